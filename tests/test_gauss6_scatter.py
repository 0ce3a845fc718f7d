"""The 6-cell Gaussians' scatter (k_scatter_gauss6 in insert_kernels.hip).

On the CPU: the table index by one FMA rounded toward zero equals the
reference's double expression (Util::fast_exp, libEM/util.cpp:788-800), and
the binning on bricks of 3 x 3 x 5 stencil origins with the kernel's row
enumeration reaches every pixel of the reference loop
(libEM/reconstructor.cpp:1166-1209) once, in the brick owning its origin.  On
the GPU: parity with the oracle where each of the kernel's three forms of the
passes runs (stencils inside the table, past it, clamped or dropped)."""
import math
from fractions import Fraction

import numpy as np
import pytest

from eman2_amd import synthetic as S
from eman2_amd.metrics import max_rel_err, weight_rel_err
from eman2_amd.transform import euler_eman_matrix
from test_binning import _frame
from test_brick_scatter import ANGLES, DLT, EPS, exact_coords, f32

BS = (3, 3, 5)
CAND = f32(3.2838)
CTF = dict(voltage=300.0, cs=2.7, ampcont=10.0, apix=1.0)


def table_offset(f):
    """bits & 0xffc of f * 50 + (2^21 + 1/2) rounded toward zero to float32"""
    exact = Fraction(float(f)) * 50 + Fraction(4194305, 2)
    quarter = exact * 4                       # the spacing of floats in [2^21, 2^22) is 1/4
    return (quarter.numerator // quarter.denominator - (1 << 23)) & 0xffc


def test_table_index_by_one_rounded_down_fma():
    rng = np.random.default_rng(3)
    edges = ((np.arange(1000) - 0.5) / 50.0).clip(min=0).astype(np.float32)
    near = [np.nextafter(edges, d).astype(np.float32) for d in (f32(0), f32(30))]
    f = np.concatenate([edges, *near, rng.uniform(0, 19.98, 4000).astype(np.float32), [f32(0), f32(1e-30)],
                        (rng.integers(0, 1279, 500) / 64.0).astype(np.float32)])  # dyadic: exact halves of an index
    f = f[(f >= 0) & (f <= 19.98)]
    want = (f.astype(np.float64) * 50.0 + 0.5).astype(np.int64)
    assert [table_offset(v) for v in f] == list(4 * want)
    assert want.max() < 1000


def bricks(m, P, corners):
    """k_bin_cols on 3 x 3 x 5 bricks from origin -P/2 - 4 (p from -P/2 - 1.5)"""
    H = P // 2
    ow, po = -H - 4, -H - 4 + 2.5
    nb = [-(-(H - ow + 1) // b) for b in BS]
    u, v, n, a, b1, b2 = _frame(m)
    dlt, hd = 1e-3, 0.5 * math.sqrt(sum(b * b for b in BS))
    rr = math.sqrt(H * H + H) + hd + 0.01
    r1, r2 = -n[b1] / n[a], -n[b2] / n[a]
    for c2 in range(nb[b2]):
        for c1 in range(nb[b1]):
            L1, L2 = po + BS[b1] * c1 - dlt, po + BS[b2] * c2 - dlt
            pas = [r1 * p1 + r2 * p2 for p1 in (L1, L1 + BS[b1] + 2 * dlt) for p2 in (L2, L2 + BS[b2] + 2 * dlt)]
            lo = max(math.floor((min(pas) - dlt - po) / BS[a]), 0)
            hi = min(math.floor((max(pas) + dlt - po) / BS[a]), nb[a] - 1)
            assert hi - lo < 5                # the room of the brick list
            for ca in range(lo, hi + 1):
                bc = [0, 0, 0]
                bc[a], bc[b1], bc[b2] = ca, c1, c2
                c = np.array([po + BS[d] * bc[d] + 0.5 * BS[d] for d in range(3)])
                s, t = c @ u, c @ v
                rh = hd + 0.01
                if s < -rh or not ((s <= H + rh and -H - rh <= t <= H - 1 + rh) if corners else s * s + t * t <= rr * rr):
                    continue
                yield bc, [ow + BS[d] * bc[d] for d in range(3)], [f32(po + BS[d] * bc[d]) for d in range(3)]


def enumerated(m, pl, H, corners):
    """the pixels the kernel's rows give for one (slice, brick) pair: at most 7 rows"""
    mm = [f32(v) for v in (*m[0, :3], *m[1, :3])]
    pc = [f32(pl[d] + f32(0.5 * BS[d])) for d in range(3)]
    sc = f32(f32(f32(pc[0] * mm[0]) + f32(pc[1] * mm[1])) + f32(pc[2] * mm[2]))
    tc = f32(f32(f32(pc[0] * mm[3]) + f32(pc[1] * mm[4])) + f32(pc[2] * mm[5]))
    xc0, yc0 = int(np.rint(sc)), int(np.rint(tc))
    fs, ft = f32(sc - f32(xc0)), f32(tc - f32(yc0))
    for r in range(8):
        dy = math.ceil(f32(ft - CAND)) + r
        y = yc0 + dy
        if not (f32(dy) <= f32(ft + CAND) and -H <= y <= H - 1):
            continue
        assert r < 7
        xl, xh = f32(fs - CAND), f32(fs + CAND)
        for d in range(3):
            if abs(mm[d]) >= 0.05:
                b0 = f32(f32(pl[d] - f32(f32(f32(xc0) * mm[d]) + f32(f32(yc0) * mm[3 + d]))) - f32(f32(dy) * mm[3 + d]))
                iu = f32(f32(1) / mm[d])
                t0, t1 = f32(f32(b0 - DLT) * iu), f32(f32(f32(b0 + f32(BS[d])) + DLT) * iu)
                xl, xh = max(xl, min(t0, t1)), min(xh, max(t0, t1))
        a, b = max(math.ceil(f32(xl - EPS)), -xc0), min(math.floor(f32(xh + EPS)), H - xc0)
        if not corners:
            b = min(b, math.isqrt(H * H + H - y * y) - xc0)
        yield from ((xc0 + dx, y) for dx in range(a, b + 1))


@pytest.mark.parametrize("P", [16, 26, 32])
def test_every_pixel_in_the_brick_of_its_origin(P):
    H = P // 2
    rng = np.random.default_rng(P)
    for ang in ANGLES + [tuple(rng.random(3) * (360, 180, 360)) for _ in range(3)]:
        m = euler_eman_matrix(*ang)
        for corners in (False, True):
            want = {}
            for y in range(-H, H):
                for x in range(H + 1):
                    if corners or x * x + y * y <= H * H + H:
                        org = [math.floor(float(q) - 2.5) for q in exact_coords(x, y, m, P)]
                        if min(org) >= -H - 4 and max(org) <= H:   # higher origins reach no cell
                            want[x, y] = org
            got = {}
            for _, lo, pl in bricks(m, P, corners):
                pix = list(enumerated(m, pl, H, corners))
                assert len(pix) == len(set(pix))
                for p in pix:
                    if p in want and all(lo[d] <= want[p][d] < lo[d] + BS[d] for d in range(3)):
                        got[p] = got.get(p, 0) + 1
            assert set(got) == set(want) and set(got.values()) == {1}, (ang, corners)


@pytest.mark.gpu
@pytest.mark.parametrize("P,sym,mode,n,corners", [
    (26, "c1", "gauss_var", 30, False),    # the whole stencil grid within a few bricks, clamped on most
    (48, "d2", "gauss_5", 20, True),       # one width, past the table in the stencils' corners
    (240, "c1", "gauss_var", 4, False),    # |p| to 120: stencils inside the table beyond 87
    (240, "c2", "fourier_iter", 3, False),
])
def test_parity(oracle, P, sym, mode, n, corners):
    from eman2_amd import Reconstructors
    print("gauss6 P=%d %s %s" % (P, sym, mode), flush=True)
    B = int(P * 0.66) // 2 * 2
    imgs, mats, _ = S.particles(S.phantom(8, 0.2 * P, seed=P), n, B, seed=P + 1, snr=1.0)
    for i, ang in enumerate(ANGLES[:3]):       # axis-aligned slices: positions on cell boundaries
        mats[i, :, :3] = euler_eman_matrix(*ang)[:, :3]
    w = np.linspace(0.5, 1.5, n).astype(np.float32)
    w[1], w[-1] = 2e-3, 3e-27                  # weights of the general form
    if mode == "fourier_iter":
        r = Reconstructors.get("fourier_iter_hip", dict(size=(P, P, P), sym=sym))
    else:
        r = Reconstructors.get("fourier_hip", dict(size=(P, P, P), sym=sym, mode=mode, corners=corners))
    r.setup()
    r.insert_batch(imgs, mats, w)
    gd, gn = r.get_state()
    v = oracle.Volume(P, sym, mode)
    for im, m, wi in zip(imgs, mats, w):
        kw = {} if mode == "fourier_iter" else {"corners": corners}
        v.insert(oracle.prep_particle(im, P), m, float(wi), **kw)
    # float32 sums of at most a few hundred terms each: relative 1e-5 of the voxel's own sum
    big = v.norm > 1e-20
    assert weight_rel_err(np.where(big, gn, 0), np.where(big, v.norm, 0)) <= 1e-5
    assert np.array_equal(gn > 0, v.norm > 0)
    assert max_rel_err(gd, v.data) <= 1e-5


@pytest.mark.gpu
def test_not_finite_pixels_stay_in_their_stencils(oracle):
    """an infinite pixel value reaches the cells of its stencil that are not dropped, and no other"""
    from eman2_amd import Reconstructors
    P, n = 32, 3
    imgs, mats, _ = S.particles(S.phantom(6, 6.0, seed=5), n, 20, seed=6, snr=2.0)
    imgs[1, 4, 4] = np.inf
    r = Reconstructors.get("fourier_hip", dict(size=(P, P, P), mode="gauss_var"))
    r.setup()
    r.insert_batch(imgs, mats, np.ones(n, np.float32))
    gd, gn = r.get_state()
    v = oracle.Volume(P, "c1", "gauss_var")
    for im, m in zip(imgs, mats):
        v.insert(oracle.prep_particle(im, P), m, 1.0)
    assert np.array_equal(np.isfinite(gd), np.isfinite(v.data)) and not np.isfinite(gd).all()
    assert weight_rel_err(gn, v.norm) <= 1e-5
