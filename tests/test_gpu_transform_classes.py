"""The transform passes at the edges of their length classes: pads up to 128,
256, 400, 512, 640 and 1,024 take tiles of different widths and register
arrays, with every radix of the plans (2-8, 11, 13) among them.  The prep of
odd and even boxes, the flip and resampling, and the finish, each at the smallest pad, at a class's last length and at one just
past it.  Bars: the prep's 2e-5 and the flip's 1e-4 as elsewhere; the finish
is two or three passes of the same transforms (2e-5)."""
import numpy as np
import pytest
import scipy.fft

from eman2_amd.metrics import max_rel_err, weight_rel_err
from test_gpu_configs import _xforms_with_2d, recon

pytestmark = pytest.mark.gpu
CTF = dict(voltage=300.0, cs=2.7, ampcont=10.0, apix=1.0)


@pytest.mark.parametrize("B,P,ctf", [(5, 8, True), (8, 8, False), (17, 22, True), (85, 128, True), (87, 130, False),
                                     (169, 256, True), (173, 260, True), (267, 400, False), (271, 416, True),
                                     (341, 512, True), (347, 520, False), (426, 640, True), (433, 650, True),
                                     (682, 1024, True)])
def test_prep(oracle, B, P, ctf):
    n = 3
    rng = np.random.default_rng(B + P)
    imgs = (rng.standard_normal((n, B, B)) + 3.0).astype(np.float32)
    dfs = rng.uniform(0.8, 2.5, n).astype(np.float32) if ctf else None
    g = recon(P).prep_batch(imgs, defocus=dfs, ctf=CTF if ctf else None)
    for i in range(n):
        o = oracle.prep_particle(imgs[i], P, dict(CTF, defocus=float(dfs[i])) if ctf else None)
        assert max_rel_err(g[i], o) <= 2e-5, (i, max_rel_err(g[i], o))


@pytest.mark.parametrize("B,P,flip", [(5, 8, True), (17, 22, True), (85, 128, False), (87, 130, True), (169, 256, True),
                                      (173, 260, True), (271, 400, False),
                                      (273, 416, True), (351, 528, True), (433, 650, True)])
def test_flip_and_resample(oracle, B, P, flip):
    n = 3
    rng = np.random.default_rng(B + P)
    imgs = (rng.standard_normal((n, B, B)) + 1.0).astype(np.float32)
    dfs = rng.uniform(0.8, 2.5, n).astype(np.float32) if flip else None
    mats = _xforms_with_2d(n, P, scale=True)
    w = np.ones(n, np.float32)
    r = recon(P)
    r.insert_batch(imgs, mats, w, defocus=dfs, ctf=CTF if flip else None)
    gd, gn = r.get_state()
    v = oracle.Volume(P, "c1", "gauss_2")
    for i in range(n):
        c = dict(CTF, defocus=float(dfs[i])) if flip else None
        v.insert(oracle.prep_particle(imgs[i], P, c, xform=mats[i]), mats[i], 1.0)
    assert weight_rel_err(gn, v.norm) <= 1e-4
    assert max_rel_err(gd, v.data) <= 1e-4


@pytest.mark.parametrize("P", [8, 22, 128, 130, 260, 416, 520, 650])
def test_finish(P):
    """setup_seedandweights + finish: the inverse of the map's own transform"""
    rng = np.random.default_rng(P)
    a = rng.standard_normal((3, P)).astype(np.float32)
    vol = (a[0][:, None, None] * a[1][None, :, None] * a[2][None, None, :]).astype(np.float32)
    vol[P // 3, P // 2, P // 4] += np.float32(5.0)
    f = scipy.fft.rfftn(scipy.fft.ifftshift(vol), workers=8)
    norm = np.ones((P, P, P // 2 + 1), np.float32)
    # normalize_threed takes self + partner on the planes x = 0 and x = P/2, the
    # self-paired cells (coordinates 0 or P/2 each) apart: undo it in the weights
    norm[:, :, 0] = norm[:, :, -1] = 0.5
    H = P // 2
    for z in (0, H):
        for y in (0, H):
            for x, once in ((0, ((0, 0),)), (H, ((0, 0), (H, H)))):
                norm[z, y, x] = 1.0 if (z, y) in once else 0.5
    data = np.empty((P, P, P + 2), np.float32)
    data[..., 0::2] = f.real
    data[..., 1::2] = f.imag
    del f
    r = recon(P)
    r.setup_seedandweights(data, norm)
    del data, norm
    out = r.finish(True)
    got = out.numpy() if hasattr(out, "numpy") else np.asarray(out)
    assert max_rel_err(got, vol) <= 2e-5
