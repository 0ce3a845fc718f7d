"""The batched agreement kernel (k_agree_batch) against the oracle where its
branches change: the packed volume (particles times operators >= P) with P/2
odd, tiles wholly beyond the insertion radius over a volume that is not zero
there, and many symmetry planes through one tile (the queue and what it does
not hold).  Bar: 1e-4 relative on the five outputs, as for the other
agreement tests (each is a ratio of float64 sums over some thousand float32
terms; the voxels hold float32 sums whose order differs)."""
import numpy as np
import pytest

from eman2_amd import synthetic as S

pytestmark = pytest.mark.gpu
KEYS = ("reconstruct_norm", "reconstruct_absqual", "reconstruct_absqual_lowres", "reconstruct_qual",
        "reconstruct_weight")


def compare(oracle, r, v, imgs, mats, w, picks, sub):
    got = r.agreement_batch(imgs, mats, w, sub=sub, apix=1.0)
    for i in picks:
        o = v.agreement(oracle.prep_particle(imgs[i], v.P), mats[i], float(w[i]), sub=sub, apix=1.0)
        for j, k in enumerate(KEYS):
            assert abs(got[i, j] - o[k]) <= 1e-4 * max(1.0, abs(o[k])), (sub, i, k, got[i, j], o[k])


@pytest.mark.parametrize("P,sym,mode,n", [(50, "c1", "gauss_2", 700), (50, "c2", "trilinear", 400),
                                          (32, "icos", "gauss_2", 40), (70, "d7", "gauss_2", 90)])
def test_packed_volume_and_planes(oracle, P, sym, mode, n):
    from eman2_amd import Reconstructors
    print("agree tiles P=%d %s %s" % (P, sym, mode), flush=True)
    B = 2 * P // 3
    imgs, mats, _ = S.particles(S.phantom(8, B / 4.0, seed=P), n, B, seed=P + 1, snr=0.5)
    w = np.linspace(0.7, 1.3, n).astype(np.float32)
    r = Reconstructors.get("fourier_hip", dict(size=(P, P, P), sym=sym, mode=mode))
    r.setup()
    r.insert_batch(imgs, mats, w)
    v = oracle.Volume(P, sym, mode)
    for im, m, wi in zip(imgs, mats, w):
        v.insert(oracle.prep_particle(im, P), m, float(wi))
    compare(oracle, r, v, imgs, mats, w, range(0, n, n // 4), True)


def test_volume_beyond_the_insertion_radius(oracle):
    from eman2_amd import Reconstructors
    P, n = 96, 120
    rng = np.random.default_rng(9)
    data = rng.standard_normal((P, P, P + 2)).astype(np.float32)
    norm = rng.uniform(0.5, 2.0, (P, P, P // 2 + 1)).astype(np.float32)
    imgs, mats, _ = S.particles(S.phantom(8, 14.0, seed=3), n, 60, seed=4, snr=0.5)
    w = np.ones(n, np.float32)
    r = Reconstructors.get("fourier_hip", dict(size=(P, P, P)))
    r.setup_seedandweights(data, norm)
    v = oracle.Volume(P, "c1", "gauss_2")
    v.data[...] = data.reshape(v.data.shape)
    v.norm[...] = norm.reshape(v.norm.shape)
    # compared as if their contributions were in the volume: the removal leaves weights of either sign on
    # both sides, away from zero
    compare(oracle, r, v, imgs, mats, w, (0, 5, 50), False)
    r.insert_batch(imgs, mats, w)
    for im, m in zip(imgs, mats):
        v.insert(oracle.prep_particle(im, P), m, 1.0)
    compare(oracle, r, v, imgs, mats, w, (0, 5, 50), True)
