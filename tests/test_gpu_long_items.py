"""Work items of many times 64 slices: the list entries of an item are read 64
at a time, one group of slices ahead.  Thousands of particles that share a few
images and orientations fill the bricks' items up to the cap; the oracle takes
each image once with the sum of its weights (the insertion is linear in them).
Items of 65 to 250 slices, whole and not in the groups of 4, 8 or 64.
Tolerance: a cell is the float32 sum of some 4,000 terms per item (gauss_2:
1,000), whose roundings add up like a random walk to 64 x 2^-24, over tens of
items summed the same way: 2e-5 of the voxel's weight and of the largest sum."""
import numpy as np
import pytest

from eman2_amd import synthetic as S
from eman2_amd.metrics import max_rel_err, weight_rel_err
from eman2_amd.transform import euler_eman_matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,P,n,most", [("gauss_var", 48, 13001, 1024), ("gauss_var", 48, 12000, 65),
                                           ("gauss_5", 40, 16000, 127), ("fourier_iter", 48, 13001, 1024),
                                           ("reference", 48, 13001, 129), ("gauss_2", 96, 10301, 1024),
                                           ("gauss_2", 96, 10301, 65), ("trilinear", 96, 10301, 126),
                                           ("gridding_5", 40, 13000, 131)])
def test_items_of_many_slices(oracle, mode, P, n, most):
    from eman2_amd import Reconstructors
    print("long items %s P=%d n=%d" % (mode, P, n), flush=True)
    B, d = 20, 6
    ph = S.phantom(6, 5.0, seed=3)
    imgs, mats, _ = S.particles(ph, d, B, seed=4, snr=1.0)
    mats[0, :, :3] = euler_eman_matrix(0.0, 0.0, 0.0)[:, :3]   # one axis-aligned slice
    rng = np.random.default_rng(5)
    pick = rng.integers(0, d, n)
    w = rng.uniform(0.5, 1.5, n).astype(np.float32)
    it = mode in ("fourier_iter", "reference")
    if it:
        r = Reconstructors.get("fourier_iter_hip", dict(size=(P, P, P)))
    else:
        r = Reconstructors.get("fourier_hip", dict(size=(P, P, P), mode=mode))
    r.set_tuning(slices_per_item=most)
    v = oracle.Volume(P, "c1", "fourier_iter" if it else mode)
    if mode == "reference":
        ref = (S.phantom_volume(ph, P) * 40.0).astype(np.float32)
        r.setup_seed(ref, 1.0)
        v.setup_iter_ref(ref)
    else:
        r.setup()
    r.insert_batch(imgs[pick], mats[pick], w)
    st = r.get_stats()
    per_item = st["pairs"] / st["items"]
    print("%.0f slices per item" % per_item, flush=True)
    assert st["chunks"] == 1 and min(most, 110) * 0.5 < per_item <= most
    gd, gn = r.get_state()
    for k in range(d):
        v.insert(oracle.prep_particle(imgs[k], P), mats[k], float(w[pick == k].astype(np.float64).sum()))
    big = v.norm > 1e-20
    assert weight_rel_err(np.where(big, gn, 0), np.where(big, v.norm, 0)) <= 2e-5
    assert max_rel_err(gd, v.data) <= 2e-5
