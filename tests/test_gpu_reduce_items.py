"""Batches whose bricks have several work items each (summed into the first
one before the merge) against the same particles inserted in calls of one,
which have fewer items than the grid has bricks and go to the merge as they
are.  The partial brick's length differs by mode (2187, 1920, 648-3000 floats
for units of 256), the items per brick with the cap on slices per item: 1 to
several hundred, in groups of 4.  Tolerance: float32 sums of the same at most
few hundred contributions per voxel in another order: 1e-5."""
import numpy as np
import pytest

from eman2_amd import synthetic as S
from eman2_amd.metrics import max_rel_err, weight_rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,sym,mode,spi", [(16, "c1", "gauss_2", 1), (16, "c1", "gauss_2", 1024), (24, "d2", "trilinear", 3),
                                            (40, "c4", "gauss_2", 16), (24, "c1", "gauss_var", 1), (20, "c1", "gridding_5", 2),
                                            (20, "c1", "gauss_3", 5)])
def test_several_items_per_brick(P, sym, mode, spi):
    from eman2_amd import Reconstructors
    print("reduce items P=%d %s %s spi=%d" % (P, sym, mode, spi), flush=True)
    n, B = 300, 12
    imgs, mats, _ = S.particles(S.phantom(5, 4.0, seed=2), n, B, seed=4, snr=1.0)
    w = np.linspace(0.5, 1.5, n).astype(np.float32)
    state = []
    for step in (n, 1):
        r = Reconstructors.get("fourier_hip", dict(size=(P, P, P), sym=sym, mode=mode))
        r.set_tuning(slices_per_item=spi)
        r.setup()
        for a in range(0, n, step):
            r.insert_batch(imgs[a:a + step], mats[a:a + step], w[a:a + step])
        state.append(r.get_state())
    assert weight_rel_err(state[0][1], state[1][1]) <= 1e-5
    assert max_rel_err(state[0][0], state[1][0]) <= 1e-5
