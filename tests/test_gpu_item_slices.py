"""Slices per work item chosen by the batch's size (item_slices in
engine.cpp): batches of any size on one handle, in any order, give the sums
that items of two slices give, and fit the item buffers sized for the largest
batch.  Tolerance: both are float32 sums of the same contributions in another
order, at most a few hundred per voxel: 1e-5 of the voxel's weight, of the
largest sum."""
import numpy as np
import pytest

from eman2_amd import synthetic as S
from eman2_amd.metrics import max_rel_err, weight_rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,sym,mode,graph", [(24, "d2", "gauss_2", 0), (24, "d2", "gauss_2", 1), (32, "c1", "gauss_var", 0),
                                              (32, "c4", "gridding_7", 0)])
def test_batches_of_any_size(P, sym, mode, graph):
    import ctypes

    from eman2_amd import Reconstructors
    from test_gpu_parity import _hip_runtime
    print("item slices P=%d %s %s graph=%d" % (P, sym, mode, graph), flush=True)
    n, B = 700, 16
    imgs, mats, _ = S.particles(S.phantom(5, 5.0, seed=2), n, B, seed=3, snr=1.0)
    hip = _hip_runtime()
    dev = ctypes.c_void_p()
    assert hip.hipMalloc(ctypes.byref(dev), imgs.nbytes) == 0
    assert hip.hipMemcpy(dev, imgs.ctypes.data, imgs.nbytes, 1) == 0  # host to device
    w = np.linspace(0.5, 1.5, n).astype(np.float32)
    state = {}
    for spi in (2, 1024):
        r = Reconstructors.get("fourier_hip", dict(size=(P, P, P), sym=sym, mode=mode))
        r.set_tuning(slices_per_item=spi, graph=graph)
        r.setup()
        for a, b in ((0, 500), (500, 501), (501, 560), (560, 700)):
            r.insert_batch(dev.value + 4 * B * B * a, mats[a:b], w[a:b], box=B)
        state[spi] = r.get_state()
    assert hip.hipFree(dev) == 0
    assert weight_rel_err(state[1024][1], state[2][1]) <= 1e-5
    assert max_rel_err(state[1024][0], state[2][0]) <= 1e-5
