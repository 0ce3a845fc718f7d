"""trim() gives the memory of finished volumes back while other handles live:
what other allocators of the process get is what they got before."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_trim_gives_idle_blocks_back():
    from eman2_amd import Reconstructors, trim
    from test_gpu_serving_budget import free_bytes
    P = 256                                   # 135 MB of voxels, 68 MB of weights, 67 MB of real map
    keep = Reconstructors.get("fourier_hip", dict(size=(32, 32, 32)))
    keep.setup()
    r = Reconstructors.get("fourier_hip", dict(size=(P, P, P)))
    trim()
    start = free_bytes()
    for k in range(2):
        r.setup()
        r.finish(True, return_numpy=True)
        assert start - free_bytes() >= 100 << 20   # kept for the next volume
        trim()
        assert start - free_bytes() <= 16 << 20
    with pytest.raises(Exception):
        r.finish(True)                        # nothing but the idle blocks went
    r.setup()
    rng = np.random.default_rng(1)
    r.insert_slice(rng.standard_normal((P, P)).astype(np.float32), np.eye(3, 4, dtype=np.float32), 1.0)
    assert np.isfinite(r.get_state()[0]).all()
