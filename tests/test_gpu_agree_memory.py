"""The batched agreement's packed copy of the volume (16 bytes a voxel) is
taken for the call and given back with it, with and without a phase flip and a
2-D transform."""
import numpy as np
import pytest

from eman2_amd import synthetic as S

pytestmark = pytest.mark.gpu
CTF = {"voltage": 300.0, "cs": 2.7, "ampcont": 10.0, "apix": 1.0}


@pytest.mark.parametrize("shifts", [False, True])
def test_packed_volume_is_given_back(shifts):
    from eman2_amd import Reconstructors, trim
    from test_gpu_serving_budget import free_bytes
    P, B, n = 256, 64, 256
    print("agreement memory shifts=%d" % shifts, flush=True)
    imgs, mats, dfs = S.particles(S.phantom(3, 16.0, seed=1), n, B, seed=2, snr=1.0, ctf={})
    if shifts:
        mats[:, :2, 3] = 2.5
    w = np.ones(n, np.float32)
    r = Reconstructors.get("fourier_hip", dict(size=(P, P, P)))
    r.set_tuning(chunk=64)                     # the same staging for both calls
    r.setup()
    r.insert_batch(imgs, mats, w, dfs, CTF)
    r.agreement_batch(imgs[:200], mats[:200], w[:200], dfs[:200], CTF)  # fewer than P: the volume as it is
    trim()
    before = free_bytes()
    r.agreement_batch(imgs, mats, w, dfs, CTF)
    trim()
    assert before - free_bytes() <= 8 << 20    # the packed volume takes 136 MB
