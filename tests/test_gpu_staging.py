"""Copies to the host through the staging ring, which a pool sets up for a
copy of 16 MB or after its first small ones: with a handle that has made one, volumes come back byte
for byte at sizes around the thresholds (64 KB, the 512 KB smallest chunk, 16
MB slots and a ring's four), from one thread and from several at once."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture
def warm():
    from eman2_amd import Reconstructors
    r = Reconstructors.get("fourier_hip", dict(size=(192, 192, 192)))
    r.setup()
    r.get_state()                              # 28 MB and 14 MB
    return r


@pytest.mark.parametrize("P", [8, 24, 26, 50, 64, 128, 162, 270])
def test_volume_round_trip(warm, P):
    from test_gpu_host_pool import round_trip
    assert round_trip(P, P)


def test_several_threads(warm):
    from test_gpu_host_pool import round_trip
    ok = []
    threads = [threading.Thread(target=lambda k=k: ok.extend(round_trip(P, 10 * k + P) for P in (48, 64, 130, 96, 26)))
               for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert len(ok) == 30 and all(ok)


def test_projections_and_slices(warm):
    """the batched prep and the projector against themselves in smaller calls"""
    from eman2_amd import Reconstructors
    from eman2_amd.projector import Projectors
    rng = np.random.default_rng(2)
    vol = rng.standard_normal((100, 100, 100)).astype(np.float32)
    m = np.zeros((40, 3, 4), np.float32)
    for i in range(len(m)):
        q, _ = np.linalg.qr(rng.standard_normal((3, 3)))
        m[i, :, :3] = q * np.sign(np.linalg.det(q))
    pr = Projectors.get("gauss_fft", {"returnfft": 1})
    whole = pr.project_batch(vol, m)           # 1.6 MB; one slice: 41 KB, not staged
    assert np.array_equal(whole, np.concatenate([pr.project_batch(vol, m[i:i + 1]) for i in range(len(m))]))
    imgs = rng.standard_normal((40, 64, 64)).astype(np.float32)
    r = Reconstructors.get("fourier_hip", dict(size=(100, 100, 100)))
    whole = r.prep_batch(imgs)
    assert np.array_equal(whole, np.concatenate([r.prep_batch(imgs[i:i + 1]) for i in range(len(imgs))]))
