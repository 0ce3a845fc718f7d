"""A projector that is given one map after another projects the map of the
call: the same array changed in place, where its content differs in a few
voxels only, and another array at the address of one that is gone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROT = np.array([[0.36, 0.48, -0.8, 0], [-0.8, 0.6, 0, 0], [0.48, 0.64, 0.6, 0]], np.float32)


@pytest.mark.parametrize("P", [8, 64, 96])
def test_map_changed_in_place(P):
    from eman2_amd.projector import Projectors
    print("projector maps P=%d" % P, flush=True)
    rng = np.random.default_rng(P)
    vol = rng.standard_normal((P, P, P)).astype(np.float32)
    pr = Projectors.get("gauss_fft", {"returnfft": 1})
    before = pr.project_batch(vol, [ROT])
    vol[P // 2 + 1, P // 2 + 1, P // 2 - 1] += 50.0
    after = pr.project_batch(vol, [ROT])
    fresh = Projectors.get("gauss_fft", {"returnfft": 1}).project_batch(vol.copy(), [ROT])
    assert np.array_equal(after, fresh)
    assert not np.array_equal(after, before)
    vol[:] = vol[::-1, ::-1, ::-1].copy()      # the same sum of voxels
    assert np.array_equal(pr.project_batch(vol, [ROT]),
                          Projectors.get("gauss_fft", {"returnfft": 1}).project_batch(vol.copy(), [ROT]))


def test_maps_one_after_another():
    from eman2_amd.projector import Projectors
    P = 48
    pr = Projectors.get("gauss_fft", {"transform": ROT})
    for k in range(4):
        vol = np.zeros((P, P, P), np.float32)  # masked: most of it zero
        vol[20 + k:28, 18:30, 22:30] = 1.0 + k
        assert np.array_equal(pr.project3d(vol).numpy(),
                              Projectors.get("gauss_fft", {"transform": ROT}).project3d(vol).numpy())
        del vol
