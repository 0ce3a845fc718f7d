"""The footprint by which the server admits a job covers the device memory
that the job's handle takes, over inserters, symmetries and batch sizes (small
batches take fewer slices per work item, so more partial bricks per slice).
32 MB are allowed for what the runtime takes itself.  The handle's memory stays
within 1.1 times `mb` MB, what it takes with bricks of 8^3 (gauss_2) and 4^3
origins (the others) and 1,024 slices per item, where work items by the
thousand are not what a small volume needs to fill the GPU (None)."""
import numpy as np
import pytest

from eman2_amd import synthetic as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,sym,P,n,mb", [("gauss_2", "c1", 96, 30, 42), ("gauss_2", "c1", 192, 250, 352),
                                             ("gauss_2", "d7", 160, 60, 188), ("gauss_2", "icos", 192, 100, 394),
                                             ("gauss_var", "c1", 96, 100, 124), ("gauss_var", "c1", 256, 300, 1780),
                                             ("gauss_var", "d7", 192, 100, 844), ("gridding_7", "c1", 128, 120, 330), ("gauss_3", "c4", 192, 200, 362),
                                             ("gauss_var", "c1", 36, 500, None), ("kaiser_bessel", "c1", 96, 3, 24)])
def test_footprint_covers_the_handle(mode, sym, P, n, mb):
    from eman2_amd import Reconstructors, trim
    from eman2_amd.serving import Server
    from test_gpu_serving_budget import free_bytes
    print("footprint %s %s P=%d n=%d" % (mode, sym, P, n), flush=True)
    B = 32
    imgs, mats, _ = S.particles(S.phantom(3, 8.0, seed=P), n, B, seed=P + 1, snr=1.0)
    s = Server(max_active=1, chunk=n)
    said = s.poll(s.submit(size=P, imgs=imgs, xforms=mats, sym=sym, mode=mode))["footprint_bytes"]
    s.drain()
    s.close()
    trim()
    before = free_bytes()
    r = Reconstructors.get("fourier_hip", dict(size=(P, P, P), sym=sym, mode=mode))
    r.set_tuning(chunk=n)
    r.setup()
    r.insert_batch(imgs, mats, np.ones(n, np.float32))
    trim()
    held = before - free_bytes()
    print("footprint %.1f MB, held %.1f MB" % (said / 2 ** 20, held / 2 ** 20), flush=True)
    assert held <= said + (32 << 20)
    assert mb is None or held <= 1.1 * (mb << 20) + (8 << 20)


@pytest.mark.parametrize("mode,sym,P,n,mb", [("gauss_var", "c1", 96, 100, 252), ("gauss_var", "c1", 256, 300, 4140),
                                             ("gauss_5", "d7", 192, 100, 2222)])
def test_budget_of_the_larger_bricks_admits(mode, sym, P, n, mb):
    """a budget (MB) that admitted the job with bricks of 4^3 origins still does"""
    from eman2_amd.serving import Server
    imgs, mats, _ = S.particles(S.phantom(3, 8.0, seed=P), n, 32, seed=P + 1, snr=1.0)
    s = Server(max_active=1, chunk=n, hbm_budget_bytes=mb << 20)
    i = s.submit(size=P, imgs=imgs, xforms=mats, sym=sym, mode=mode)
    s.drain()
    st = s.poll(i)
    s.close()
    print("footprint %s %s P=%d: %.1f MB, %s" % (mode, sym, P, st["footprint_bytes"] / 2 ** 20, st["state"]), flush=True)
    assert st["state"] == "done"
