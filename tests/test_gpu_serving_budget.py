"""A server's jobs and the idle blocks of finished ones together stay within
its budget: jobs of mixed sizes, one after another and two at a time, and the
device memory in use beyond that before the server at every moment.  64 MB
are allowed for what the runtime takes itself (queues, code, scratch)."""
import ctypes
import threading
import time

import numpy as np
import pytest

from eman2_amd import synthetic as S

pytestmark = pytest.mark.gpu
SLACK = 64 << 20


def free_bytes():
    from test_gpu_parity import _hip_runtime
    f, t = ctypes.c_size_t(), ctypes.c_size_t()
    assert _hip_runtime().hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
    return f.value


def job(P, n):
    B = P // 2
    imgs, mats, _ = S.particles(S.phantom(3, B * 0.2, seed=P), n, B, seed=P + 1, snr=1.0)
    return dict(size=P, imgs=imgs, xforms=mats)


@pytest.mark.parametrize("active", [1, 2])
def test_admitted_and_idle_bytes_within_the_budget(active):
    from eman2_amd.serving import Server
    jobs = [job(P, 64) for P in (96, 128, 160, 112, 192, 144, 128)]
    with_all = Server(max_active=1, chunk=64)  # loads the kernels, and tells the footprints
    need = max(with_all.poll(with_all.submit(**j))["footprint_bytes"] for j in jobs)
    with_all.drain()
    with_all.close()
    budget = int(need * (1.05 if active == 1 else 1.6))
    start = free_bytes()
    least, stop = [start], threading.Event()

    def watch():
        while not stop.is_set():
            least[0] = min(least[0], free_bytes())
            time.sleep(0.0005)

    t = threading.Thread(target=watch)
    t.start()
    s = Server(hbm_budget_bytes=budget, max_active=active, chunk=64)
    for k in range(3):
        ids = [s.submit(**j) for j in jobs]
        s.drain()
        assert [s.poll(i)["state"] for i in ids] == ["done"] * len(jobs)
        assert all(np.isfinite(s.result(i)).all() for i in ids)
    stop.set()
    t.join()
    print("budget %d MB, most %d MB, idle %d MB" % (budget >> 20, (start - least[0]) >> 20, (start - free_bytes()) >> 20),
          flush=True)
    assert start - free_bytes() <= budget + SLACK
    assert start - least[0] <= budget + SLACK
    s.close()
    assert start - free_bytes() <= SLACK
