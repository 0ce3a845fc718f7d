"""Device blocks, streams and pinned staging shared by the handles
(host_pool.hpp): volumes come back byte for byte at sizes around the staging
thresholds (64 KB, the 512 KB smallest chunk, 16 MB slots and a ring's four),
from handles created and destroyed by several threads at once, whose blocks
pass from one to the other."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def round_trip(P, seed):
    from eman2_amd import Reconstructors
    rng = np.random.default_rng(seed)
    data = rng.standard_normal((P, P, P + 2)).astype(np.float32)
    norm = rng.standard_normal((P, P, P // 2 + 1)).astype(np.float32)
    r = Reconstructors.get("fourier_hip", dict(size=(P, P, P)))
    r.setup_seedandweights(data, norm)
    d, n = r.get_state()
    return np.array_equal(d, data) and np.array_equal(n, norm)


@pytest.mark.parametrize("P", [8, 24, 26, 50, 64, 128, 162, 270])
def test_volume_round_trip(P):
    assert round_trip(P, P)


def test_handles_of_several_threads():
    ok = []

    def work(k):
        for i, P in enumerate((48, 26, 96, 64, 130, 48)):
            ok.append(round_trip(P, 10 * k + i))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert len(ok) == 24 and all(ok)
