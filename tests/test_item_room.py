"""The room of the batched insertion's work item list (ensure_bins in
engine.cpp): sized for the largest batch of a handle, it holds every smaller
batch too, whose items take fewer slices each (item_slices).  Replays the
sizing over inserters, pads, caps on the slices per item and batch sizes, with
at most 4 bricks of a brick column per slice (along the dominant axis a brick
column spans (sum of the other two edges) / edge <= 2.7 bricks).  (CPU only.)"""
import math

import pytest

CUS = 256


def geom(P, kind):
    """nb, nbz, bs, bsz, wide of brick_geom (the origin ranges' lower ends: floor(p - 2.5) etc.)"""
    H = P // 2
    bs, bsz, ow = {"gauss_2": (8, 8, -H - 1), "gauss6": (3, 5, -H - 4), "wide": (4, 4, -H - 4)}[kind]
    return (H - ow + 1 + bs - 1) // bs, (H - ow + 1 + bsz - 1) // bsz, bs, bsz, kind != "gauss_2"


def item_slices(P, g, n, most):
    nb, nbz, bs, bsz, wide = g
    pb2 = (P + 8.0) ** 2 * (2 * bs + bsz) / (3.0 * bs * bs * bsz)
    k = (6.0 if wide else 8.0) * math.sqrt(0.63 * pb2 * n / (16.0 * CUS))
    return int(min(float(most), max(16.0, k)))


@pytest.mark.parametrize("kind", ["gauss_2", "gauss6", "wide"])
@pytest.mark.parametrize("most", [1, 2, 16, 17, 33, 250, 1024, 5000])
def test_smaller_batches_fit(kind, most):
    for P in (8, 26, 96, 384, 1024):
        g = geom(P, kind)
        nb, nbz = g[:2]
        keys, columns = 3 * nb * nb * nbz, nb * max(nb, nbz)
        for N in (1, 7, 100, 1000, 3001, 12000, 40000):
            if 5 * columns * N > 2 ** 31 - 1:
                continue
            K = item_slices(P, g, N, most)
            room = 5 * columns * N // K * (5 if K < most else 4) // 4 + keys + 1
            steps = set(range(1, N + 1, max(1, N // 400))) | {N}
            for n in steps:
                assert 4 * columns * n / item_slices(P, g, n, most) + keys <= room, (P, N, n)
