"""The room of the batched insertion's work item list (ensure_bins in
engine.cpp): sized for the largest batch of a handle, it holds every smaller
batch too, whose items take fewer slices each (item_slices).  Replays the sizing
over inserters, pads, caps on the slices per item and batch sizes, with as
many list entries as a slice can take (list_per_slice: its span along the
dominant axis in each brick column, tested over random planes).  (CPU only.)"""
import math

import numpy as np
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


def column_bricks(g):
    """most bricks of a column along x or y, and along z"""
    _, _, bs, bsz, _ = g
    return int((bs + bsz + 0.01) / bs) + 2, int((2 * bs + 0.01) / bsz) + 2


def list_per_slice(g):
    (xy, z), (nb, nbz) = column_bricks(g), g[:2]
    return max(xy * nb * nbz, z * nb * nb)


@pytest.mark.parametrize("kind", ["gauss_2", "gauss6", "wide"])
def test_bricks_of_a_column(kind):
    g = geom(96, kind)
    edge, most = [g[2], g[2], g[3]], column_bricks(g)
    rng = np.random.default_rng(3)
    corner = np.concatenate([[(1.0, 1.0), (1.0, -1.0), (-1.0, -1.0), (0.0, 1.0)], rng.uniform(-1, 1, (400, 2))])
    for a, (b1, b2) in enumerate(((1, 2), (0, 2), (0, 1))):
        for r1, r2 in corner:                  # the plane's slopes along the dominant axis a
            off = rng.uniform(-50, 50, 50)
            x = r1 * edge[b1] * np.array([0.0, 1, 0, 1]) + r2 * edge[b2] * np.array([0.0, 0, 1, 1])
            pad = (abs(r1) + abs(r2)) * 1e-3 + 1e-3
            lo, hi = np.floor((off + x.min() - pad) / edge[a]), np.floor((off + x.max() + pad) / edge[a])
            assert (hi - lo + 1).max() <= most[0 if a < 2 else 1]


@pytest.mark.parametrize("kind", ["gauss_2", "gauss6", "wide"])
@pytest.mark.parametrize("most", [1, 2, 16, 17, 33, 250, 1024, 5000])
def test_smaller_batches_fit(kind, most):
    for P in (8, 26, 96, 384, 1024):
        g = geom(P, kind)
        nb, nbz = g[:2]
        keys, pairs = 3 * nb * nb * nbz, list_per_slice(g)
        for N in (1, 7, 100, 1000, 3001, 12000, 40000):
            if pairs * N > 2 ** 31 - 1:
                continue
            K = item_slices(P, g, N, most)
            room = pairs * N // K * 5 // 4 + keys + 1
            steps = set(range(1, N + 1, max(1, N // 400))) | {N}
            for n in steps:
                assert pairs * n / item_slices(P, g, n, most) + keys <= room, (P, N, n)
