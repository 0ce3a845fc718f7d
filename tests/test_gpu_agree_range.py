"""The batched agreement over the range of the particle weights: amp, cc and
low-resolution cc do not depend on a common factor of all weights, also where
the squares of weighted sums leave the float range (weights of 1e-21: squares
below the smallest normal; 1e19: above the largest).  Tolerance: the sums
scale by a power of two, so float32 rounding is the same away from the ends of
the range; 2e-6, some float32 roundings of the outputs, for the rest."""
import numpy as np
import pytest

from eman2_amd import synthetic as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,sym", [("gauss_2", "c1"), ("gauss_2", "d2"), ("trilinear", "c1")])
@pytest.mark.parametrize("sub", [False, True])
def test_common_weight_factor(mode, sym, sub):
    from eman2_amd import Reconstructors
    P, B, n = 24, 16, 480
    print("agreement range %s %s sub=%d" % (mode, sym, sub), flush=True)
    imgs, mats, _ = S.particles(S.phantom(8, 4.5, seed=1), n, B, seed=2, snr=1.0)
    w = np.linspace(0.5, 1.5, n).astype(np.float32)
    found = []
    for e in (0, -70, 63):
        we = np.ldexp(w, e).astype(np.float32)
        r = Reconstructors.get("fourier_hip", dict(size=(P, P, P), sym=sym, mode=mode))
        r.setup()
        r.insert_batch(imgs, mats, we)
        found.append(np.asarray(r.agreement_batch(imgs, mats, we, sub=sub))[:, :3])
    assert np.isfinite(found[0]).all()
    for f in found[1:]:
        assert np.isfinite(f).all()
        assert np.abs(f - found[0]).max() <= 2e-6 * np.abs(found[0]).max()
