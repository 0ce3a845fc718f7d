"""Single-slice insertion by a thread per (pixel, corner): pads whose half row
is just below and just past the 32 pixels of a block, with the corners of the
slice, the x = 0 and x = P/2 planes and symmetry copies, against the oracle.
Bar: float32 sums of a few contributions per voxel, 1e-5."""
import numpy as np
import pytest

from eman2_amd.metrics import max_rel_err, weight_rel_err
from eman2_amd.transform import Transform, euler_eman_matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,sym,mode,corners", [(8, "c1", "gauss_2", 1), (22, "c4", "trilinear", 1), (60, "c1", "gauss_2", 0),
                                                (64, "d2", "gauss_2", 1), (66, "c1", "trilinear", 0), (128, "c2", "gauss_2", 1)])
def test_slices(oracle, P, sym, mode, corners):
    from eman2_amd import Reconstructors
    from eman2_amd.reconstructor import EMData
    print("corners P=%d %s %s %d" % (P, sym, mode, corners), flush=True)
    rng = np.random.default_rng(P)
    r = Reconstructors.get("fourier_hip", dict(size=(P, P, P), sym=sym, mode=mode, corners=bool(corners)))
    r.setup()
    v = oracle.Volume(P, sym, mode)
    mats = [euler_eman_matrix(0.0, 0.0, 0.0), euler_eman_matrix(0.0, 90.0, 0.0)]
    mats += [euler_eman_matrix(*(rng.random(3) * (360, 180, 360))) for _ in range(4)]
    for m in mats:
        m = m.astype(np.float32)
        s = rng.standard_normal((P, P + 2)).astype(np.float32)
        r.insert_slice(EMData(s, True, {"reconstruct_preproc": 1}), Transform(m), 0.75)
        v.insert(s, m, 0.75, corners=bool(corners))
    gd, gn = r.get_state()
    assert weight_rel_err(gn, v.norm) <= 1e-5
    assert max_rel_err(gd, v.data) <= 1e-5
