"""Both sides of the lines at which FP64 calls change between the 32 x 32 ring tiles,
the 64 x 64 ones and the tiles without a ring: 192, 256 and 512 tiles of 64 x 64, and
numbers of bands by frequencies.  Tolerance: the FP64 bar, 1e-12."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,C,G,nw,config", [
    (48, 64 * 385, 30, 1, 0), (49, 64 * 385, 30, 1, 0), (160, 64 * 193, 64, 1, 0), (161, 64 * 192, 60, 1, 0),
    (161, 64 * 193, 64, 1, 0), (161, 64 * 128 - 5, 128, 1, 0), (160, 64 * 86, 190, 1, 0), (161, 64 * 86, 190, 1, 0),
    (335, 64 * 97, 100, 2, 0), (336, 64 * 97, 100, 2, 0), (61, 1000, 70, 1, 2), (60, 1000, 70, 1, 2),
    (161, 64 * 513, 10, 1, 0), (161, 64 * 512, 10, 1, 0),
])
def test_both_sides(fk, fko, nb, C, G, nw, config):
    p = fko.gpp_random(nb, 3, C, G, nw=nw, seed=nb + C, wtilde_re=(0.5, 5.5))
    ref_ach, ref_asx, _ = fko.gpp(p, nthreads=0)
    ach, asx, _ = fk.gpp_problem(p, config=config)
    assert np.max(np.abs(ach - ref_ach)) <= 1e-12 * np.max(np.abs(ref_ach))
    assert np.max(np.abs(asx - ref_asx)) <= 1e-12 * np.max(np.abs(ref_asx))
    out = fk.gpp_problem(p, config=config, achstemp=True)
    assert out[0].tobytes() == ach.tobytes() and out[1].tobytes() == asx.tobytes()
