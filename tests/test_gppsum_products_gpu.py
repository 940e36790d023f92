"""gppsum = 1 on nearly real inputs: the imaginary parts of the band sums keep
their own relative accuracy (four real products per complex one; the three of the
3M form would leave errors of the size of the real parts in them).

Every input has imaginary parts 1e-8 of its real ones, so the results have too.
Each term's imaginary part is a sum of products with one factor of 1e-8, good to a
few units of 2^-53 of itself, and a result sums at most 1e6 of them without
systematic cancellation: 1e-12 of the largest imaginary part is the repository's
FP64 bar.  3M misses it by four orders of magnitude (2e-8)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,nv,C,G,nw", [(40, 0, 300, 70, 3), (64, 6, 700, 96, 4), (9, 9, 200, 64, 2)])
def test_imaginary_parts_of_nearly_real_sums(fk, fko, nb, nv, C, G, nw):
    p = fko.gpp_random(nb, nv, C, G, nw=nw, seed=nb, wtilde_re=(0.5, 5.5))
    for k in ("aqsm", "aqsn", "I_eps", "wtilde"):
        a = getattr(p, k)
        setattr(p, k, np.ascontiguousarray(a.real + 1e-8j * a.imag))
    ref_ach, ref_asx, _ = fko.gpp_gppsum(p)
    ach, asx, _ = fk.gpp_problem(p, semantics=fk.FK_GPP_GPPSUM)
    for got, ref in ((ach, ref_ach), (asx, ref_asx)):
        for part in ("real", "imag"):
            g, r = getattr(got, part), getattr(ref, part)
            assert np.max(np.abs(g - r)) <= 1e-12 * np.max(np.abs(r)), part
