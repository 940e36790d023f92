"""achtemp and asxtemp with and without achstemp, bit for bit, at the frequency
counts where the two calls take passes of different width over the frequencies
(3 take one pass in both), with |wtilde| inside and outside the range of the short
pole terms."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["fp64", "mixed"])
@pytest.mark.parametrize("config", [0, 2])
@pytest.mark.parametrize("nw", [4, 5, 6, 7, 11, 16])
def test_achstemp_leaves_the_other_outputs_alone(fk, fko, kind, config, nw):
    p = fko.gpp_random(41, 5, 700, 150, nw=nw, seed=nw, wtilde_re=(0.5, 5.5))
    rng = np.random.default_rng(nw)
    w = p.wtilde.reshape(-1)
    k = rng.choice(w.size, 2000, replace=False)
    w[k[:700]] = 0.0
    w[k[700:1400]] = 10.0 ** rng.uniform(2.5, 4, 700)
    w[k[1400:]] = 10.0 ** rng.uniform(-5, -3, 600)
    if kind == "mixed":
        if config:
            pytest.skip("the tile configurations of complex64 inputs have tests of their own")
        for name in ("aqsm", "aqsn", "I_eps", "wtilde"):
            setattr(p, name, getattr(p, name).astype(np.complex64))
    plain = fk.gpp_problem(p, precision=kind, config=config)
    out = fk.gpp_problem(p, precision=kind, config=config, achstemp=True)
    assert out[0].tobytes() == plain[0].tobytes() and out[1].tobytes() == plain[1].tobytes()
