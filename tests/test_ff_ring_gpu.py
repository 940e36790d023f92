"""The FF contraction's FP64 tiles at the edges of their LDS ring and tiles:
ig ranges of one stage (8 ig) and of fewer, as many and more stages than ring
slots, with and without a remainder; bands and columns at the tile edges; the
ig range split over workgroups.

Tolerance: a result sums G * C products of three FP64 factors; each product
of the 3M form carries at most a few units of 2^-53 of |a||x||c|, so with
|result| of the order of sqrt(G C) |a||x||c| and G C <= 2e5 the error stays
below 4 * 2^-53 * sqrt(G C) ~ 2e-13 of the largest result; 1e-12 is the
repository's FP64 bar."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.max(np.abs(a - b)) / np.max(np.abs(b)))


@pytest.mark.parametrize("config", [0, 1, 2])
@pytest.mark.parametrize("nb,C,G,nf", [
    (1, 1, 1, 1), (3, 7, 5, 2), (16, 8, 8, 1), (17, 9, 9, 2), (31, 16, 15, 1), (32, 17, 17, 1),
    (33, 24, 24, 3), (63, 25, 23, 1), (64, 40, 33, 1), (65, 63, 63, 2), (64, 64, 64, 1), (65, 129, 65, 1),
    (127, 200, 127, 1), (129, 385, 130, 1), (10, 3000, 40, 1), (70, 2563, 65, 1),
])
def test_ring_edges(fk, fko, config, nb, C, G, nf):
    p = fko.ff_random(nb, C, G, nf, seed=nb + C)
    rt, rv, ra = fko.ff(p, achs_freq=0)
    t, v, a, _ = fk.ff_problem(p, achs_freq=0, config=config)
    assert _rel(t, rt) <= 1e-12 and _rel(v, rv) <= 1e-12
    assert abs(complex(a[0]) - ra) <= 1e-12 * max(abs(ra), float(np.max(np.abs(rv))))
