"""The gppsum = 1 tiles at the edges of their ring, tiles and rules: unoccupied
bands of no stage (8 bands), of one, of as many and more than ring slots, with
and without a remainder; occupied bands at k-step edges; rows and columns at the
tile edges; frequencies of one and more passes; column maps that use every tile
(two tiles per workgroup) and none; more row blocks than the kernel arguments
list; elements at the branch thresholds and outside the range of the short
terms, which keep the reference's operations.

Tolerance: the repository's FP64 bar, 1e-12 of the largest result: a result sums
at most 2e6 terms, each good to a few units of 2^-53 of its size."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RTOL = 1e-12


def _rel(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300))


def _check(fk, fko, p):
    ref_ach, ref_asx, _ = fko.gpp_gppsum(p)
    ach, asx, _ = fk.gpp_problem(p, semantics=fk.FK_GPP_GPPSUM)
    if np.any(ref_ach):
        assert _rel(ach, ref_ach) <= RTOL
    else:
        assert not np.any(ach)
    if p.nv and np.any(ref_asx):
        assert _rel(asx, ref_asx) <= RTOL
    else:
        assert not np.any(asx)


@pytest.mark.parametrize("nb,nv,C,G,nw", [
    (1, 0, 1, 1, 1), (3, 3, 40, 9, 2), (7, 0, 31, 31, 3), (8, 0, 32, 32, 3), (9, 1, 33, 33, 4), (16, 0, 64, 63, 3),
    (21, 4, 65, 64, 1), (22, 5, 96, 65, 7), (29, 5, 97, 97, 3), (33, 8, 600, 130, 3), (34, 9, 1100, 129, 6),
    (18, 1, 2000, 70, 3),
])
def test_ring_edges(fk, fko, nb, nv, C, G, nw):
    _check(fk, fko, fko.gpp_random(nb, nv, C, G, nw=nw, seed=nb + C, wtilde_re=(0.5, 5.5)))


@pytest.mark.parametrize("kind", ["last", "first", "mixed"])
def test_column_maps(fk, fko, kind):
    """Every column at the last G-vector (all tiles used), at the first (one tile
    column), and both in one row block."""
    p = fko.gpp_random(12, 3, 300, 150, seed=4, wtilde_re=(0.5, 5.5))
    inv = np.asarray(p.inv_igp_index)
    inv[:] = {"last": p.ncouls - 1, "first": 0, "mixed": 0}[kind]
    if kind == "mixed":
        inv[70] = p.ncouls - 1
    _check(fk, fko, p)


def test_many_row_blocks(fk, fko):
    p = fko.gpp_random(5, 1, 40, 32900, seed=6, wtilde_re=(0.5, 5.5))
    p.inv_igp_index[:] = np.arange(p.ngpown) % p.ncouls
    _check(fk, fko, p)


@pytest.mark.parametrize("nw", [1, 3, 4])
def test_threshold_and_general_elements(fk, fko, nw):
    """|wtilde| from 1e-8 to 1e5, and |wx - wtilde| at gamma to the last bits."""
    p = fko.gpp_random(19, 4, 321, 90, nw=nw, seed=3, wtilde_re=(0.5, 5.5))
    rng = np.random.default_rng(5)
    w = p.wtilde.reshape(-1)
    k = rng.choice(w.size, 600, replace=False)
    w[k[:200]] = 10.0 ** rng.uniform(-2.5, -2, 200) * np.exp(1j * rng.uniform(0, 6, 200))
    w[k[200:400]] = 10.0 ** rng.uniform(2, 5, 200) * np.exp(1j * rng.uniform(0, 6, 200))
    s = rng.choice([-1.0, 1.0], 200)
    w[k[400:]] = p.wx[rng.integers(0, nw, 200)] + s * np.sqrt(p.limittwo) * (1 + 2.0 ** -52 * rng.integers(-3, 4, 200))
    _check(fk, fko, p)


def test_stop_positions(fk, fko):
    """The occupied loop's break at the edges of the scan's steps (256 threads of
    4 ig), at to1 to the last bits, and two breaks in one column."""
    p = fko.gpp_random(6, 3, 2300, 12, seed=8, wtilde_re=(0.5, 5.5))
    p.inv_igp_index[:] = p.ncouls - 1 - np.arange(p.ngpown)
    for m, at in enumerate([0, 1, 255, 256, 511, 767, 768, 1023, 1024, 2047, 2048]):
        p.I_eps[m, at] = p.to1 * (1 - 1e-12) / p.wtilde[m, at] ** 2
    p.I_eps[2, 100] = p.to1 * (1 + 1e-12) / p.wtilde[2, 100] ** 2
    p.I_eps[5, 2000] = 0.0
    _check(fk, fko, p)
