"""Mixed GPP at the edges of its preparation and pole kernels: bands at the 16 of
a fragment, the 512 (aqsn) and 1024 (coefficients) that a thread keeps in
registers, and past them; rows at the 4 (2 past eight frequencies) of a pole
workgroup, columns at its 256; every class of frequency counts; elements that the
short pole terms leave to the general ones.

Tolerance: the mixed form's bar, 1e-8 of the largest result."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RTOL = 1e-8


def _rel(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300))


def _round64(p):
    for k in ("aqsm", "aqsn", "I_eps", "wtilde"):
        setattr(p, k, getattr(p, k).astype(np.complex64).astype(np.complex128))
    return p


def _check(fk, fko, p):
    h = {k: np.ascontiguousarray(getattr(p, k).astype(np.complex64)) for k in ("aqsm", "aqsn", "I_eps", "wtilde")}
    out = fk.gpp_kernel(p.nb, p.nv, p.ncouls, p.ngpown, p.wx, h["aqsm"], h["aqsn"], h["I_eps"], h["wtilde"], p.vcoul,
                        p.inv_igp_index, p.indinv, precision="mixed")
    ref_ach, ref_asx, _ = fko.gpp(p, nthreads=0)
    assert _rel(out[0], ref_ach) <= RTOL
    assert _rel(out[1], ref_asx) <= RTOL if p.nv else not np.any(out[1])


@pytest.mark.parametrize("nb,nv,C,G,nw", [
    (1, 1, 1, 1, 1), (15, 0, 255, 3, 2), (16, 2, 256, 4, 3), (17, 3, 257, 5, 4), (64, 0, 300, 6, 5), (65, 9, 511, 7, 8),
    (512, 2, 513, 9, 3), (513, 16, 300, 8, 9), (600, 5, 257, 3, 12), (1024, 3, 130, 2, 13), (1040, 17, 100, 1, 16),
    (33, 70, 1000, 11, 6),
])
def test_edges(fk, fko, nb, nv, C, G, nw):
    _check(fk, fko, _round64(fko.gpp_random(nb, min(nv, nb), C, G, nw=nw, seed=nb + C, wtilde_re=(0.5, 5.5))))


@pytest.mark.parametrize("nw", [3, 7, 11])
def test_general_elements(fk, fko, nw):
    p = fko.gpp_random(37, 6, 321, 90, nw=nw, seed=3, wtilde_re=(0.5, 5.5))
    rng = np.random.default_rng(5)
    w = p.wtilde.reshape(-1)
    k = rng.choice(w.size, 600, replace=False)
    w[k[:300]] = 10.0 ** rng.uniform(-6, -2, 300) * np.exp(1j * rng.uniform(0, 6, 300))
    w[k[300:]] = 10.0 ** rng.uniform(2, 5, 300) * np.exp(1j * rng.uniform(0, 6, 300))
    _check(fk, fko, _round64(p))
