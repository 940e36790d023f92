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


def _off8(a):
    """A device copy of a complex array that starts 8 bytes past a 16-byte line."""
    import torch
    f = np.ascontiguousarray(a).view(np.float64).reshape(-1)
    v = torch.empty(f.size + 2, dtype=torch.float64, device="cuda:0")[1:1 + f.size]
    v.copy_(torch.from_numpy(f))
    assert v.data_ptr() % 16 == 8
    return v


def _device_options(fk):
    o = fk.default_options()
    o.memory, o.precision, o.config = fk.FK_MEM_DEVICE, fk.FK_PREC_FP64, 0
    return o


def test_inputs_aligned_to_8_bytes(fk, fko):
    import ctypes

    import torch
    p = fko.ff_random(37, 150, 70, 3, seed=4)
    m = torch.from_numpy(np.ascontiguousarray(p.aqsm)).to("cuda:0")
    v = torch.from_numpy(np.ascontiguousarray(p.vcoul)).to("cuda:0")
    n, x = _off8(p.aqsn), _off8(p.I_eps)
    inv, ind = np.ascontiguousarray(p.inv_igp_index, np.int32), np.ascontiguousarray(p.indinv, np.int32)
    t = torch.zeros(2, 37, 3, dtype=torch.complex128, device="cuda:0")
    prob = fk.FfProblem(37, 150, 70, 3, m.data_ptr(), n.data_ptr(), x.data_ptr(), v.data_ptr(), inv.ctypes.data,
                        ind.ctypes.data, 0)
    torch.cuda.synchronize()
    assert fk.lib.ff_kernel(ctypes.byref(prob), ctypes.byref(_device_options(fk)), t[0].data_ptr(), t[1].data_ptr(),
                            None) == 0
    torch.cuda.synchronize()
    rt, rv, _ = fko.ff(p, achs_freq=0)
    assert _rel(t[0].cpu().numpy(), rt) <= 1e-12 and _rel(t[1].cpu().numpy(), rv) <= 1e-12
