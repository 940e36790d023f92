"""The FP64 GPP tiles on the LDS ring (at most 16 occupied bands) at the edges
of their ring, tiles and rules: unoccupied bands of no stage (8 bands), of one,
of as many and more stages than ring slots, with and without a remainder;
occupied bands at k-step edges and across the rule's limit of 16; rows and
columns at the tile edges; one to four passes over the frequencies; elements
that the short pole terms leave to the general ones (|wtilde| tiny or large,
NaN-free limits, wx = wtilde); input arrays aligned to 8 bytes only.

Tolerance: the repository's FP64 bar, 1e-12 of the largest result.  A result
sums at most 3e6 terms, each good to a few units of 2^-53 of its size, so
with sums of the order of the root of their number times a term the error
stays below 1e-14 to 1e-13 of them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RTOL = 1e-12


def _rel(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300))


def _check(fk, fko, p, **kw):
    ref_ach, ref_asx, _ = fko.gpp(p, nthreads=0)
    ach, asx, _ = fk.gpp_problem(p, **kw)
    assert _rel(ach, ref_ach) <= RTOL
    if p.nv == 0:
        assert not np.any(asx)
    else:
        assert _rel(asx, ref_asx) <= RTOL


@pytest.mark.parametrize("config", [0, 2])     # 0: 32 x 32 tiles at these sizes, 2: 64 x 64
@pytest.mark.parametrize("nb,nv,C,G,nw", [
    (1, 0, 1, 1, 1), (1, 1, 1, 1, 2), (8, 0, 63, 7, 3), (9, 2, 31, 33, 3), (25, 3, 33, 32, 6), (9, 1, 64, 64, 3), (16, 0, 65, 63, 4), (17, 17, 64, 64, 3),
    (16, 16, 130, 65, 5), (20, 4, 200, 64, 3), (29, 5, 129, 128, 1), (32, 8, 127, 129, 2), (40, 15, 500, 66, 8),
    (33, 16, 257, 65, 9), (33, 17, 257, 65, 9), (24, 0, 640, 31, 16), (57, 9, 1000, 200, 11), (130, 12, 4099, 70, 3),
    (20, 2, 2561, 1000, 3),       # 640 tiles of 64 x 64 and more: the other side of the rule
])
def test_ring_edges(fk, fko, config, nb, nv, C, G, nw):
    _check(fk, fko, fko.gpp_random(nb, nv, C, G, nw=nw, seed=nb + C, wtilde_re=(0.5, 5.5)), config=config)


@pytest.mark.parametrize("config", [0, 2])
@pytest.mark.parametrize("nw", [2, 3, 7, 12])
def test_general_elements(fk, fko, config, nw):
    """|wtilde| from 1e-6 to 1e5 and wx = wtilde among ordinary elements."""
    p = fko.gpp_random(37, 6, 321, 90, nw=nw, seed=3, wtilde_re=(0.5, 5.5))
    rng = np.random.default_rng(5)
    w = p.wtilde.reshape(-1)
    k = rng.choice(w.size, 600, replace=False)
    w[k[:200]] = 10.0 ** rng.uniform(-6, -2, 200) * np.exp(1j * rng.uniform(0, 6, 200))
    w[k[200:400]] = 10.0 ** rng.uniform(2, 5, 200) * np.exp(1j * rng.uniform(0, 6, 200))
    w[k[400:500]] = p.wx[rng.integers(0, nw, 100)] + 1e-9 * rng.normal(size=100)
    w[k[500:]] = -p.wx[rng.integers(0, nw, 100)] + 1e-3j
    _check(fk, fko, p, config=config)


def test_band_edges_with_batch(fk, fko):
    """The batch kernel of the same tiles, problems of different edges."""
    import torch
    shapes = [(9, 1, 64, 64, 3), (16, 16, 130, 65, 5), (24, 0, 640, 31, 11), (57, 9, 1000, 200, 4)]
    ps = [fko.gpp_random(nb, nv, C, G, nw=nw, seed=nb, wtilde_re=(0.5, 5.5)) for nb, nv, C, G, nw in shapes]
    dev = [dict(nb=p.nb, nv=p.nv, ncouls=p.ncouls, ngpown=p.ngpown, wx=p.wx, inv_igp_index=p.inv_igp_index,
                indinv=p.indinv, **{k: torch.from_numpy(np.ascontiguousarray(getattr(p, k))).to("cuda:0")
                                    for k in ("aqsm", "aqsn", "I_eps", "wtilde", "vcoul")}) for p in ps]
    torch.cuda.synchronize()
    ach, asx, _ = fk.GppBatch(dev, precision="fp64", config=2).run()
    torch.cuda.synchronize()
    for p, a, x in zip(ps, ach, asx):
        ref_ach, ref_asx, _ = fko.gpp(p, nthreads=0)
        assert _rel(a.cpu().numpy(), ref_ach) <= RTOL
        assert _rel(x.cpu().numpy(), ref_asx) <= RTOL or p.nv == 0


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
    p = fko.gpp_random(45, 3, 300, 70, seed=2, wtilde_re=(0.5, 5.5))
    d = {k: torch.from_numpy(np.ascontiguousarray(getattr(p, k))).to("cuda:0") for k in ("aqsm", "I_eps", "wtilde", "vcoul")}
    n = _off8(p.aqsn)
    out = torch.zeros(2, 3, dtype=torch.complex128, device="cuda:0")
    wx, inv, ind = (np.ascontiguousarray(x, t) for x, t in ((p.wx, np.float64), (p.inv_igp_index, np.int32),
                                                            (p.indinv, np.int32)))
    prob = fk.GppProblem(p.nb, p.nv, p.ncouls, p.ngpown, 3, wx.ctypes.data, d["aqsm"].data_ptr(), n.data_ptr(),
                         d["I_eps"].data_ptr(), d["wtilde"].data_ptr(), d["vcoul"].data_ptr(), inv.ctypes.data,
                         ind.ctypes.data, p.to1, p.limittwo, p.limitone, p.occ, 0)
    torch.cuda.synchronize()
    assert fk.lib.gpp_kernel(ctypes.byref(prob), ctypes.byref(_device_options(fk)), out[0].data_ptr(),
                             out[1].data_ptr(), None) == 0
    torch.cuda.synchronize()
    ref_ach, ref_asx, _ = fko.gpp(p, nthreads=0)
    assert _rel(out[0].cpu().numpy(), ref_ach) <= RTOL and _rel(out[1].cpu().numpy(), ref_asx) <= RTOL


@pytest.mark.parametrize("nb,nv,C,G,nw", [(25, 0, 300, 40, 3), (37, 5, 700, 130, 2), (150, 9, 5000, 300, 4)])
def test_workspace_serves_gppsum(fk, fko, nb, nv, C, G, nw):
    """The canonical workspace and a stop per column hold the gppsum = 1 form."""
    import torch
    p = fko.gpp_random(nb, nv, C, G, nw=nw, seed=nb)
    d = {k: torch.from_numpy(np.ascontiguousarray(getattr(p, k))).to("cuda:0")
         for k in ("aqsm", "aqsn", "I_eps", "wtilde", "vcoul")}
    ws = torch.empty(fk.gpp_workspace_size(nb, nv, C, G, nw) + 4 * G + 256, dtype=torch.uint8, device="cuda:0")
    fk.gpp_kernel(nb, nv, C, G, p.wx, d["aqsm"], d["aqsn"], d["I_eps"], d["wtilde"], d["vcoul"], p.inv_igp_index,
                  p.indinv, semantics=fk.FK_GPP_GPPSUM, workspace=ws)
    torch.cuda.synchronize()
