"""Inputs aligned to 8 bytes only, in every kernel that fills its LDS ring by
direct loads or through registers: the gppsum = 1 tiles (aqsn and aqsm), the 64 x 64
and 32 x 32 tiles of single calls and the batch's.  Only the way into LDS differs, so
the results are those of aligned inputs bit for bit."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dev(a, off8):
    """A device copy of an array, 8 bytes past a 16-byte line or on one."""
    import torch
    f = np.ascontiguousarray(a).view(np.float64).reshape(-1)
    k = 1 if off8 else 0
    v = torch.empty(f.size + 2, dtype=torch.float64, device="cuda:0")[k:k + f.size]
    v.copy_(torch.from_numpy(f))
    assert v.data_ptr() % 16 == 8 * k
    return v


class _Case:
    """One problem on the device with some of its arrays off by 8 bytes."""

    def __init__(self, fk, p, off, semantics=0):
        self.d = {k: _dev(getattr(p, k), k in off) for k in ("aqsm", "aqsn", "I_eps", "wtilde", "vcoul")}
        self.h = [np.ascontiguousarray(x, t) for x, t in ((p.wx, np.float64), (p.inv_igp_index, np.int32),
                                                          (p.indinv, np.int32))]
        ptr = {k: v.data_ptr() for k, v in self.d.items()}
        self.s = fk.GppProblem(p.nb, p.nv, p.ncouls, p.ngpown, len(p.wx), self.h[0].ctypes.data, ptr["aqsm"], ptr["aqsn"],
                               ptr["I_eps"], ptr["wtilde"], ptr["vcoul"], self.h[1].ctypes.data, self.h[2].ctypes.data,
                               p.to1, p.limittwo, p.limitone, p.occ, semantics)


def _options(fk, config):
    o = fk.default_options()
    o.memory, o.precision, o.config = fk.FK_MEM_DEVICE, fk.FK_PREC_FP64, config
    return o


def _single(fk, c, config):
    import torch
    out = torch.zeros(2, c.s.nfreq, dtype=torch.complex128, device="cuda:0")
    torch.cuda.synchronize()
    assert fk.lib.gpp_kernel(ctypes.byref(c.s), ctypes.byref(_options(fk, config)), out[0].data_ptr(),
                             out[1].data_ptr(), None) == 0
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("config", [0, 2])
@pytest.mark.parametrize("nb,nv,C,G", [(45, 3, 300, 70), (24, 16, 129, 33), (9, 0, 65, 64)])
def test_gpp(fk, fko, config, nb, nv, C, G):
    p = fko.gpp_random(nb, nv, C, G, seed=2, wtilde_re=(0.5, 5.5))
    ref = _single(fk, _Case(fk, p, ()), config)
    for off in (("aqsn",), ("aqsm", "aqsn", "I_eps", "wtilde", "vcoul")):
        assert _single(fk, _Case(fk, p, off), config).tobytes() == ref.tobytes(), off


@pytest.mark.parametrize("off", [("aqsn",), ("aqsm",), ("aqsm", "aqsn", "I_eps", "wtilde", "vcoul")])
@pytest.mark.parametrize("nb,nv,C,G", [(45, 3, 300, 70), (24, 9, 129, 33), (30, 0, 65, 64)])
def test_gppsum(fk, fko, off, nb, nv, C, G):
    p = fko.gpp_random(nb, nv, C, G, seed=2, wtilde_re=(0.5, 5.5))
    ref = _single(fk, _Case(fk, p, (), fk.FK_GPP_GPPSUM), 0)
    assert _single(fk, _Case(fk, p, off, fk.FK_GPP_GPPSUM), 0).tobytes() == ref.tobytes()


def _batch(fk, cases):
    import torch
    n = len(cases)
    arr = (ctypes.POINTER(fk.GppProblem) * n)(*[ctypes.pointer(c.s) for c in cases])
    out = [torch.zeros(2, c.s.nfreq, dtype=torch.complex128, device="cuda:0") for c in cases]
    pa = (ctypes.c_void_p * n)(*[t[0].data_ptr() for t in out])
    px = (ctypes.c_void_p * n)(*[t[1].data_ptr() for t in out])
    torch.cuda.synchronize()
    assert fk.lib.gpp_kernel_batched(n, arr, ctypes.byref(_options(fk, 2)), pa, px) == 0
    torch.cuda.synchronize()
    return [t.cpu().numpy() for t in out]


def test_gpp_batch(fk, fko):
    """Aligned and misaligned problems side by side in one batch."""
    ps = [fko.gpp_random(nb, nv, C, G, nw=nw, seed=nb, wtilde_re=(0.5, 5.5))
          for nb, nv, C, G, nw in [(45, 3, 300, 70, 3), (24, 16, 129, 33, 7), (9, 0, 65, 64, 11)]]
    ref = _batch(fk, [_Case(fk, p, ()) for p in ps])
    got = _batch(fk, [_Case(fk, p, off) for p, off in zip(ps, (("aqsn",), (), ("aqsm", "aqsn", "I_eps", "wtilde")))])
    for a, b in zip(got, ref):
        assert a.tobytes() == b.tobytes()
