"""A caller's workspace at any address: the coefficient matrix and the operand
slices lie in it and move into LDS by direct 16-byte loads only where they are
16-byte aligned.  Results are those of an aligned workspace: bit for bit, since
only the way into LDS differs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _device(p, dtype):
    import torch
    d = {k: torch.from_numpy(np.ascontiguousarray(getattr(p, k).astype(dtype))).to("cuda:0")
         for k in ("aqsm", "aqsn", "I_eps", "wtilde")}
    return dict(d, vcoul=torch.from_numpy(np.ascontiguousarray(p.vcoul)).to("cuda:0"))


@pytest.mark.parametrize("kw", [dict(), dict(config=2), dict(config=2, achstemp=True), dict(sym=True), dict(mixed=True),
                                dict(acht_n1=True)])
@pytest.mark.parametrize("offset", [8])
def test_results_do_not_depend_on_the_address(fk, fko, kw, offset):
    import torch
    kw = dict(kw)
    mixed, sym = kw.pop("mixed", False), kw.pop("sym", False)
    p = fko.gpp_random(45, 3, 300, 70, seed=2, wtilde_re=(0.5, 5.5))
    d = _device(p, np.complex64 if mixed else np.complex128)
    prec = "mixed" if mixed else "fp64"
    n = fk.gpp_workspace_size(p.nb, p.nv, p.ncouls, p.ngpown, len(p.wx), precision=prec, config=kw.get("config", 0),
                              acht_n1=kw.get("acht_n1", False)) + (4 * p.ngpown + 256 if sym else 0)
    buf = torch.empty(n + 64, dtype=torch.uint8, device="cuda:0")
    if sym:
        kw["semantics"] = fk.FK_GPP_GPPSUM
    res = []
    for off in (0, offset):
        buf.fill_(0xA5)
        ws = buf[off:off + n]
        assert ws.data_ptr() % 16 == off
        out = fk.gpp_kernel(p.nb, p.nv, p.ncouls, p.ngpown, p.wx, d["aqsm"], d["aqsn"], d["I_eps"], d["wtilde"],
                            d["vcoul"], p.inv_igp_index, p.indinv, precision=prec, workspace=ws, **kw)
        torch.cuda.synchronize()
        assert bool((buf[:off] == 0xA5).all()) and bool((buf[off + n:] == 0xA5).all())
        res.append([x.cpu().numpy() for x in out if x is not None])
    for a, b in zip(*res):
        assert a.tobytes() == b.tobytes()
