"""gppsum = 1: |wtilde| down to 1e-8, where the general terms and their own branch
for |wtilde| <= to1 are taken, and partials that stay inside the workspace."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RTOL = 1e-12      # the repository's FP64 bar, of the largest result


def _rel(a, b):
    return float(np.max(np.abs(a - b)) / np.max(np.abs(b)))


@pytest.mark.parametrize("nw", [1, 3, 4])
def test_tiny_wtilde(fk, fko, nw):
    """|wtilde| from 1e-8 to 1e-2 with I_eps so large that the occupied loop does not
    stop (|wtilde^2 I_eps| >= 10 to1), at frequencies from 1e-7 on, so that elements
    are near the pole and |wtilde| falls on both sides of to1 there."""
    p = fko.gpp_random(19, 4, 321, 90, nw=nw, seed=3, wtilde_re=(0.5, 5.5))
    p.wx = np.array([1e-7, 0.3, 3.0, 1e-3])[:nw]
    p.inv_igp_index[:] = p.ncouls - 1 - np.arange(p.ngpown)
    rng = np.random.default_rng(5)
    size = p.wtilde.size
    k = rng.choice(size, 4000, replace=False)
    w = 10.0 ** rng.uniform(-8, -2, 4000) * np.exp(1j * rng.uniform(0, 6.28, 4000))
    assert np.sum(np.abs(w) < p.to1) > 500
    p.wtilde.reshape(-1)[k] = w
    p.I_eps.reshape(-1)[k] = 10.0 * p.to1 / np.abs(w) ** 2 * np.exp(1j * rng.uniform(0, 6.28, 4000))
    small = np.abs(p.wtilde ** 2 * p.I_eps) < p.to1
    p.I_eps[small] = 1.0
    ref_ach, ref_asx, _ = fko.gpp_gppsum(p)
    ach, asx, _ = fk.gpp_problem(p, semantics=fk.FK_GPP_GPPSUM)
    assert _rel(ach, ref_ach) <= RTOL and _rel(asx, ref_asx) <= RTOL


@pytest.mark.parametrize("last", [False, True])
@pytest.mark.parametrize("nb,nv,C,G,nw", [(25, 0, 300, 40, 3), (37, 5, 700, 130, 2), (9, 3, 65, 64, 1), (30, 9, 3000, 300, 4)])
def test_workspace_bounds(fk, fko, last, nb, nv, C, G, nw):
    """The canonical workspace and a stop per column hold the form, with one and two
    tiles per workgroup, and nothing behind them is written."""
    import torch
    p = fko.gpp_random(nb, nv, C, G, nw=nw, seed=nb, wtilde_re=(0.5, 5.5))
    if last:
        p.inv_igp_index[:] = C - 1 - np.arange(G) % 5
    d = {k: torch.from_numpy(np.ascontiguousarray(getattr(p, k))).to("cuda:0")
         for k in ("aqsm", "aqsn", "I_eps", "wtilde", "vcoul")}
    n = fk.gpp_workspace_size(nb, nv, C, G, nw) + 4 * G + 256
    buf = torch.full((n + 4096,), 0x5A, dtype=torch.uint8, device="cuda:0")
    ach, asx, _ = fk.gpp_kernel(nb, nv, C, G, p.wx, d["aqsm"], d["aqsn"], d["I_eps"], d["wtilde"], d["vcoul"],
                                p.inv_igp_index, p.indinv, semantics=fk.FK_GPP_GPPSUM, workspace=buf[:n])
    torch.cuda.synchronize()
    assert bool((buf[n:] == 0x5A).all())
    ref_ach, ref_asx, _ = fko.gpp_gppsum(p)
    assert _rel(ach.cpu().numpy(), ref_ach) <= RTOL
    assert _rel(asx.cpu().numpy(), ref_asx) <= RTOL if nv else not np.any(asx.cpu().numpy())
