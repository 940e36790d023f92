"""The forms of the gppsum = 1 kernel: 3 or 4 frequencies per pass, one or two tiles
per workgroup, two of them side by side on eight waves or one after the other.

Which form a problem takes follows from its frequencies (3 per pass unless 4 take
fewer passes), its tiles of 64 x 32 against the partials that the workspace holds,
and its workgroups against the GPU's 256 CUs.  Tolerance: the FP64 bar, 1e-12 of the
largest result."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300))


@pytest.mark.parametrize("nw", [3, 4, 5, 7, 16])
@pytest.mark.parametrize("nb,nv,C,G,last", [
    (20, 3, 65, 9, True),        # a second tile that ends past the last column
    (11, 0, 97, 64, True),       # an odd number of tiles per row block
    (19, 5, 300, 130, True),     # two tiles side by side, several row blocks
    (9, 2, 2100, 700, False),    # one tile per workgroup
    (5, 1, 1700, 1300, True),    # two tiles one after the other, more than 256 workgroups
])
def test_forms(fk, fko, nb, nv, C, G, last, nw):
    p = fko.gpp_random(nb, nv, C, G, nw=nw, seed=nb + nw, wtilde_re=(0.5, 5.5))
    if last:                     # every tile of every row block in use
        p.inv_igp_index[:] = C - 1 - np.arange(G) % 3
    ref_ach, ref_asx, _ = fko.gpp_gppsum(p)
    ach, asx, _ = fk.gpp_problem(p, semantics=fk.FK_GPP_GPPSUM)
    assert _rel(ach, ref_ach) <= 1e-12
    assert _rel(asx, ref_asx) <= 1e-12 if nv else not np.any(asx)


def test_four_frequencies_take_one_pass(fk):
    """A fourth frequency costs a small call a few per cent (39% as a second pass over
    the elements), at most a fifth."""
    import torch
    nb, C, G = 84, 405, 16
    g = torch.Generator(device="cuda:0")
    g.manual_seed(1)

    def uniform(shape, lo=-0.5, hi=0.5, im=0.5):
        t = torch.empty(shape, dtype=torch.complex128, device="cuda:0")
        v = torch.view_as_real(t)
        v[..., 0].uniform_(lo, hi, generator=g)
        v[..., 1].uniform_(-im, im, generator=g)
        return t

    aqsm, aqsn, ieps, wt = uniform((nb, C)), uniform((nb, C)), uniform((G, C)), uniform((G, C), 0.5, 5.5, 0.01)
    vcoul = torch.empty(C, dtype=torch.float64, device="cuda:0").uniform_(0.1, 10.0, generator=g)
    inv = (np.arange(G) * C // G).astype(np.int32)
    ind = np.arange(C + 1, dtype=np.int32)
    ind[C] = C - 1
    ms = {}
    for nw in (3, 4):
        wx = np.array([3.0, 4.0, 5.0, 6.0][:nw])
        ws = torch.empty(fk.gpp_workspace_size(nb, 0, C, G, nw) + 4 * G + 256, dtype=torch.uint8, device="cuda:0")
        ms[nw] = min(fk.gpp_kernel(nb, 0, C, G, wx, aqsm, aqsn, ieps, wt, vcoul, inv, ind, semantics=fk.FK_GPP_GPPSUM,
                                   workspace=ws, time_kernel=True)[2] for _ in range(40))
    assert ms[4] <= 1.2 * ms[3]
