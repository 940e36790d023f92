"""Mixed batches whose problems fall into several frequency classes of the pole
kernel (up to 4, 8, 12 and 16 frequencies): all in one launch up to 2048 blocks, one
launch per class past them, with the mask on and off.  Each problem's results are
those of its own call to the mixed bar, 1e-8 of the largest, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mask", [True, False])
@pytest.mark.parametrize("nws,C,G", [
    ((3, 7, 11, 16), 300, 40), ((16, 1), 257, 5), ((5, 1, 12), 513, 9), ((4, 4), 300, 40), ((2, 9, 14, 6), 2100, 700),
])
def test_classes(fk, fko, nws, C, G, mask):
    import torch
    ps, dev = [], []
    for k, nw in enumerate(nws):
        p = fko.gpp_random(17 + 5 * k, 2 + k, C - 31 * k, G + k, nw=nw, seed=k, wtilde_re=(0.5, 2.5))
        p.wx = 3.0 + np.arange(nw)
        for name in ("aqsm", "aqsn", "I_eps", "wtilde"):
            setattr(p, name, getattr(p, name).astype(np.complex64).astype(np.complex128))
        ps.append(p)
        dev.append(dict(nb=p.nb, nv=p.nv, ncouls=p.ncouls, ngpown=p.ngpown, wx=p.wx, inv_igp_index=p.inv_igp_index,
                        indinv=p.indinv, vcoul=torch.from_numpy(np.ascontiguousarray(p.vcoul)).to("cuda:0"),
                        **{n: torch.from_numpy(np.ascontiguousarray(getattr(p, n).astype(np.complex64))).to("cuda:0")
                           for n in ("aqsm", "aqsn", "I_eps", "wtilde")}))
    torch.cuda.synchronize()
    batch = fk.GppBatch(dev, precision="mixed", mask=mask)
    for _ in range(2):
        ach, asx, _ = batch.run()
        torch.cuda.synchronize()
        for p, a, x in zip(ps, ach, asx):
            ref_ach, ref_asx, _ = fko.gpp(p, nthreads=0, mask_on=mask)
            assert np.max(np.abs(a.cpu().numpy() - ref_ach)) <= 1e-8 * np.max(np.abs(ref_ach))
            assert np.max(np.abs(x.cpu().numpy() - ref_asx)) <= 1e-8 * np.max(np.abs(ref_asx))
