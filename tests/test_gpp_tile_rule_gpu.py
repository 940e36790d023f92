"""Both sides of the lines at which FP64 calls change between the 32 x 32 ring tiles,
the 64 x 64 ones and the tiles without a ring: 192, 256 and 512 tiles of 64 x 64, and
numbers of bands by frequencies.  Tolerance: the FP64 bar, 1e-12."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,C,G,nw,config", [
    (48, 64 * 385, 30, 1, 0), (49, 64 * 385, 30, 1, 0), (160, 64 * 193, 64, 1, 0), (161, 64 * 192, 60, 1, 0),
    (161, 64 * 193, 64, 1, 0), (161, 64 * 128 - 5, 128, 1, 0), (160, 64 * 86, 190, 1, 0), (161, 64 * 86, 190, 1, 0),
    (335, 64 * 97, 100, 2, 0), (336, 64 * 97, 100, 2, 0), (61, 1000, 70, 1, 2), (60, 1000, 70, 1, 2),
    (161, 64 * 513, 10, 1, 0), (161, 64 * 512, 10, 1, 0),
])
def test_both_sides(fk, fko, nb, C, G, nw, config):
    p = fko.gpp_random(nb, 3, C, G, nw=nw, seed=nb + C, wtilde_re=(0.5, 5.5))
    ref_ach, ref_asx, _ = fko.gpp(p, nthreads=0)
    ach, asx, _ = fk.gpp_problem(p, config=config)
    assert np.max(np.abs(ach - ref_ach)) <= 1e-12 * np.max(np.abs(ref_ach))
    assert np.max(np.abs(asx - ref_asx)) <= 1e-12 * np.max(np.abs(ref_asx))
    out = fk.gpp_problem(p, config=config, achstemp=True)
    assert out[0].tobytes() == ach.tobytes() and out[1].tobytes() == asx.tobytes()


@pytest.mark.parametrize("config", [0, 2])
@pytest.mark.parametrize("nb,nv,C,G,nw", [(40, 17, 300, 70, 3), (40, 24, 300, 70, 3), (40, 25, 300, 70, 3), (24, 24, 129, 65, 8),
                                          (60, 23, 2561, 1000, 2)])
def test_occupied_bands(fk, fko, config, nb, nv, C, G, nw):
    """Up to 24 occupied bands on the ring, more without it."""
    p = fko.gpp_random(nb, nv, C, G, nw=nw, seed=nb + nv, wtilde_re=(0.5, 5.5))
    ref_ach, ref_asx, _ = fko.gpp(p, nthreads=0)
    ach, asx, _ = fk.gpp_problem(p, config=config)
    assert np.max(np.abs(ach - ref_ach)) <= 1e-12 * np.max(np.abs(ref_ach))
    assert np.max(np.abs(asx - ref_asx)) <= 1e-12 * np.max(np.abs(ref_asx))


@pytest.mark.parametrize("shapes", [
    [(336, 3, 1000, 64, 2), (400, 0, 1500, 130, 1)],                     # all idle on the ring: none of it
    [(335, 3, 1000, 64, 2), (400, 3, 1500, 130, 1), (60, 9, 700, 60, 7)],   # both kernels
    [(20, 24, 900, 100, 3), (30, 25, 900, 100, 3), (90, 60, 300, 70, 11)],
    [(20, 3, 900, 100, 3), (9, 1, 64, 64, 7), (30, 2, 5000, 500, 1)],    # more tiles than workgroups
    [(5, 3, 64, 64, 1)],                                                 # one tile
])
def test_batch_kernel_by_problem(fk, fko, shapes):
    """Each problem of a batch takes the kernel of its single call of the same
    configuration, and gives its bits."""
    import torch
    ps = [fko.gpp_random(max(nb, nv), nv, C, G, nw=nw, seed=nb, wtilde_re=(0.5, 5.5)) for nb, nv, C, G, nw in shapes]
    dev = [dict(nb=p.nb, nv=p.nv, ncouls=p.ncouls, ngpown=p.ngpown, wx=p.wx, inv_igp_index=p.inv_igp_index,
                indinv=p.indinv, **{k: torch.from_numpy(np.ascontiguousarray(getattr(p, k))).to("cuda:0")
                                    for k in ("aqsm", "aqsn", "I_eps", "wtilde", "vcoul")}) for p in ps]
    torch.cuda.synchronize()
    batch = fk.GppBatch(dev, precision="fp64", config=2)
    for _ in range(2):
        ach, asx, _ = batch.run()
        torch.cuda.synchronize()
        for p, a, x in zip(ps, ach, asx):
            ref_ach, ref_asx, _ = fko.gpp(p, nthreads=0)
            one_ach, one_asx, _ = fk.gpp_problem(p, config=2)
            assert a.cpu().numpy().tobytes() == one_ach.tobytes() and x.cpu().numpy().tobytes() == one_asx.tobytes()
            assert np.max(np.abs(one_ach - ref_ach)) <= 1e-12 * np.max(np.abs(ref_ach))
            if p.nv:
                assert np.max(np.abs(one_asx - ref_asx)) <= 1e-12 * np.max(np.abs(ref_asx))
