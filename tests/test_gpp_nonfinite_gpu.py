"""Infinities and NaNs in the band arrays reach the outputs that the reference
lets them reach, and no others (FP64, canonical and gppsum = 1)."""
import warnings

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(fk, p, form):
    if form == "batch":
        import torch
        d = dict(nb=p.nb, nv=p.nv, ncouls=p.ncouls, ngpown=p.ngpown, wx=p.wx, inv_igp_index=p.inv_igp_index,
                 indinv=p.indinv, **{k: torch.from_numpy(np.ascontiguousarray(getattr(p, k))).to("cuda:0")
                                     for k in ("aqsm", "aqsn", "I_eps", "wtilde", "vcoul")})
        torch.cuda.synchronize()
        ach, asx, _ = fk.GppBatch([d], precision="fp64", config=2).run()
        torch.cuda.synchronize()
        return ach[0].cpu().numpy(), asx[0].cpu().numpy()
    if form == "gppsum":
        return fk.gpp_problem(p, semantics=fk.FK_GPP_GPPSUM)[:2]
    return fk.gpp_problem(p, config=0 if form == "small" else 2)[:2]


def _oracle(fko, p, form):
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        return (fko.gpp_gppsum(p) if form == "gppsum" else fko.gpp(p, nthreads=0))[:2]


@pytest.mark.parametrize("form", ["small", "large", "batch", "gppsum"])
@pytest.mark.parametrize("nv", [1, 2, 3, 5, 6])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_an_unoccupied_band_leaves_asxtemp_alone(fk, fko, form, nv, bad):
    """asxtemp sums over the occupied bands: an infinity in any other (the first
    unoccupied ones share a k-step of 4 bands with the last occupied) has no
    part in it.  Tolerance: the FP64 bar."""
    p = fko.gpp_random(20, nv, 300, 70, seed=3, wtilde_re=(0.5, 5.5))
    clean = _oracle(fko, p, form)[1]
    for band in range(nv, nv + 4):
        p.aqsn[band, 17 + band] = bad
        if form == "gppsum":
            p.aqsm[band, 19 + band] = bad
    ach, asx = _run(fk, p, form)
    assert not np.all(np.isfinite(ach.real))
    assert np.max(np.abs(asx - clean)) <= 1e-12 * np.max(np.abs(clean))


@pytest.mark.parametrize("form,occupied", [("small", True), ("large", True), ("batch", True), ("gppsum", True),
                                           ("small", False), ("large", False), ("batch", False)])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_a_band_element_near_the_pole(fk, fko, form, occupied, bad):
    """One element of aqsn is not finite and every factor that it meets is near the
    pole at frequency 0, where sch = 0: an occupied band adds 0 times it (a NaN), an
    unoccupied one is left out.  (The sequential program adds 0 times it in the
    gppsum = 1 form, which the library has always left out: not compared.)"""
    p = fko.gpp_random(20, 3, 300, 70, seed=3, wtilde_re=(0.5, 2.0))
    ig = 33
    p.aqsn[1 if occupied else 9, ig] = bad
    p.wtilde[:, ig] = p.wx[0] + 0.1
    ref, got = _oracle(fko, p, form), _run(fk, p, form)
    for g, r in zip(got, ref):
        assert np.array_equal(np.isfinite(g), np.isfinite(r)), (g, r)
        ok = np.isfinite(r)
        assert np.all(np.abs(g[ok] - r[ok]) <= 1e-12 * np.max(np.abs(r[ok]), initial=0.0))
    assert not np.all(np.isfinite(ref[0]))
