"""Performance cases of the GPP / FF library: what programs ask of it.

A case is a dict of plain values.  `kind` names the entry point:

  gpp       gpp_kernel on device arrays, FP64 or mixed (complex64), with the
            optional outputs acht_n1_loc and achstemp when `extra` is set
  gppsum    gpp_kernel with the gppsum = 1 semantics (FP64 only)
  gpp_batch a GppBatch over `count` uneven problems, FP64 or mixed
  ff        ff_kernel, FP64 or mixed (split BF16)
  ff_full   ff_kernel_full with the program's own frequency axes
  ff_batch  an FfBatch over `count` uneven problems

Sizes are number_bands (nb), nvband (nv), ncouls (C), ngpown (G), frequencies
(nw; FF: nf grid frequencies, ne evaluation frequencies).  They come from the
benchmark's and the tests' workloads and the ranges around them.

`prepare` makes the inputs on the device from the seed, with the caller-owned
workspace (or the batch handle) that a program keeps from call to call;
`run` is one call; `exact` is the same result from plain torch in FP64.
"""
import importlib.util
import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEV = "cuda:0"


def _load():
    """The package directory has a hyphen in its name, so it is imported by path."""
    if "fortkernels_amd" in sys.modules:
        return sys.modules["fortkernels_amd"]
    pkg = os.path.join(ROOT, "fortkernels-_amd")
    spec = importlib.util.spec_from_file_location("fortkernels_amd", os.path.join(pkg, "__init__.py"),
                                                  submodule_search_locations=[pkg])
    mod = importlib.util.module_from_spec(spec)
    sys.modules["fortkernels_amd"] = mod
    spec.loader.exec_module(mod)
    return mod


# --------------------------------------------------------------------------
# the cases
# --------------------------------------------------------------------------
def listed():
    return [
        # a call where launches and latency are all there is: a unit-test or
        # few-band model problem
        dict(name="gpp_small", kind="gpp", precision="fp64", nb=16, nv=2, C=300, G=60, nw=3, extra=False),
        # the reference program's own command line, gppKer 128 2 8192 20
        dict(name="gpp_program", kind="gpp", precision="fp64", nb=128, nv=2, C=8192, G=409, nw=3, extra=False),
        # the headline workload, gppKer 512 2 32768 20
        dict(name="gpp_headline", kind="gpp", precision="fp64", nb=512, nv=2, C=32768, G=1638, nw=3, extra=False),
        # every output of a real run (per-band sums and the static-CH
        # remainder), at sizes that are multiples of nothing
        dict(name="gpp_all_outputs", kind="gpp", precision="fp64", nb=333, nv=11, C=10007, G=1001, nw=7, extra=True),
        # complex64 inputs on a mid-sized ragged problem with more frequencies
        dict(name="gpp_mixed_ragged", kind="gpp", precision="mixed", nb=100, nv=7, C=6151, G=307, nw=5, extra=False),
        # complex64 inputs, the headline workload
        dict(name="gpp_mixed_headline", kind="gpp", precision="mixed", nb=512, nv=2, C=32768, G=1638, nw=3, extra=False),
        # the sequential program's gppsum = 1 loop
        dict(name="gppsum", kind="gppsum", precision="fp64", nb=256, nv=4, C=16384, G=819, nw=3),
        # a run over q-points: uneven GPP problems as one batch, both precisions
        dict(name="gpp_batch", kind="gpp_batch", precision="fp64", count=12, shapes=3, cmax=20000),
        dict(name="gpp_batch_mixed", kind="gpp_batch", precision="mixed", count=12, shapes=4, cmax=20000),
        # the FF contraction of one dielectric matrix, FP64
        dict(name="ff_headline", kind="ff", precision="fp64", nb=256, C=4096, G=4096, nf=32),
        # the whole FF evaluation of the Fortran program on the split-BF16 contraction
        dict(name="ff_full_mixed", kind="ff_full", precision="mixed", nb=256, nv=8, C=4096, G=4096, nf=32, ne=10),
        # many small FF contractions as one batch
        dict(name="ff_batch", kind="ff_batch", precision="fp64", count=8, shapes=5, cmax=2048),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed kinds, its sizes spread over their ranges."""
    kind = rng.choice(["gpp", "gpp", "gpp", "gppsum", "gpp_batch", "ff", "ff_full", "ff_batch"])
    precision = rng.choice(["fp64", "mixed"])
    if kind in ("gpp", "gppsum"):
        top = 512 * 32768 * 1638 if kind == "gpp" else 256 * 16384 * 819
        while True:
            nb, C = _log_int(rng, 16, 800), _log_int(rng, 256, 32768)
            G = max(1, C // rng.randint(5, 40))
            if nb * C * G <= top:
                break
        nv = rng.randint(0, min(16, nb))
        nw = rng.randint(1, 11)
        if kind == "gppsum":
            return dict(kind=kind, precision="fp64", nb=nb, nv=nv, C=C, G=G, nw=nw)
        extra = nw >= 3 and rng.random() < 0.25
        return dict(kind=kind, precision=precision, nb=nb, nv=nv, C=C, G=G, nw=nw, extra=extra)
    if kind == "gpp_batch":
        return dict(kind=kind, precision=precision, count=rng.randint(2, 12), shapes=rng.randint(10, 10 ** 6),
                    cmax=_log_int(rng, 4500, 16000))
    if kind == "ff_batch":
        return dict(kind=kind, precision=precision, count=rng.randint(2, 8), shapes=rng.randint(10, 10 ** 6),
                    cmax=_log_int(rng, 600, 2000))
    while True:
        nb, C, nf = _log_int(rng, 8, 400), _log_int(rng, 200, 4096), rng.randint(2, 32)
        G = max(1, C // rng.choice([1, 1, 2, 3, 5]))
        if nb * C * G * nf <= 256 * 4096 * 4096 * 32 and G * C * nf <= 4096 * 4096 * 32:
            break
    if kind == "ff":
        return dict(kind=kind, precision=precision, nb=nb, C=C, G=G, nf=nf)
    return dict(kind=kind, precision=precision, nb=nb, nv=rng.randint(0, min(16, nb)), C=C, G=G, nf=nf,
                ne=rng.randint(1, 12))


def _gpp_batch_shapes(case):
    """number_bands U{128..1024}, ncouls U{4096..cmax}/64*64, ngpown ncouls/20,
    nvband U{2..16}, frequencies U{3..11}."""
    rng = random.Random(case["shapes"])
    out = []
    for _ in range(case["count"]):
        C = rng.randint(4096, case["cmax"]) // 64 * 64
        out.append((rng.randint(128, 1024), rng.randint(2, 16), C, C // 20, rng.randint(3, 11)))
    return out


def _ff_batch_shapes(case):
    """number_bands U{32..256}, ncouls U{512..cmax}/64*64, ngpown ncouls/2, nFreq U{8..32}."""
    rng = random.Random(case["shapes"])
    out = []
    for _ in range(case["count"]):
        C = rng.randint(512, case["cmax"]) // 64 * 64
        out.append((rng.randint(32, 256), C, C // 2, rng.randint(8, 32)))
    return out


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
def _uniform(gen, shape, dtype, re=(-0.5, 0.5), im=(-0.5, 0.5)):
    t = torch.empty(shape, dtype=dtype, device=DEV)
    v = torch.view_as_real(t)
    if re == im:
        v.uniform_(re[0], re[1], generator=gen)
    else:
        v[..., 0].uniform_(re[0], re[1], generator=gen)
        v[..., 1].uniform_(im[0], im[1], generator=gen)
    return t


def _maps(C, G):
    """inv_igp_index and indinv as the reference program sets them."""
    inv = (np.arange(G, dtype=np.int64) * C // G).astype(np.int32)
    ind = np.arange(C + 1, dtype=np.int32)
    ind[C] = C - 1
    return inv, ind


def _gpp_inputs(gen, nb, C, G, nw, precision):
    """Plane-wave matrix elements, the static inverse dielectric matrix and
    plasmon energies from below to above the evaluation axis, so that all
    three branches of the pole factor are taken."""
    dt = torch.complex128 if precision == "fp64" else torch.complex64
    inv, ind = _maps(C, G)
    return dict(aqsm=_uniform(gen, (nb, C), dt), aqsn=_uniform(gen, (nb, C), dt), I_eps=_uniform(gen, (G, C), dt),
                wtilde=_uniform(gen, (G, C), dt, (0.5, 5.5), (-0.01, 0.01)),
                vcoul=torch.empty(C, dtype=torch.float64, device=DEV).uniform_(0.1, 10.0, generator=gen),
                wx=np.array([10.0 - 6.0 + 1.0 * ((iw + 1) - 2) for iw in range(nw)]), inv_igp_index=inv, indinv=ind)


def _ff_inputs(gen, nb, C, G, nf, arrays=("I_eps",)):
    inv, ind = _maps(C, G)
    t = dict(aqsm=_uniform(gen, (nb, C), torch.complex128), aqsn=_uniform(gen, (nb, C), torch.complex128))
    for name in arrays:
        t[name] = _uniform(gen, (nf, G, C), torch.complex128)
    t["vcoul"] = torch.empty(C, dtype=torch.float64, device=DEV).uniform_(0.1, 10.0, generator=gen)
    return dict(t, inv_igp_index=inv, indinv=ind)


def _ff_axes(nb, nf):
    """Band energies, grid, weights and broadening of the Fortran program."""
    ekq = -10.0 + np.arange(nb, dtype=np.float64)
    grid = 2.0 * np.arange(nf, dtype=np.float64)
    pref = np.empty(nf)
    pref[:-1] = (grid[1:] - grid[:-1]) / 3.14
    pref[-1] = pref[-2]
    pref[0] *= 0.5
    pref[-1] *= 0.5
    return ekq, grid, pref, np.full(nf, 0.1j)


def _inputs(case, seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed))
    kind = case["kind"]
    if kind in ("gpp", "gppsum"):
        return _gpp_inputs(gen, case["nb"], case["C"], case["G"], case["nw"], case["precision"])
    if kind == "gpp_batch":
        return [dict(_gpp_inputs(gen, nb, C, G, nw, case["precision"]), nb=nb, nv=nv, ncouls=C, ngpown=G)
                for nb, nv, C, G, nw in _gpp_batch_shapes(case)]
    if kind == "ff":
        return _ff_inputs(gen, case["nb"], case["C"], case["G"], case["nf"])
    if kind == "ff_batch":
        return [dict(_ff_inputs(gen, nb, C, G, nf), nb=nb, ncouls=C, ngpown=G, nfreq=nf)
                for nb, C, G, nf in _ff_batch_shapes(case)]
    t = _ff_inputs(gen, case["nb"], case["C"], case["G"], case["nf"], ("I_epsR", "I_epsA"))
    t["ekq"], t["grid"], t["pref"], t["brd"] = _ff_axes(case["nb"], case["nf"])
    return t


def prepare(case, seed):
    fk = _load()
    t = _inputs(case, seed)
    c, kind = case, case["kind"]
    if kind == "gpp_batch":
        torch.cuda.synchronize()   # the batch reads its inputs on its own stream
        return dict(case=c, batch=fk.GppBatch(t, precision=c["precision"], config=0))
    if kind == "ff_batch":
        torch.cuda.synchronize()
        return dict(case=c, batch=fk.FfBatch(t, precision=c["precision"], config=0))
    if kind == "ff":
        n = fk.ff_workspace_size(c["nb"], c["C"], c["G"], c["nf"], precision=c["precision"])
    elif kind == "ff_full":
        n = fk.ff_full_workspace_size(c["nb"], c["nv"], c["C"], c["G"], c["nf"], c["ne"], t["ekq"], t["grid"],
                                      precision=c["precision"])
    else:
        # the gppsum = 1 form needs a stop per column beside the canonical workspace
        n = fk.gpp_workspace_size(c["nb"], c["nv"], c["C"], c["G"], c["nw"], precision=c["precision"],
                                  acht_n1=c.get("extra", False))
        n += 4 * c["G"] + 256 if kind == "gppsum" else 0
    return dict(case=c, t=t, ws=torch.empty(n, dtype=torch.uint8, device=DEV))


def run(state):
    fk = _load()
    c = state["case"]
    kind = c["kind"]
    stream = torch.cuda.current_stream()
    if kind == "gpp_batch":
        ach, asx, _ = state["batch"].run(stream=stream)
        return dict(achtemp=ach, asxtemp=asx)
    if kind == "ff_batch":
        schDt, schDv, achs, _ = state["batch"].run(stream=stream)
        return dict(schDt=schDt, schDv=schDv, achs=achs)
    t = state["t"]
    if kind == "gpp":
        out = fk.gpp_kernel(c["nb"], c["nv"], c["C"], c["G"], t["wx"], t["aqsm"], t["aqsn"], t["I_eps"], t["wtilde"],
                            t["vcoul"], t["inv_igp_index"], t["indinv"], precision=c["precision"], stream=stream,
                            workspace=state["ws"], acht_n1=c["extra"], achstemp=c["extra"])
        if c["extra"]:
            return dict(achtemp=out[0], asxtemp=out[1], acht_n1_loc=out[3], achstemp=out[4])
        return dict(achtemp=out[0], asxtemp=out[1])
    if kind == "gppsum":
        out = fk.gpp_kernel(c["nb"], c["nv"], c["C"], c["G"], t["wx"], t["aqsm"], t["aqsn"], t["I_eps"], t["wtilde"],
                            t["vcoul"], t["inv_igp_index"], t["indinv"], semantics=fk.FK_GPP_GPPSUM, stream=stream,
                            workspace=state["ws"])
        return dict(achtemp=out[0], asxtemp=out[1])
    if kind == "ff":
        out = fk.ff_kernel(c["nb"], c["C"], c["G"], c["nf"], t["aqsm"], t["aqsn"], t["I_eps"], t["vcoul"],
                           t["inv_igp_index"], t["indinv"], precision=c["precision"], stream=stream,
                           workspace=state["ws"])
        return dict(schDt=out[0], schDv=out[1], achs=out[2])
    out = fk.ff_kernel_full(c["nb"], c["nv"], c["C"], c["G"], c["nf"], c["ne"], t["aqsm"], t["aqsn"], t["I_epsR"],
                            t["I_epsA"], t["vcoul"], t["inv_igp_index"], t["indinv"], t["ekq"], t["grid"], t["pref"],
                            t["brd"], precision=c["precision"], stream=stream, workspace=state["ws"])
    out.pop("kernel_ms")
    return out


# --------------------------------------------------------------------------
# work that the path cannot do without
# --------------------------------------------------------------------------
def _gpp_work(nb, nv, C, G, nw, elem, extra=False):
    """Inputs once; a complex multiply-add as 8 flops, the band contraction
    once (the pole factor does not depend on the band)."""
    gc = float(G) * C
    flops = 8.0 * nb * gc + gc * (8.0 * nv + 9.0 + 42.0 * nw)
    if extra:
        flops += 8.0 * nb * gc + 8.0 * gc
    return elem * (float(nb) * C + float(nb) * G + 2.0 * gc) + 8.0 * C, flops


def _ff_work(nb, C, G, nf):
    return 16.0 * (float(nf) * G * C + float(nb) * C + float(nb) * G + 2.0 * nb * nf) + 8.0 * G, \
        8.0 * float(nb) * G * C * nf


def work(case):
    kind = case["kind"]
    elem = 8.0 if case["precision"] == "mixed" and kind.startswith("gpp") else 16.0
    if kind == "gpp":
        b, f = _gpp_work(case["nb"], case["nv"], case["C"], case["G"], case["nw"], elem, case["extra"])
    elif kind == "gppsum":
        # two band contractions over the half plane ig <= igp
        nb, nv, C, G, nw = (case[k] for k in ("nb", "nv", "C", "G", "nw"))
        half = 0.5 * G * C
        b = 16.0 * (2.0 * nb * C + 2.0 * half)
        f = 16.0 * nb * half + half * nw * 42.0
    elif kind == "gpp_batch":
        w = [_gpp_work(*s, elem) for s in _gpp_batch_shapes(case)]
        b, f = sum(x[0] for x in w), sum(x[1] for x in w)
    elif kind == "ff":
        b, f = _ff_work(case["nb"], case["C"], case["G"], case["nf"])
    elif kind == "ff_batch":
        w = [_ff_work(*s) for s in _ff_batch_shapes(case)]
        b, f = sum(x[0] for x in w), sum(x[1] for x in w)
    else:
        b, f = _ff_work(case["nb"], case["C"], case["G"], case["nf"])
        nbA, nfA = _ff_box(case)
        b += 16.0 * float(nfA) * case["G"] * case["C"]
        f += 8.0 * float(nbA) * case["G"] * case["C"] * nfA
    return {"bytes": b, "flops": f}


def _ff_box(case):
    """Bands and frequencies of I_epsA that the SX and delta terms read."""
    ekq, grid, _, _ = _ff_axes(case["nb"], case["nf"])
    wx = 0.0 - ekq[:, None] + 0.5 * np.arange(case["ne"])[None, :]
    read = (wx >= 0.0) | (np.arange(case["nb"])[:, None] < case["nv"])
    if not read.any():
        return 0, 0
    f = _interval(grid, np.abs(wx))[read]
    bands = np.nonzero(read.any(axis=1))[0]
    return int(bands[-1] - bands[0] + 1), int(f.max() + 1 - f.min() + 1)


# --------------------------------------------------------------------------
# the same results in plain torch, FP64
# --------------------------------------------------------------------------
def _columns(t):
    return torch.from_numpy(t["indinv"].astype(np.int64)[t["inv_igp_index"]]).to(DEV)


def _exact_gpp(t, nb, nv, C, G, extra=False, to1=1e-6, limittwo=0.25, limitone=2.5e5):
    w = {k: t[k].to(torch.complex128) for k in ("aqsm", "aqsn")}
    igp = _columns(t)
    coef = 0.5 * t["vcoul"][igp][None, :] * w["aqsm"][:, igp].conj()          # [nb][G]
    wx = [float(x) for x in t["wx"]]
    ach = torch.zeros(len(wx), dtype=torch.complex128, device=DEV)
    asx, achs = torch.zeros_like(ach), torch.zeros(1, dtype=torch.complex128, device=DEV)
    n1 = torch.zeros(nb, dtype=torch.complex128, device=DEV)
    rows = max(1, min(G, (1 << 22) // C))
    for r0 in range(0, G, rows):
        c = coef[:, r0:r0 + rows].t().contiguous()
        B = c @ w["aqsn"]
        Bo = c[:, :nv].contiguous() @ w["aqsn"][:nv] if nv else None
        ie, wt = t["I_eps"][r0:r0 + rows].to(torch.complex128), t["wtilde"][r0:r0 + rows].to(torch.complex128)
        achs -= (B * ie).sum()
        Om = wt * wt * ie
        for iw, x in enumerate(wx):
            wdiff = x - wt
            d2 = wdiff.real * wdiff.real + wdiff.imag * wdiff.imag
            delw = wt * wdiff.conj() * (1.0 / d2)
            e2 = delw.real * delw.real + delw.imag * delw.imag
            m = (d2 > limittwo) & (e2 < limitone)
            X = torch.where(m, delw * ie, torch.zeros_like(ie))
            ach[iw] += (B * X).sum()
            if extra and iw == 2:
                n1 += ((w["aqsn"] @ X.t().contiguous()) * c.t()).sum(dim=1)
            if nv:
                z = delw + 0.5
                near = -ie * delw * z.conj() / (4.0 * (z.real * z.real + z.imag * z.imag))
                S = torch.where(m, Om / (x * x), torch.where(e2 > to1, near, torch.zeros_like(ie)))
                asx[iw] += 2.0 * (Bo * S).sum()
    out = dict(achtemp=ach, asxtemp=asx)
    return dict(out, acht_n1_loc=n1, achstemp=achs) if extra else out


def _exact_gppsum(t, nb, nv, C, G, to1=1e-6, limittwo=0.25, limitone=2.5e5):
    igp = _columns(t)
    aqsm, aqsn = t["aqsm"], t["aqsn"]
    coef = 0.5 * t["vcoul"][igp][None, :] * aqsm[:, igp].conj()
    wx = [float(x) for x in t["wx"]]
    ach = torch.zeros(len(wx), dtype=torch.complex128, device=DEV)
    asx = torch.zeros_like(ach)
    ig = torch.arange(C, device=DEV)[None, :]
    rows = max(1, min(G, (1 << 22) // C))
    for r0 in range(0, G, rows):
        g = igp[r0:r0 + rows][:, None]
        c = coef[:, r0:r0 + rows].t().contiguous()
        cu, co = c[:, nv:].contiguous(), c[:, :nv].contiguous()
        Bu, Bp = cu @ aqsn[nv:], cu @ aqsm[nv:]
        Bo, Bpo = co @ aqsn[:nv], co @ aqsm[:nv]
        ie, wt = t["I_eps"][r0:r0 + rows], t["wtilde"][r0:r0 + rows]
        zero = torch.zeros_like(ie)
        Om = wt * wt * ie
        # the occupied loop stops at the first ig < igp with |wtilde^2 I_eps| < to1
        small = (Om.abs() < to1) & (ig < g)
        stop = torch.where(small, ig, g).amin(dim=1, keepdim=True)
        occ = ig < stop
        diag = (ig == g) & (g > 0) & (g % 512 == 0)
        both = (ig < g - 1) & (ig % 512 != 511)
        mirror = ig != g - 1
        for iw, x in enumerate(wx):
            wdiff = x - wt
            d2 = wdiff.real * wdiff.real + wdiff.imag * wdiff.imag
            delw = wt / wdiff
            keep = (d2 < limittwo) | (delw.abs() ** 2 > limitone)
            sch = delw * ie
            term = Bu * sch + torch.where(both, (Bp * sch).conj(), zero)
            ach[iw] += torch.where(keep & (both | diag), term, zero).sum()
            if nv:
                dl = wdiff * (0.5 / wt)
                near = (wdiff.abs() < math.sqrt(limittwo)) | (dl.abs() ** 2 < to1)
                sch = torch.where(near, zero, wt * ie / wdiff)
                ssx = torch.where(near, torch.where(wt.abs() > to1, -Om / (4.0 * wt * wt * (1.0 + dl)), zero),
                                  Om / (x * x - wt * wt))
                for out, f, s in ((ach, sch, 1.0), (asx, ssx, 2.0)):
                    term = Bo * f + torch.where(mirror, (Bpo * f).conj(), zero)
                    out[iw] += s * torch.where(occ, term, zero).sum()
    return dict(achtemp=ach, asxtemp=asx)


def _exact_ff(t, X, nb, C, G, nf):
    """schDt, schDv [nb][nf] of one dielectric matrix."""
    igp = _columns(t)
    cf, v = t["aqsm"][:, igp].conj(), t["vcoul"][igp]
    at = t["aqsn"].t().contiguous()
    schDt = torch.empty(nb, nf, dtype=torch.complex128, device=DEV)
    schDv = torch.empty_like(schDt)
    for f in range(nf):
        p = (X[f] @ at).t() * cf
        schDt[:, f] = p.sum(dim=1)
        schDv[:, f] = (p * v).sum(dim=1)
    return schDt, schDv


def _interval(grid, w):
    f = np.searchsorted(grid, w, side="right") - 1
    return np.where((f < 0) | (f > len(grid) - 2), len(grid) - 2, f)


def _exact_ff_full(t, case):
    nb, nv, C, G, nf, ne = (case[k] for k in ("nb", "nv", "C", "G", "nf", "ne"))
    S, VR = (x.cpu().numpy() for x in _exact_ff(t, t["I_epsR"], nb, C, G, nf))
    VA = _exact_ff(t, t["I_epsA"], nb, C, G, nf)[1].cpu().numpy()
    grid, pref, brd, zb = t["grid"], t["pref"], t["brd"], 0.5 / 3.14
    wx = 0.0 - t["ekq"][:, None] + np.arange(ne)[None, :] * 0.5
    wxp = -0.0 - t["ekq"][:, None] + np.arange(ne)[None, :] * 0.5
    occ = (np.arange(nb) < nv)[:, None]
    n1 = np.arange(nb)[:, None]
    f = _interval(grid, np.abs(wx))
    d = grid[f + 1] - grid[f]
    fa, fb = (grid[f + 1] - np.abs(wx)) / d, (np.abs(wx) - grid[f]) / d
    sxr, sxa = fa * VR[n1, f] + fb * VR[n1, f + 1], fa * VA[n1, f] + fb * VA[n1, f + 1]
    asx = np.where(occ, np.where(wx >= 0.0, sxr, sxa), 0.0)
    w, wp = wx[:, :, None], wxp[:, :, None]
    num = 1j * pref[:-1] * S[:, None, :-1]
    ach = -(num / (w - (grid - brd)[:-1])).sum(axis=2)
    corb = -(num / (w - np.where(occ[:, :, None], (-grid - brd)[:-1], (grid - brd)[:-1]))).sum(axis=2)
    zl, zr = grid[:-1], grid[1:]
    left, right = S[:, None, :-1], S[:, None, 1:]

    def ratio(a, b):
        with np.errstate(divide="ignore", invalid="ignore"):
            return np.log(np.clip(np.abs(a / b), 1e-4, 1e4))

    it = -ratio(w - zr, w - zl)
    s2 = -(1j * zb * 0.5 * (left + right) * it).sum(axis=2)
    lin, lin2 = right - left, (right - left) / (zr - zl)
    lin3 = np.where(occ[:, :, None], (left + lin2 * (wp - zl)) * ratio(w + zr, w + zl),
                    (left + lin2 * (w - zl)) * it) + lin
    cor = -(1j * zb * lin3).sum(axis=2)
    delta = -0.5 * (sxr - sxa)
    s2 = s2 + np.where(wx >= 0.0, delta, 0.0)
    cor = cor + np.where((wx >= 0.0) != occ, delta, 0.0)
    return dict(achsDtemp=np.array([-0.5 * VR[:, 0].sum()]), asxDtemp=asx.sum(axis=0), achDtemp=ach.sum(axis=0),
                achDtemp_cor=cor.sum(axis=0), achDtemp_corb=corb.sum(axis=0), ach2Dtemp=s2.sum(axis=0), schDt=S)


def exact(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    if kind == "gpp":
        return _exact_gpp(t, case["nb"], case["nv"], case["C"], case["G"], case["extra"])
    if kind == "gppsum":
        return _exact_gppsum(t, case["nb"], case["nv"], case["C"], case["G"])
    if kind == "gpp_batch":
        out = [_exact_gpp(p, p["nb"], nv, C, G) for p, (_, nv, C, G, _) in zip(t, _gpp_batch_shapes(case))]
        return dict(achtemp=[o["achtemp"] for o in out], asxtemp=[o["asxtemp"] for o in out])
    if kind == "ff":
        schDt, schDv = _exact_ff(t, t["I_eps"], case["nb"], case["C"], case["G"], case["nf"])
        return dict(schDt=schDt, schDv=schDv, achs=-0.5 * schDv[:, :1].sum(dim=0))
    if kind == "ff_batch":
        out = [_exact_ff(p, p["I_eps"], p["nb"], p["ncouls"], p["ngpown"], p["nfreq"]) for p in t]
        return dict(schDt=[o[0] for o in out], schDv=[o[1] for o in out],
                    achs=[-0.5 * o[1][:, :1].sum(dim=0) for o in out])
    return _exact_ff_full(t, case)
