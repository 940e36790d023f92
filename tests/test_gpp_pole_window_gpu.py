"""The short pole terms over the whole range of |wtilde| and with the mask off.

They take an element where one comparison decides both branches: |wtilde| in a
window set by the limits, which has no lower end when every |wx| is well above
sqrt(limittwo) and no upper end when every |wx| is well below it, and any wtilde of
0.  Results at frequencies on both sides of those rules, with |wtilde| from 0 to
1e6, wx = +-wtilde to the last bits and thresholds to the last bits, against the
oracle: 1e-12 of the largest result (FP64), 1e-8 (mixed), the repository's bars.

The last test holds the speed: a call with the mask off, or with zeros and large
values among its wtilde, takes about the time of a plain one (1.0 to 1.1 of it; 1.4
to 2 where these elements are evaluated one at a time), so at most 1.3 times."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

AXES = {
    "plain": [3.0, 4.0, 5.0],
    "low": [0.3, 1.3, 2.3],                       # below sqrt(limittwo): tiny wtilde may be near the pole
    "edge": [0.5026, -0.5026, 0.75],              # just above 1.005 sqrt(limittwo)
    "zero": [0.0, 1e-6, 7.0, -0.2, 0.5],
    "signs": [-3.0, -0.8, 0.8, 2.0, 5.0, 6.5, 9.0],
    "high": [200.0, 247.0, 260.0, 3000.0],
}


def _problem(fko, axis, seed, nv=5):
    wx = np.array(AXES[axis])
    p = fko.gpp_random(37, nv, 321, 90, nw=len(wx), seed=seed, wtilde_re=(0.5, 5.5))
    p.wx = wx
    rng = np.random.default_rng(seed)
    w = p.wtilde.reshape(-1)
    k = rng.choice(w.size, 7000, replace=False).reshape(7, 1000)
    ph = lambda: np.exp(1j * rng.uniform(0, 6.28, 1000))                                 # noqa: E731
    w[k[0]] = 0.0
    w[k[1]] = 10.0 ** rng.uniform(-9, -2, 1000) * ph()
    w[k[2]] = 10.0 ** rng.uniform(1, 6, 1000) * ph()
    pick = wx[rng.integers(0, len(wx), (4, 1000))]
    ulp = 2.0 ** -52 * rng.integers(-3, 4, 1000)
    w[k[3]] = pick[0] * (1 + 1e-3 * rng.normal(size=1000)) + 1e-3j
    w[k[4]] = -pick[1] * (1 + 1e-2 * rng.normal(size=1000)) + 0.1j
    w[k[5]] = pick[2] + rng.choice([-0.5, 0.5], 1000) * (1 + ulp)                        # |u|^2 at limittwo
    # |wtilde|^2 at to1 |u|^2: u = wx - wtilde real, wtilde = wx / (1001 or -999)
    w[k[6]] = pick[3] / rng.choice([1001.0, -999.0], 1000) * (1 + ulp)
    return p


@pytest.mark.parametrize("axis", AXES)
@pytest.mark.parametrize("config", [0, 2])
@pytest.mark.parametrize("mask", [True, False])
def test_fp64(fk, fko, axis, config, mask):
    p = _problem(fko, axis, 1)
    if axis == "zero":
        p.wtilde[np.abs(p.wtilde) < 1e-6] = 1e-3         # |wx - wtilde| = 0 and 1/wx^2 of 0: not numbers
        if not mask:
            p.wtilde[np.abs(p.wtilde[..., None] - p.wx).min(axis=-1) < 1e-12] = 1e-3
    for iw in np.nonzero(p.wx == 0.0)[0]:
        # the static SX factor divides by wx^2: keep |wx - wtilde|^2 <= limittwo there
        far = np.abs(p.wtilde) > 0.45
        p.wtilde[far] = 0.2 + 0.01j
    ref_ach, ref_asx, _ = fko.gpp(p, nthreads=0, mask_on=mask)
    ach, asx, _ = fk.gpp_problem(p, config=config, mask=mask)
    assert np.max(np.abs(ach - ref_ach)) <= 1e-12 * np.max(np.abs(ref_ach))
    assert np.max(np.abs(asx - ref_asx)) <= 1e-12 * np.max(np.abs(ref_asx))


@pytest.mark.parametrize("axis", ["plain", "low", "signs", "high"])
@pytest.mark.parametrize("mask", [True, False])
def test_mixed(fk, fko, axis, mask):
    p = _problem(fko, axis, 2)
    h = {k: np.ascontiguousarray(getattr(p, k).astype(np.complex64)) for k in ("aqsm", "aqsn", "I_eps", "wtilde")}
    for k, v in h.items():
        setattr(p, k, v.astype(np.complex128))
    if not mask:      # keep |wx - wtilde| off 0, where the unmasked factor has its pole
        near = np.abs(p.wtilde[..., None] - p.wx).min(axis=-1) < 1e-2
        p.wtilde[near] = 2.7
        h["wtilde"] = p.wtilde.astype(np.complex64)
        p.wtilde = h["wtilde"].astype(np.complex128)
    out = fk.gpp_kernel(p.nb, p.nv, p.ncouls, p.ngpown, p.wx, h["aqsm"], h["aqsn"], h["I_eps"], h["wtilde"], p.vcoul,
                        p.inv_igp_index, p.indinv, precision="mixed", mask=mask)
    ref_ach, ref_asx, _ = fko.gpp(p, nthreads=0, mask_on=mask)
    assert np.max(np.abs(out[0] - ref_ach)) <= 1e-8 * np.max(np.abs(ref_ach))
    assert np.max(np.abs(out[1] - ref_asx)) <= 1e-8 * np.max(np.abs(ref_asx))


def _time(f):
    """Milliseconds per call, the smallest of 7 groups of 10."""
    import torch
    best = 1e30
    for _ in range(8):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(10):
            f()
        e1.record()
        torch.cuda.synchronize()
        best = min(best, e0.elapsed_time(e1) / 10)
    return best


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("nb,nv,C,G,nw", [(128, 2, 8192, 409, 3), (100, 11, 6007, 601, 7)])
def test_speed_with_the_mask_off_and_outside_the_window(fk, precision, batch, nb, nv, C, G, nw):
    import torch
    g = torch.Generator(device="cuda:0")
    g.manual_seed(3)
    dt = torch.complex64 if precision == "mixed" else torch.complex128

    def uniform(shape, lo=-0.5, hi=0.5, im=0.5):
        t = torch.empty(shape, dtype=dt, device="cuda:0")
        v = torch.view_as_real(t)
        v[..., 0].uniform_(lo, hi, generator=g)
        v[..., 1].uniform_(-im, im, generator=g)
        return t

    aqsm, aqsn, ieps, wt = uniform((nb, C)), uniform((nb, C)), uniform((G, C)), uniform((G, C), 0.5, 5.5, 0.01)
    outside = wt.clone()
    r = torch.rand((G, C), generator=g, device="cuda:0")
    outside[r < 0.05] = 0.0
    outside[r > 0.95] = 1000.0
    vcoul = torch.empty(C, dtype=torch.float64, device="cuda:0").uniform_(0.1, 10.0, generator=g)
    wx = np.array([3.0 + iw for iw in range(nw)])
    inv = (np.arange(G, dtype=np.int64) * C // G).astype(np.int32)
    ind = np.arange(C + 1, dtype=np.int32)
    ind[C] = C - 1
    stream = torch.cuda.current_stream()
    ws = torch.empty(fk.gpp_workspace_size(nb, nv, C, G, nw, precision=precision), dtype=torch.uint8, device="cuda:0")

    def call(w, mask):
        if batch:
            torch.cuda.synchronize()
            b = fk.GppBatch([dict(nb=nb, nv=nv, ncouls=C, ngpown=G, wx=wx, aqsm=aqsm, aqsn=aqsn, I_eps=ieps, wtilde=w,
                                  vcoul=vcoul, inv_igp_index=inv, indinv=ind)] * 2, precision=precision,
                            config=2 if precision == "fp64" else 0, mask=mask)
            return lambda: b.run(stream=stream)
        return lambda: fk.gpp_kernel(nb, nv, C, G, wx, aqsm, aqsn, ieps, w, vcoul, inv, ind, precision=precision,
                                     mask=mask, stream=stream, workspace=ws)

    plain = _time(call(wt, True))
    assert _time(call(wt, False)) <= 1.3 * plain
    assert _time(call(outside, True)) <= 1.3 * plain
