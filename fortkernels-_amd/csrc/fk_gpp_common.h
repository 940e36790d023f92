// fk_gpp_common.h -- device code shared by the GPP kernels: the pole factor
// and SX factor of one (my_igp, ig) element (BGW-Kernels/gppKer.cpp:19-65,
// :394-411) and the reductions around them.
#pragma once

#include "fk_complex.h"

namespace fk {
namespace gpp {

constexpr int kMaxFreq = 16;
constexpr int kXcds = 8;       // MI355X: consecutive workgroups go to different XCDs

struct PoleConst {
    double wx[kMaxFreq];
    double iwx2[kMaxFreq];     // 1 / wx^2: conj(cden) / |cden|^2 of the mask branch, cden = wx^2 real (:41-44)
};

// Scalars of the per-element epilogue.
struct PoleParams {
    double limittwo, limitone, to1;
    double lo, hi;             // pole_terms takes an element with lo < |wtilde|^2 < hi
    int mask_on;
    int nw;
    PoleConst pc;
};

inline PoleParams make_pole_params(const double *wx, int nfreq, double limittwo, double limitone, double to1,
                                   bool mask_on)
{
    PoleParams pp;
    pp.limittwo = limittwo;
    pp.limitone = limitone;
    pp.to1 = to1;
    pp.mask_on = mask_on ? 1 : 0;
    pp.nw = nfreq;
    pp.lo = pp.hi = 0.0;
    if (limittwo > 0.0 && limitone > 0.0 && to1 == to1) {
        pp.lo = 1.01 * (to1 > 0.0 ? to1 : 0.0) * limittwo;
        pp.hi = 0.99 * limitone * limittwo;
        // |wtilde| so far from every frequency that the mask is on at each
        double near = INFINITY, far = 0.0;      // the smallest and largest |wx|
        for (int iw = 0; iw < nfreq; ++iw) {
            near = !(std::fabs(wx[iw]) >= near) ? std::fabs(wx[iw]) : near;
            far = !(std::fabs(wx[iw]) <= far) ? std::fabs(wx[iw]) : far;
        }
        const double pole = std::sqrt(1.01 * limittwo), below = near - pole;
        const double above = std::max(far + pole, far / (1.0 - std::sqrt(1.01 / limitone)));
        const double lo = pp.lo, hi = pp.hi;
        if (lo < hi && below > 0.0 && below * below > 1.01 * lo) pp.lo = -1.0;
        if (limitone > 1.02 && above * above < 0.99 * hi) pp.hi = 1e300;
    }
    for (int iw = 0; iw < kMaxFreq; ++iw) {
        const double w = iw < nfreq ? wx[iw] : 0.0;
        pp.pc.wx[iw] = w;
        pp.pc.iwx2[iw] = iw < nfreq ? 1.0 / (w * w) : 0.0;
    }
    return pp;
}

__device__ __forceinline__ double2 widen(double2 v) { return v; }
__device__ __forceinline__ double2 widen(float2 v) { return make_double2((double)v.x, (double)v.y); }

// 1/x from v_rcp_f64 and one step of third order.  Measured over 4M inputs
// spanning 2^-40 .. 2^40, v_rcp_f64 alone is within 4.2e8 units of 2^-53
// (about 2^-24 relative); with e = 1 - x r, r (1 + e + e^2) is off by e^3,
// below the last rounding, in three fused operations where two Newton steps
// (equal to the IEEE quotient) take four.
__device__ __forceinline__ double rcp_cubic(double x)
{
    const double r = __builtin_amdgcn_rcp(x);
    const double e = __builtin_fma(-x, r, 1.0);
    return __builtin_fma(r, __builtin_fma(e, e, e), r);
}

// delw = wtilde * conj(wdiff) * rden and |delw|^2 in the reference's FP64
// evaluation order (BGW-Kernels/gppKer.cpp:30-36, :396-402).  Contraction is
// off so, given the same rden, they round exactly as the reference's.
__device__ __forceinline__ void pole_delw(double2 wt, double wdr, double rden, double2 &delw, double &delwr)
{
#pragma clang fp contract(off)
    const double wdi = -wt.y;
    delw = make_double2((wt.x * wdr - wt.y * (-wdi)) * rden, (wt.x * (-wdi) + wt.y * wdr) * rden);
    delwr = delw.x * delw.x + delw.y * delw.y;
}

__device__ __forceinline__ double pole_wdiffr(double wdr, double wdi)
{
#pragma clang fp contract(off)
    return wdr * wdr + wdi * wdi;
}

// The sum over the wave in every lane: lanes l and l ^ 1 first, then l ^ 2, ...
__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Sums of 8 values over the wave through `buf`, 8 * 65 doubles of LDS of its own:
// lane q < 8 returns wave_sum(v[q]), the same bits.  Lane q + 8 h adds value q of
// lanes 8 h .. 8 h + 7, pairs first, then the parts meet: 8 writes, 8 reads and 10
// additions where 8 butterflies take 96 shuffles and 48 additions (13312 tiles
// of 12 values: 0.05 ms less).
__device__ __forceinline__ double wave_sums_lds(const double (&v)[8], int lane, double *buf)
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int q = 0; q < 8; ++q) buf[q * 65 + lane] = v[q];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const double *p = buf + (lane & 7) * 65 + (lane & ~7);
    double x = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
#pragma unroll
    for (int off = 8; off < 64; off <<= 1) x += __shfl_xor(x, off, 64);
    return x;
}

// One (my_igp, ig) element for the NWC frequencies w0 .. w0+NWC-1: adds
// B * D to sach[q] and Bo * ssx to sasx[q], where D = mask * delw * I_eps
// and ssx is the three-way SX factor (:37-57).  `ok` = a real, kept
// element; a frequency past nw repeats the last one and adds nothing.
// The SX factor of the mask branch (:41-44) is Omega2 / wx^2 (cden = wx^2
// is real); that of the near-pole branch (:49-52) is
// -I_eps delw conj(z) / (4 |z|^2), z = delw + 0.5 (Omega2 conj(cden) /
// |cden|^2 with cden = 4 wtilde^2 z and Omega2 = wtilde^2 I_eps loses its
// wtilde^2).
template <int NWC>
__device__ __forceinline__ void pole_element(const PoleParams &pp, int w0, bool ok, double2 wt, double2 ie,
                                             double2 B, double2 Bo, bool want_ssx, double2 (&sach)[NWC],
                                             double2 (&sasx)[NWC])
{
    const double tol1 = 1e-13 * pp.limitone, tol2 = 1e-13 * pp.to1;
    const double2 Om = cmul(cmul(wt, wt), ie);
#pragma unroll
    for (int q = 0; q < NWC; ++q) {
        const int iw = min(w0 + q, pp.nw - 1);
        const bool live = ok && (w0 + q < pp.nw);
        const double wdr = pp.pc.wx[iw] - wt.x;
        const double wdiffr = pole_wdiffr(wdr, -wt.y);
        double2 delw;
        double delwr;
        pole_delw(wt, wdr, rcp_cubic(wdiffr), delw, delwr);
        // points within 1e-13 of a branch threshold take the IEEE quotient,
        // so every branch decision is the reference's
        const bool near = fabs(delwr - pp.limitone) <= tol1 || fabs(delwr - pp.to1) <= tol2;
        if (__ballot(near)) {
            if (near) pole_delw(wt, wdr, 1.0 / wdiffr, delw, delwr);
        }
        const bool m = (wdiffr > pp.limittwo) && (delwr < pp.limitone);
        const double2 D = (m || !pp.mask_on) ? cmul(delw, ie) : make_double2(0.0, 0.0);
        const double2 t = cmul(B, D);
        if (live) sach[q] = cadd(sach[q], t);
        if (want_ssx) {
            double2 S = m ? make_double2(Om.x * pp.pc.iwx2[iw], Om.y * pp.pc.iwx2[iw]) : make_double2(0.0, 0.0);
            const bool need2 = !m && delwr > pp.to1;
            if (__ballot(need2)) {
                if (need2) {
                    const double2 z = make_double2(delw.x + 0.5, delw.y);
                    const double sc = -0.25 * rcp_cubic(z.x * z.x + z.y * z.y);
                    const double2 v = cmul(ie, cmul(delw, cconj(z)));
                    S = make_double2(sc * v.x, sc * v.y);
                }
            }
            const double2 u = cmul(Bo, S);
            if (live) sasx[q] = cadd(sasx[q], u);
        }
    }
}

__device__ __forceinline__ double2 cmul_fused(double2 a, double2 b)
{
#pragma clang fp contract(off)
    return make_double2(__builtin_fma(a.x, b.x, -(a.y * b.y)), __builtin_fma(a.x, b.y, a.y * b.x));
}

// One kept (my_igp, ig) element for the frequencies w0 .. w0+NWC-1 that
// exist: adds B D to sach[q] and Bo ssx to sasx[q], what pole_element adds, in
// less than half its operations (27 per frequency).  FP64 vector operations and
// FP64 MFMAs take turns on the same units here, so the epilogue adds to the
// MFMA time however well the two are interleaved, and its length is what it
// costs (512/2/32768/1638, 3 frequencies, an earlier form of the ring tiles: 3.00
// ms with pole_element's operations, 2.89 with these).
//
// With u = wx - wtilde and s = wx + wtilde,
//     D   = I_eps wtilde / u                     where the mask is on,
//     ssx = wtilde^2 I_eps / wx^2                where the mask is on,
//     ssx = -I_eps wtilde / (2 s)                near the pole:
// delw = wtilde / u, so delw + 1/2 = s / (2 u), and delw / (delw + 1/2) =
// 2 wtilde / s.  One reciprocal serves either branch, and the products with B
// and Bo are formed once per element.
//
// The branch is the sign of |u|^2 - limittwo alone (|u|^2 rounded as the
// reference rounds it): the mask's second test |delw|^2 < limitone follows
// from |u|^2 > limittwo when |wtilde|^2 < 0.99 limitone limittwo, and the
// near-pole test |delw|^2 > to1 from |u|^2 <= limittwo when |wtilde|^2 >
// 1.01 to1 limittwo (u = 0, where |delw|^2 is a NaN, adds nothing).  That is 5e-4 ..
// 249 with the default limits.  A larger |wtilde| keeps the mask on where |u| >=
// |wtilde| - |wx| alone is beyond both lines at every frequency, a smaller one
// where |wx| - |wtilde| is, so with every |wx| between 0.51 and 248 the range has
// no end; a wtilde of 0 (padding) adds nothing but zeros anywhere.  Other elements,
// NaNs and those whose Bo is not finite (0 Bo, added where the mask is off, is a
// NaN then) return false and are left to pole_element.
//
// The branches are taken under the execution mask: with selected factors instead
// (five more operations, no branch) every kernel that uses this is slower, by 7%
// at 3 frequencies and 20% at 7.
//
// Without occupied bands (Bo = 0) the sums of sasx are to be dropped: a 0 / wx^2
// at wx = 0 leaves a NaN there.
// MASK: pp.mask_on, a kernel of its own (tested here per element, it costs a tile's
// epilogue 10%).  wx, iwx2: the frequencies' tables (PoleConst).
template <int NWC, bool ALL, bool MASK, class Table>
__device__ __forceinline__ bool pole_terms(const PoleParams &pp, Table wx, Table iwx2, int w0, double2 wt, double2 ie, double2 B,
                                           double2 Bo, double2 (&sach)[NWC], double2 (&sasx)[NWC])
{
    // fused operations only where written, so every kernel rounds alike
#pragma clang fp contract(off)
    const double wy2 = wt.y * wt.y;
    const double wt2 = __builtin_fma(wt.x, wt.x, wy2);
    const double2 T = cmul_fused(ie, wt), P = cmul_fused(B, T);
    const double2 PQ = make_double2(P.y * wt.y, P.x * wt.y);
    const double2 BoOm = cmul_fused(Bo, cmul_fused(T, wt));
    const double2 R = cmul_fused(Bo, make_double2(-0.5 * T.x, -0.5 * T.y));
    if (!((wt2 > pp.lo || wt2 == 0.0) && wt2 < pp.hi && fabs(R.x + R.y) < __builtin_inf())) return false;
    const double2 RQ = make_double2(R.y * wt.y, R.x * wt.y);
#pragma unroll
    for (int q = 0; q < NWC; ++q) {
        if (!ALL && q > 0 && w0 + q >= pp.nw) break;
        const double yu = wx[w0 + q] - wt.x, du = yu * yu + wy2;
        const double ys = wx[w0 + q] + wt.x, ds = __builtin_fma(ys, ys, wy2);
        const bool m = du > pp.limittwo;
        const double r = rcp_cubic(m ? du : ds);
        if (m) {
            sach[q].x = __builtin_fma(__builtin_fma(P.x, yu, -PQ.x), r, sach[q].x);
            sach[q].y = __builtin_fma(__builtin_fma(P.y, yu, PQ.y), r, sach[q].y);
            sasx[q].x = __builtin_fma(BoOm.x, iwx2[w0 + q], sasx[q].x);
            sasx[q].y = __builtin_fma(BoOm.y, iwx2[w0 + q], sasx[q].y);
        } else {
            const double rs = du > 0.0 ? r : 0.0;
            sasx[q].x = __builtin_fma(__builtin_fma(R.x, ys, RQ.x), rs, sasx[q].x);
            sasx[q].y = __builtin_fma(__builtin_fma(R.y, ys, -RQ.y), rs, sasx[q].y);
        }
    }
    if constexpr (!MASK) {
        // B D where the mask would be off
#pragma unroll
        for (int q = 0; q < NWC; ++q) {
            if (!ALL && q > 0 && w0 + q >= pp.nw) break;
            const double yu = wx[w0 + q] - wt.x, du = yu * yu + wy2;
            if (!(du > pp.limittwo)) {
                const double r = rcp_cubic(du);
                sach[q].x = __builtin_fma(__builtin_fma(P.x, yu, -PQ.x), r, sach[q].x);
                sach[q].y = __builtin_fma(__builtin_fma(P.y, yu, PQ.y), r, sach[q].y);
            }
        }
    }
    return true;
}

}  // namespace gpp
}  // namespace fk
