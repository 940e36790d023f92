// fk_gpp_sym.hip -- the gppsum = 1 form of the GPP band loop on MI355X.
//
// gppKerSeq.cpp (the reference's sequential program, fifth argument gppsum)
// sums, for gppsum = 1, per band n1, column my_igp (igp from the column map)
// and frequency, only over ig <= igp, and adds beside every term m1 x its
// mirror m2 conj(x), m1 = aqsn[n1][ig] conj(aqsm[n1][igp]),
// m2 = conj(aqsm[n1][ig]) aqsm[n1][igp]:
//   occupied bands (flagOCC_solver :90-139): ig < igp, stopping at the first
//     ig with |wtilde^2 I_eps| < to1; near-pole (|wx - wtilde| < gamma or
//     |delw|^2 < to1, delw = (wx - wtilde) (0.5 / wtilde)): sch = 0,
//     ssx = -Omega2 / (4 wtilde^2 (1 + delw)); else sch = wtilde I_eps /
//     (wx - wtilde), ssx = Omega2 / (wx^2 - wtilde^2); the mirror is left
//     out at ig = igp - 1;
//   unoccupied bands (noflagOCC_solver :206-242, called per 512-wide block,
//     :438-450): every ig < igp - 1 except ig = 511 mod 512, plus the
//     diagonal ig = igp (m1 term only) when igp is a positive multiple of
//     512; only the near-pole terms are kept (|wdiff|^2 < limittwo or
//     |delw|^2 > limitone, delw = wtilde / wdiff), sch = delw I_eps.
//
// Summed over bands the m1 and m2 factors are two GEMMs with one left
// operand, c[n1][my_igp] = 0.5 vcoul[igp] conj(aqsm[n1][igp]) (the
// coefficient matrix of the canonical path):
//   Bu  = sum_{n1 >= nv} c aqsn[n1][ig],   Bu' = sum_{n1 >= nv} c aqsm[n1][ig],
// and m2-sums are conj(Bu'), so a term is Bu x + conj(Bu' x).  The kernel
// runs both on FP64 MFMA over the unoccupied bands of a 64 x 32 tile of
// (my_igp, ig) (a tile with no ig <= igp of its rows is skipped), forms the
// occupied-band sums Bo, Bo' by MFMA in the epilogue and evaluates the factors
// per element and frequency in FP64.  Near a branch threshold complex division
// is Smith's algorithm (R. L. Smith, "Algorithm 116: Complex
// division", CACM 5(8), 1962), the order of libgcc's __divdc3 that the
// reference's std::complex<double> calls, with IEEE quotients and no
// contraction; |z| is hypot.  Per-tile partials go to the reduction of the
// canonical path.
#include "fk_complex.h"
#include "fk_gpp_common.h"
#include "fk_internal.h"
#include "fk_mfma_ring.h"

#include <algorithm>
#include <climits>
#include <cmath>

namespace fk {
namespace {

using namespace gpp;

constexpr int kSymTile = 64, kSymCols = 32;   // rows and columns of a tile
constexpr int kSymBlocks = 512;  // row blocks whose tiles the kernel arguments can list
constexpr int kSymStages = 3, kSymWgs = 3;   // ring stages, workgroups per CU
constexpr int kSymWide = 256;    // workgroups of two tiles side by side, at most

// std::complex<double> product and quotient as the reference rounds them.
__device__ __forceinline__ double2 zmul(double2 a, double2 b)
{
#pragma clang fp contract(off)
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

__device__ __forceinline__ double2 zdiv(double2 a, double2 b)
{
#pragma clang fp contract(off)
    double ratio, denom;
    if (fabs(b.x) < fabs(b.y)) {
        ratio = b.x / b.y;
        denom = b.x * ratio + b.y;
        return make_double2((a.x * ratio + a.y) / denom, (a.y * ratio - a.x) / denom);
    }
    ratio = b.y / b.x;
    denom = b.y * ratio + b.x;
    return make_double2((a.y * ratio + a.x) / denom, (a.y - a.x * ratio) / denom);
}

__device__ __forceinline__ double znorm2(double2 a)
{
#pragma clang fp contract(off)
    return a.x * a.x + a.y * a.y;
}

// ig of the unoccupied sum of column igp: 1 both terms, 2 diagonal, 0 none
__device__ __forceinline__ int unocc_kind(int ig, int igp)
{
    if (ig == igp) return (igp > 0 && (igp & 511) == 0) ? 2 : 0;
    if (ig >= igp - 1) return 0;
    return (ig & 511) == 511 ? 0 : 1;
}

// stop[m] = the first ig < igp with |wtilde^2 I_eps| < to1, or igp (the
// occupied loop's break, gppKerSeq.cpp:99); 0 for a skipped column.  Four ig per
// thread and step, loaded together; |.| is the reference's hypot where the square
// does not settle it.  (One ig per step and a hypot for each: 60 us for
// 819 x 16384; this form 47.)
constexpr int kStopPer = 4;

__global__ __launch_bounds__(256) void gpp_sym_stop_kernel(const double2 *wtilde, const double2 *ieps, const int *igp,
                                                           int C, double to1, int *stop)
{
    __shared__ int found;
    const int m = blockIdx.x;
    const int g = igp[m];
    const double sure = 1.01 * to1 * to1;
    if (threadIdx.x == 0) found = INT_MAX;
    __syncthreads();
    const double2 *wr = wtilde + (size_t)m * C, *er = ieps + (size_t)m * C;
    for (int base = 0; base < g; base += 256 * kStopPer) {
        double2 w[kStopPer], e[kStopPer];
#pragma unroll
        for (int k = 0; k < kStopPer; ++k) {
            const int ig = min(base + 256 * k + (int)threadIdx.x, C - 1);
            w[k] = wr[ig];
            e[k] = er[ig];
        }
#pragma unroll
        for (int k = 0; k < kStopPer; ++k) {
            const int ig = base + 256 * k + (int)threadIdx.x;
            const double2 om = zmul(zmul(w[k], w[k]), e[k]);
            if (ig < g && !(to1 > 0.0 && sure > 1e-300 && znorm2(om) > sure) && hypot(om.x, om.y) < to1)
                atomicMin(&found, ig);
        }
        __syncthreads();
        // every thread reads `found` between the same two barriers: the
        // decision to stop is uniform
        const bool done = found != INT_MAX;
        __syncthreads();
        if (done) break;
    }
    if (threadIdx.x == 0) stop[m] = g < 0 ? 0 : min(found, g);
}

struct SymArgs {
    const double2 *c;        // [Kpad][ldc]: occupied rows 0..nv-1, zero rows to nvpad, unoccupied rows
    const double2 *aqsn;     // [nb][C]
    const double2 *aqsm;     // [nb][C]
    const double2 *I_eps;    // [G][C]
    const double2 *wtilde;   // [G][C]
    const int *igp;          // [G], -1 = skipped column
    const int *stop;         // [G] (read when nv > 0)
    double2 *partials;       // [workgroups][nw][2]
    int nb, nv, C, G, nw, ldc, nvpad, nks;
    int nblk, per;           // row blocks; tiles per workgroup
    int every;               // > 0: workgroups of every row block (more than kSymBlocks blocks)
    int first[kSymBlocks + 1];   // first workgroup of each row block
    double limittwo, limitone, to1, gamma;
    double lo, hi;           // sym_terms takes an element with lo < |wtilde|^2 < hi
    int aligned;             // 16-byte aligned: c (bit 0), aqsn and aqsm (bit 1)
    double wx[kMaxFreq];
};

// One element's unocc_kind, its occupied flag and whether its mirror counts.
struct SymElem { int kind; bool occ, mirror; };

__device__ __forceinline__ SymElem sym_elem(const SymArgs &a, int row, int col)
{
    SymElem e;
    const int g = (row < a.G && col < a.C) ? a.igp[row] : -1;
    e.kind = g >= 0 ? unocc_kind(col, g) : 0;
    e.occ = g >= 0 && a.nv > 0 && col < a.stop[row];
    e.mirror = col != g - 1;
    return e;
}

// The terms of one element at the NWC frequencies from w0, in the reference's
// operations and order (any wtilde, any limits).
template <int NWC>
__device__ __forceinline__ void sym_element(const SymArgs &a, int w0, SymElem e, double2 wt, double2 ie, double2 Bu,
                                            double2 Bp, double2 Bo, double2 Bpo, double2 (&sach)[NWC],
                                            double2 (&sasx)[NWC])
{
    const double2 wt2 = zmul(wt, wt);
    const double2 Om = zmul(wt2, ie);
    const double2 half = e.occ ? zdiv(make_double2(0.5, 0.0), wt) : make_double2(0.0, 0.0);
#pragma unroll
    for (int q = 0; q < NWC; ++q) {
        if (w0 + q >= a.nw) break;
        const double wxt = a.wx[w0 + q];
        const double2 wdiff = make_double2(wxt - wt.x, -wt.y);
        if (e.kind) {
            const double2 delw = zdiv(wt, wdiff);
            const double delw2 = znorm2(delw), wdiffr = znorm2(wdiff);
            if (fabs(wdiffr) < a.limittwo || delw2 > a.limitone) {
                const double2 sch = zmul(delw, ie);
                double2 t = cmul(Bu, sch);
                if (e.kind == 1) t = cadd(t, cconj(cmul(Bp, sch)));
                sach[q] = cadd(sach[q], t);
            }
        }
        if (e.occ) {
            const double2 delw = zmul(wdiff, half);
            const double ad = hypot(delw.x, delw.y);
            double2 sch = make_double2(0.0, 0.0), ssx = make_double2(0.0, 0.0);
            if (hypot(wdiff.x, wdiff.y) < a.gamma || ad * ad < a.to1) {
                if (hypot(wt.x, wt.y) > a.to1) {
                    const double2 den =
                        zmul(make_double2(4.0 * wt2.x, 4.0 * wt2.y), make_double2(1.0 + delw.x, delw.y));
                    ssx = zdiv(make_double2(-Om.x, -Om.y), den);
                }
            } else {
                sch = zdiv(zmul(wt, ie), wdiff);
                ssx = zdiv(Om, make_double2(wxt * wxt - wt2.x, -wt2.y));
            }
            double2 th = cmul(Bo, sch), ts = cmul(Bo, ssx);
            if (e.mirror) {
                th = cadd(th, cconj(cmul(Bpo, sch)));
                ts = cadd(ts, cconj(cmul(Bpo, ssx)));
            }
            sach[q] = cadd(sach[q], th);
            sasx[q] = cadd(sasx[q], ts);
        }
    }
}

// B x + conj(B' x) with (B + B').re etc. formed once.  A term is formed before it
// meets the sum, which is larger and rounds at its own size: with its two products
// added one by one the error against long double (rms of 150 problems of
// 30/4/400/64, 3M) is 3.5e-16 of the largest achtemp and 3.6e-16 of the largest
// asxtemp, so 3.4e-16 and 3.45e-16.
struct SymPair {
    double xr, xi, yr, yi;     // Re B + Re B', Im B + Im B', Re B - Re B', Im B - Im B'
    __device__ __forceinline__ SymPair(double2 b, double2 p)
        : xr(b.x + p.x), xi(b.y + p.y), yr(b.x - p.x), yi(b.y - p.y) {}
    __device__ __forceinline__ void add(double2 &sum, double2 x) const
    {
        sum.x += __builtin_fma(xr, x.x, -(xi * x.y));
        sum.y += __builtin_fma(yr, x.y, yi * x.x);
    }
};

// The same terms in a fifth of the operations, for lo < |wtilde|^2 < hi (else
// false, and nothing is added).  With u = wx - wtilde, s = wx + wtilde, T =
// wtilde I_eps:
//   near the pole (|u|^2 < limittwo):  unoccupied sch = T / u,
//                                      occupied   ssx = -T / (2 s)
//     (1 + delw = s / (2 wtilde), so Omega2 / (4 wtilde^2 (1 + delw)) = T / (2 s));
//   elsewhere, occupied only:          sch = T / u,  ssx = Omega2 / (wx^2 - wtilde^2).
// |wtilde|^2 < 0.99 limitone limittwo makes |delw|^2 > limitone imply |u|^2 <
// limittwo, and |wtilde|^2 < limittwo / (4.04 to1) makes |u / (2 wtilde)|^2 < to1
// imply it; |wtilde|^2 > 1.01 to1^2 decides |wtilde| > to1.  |u|^2 is rounded as
// the reference rounds it, but its occupied loop compares hypot(u) with gamma =
// sqrt(limittwo): an occupied element within 1e-12 of that line returns false too.
template <int NWC>
__device__ __forceinline__ bool sym_terms(const SymArgs &a, int w0, SymElem e, double2 wt, double2 ie, double2 Bu,
                                          double2 Bp, double2 Bo, double2 Bpo, double2 (&sach)[NWC],
                                          double2 (&sasx)[NWC])
{
#pragma clang fp contract(off)
    const double wy2 = wt.y * wt.y;
    const double wt2 = __builtin_fma(wt.x, wt.x, wy2);
    // 0 Bo near the pole is a NaN where Bo is not finite
    bool fast = wt2 > a.lo && wt2 < a.hi && fabs((Bo.x + Bo.y) + (Bpo.x + Bpo.y)) < __builtin_inf();
#pragma unroll
    for (int q = 0; q < NWC; ++q) {
        const double wdr = a.wx[min(w0 + q, a.nw - 1)] - wt.x, d = wdr * wdr + wy2;
        fast = fast && !(e.occ && fabs(d - a.limittwo) <= 1e-12 * a.limittwo);
    }
    if (!fast) return false;
    const double2 zero = make_double2(0.0, 0.0);
    const double2 T = cmul_fused(ie, wt), Om = cmul_fused(T, wt);
    const double w2r = __builtin_fma(wt.x, wt.x, -wy2), w2i = 2.0 * wt.x * wt.y;
    const SymPair U(Bu, e.kind == 1 ? Bp : zero), O(Bo, e.mirror ? Bpo : zero);
#pragma unroll
    for (int q = 0; q < NWC; ++q) {
        if (w0 + q >= a.nw) break;
        const double wx = a.wx[w0 + q];
        const double wdr = wx - wt.x, d = wdr * wdr + wy2;
        const bool near = d < a.limittwo;
        if (near ? e.kind != 0 : e.occ) {
            const double r = rcp_cubic(d);
            const double2 sch = make_double2(__builtin_fma(T.x, wdr, -(T.y * wt.y)) * r,
                                             __builtin_fma(T.y, wdr, T.x * wt.y) * r);
            if (near) U.add(sach[q], sch);
            else O.add(sach[q], sch);
        }
        if (e.occ) {
            // N conj(D) / |D|^2
            const double2 N = near ? make_double2(-0.5 * T.x, -0.5 * T.y) : Om;
            const double2 D = near ? make_double2(wx + wt.x, wt.y) : make_double2(wx * wx - w2r, -w2i);
            const double r = rcp_cubic(__builtin_fma(D.x, D.x, D.y * D.y));
            O.add(sasx[q], make_double2(__builtin_fma(N.x, D.x, N.y * D.y) * r, __builtin_fma(N.y, D.x, -(N.x * D.y)) * r));
        }
    }
    return true;
}

template <int NWC, int NG>
struct SymLds {
    union {
        double2 ring[kSymStages][2][8][64];      // [slot][coefficients; aqsn, aqsm][k][column]
        double2 b[4][3][4][64];                  // [wave][block - 1][register][lane]
    } tile[NG];
    double red[4 * NG][4 * NWC];
    double tot[kMaxFreq * 4];
    int last;                                    // the largest igp of the row block
};

// A 64 x 32 tile of (my_igp, ig) with both right operands side by side: 32
// columns of aqsn and the same 32 of aqsm are the 64
// columns of an LDS ring stage (fk_mfma_ring.h), and of a wave's two column blocks
// one is Bu and one Bu' of the same 16 ig.  Its three workgroups per CU are the
// FP64 tiles' of fk_gpp.hip, where the reasons stand, as is the epilogue: three of
// a wave's four blocks wait in the ring's memory, and the occupied bands are
// contracted per block.  The complex products are four real ones (ring::Acc4):
// with three (3M) the call below takes 550 us, but the imaginary parts of nearly
// real sums are lost (wavefunctions and matrices with inversion symmetry), and the
// error of the case itself is larger: 3.4e-16 against 3.0e-16 of the largest
// achtemp, 3.45e-16 against 3.2e-16 of the largest asxtemp (150 problems of
// 30/4/400/64 against long double).
//
// Only the tiles with some ig <= igp have a workgroup: the host lists them by
// row block (`per` of them in one workgroup where there are more than partials).
// Past kSymBlocks row blocks all tiles have one and those with none end at once,
// row blocks fastest (the kernel at 64/2/2000/40000: 1.39 ms with igp spread over
// all G-vectors, 0.11 with every igp below 64; with every tile evaluated, tile
// columns fastest, 2.33 and 2.28).
// Measured at 256/4/16384/819, 3 frequencies: the call 640 us, with contiguous ranges
// of 64 x 64 tiles per XCD, half of them empty, two workgroups per CU and every
// quotient and hypot evaluated 1486.
//
// NWC frequencies per epilogue pass: 4 where that takes fewer passes than 3
// (84/0/405/16 with 4 frequencies 41 us, in two passes 60; 422/13/14154/2971 with 16
// 4.2 ms, in six passes 4.5), else 3, which spills nothing (39/5/306/43 with 5
// frequencies 71 us, with 4 per pass 77).
//
// NG = 2: two tiles of a workgroup side by side on eight waves, for calls with two
// tiles per workgroup that do not fill the GPU (a few row blocks): 800/0/4000/50,
// the kernel 222 us, one after the other 256 (two workgroups would take 130, but the
// workspace holds a partial for each 64 x 64 tile only).
template <int NWC, int NG>
__global__ __launch_bounds__(256 * NG, NG == 1 ? kSymWgs : 1) void gpp_sym_kernel(SymArgs a)
{
    constexpr int MB = 2, NB = 2, NWAVES = 4 * NG, LPW = 4;
    __shared__ SymLds<NWC, NG> lds;
    const int tid = threadIdx.x, lane = tid & 63, wave_id = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave = wave_id & 3, group = wave_id >> 2;
    auto &sh = lds.tile[group];
    const int wm = wave & 1, wn = wave >> 1;
    int tm, h0;
    if (a.every > 0) {                             // row blocks fastest: few tile columns spread over all XCDs
        tm = blockIdx.x % a.nblk;
        h0 = (int)blockIdx.x / a.nblk * a.per;
    } else {
        int lo = 0, hi = a.nblk - 1;               // last row block with first <= this workgroup
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (a.first[mid] <= (int)blockIdx.x) lo = mid;
            else hi = mid - 1;
        }
        tm = lo;
        h0 = ((int)blockIdx.x - a.first[lo]) * a.per;
    }
    const int rowbase = tm * kSymTile + wm * 32, nmax = a.C - 1;
    const int kl = lane >> 4, cl = lane & 15;
    if (tid < kMaxFreq * 4) lds.tot[tid] = 0.0;
    if (a.every > 0 && wave_id == 0) {              // not listed: some of the tiles have no ig <= igp
        int g = tm * kSymTile + lane < a.G ? a.igp[tm * kSymTile + lane] : -1;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) g = max(g, __shfl_xor(g, off, 64));
        if (lane == 0) lds.last = min(g, nmax);
    }
    __syncthreads();
    const int n_last = a.every > 0 ? __builtin_amdgcn_readfirstlane(lds.last) : nmax;

    const bool side_a = wave < 2;
    const int k0 = 4 * (wave & 1);
    const int nun = a.nb - a.nv, nst = (nun + 7) / 8;
    const size_t ld = side_a ? (size_t)a.ldc : (size_t)a.C;
    const int row0 = (side_a ? a.nvpad : a.nv) + k0;
    const int last = side_a ? a.nks * 4 - 1 : a.nb - 1;
    const bool direct = a.aligned & (side_a ? 1 : 2);
    const int nko = (a.nv + 3) / 4;

    // (a second group past the last column has clamped ones and adds nothing)
    for (int h = h0; h < h0 + a.per && h * kSymCols <= n_last; h += NG) {
        const int n0 = (h + group) * kSymCols;
        // ---- GEMM over the unoccupied bands: Bu (right operand aqsn), Bu' (aqsm)
        const int lcol = min(n0 + (lane & 31), nmax);
        const double2 *src = side_a ? a.c + tm * kSymTile + lane : (lane < 32 ? a.aqsn : a.aqsm) + lcol;
        auto issue = [&](int s, int slot) {
            const int r = row0 + 8 * s;
            double2 *dst = &sh.ring[slot][side_a ? 0 : 1][k0][0];
            if (direct) {
#pragma unroll
                for (int j = 0; j < LPW; ++j) ring::lds_load16(src + (size_t)min(r + j, last) * ld, dst + 64 * j);
            } else {
#pragma unroll
                for (int j = 0; j < LPW; ++j) dst[64 * j + lane] = ring::load16(src + (size_t)min(r + j, last) * ld);
            }
        };
        auto read = [&](ring::Frags<MB, NB> &f, int s, int slot, int q) {
            const double2 *st = &sh.ring[slot][0][4 * q + kl][cl];
#pragma unroll
            for (int i = 0; i < MB; ++i) f.a[i] = st[wm * 32 + 16 * i];
#pragma unroll
            for (int j = 0; j < NB; ++j) f.b[j] = st[8 * 64 + 32 * j + wn * 16];
            if (8 * s + 8 > nun) {   // rows past the last band
                const bool kok = 8 * s + 4 * q + kl < nun;
#pragma unroll
                for (int i = 0; i < MB; ++i) f.a[i] = kok ? f.a[i] : make_double2(0.0, 0.0);
            }
        };
        ring::Acc4<MB, NB> acc;
        acc.zero();
        ring::main_loop<MB, NB, kSymStages, LPW>(nst, acc, issue, read);
        ring::wait_barrier<0>();

        // ---- epilogue
        double2 Bu0[4];
#pragma unroll
        for (int k = 0; k < MB * NB; ++k)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const double2 v = acc.value(k / NB, k % NB, r);
                if (k == 0) Bu0[r] = v;
                else sh.b[wave][k - 1][r][lane] = v;
            }
        for (int w0 = 0; w0 < a.nw; w0 += NWC) {
            double2 sach[NWC], sasx[NWC];
#pragma unroll
            for (int q = 0; q < NWC; ++q) { sach[q] = make_double2(0.0, 0.0); sasx[q] = make_double2(0.0, 0.0); }
            unsigned general = 0;
            int kp = kl, cp = cl;      // opaque in each pass (gpp_ring_tile)
            asm volatile("" : "+v"(kp), "+v"(cp));
            const int col = n0 + wn * 16 + cp;
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                __builtin_amdgcn_sched_barrier(0);
                double2 cwt[4], cie[4];
                auto load = [&](int r) {
                    const int row = rowbase + i * 16 + 4 * r + kp;
                    const size_t e = (size_t)min(row, a.G - 1) * a.C + min(col, nmax);
                    cwt[r] = a.wtilde[e];
                    cie[r] = a.I_eps[e];
                };
                load(0);
                load(1);
                ring::Acc4<1, 2> o;
                o.zero();
                for (int ks = 0; ks < nko; ++ks) {
                    ring::Frags<1, 2> f;
                    const size_t rb = (size_t)min(4 * ks + kp, a.nv - 1) * a.C + min(col, nmax);   // occupied bands only (gpp_ring_tile)
                    f.a[0] = a.c[(size_t)(4 * ks + kp) * a.ldc + rowbase + 16 * i + cp];
                    f.b[0] = a.aqsn[rb];
                    f.b[1] = a.aqsm[rb];
                    o.mma(f);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    __builtin_amdgcn_sched_barrier(0);
                    if (r == 1) {
                        load(2);
                        load(3);
                    }
                    const SymElem e = sym_elem(a, rowbase + i * 16 + 4 * r + kp, col);
                    if (e.kind || e.occ) {
                        const double2 Bu = i == 0 ? Bu0[r] : sh.b[wave][1][r][lane];
                        const double2 Bp = sh.b[wave][2 * i][r][lane];
                        if (!sym_terms<NWC>(a, w0, e, cwt[r], cie[r], Bu, Bp, o.value(0, 0, r), o.value(0, 1, r), sach,
                                                sasx))
                            general |= 1u << (4 * i + r);
                    }
                }
            }
            // the elements sym_terms left out, one at a time
            if (__ballot(general != 0)) {
#pragma unroll 1
                for (int el = 0; el < MB * 4; ++el) {
                    if ((general >> el) & 1u) {
                        const int i = el >> 2, r = el & 3, row = rowbase + 16 * i + 4 * r + kp;
                        double2 Bu;
                        switch (el) {             // constant register indices
                        case 0: Bu = Bu0[0]; break;
                        case 1: Bu = Bu0[1]; break;
                        case 2: Bu = Bu0[2]; break;
                        case 3: Bu = Bu0[3]; break;
                        default: Bu = sh.b[wave][1][r][lane];
                        }
                        const double2 Bp = sh.b[wave][2 * i][r][lane];
                        double2 Bo = make_double2(0.0, 0.0), Bpo = Bo;
                        for (int n1 = 0; n1 < a.nv; ++n1) {
                            const double2 cn = a.c[(size_t)n1 * a.ldc + row];
                            Bo = cfma(Bo, cn, a.aqsn[(size_t)n1 * a.C + col]);
                            Bpo = cfma(Bpo, cn, a.aqsm[(size_t)n1 * a.C + col]);
                        }
                        const size_t x = (size_t)row * a.C + col;
                        sym_element<NWC>(a, w0, sym_elem(a, row, col), a.wtilde[x], a.I_eps[x], Bu, Bp, Bo, Bpo, sach,
                                             sasx);
                    }
                }
            }
            // wave reduction, then a fixed-order sum over the waves and tiles
            double v[4 * NWC];
#pragma unroll
            for (int q = 0; q < NWC; ++q) {
                v[4 * q + 0] = sach[q].x;
                v[4 * q + 1] = sach[q].y;
                v[4 * q + 2] = sasx[q].x;
                v[4 * q + 3] = sasx[q].y;
            }
#pragma unroll
            for (int q = 0; q < 4 * NWC; ++q) {
                const double x = wave_sum(v[q]);
                if (lane == 0) lds.red[wave_id][q] = x;
            }
            __syncthreads();
            if (tid < 4 * NWC && w0 + (tid >> 2) < a.nw) {
                double sum = lds.red[0][tid];
#pragma unroll
                for (int w = 1; w < NWAVES; ++w) sum += lds.red[w][tid];
                lds.tot[4 * w0 + tid] += sum;
            }
            __syncthreads();
        }
    }
    __syncthreads();
    if (tid < 4 * a.nw) reinterpret_cast<double *>(a.partials + (size_t)blockIdx.x * a.nw * 2)[tid] = lds.tot[tid];
}

}  // namespace

int gpp_sym_launch(const fk_gpp_problem *p, const std::vector<int32_t> &cols, const double2 *c, int ldc, int Kpad,
                   int nvpad, const int *d_igp, int *d_stop, const double2 *aqsm, const double2 *aqsn, const double2 *ieps,
                   const double2 *wt, double2 *partials, size_t max_partials, int *count, float *kernel_ms, hipStream_t s)
{
    if (p->nvband > 0) {
        hipLaunchKernelGGL(gpp_sym_stop_kernel, dim3(p->ngpown), dim3(256), 0, s, wt, ieps, d_igp, p->ncouls, p->to1,
                           d_stop);
        FK_HIP(hipGetLastError());
    }
    SymArgs a;
    a.c = c; a.aqsn = aqsn; a.aqsm = aqsm; a.I_eps = ieps; a.wtilde = wt; a.igp = d_igp; a.stop = d_stop;
    a.partials = partials;
    a.nb = p->number_bands; a.nv = p->nvband; a.C = p->ncouls; a.G = p->ngpown; a.nw = p->nfreq;
    a.ldc = ldc; a.nvpad = nvpad; a.nks = Kpad / 4;
    // the tiles of each row block: columns 0 .. its largest igp
    a.nblk = div_up(p->ngpown, kSymTile);
    std::vector<int> tiles(a.nblk, div_up(p->ncouls, kSymCols));
    const bool listed = a.nblk <= kSymBlocks;
    int64_t total = 0;
    for (int b = 0; b < a.nblk; ++b) {
        if (listed) {
            int g = -1;
            for (int m = b * kSymTile; m < std::min((b + 1) * kSymTile, p->ngpown); ++m) g = std::max(g, (int)cols[m]);
            tiles[b] = (std::min(g, p->ncouls - 1) + kSymCols) / kSymCols;   // 0 for g = -1
        }
        total += tiles[b];
    }
    a.per = total <= (int64_t)max_partials ? 1 : 2;   // two per workgroup are a 64 x 64 tile's worth of partials
    a.every = listed ? 0 : div_up(tiles[0], a.per);
    int blocks = 0;
    for (int b = 0; b < a.nblk; ++b) {
        if (listed) a.first[b] = blocks;
        blocks += div_up(tiles[b], a.per);
    }
    *count = blocks;
    a.limittwo = p->limittwo; a.limitone = p->limitone; a.to1 = p->to1; a.gamma = std::sqrt(p->limittwo);
    a.lo = a.hi = 0.0;
    if (p->limittwo > 0.0 && p->limitone > 0.0 && p->to1 >= 0.0) {
        a.lo = 1.01 * p->to1 * p->to1;
        a.hi = 0.99 * p->limitone * p->limittwo;
        if (p->to1 > 0.0) a.hi = std::min(a.hi, p->limittwo / (4.04 * p->to1));
    }
    a.aligned = ring::aligned16(c) | (ring::aligned16(aqsn) & ring::aligned16(aqsm)) << 1;
    for (int iw = 0; iw < kMaxFreq; ++iw) a.wx[iw] = iw < p->nfreq ? p->wx[iw] : 0.0;
    KernelTimer timer(kernel_ms, s);
    FK_TRY(timer.start());
    if (blocks > 0) {
        const bool four = div_up(p->nfreq, 4) < div_up(p->nfreq, 3);
        if (a.per == 2 && blocks <= kSymWide) {
            if (four) hipLaunchKernelGGL((gpp_sym_kernel<4, 2>), dim3(blocks), dim3(512), 0, s, a);
            else hipLaunchKernelGGL((gpp_sym_kernel<3, 2>), dim3(blocks), dim3(512), 0, s, a);
        } else {
            if (four) hipLaunchKernelGGL((gpp_sym_kernel<4, 1>), dim3(blocks), dim3(256), 0, s, a);
            else hipLaunchKernelGGL((gpp_sym_kernel<3, 1>), dim3(blocks), dim3(256), 0, s, a);
        }
    }
    FK_HIP(hipGetLastError());
    FK_TRY(timer.stop());
    return timer.finish();
}

}  // namespace fk
