// fk_gpp_oz.hip -- mixed-precision GPP band sum on MI355X (gfx950): the
// band contraction B = sum_n1 c[n1] aqsn[n1] runs on int8 MFMA with exact
// int32 accumulation (an Ozaki-style split, Ozaki, Ogita, Oishi & Rump,
// "Error-free transformations of matrix multiplication", Numer. Algorithms
// 59 (2012); on integer matrix units: Ootomo, Ozaki & Yokota, IJHPCA 2024);
// everything else is FP64.
//
// Inputs are complex64 (fk_cfloat).  The complex product runs as three real
// products (Gauss):
//     P0 = cr ar,   P1 = ci ai,   P2 = (cr + ci)(ar + ai),
//     re B = P0 - P1,   im B = P2 - P0 - P1,
// over the matrices cr, ci, cr + ci of the coefficients c[n1][my_igp] =
// 0.5 vcoul[igp] conj(aqsm[n1][igp]) (FP64) and ar, ai, ar + ai of aqsn.
// Each row of each coefficient matrix and each column of each aqsn matrix
// is scaled so that its largest magnitude (M) maps to 127 and split into
// four int8 slices:
//     x = M / 127 * (s0 + s1/254 + s2/254^2 + s3/254^3),  |s_k| <= 127,
// 31 bits of the row's or column's range.  The slice pairs (i, j) with
// i + j = L share the weight 254^-L, so four int32 accumulators per product
// (L = 0..3; the pairs with i + j > 3 are below 254^-4 of the leading term
// and dropped) hold the contraction exactly: 3 x 10 slice pairs, 30 int8
// MFMAs per 32 bands.  The error against the FP64 evaluation on the same
// complex64 values is the slice truncation's, a few 1e-9 relative at most
// (2.4e-9 at 512/2/32768/1638).
//
// Kernels (one call = four launches on the caller's stream):
//   oz_prep_kernel       row / column maxima of the six matrices, their
//                        int8 slices, FP64 occupied rows
//   gpp_oz_gemm_kernel   int8 MFMA tile, operands staged through a
//                        three-stage LDS ring by direct global->LDS loads;
//                        B rebuilt in FP64 and stored
//   gpp_oz_pole_kernel   per (my_igp, ig): occupied-band sum Bo in FP64, the
//                        pole and SX factors in FP64, per-block partials
//   gpp_reduce_kernel    fixed-order sum of the partials (shared with FP64)
//
// Slices are stored in MFMA-lane order: a 1 KB block per (plane, 32 rows,
// 32 bands) in which lane L's 16 bytes (row L%32, bands 16 (L/32) .. +15)
// sit at byte 16 L, so one direct-to-LDS load moves a whole operand
// fragment of the 32x32x32 int8 MFMA and the MFMA reads it back with one
// conflict-free ds_read_b128 per lane.  (The 16x16x64 int8 MFMA runs at
// half the int8 rate on this part; the 32x32x32 form reaches it.)
#include "fk_complex.h"
#include "fk_gpp_common.h"
#include "fk_internal.h"
#include "fk_mfma_ring.h"

#include <algorithm>
#include <cstddef>
#include <cstring>
#include <type_traits>

namespace fk {
namespace {

using namespace gpp;
typedef int i4 __attribute__((ext_vector_type(4)));

constexpr int kSlices = 4;
constexpr int kProds = 3;       // P0 = cr ar, P1 = ci ai, P2 = (cr + ci)(ar + ai)
constexpr int kLevels = 4;      // slice pairs with i + j < kLevels
constexpr int kKStep = 32;      // bands per pipeline step = the K of one 32x32x32 int8 MFMA
constexpr int kPlanes = kProds * kSlices;   // slice planes per operand
constexpr int kFrag = 1024;     // bytes per lane-ordered fragment
constexpr int kMaxBandsOz = 16000;   // keeps the level-3 int32 sums (4 pairs) below 2^31

// Slices of x, |x| <= M (scale = 127 / M), in units of M/127 (first) and
// /254 per level.  The scaling rounds once at 2^-53 relative; every later
// step is exact.
__device__ __forceinline__ void split4(double x, double scale, int8_t (&s)[kSlices])
{
    double t = x * scale;
    double q = rint(t);
    s[0] = (int8_t)q;
#pragma unroll
    for (int k = 1; k < kSlices; ++k) {
        t = (t - q) * 254.0;
        q = rint(t);
        s[k] = (int8_t)q;
    }
}


// ---------------------------------------------------------------------------
// Slices of both operands in one launch.  A workgroup takes 8 coefficient
// rows (the first ldm/8 workgroups) or 16 aqsn columns (the rest).  Each
// row (column) feeds three real matrices, cr, ci, cr + ci (ar, ai, ar + ai),
// each with its own scale: the workgroup finds the three maxima over all
// bands, then splits the three values of each band into four slices, band
// block by band block (16 bands = the 16 bytes of one fragment lane); a
// thread's first block stays in registers in between, the others are read
// again.  Thread t of an R-wide slab: row or column R x + t%R, band blocks t/R,
// t/R + 512/R, ...
// ---------------------------------------------------------------------------
struct PrepArgs {
    const float2 *aqsm, *aqsn;
    const double *vcoul;
    const int *igp;
    int8_t *as, *bs;         // [12][ldm/32][nkb][1024], [12][ldn/32][nkb][1024]: plane = matrix * 4 + slice
    double *ra, *rb;         // [3][ldm], [3][ldn]: M / 127 of each row, column of each matrix
    double2 *c_occ;          // [nv][ldm] coefficients of the occupied bands
    int nb, nv, C, G, ldm, ldn, nkb, blocks_a;
};

// R rows (coefficients, IS_A) or columns (aqsn) per workgroup, kPrepThreads / R
// band groups: the coefficients are gathered at scattered igp columns, so their
// slabs are kept thin to spread the gathers over more workgroups.  A thread's
// first 16 bands stay in registers between the two passes (all of them up to 512
// bands of aqsn), loaded 16 at once.  Measured at 512/2/32768/1638: 114 us, with
// 256 threads that read every band twice 184.
constexpr int kPrepThreads = 512;

template <int R, bool IS_A>
__device__ __forceinline__ void prep_slab(const PrepArgs &a, int slab)
{
    constexpr int NG = kPrepThreads / R, NW = kPrepThreads / 64;
    __shared__ double sm[kProds][NW][R];
    const int tid = threadIdx.x, c = tid % R, grp = tid / R;
    const int idx = slab * R + c;
    const int g = IS_A ? (idx < a.G ? a.igp[idx] : -1) : idx;
    const bool in = IS_A ? g >= 0 : idx < a.C;
    const float2 *src = (IS_A ? a.aqsm : a.aqsn) + (in ? g : 0);
    const double vs = IS_A && in ? 0.5 * a.vcoul[g] : 0.0;
    // bands 16 j .. 16 j + 15 of this row or column, as stored
    float2 raw[16];
    auto load = [&](int j) {
#pragma unroll
        for (int b = 0; b < 16; ++b)
            raw[b] = in && 16 * j + b < a.nb ? src[(size_t)(16 * j + b) * a.C] : make_float2(0.f, 0.f);
    };
    // the coefficient c or the value of aqsn
    auto value = [&](float2 v) -> double2 {
        if constexpr (IS_A) return make_double2((double)v.x * vs, -(double)v.y * vs);
        else return make_double2((double)v.x, (double)v.y);
    };
    const int nblk = (a.nb + 15) / 16;
    double mx[kProds] = {0.0, 0.0, 0.0};
    auto maxima = [&]() {
#pragma unroll
        for (int b = 0; b < 16; ++b) {
            const double2 v = value(raw[b]);
            mx[0] = fmax(mx[0], fabs(v.x));
            mx[1] = fmax(mx[1], fabs(v.y));
            mx[2] = fmax(mx[2], fabs(v.x + v.y));
        }
    };
    for (int j = grp + NG; j < nblk; j += NG) {
        load(j);
        maxima();
    }
    load(grp);
    maxima();
#pragma unroll
    for (int pr = 0; pr < kProds; ++pr) {
#pragma unroll
        for (int off = R; off < 64; off <<= 1) mx[pr] = fmax(mx[pr], __shfl_xor(mx[pr], off, 64));
        if ((tid & 63) < R) sm[pr][tid >> 6][c] = mx[pr];
    }
    __syncthreads();
    const int ld = IS_A ? a.ldm : a.ldn;
    double scale[kProds];
#pragma unroll
    for (int pr = 0; pr < kProds; ++pr) {
        double m = 0.0;
#pragma unroll
        for (int k = 0; k < NW; ++k) m = fmax(m, sm[pr][k][c]);
        scale[pr] = m > 0.0 ? 127.0 / m : 0.0;
        if (grp == 0) (IS_A ? a.ra : a.rb)[(size_t)pr * ld + idx] = m / 127.0;
    }

    int8_t *base = IS_A ? a.as : a.bs;
    const size_t blk = idx >> 5, nblks = (size_t)ld / 32;
    // 16-band blocks of the padded K, one 16-byte store per plane
    for (int j = grp; j < a.nkb * 2; j += NG) {
        if (j != grp) load(j);
        const int lane = (idx & 31) + 32 * (j & 1), kb = j >> 1;
        // One product's planes at a time: 16 registers of packed bytes.  The
        // stored values are opaque in each, or their 32 FP64 forms would be kept
        // from one to the next (spilled).
#pragma unroll
        for (int pr = 0; pr < kProds; ++pr) {
            uint32_t q[kSlices][4] = {};
#pragma unroll
            for (int b = 0; b < 16; ++b) asm volatile("" : "+v"(raw[b].x), "+v"(raw[b].y));
#pragma unroll
            for (int b = 0; b < 16; ++b) {
                const double2 v = value(raw[b]);
                if (IS_A && pr == 0 && 16 * j + b < a.nv) a.c_occ[(size_t)(16 * j + b) * a.ldm + idx] = v;
                int8_t sl[kSlices];
                split4(pr == 0 ? v.x : pr == 1 ? v.y : v.x + v.y, scale[pr], sl);
#pragma unroll
                for (int k = 0; k < kSlices; ++k) q[k][b >> 2] |= (uint32_t)(uint8_t)sl[k] << (8 * (b & 3));
            }
#pragma unroll
            for (int k = 0; k < kSlices; ++k) {
                int8_t *dst = base + (((size_t)(pr * kSlices + k) * nblks + blk) * a.nkb + kb) * kFrag + 16 * lane;
                *reinterpret_cast<uint4 *>(dst) = make_uint4(q[k][0], q[k][1], q[k][2], q[k][3]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

constexpr int kPrepRowsA = 8, kPrepColsB = 16;

__device__ __forceinline__ void oz_prep_block(const PrepArgs &a, int b)
{
    if (b < a.blocks_a) prep_slab<kPrepRowsA, true>(a, b);
    else prep_slab<kPrepColsB, false>(a, b - a.blocks_a);
}

__global__ __launch_bounds__(kPrepThreads, 4) void oz_prep_kernel(PrepArgs a)
{
    oz_prep_block(a, blockIdx.x);
}

// ---------------------------------------------------------------------------
// int8 MFMA GEMM.  64x64 workgroup tile of 2x2 blocks of 32x32.
// 32x32x32 int8 MFMA: lane l supplies 16 bytes of row l%32 of A and
// of column l%32 of B at the same 16 bands; accumulator register j of lane
// l holds row 8 (j/4) + 4 (l/32) + j%4, column l%32.
//
// The complex product as three real products (Gauss):
//     P0 = cr ar,   P1 = ci ai,   P2 = (cr + ci)(ar + ai),
//     re B = P0 - P1,   im B = P2 - P0 - P1,
// each matrix with its own row (column) scales.  Each product runs the ten
// slice pairs of levels 0..3: 30 MFMAs per 32 bands.  (The complex product
// as two real products over an interleaved K' = 2 nb with one scale per row
// and column needs all 13 pairs of levels 0..4 for the same accuracy: 52
// MFMAs.)
//
// LDS ring of kStages steps of 32 bands; a stage holds the workgroup's 24 A
// fragments ([matrix][slice][row block]) and 24 B fragments
// ([matrix][slice][column block]), 48 KB.  Twelve waves, three per SIMD:
// wave w owns the 32x32 block w % 4 and the product w / 4.  Each wave moves
// 4 fragments per step with direct global->LDS loads, issued over the first
// MFMAs of step s for step s+2, into the stage step s-1 used; after its
// fifth MFMA it waits for its loads of step s+1 and passes a barrier that
// covers every wave's loads, and its next MFMAs carry the 8 LDS reads of
// its fragments of step s+1 into the other register set.  With three waves
// per SIMD the MFMA pipe is fed by whichever wave is ready (one wave per
// SIMD, each computing all three products of its block, left the pipes
// busy 47% of the time).
// ---------------------------------------------------------------------------
constexpr int kBM = 64, kBN = 64, kGroupM = 4, kStages = 3;
constexpr int kFragsA = kPlanes * (kBM / 32), kFragsB = kPlanes * (kBN / 32);   // 24, 24
constexpr int kFragsPerStage = kFragsA + kFragsB;          // 48

// slice pairs of a wave's step in MFMA order; levels si + sj: 3 2 1 3 2 1
// 3 2 0 3 (an accumulator is reused at most every third MFMA)
struct PairStep { int si, sj; };
constexpr int kPairs = 10;
constexpr PairStep kOrder[kPairs] = {{0, 3}, {0, 2}, {0, 1}, {1, 2}, {1, 1},
                                     {1, 0}, {2, 1}, {2, 0}, {0, 0}, {3, 0}};

struct GemmArgs {
    const int8_t *as, *bs;
    const double *ra, *rb;   // [3][ldm], [3][ldn]: M / 127 of each row, column of each matrix
    double2 *bmat;           // [ldm][ldn] B in FP64
    int ldm, ldn, nkb, tiles_m, tiles_n, group_m;
};

typedef int i16v __attribute__((ext_vector_type(16)));

__device__ __forceinline__ i16v mfma_i8(i4 a, i4 b, i16v c)
{
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
}

// Workgroup b -> tile.  Each XCD runs a contiguous range of the logical
// order; the logical order walks bands of group_m row tiles, column by
// column, so a band's coefficient slices stay in the XCD's L2 while the
// aqsn slices stream past.
__device__ __forceinline__ void oz_tile(int b, int tiles_m, int tiles_n, int group_m, int &tm, int &tn)
{
    const int total = tiles_m * tiles_n;
    const int q = total / kXcds, r = total % kXcds, x = b % kXcds, i = b / kXcds;
    const int t = (x < r) ? x * (q + 1) + i : r * (q + 1) + (x - r) * q + i;
    const int band = t / (group_m * tiles_n);
    const int first = band * group_m;
    const int gm = min(tiles_m - first, group_m);
    const int u = t - band * group_m * tiles_n;
    tm = first + u % gm;
    tn = u / gm;
}


// ring::lds_load16 from a wave-uniform base (kept in SGPRs) plus a per-lane byte
// offset: one VGPR serves every load of the kernel.
__device__ __forceinline__ void lds_load16(const int8_t *base, unsigned voff, const int8_t *lds)
{
    const unsigned la = (unsigned)__builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)lds);
    const uint64_t bu = (uint64_t)(uintptr_t)base;
    // readfirstlane yields an int: widen through unsigned (no sign extension)
    const uint64_t ub = ((uint64_t)(unsigned)__builtin_amdgcn_readfirstlane((unsigned)(bu >> 32)) << 32) |
                        (uint64_t)(unsigned)__builtin_amdgcn_readfirstlane((unsigned)bu);
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(ub), "s"(la)
                 : "memory", "m0");
}

// ---------------------------------------------------------------------------
// The same 64x64 tile with 12 waves, three per SIMD: wave w owns the 32x32
// block w % 4 and the product w / 4 (4 accumulators, 10 MFMAs per step).
// The LDS ring and its layout are those above; each wave moves 4 of a
// step's 48 fragments and reads the 8 of its block and product.  With three
// waves per SIMD the MFMA pipe is fed by whichever wave is ready.  The
// epilogue meets the three products of a block in the (then free) ring:
// the waves of products 1 and 2 leave P there, those of product 0 form B.
// ---------------------------------------------------------------------------
constexpr int kWaves12 = 12;
constexpr int kLoads12 = kFragsPerStage / kWaves12;   // 4
constexpr int kWait12 = 4;                            // MFMA after which a wave waits
// a wave's 8 fragments in the order of their first use by its step
struct Frag8 { bool a; int sl; };
constexpr Frag8 kRead12[2 * kSlices] = {{true, 0}, {false, 3}, {false, 2}, {false, 1},
                                        {true, 1}, {false, 0}, {true, 2}, {true, 3}};

__device__ __forceinline__ void wait_loads_barrier4(int n)
{
    if (n == 4) asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

struct Frags12 {
    i4 a[kSlices];   // this wave's product, row block
    i4 b[kSlices];   // this wave's product, column block
};

// Tiles first, first + stride, ... (count >= 1 of them) in launch order on
// one workgroup.  With PERSIST, the last two steps of a tile load the first
// two of the next (the last tile reloads its own: one code path), and the
// tile's scales travel as three more direct loads (waves 0..2, 1 KB each)
// into a double-buffered LDS area; without it (one tile per workgroup) the
// last two steps load nothing.  The epilogue forms this wave's scaled P,
// waits for and reads the next tile's step-0 fragments, then meets the
// three products of its block in the ring stage no load is writing (two
// rounds of 8 rows), and the product-0 waves store B.
template <bool PERSIST>
__device__ __forceinline__ void oz_gemm12_tiles(const GemmArgs &a, int first, int stride, int count)
{
    __shared__ __attribute__((aligned(16))) int8_t lds[kStages][kFragsPerStage][kFrag];
    __shared__ __attribute__((aligned(16))) double scl[2][2 * kProds][kBM];   // [tile parity][ra 0..2, rb 0..2][64]

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int blk = wave & 3, pr = wave >> 2;
    const int wm = blk & 1, wn = blk >> 1;
    const int nks = a.nkb;

    // this wave's loads: stage fragment f = 4 wave + k, A (plane f/2, row
    // block 2 tm + f%2) for f < 24, else B (plane (f-24)/2, column block
    // 2 tn + f%2); waves 0..5 move A, 6..11 B.  koff: from the tile's base.
    const bool side_a = kLoads12 * wave < kFragsA;
    const size_t nblk = (size_t)(side_a ? a.ldm : a.ldn) / 32;
    const int8_t *uside = side_a ? a.as : a.bs;
    auto koff = [&](int k) -> size_t {
        const int q = kLoads12 * wave + k - (side_a ? 0 : kFragsA);
        return ((size_t)(q >> 1) * nblk + (q & 1)) * a.nkb * kFrag;
    };
    auto tile_src = [&](int b) -> const int8_t * {
        int tm, tn;
        oz_tile(b, a.tiles_m, a.tiles_n, a.group_m, tm, tn);
        return uside + (size_t)(2 * (side_a ? tm : tn)) * a.nkb * kFrag;
    };
    const unsigned voff = 16 * lane;
    auto stage = [&](int g) -> int8_t * { return &lds[g % kStages][0][0]; };
    auto issue = [&](const int8_t *src, int g, int k) {
        lds_load16(src + koff(k), voff, stage(g) + (kLoads12 * wave + k) * kFrag);
    };
    // scale pieces of tile b (waves 0..2): lanes 0..31 piece 2w, lanes
    // 32..63 piece 2w+1 (0..2 ra rows, 3..5 rb columns), 2 doubles a lane
    auto issue_scales = [&](int b, int t) {
        if (wave < kProds) {
            int tm, tn;
            oz_tile(b, a.tiles_m, a.tiles_n, a.group_m, tm, tn);
            const int q = 2 * wave + (lane >> 5);
            const double *g = q < kProds ? a.ra + (size_t)q * a.ldm + tm * kBM
                                         : a.rb + (size_t)(q - kProds) * a.ldn + tn * kBN;
            ring::lds_load16(g + 2 * (lane & 31), &scl[t & 1][2 * wave][0]);
        }
    };
    auto read_frag = [&](const int8_t *st, Frags12 &f, int r) {
        const Frag8 fr = kRead12[r];
        if (fr.a) f.a[fr.sl] = *reinterpret_cast<const i4 *>(st + (pr * 8 + fr.sl * 2 + wm) * kFrag + 16 * lane);
        else f.b[fr.sl] = *reinterpret_cast<const i4 *>(st + (kFragsA + pr * 8 + fr.sl * 2 + wn) * kFrag + 16 * lane);
    };

    i16v acc[kLevels];

    // the g-th step of this workgroup: MFMAs from `cur`; with LOADS, the 4
    // loads from `src` into the stage of step g+2 (and with SCALES tile
    // b's scales after them); with NEXT, the wait for step g+1 after MFMA
    // kWait12 and its fragments read into `nxt`
    auto step = [&](auto next_t, auto loads_t, auto scales_t, const Frags12 &cur, Frags12 &nxt, int g,
                    const int8_t *src, int b, int t) {
        constexpr bool NEXT = decltype(next_t)::value;
        constexpr bool LOADS = decltype(loads_t)::value;
        constexpr bool SCALES = decltype(scales_t)::value;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int o = 0; o < kPairs; ++o) {
            const PairStep ps = kOrder[o];
            acc[ps.si + ps.sj] = mfma_i8(cur.a[ps.si], cur.b[ps.sj], acc[ps.si + ps.sj]);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (LOADS) {
                if (o < kLoads12) issue(src, g + 2, o);
                if constexpr (SCALES) {
                    if (o == kLoads12 - 1) issue_scales(b, t);
                }
            }
            if constexpr (NEXT) {
                if (o == kWait12) wait_loads_barrier4(LOADS ? 4 : 0);
                if (o > kWait12 && o <= kWait12 + kSlices) {
                    read_frag(stage(g + 1), nxt, 2 * (o - kWait12 - 1));
                    read_frag(stage(g + 1), nxt, 2 * (o - kWait12 - 1) + 1);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    using yes = std::integral_constant<bool, true>;
    using no = std::integral_constant<bool, false>;

    // Waits: vmcnt counts this wave's direct loads (4 a step, plus one
    // scale piece for waves 0..2 issued after a step's loads) and B stores;
    // the loads complete in issue order, and a wait allows only the 4 loads
    // issued after the step waited for, so it is correct whatever the
    // stores do.
    Frags12 h0, h1;
    const int8_t *src = tile_src(first);
#pragma unroll
    for (int k = 0; k < kLoads12; ++k) issue(src, 0, k);
    issue_scales(first, 0);
#pragma unroll
    for (int k = 0; k < kLoads12; ++k) issue(src + kFrag, 1, k);
    wait_loads_barrier4(4);
#pragma unroll
    for (int r = 0; r < 2 * kSlices; ++r) read_frag(stage(0), h0, r);

    typedef double d2v __attribute__((ext_vector_type(2)));
    const double W[kLevels] = {1.0, 1.0 / 254.0, 1.0 / 64516.0, 1.0 / 16387064.0};
    int g = 0, b = first;
    for (int t = 0; t < count; ++t, b += stride, g += nks) {
#pragma unroll
        for (int L = 0; L < kLevels; ++L) acc[L] = i16v{};
        int s = 0;
        for (; s + 2 < nks; s += 2) {
            step(yes{}, yes{}, no{}, h0, h1, g + s, src + (size_t)(s + 2) * kFrag, b, t);
            step(yes{}, yes{}, no{}, h1, h0, g + s + 1, src + (size_t)(s + 3) * kFrag, b, t);
        }
        const int8_t *nsrc = src;
        if constexpr (PERSIST) {
            const bool more = t + 1 < count;
            const int bn = more ? b + stride : b;
            nsrc = tile_src(bn);
            step(yes{}, yes{}, yes{}, h0, h1, g + s, nsrc, bn, t + 1);
            step(no{}, yes{}, no{}, h1, h0, g + s + 1, nsrc + kFrag, b, t);
        } else {
            step(yes{}, no{}, no{}, h0, h1, g + s, src, b, t);
            step(no{}, no{}, no{}, h1, h0, g + s + 1, src, b, t);
        }
        src = nsrc;

        // P of this wave's product, scaled
        int tm, tn;
        oz_tile(b, a.tiles_m, a.tiles_n, a.group_m, tm, tn);
        const double *sc = &scl[t & 1][0][0];
        const double rbc = sc[(kProds + pr) * kBM + wn * 32 + (lane & 31)];
        double P[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int r = wm * 32 + 8 * (j >> 2) + 4 * (lane >> 5) + (j & 3);
            double v = 0.0;
#pragma unroll
            for (int L = kLevels - 1; L >= 0; --L) v += W[L] * (double)acc[L][j];
            P[j] = v * sc[pr * kBM + r] * rbc;
        }
        __builtin_amdgcn_sched_barrier(0);
        // the next tile's step-0 fragments (PERSIST), or just a barrier:
        // after it every wave is done with the ring of this tile
        if constexpr (PERSIST) {
            wait_loads_barrier4(4);
#pragma unroll
            for (int r = 0; r < 2 * kSlices; ++r) read_frag(stage(g + nks), h0, r);
        } else {
            wait_loads_barrier4(0);
        }
        // the stage of this tile's last step is free (the next tile's steps
        // 0 and 1 occupy the other two): the products meet there, 8 rows a
        // round, [2 products][4 blocks][8][64] doubles = 32 KB
        double *X = reinterpret_cast<double *>(stage(g + nks - 1));
        const int col = tn * kBN + wn * 32 + (lane & 31);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (pr > 0) {
#pragma unroll
                for (int jj = 0; jj < 8; ++jj) X[(((pr - 1) * 4 + blk) * 8 + jj) * 64 + lane] = P[8 * h + jj];
            }
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            if (pr == 0) {
#pragma unroll
                for (int jj = 0; jj < 8; ++jj) {
                    const int j = 8 * h + jj;
                    const int r = wm * 32 + 8 * (j >> 2) + 4 * (lane >> 5) + (j & 3);
                    const double P1 = X[((0 * 4 + blk) * 8 + jj) * 64 + lane];
                    const double P2 = X[((1 * 4 + blk) * 8 + jj) * 64 + lane];
                    const d2v bv = {P[j] - P1, P2 - P[j] - P1};
                    __builtin_nontemporal_store(bv,
                                                reinterpret_cast<d2v *>(&a.bmat[(size_t)(tm * kBM + r) * a.ldn + col]));
                }
            }
            // the round's values are read before the next round (or the
            // next tile's loads, and the scale buffer's refill) overwrite
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
    }
    // a last tile's loads for a next tile may still be in flight: they
    // write LDS, which must not be released before they land
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// one workgroup per CU, each walking its share of the tiles
__global__ __launch_bounds__(768, 1) void gpp_oz_gemm_kernel(GemmArgs a, int tiles)
{
    const int first = blockIdx.x, stride = gridDim.x;
    if (first >= tiles) return;
    oz_gemm12_tiles<true>(a, first, stride, (tiles - 1 - first) / stride + 1);
}

// ---------------------------------------------------------------------------
// Pole/SX epilogue over every (my_igp, ig): B from bmat, Bo = sum over the
// occupied bands in FP64, then the pole and SX factors in FP64 (pole_terms).
// A workgroup takes R rows my_igp and a run of their columns, one column of
// all R rows per thread and iteration: the R rows' loads are independent (R
// times the bytes in flight of a wave that takes one row), the occupied bands'
// aqsn values are loaded and widened once for R rows, and the rows'
// coefficients are uniform loads.  All W >= nw frequencies of a thread's
// elements are summed in registers, over the workgroup once at the end: one
// partial per workgroup and frequency, a fixed order.
//
// Measured: 512/2/32768/1638, 3 frequencies 367 us (4.7 TB/s; without the pole
// terms 300 us, 5.7 TB/s), the form of one row and two quotients 558; a batch of
// 12 problems of 3 to 11 frequencies 1.35 ms, before 2.65.  Two rows cost the
// same at 3 frequencies and 8% more at 7, loading one iteration ahead 5% more.
//
// W is the kernel's class, 4, 8, 12 or 16 frequencies (exact for a single call
// of up to 4): 8 W registers of sums decide how many waves fit, so a kernel
// for every nw would run all at the occupancy of 16.
// ---------------------------------------------------------------------------
constexpr int oz_class(int nw) { return (nw - 1) / 4; }
constexpr int pole_rows(int W) { return W <= 8 ? 4 : 2; }
// waves per SIMD that the kernels are held to: 128, 168 and 256 registers
constexpr int pole_waves(int W) { return W <= 4 ? 4 : W <= 8 ? 3 : 2; }

struct PoleArgs {
    const double2 *bmat;     // [ldm][ldn] B
    const double2 *c_occ;    // [nv][ldm]
    const float2 *aqsn, *I_eps, *wtilde;
    const int *igp;
    double2 *partials;       // [blocks][nw][2]
    double2 *achs_part;      // [blocks] static-CH remainder, or NULL
    int nv, C, G, ldm, ldn, chunks;
    PoleParams pp;
};

// Workgroups per group of rows: runs of at most 16 iterations of 256 columns,
// shorter where the rows alone give fewer than about 8 workgroups per CU (two to
// three rounds of what the kernels' registers let onto one: 3 or 4, 2 for the class
// of 16; sized without a device, so for the MI355X's 256 CUs).
inline int pole_chunks(int G, int C, int nw)
{
    const int iters = div_up(C, 256), groups = div_up(G, pole_rows(4 * oz_class(nw) + 4));
    return std::min(iters, std::max(div_up(iters, 16), div_up(2048, groups)));
}
inline int pole_blocks(int G, int C, int nw)
{
    return div_up(G, pole_rows(4 * oz_class(nw) + 4)) * pole_chunks(G, C, nw);
}

template <int W>
struct PoleLds {
    double buf[4][8 * 65];
    double red[4][4 * W + 2];
};

// tab: the wx and iwx2 tables of a.pp, read through scalar loads
typedef const __attribute__((address_space(4))) double cdbl;
static_assert(offsetof(PoleConst, iwx2) == sizeof(double) * kMaxFreq, "tab + kMaxFreq is iwx2");

template <int W, bool ALL, bool ACHS, bool MASK>
__device__ __forceinline__ void oz_pole_block(const PoleArgs &a, cdbl *tab, int b, PoleLds<W> &L)
{
    constexpr int R = pole_rows(W);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int mg = __builtin_amdgcn_readfirstlane(b / a.chunks);
    const int ch = __builtin_amdgcn_readfirstlane(b - mg * a.chunks);
    const int iters = (a.C + 255) / 256, m0 = mg * R;
    const int c_lo = 256 * (int)((int64_t)ch * iters / a.chunks);
    const int c_hi = min(256 * (int)((int64_t)(ch + 1) * iters / a.chunks), a.C);
    const bool want_ssx = a.nv > 0;
    // coefficients of the rows' occupied bands: uniform, read-only here (the
    // rows of c_occ are padded to ldm, a multiple of R)
    cdbl *occ = (cdbl *)(const double *)(a.c_occ + m0);
    bool ok[R];
    size_t row[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        row[r] = (size_t)min(m0 + r, a.G - 1);
        ok[r] = m0 + r < a.G && __builtin_amdgcn_readfirstlane(a.igp[row[r]]) >= 0;
    }
    double2 sach[W], sasx[W], sachs = make_double2(0.0, 0.0);
#pragma unroll
    for (int q = 0; q < W; ++q) { sach[q] = make_double2(0.0, 0.0); sasx[q] = make_double2(0.0, 0.0); }
    for (int ig = c_lo + tid; ig < c_hi; ig += 256) {
        double2 B[R], Bo[R];
        float2 wt[R], ie[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            B[r] = a.bmat[row[r] * a.ldn + ig];
            wt[r] = a.wtilde[row[r] * a.C + ig];
            ie[r] = a.I_eps[row[r] * a.C + ig];
            Bo[r] = make_double2(0.0, 0.0);
        }
        // unrolled for the latency of the coefficients' scalar loads (512/64/32768/1638
        // 2.68 ms, so 2.37; 1000/1000/200/200, 1 frequency, 331 us, so 162)
#pragma unroll 4
        for (int n1 = 0; n1 < a.nv; ++n1) {
            const double2 x = widen(a.aqsn[(size_t)n1 * a.C + ig]);
            cdbl *co = occ + (size_t)n1 * a.ldm * 2;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                Bo[r].x = __builtin_fma(co[2 * r], x.x, __builtin_fma(-co[2 * r + 1], x.y, Bo[r].x));
                Bo[r].y = __builtin_fma(co[2 * r], x.y, __builtin_fma(co[2 * r + 1], x.x, Bo[r].y));
            }
        }
        unsigned general = 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (!ok[r]) continue;
            // past four frequencies the tables are read again for each row:
            // kept in scalar registers all along they push others out of them
            // (nw 7: 119 to 150 us at 12000 x 600)
            if constexpr (W > 4) asm volatile("" : "+s"(tab));
            if (!pole_terms<W, ALL, MASK>(a.pp, tab, tab + kMaxFreq, 0, widen(wt[r]), widen(ie[r]), B[r], Bo[r], sach, sasx))
                general |= 1u << r;
            // static-CH remainder -sum B I_eps (gppkernel.deslippe.09.30.2014.f90:192-230)
            if constexpr (ACHS) sachs = csub(sachs, cmul(B[r], widen(ie[r])));
        }
        // the elements pole_terms left out (hardly ever any), one at a time
        if (__ballot(general != 0)) {
#pragma unroll 1
            for (int r = 0; r < R; ++r) {
                if (!((general >> r) & 1u)) continue;
                const size_t m = (size_t)(m0 + r);
                double2 o = make_double2(0.0, 0.0);
                for (int n1 = 0; n1 < a.nv; ++n1)
                    o = cfma(o, a.c_occ[(size_t)n1 * a.ldm + m], widen(a.aqsn[(size_t)n1 * a.C + ig]));
                pole_element<W>(a.pp, 0, true, widen(a.wtilde[m * a.C + ig]), widen(a.I_eps[m * a.C + ig]),
                                a.bmat[m * a.ldn + ig], o, want_ssx, sach, sasx);
            }
        }
    }
    // sums over the wave, two frequencies at a time, then over the waves
#pragma unroll
    for (int q = 0; q < W; q += 2) {
        constexpr int kNone = W - 1;
        const int q1 = q + 1 < W ? q + 1 : kNone;
        double v[8] = {sach[q].x, sach[q].y, sasx[q].x, sasx[q].y, sach[q1].x, sach[q1].y, sasx[q1].x, sasx[q1].y};
        if (!want_ssx) v[2] = v[3] = v[6] = v[7] = 0.0;
        const double x = wave_sums_lds(v, lane, L.buf[wave]);
        if (lane < (q + 1 < W ? 8 : 4)) L.red[wave][4 * q + lane] = x;
    }
    if constexpr (ACHS) {
        const double v0 = wave_sum(sachs.x), v1 = wave_sum(sachs.y);
        if (lane == 0) {
            L.red[wave][4 * W] = v0;
            L.red[wave][4 * W + 1] = v1;
        }
    }
    __syncthreads();
    const int nw = ALL ? W : a.pp.nw;
    if (tid < 4 * nw)
        reinterpret_cast<double *>(a.partials + (size_t)b * nw * 2)[tid] =
            ((L.red[0][tid] + L.red[1][tid]) + L.red[2][tid]) + L.red[3][tid];
    if (ACHS && tid >= 128 && tid < 130) {
        const int k = 4 * W + tid - 128;
        reinterpret_cast<double *>(a.achs_part + b)[tid - 128] = ((L.red[0][k] + L.red[1][k]) + L.red[2][k]) + L.red[3][k];
    }
}

template <int W, bool ALL, bool ACHS, bool MASK>
__global__ __launch_bounds__(256, pole_waves(W)) void gpp_oz_pole_kernel(PoleArgs a)
{
    __shared__ PoleLds<W> L;
    cdbl *args = (cdbl *)__builtin_amdgcn_kernarg_segment_ptr();   // a is the first argument
    oz_pole_block<W, ALL, ACHS, MASK>(a, args + (offsetof(PoleArgs, pp) + offsetof(PoleParams, pc)) / sizeof(double), blockIdx.x, L);
}

template <bool ACHS>
void launch_pole(int blocks, hipStream_t s, const PoleArgs &a)
{
    const dim3 grid(blocks), block(256);
    const int c = oz_class(a.pp.nw);
    if (!a.pp.mask_on) {
        switch (c) {
        case 0: hipLaunchKernelGGL((gpp_oz_pole_kernel<4, false, ACHS, false>), grid, block, 0, s, a); break;
        case 1: hipLaunchKernelGGL((gpp_oz_pole_kernel<8, false, ACHS, false>), grid, block, 0, s, a); break;
        case 2: hipLaunchKernelGGL((gpp_oz_pole_kernel<12, false, ACHS, false>), grid, block, 0, s, a); break;
        default: hipLaunchKernelGGL((gpp_oz_pole_kernel<16, false, ACHS, false>), grid, block, 0, s, a); break;
        }
        return;
    }
    switch (a.pp.nw) {
    case 1: hipLaunchKernelGGL((gpp_oz_pole_kernel<1, true, ACHS, true>), grid, block, 0, s, a); break;
    case 2: hipLaunchKernelGGL((gpp_oz_pole_kernel<2, true, ACHS, true>), grid, block, 0, s, a); break;
    case 3: hipLaunchKernelGGL((gpp_oz_pole_kernel<3, true, ACHS, true>), grid, block, 0, s, a); break;
    case 4: hipLaunchKernelGGL((gpp_oz_pole_kernel<4, true, ACHS, true>), grid, block, 0, s, a); break;
    default:
        switch (c) {
        case 1: hipLaunchKernelGGL((gpp_oz_pole_kernel<8, false, ACHS, true>), grid, block, 0, s, a); break;
        case 2: hipLaunchKernelGGL((gpp_oz_pole_kernel<12, false, ACHS, true>), grid, block, 0, s, a); break;
        default: hipLaunchKernelGGL((gpp_oz_pole_kernel<16, false, ACHS, true>), grid, block, 0, s, a); break;
        }
    }
}

// ---------------------------------------------------------------------------
// Batches: one launch of each kernel above for many problems.  Every
// problem has a record of its three kernels' arguments; block b of a batched
// prep or pole launch belongs to the problem p with first[p] <= b <
// first[p + 1] and runs that problem's block b - first[p].  The GEMM launch
// is persistent and walks the problems in turn; a problem's GEMM range
// starts at a multiple of the XCD count, so its tile order keeps its XCD
// locality.
// ---------------------------------------------------------------------------
struct OzRecord {
    PrepArgs pr;
    GemmArgs ga;
    PoleArgs pa;
    int gemm_tiles;          // tiles of the problem (its GEMM range may be longer)
};

// the problem whose range of a launch holds block b (first: n + 1 entries)
__device__ __forceinline__ int batch_problem(const int *first, int n, int b)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (first[mid] <= b) lo = mid;
        else hi = mid - 1;
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

__global__ __launch_bounds__(kPrepThreads, 4) void oz_prep_batch_kernel(const OzRecord *rec, const int *first, int n)
{
    const int b = (int)blockIdx.x, p = batch_problem(first, n, b);
    const PrepArgs pr = rec[p].pr;   // in registers: not reloaded after each barrier
    oz_prep_block(pr, b - first[p]);
}

// The GEMM of every problem, persistent: one workgroup per CU walks the
// problems in order and takes, of problem p, the tiles f, f + grid, ... with
// f = (w - first[p]) mod grid.  The rotation continues from problem to
// problem (first[p] is the problem's running tile offset, a multiple of the
// XCD count, so a tile runs on the XCD the single-problem kernel gives it),
// and within a problem the next tile's first steps load during the current
// tile's last two, as in gpp_oz_gemm_kernel.  Between problems a workgroup
// needs no barrier: each wave's LDS slots are its own and every wave drains
// its loads and passes the epilogue's last barrier before returning.
__global__ __launch_bounds__(768, 1) void gpp_oz_gemm_batch_kernel(const OzRecord *rec, const int *first, int n)
{
    const int w = (int)blockIdx.x, grid = (int)gridDim.x;
    for (int p = 0; p < n; ++p) {
        const int tiles = __builtin_amdgcn_readfirstlane(rec[p].gemm_tiles);
        const int f = (w - __builtin_amdgcn_readfirstlane(first[p]) % grid + grid) % grid;
        if (f >= tiles) continue;
        // a copy in registers: the tile's direct loads are asm statements that
        // clobber memory, after which fields read through rec would be reloaded
        const GemmArgs ga = rec[p].ga;
        oz_gemm12_tiles<true>(ga, f, grid, (tiles - 1 - f) / grid + 1);
    }
}

// The problems of one frequency class (first: no blocks for the others).  The
// arguments by reference: a register copy of them (with the pole parameters of
// up to 16 frequencies) made this kernel 1.7x slower.
template <int W, bool MASK>
__global__ __launch_bounds__(256, pole_waves(W)) void gpp_oz_pole_batch_kernel(const OzRecord *__restrict__ rec,
                                                                               const int *first, int n)
{
    __shared__ PoleLds<W> L;
    const int b = (int)blockIdx.x, p = batch_problem(first, n, b);
    oz_pole_block<W, false, false, MASK>(rec[p].pa, (cdbl *)&rec[p].pa.pp.pc, b - first[p], L);
}

// All classes in one launch, in the registers of the largest: for batches of few
// blocks, where the launches count.  A batch's run with one launch and with one per
// class, by blocks: 71 58 us and 73; 105 46 and 62; 464 58 and 78; 1196 87 and 92;
// 1946 115 and 119; 2933 166 and 159; 7417 320 and 285.
constexpr int kPoleSmallBatch = 2048;

template <bool MASK>
__global__ __launch_bounds__(256, pole_waves(16)) void gpp_oz_pole_small_batch_kernel(const OzRecord *__restrict__ rec,
                                                                                     const int *first, int n)
{
    __shared__ PoleLds<16> L;
    int b = (int)blockIdx.x, c = 0;
    while (b >= first[c * (n + 1) + n]) b -= first[c++ * (n + 1) + n];     // first[n]: the class's blocks
    c = __builtin_amdgcn_readfirstlane(c);
    first += c * (n + 1);
    const int p = batch_problem(first, n, b);
    cdbl *tab = (cdbl *)&rec[p].pa.pp.pc;
    const int k = b - first[p];
    if (c == 0) oz_pole_block<4, false, false, MASK>(rec[p].pa, tab, k, reinterpret_cast<PoleLds<4> &>(L));
    else if (c == 1) oz_pole_block<8, false, false, MASK>(rec[p].pa, tab, k, reinterpret_cast<PoleLds<8> &>(L));
    else if (c == 2) oz_pole_block<12, false, false, MASK>(rec[p].pa, tab, k, reinterpret_cast<PoleLds<12> &>(L));
    else oz_pole_block<16, false, false, MASK>(rec[p].pa, tab, k, L);
}

template <bool MASK>
void launch_pole_batch(int c, int blocks, hipStream_t s, const OzRecord *rec, const int *first, int n)
{
    const dim3 grid(blocks), block(256);
    switch (c) {
    case 0: hipLaunchKernelGGL((gpp_oz_pole_batch_kernel<4, MASK>), grid, block, 0, s, rec, first, n); break;
    case 1: hipLaunchKernelGGL((gpp_oz_pole_batch_kernel<8, MASK>), grid, block, 0, s, rec, first, n); break;
    case 2: hipLaunchKernelGGL((gpp_oz_pole_batch_kernel<12, MASK>), grid, block, 0, s, rec, first, n); break;
    default: hipLaunchKernelGGL((gpp_oz_pole_batch_kernel<16, MASK>), grid, block, 0, s, rec, first, n); break;
    }
}

}  // namespace

size_t gpp_oz_batch_record_bytes() { return sizeof(OzRecord); }

OzBlocks gpp_oz_batch_record(const fk_gpp_problem *p, const fk_options *o, const OzLayout &L, const Scratch &ws,
                             const int *d_igp, void *record)
{
    OzRecord r;
    PrepArgs &pr = r.pr;
    pr.aqsm = static_cast<const float2 *>(p->aqsmtemp); pr.aqsn = static_cast<const float2 *>(p->aqsntemp);
    pr.vcoul = p->vcoul; pr.igp = d_igp;
    pr.as = static_cast<int8_t *>(ws.at(L.off_as));
    pr.bs = static_cast<int8_t *>(ws.at(L.off_bs));
    pr.ra = static_cast<double *>(ws.at(L.off_ea));
    pr.rb = static_cast<double *>(ws.at(L.off_eb));
    pr.c_occ = static_cast<double2 *>(ws.at(L.off_cocc));
    pr.nb = p->number_bands; pr.nv = p->nvband; pr.C = p->ncouls; pr.G = p->ngpown;
    pr.ldm = L.ldm; pr.ldn = L.ldn; pr.nkb = L.Kb / kKStep; pr.blocks_a = L.ldm / kPrepRowsA;
    GemmArgs &ga = r.ga;
    ga.as = pr.as; ga.bs = pr.bs; ga.ra = pr.ra; ga.rb = pr.rb;
    ga.bmat = static_cast<double2 *>(ws.at(L.off_bmat));
    ga.ldm = L.ldm; ga.ldn = L.ldn; ga.nkb = pr.nkb;
    ga.tiles_m = L.tiles_m; ga.tiles_n = L.tiles_n; ga.group_m = kGroupM;
    PoleArgs &pa = r.pa;
    pa.bmat = ga.bmat; pa.c_occ = pr.c_occ; pa.aqsn = pr.aqsn;
    pa.I_eps = static_cast<const float2 *>(p->I_eps_array); pa.wtilde = static_cast<const float2 *>(p->wtilde_array);
    pa.igp = d_igp;
    pa.partials = static_cast<double2 *>(ws.at(L.off_part));
    pa.achs_part = nullptr;
    pa.nv = p->nvband; pa.C = p->ncouls; pa.G = p->ngpown; pa.ldm = L.ldm; pa.ldn = L.ldn;
    pa.chunks = pole_chunks(p->ngpown, p->ncouls, p->nfreq);
    pa.pp = make_pole_params(p->wx, p->nfreq, p->limittwo, p->limitone, p->to1, o->mask != 0);
    r.gemm_tiles = L.tiles_m * L.tiles_n;
    std::memcpy(record, &r, sizeof(r));
    OzBlocks nb;
    const bool any = p->number_bands > 0;
    nb.prep = any ? L.ldm / kPrepRowsA + L.ldn / kPrepColsB : 0;
    nb.gemm = any ? div_up(r.gemm_tiles, kXcds) * kXcds : 0;
    nb.pole = any ? pole_blocks(p->ngpown, p->ncouls, p->nfreq) : 0;
    nb.pole_class = oz_class(p->nfreq);
    return nb;
}

int gpp_oz_batch_launch(const void *records, const int *first_prep, const int *first_gemm, const int *first_pole,
                        int n, int total_prep, int total_gemm, const int *total_pole, bool mask, hipStream_t s)
{
    const OzRecord *rec = static_cast<const OzRecord *>(records);
    if (total_prep > 0)
        hipLaunchKernelGGL(oz_prep_batch_kernel, dim3(total_prep), dim3(kPrepThreads), 0, s, rec, first_prep, n);
    if (total_gemm > 0) {
        int dev = 0, ncu = 0;
        FK_HIP(hipGetDevice(&dev));
        FK_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
        const int grid = std::max(1, std::min(total_gemm, ncu));
        hipLaunchKernelGGL(gpp_oz_gemm_batch_kernel, dim3(grid), dim3(kWaves12 * 64), 0, s, rec, first_gemm, n);
    }
    int pole = 0, classes = 0;
    for (int c = 0; c < kOzPoleClasses; ++c) {
        pole += total_pole[c];
        classes += total_pole[c] > 0;
    }
    if (classes > 1 && pole <= kPoleSmallBatch) {
        const dim3 grid(pole), block(256);
        if (mask) hipLaunchKernelGGL(gpp_oz_pole_small_batch_kernel<true>, grid, block, 0, s, rec, first_pole, n);
        else hipLaunchKernelGGL(gpp_oz_pole_small_batch_kernel<false>, grid, block, 0, s, rec, first_pole, n);
        FK_HIP(hipGetLastError());
        return FK_OK;
    }
    for (int c = 0; c < kOzPoleClasses; ++c) {
        if (total_pole[c] <= 0) continue;
        const int *first = first_pole + c * (n + 1);
        if (mask) launch_pole_batch<true>(c, total_pole[c], s, rec, first, n);
        else launch_pole_batch<false>(c, total_pole[c], s, rec, first, n);
    }
    FK_HIP(hipGetLastError());
    return FK_OK;
}

void gpp_oz_plan(const fk_gpp_problem *p, Scratch &ws, OzLayout &L)
{
    const int nb = std::max(p->number_bands, 1);
    L.ldm = div_up(p->ngpown, kBM) * kBM;
    L.ldn = div_up(p->ncouls, kBN) * kBN;
    L.Kb = div_up(nb, 2 * kKStep) * 2 * kKStep;   // an even number of GEMM steps
    L.tiles_m = L.ldm / kBM;
    L.tiles_n = L.ldn / kBN;
    L.off_as = ws.plan((size_t)kPlanes * L.ldm * L.Kb);
    L.off_bs = ws.plan((size_t)kPlanes * L.ldn * L.Kb);
    L.off_ea = ws.plan(sizeof(double) * kProds * (size_t)L.ldm);
    L.off_eb = ws.plan(sizeof(double) * kProds * (size_t)L.ldn);
    L.off_cocc = ws.plan(sizeof(double2) * (size_t)std::max(p->nvband, 1) * L.ldm);
    L.off_bmat = ws.plan(sizeof(double2) * (size_t)L.ldm * L.ldn);
    const size_t blocks = (size_t)pole_blocks(p->ngpown, p->ncouls, p->nfreq);
    L.off_part = ws.plan(sizeof(double2) * 2 * (size_t)p->nfreq * blocks);
    L.off_achs = ws.plan(sizeof(double2) * blocks);
}

int gpp_oz_check(const fk_gpp_problem *p)
{
    if (p->number_bands > kMaxBandsOz) {
        set_error("gpp_kernel: the mixed-precision path takes at most %d bands (got %d)", kMaxBandsOz,
                  p->number_bands);
        return FK_ERR_UNSUPPORTED;
    }
    return FK_OK;
}

int gpp_oz_launch(const fk_gpp_problem *p, const fk_options *o, const OzLayout &L, Scratch &ws, const int *d_igp,
                  const float2 *aqsm, const float2 *aqsn, const float2 *ieps, const float2 *wt, const double *vcoul,
                  double2 *d_ach, double2 *d_asx, double2 *d_achs, hipStream_t s)
{
    const int nkb = L.Kb / kKStep;
    PrepArgs pr;
    pr.aqsm = aqsm; pr.aqsn = aqsn; pr.vcoul = vcoul; pr.igp = d_igp;
    pr.as = static_cast<int8_t *>(ws.at(L.off_as));
    pr.bs = static_cast<int8_t *>(ws.at(L.off_bs));
    pr.ra = static_cast<double *>(ws.at(L.off_ea));
    pr.rb = static_cast<double *>(ws.at(L.off_eb));
    pr.c_occ = static_cast<double2 *>(ws.at(L.off_cocc));
    pr.nb = p->number_bands; pr.nv = p->nvband; pr.C = p->ncouls; pr.G = p->ngpown;
    pr.ldm = L.ldm; pr.ldn = L.ldn; pr.nkb = nkb; pr.blocks_a = L.ldm / kPrepRowsA;
    hipLaunchKernelGGL(oz_prep_kernel, dim3(L.ldm / kPrepRowsA + L.ldn / kPrepColsB), dim3(kPrepThreads), 0, s, pr);
    FK_HIP(hipGetLastError());

    GemmArgs ga;
    ga.as = pr.as; ga.bs = pr.bs; ga.ra = pr.ra; ga.rb = pr.rb;
    ga.bmat = static_cast<double2 *>(ws.at(L.off_bmat));
    ga.ldm = L.ldm; ga.ldn = L.ldn; ga.nkb = nkb;
    ga.tiles_m = L.tiles_m; ga.tiles_n = L.tiles_n; ga.group_m = kGroupM;
    const int tiles = L.tiles_m * L.tiles_n;
    KernelTimer timer(o->kernel_ms, s);
    FK_TRY(timer.start());
    int dev = 0, ncu = 0;
    FK_HIP(hipGetDevice(&dev));
    FK_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    hipLaunchKernelGGL(gpp_oz_gemm_kernel, dim3(std::min(tiles, std::max(ncu, 1))), dim3(kWaves12 * 64), 0, s, ga,
                       tiles);
    FK_HIP(hipGetLastError());
    FK_TRY(timer.stop());

    PoleArgs pa;
    pa.bmat = ga.bmat; pa.c_occ = pr.c_occ; pa.aqsn = aqsn; pa.I_eps = ieps; pa.wtilde = wt; pa.igp = d_igp;
    pa.partials = static_cast<double2 *>(ws.at(L.off_part));
    pa.achs_part = d_achs ? static_cast<double2 *>(ws.at(L.off_achs)) : nullptr;
    pa.nv = p->nvband; pa.C = p->ncouls; pa.G = p->ngpown; pa.ldm = L.ldm; pa.ldn = L.ldn;
    pa.chunks = pole_chunks(p->ngpown, p->ncouls, p->nfreq);
    pa.pp = make_pole_params(p->wx, p->nfreq, p->limittwo, p->limitone, p->to1, o->mask != 0);
    const int blocks = pole_blocks(p->ngpown, p->ncouls, p->nfreq);
    if (pa.achs_part) launch_pole<true>(blocks, s, pa);
    else launch_pole<false>(blocks, s, pa);
    FK_HIP(hipGetLastError());
    FK_TRY(gpp_reduce_launch(pa.partials, blocks, p->nfreq, 2.0 * p->occ, d_ach, d_asx, s));
    if (d_achs) FK_TRY(gpp_sum_launch(pa.achs_part, blocks, d_achs, s));
    return timer.finish();
}

}  // namespace fk
