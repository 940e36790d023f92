// fk_mfma_ring.h -- the FP64 MFMA main loop shared by the GPP and FF GEMMs:
// operands staged through an LDS ring by direct global->LDS loads, the
// complex product as three or four real MFMA products.
//
// Why LDS and not fragments loaded straight into registers (the form before):
// a CU's eight waves then issue four 1 KB fragment loads per 12 MFMAs, each
// operand fragment twice, and the vector memory path, not the MFMA pipes, set
// the pace: 70-72% of the cycles busy at any ring depth (3 to 8 k-steps),
// row stride or register budget, against 97% with the loads taken out.  Through
// LDS every operand element crosses the vector memory path once per workgroup,
// in full 128-byte lines, and the fragments come back as conflict-free
// ds_read_b128.  FF contraction 256/4096/4096/16: 7.6 ms (54 TFLOP/s of
// executed flops) to 6.3 ms (65); at 256/4096/4096/32 its MFMA pipes are
// busy 88% of the cycles, at 2.34 GHz, without a bank conflict.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace fk {
namespace ring {

typedef double d4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ d4 mfma(double a, double b, d4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
// -a * b + c (the neg modifier on A, the blgp field of the builtin)
__device__ __forceinline__ d4 mfma_nega(double a, double b, d4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 1);
}

// One direct global->LDS load, 16 bytes per lane: lane l's bytes land at LDS
// byte address lds + 16 l (lds wave-uniform).  As inline asm, because the
// compiler cannot tell which LDS a direct load writes and would put a
// vmcnt(0) wait in front of every LDS read; the callers order loads and reads
// with wait_barrier.  No register outputs.
__device__ __forceinline__ void lds_load16(const void *g, const void *lds)
{
    const unsigned la = (unsigned)__builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)lds);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(la) : "memory", "m0");
}

// Whether p may be the source of direct loads (16-byte aligned).
inline int aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// The element at g where g need not be 16-byte aligned (an array of complex
// numbers is aligned to its 8-byte parts only, and a workspace may start
// anywhere): such sources are staged by way of registers, stored to LDS when the
// direct load would be issued.
__device__ __forceinline__ double2 load16(const double2 *g)
{
    const __attribute__((address_space(1))) double *p = (const __attribute__((address_space(1))) double *)g;
    return make_double2(p[0], p[1]);
}

// Wait until at most N of this wave's loads are in flight and its LDS reads
// are done, then meet the other waves of the workgroup.
template <int N>
__device__ __forceinline__ void wait_barrier()
{
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// Operand fragments of one k-step (4 k) of a wave's (16 MB) x (16 NB) tile:
// lane l holds A[l % 16][l / 16] and B[l / 16][l % 16] of each 16-row and
// 16-column block.
template <int MB, int NB>
struct Frags {
    double2 a[MB], b[NB];
};

// The complex product as three real GEMMs (the 3M method; Higham, SIAM J.
// Matrix Anal. Appl. 13(3), 1992):
//   T1 = (ar + ai) br,  T2 = ar (bi - br),  T3 = ai (br + bi),
//   re = T1 - T3,       im = T1 + T2,
// 12 MFMAs per k-step of a 2 x 2 wave tile where four real products take 16.
// Accumulator register r of lane l is row 4 r + l / 16, column l % 16.
template <int MB, int NB>
struct Acc3 {
    d4 t1[MB][NB], t2[MB][NB], t3[MB][NB];

    __device__ __forceinline__ void zero()
    {
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) t1[i][j] = t2[i][j] = t3[i][j] = d4{0, 0, 0, 0};
    }
    __device__ __forceinline__ void mma(const Frags<MB, NB> &f)
    {
        double as[MB], bd[NB], bs[NB];
#pragma unroll
        for (int i = 0; i < MB; ++i) as[i] = f.a[i].x + f.a[i].y;
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            bd[j] = f.b[j].y - f.b[j].x;
            bs[j] = f.b[j].x + f.b[j].y;
        }
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                t1[i][j] = mfma(as[i], f.b[j].x, t1[i][j]);
                t2[i][j] = mfma(f.a[i].x, bd[j], t2[i][j]);
                t3[i][j] = mfma(f.a[i].y, bs[j], t3[i][j]);
            }
    }
    __device__ __forceinline__ double2 value(int i, int j, int r) const
    {
        return make_double2(t1[i][j][r] - t3[i][j][r], t1[i][j][r] + t2[i][j][r]);
    }
};

// The complex product as four real ones: a third more MFMAs, but the error of
// each part stays relative to that part's own products, while the 3M form adds
// errors of the size of |re| to im.  With operands whose imaginary parts are
// 1e-8 of the real ones, sums of 32 and 256 products: im good to 3e-16 and
// 8e-16 of itself, 3M 2e-8 and 5e-8.
template <int MB, int NB>
struct Acc4 {
    d4 re[MB][NB], im[MB][NB];

    __device__ __forceinline__ void zero()
    {
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) re[i][j] = im[i][j] = d4{0, 0, 0, 0};
    }
    __device__ __forceinline__ void mma(const Frags<MB, NB> &f)
    {
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                re[i][j] = mfma(f.a[i].x, f.b[j].x, re[i][j]);
                im[i][j] = mfma(f.a[i].x, f.b[j].y, im[i][j]);
            }
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                re[i][j] = mfma_nega(f.a[i].y, f.b[j].y, re[i][j]);
                im[i][j] = mfma(f.a[i].y, f.b[j].x, im[i][j]);
            }
    }
    __device__ __forceinline__ double2 value(int i, int j, int r) const { return make_double2(re[i][j][r], im[i][j][r]); }
};

// The main loop: nst stages of 8 k (two k-steps) through a ring of NS LDS
// slots.  issue(stage, slot) starts this wave's LPW direct loads of a stage;
// read(frags, stage, slot, q) reads its fragments of k-step q.  Stage s+NS-1
// is issued at the start of stage s, into the slot stage s-1 used: every wave
// has read that slot before the barrier that opens stage s (wait_barrier
// waits for the LDS reads too).  The loads complete in issue order, so waiting
// for all but the newest (NS-2) LPW means stage s+1 has landed; near the
// end, where fewer are in flight, everything is waited for.  On return no
// load is in flight and every wave may still be reading the last slot: meet a
// barrier before the ring is used for something else.
template <int MB, int NB, int NS, int LPW, class Acc, class Issue, class Read>
__device__ __forceinline__ void main_loop(int nst, Acc &acc, Issue issue, Read read)
{
    auto arrived = [&](int s) {
        if (s + NS - 2 < nst) wait_barrier<LPW *(NS - 2)>();
        else wait_barrier<0>();
    };
#pragma unroll
    for (int s = 0; s < NS - 1; ++s)
        if (s < nst) issue(s, s);
    arrived(0);
    Frags<MB, NB> f0, f1;
    read(f0, 0, 0, 0);
    int slot = 0, fill = NS - 1;
    for (int s = 0; s < nst; ++s) {
        if (s + NS - 1 < nst) issue(s + NS - 1, fill);
        fill = fill + 1 == NS ? 0 : fill + 1;
        read(f1, s, slot, 1);
        acc.mma(f0);
        slot = slot + 1 == NS ? 0 : slot + 1;
        if (s + 1 < nst) {
            arrived(s + 1);
            read(f0, s + 1, slot, 0);
        }
        acc.mma(f1);
    }
}

}  // namespace ring
}  // namespace fk
