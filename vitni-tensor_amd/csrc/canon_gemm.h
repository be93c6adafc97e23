// canon_gemm.h -- shared pieces of the batched pinned dot (canon_gemm.hip,
// canon_gemm_split.hip).
//
// Same contract as canon_gemv.hip (src/ops/quant.rs:429-448, :482-566): per
// output and chunk of 8192 inputs, chain j sums the products x_i * w_i with
// i % 8 == j from +0.0 in increasing i, each product rounded before its add;
// fixed_tree combines the 8 chains, then the chunks.
//
// A GEMV per batch row decodes and multiplies every weight again for every
// row (Q8_0 4096 x 4096 at 128 tokens: 556 us).  Here a wave owns 16 weight
// rows x 16*NT tokens and decodes a weight once, and the products come from
// v_mfma_f32_16x16x1_4b_f32: with K = 1 and a zero C operand each of its
// 4 x 16 x 16 results is one product, rounded once (checked bit for bit
// against the host's product over 25 M pairs, subnormal results and inputs
// included; the sign of a zero product cannot show, because a chain starts at
// +0.0 and no sum of it is ever -0.0).  It hands every operand to 16 others
// without moving it, at the price of a vector multiply: 16 MFMAs take 218 ns
// of a SIMD, and the 256 adds of their results 236 ns, one after the other
// (f32 MFMA and f32 vector work share the pipe; a multiply and an add per
// product on the vector unit alone take 550 ns).  Those 454 ns bound a step:
// 58 us for the shape above, which takes 103 us (decoding 60 ns a step, the
// rest waits of two waves a SIMD for issue, barriers and loads).
//
// Work split.  A step is 64 consecutive inputs, in four parts of 16.  Lane
// 16g + r holds inputs 4g .. 4g+3 of each part for row r (A) and for token r
// (B).  MFMA (part, c) multiplies input 4g + c of the part for every group g:
// its blocks 0 and 1 are the next products of chains c and 4 + c, blocks 2
// and 3 the ones after them.
//
// The activations go through LDS, loaded in contiguous rows and shared by the
// workgroup's waves: in the operand order every lane is at another row, and
// the vector memory path takes such a load lane by lane (84 cache accesses a
// load by counter).  With every wave loading its own operands a wave step took
// 850 ns whatever it computed.
#pragma once

#include "vtq_device.h"
#include "vtq_kernels.h"

namespace vtq {
namespace gm {

constexpr int kChunk = 8192;
constexpr int kStep = kGmStep;
constexpr int kMaxLevels = 3;                // at most 8 chunks (in_feat <= 65536)
constexpr int kWord3 = 0x00020000;           // raw buffer descriptor word 3, gfx9 family
constexpr uint32_t kOutOfRange = 0x80000000u;

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));  // y promises no more than 4 bytes

// Operands in flight are held as whole vector values: split into words, the
// words' copies would wait for a load right where it is issued.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u32x4 load16(__amdgpu_buffer_rsrc_t rs, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff, soff, 0));
}
__device__ __forceinline__ u32x2 load8(__amdgpu_buffer_rsrc_t rs, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, voff, soff, 0));
}
// no load moves across (the wait counts of the loops rest on their order)
__device__ __forceinline__ void fence() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
// clamp to 0 .. m as a scalar (the compiler's clamp is a vector instruction,
// and a descriptor it touches costs a loop at every load)
__device__ __forceinline__ int left(int v, int m) { return __builtin_amdgcn_readfirstlane(max(0, min(m, v))); }

// The row group and the token group of this workgroup.  Workgroup i runs on
// XCD i % 8: the token groups of one row group take consecutive slots of one
// XCD, so its L2 holds the rows between them.
__device__ __forceinline__ void groups(int NR, int TP, int* rg, int* tp) {
    const int id = blockIdx.x, full = (NR / 8) * 8 * TP;
    if (id < full) {
        const int k = id >> 3;
        *rg = (k / TP) * 8 + (id & 7);
        *tp = k % TP;
    } else {
        *rg = (NR / 8) * 8 + (id - full) / TP;
        *tp = (id - full) % TP;
    }
}

// One step's products and adds for C4 values of c and NT token tiles: acc[tile]
// [chains c, 4 + c][c][row of the lane's four].  MFMA u + 1 is issued before
// MFMA u's results are added.
template <int C4, int NT, class X>
__device__ __forceinline__ void mul_add(float (&acc)[NT][2][C4][4], const float (&wv)[4][C4], const X (&xv)[NT][4]) {
    constexpr int U = 4 * C4 * NT;
    v16f d[2];
    auto mul = [&](int u) __attribute__((always_inline)) {
        const int t = u % NT, k = u / NT % C4, p = u / (NT * C4);
        d[u & 1] = __builtin_amdgcn_mfma_f32_16x16x1f32(wv[p][k], xv[t][p][k], v16f{}, 0, 0, 0);
    };
    mul(0);
#pragma unroll
    for (int u = 0; u < U; u++) {
        if (u + 1 < U) mul(u + 1);
        __builtin_amdgcn_sched_barrier(0);
        const int t = u % NT, k = u / NT % C4;
#pragma unroll
        for (int b = 0; b < 4; b++)
#pragma unroll
            for (int i = 0; i < 4; i++) acc[t][b & 1][k][i] = acc[t][b & 1][k][i] + d[u & 1][4 * b + i];
        // the adds stay in their unit (left alone, several steps' adds gather
        // at the loop's end, with every product kept until then)
        float(&a)[4] = acc[t][0][k], (&b)[4] = acc[t][1][k];
        asm volatile("" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]));
        __builtin_amdgcn_sched_barrier(0);
    }
}

// The first two levels of fixed_tree over the 8 chains, within c = 0..C4-1:
// h[tile][0] from chains c, h[tile][1] from chains 4 + c.
template <int C4, int NT>
__device__ __forceinline__ void chain_tree(const float (&acc)[NT][2][C4][4], float (&h)[NT][2][4]) {
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int e = 0; e < 2; e++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float q[C4];
#pragma unroll
                for (int k = 0; k < C4; k++) q[k] = acc[t][e][k][i];
#pragma unroll
                for (int st = 1; st < C4; st <<= 1)
#pragma unroll
                    for (int k = 0; k < C4; k += 2 * st) q[k] = q[k] + q[k + st];
                h[t][e][i] = q[0];
            }
}

// fixed_tree over the chunks, as a binary counter: after chunk c the levels
// below L = (trailing ones of c) merge into level L, the stored group on the
// left; at the last chunk the open groups fold right to left into v.
template <int NT>
__device__ __forceinline__ void chunk_tree(float (&stk)[kMaxLevels][NT][4], float (&v)[NT][4], int c, int nchunks) {
    const int L = __builtin_ctz(~(unsigned)c);
    auto merge = [&](int l) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) v[t][i] = stk[l][t][i] + v[t][i];
    };
#pragma unroll
    for (int l = 0; l < kMaxLevels; l++)
        if (l < L) merge(l);
#pragma unroll
    for (int l = 0; l < kMaxLevels; l++) {
        if (c + 1 == nchunks) {
            if (l > L && ((nchunks >> l) & 1)) merge(l);
        } else if (l == L) {
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int i = 0; i < 4; i++) stk[l][t][i] = v[t][i];
        }
    }
}

// Element i of a lane is row o + i, token tok.
__device__ __forceinline__ void store(float* y, const float (&v)[4], int tok, int o, int batch, int out_feat) {
    if (tok >= batch) return;
    float* yp = y + (size_t)tok * out_feat + o;
    if ((out_feat & 3) == 0 && o + 3 < out_feat) {
        *reinterpret_cast<f32x4_a4*>(yp) = f32x4_a4{v[0], v[1], v[2], v[3]};
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (o + i < out_feat) yp[i] = v[i];
    }
}

}  // namespace gm
}  // namespace vtq
