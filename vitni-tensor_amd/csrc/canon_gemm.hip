// canon_gemm.hip -- the pinned 8-lane fp32 dot over a batch of activation rows.
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
// and 3 the ones after them.  CS waves share a tile by c (chains c and 4 + c
// for 4/CS values of c each), which fills the chip when the tiles alone do
// not; their sums meet in LDS once per chunk.
//
// The activations of a step go through LDS, loaded in rows of 256 contiguous
// bytes and shared by the workgroup's waves: in the operand order every lane
// is at another row, and the vector memory path takes such a load lane by
// lane (84 cache accesses a load by counter).  With every wave loading its
// own operands a wave step took 850 ns whatever its share of the chains: 58 /
// 55 us instead of 65 / 31 for 4096 x 4096 at 16 tokens (CS 1 / 4), 112 / 420
// instead of 103 / 213 at 128.
#include "vtq_device.h"
#include "vtq_kernels.h"

namespace vtq {

namespace {

constexpr int kGmChunk = 8192;
constexpr int kGmStep = 64;
constexpr int kGmMaxLevels = 3;               // at most 8 chunks (in_feat <= 65536)
constexpr int kGmWord3 = 0x00020000;          // raw buffer descriptor word 3, gfx9 family
constexpr uint32_t kGmOutOfRange = 0x80000000u;

// no load moves across (the wait counts of the loop rest on their order)
__device__ __forceinline__ void gm_fence() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
// the upper 32 lanes of a change places with the lower 32 of b
__device__ __forceinline__ void gm_swap32(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0], b = r[1];
}
// in each half of the wave, the upper 16 lanes of a with the lower 16 of b
__device__ __forceinline__ void gm_swap16(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0], b = r[1];
}

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));  // y promises no more than 4 bytes

// Operands in flight are held as whole vector values: split into words, the
// words' copies would wait for a load right where it is issued.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u32x4 gm_load16(__amdgpu_buffer_rsrc_t rs, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff, soff, 0));
}
__device__ __forceinline__ u32x2 gm_load8(__amdgpu_buffer_rsrc_t rs, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, voff, soff, 0));
}

// Each format, for a wave that owns c = cw*C4 .. cw*C4 + C4-1 (C4 = 4/CS): Raw
// holds a lane's bytes of one step; ready() turns them into the weights
// w[part][k] of inputs 4g + cw*C4 + k of the four parts.  off: byte offset of
// the lane's row (out of range: everything reads as zero, and so do the
// weights); half: the step's second 32 inputs are past the row's end.

// d * code for the wave's codes among the four signed bytes of q
template <int CS>
__device__ __forceinline__ void gm_scale_s8(float (&w)[4 / CS], uint32_t q, float d, int cw) {
    if (CS > 1) q >>= 32 / CS * cw;
#pragma unroll
    for (int k = 0; k < 4 / CS; k++) w[k] = d * (float)(int8_t)(uint8_t)(q >> (8 * k));
}

template <int CS>
struct GmQ8_0 {  // src/ops/quant.rs:193-210
    static constexpr bool kFine = false;
    struct Raw {
        u32x4 q;
        uint32_t d;
    };
    // the lane loads the 16 codes of half g%2 of block g/2, and the scale of
    // that block; 4 x 4 words change places between the groups in ready()
    __device__ static void load(Raw& r, __amdgpu_buffer_rsrc_t rs, uint32_t off, int s, int g, int, bool half) {
        const uint32_t o = (half && g >= 2) ? kGmOutOfRange : off + 34u * (g >> 1), so = 68u * (uint32_t)s;
        r.q = gm_load16(rs, o + 2 + 16 * (g & 1), so);
        r.d = __builtin_amdgcn_raw_buffer_load_b16(rs, o, so, 0);
    }
    __device__ static void ready(float (&w)[4][4 / CS], const Raw& r, int, int, int cw) {
        uint32_t q[4] = {r.q.x, r.q.y, r.q.z, r.q.w};
        gm_swap32(q[0], q[2]);
        gm_swap32(q[1], q[3]);
        gm_swap16(q[0], q[1]);
        gm_swap16(q[2], q[3]);
        uint32_t da = r.d, db = r.d;
        gm_swap32(da, db);
        const float d0 = f16_hw(da), d1 = f16_hw(db);
#pragma unroll
        for (int p = 0; p < 4; p++) gm_scale_s8<CS>(w[p], q[p], p < 2 ? d0 : d1, cw);
    }
};

template <int CS>
struct GmQ5_0 {  // src/ops/quant.rs:160-186: elements 0..15 in the low halves, 16..31 in the high halves
    static constexpr bool kFine = false;
    struct Raw {
        u32x2 h[2];  // d, qh of each block
        uint32_t q[2];
    };
    __device__ static void load(Raw& r, __amdgpu_buffer_rsrc_t rs, uint32_t off, int s, int g, int, bool half) {
        const uint32_t so = 44u * (uint32_t)s;
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const uint32_t o = (b && half) ? kGmOutOfRange : off + 22u * b;
            r.h[b] = gm_load8(rs, o, so);
            r.q[b] = __builtin_amdgcn_raw_buffer_load_b32(rs, o + 6 + 4 * g, so, 0);
        }
    }
    __device__ static void ready(float (&w)[4][4 / CS], const Raw& r, int, int g, int cw) {
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const float d = f16_hw(r.h[b].x & 0xFFFFu);
            const uint32_t qh = __builtin_amdgcn_alignbyte(r.h[b].y, r.h[b].x, 2) >> (4 * g);
#pragma unroll
            for (int e = 0; e < 2; e++) {
                // four high bits to bit 4 of the four bytes, then code - 16 as a signed byte
                const uint32_t hi = ((((qh >> (16 * e)) & 15u) * 0x00204081u) & 0x01010101u) << 4;
                const uint32_t u = ((r.q[b] >> (4 * e)) & 0x0F0F0F0Fu) | hi;
                gm_scale_s8<CS>(w[2 * b + e], (u + 0x70707070u) ^ 0x80808080u, d, cw);
            }
        }
    }
};

template <int CS>
struct GmQ4_0 {  // src/ops/quant.rs:91-111: element 2k low half of byte k, 2k + 1 high half
    static constexpr bool kFine = false;
    struct Raw {
        u32x4 q[2];  // both blocks' codes
        uint32_t d[2];
    };
    __device__ static void load(Raw& r, __amdgpu_buffer_rsrc_t rs, uint32_t off, int s, int, int, bool half) {
        const uint32_t so = 36u * (uint32_t)s;
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const uint32_t o = (b && half) ? kGmOutOfRange : off + 18u * b;
            r.q[b] = gm_load16(rs, o + 2, so);
            r.d[b] = __builtin_amdgcn_raw_buffer_load_b16(rs, o, so, 0);
        }
    }
    __device__ static void ready(float (&w)[4][4 / CS], const Raw& r, int, int g, int cw) {
        // bytes 2g, 2g+1 of a part's eight: elements 4g .. 4g+3 as nibbles
        const int sh = 16 * (g & 1);
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const u32x4 q = r.q[p >> 1];
            const uint32_t a = (p & 1) ? q.z : q.x, b = (p & 1) ? q.w : q.y;
            const uint32_t n = (g >= 2 ? b : a) >> sh;
            // nibbles 0, 1, 2, 3 to bytes, then code - 8 as a signed byte
            const uint32_t lo = n & 0x0F0Fu, hi = (n >> 4) & 0x0F0Fu;
            const uint32_t u = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
            gm_scale_s8<CS>(w[p], (u + 0x78787878u) ^ 0x80808080u, f16_hw(r.d[p >> 1]), cw);
        }
    }
};

template <int CS>
struct GmQ4KFloat {  // src/ops/quant.rs:649-667: w = d1*q - m1f per sub-block of 32
    static constexpr bool kFine = false;
    struct Raw {
        u32x4 h;
        uint32_t q[2];
    };
    // step s is sub-blocks 2(s%4) and 2(s%4)+1 of super-block s/4, in the low
    // and the high halves of 32 bytes
    __device__ static void load(Raw& r, __amdgpu_buffer_rsrc_t rs, uint32_t off, int s, int g, int, bool) {
        const uint32_t blk = 144u * (uint32_t)(s >> 2), qs = blk + 32u * (uint32_t)(s & 3);
        r.h = gm_load16(rs, off, blk);
#pragma unroll
        for (int e = 0; e < 2; e++) r.q[e] = __builtin_amdgcn_raw_buffer_load_b32(rs, off + 16 + 16 * e + 4 * g, qs, 0);
    }
    __device__ static void ready(float (&w)[4][4 / CS], const Raw& r, int s, int, int cw) {
        const float d = f16_hw(r.h.x & 0xFFFFu), dmin = f16_hw(r.h.x >> 16);
        const uint32_t up = (s & 2) ? ~0u : 0u;  // sub-blocks 4..7 take the split encoding
#pragma unroll
        for (int b = 0; b < 2; b++) {
            // get_scale_min_k4 (src/ops/quant.rs:267-276) of sub-block 2(s%4) + b
            const int sh = 16 * (s & 1) + 8 * b;
            const uint32_t A = r.h.w >> sh, B = r.h.y >> sh, C = r.h.z >> sh;
            const uint32_t sc = (((A & 15u) | ((B >> 2) & 0x30u)) & up) | (B & 63u & ~up);
            const uint32_t mn = ((((A >> 4) & 15u) | ((C >> 2) & 0x30u)) & up) | (C & 63u & ~up);
            const float d1 = d * (float)sc, nm = -(dmin * (float)mn);
            // d1*q is exact (an f16 times 6 and 4 bits), so the fused form
            // rounds exactly where the reference's subtraction does
#pragma unroll
            for (int e = 0; e < 2; e++) {
                uint32_t q = (r.q[e] >> (4 * b)) & 0x0F0F0F0Fu;
                if (CS > 1) q >>= 32 / CS * cw;
#pragma unroll
                for (int k = 0; k < 4 / CS; k++)
                    w[2 * b + e][k] = __builtin_fmaf(d1, (float)((q >> (8 * k)) & 0xFFu), nm);
            }
        }
    }
};

// 4/CS floats as one value
template <int CS>
struct GmFloats {
    typedef float T __attribute__((ext_vector_type(4 / CS)));
};
// A lane's floats of each part of a step
template <int CS>
__device__ __forceinline__ void gm_load_floats(typename GmFloats<CS>::T (&o)[4], __amdgpu_buffer_rsrc_t rs, uint32_t off,
                                               uint32_t off2, uint32_t so) {
    using T = typename GmFloats<CS>::T;
#pragma unroll
    for (int p = 0; p < 4; p++) {
        const uint32_t a = (p < 2 ? off : off2) + 64 * p;
        if constexpr (CS == 4)
            o[p] = __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(rs, a, so, 0));
        else if constexpr (CS == 2)
            o[p] = __builtin_bit_cast(T, gm_load8(rs, a, so));
        else
            o[p] = __builtin_bit_cast(T, gm_load16(rs, a, so));
    }
}

template <int CS>
struct GmF32 {  // src/model/forward_quantized.rs:674-697; any row length
    static constexpr bool kFine = true;
    struct Raw {
        typename GmFloats<CS>::T w[4];
    };
    __device__ static void load(Raw& r, __amdgpu_buffer_rsrc_t rs, uint32_t off, int s, int g, int cw, bool) {
        const uint32_t o = off + 16u * g + 16u / CS * cw;
        gm_load_floats<CS>(r.w, rs, o, o, 256u * (uint32_t)s);
    }
    __device__ static void ready(float (&w)[4][4 / CS], const Raw& r, int, int, int) {
#pragma unroll
        for (int p = 0; p < 4; p++)
#pragma unroll
            for (int k = 0; k < 4 / CS; k++) w[p][k] = r.w[p][k];
    }
};

// One 16 x 16*NT tile by CS waves; 4/CS row tiles to a workgroup.  PD: ring
// slots of operands (PD - 1 steps in flight during a step).
template <template <int> class FmtT, int NT, int CS, int PD>
__global__ __launch_bounds__(256, 2) void canon_gemm_kernel(const float* x, const uint8_t* W,
                                                            size_t row_bytes, float* y, int n,
                                                            int out_feat, int batch, int NR, int TP) {
    using Fmt = FmtT<CS>;
    constexpr int C4 = 4 / CS;
    constexpr int RW = 4 / CS;      // row tiles of a workgroup
    constexpr int U = 4 * C4 * NT;  // MFMAs of a step
    static_assert((kGmChunk / kGmStep) % PD == 0 && PD % 2 == 0, "ring slots and LDS buffers restart at 0 in every chunk");
    const int lane = threadIdx.x & 63, wave = wave_id();
    const int g = lane >> 4, r = lane & 15;
    const int cw = wave % CS, rw = wave / CS;
    // Workgroup i runs on XCD i % 8: the token groups of one row group take
    // consecutive slots of one XCD, so its L2 holds the rows between them.
    const int id = blockIdx.x, full = (NR / 8) * 8 * TP;
    int rg, tp;
    if (id < full) {
        const int k = id >> 3;
        rg = (k / TP) * 8 + (id & 7);
        tp = k % TP;
    } else {
        rg = (NR / 8) * 8 + (id - full) / TP;
        tp = (id - full) % TP;
    }
    const int row0 = (rg * RW + rw) * 16;
    // clamp to 0 .. 16 as a scalar (the compiler's clamp is a vector
    // instruction, and a descriptor it touches costs a loop at every load)
    auto left = [](int m) { return __builtin_amdgcn_readfirstlane(max(0, min(16, m))); };
    const int rows = left(out_feat - row0);  // 0: nothing to store, every weight reads as zero
    // 16 rows are a multiple of 16 bytes in every format, so the base keeps W's alignment
    const __amdgpu_buffer_rsrc_t rsw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(W + (rows ? (size_t)row0 * row_bytes : 0)), (short)0, (int)(row_bytes * (size_t)rows),
        kGmWord3);
    __amdgpu_buffer_rsrc_t rsx[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const int t0 = (tp * NT + t) * 16, nt = left(batch - t0);
        rsx[t] = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x + (nt ? (size_t)t0 * n : 0)), (short)0,
                                                   (int)(4u * (uint32_t)nt * (uint32_t)n), kGmWord3);
    }
    const uint32_t wbase = r < rows ? (uint32_t)r * (uint32_t)row_bytes : kGmOutOfRange;

    // Staging: thread 16a + q loads the 16 bytes of chunk q (inputs 4q .. 4q+3
    // of the step) of token a of each tile; in LDS token a's chunk q lies at
    // slot q ^ a, so neither the writes nor the operand reads (8 lanes at 8
    // tokens, one chunk) meet in a bank.
    __shared__ u32x4 xs[2][NT][256];
    const int sa = (int)threadIdx.x >> 4, sq = (int)threadIdx.x & 15;
    const uint32_t sbase = 4u * ((uint32_t)sa * (uint32_t)n + 4u * (uint32_t)sq);
    const int sslot = 16 * sa + (sq ^ sa);

    typename Fmt::Raw raw[PD];
    u32x4 xr[PD][NT];
    // Steps past the row's end read as zero (products +-0, which change no
    // chain), so the loop has no branch around a load and the compiler's wait
    // counts stay exact; so does the second half of the last step where the
    // row length is an odd multiple of 32 (block formats).  An f32 row's last
    // step, of any length, is taken after the loop.
    constexpr int kWhole = Fmt::kFine ? kGmStep : 1;  // inputs a step of the loop must have
    auto load_w = [&](int slot, int s) __attribute__((always_inline)) {
        Fmt::load(raw[slot], rsw, kGmStep * s + kWhole <= n ? wbase : kGmOutOfRange, s, g, cw, kGmStep * s + 32 >= n);
    };
    auto load_x = [&](int slot, int s) __attribute__((always_inline)) {
        const uint32_t o = kGmStep * s + (Fmt::kFine ? kGmStep - 1 : 4 * sq) < n ? sbase : kGmOutOfRange;
#pragma unroll
        for (int t = 0; t < NT; t++) xr[slot][t] = gm_load16(rsx[t], o, 256u * (uint32_t)s);
    };
    auto stage_x = [&](int slot, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < NT; t++) xs[buf][t][sslot] = xr[slot][t];
    };
    auto read_x = [&](typename GmFloats<CS>::T (&xv)[NT][4], int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < 4; p++)
#pragma unroll
            for (int t = 0; t < NT; t++)
                xv[t][p] = reinterpret_cast<const typename GmFloats<CS>::T*>(&xs[buf][t][16 * r + ((4 * p + g) ^ r)])[cw];
    };

    const int nchunks = (n + kGmChunk - 1) / kGmChunk;
    float acc[NT][2][C4][4];         // [tile][chains c, 4 + c][c][row of the lane's four]
    float stk[kGmMaxLevels][NT][4];  // completed chunk groups of fixed_tree (a binary counter)
#pragma unroll
    for (int l = 0; l < kGmMaxLevels; l++)
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) stk[l][t][i] = 0.0f;
    float res[NT][4];
    __shared__ float4 part[CS > 1 ? 4 * NT * 2 * 64 : 1];

    // one step's products and adds: MFMA u + 1 is issued before MFMA u's results are added
    auto mul_add = [&](const float (&wv)[4][C4], const typename GmFloats<CS>::T (&xv)[NT][4]) __attribute__((always_inline)) {
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
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // Step s (ring slot s % PD, LDS buffer s % 2) computes from the buffer the
    // barrier before it completed and stages step s + 1 into the other.
    auto step = [&](int slot, int s) __attribute__((always_inline)) {
        float wv[4][C4];
        typename GmFloats<CS>::T xv[NT][4];
        read_x(xv, slot & 1);
        Fmt::ready(wv, raw[slot], s, g, cw);
        gm_fence();
        load_w(slot, s + PD);
        stage_x((slot + 1) % PD, (slot & 1) ^ 1);
        gm_fence();
        load_x((slot + 1) % PD, s + 1 + PD);
        gm_fence();
        mul_add(wv, xv);
        __syncthreads();
    };

#pragma unroll
    for (int i = 0; i < PD; i++) {
        // the loop's load order, so that its wait counts hold from the first step
        if (i > 0) load_w(i - 1, i - 1);
        gm_fence();
        load_x(i, i);
        gm_fence();
    }
    load_w(PD - 1, PD - 1);
    gm_fence();
    stage_x(0, 0);
    gm_fence();
    load_x(0, PD);
    gm_fence();
    __syncthreads();
    for (int c = 0; c < nchunks; c++) {
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int k = 0; k < C4; k++)
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[t][h][k][i] = 0.0f;
        const int s1 = min((c + 1) * (kGmChunk / kGmStep), (n + kGmStep - kWhole) / kGmStep);
        for (int s = c * (kGmChunk / kGmStep); s < s1; s += PD) {
#pragma unroll
            for (int i = 0; i < PD; i++) step(i, s + i);
        }
        if (Fmt::kFine && c + 1 == nchunks && n % kGmStep) {
            // the rest of an f32 row: what lies past its end belongs to the next row
            const int s = n / kGmStep;
            typename Fmt::Raw rt;
            typename GmFloats<CS>::T xt[NT][4];
            float wv[4][C4];
            Fmt::load(rt, rsw, wbase, s, g, cw, false);
#pragma unroll
            for (int t = 0; t < NT; t++) xs[0][t][sslot] = gm_load16(rsx[t], sbase, 256u * (uint32_t)s);
            __syncthreads();
            read_x(xt, 0);
            Fmt::ready(wv, rt, s, g, cw);
#pragma unroll
            for (int p = 0; p < 4; p++)
#pragma unroll
                for (int k = 0; k < C4; k++) {
                    const bool in = kGmStep * s + 16 * p + 4 * g + cw * C4 + k < n;
                    wv[p][k] = in ? wv[p][k] : 0.0f;
#pragma unroll
                    for (int t = 0; t < NT; t++) xt[t][p][k] = in ? xt[t][p][k] : 0.0f;
                }
            mul_add(wv, xt);
        }
        // fixed_tree over the 8 chains: ((0+1)+(2+3)) + ((4+5)+(6+7))
        float hv[NT][2][4], v[NT][4];
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    float q[C4];
#pragma unroll
                    for (int k = 0; k < C4; k++) q[k] = acc[t][h][k][i];
#pragma unroll
                    for (int st = 1; st < C4; st <<= 1)
#pragma unroll
                        for (int k = 0; k < C4; k += 2 * st) q[k] = q[k] + q[k + st];
                    hv[t][h][i] = q[0];
                }
        if constexpr (CS > 1) {
            if (c) __syncthreads();  // the previous chunk's parts have been read
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int h = 0; h < 2; h++)
                    part[((wave * NT + t) * 2 + h) * 64 + lane] =
                        make_float4(hv[t][h][0], hv[t][h][1], hv[t][h][2], hv[t][h][3]);
            __syncthreads();
            if (cw == 0) {
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        float4 p[CS];
#pragma unroll
                        for (int q = 0; q < CS; q++) p[q] = part[(((wave + q) * NT + t) * 2 + h) * 64 + lane];
#pragma unroll
                        for (int st = 1; st < CS; st <<= 1)
#pragma unroll
                            for (int q = 0; q < CS; q += 2 * st)
                                p[q] = make_float4(p[q].x + p[q + st].x, p[q].y + p[q + st].y, p[q].z + p[q + st].z,
                                                   p[q].w + p[q + st].w);
                        hv[t][h][0] = p[0].x, hv[t][h][1] = p[0].y, hv[t][h][2] = p[0].z, hv[t][h][3] = p[0].w;
                    }
            }
        }
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) v[t][i] = hv[t][0][i] + hv[t][1][i];
        // fixed_tree over the chunks: after chunk c the levels below L =
        // (trailing ones of c) merge into level L, the stored group on the left;
        // at the last chunk the open groups fold right to left
        const int L = __builtin_ctz(~(unsigned)c);
        const bool end = c + 1 == nchunks;
#pragma unroll
        for (int l = 0; l < kGmMaxLevels; l++)
            if (l < L)
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int i = 0; i < 4; i++) v[t][i] = stk[l][t][i] + v[t][i];
        if (!end) {
#pragma unroll
            for (int l = 0; l < kGmMaxLevels; l++)
                if (l == L)
#pragma unroll
                    for (int t = 0; t < NT; t++)
#pragma unroll
                        for (int i = 0; i < 4; i++) stk[l][t][i] = v[t][i];
        } else {
#pragma unroll
            for (int l = 0; l < kGmMaxLevels; l++)
                if (l > L && ((nchunks >> l) & 1))
#pragma unroll
                    for (int t = 0; t < NT; t++)
#pragma unroll
                        for (int i = 0; i < 4; i++) v[t][i] = stk[l][t][i] + v[t][i];
        }
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) res[t][i] = v[t][i];
    }
    if (cw != 0) return;
    // element i of a lane is row 4*(lane/16) + i, token lane%16
    const int o = row0 + 4 * g;
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const int tok = (tp * NT + t) * 16 + r;
        if (tok >= batch) continue;
        float* yp = y + (size_t)tok * out_feat + o;
        if ((out_feat & 3) == 0 && o + 3 < out_feat) {
            *reinterpret_cast<f32x4_a4*>(yp) = f32x4_a4{res[t][0], res[t][1], res[t][2], res[t][3]};
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (o + i < out_feat) yp[i] = res[t][i];
        }
    }
}

template <template <int> class FmtT, int NT, int CS, int PD>
hipError_t launch_gm(const float* x, const uint8_t* w, size_t row_bytes, float* y, int batch, int n, int out_feat,
                     hipStream_t stream) {
    const int NR = (out_feat + 16 * (4 / CS) - 1) / (16 * (4 / CS)), TP = (batch + 16 * NT - 1) / (16 * NT);
    hipLaunchKernelGGL((canon_gemm_kernel<FmtT, NT, CS, PD>), dim3((unsigned)NR * (unsigned)TP), dim3(256), 0, stream, x,
                       w, row_bytes, y, n, out_feat, batch, NR, TP);
    return hipGetLastError();
}

// The kernel's forms and the time of one in nanoseconds, as measured over 21
// shapes (2 to 512 tokens, 256 to 11008 inputs, 64 to 32000 rows): what
// counts is the steps of a row and how many waves each of the 1024 SIMDs gets
// in turn.  A lone wave waits for its own loads and barriers, so its step
// costs more than a shared SIMD's.  (Q8_0 4096 x 4096, us: 16 tokens 65 / 42 /
// 31 with CS = 1 / 2 / 4; 32 tokens 65 / 44 / 58; 128 tokens 103 / 117 / 213,
// 115 with NT = 2; 2048 x 2048 at 512 tokens 98 with NT = 1, 94 with NT = 2.)
struct GmForm {
    int nt, cs;
    long lone, pair, more;  // ns a step: one wave per SIMD, two, each of more
};
constexpr GmForm kGmForms[] = {{1, 4, 490, 910, 455}, {1, 2, 685, 1062, 465}, {1, 1, 1000, 1600, 800},
                               {2, 1, 1780, 2950, 1475}};

int gm_pick(int batch, int n, int out_feat, long* ns) {
    const long steps = (n + kGmStep - 1) / kGmStep;
    int best = 0;
    *ns = 0;
    for (int f = 0; f < 4; f++) {
        const GmForm& k = kGmForms[f];
        const long tiles = (long)((out_feat + 15) / 16) * ((batch + 16 * k.nt - 1) / (16 * k.nt));
        const long waves = (tiles * k.cs + 1023) / 1024;
        const long t = steps * (waves == 1 ? k.lone : waves == 2 ? k.pair : k.more * waves) + 3000;
        if (f == 0 || t < *ns) best = f, *ns = t;
    }
    return best;
}

template <template <int> class FmtT>
hipError_t launch_gm_fmt(const float* x, const uint8_t* w, size_t row_bytes, float* y, int batch, int n, int out_feat,
                         hipStream_t stream) {
    long ns;
    switch (gm_pick(batch, n, out_feat, &ns)) {
    case 0: return launch_gm<FmtT, 1, 4, 4>(x, w, row_bytes, y, batch, n, out_feat, stream);
    case 1: return launch_gm<FmtT, 1, 2, 2>(x, w, row_bytes, y, batch, n, out_feat, stream);
    case 2: return launch_gm<FmtT, 1, 1, 2>(x, w, row_bytes, y, batch, n, out_feat, stream);
    default: return launch_gm<FmtT, 2, 1, 2>(x, w, row_bytes, y, batch, n, out_feat, stream);
    }
}

}  // namespace

// Whether the batch kernel is faster than one GEMV slice per batch row, whose
// time is its weights decoded per nanosecond (measured with the shapes above:
// Q8_0 3600 in the LDS-resident kernel, 2000 in the windowed one; Q4_K float
// 2300, Q4_0 2000, Q5_0 1200, F32 1000).  With those the line for Q8_0 4096 x 4096
// lies between 4 tokens (22 us against 31) and 8 (40 against 31).
bool canon_gemm_faster(CanonFormat fmt, int batch, int in_feat, int out_feat) {
    if (batch < 2 || in_feat > canon_max_in_feat()) return false;
    const double rate = fmt == kCanonQ8_0 ? (in_feat % 256 == 0 && in_feat <= 4096 ? 3600 : 2000)
                        : fmt == kCanonQ4KFloat ? 2300 : fmt == kCanonQ4_0 ? 2000 : fmt == kCanonQ5_0 ? 1200 : 1000;
    long ns;
    gm_pick(batch, in_feat, out_feat, &ns);
    return (double)batch * in_feat * out_feat / rate * 0.9 > (double)ns;
}

hipError_t launch_canon_gemm(CanonFormat fmt, const float* x, const uint8_t* w, size_t row_bytes, float* y, int batch,
                             int in_feat, int out_feat, hipStream_t stream) {
    if (in_feat <= 0 || in_feat > canon_max_in_feat()) return hipErrorInvalidValue;
    switch (fmt) {
    case kCanonQ8_0: return launch_gm_fmt<GmQ8_0>(x, w, row_bytes, y, batch, in_feat, out_feat, stream);
    case kCanonQ5_0: return launch_gm_fmt<GmQ5_0>(x, w, row_bytes, y, batch, in_feat, out_feat, stream);
    case kCanonQ4_0: return launch_gm_fmt<GmQ4_0>(x, w, row_bytes, y, batch, in_feat, out_feat, stream);
    case kCanonF32: return launch_gm_fmt<GmF32>(x, w, row_bytes, y, batch, in_feat, out_feat, stream);
    case kCanonQ4KFloat: return launch_gm_fmt<GmQ4KFloat>(x, w, row_bytes, y, batch, in_feat, out_feat, stream);
    }
    return hipErrorInvalidValue;
}

}  // namespace vtq
