// canon_gemm.hip -- the pinned 8-lane fp32 dot over a batch of activation rows
// (see canon_gemm.h): the kernel of large grids, and the launcher of the batch
// kernels (their choice: vtq_rules.h).
//
// A wave owns all eight chains of its 16 rows and gathers its own weights, the
// activations pass through LDS a step at a time.
#include "canon_gemm.h"

namespace vtq {

using namespace gm;

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// the upper 32 lanes of a change places with the lower 32 of b
__device__ __forceinline__ void swap32(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0], b = r[1];
}
// in each half of the wave, the upper 16 lanes of a with the lower 16 of b
__device__ __forceinline__ void swap16(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0], b = r[1];
}

// Each format: Raw holds a lane's bytes of one step; ready() turns them into
// the weights w[part][k] of inputs 4g + k of the four parts.  off: byte offset of
// the lane's row (out of range: everything reads as zero, and so do the
// weights); half: the step's second 32 inputs are past the row's end.

// d * code for the four signed bytes of q
__device__ __forceinline__ void scale_s8(float (&w)[4], uint32_t q, float d) {
#pragma unroll
    for (int k = 0; k < 4; k++) w[k] = d * (float)(int8_t)(uint8_t)(q >> (8 * k));
}

struct WideQ8_0 {  // src/ops/quant.rs:193-210
    static constexpr bool kFine = false;
    struct Raw {
        u32x4 q;
        uint32_t d;
    };
    // the lane loads the 16 codes of half g%2 of block g/2, and the scale of
    // that block; 4 x 4 words change places between the groups in ready()
    __device__ static void load(Raw& r, __amdgpu_buffer_rsrc_t rs, uint32_t off, int s, int g, bool half) {
        const uint32_t o = (half && g >= 2) ? kOutOfRange : off + 34u * (g >> 1), so = 68u * (uint32_t)s;
        r.q = load16(rs, o + 2 + 16 * (g & 1), so);
        r.d = __builtin_amdgcn_raw_buffer_load_b16(rs, o, so, 0);
    }
    __device__ static void ready(float (&w)[4][4], const Raw& r, int, int) {
        uint32_t q[4] = {r.q.x, r.q.y, r.q.z, r.q.w};
        swap32(q[0], q[2]);
        swap32(q[1], q[3]);
        swap16(q[0], q[1]);
        swap16(q[2], q[3]);
        uint32_t da = r.d, db = r.d;
        swap32(da, db);
        const float d0 = f16_hw(da), d1 = f16_hw(db);
#pragma unroll
        for (int p = 0; p < 4; p++) scale_s8(w[p], q[p], p < 2 ? d0 : d1);
    }
};

struct WideQ5_0 {  // src/ops/quant.rs:160-186: elements 0..15 in the low halves, 16..31 in the high halves
    static constexpr bool kFine = false;
    struct Raw {
        u32x2 h[2];  // d, qh of each block
        uint32_t q[2];
    };
    __device__ static void load(Raw& r, __amdgpu_buffer_rsrc_t rs, uint32_t off, int s, int g, bool half) {
        const uint32_t so = 44u * (uint32_t)s;
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const uint32_t o = (b && half) ? kOutOfRange : off + 22u * b;
            r.h[b] = load8(rs, o, so);
            r.q[b] = __builtin_amdgcn_raw_buffer_load_b32(rs, o + 6 + 4 * g, so, 0);
        }
    }
    __device__ static void ready(float (&w)[4][4], const Raw& r, int, int g) {
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const float d = f16_hw(r.h[b].x & 0xFFFFu);
            const uint32_t qh = __builtin_amdgcn_alignbyte(r.h[b].y, r.h[b].x, 2) >> (4 * g);
#pragma unroll
            for (int e = 0; e < 2; e++) {
                // four high bits to bit 4 of the four bytes, then code - 16 as a signed byte
                const uint32_t hi = ((((qh >> (16 * e)) & 15u) * 0x00204081u) & 0x01010101u) << 4;
                const uint32_t u = ((r.q[b] >> (4 * e)) & 0x0F0F0F0Fu) | hi;
                scale_s8(w[2 * b + e], (u + 0x70707070u) ^ 0x80808080u, d);
            }
        }
    }
};

struct WideQ4_0 {  // src/ops/quant.rs:91-111: element 2k low half of byte k, 2k + 1 high half
    static constexpr bool kFine = false;
    struct Raw {
        u32x4 q[2];  // both blocks' codes
        uint32_t d[2];
    };
    __device__ static void load(Raw& r, __amdgpu_buffer_rsrc_t rs, uint32_t off, int s, int, bool half) {
        const uint32_t so = 36u * (uint32_t)s;
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const uint32_t o = (b && half) ? kOutOfRange : off + 18u * b;
            r.q[b] = load16(rs, o + 2, so);
            r.d[b] = __builtin_amdgcn_raw_buffer_load_b16(rs, o, so, 0);
        }
    }
    __device__ static void ready(float (&w)[4][4], const Raw& r, int, int g) {
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
            scale_s8(w[p], (u + 0x78787878u) ^ 0x80808080u, f16_hw(r.d[p >> 1]));
        }
    }
};

struct WideQ4KFloat {  // src/ops/quant.rs:649-667: w = d1*q - m1f per sub-block of 32
    static constexpr bool kFine = false;
    struct Raw {
        u32x4 h;
        uint32_t q[2];
    };
    // step s is sub-blocks 2(s%4) and 2(s%4)+1 of super-block s/4, in the low
    // and the high halves of 32 bytes
    __device__ static void load(Raw& r, __amdgpu_buffer_rsrc_t rs, uint32_t off, int s, int g, bool) {
        const uint32_t blk = 144u * (uint32_t)(s >> 2), qs = blk + 32u * (uint32_t)(s & 3);
        r.h = load16(rs, off, blk);
#pragma unroll
        for (int e = 0; e < 2; e++) r.q[e] = __builtin_amdgcn_raw_buffer_load_b32(rs, off + 16 + 16 * e + 4 * g, qs, 0);
    }
    __device__ static void ready(float (&w)[4][4], const Raw& r, int s, int) {
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
                const uint32_t q = (r.q[e] >> (4 * b)) & 0x0F0F0F0Fu;
#pragma unroll
                for (int k = 0; k < 4; k++)
                    w[2 * b + e][k] = __builtin_fmaf(d1, (float)((q >> (8 * k)) & 0xFFu), nm);
            }
        }
    }
};

// A lane's floats of each part of a step
__device__ __forceinline__ void load_floats(f32x4 (&o)[4], __amdgpu_buffer_rsrc_t rs, uint32_t off, uint32_t so) {
#pragma unroll
    for (int p = 0; p < 4; p++) o[p] = __builtin_bit_cast(f32x4, load16(rs, off + 64 * p, so));
}

struct WideF32 {  // src/model/forward_quantized.rs:674-697; any row length
    static constexpr bool kFine = true;
    struct Raw {
        f32x4 w[4];
    };
    __device__ static void load(Raw& r, __amdgpu_buffer_rsrc_t rs, uint32_t off, int s, int g, bool) {
        load_floats(r.w, rs, off + 16u * g, 256u * (uint32_t)s);
    }
    __device__ static void ready(float (&w)[4][4], const Raw& r, int, int) {
#pragma unroll
        for (int p = 0; p < 4; p++)
#pragma unroll
            for (int k = 0; k < 4; k++) w[p][k] = r.w[p][k];
    }
};

// Four row tiles of 16 rows a workgroup, one a wave, by NT token tiles of 16.
// PD: ring slots of operands (PD - 1 steps in flight during a step).
template <class Fmt, int NT, int PD>
__global__ __launch_bounds__(256, 2) void canon_gemm_wide_kernel(const float* x, const uint8_t* W, size_t row_bytes,
                                                                 float* y, int n, int out_feat, int batch, int NR, int TP) {
    static_assert((kChunk / kStep) % PD == 0 && PD % 2 == 0, "ring slots and LDS buffers restart at 0 in every chunk");
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, r = lane & 15;
    int rg, tp;
    groups(NR, TP, &rg, &tp);
    const int row0 = (rg * 4 + wave_id()) * 16;
    const int rows = left(out_feat - row0, 16);  // 0: nothing to store, every weight reads as zero
    // 16 rows are a multiple of 16 bytes in every format, so the base keeps W's alignment
    const __amdgpu_buffer_rsrc_t rsw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(W + (rows ? (size_t)row0 * row_bytes : 0)), (short)0, (int)(row_bytes * (size_t)rows), kWord3);
    __amdgpu_buffer_rsrc_t rsx[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const int t0 = (tp * NT + t) * 16, nt = left(batch - t0, 16);
        rsx[t] = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x + (nt ? (size_t)t0 * n : 0)), (short)0,
                                                   (int)(4u * (uint32_t)nt * (uint32_t)n), kWord3);
    }
    const uint32_t wbase = r < rows ? (uint32_t)r * (uint32_t)row_bytes : kOutOfRange;

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
    constexpr int kWhole = Fmt::kFine ? kStep : 1;  // inputs a step of the loop must have
    auto load_w = [&](int slot, int s) __attribute__((always_inline)) {
        Fmt::load(raw[slot], rsw, kStep * s + kWhole <= n ? wbase : kOutOfRange, s, g, kStep * s + 32 >= n);
    };
    auto load_x = [&](int slot, int s) __attribute__((always_inline)) {
        const uint32_t o = kStep * s + (Fmt::kFine ? kStep - 1 : 4 * sq) < n ? sbase : kOutOfRange;
#pragma unroll
        for (int t = 0; t < NT; t++) xr[slot][t] = load16(rsx[t], o, 256u * (uint32_t)s);
    };
    auto stage_x = [&](int slot, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < NT; t++) xs[buf][t][sslot] = xr[slot][t];
    };
    auto read_x = [&](f32x4 (&xv)[NT][4], int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < 4; p++)
#pragma unroll
            for (int t = 0; t < NT; t++)
                xv[t][p] = __builtin_bit_cast(f32x4, xs[buf][t][16 * r + ((4 * p + g) ^ r)]);
    };

    const int nchunks = (n + kChunk - 1) / kChunk;
    float acc[NT][2][4][4];         // [tile][chains c, 4 + c][c][row of the lane's four]
    float stk[kMaxLevels][NT][4];  // completed chunk groups of fixed_tree (a binary counter)
#pragma unroll
    for (int l = 0; l < kMaxLevels; l++)
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) stk[l][t][i] = 0.0f;
    float v[NT][4];

    // Step s (ring slot s % PD, LDS buffer s % 2) computes from the buffer the
    // barrier before it completed and stages step s + 1 into the other.
    auto step = [&](int slot, int s) __attribute__((always_inline)) {
        float wv[4][4];
        f32x4 xv[NT][4];
        read_x(xv, slot & 1);
        Fmt::ready(wv, raw[slot], s, g);
        fence();
        load_w(slot, s + PD);
        stage_x((slot + 1) % PD, (slot & 1) ^ 1);
        fence();
        load_x((slot + 1) % PD, s + 1 + PD);
        fence();
        mul_add<4>(acc, wv, xv);
        __syncthreads();
    };

#pragma unroll
    for (int i = 0; i < PD; i++) {
        // the loop's load order, so that its wait counts hold from the first step
        if (i > 0) load_w(i - 1, i - 1);
        fence();
        load_x(i, i);
        fence();
    }
    load_w(PD - 1, PD - 1);
    fence();
    stage_x(0, 0);
    fence();
    load_x(0, PD);
    fence();
    __syncthreads();
    for (int c = 0; c < nchunks; c++) {
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int k = 0; k < 4; k++)
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[t][h][k][i] = 0.0f;
        const int s1 = min((c + 1) * (kChunk / kStep), (n + kStep - kWhole) / kStep);
        for (int s = c * (kChunk / kStep); s < s1; s += PD) {
#pragma unroll
            for (int i = 0; i < PD; i++) step(i, s + i);
        }
        if (Fmt::kFine && c + 1 == nchunks && n % kStep) {
            // the rest of an f32 row: what lies past its end belongs to the next row
            const int s = n / kStep;
            typename Fmt::Raw rt;
            f32x4 xt[NT][4];
            float wv[4][4];
            Fmt::load(rt, rsw, wbase, s, g, false);
#pragma unroll
            for (int t = 0; t < NT; t++) xs[0][t][sslot] = load16(rsx[t], sbase, 256u * (uint32_t)s);
            __syncthreads();
            read_x(xt, 0);
            Fmt::ready(wv, rt, s, g);
#pragma unroll
            for (int p = 0; p < 4; p++)
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const bool in = kStep * s + 16 * p + 4 * g + k < n;
                    wv[p][k] = in ? wv[p][k] : 0.0f;
#pragma unroll
                    for (int t = 0; t < NT; t++) xt[t][p][k] = in ? xt[t][p][k] : 0.0f;
                }
            mul_add<4>(acc, wv, xt);
        }
        // fixed_tree over the 8 chains: ((0+1)+(2+3)) + ((4+5)+(6+7))
        float h[NT][2][4];
        chain_tree(acc, h);
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) v[t][i] = h[t][0][i] + h[t][1][i];
        chunk_tree(stk, v, c, nchunks);
    }
#pragma unroll
    for (int t = 0; t < NT; t++) store(y, v[t], (tp * NT + t) * 16 + r, row0 + 4 * g, batch, out_feat);
}

template <class Fmt>
hipError_t launch_wide(int nt, const float* x, const uint8_t* w, size_t row_bytes, float* y, int batch, int n, int out_feat,
                       hipStream_t stream) {
    const int NR = (out_feat + 63) / 64, TP = (batch + 16 * nt - 1) / (16 * nt);
    const dim3 grid((unsigned)NR * (unsigned)TP);
    if (nt == 2)
        hipLaunchKernelGGL((canon_gemm_wide_kernel<Fmt, 2, 2>), grid, dim3(256), 0, stream, x, w, row_bytes, y, n, out_feat,
                           batch, NR, TP);
    else
        hipLaunchKernelGGL((canon_gemm_wide_kernel<Fmt, 1, 2>), grid, dim3(256), 0, stream, x, w, row_bytes, y, n, out_feat,
                           batch, NR, TP);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_canon_gemm(CanonFormat fmt, const float* x, const uint8_t* w, size_t row_bytes, float* y, int batch,
                             int in_feat, int out_feat, hipStream_t stream) {
    if (in_feat <= 0 || in_feat > canon_max_in_feat()) return hipErrorInvalidValue;
    long ns;
    const GmForm& f = kGmForms[gm_pick(fmt, batch, in_feat, out_feat, &ns)];
    if (f.cs > 1) return launch_canon_gemm_split(fmt, f.cs, x, w, row_bytes, y, batch, in_feat, out_feat, stream);
    switch (fmt) {
    case kCanonQ8_0: return launch_wide<WideQ8_0>(f.nt, x, w, row_bytes, y, batch, in_feat, out_feat, stream);
    case kCanonQ5_0: return launch_wide<WideQ5_0>(f.nt, x, w, row_bytes, y, batch, in_feat, out_feat, stream);
    case kCanonQ4_0: return launch_wide<WideQ4_0>(f.nt, x, w, row_bytes, y, batch, in_feat, out_feat, stream);
    case kCanonF32: return launch_wide<WideF32>(f.nt, x, w, row_bytes, y, batch, in_feat, out_feat, stream);
    case kCanonQ4KFloat: return launch_wide<WideQ4KFloat>(f.nt, x, w, row_bytes, y, batch, in_feat, out_feat, stream);
    }
    return hipErrorInvalidValue;
}

}  // namespace vtq
