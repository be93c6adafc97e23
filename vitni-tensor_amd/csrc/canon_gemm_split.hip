// canon_gemm_split.hip -- the pinned 8-lane fp32 dot over a batch of activation
// rows (see canon_gemm.h): the kernel of small grids.
//
// Where the 16 x 16 tiles alone would leave SIMDs idle, CS waves share a tile by
// c (chains c and 4 + c for 4/CS values of c each); their sums meet in LDS once
// per chunk.  A wave's step is then short, so what it waits for counts: both
// operands pass through LDS in windows of four steps, loaded in contiguous
// rows a window ahead, with one barrier a window, and a step's LDS reads are
// issued before the adds of the step before it.  Q8_0 4096 x 4096 at 16 tokens
// (CS = 4): 30.9 us with a barrier a step and the weights gathered by every
// wave, 30.7 with the weights through LDS, 25.4 with the window's one barrier;
// at 32 tokens 44 / 39 / 35.  What is left is the decoding beside 64 adds a step
// (100 vector instructions) on the one wave that each SIMD has.
#include "canon_gemm.h"

namespace vtq {

using namespace gm;

namespace {

typedef uint32_t u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));

// Block formats.  A window is four steps (256 inputs, kRow bytes of a row, a
// multiple of 16) and lies in LDS, rows kRow bytes apart (for every format the
// 16 rows' words of one lane group fall on 16 different quads of banks).
// fetch() reads what the lane needs of step si of its row's window, and
// ready() makes of it the weights w[part][k] of inputs 4g + cw*C4 + k of the
// four parts, for a wave that owns c = cw*C4 .. cw*C4 + C4-1 (C4 = 4/CS, CS 2
// or 4); m0, m1: all ones, or zero where the step's first or second 32 inputs
// are past the row's end (whatever lies there, their scales and so their
// weights are zero).

// d * code for the wave's codes among the four signed bytes of q
template <int CS>
__device__ __forceinline__ void scale_s8(float (&w)[4 / CS], uint32_t q, float d, int cw) {
    q >>= 32 / CS * cw;
#pragma unroll
    for (int k = 0; k < 4 / CS; k++) w[k] = d * (float)(int8_t)(uint8_t)(q >> (8 * k));
}
// the upper half of q[0] and the lower half of q[1]
__device__ __forceinline__ uint32_t mid(const uint32_t (&q)[2]) { return __builtin_amdgcn_alignbyte(q[1], q[0], 2); }

template <int CS>
struct SplitQ8_0 {  // src/ops/quant.rs:193-210
    static constexpr bool kFine = false;
    static constexpr int kRow = 272;
    struct Raw {
        uint32_t d0, d1, a[2], b[2], c, e;
    };
    __device__ static void fetch(Raw& r, const uint8_t* row, int si, int g) {
        const uint32_t* q = reinterpret_cast<const uint32_t*>(row) + 17 * si;  // two blocks of 34 bytes
        r.d0 = q[0], r.d1 = q[8];
        r.a[0] = q[g], r.a[1] = q[g + 1], r.b[0] = q[4 + g], r.b[1] = q[5 + g];
        r.c = q[9 + g], r.e = q[13 + g];
    }
    __device__ static void ready(float (&w)[4][4 / CS], const Raw& r, int, int, int cw, uint32_t m0, uint32_t m1) {
        const float d0 = f16_hw(r.d0 & 0xFFFFu & m0), d1 = f16_hw((r.d1 >> 16) & m1);
        scale_s8<CS>(w[0], mid(r.a), d0, cw);
        scale_s8<CS>(w[1], mid(r.b), d0, cw);
        scale_s8<CS>(w[2], r.c, d1, cw);
        scale_s8<CS>(w[3], r.e, d1, cw);
    }
};

template <int CS>
struct SplitQ5_0 {  // src/ops/quant.rs:160-186: elements 0..15 in the low halves, 16..31 in the high halves
    static constexpr bool kFine = false;
    static constexpr int kRow = 176;
    __device__ static void block(float (&lo)[4 / CS], float (&hi)[4 / CS], uint32_t q, uint32_t qh, float d, int g, int cw) {
        qh >>= 4 * g;
#pragma unroll
        for (int e = 0; e < 2; e++) {
            // four high bits to bit 4 of the four bytes, then code - 16 as a signed byte
            const uint32_t h = ((((qh >> (16 * e)) & 15u) * 0x00204081u) & 0x01010101u) << 4;
            const uint32_t u = ((q >> (4 * e)) & 0x0F0F0F0Fu) | h;
            scale_s8<CS>(e ? hi : lo, (u + 0x70707070u) ^ 0x80808080u, d, cw);
        }
    }
    struct Raw {
        uint32_t h[2], q0[2], d1, h1, q1;
    };
    __device__ static void fetch(Raw& r, const uint8_t* row, int si, int g) {
        const uint32_t* q = reinterpret_cast<const uint32_t*>(row) + 11 * si;  // two blocks of 22 bytes
        r.h[0] = q[0], r.h[1] = q[1], r.q0[0] = q[1 + g], r.q0[1] = q[2 + g];
        r.d1 = q[5], r.h1 = q[6], r.q1 = q[7 + g];
    }
    __device__ static void ready(float (&w)[4][4 / CS], const Raw& r, int, int g, int cw, uint32_t m0, uint32_t m1) {
        block(w[0], w[1], mid(r.q0), mid(r.h), f16_hw(r.h[0] & 0xFFFFu & m0), g, cw);
        block(w[2], w[3], r.q1, r.h1, f16_hw((r.d1 >> 16) & m1), g, cw);
    }
};

template <int CS>
struct SplitQ4_0 {  // src/ops/quant.rs:91-111: element 2k low half of byte k, 2k + 1 high half
    static constexpr bool kFine = false;
    static constexpr int kRow = 144;
    struct Raw {
        uint32_t d0, d1, n[4];
    };
    __device__ static void fetch(Raw& r, const uint8_t* row, int si, int g) {
        const uint32_t* q = reinterpret_cast<const uint32_t*>(row) + 9 * si;  // two blocks of 18 bytes
        const uint16_t* h = reinterpret_cast<const uint16_t*>(row) + 18 * si + g;
        r.d0 = q[0], r.d1 = q[4];
#pragma unroll
        for (int p = 0; p < 4; p++) r.n[p] = h[4 * p + (p < 2 ? 1 : 2)];
    }
    __device__ static void ready(float (&w)[4][4 / CS], const Raw& r, int, int, int cw, uint32_t m0, uint32_t m1) {
        const float d0 = f16_hw(r.d0 & 0xFFFFu & m0), d1 = f16_hw((r.d1 >> 16) & m1);
#pragma unroll
        for (int p = 0; p < 4; p++) {
            // elements 4g .. 4g+3 of the part as nibbles 0..3, to bytes, then code - 8 as a signed byte
            const uint32_t u = __builtin_amdgcn_perm((r.n[p] >> 4) & 0x0F0Fu, r.n[p] & 0x0F0Fu, 0x05010400u);
            scale_s8<CS>(w[p], (u + 0x78787878u) ^ 0x80808080u, p < 2 ? d0 : d1, cw);
        }
    }
};

template <int CS>
struct SplitQ4KFloat {  // src/ops/quant.rs:649-667: w = d1*q - m1f per sub-block of 32
    static constexpr bool kFine = false;
    static constexpr int kRow = 144;
    // a window is a super-block; step si its sub-blocks 2si and 2si + 1, in
    // the low and the high halves of 32 bytes
    struct Raw {
        u32x4 h;
        uint32_t q[2];
    };
    __device__ static void fetch(Raw& r, const uint8_t* row, int si, int g) {
        const uint32_t* qs = reinterpret_cast<const uint32_t*>(row) + 4 + 8 * si + g;
        r.h = *reinterpret_cast<const u32x4*>(row);
        r.q[0] = qs[0], r.q[1] = qs[4];
    }
    __device__ static void ready(float (&w)[4][4 / CS], const Raw& r, int si, int, int cw, uint32_t m0, uint32_t) {
        const u32x4 h = r.h;
        const float d = f16_hw(h[0] & 0xFFFFu & m0), dmin = f16_hw((h[0] >> 16) & m0);
#pragma unroll
        for (int b = 0; b < 2; b++) {
            // get_scale_min_k4 (src/ops/quant.rs:267-276) of sub-block 2si + b
            const int sh = 16 * (si & 1) + 8 * b;
            const uint32_t A = h[3] >> sh, B = h[1] >> sh, C = h[2] >> sh;
            const uint32_t sc = si >= 2 ? (A & 15u) | ((B >> 2) & 0x30u) : B & 63u;
            const uint32_t mn = si >= 2 ? ((A >> 4) & 15u) | ((C >> 2) & 0x30u) : C & 63u;
            const float d1 = d * (float)sc, nm = -(dmin * (float)mn);
            // d1*q is exact (an f16 times 6 and 4 bits), so the fused form
            // rounds exactly where the reference's subtraction does
#pragma unroll
            for (int e = 0; e < 2; e++) {
                uint32_t q = (r.q[e] >> (4 * b)) & 0x0F0F0F0Fu;
                q >>= 32 / CS * cw;
#pragma unroll
                for (int k = 0; k < 4 / CS; k++)
                    w[2 * b + e][k] = __builtin_fmaf(d1, (float)((q >> (8 * k)) & 0xFFu), nm);
            }
        }
    }
};

// 4/CS floats as one value
template <int CS>
struct Floats {
    typedef float T __attribute__((ext_vector_type(4 / CS)));
};
// A lane's floats of each part of a step
template <int CS>
__device__ __forceinline__ void load_floats(typename Floats<CS>::T (&o)[4], __amdgpu_buffer_rsrc_t rs, uint32_t off,
                                            uint32_t so) {
    using T = typename Floats<CS>::T;
#pragma unroll
    for (int p = 0; p < 4; p++) {
        const uint32_t a = off + 64 * p;
        if constexpr (CS == 4)
            o[p] = __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(rs, a, so, 0));
        else
            o[p] = __builtin_bit_cast(T, load8(rs, a, so));
    }
}

// F32 rows of any length, each lane its own words from global memory (256
// bytes a step and row: staging them would cost as many registers as it saves
// cache accesses).  off: byte offset of the lane's row, or out of range.
template <int CS>
struct SplitF32 {  // src/model/forward_quantized.rs:674-697
    static constexpr bool kFine = true;
    static constexpr int kRow = 16;  // no window in LDS
    struct Raw {
        typename Floats<CS>::T w[4];
    };
    __device__ static void load(Raw& r, __amdgpu_buffer_rsrc_t rs, uint32_t off, int s, int g, int cw) {
        const uint32_t o = off + 16u * g + 16u / CS * cw;
        load_floats<CS>(r.w, rs, o, 256u * (uint32_t)s);
    }
    __device__ static void ready(float (&w)[4][4 / CS], const Raw& r, int, int, int, uint32_t, uint32_t) {
#pragma unroll
        for (int p = 0; p < 4; p++)
#pragma unroll
            for (int k = 0; k < 4 / CS; k++) w[p][k] = r.w[p][k];
    }
};

// One 16 x 16 tile by CS waves (c = cw*C4 .. for wave cw); 4/CS row tiles to a
// workgroup.
template <template <int> class FmtT, int CS>
__global__ __launch_bounds__(256, 2) void canon_gemm_split_kernel(const float* x, const uint8_t* W, size_t row_bytes, float* y,
                                                                  int n, int out_feat, int batch, int NR, int TP) {
    using Fmt = FmtT<CS>;
    constexpr bool kFine = Fmt::kFine;
    constexpr int C4 = 4 / CS;
    constexpr int RW = 4 / CS;      // row tiles of a workgroup
    constexpr int WS = 4;           // steps of a window
    constexpr int kWinChunk = kChunk / (kStep * WS);
    const int lane = threadIdx.x & 63, wave = wave_id();
    const int g = lane >> 4, r = lane & 15;
    const int cw = wave % CS, rw = wave / CS;
    int rg, tp;
    groups(NR, TP, &rg, &tp);
    const int row0 = rg * RW * 16;  // the workgroup's first row
    const int rows = left(out_feat - row0, 16 * RW);
    const uint32_t wbytes = (uint32_t)row_bytes * (uint32_t)rows;
    // 16 rows are a multiple of 16 bytes in every format, so the base keeps W's alignment
    const __amdgpu_buffer_rsrc_t rsw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(W + (size_t)row0 * row_bytes),
                                                                         (short)0, (int)wbytes, kWord3);
    const int toks = left(batch - 16 * tp, 16);
    const __amdgpu_buffer_rsrc_t rsx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(x + (size_t)(16 * tp) * n), (short)0, (int)(4u * (uint32_t)toks * (uint32_t)n), kWord3);

    // Activations, a window at a time: load k of thread i takes 16-byte chunk
    // i % 64 (inputs 4 (i % 64) .. of the window) of token 4k + i/64, a
    // row's 1 KB per wave; in LDS token a's chunk q lies at slot q ^ a,
    // so neither the writes nor the operand reads (8 lanes at 8 tokens, one
    // chunk) meet in a bank.
    __shared__ u32x4 xs[2][1024];
    const int sa = (int)threadIdx.x >> 6, sq = (int)threadIdx.x & 63;
    u32x4 xr[4];
    // Inputs past the row's end read as zero.  (A step of an f32 row has all
    // its inputs; the rest of such a row is taken after the loop.)
    auto load_x = [&](int w) __attribute__((always_inline)) {
        const int e = kStep * WS * w + 4 * sq;
        const bool in = kFine ? (e / kStep + 1) * kStep <= n : e < n;
#pragma unroll
        for (int k = 0; k < 4; k++)
            xr[k] = load16(rsx, in ? 4u * ((uint32_t)(4 * k + sa) * (uint32_t)n + 4u * (uint32_t)sq) : kOutOfRange,
                           1024u * (uint32_t)w);
    };
    auto stage_x = [&](int w) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < 4; k++) xs[w & 1][64 * (4 * k + sa) + (sq ^ (4 * k + sa))] = xr[k];
    };
    auto read_x = [&](typename Floats<CS>::T (&xv)[1][4], int buf, int si) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < 4; p++)
            xv[0][p] = reinterpret_cast<const typename Floats<CS>::T*>(&xs[buf][64 * r + ((16 * si + 4 * p + g) ^ r)])[cw];
    };

    // Weights (block formats): load k of thread i takes 16-byte chunk i + 256k
    // of the workgroup's rows' windows, row by row.  The last chunk of the last
    // row ends with the row: it is loaded, and lies, as far back as that takes.
    // (Chunks past the rows' last are loaded as zeros and stored behind it: a
    // branch here would let the compiler move the adds of a step across it.)
    constexpr int kCh = Fmt::kRow / 16, kLoads = kFine ? 1 : (16 * RW * kCh + 255) / 256, kWinBytes = kLoads * 4096;
    __shared__ __align__(16) uint8_t wsh[kFine ? 16 : 2 * kWinBytes];
    uint32_t wo[kLoads];  // offset of the chunk at window 0
    u32x4 wt[kLoads];
    if constexpr (!kFine) {
#pragma unroll
        for (int k = 0; k < kLoads; k++) {
            const int i = (int)threadIdx.x + 256 * k, row = i / kCh;
            wo[k] = row < rows ? (uint32_t)row * (uint32_t)row_bytes + 16u * (uint32_t)(i % kCh) : kOutOfRange;
        }
    }
    // bytes by which the chunk at offset o hangs over the end
    auto over = [&](uint32_t o) { return o < wbytes && o + 16 > wbytes ? o + 16 - wbytes : 0u; };
    auto load_w = [&](int w) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < kLoads; k++) {
            const uint32_t o = wo[k] + (uint32_t)(w * Fmt::kRow);
            wt[k] = load16(rsw, o - over(o), 0);
        }
    };
    auto stage_w = [&](int w) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < kLoads; k++) {
            const uint32_t o = wo[k] + (uint32_t)(w * Fmt::kRow);
            *reinterpret_cast<u32x4_a2*>(wsh + (w & 1) * kWinBytes + 16 * ((int)threadIdx.x + 256 * k) - over(o)) = wt[k];
        }
    };
    // (f32: each lane its own words, two steps ahead)
    typename SplitF32<CS>::Raw fr[kFine ? 2 : 1];
    const uint32_t fbase = 16 * rw + r < rows ? (uint32_t)(16 * rw + r) * (uint32_t)row_bytes : kOutOfRange;
    auto load_f = [&](int slot, int s) __attribute__((always_inline)) {
        SplitF32<CS>::load(fr[slot], rsw, kStep * (s + 1) <= n ? fbase : kOutOfRange, s, g, cw);
    };

    const int nchunks = (n + kChunk - 1) / kChunk;
    const int nsteps = kFine ? n / kStep : (n + kStep - 1) / kStep, nwin = (nsteps + WS - 1) / WS;
    float acc[1][2][C4][4];
    float stk[kMaxLevels][1][4];  // completed chunk groups of fixed_tree (a binary counter)
#pragma unroll
    for (int l = 0; l < kMaxLevels; l++)
#pragma unroll
        for (int i = 0; i < 4; i++) stk[l][0][i] = 0.0f;
    float v[1][4];
    __shared__ float4 part[4 * 2 * 64];

    // Window w computes from the LDS buffers that the barrier before it
    // completed; its operands for step si + 1 are read before the adds of step
    // si, which hide the reads.  The next window's loads, issued at its start,
    // are stored at its end.  Steps past the row's end add zero products, which
    // change no chain.
    auto window = [&](int w) __attribute__((always_inline)) {
        const uint8_t* row = wsh + (w & 1) * kWinBytes + (16 * rw + r) * Fmt::kRow;
        typename Fmt::Raw raw[2];
        typename Floats<CS>::T xv[2][1][4];
        float wv[4][C4];
        auto fetch = [&](int si) __attribute__((always_inline)) {
            read_x(xv[si & 1], w & 1, si);
            if constexpr (!kFine) Fmt::fetch(raw[si & 1], row, si, g);
        };
        fetch(0);
        fence();
        load_x(w + 1);
        fence();
        if constexpr (!kFine) load_w(w + 1);
        fence();
#pragma unroll
        for (int si = 0; si < WS; si++) {
            const int s = WS * w + si;
            if constexpr (kFine) {
                Fmt::ready(wv, fr[si & 1], si, g, cw, 0, 0);
                fence();
                load_f(si & 1, s + 2);
            } else {
                Fmt::ready(wv, raw[si & 1], si, g, cw, kStep * s < n ? ~0u : 0u, kStep * s + 32 < n ? ~0u : 0u);
            }
            fence();
            if (si + 1 < WS) fetch(si + 1);
            fence();
            mul_add<C4>(acc, wv, xv[si & 1]);
        }
        fence();
        stage_x(w + 1);
        if constexpr (!kFine) stage_w(w + 1);
        __syncthreads();
    };

    load_x(0);
    fence();
    if constexpr (!kFine) load_w(0);
    stage_x(0);
    if constexpr (!kFine) stage_w(0);
    fence();
    if constexpr (kFine) {
        load_f(0, 0);
        fence();
        load_f(1, 1);
        fence();
    }
    __syncthreads();
    for (int c = 0; c < nchunks; c++) {
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int k = 0; k < C4; k++)
#pragma unroll
                for (int i = 0; i < 4; i++) acc[0][h][k][i] = 0.0f;
        const int w1 = min((c + 1) * kWinChunk, nwin);
        for (int w = c * kWinChunk; w < w1; w++) window(w);
        if (kFine && c + 1 == nchunks && n % kStep) {
            // the rest of an f32 row: what lies past its end belongs to the next row
            const int s = n / kStep;
            typename SplitF32<CS>::Raw rt;
            typename Floats<CS>::T xt[1][4];
            float wv[4][C4];
            SplitF32<CS>::load(rt, rsw, fbase, s, g, cw);
            {
                const int i = (int)threadIdx.x, a = i >> 4, q = i & 15;
                xs[0][64 * a + (q ^ a)] = load16(rsx, 4u * ((uint32_t)a * (uint32_t)n + 4u * (uint32_t)q), 256u * (uint32_t)s);
            }
            __syncthreads();
            read_x(xt, 0, 0);
            SplitF32<CS>::ready(wv, rt, 0, g, cw, 0, 0);
#pragma unroll
            for (int p = 0; p < 4; p++)
#pragma unroll
                for (int k = 0; k < C4; k++) {
                    const bool in = kStep * s + 16 * p + 4 * g + cw * C4 + k < n;
                    wv[p][k] = in ? wv[p][k] : 0.0f;
                    xt[0][p][k] = in ? xt[0][p][k] : 0.0f;
                }
            mul_add<C4>(acc, wv, xt);
        }
        // fixed_tree over the 8 chains: ((0+1)+(2+3)) + ((4+5)+(6+7))
        float h[1][2][4];
        chain_tree(acc, h);
        if (c) __syncthreads();  // the previous chunk's parts have been read
#pragma unroll
        for (int e = 0; e < 2; e++) part[(wave * 2 + e) * 64 + lane] = make_float4(h[0][e][0], h[0][e][1], h[0][e][2], h[0][e][3]);
        __syncthreads();
        if (cw == 0) {
#pragma unroll
            for (int e = 0; e < 2; e++) {
                float4 p[CS];
#pragma unroll
                for (int q = 0; q < CS; q++) p[q] = part[((wave + q) * 2 + e) * 64 + lane];
#pragma unroll
                for (int st = 1; st < CS; st <<= 1)
#pragma unroll
                    for (int q = 0; q < CS; q += 2 * st)
                        p[q] = make_float4(p[q].x + p[q + st].x, p[q].y + p[q + st].y, p[q].z + p[q + st].z,
                                           p[q].w + p[q + st].w);
                h[0][e][0] = p[0].x, h[0][e][1] = p[0].y, h[0][e][2] = p[0].z, h[0][e][3] = p[0].w;
            }
        }
#pragma unroll
        for (int i = 0; i < 4; i++) v[0][i] = h[0][0][i] + h[0][1][i];
        chunk_tree(stk, v, c, nchunks);
    }
    if (cw == 0) store(y, v[0], 16 * tp + r, row0 + 16 * rw + 4 * g, batch, out_feat);
}

template <template <int> class FmtT>
hipError_t launch_split(int cs, const float* x, const uint8_t* w, size_t row_bytes, float* y, int batch, int n, int out_feat,
                        hipStream_t stream) {
    const int rows = 16 * (4 / cs), NR = (out_feat + rows - 1) / rows, TP = (batch + 15) / 16;
    const dim3 grid((unsigned)NR * (unsigned)TP);
    if (cs == 4)
        hipLaunchKernelGGL((canon_gemm_split_kernel<FmtT, 4>), grid, dim3(256), 0, stream, x, w, row_bytes, y, n, out_feat,
                           batch, NR, TP);
    else
        hipLaunchKernelGGL((canon_gemm_split_kernel<FmtT, 2>), grid, dim3(256), 0, stream, x, w, row_bytes, y, n, out_feat,
                           batch, NR, TP);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_canon_gemm_split(CanonFormat fmt, int cs, const float* x, const uint8_t* w, size_t row_bytes, float* y,
                                   int batch, int in_feat, int out_feat, hipStream_t stream) {
    switch (fmt) {
    case kCanonQ8_0: return launch_split<SplitQ8_0>(cs, x, w, row_bytes, y, batch, in_feat, out_feat, stream);
    case kCanonQ5_0: return launch_split<SplitQ5_0>(cs, x, w, row_bytes, y, batch, in_feat, out_feat, stream);
    case kCanonQ4_0: return launch_split<SplitQ4_0>(cs, x, w, row_bytes, y, batch, in_feat, out_feat, stream);
    case kCanonF32: return launch_split<SplitF32>(cs, x, w, row_bytes, y, batch, in_feat, out_feat, stream);
    case kCanonQ4KFloat: return launch_split<SplitQ4KFloat>(cs, x, w, row_bytes, y, batch, in_feat, out_feat, stream);
    }
    return hipErrorInvalidValue;
}

}  // namespace vtq
