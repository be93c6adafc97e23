// vtq_probe.hip -- helpers of the benchmark and the tests (libvtq_probe.so).
//
// Not part of the quantized-linear boundary (include/vtq.h).  The kernels
// exist only to measure what the hardware gives a plain access pattern on
// the same buffers the benchmark's GEMVs read, so that each GEMV's rate can
// be quoted against a measured read ceiling as well as the published peak.
// The queries name the form that the dispatch rules (vtq_rules.h) give a call,
// so that a test can say which kernel it covers; they touch no GPU.
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "vtq_rules.h"

namespace {

// Read-only stream: every thread reads 16-byte words i = g, g + G, g + 2G, ...
// (g = global thread index, G = grid threads), one load in flight per thread,
// and folds them into one word.  The store happens only if that word equals
// a constant the data never produces in practice; it keeps the loads alive
// without adding write traffic.
__global__ __launch_bounds__(256) void stream_read_kernel(const uint4* __restrict__ p, size_t n16,
                                                          uint32_t* __restrict__ sink) {
    uint32_t acc = 0;
    const size_t stride = (size_t)gridDim.x * 256;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n16; i += stride) {
        const uint4 v = p[i];
        acc ^= v.x ^ v.y ^ v.z ^ v.w;
    }
    if (acc == 0x9E3779B9u) sink[blockIdx.x] = acc;
}

}  // namespace

extern "C" {

// Launches the read of `bytes` (a multiple of 16) starting at device pointer
// `p` on `stream` with `workgroups` workgroups of 256 threads; `sink` is a
// device buffer of at least `workgroups` words.  Returns a hipError_t value.
int vtqp_stream_read(const void* p, size_t bytes, int workgroups, void* sink, void* stream) {
    if (!p || !sink || workgroups <= 0 || bytes % 16 != 0) return (int)hipErrorInvalidValue;
    hipLaunchKernelGGL(stream_read_kernel, dim3((unsigned)workgroups), dim3(256), 0, (hipStream_t)stream,
                       static_cast<const uint4*>(p), bytes / 16, static_cast<uint32_t*>(sink));
    return (int)hipGetLastError();
}

// The form a pinned-dot call takes: 0 one GEMV slice per batch row, else 10 *
// token tiles of a wave + waves to a tile.
int vtqp_canon_form(int fmt, int batch, int in_feat, int out_feat) {
    if (fmt < 0 || fmt > vtq::kCanonQ4KFloat || batch <= 0 || in_feat <= 0 || out_feat <= 0) return -1;
    const vtq::CanonFormat f = (vtq::CanonFormat)fmt;
    if (!vtq::canon_gemm_faster(f, batch, in_feat, out_feat)) return 0;
    long ns;
    const vtq::GmForm& g = vtq::kGmForms[vtq::gm_pick(f, batch, in_feat, out_feat, &ns)];
    return 10 * g.nt + g.cs;
}

// The form a k-quant call (Q4_K = 12 / Q6_K = 14, integer regime) takes: 0 one
// GEMV slice per batch row, 1 the LDS-operand kernel, 2 the per-wave kernel,
// 300 + piece the split-K kernel, 600 + piece the same with two token tiles to
// a wave.
int vtqp_kquant_form(int type, int batch, int in_feat, int out_feat) {
    if ((type != 12 && type != 14) || batch <= 0 || in_feat <= 0 || in_feat % 256 || out_feat <= 0) return -1;
    const int R = in_feat / 256, NR = (out_feat + 31) / 32;
    const int M = batch < vtq::kChunkM ? batch : vtq::kChunkM, Mt = (M + 31) / 32;
    if (type == 14) {
        if (!vtq::q6k_gemm_faster(batch, in_feat, out_feat)) return 0;
        if (const int C = vtq::q6k_two_tiles(R, NR, Mt)) return 600 + C;
        return 300 + vtq::sk_piece(R, NR * Mt);
    }
    if (!vtq::q4k_gemm_faster(batch, in_feat, out_feat)) return 0;
    const int form = vtq::gemm_form(R, out_feat, M, Mt);
    return form == 3 ? 300 + vtq::sk_piece(R, NR * Mt) : form == 2 ? 2 : 1;
}

}  // extern "C"
