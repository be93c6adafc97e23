// vtq_rules.h -- which kernel, and which form of it, takes a call: the rules of
// the dispatch on sizes and types, host code without a kernel, so that tests can
// ask them (libvtq_probe.so) without a GPU.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace vtq {

// Canonical-dot weight formats (8-lane pinned fp32 dot, src/ops/quant.rs:482-566).
enum CanonFormat { kCanonQ8_0 = 0, kCanonQ5_0 = 1, kCanonQ4_0 = 2, kCanonF32 = 3, kCanonQ4KFloat = 4 };

constexpr int kCanonMaxInFeat = 65536;  // inputs of one launch: 8 chunks of 8192

// ------------------------------------------------ pinned dot over batch rows

constexpr int kGmStep = 64;  // inputs of a step

// The forms (CS = 1 in canon_gemm.hip, CS = 2 and 4 in canon_gemm_split.hip) and the time of
// one in nanoseconds, as measured over 21 shapes (2 to 512 tokens, 256 to 11008
// inputs, 64 to 32000 rows): what counts is the steps of a row and how many
// waves each of the 1024 SIMDs gets in turn.  A lone wave waits for its own
// loads and barriers, so its step costs more than a shared SIMD's.  The split
// forms go by whole windows of four steps.  (Q8_0 4096 x 4096, us, with CS = 1 / 2
// / 4: 16 tokens 65 / 38 / 25; 32 tokens 65 / 38 / 35; 64 tokens 65 / 58 / 65;
// 128 tokens 103 / 107 / 126, 115 with NT = 2; 2048 x 2048 at 512 tokens 98 with
// NT = 1, 94 with NT = 2; 896 x 4864 at 300 tokens 65 with NT = 2, 78 with CS = 2.)
struct GmForm {
    int nt, cs;
    long lone, pair, more;  // ns a step: one wave per SIMD, two, each of more
};
constexpr GmForm kGmForms[] = {{1, 4, 350, 520, 245}, {1, 2, 550, 855, 408}, {1, 1, 1000, 1600, 800},
                               {2, 1, 1780, 2950, 1475}};
// F32 rows aren't staged, so with CS = 4 four waves gather each row, 16 loads of
// 64 cache accesses a tile and step: the vector memory path's time on a full CU.
// (64 tokens of 2048 x 2048: 33.2 us with CS = 4, 19.5 with CS = 2.)
constexpr GmForm kGmF32Split4 = {1, 4, 430, 940, 470};
constexpr long kGmLaunchNs = 3000;  // besides the steps

inline int gm_pick(CanonFormat fmt, int batch, int n, int out_feat, long* ns) {
    int best = 0;
    *ns = 0;
    for (int f = 0; f < 4; f++) {
        const GmForm& k = f == 0 && fmt == kCanonF32 ? kGmF32Split4 : kGmForms[f];
        const long tiles = (long)((out_feat + 15) / 16) * ((batch + 16 * k.nt - 1) / (16 * k.nt));
        const long waves = (tiles * k.cs + 1023) / 1024, whole = (k.cs > 1 ? 4 : 1) * kGmStep;
        const long steps = (n + whole - 1) / whole * (whole / kGmStep);
        const long t = steps * (waves == 1 ? k.lone : waves == 2 ? k.pair : k.more * waves) + kGmLaunchNs;
        if (f == 0 || t < *ns) best = f, *ns = t;
    }
    return best;
}

// Whether the batch kernel is faster than one GEMV slice per batch row, whose
// time is its weights decoded per nanosecond (measured with the shapes above:
// Q8_0 3600 in the LDS-resident kernel, 2000 in the windowed one; Q4_K float
// 2300, Q4_0 2000, Q5_0 1200, F32 1000).  With those the line for Q8_0 4096 x 4096
// lies between 4 tokens (22 us against 25) and 8 (40 against 25).  The windowed
// kernel is faster on a grid that fills the chip, rows of one chunk that are long
// enough to hide their start: Q4_0 2500 (2 tokens, us, GEMV against the batch
// kernel: 4096 -> 16384 47.5 / 57.0, -> 32000 88.4 / 105.2; 1024 -> 32000 30.0 /
// 29.7; 11008 -> 16384 190 / 148), on a smaller one 2100 (7 tokens, 3840 -> 1985 22.6 /
// 24.4; 3, 2048 -> 8192 20.8 / 19.6), Q8_0 2900 and 2200 (8192 -> 32000 162 / 200;
// 14336 -> 32000 447 / 348; 3 tokens, 7040 -> 15341 103 / 95, 6272 -> 6629 44.2 /
// 50.5, 4352 -> 8192 36.0 / 35.1).
inline bool canon_gemm_faster(CanonFormat fmt, int batch, int in_feat, int out_feat) {
    if (batch < 2 || in_feat > kCanonMaxInFeat) return false;
    // a launch holds fewer than 2^32 threads; no form has more than 256 to a tile of 16 x 16
    if ((size_t)((out_feat + 15) / 16) * ((batch + 15) / 16) >= ((size_t)1 << 24)) return false;
    const bool one = in_feat > 1024 && in_feat <= 8192, full = one && (size_t)batch * out_feat >= 32000;
    const double rate = fmt == kCanonQ8_0 ? (in_feat % 256 == 0 && in_feat <= 4096 ? 3600 : full ? 2900 : one ? 2200 : 2000)
                        : fmt == kCanonQ4KFloat ? 2300
                        : fmt == kCanonQ4_0 ? (full ? 2500 : one ? 2100 : 2000)
                        : fmt == kCanonQ5_0 ? 1200 : 1000;
    const double gemv = (double)batch * in_feat * out_feat / rate * 0.9;
    if (gemv <= kGmLaunchNs) return false;
    long ns;
    gm_pick(fmt, batch, in_feat, out_feat, &ns);
    return gemv > (double)ns;
}

// ------------------------------------------------------- k-quant batch GEMM

constexpr int kTO = 32;        // LDS-operand kernel: weight rows per workgroup
constexpr int kTB = 128;       // and tokens per workgroup (4 waves x 32)
constexpr int kChunkM = 8192;  // tokens per launch pair (bounds the workspace)
constexpr int kPwMaxR = 16;    // super-blocks of a row in the per-wave kernel
constexpr int pw_level_bytes(int NT) { return NT * 4 * 64 * 16; }  // one tree level of NT tiles

constexpr int kSkMaxWaves = 12;

// The chunks of a row of R super-blocks cut into pieces of C (q4k_gemm_sk_kernel).
inline int sk_chunks(int R, int C) {
    int n = 0;
    for (int k = 6; k >= 0; k--)
        if ((R >> k) & 1) n += (1 << k) >= C ? (1 << k) / C : 1;
    return n;
}

// The piece size for a grid of T tiles: the smallest that keeps the launch
// within 2048 waves (8 per CU), else the smallest that needs at most
// kSkMaxWaves chunks (every row length below 128 super-blocks has one).
inline int sk_piece(int R, int T) {
    int first = 0;
    for (int C = 1; C <= 16; C <<= 1) {
        const int n = sk_chunks(R, C);
        if (n > kSkMaxWaves) continue;
        if (!first) first = C;
        if ((long)T * n <= 2048) return C;
    }
    return first;
}

constexpr int kQ6StageBytes = 32 * 208;
// the weight stage, or a chunk's value where that is larger
constexpr int sk_stage_bytes(bool q6, int NT) {
    return !q6 ? 4096 : NT * 4096 > kQ6StageBytes ? NT * 4096 : kQ6StageBytes;
}
constexpr int sk_lds_per_wave(bool q6, int NT, int C) {
    return sk_stage_bytes(q6, NT) + (q6 ? 128 : 256) + (C > 8 ? 2 : C > 4 ? 1 : 0) * pw_level_bytes(NT);
}

// With NT = 2 (Q6_K) a wave's two token tiles need the registers of an 8-wave
// workgroup.
constexpr int sk_max_waves(int NT) { return NT == 2 ? 8 : kSkMaxWaves; }

// The piece size with two token tiles, or 0: chunks long enough to hide a
// wave's first loads, in as many waves and as much LDS as a workgroup has.
inline int sk_piece2(int R) {
    for (int C = 4; C <= 16; C <<= 1)
        if (sk_chunks(R, C) <= sk_max_waves(2) && sk_chunks(R, C) * sk_lds_per_wave(true, 2, C) <= 160 * 1024) return C;
    return 0;
}

// Which kernel takes a launch (M tokens in Mt 32-token tiles): 3 the
// split-K kernel, for grids too small to fill the chip; else 2 the per-wave
// kernel with two token tiles per wave for rows of at most 16 super-blocks,
// 0 the LDS-operand kernel for longer rows.  Split-K takes rows of at most 16
// super-blocks up to 1024 tiles of 32 x 32, and longer rows where the
// LDS-operand kernel would launch fewer than 256 workgroups (measured
// crossovers, pre-pass included: 4096 x 4096 at 256 tokens 25.5 against
// 26.3 us for the LDS-operand kernel, 11264 x 2048 at 96 tokens 19.5 against
// 18.8 us for the per-wave kernel; 4096 x 11008 at 128 tokens 43.4 against
// 56.5 us, at 256 tokens 76.6 against 59.3 us).  Longer rows below 32 tokens
// always take it: the LDS-operand kernel spends a workgroup of 128 tokens on
// them and folds a row in series (us, GEMV per row / LDS-operand / split-K, 4
// tokens: 14336 -> 8192 57 / 74 / 27, 4352 -> 8200 20.8 / 29.8 / 16.3, 8192 ->
// 128256 391 / 405 / 186; at 31 tokens of 14336 -> 8192 357 / 71 / 27).  The
// split-K and per-wave forms address the weights with 32-bit buffer offsets.
inline int gemm_form(int R, int N, int M, int Mt) {
    if ((size_t)N * R * 144 >= ((size_t)1 << 31)) return 0;
    if (R <= kPwMaxR) return (long)((N + 31) / 32) * Mt <= 1024 ? 3 : 2;
    if (M < 32) return 3;
    return (long)((N + kTO - 1) / kTO) * ((M + kTB - 1) / kTB) < 256 ? 3 : 0;
}

// From this many Q4_K rows on every call takes the GEMM, as the GEMV streams the
// matrix once per batch row (4096 x 4096: 34.3 us for 16 rows already, the GEMM
// 12.7).
constexpr int kGemmOnlyBatch = 32;
constexpr int kQ4MaxR = 127;

// Whether a batch takes the GEMM rather than one GEMV slice per batch row: from
// 32 rows on always; below, from 16 rows, from 8 with at least 2^22 weights,
// from 4 with at least 2^27 weights times rows (us, GEMV against GEMM: 8 x
// 4096 x 11008 24.2 / 15.5, 8 x 4096 x 4096 18.5 / 12.4, 4 x 4096 x 4096 10.9 /
// 12.0, 4 x 11008 x 4096 27.5 / 19.0, 4 x 2048 x 32000 16.8 / 15.1, 3 x 2048 x
// 32000 13.3 / 15.2, 8 x 2048 x 2048 11.6 / 11.8, 8 x 512 x 300 9.0 / 11.9,
// 16 x 256 x 64 14.5 / 12.0).  Four tokens on rows of 8 to 16 super-blocks gain
// less: past 32768 outputs, where the per-wave kernel takes them in rounds of
// 65536, they take it from 40000 on (4096 -> 33000 41.0 / 47.5, -> 40000 49.7 /
// 48.8; 3072 -> 33000 30.9 / 36.0, -> 40000 38.0 / 37.7; 2048 -> 33000 18.7 / 24.2,
// -> 40000 25.5 / 25.7).
inline bool q4k_gemm_faster(size_t batch, size_t in_feat, size_t out_feat) {
    if (in_feat == 0 || in_feat > (size_t)kQ4MaxR * 256) return false;
    if (batch >= (size_t)kGemmOnlyBatch) return true;
    if (out_feat * (in_feat / 256) >= ((size_t)1 << 31) / 144) return false;  // past the small grids' kernel
    const size_t w = in_feat * out_feat;
    if (batch == 4 && in_feat >= 2048 && in_feat <= (size_t)kPwMaxR * 256 && out_feat > 32768 && out_feat < 40000) return false;
    return batch >= 16 || (batch >= 8 && w >= ((size_t)1 << 22)) || (batch >= 4 && batch * w >= ((size_t)1 << 27));
}

// Whether a Q6_K launch of NR row and Mt token tiles takes two token tiles to a
// wave, and then the piece size: where the workgroups and waves still keep most
// of the chip busy (us, one tile against two, in brackets workgroups x waves of
// the second form): 11008 -> 4096 at 200 tokens 96.7 / 68.9 [512 x 7], at 96 52.4
// / 33.5 [256 x 7], at 64 27.7 / 32.2 [128 x 7]; 11008 -> 6000 at 64 52.2 / 31.8
// [188 x 7]; 5632 -> 2048 at 192 27.1 / 21.3 [192 x 6], at 128 17.6 / 18.9
// [128 x 6]; 4096 -> 2048 at 192 19.4 / 15.7 [192 x 4]; 4096 -> 14336 at 512 197 /
// 129; 2048 -> 32000 at 128 75.0 / 42.6.  Rows of one super-block gain at some
// sizes and lose at others (512 tokens, 10000 rows 14.9 / 15.7).
inline int q6k_two_tiles(int R, int NR, int Mt) {
    const int C = sk_piece2(R);
    const long wgs = (long)NR * ((Mt + 1) / 2);
    return C && R > 1 && Mt > 1 && wgs >= 160 && wgs * sk_chunks(R, C) >= 700 ? C : 0;
}

// From how many weights on a Q6_K batch of 3 to 7 rows takes the GEMM: its time
// below some 10 M weights is a row's chain of leaves (7.8 us and 0.3 us a
// super-block), the GEMV's a pass over the matrix per batch row, so long rows of
// small matrices stay with the GEMV.  us, GEMV against GEMM, either side of each
// line: 3 rows 1024 -> 8193 12.7 / 9.0; 2048 -> 4097 9.1 / 9.9, -> 5793 11.0 / 10.2;
// 4096 -> 2897 11.4 / 12.7, -> 4097 13.6 / 13.4; 8192 -> 2897 16.2 / 18.1, -> 4097
// 19.3 / 18.8; 14336 -> 1656 24.7 / 25.7, -> 2341 26.7 / 26.4.  4 rows 4096 -> 2049
// 12.3 / 12.4; 8192 -> 1449 15.4 / 17.8, -> 2049 17.9 / 17.9; 14336 -> 586 24.0 /
// 25.8, -> 828 26.8 / 25.5.  5 rows 8192 -> 1025 16.2 / 17.7, -> 1449 18.7 / 17.9.
inline size_t q6k_least_weights(size_t batch, int R) {
    size_t m = 8;
    if (batch == 3) m = R <= 4 ? 8 : R <= 8 ? 10 : R <= 16 ? 16 : 32;
    if (batch == 4 && R > 16) m = R <= 32 ? 16 : 11;
    if (batch == 5 && R > 16 && R <= 32) m = 11;
    return m << 20;
}

// Whether a Q6_K batch takes the GEMM rather than one GEMV slice per batch row:
// from 8 rows on, from 3 with q6k_least_weights (us, GEMV against GEMM: 4096 x
// 4096 at 2 rows 11.0 / 12.8; 11008 -> 4096 at 2 rows 19.1 / 22.7, at 4 35.3 /
// 22.7; 1024 -> 2000 at 4 rows 10.0 / 11.2; 512 -> 300 at 8 rows 13.2 / 11.3).
// 32-bit offsets address the weights; the 11 waves that rows of 127 super-blocks
// need do not fit in LDS.
constexpr int kQ6MaxR = 126;
inline bool q6k_gemm_faster(size_t batch, size_t in_feat, size_t out_feat) {
    if (in_feat == 0 || in_feat > (size_t)kQ6MaxR * 256) return false;
    const size_t R = in_feat / 256;
    return out_feat * R < ((size_t)1 << 31) / 210 &&
           (batch >= 8 || (batch >= 3 && in_feat * out_feat >= q6k_least_weights(batch, (int)R)));
}

}  // namespace vtq
