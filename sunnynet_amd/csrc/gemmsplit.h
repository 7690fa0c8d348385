// Products of many rows on the fp16 matrix cores from operands in two fp16 planes
// (gemmsplit.hip).
//
// A row x of K floats is held as 2^s x = h + l in two fp16 planes, s the power of
// two that takes the row's largest magnitude into [2^14, 2^15): h rounds 2^s x to
// 11 bits, l the exact remainder to 11 more, so h + l differs from 2^s x by at most
// 2^-22 of it or 2^-24: 22 bits where fp32 has 24, and fewer for values below 2^-17
// of their row's largest. A product is X W^T = 2^-(sx + sw) (Hx Hw + (Hx Lw + Lx Hw)),
// accumulated in fp32, the two parts apart; Lx Lw, below 2^-22 of a term, is left
// out. What these leave out is less than what the sums round: against 64 bits the
// outputs are nearer than with the fp32 matrix cores, whose sums are rounded once
// per two values of k and these once per 16. SunnyNet-100M and -small, 1 to 16
// prompts of 64 to 2048 tokens, fp32, fp16 and INT4 weights (57 calls of two seeds):
// the error of logits 0.38 to 0.75 of theirs, of states 0.76 to 0.99. (With one
// accumulator for the three products it was up to 1.16 of theirs.)
#pragma once

#include <climits>

#include "gemm.h"

namespace snhip {

constexpr int kSplitTile = 256;          // rows of planes are padded to this
constexpr int kSplitNonFinite = INT_MIN; // `ex` of a row with an infinity or NaN

// Planes of a matrix of rows: `pl` in fragment order (split_halfs(rows, K)
// uint16), `ex` the rows' s (rows padded to kSplitTile).
struct SplitMat {
    uint16_t* pl = nullptr;
    int* ex = nullptr;
};
inline size_t split_rows(size_t rows) { return (rows + kSplitTile - 1) / kSplitTile * kSplitTile; }
inline size_t split_halfs(size_t rows, size_t K) { return split_rows(rows) * K * 2; }

// Planes of g's X rows (g.M, with its shifted reads), or of its weights (g.N rows).
snhip_status launch_split_x(const GemmArgs& g, SplitMat out, hipStream_t st);
snhip_status launch_split_w(const GemmArgs& g, SplitMat out, hipStream_t st);
// Planes of the prefill's intermediate rows, made where they are computed, for rows
// of at most kSplitRegs values (a multiple of 8; all arrays 16-byte aligned):
constexpr int kSplitRegs = 2048;
// raw + depthwise conv over the rows of each sequence of T (k_conv_rows' order);
struct SplitConv {
    const float *raw, *hist;
    size_t hist_bstride;
    const float* dw;
    int T, D, taps;
};
// the gated u, with p and (1 - p) u to pa and pb (k_gate_rows' order);
struct SplitGate {
    const float *q, *delta;
    float *pa, *pb;
    int D, clamp;
    float p_floor;
};
// LayerNorm of rows of n.
struct SplitLn {
    const float *x, *g, *c;
    int n;
    float eps;
};
snhip_status launch_split_conv(const SplitConv& c, int rows, SplitMat out, hipStream_t st);
snhip_status launch_split_gate(const SplitGate& c, int rows, SplitMat out, hipStream_t st);
snhip_status launch_split_ln(const SplitLn& c, int rows, SplitMat out, hipStream_t st);
// Y = X W^T with g's epilogue from the planes of both. `work` is scratch for
// split-K partials as launch_gemm's.
snhip_status launch_gemm_split(const GemmArgs& g, SplitMat x, SplitMat w, float* work, size_t work_floats,
                               hipStream_t st);

}  // namespace snhip
