// Order-faithful RWKV-7 step kernels (rkseq.h).
//
// The reference's C runtime (sunnynet/runtime/rwkv7.c) rounds in a fixed
// order: every matrix product is a sequential fmaf chain over the inputs,
// LayerNorm and group-norm statistics are sequential sums, the head state
// dots use eight stride-8 partial sums folded as ((0+4)+(1+5))+((2+6)+(3+7)),
// and expf / tanhf are glibc's. The kernels here repeat exactly that:
//
// * Products run on the matrix cores with v_mfma_f32_16x16x4_f32, whose four
//   products are added in order with one rounding each (k_rkq_mm): issued in k
//   order they give the reference's chain. INT4 weights are dequantized in
//   registers as fma(q, s, -8 s), which equals quant.c's (q - 8) s.
// * LayerNorm: one wave per row, the row in LDS, one lane running each
//   sequential sum while the others prepare the squared deviations.
// * Heads: one wave per (head, sequence), lane i owning state row i.
// * expf / tanhf: refmath.h (glibc's algorithms).
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "lanesum.h"
#include "refmath.h"
#include "rkseq.h"
#include "snhip_rwkv7.h"

namespace snhip {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4v __attribute__((ext_vector_type(4)));

constexpr float kR2 = 0.6065306597126334f;   // 1/sqrt(e), rwkv7.c:38
constexpr float kEpsGroup = 6.4e-4f;          // rwkv7.c:39
constexpr int kHS = 64;
constexpr int kLnMax = 4096;

__device__ __forceinline__ float hsum8(const float* v) {
    const float c0 = v[0] + v[4], c1 = v[1] + v[5], c2 = v[2] + v[6], c3 = v[3] + v[7];
    return (c0 + c1) + (c2 + c3);
}

// ------------------------------------------------------------------ rows
// Sequential fp32 sum of n4 float4 in LDS (element order), by one lane.
// Rows whose length is a multiple of 64 run through a window of 16 float4:
// slot i is added, then refilled with the same slot of the next block, so
// the reads stay one block (64 dependent adds) ahead with no register copies
// and only the chain of dependent adds is exposed.
__device__ __forceinline__ float seq_sum(const float4* v, int n4) {
    float s = 0.0f;
    if (n4 % 16 == 0) {
        float4 w[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) w[i] = v[i];
        for (int base = 0; base < n4; base += 16) {
            const int nb = min(base + 16, n4 - 16);   // the next block (the last block again at the end)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                s = s + w[i].x; s = s + w[i].y; s = s + w[i].z; s = s + w[i].w;
                w[i] = v[nb + i];
            }
        }
        return s;
    }
    for (int i = 0; i < n4; ++i) {
        const float4 b = v[i];
        s = s + b.x; s = s + b.y; s = s + b.z; s = s + b.w;
    }
    return s;
}

// Row LayerNorm of rows up to kLnMax, one workgroup of LT threads per row:
// thread t owns float4 q = t + LT j of the row (elements 4q .. 4q+3); its
// row, gain, bias, shift and mix values are loaded as float4 before the sums,
// so the only exposed latencies are one round trip and the two sequential
// sums (one lane). 256 threads rather than one wave spread the row's loads
// and the mixes' stores: 9.6 -> 8.4 us per call at D = 768, B = 64.
constexpr int kLnR = 192;                  // float4 of a row held in registers (rows <= 768)
constexpr int kLnT = 256;                  // threads per row

template <int LT>
__global__ __launch_bounds__(LT) void k_rkq_ln(RkqLnArgs A) {
    constexpr int kLnQ = (kLnR + LT - 1) / LT;   // float4 per thread
    __shared__ float4 xs4[kLnMax / 4];
    __shared__ float4 sq4[kLnMax / 4];
    __shared__ float stat[2];
    const int b = blockIdx.x, t = threadIdx.x, D = A.D, n4 = D / 4;
    const float4* src;
    bool ok = true;
    if (A.mode == RKQ_LN_EMBED) {
        const int tk = A.tok[b];
        ok = tk >= 0 && tk < A.vocab;
        src = reinterpret_cast<const float4*>(A.embed + (size_t)(ok ? tk : 0) * D);
    } else {
        src = reinterpret_cast<const float4*>(A.x + (size_t)b * D);
    }
    float4* sh4 = A.shift ? reinterpret_cast<float4*>(A.shift + (size_t)b * A.shift_bstride) : nullptr;
    const float4* g4 = reinterpret_cast<const float4*>(A.g);
    const float4* c4 = reinterpret_cast<const float4*>(A.c);
    const float4* l4 = reinterpret_cast<const float4*>(A.lerp);
    const bool regs = n4 <= LT * kLnQ;
    const bool mix1 = A.mode == RKQ_LN_MIX1, mix2 = A.mode == RKQ_LN_MIX2;
    float4 gv[kLnQ], cv[kLnQ], sv[kLnQ], lv[6][kLnQ];
    for (int q = t; q < n4; q += LT) {
        float4 v = src[q];
        if (!ok) v = make_float4(__builtin_nanf(""), __builtin_nanf(""), __builtin_nanf(""), __builtin_nanf(""));
        xs4[q] = v;
    }
    if (regs) {
#pragma unroll
        for (int j = 0; j < kLnQ; ++j) {
            const int q = min(t + LT * j, n4 - 1);
            gv[j] = g4[q];
            cv[j] = c4[q];
            if (mix1 || mix2) sv[j] = sh4[q];
            if (mix1) {
#pragma unroll
                for (int s6 = 0; s6 < 6; ++s6) lv[s6][j] = l4[(size_t)s6 * n4 + q];
            } else if (mix2) {
                lv[0][j] = l4[q];
            }
        }
    }
    __syncthreads();
    // sum = sum + x[i], then vsum = vsum + d * d, in order: lane-sliced in
    // wave 0 (lanesum.h) for rows of 256, 512, 768 or 1024, else by thread 0
    const int kl = D % 256 ? 0 : D / 256;
    if (kl >= 1 && kl <= 4) {
        if (t < 64) {
            auto go = [&](auto k) {
                constexpr int KL4 = decltype(k)::value;
                float v[4 * KL4];
#pragma unroll
                for (int q = 0; q < KL4; ++q) {
                    const float4 x = xs4[t * KL4 + q];
                    v[4 * q] = x.x; v[4 * q + 1] = x.y; v[4 * q + 2] = x.z; v[4 * q + 3] = x.w;
                }
                float m, r;
                lane_ln_stats(v, D, A.eps, m, r);
                if (t == 0) {
                    stat[0] = m;
                    stat[1] = r;
                }
            };
            if (kl == 1) go(std::integral_constant<int, 1>{});
            else if (kl == 2) go(std::integral_constant<int, 2>{});
            else if (kl == 3) go(std::integral_constant<int, 3>{});
            else go(std::integral_constant<int, 4>{});
        }
        __syncthreads();
    } else {
        if (t == 0) stat[0] = seq_sum(xs4, n4) / (float)D;
        __syncthreads();
        const float m0 = stat[0];
        for (int q = t; q < n4; q += LT) {
            const float4 v = xs4[q];
            float4 d;
            d.x = v.x - m0; d.y = v.y - m0; d.z = v.z - m0; d.w = v.w - m0;
            d.x = d.x * d.x; d.y = d.y * d.y; d.z = d.z * d.z; d.w = d.w * d.w;
            sq4[q] = d;
        }
        __syncthreads();
        if (t == 0) stat[1] = 1.0f / sqrtf(seq_sum(sq4, n4) / (float)D + A.eps);
        __syncthreads();
    }
    const float mean = stat[0], rstd = stat[1];
    const size_t mat = x16_floats((int)gridDim.x, D);   // one matrix of all rows
    // float4 q of this row in x16 order (its four inputs are 64 floats apart)
    auto put = [&](float* m, int q, float4 v) {
        float* p = m + x16_at(b, 4 * q, D / 16);
        p[0] = v.x; p[64] = v.y; p[128] = v.z; p[192] = v.w;
    };
    auto norm = [&](float x, float g, float c) { return (x - mean) * rstd * g + c; };
    auto emit = [&](int q, float4 g, float4 c, float4 sh, const float4* lp) {
        const float4 x = xs4[q];
        float4 xn;
        xn.x = norm(x.x, g.x, c.x); xn.y = norm(x.y, g.y, c.y);
        xn.z = norm(x.z, g.z, c.z); xn.w = norm(x.w, g.w, c.w);
        if (mix1) {
            float4 d;
            d.x = sh.x - xn.x; d.y = sh.y - xn.y; d.z = sh.z - xn.z; d.w = sh.w - xn.w;
#pragma unroll
            for (int s6 = 0; s6 < 6; ++s6) {
                float4 r;
                r.x = xn.x + lp[s6].x * d.x; r.y = xn.y + lp[s6].y * d.y;
                r.z = xn.z + lp[s6].z * d.z; r.w = xn.w + lp[s6].w * d.w;
                put(A.out + s6 * mat, q, r);
            }
            sh4[q] = xn;
        } else if (mix2) {
            float4 r;
            r.x = xn.x + lp[0].x * (sh.x - xn.x); r.y = xn.y + lp[0].y * (sh.y - xn.y);
            r.z = xn.z + lp[0].z * (sh.z - xn.z); r.w = xn.w + lp[0].w * (sh.w - xn.w);
            put(A.out, q, r);
            sh4[q] = xn;
        } else if (A.mode == RKQ_LN_PLAIN) {
            put(A.out, q, xn);
        } else {
            reinterpret_cast<float4*>(A.out)[(size_t)b * n4 + q] = xn;
        }
    };
    if (regs) {
#pragma unroll
        for (int j = 0; j < kLnQ; ++j) {
            const int q = t + LT * j;
            if (q < n4) {
                const float4 lp[6] = {lv[0][j], lv[1][j], lv[2][j], lv[3][j], lv[4][j], lv[5][j]};
                emit(q, gv[j], cv[j], sv[j], lp);
            }
        }
    } else {
        for (int q = t; q < n4; q += LT) {   // longer rows: parameters loaded as used
            float4 lp[6], sh = make_float4(0.f, 0.f, 0.f, 0.f);
            if (mix1 || mix2) sh = sh4[q];
            if (mix1) {
                for (int s6 = 0; s6 < 6; ++s6) lp[s6] = l4[(size_t)s6 * n4 + q];
            } else if (mix2) {
                lp[0] = l4[q];
            }
            emit(q, g4[q], c4[q], sh, lp);
        }
    }
}

// ------------------------------------------------------------- products
// Y[b] = W X[b], every output the reference's chain acc = fmaf(x[k], w[k], acc)
// over k in order. v_mfma_f32_16x16x4_f32 adds its four products one after the
// other, each with one rounding, lowest k first (checked on gfx950: 51,200
// random outputs of it, and of 32x32x2, equal the sequential fmaf chain bit for
// bit, none equals another order or a single rounding throughout), so a chain
// of them in k order is that chain. A dependent one issues every 36 cycles, 9
// per input (4x4x1 chains: 13 to 19), and a wave holds only 16 outputs x 16
// sequences per chain, so a batch of 16 already spreads over many waves.
//
// One wave per 16 O outputs x 16 S sequences, one wave per workgroup, nothing
// shared and no barrier. Lane (n, g) = (l % 16, l / 16) supplies input 4 i + g
// of step i: output n's weight (A) and sequence n's x (B), and then holds
// outputs 4 g .. 4 g + 3 of sequence n. With one wave per SIMD a chain leaves
// room for about six other instructions per MFMA (one issues every ~5.4
// cycles), so both operands come in the order the steps use them (x16_at): one
// coalesced 1 KiB load each per 16 inputs, PF of them ahead in registers. Every
// producer writes its rows that way, and a product's own outputs are in that
// order already. The first version, which dequantized INT4 codes and transposed
// row-major x in the wave (11 instructions per MFMA), took 28 us for the
// channel-mix value at B = 64; this one takes 15 (the 4x4x1 chains it replaced:
// 26). The step at B = 64: 1,350 -> 1,030 us (12 x 768 INT4 g32); a 512-token
// prefill chunk, kernels, 4.8 -> 3.4 ms (2.9 since the recurrence's interleaving).
//
// Weights (BLK): -1, tiled fp32 copies of the layer matrices, made at load
// (k_rkq_tile); 32 / 64, INT4 codes: byte g of dword i of a group is exactly
// lane group g's input, so the wave dequantizes its operand in registers
// (fma(q, s, -8 s), quant.c's (q - 8) s), which the vocabulary head's eight
// chains hide; 0, fp32 rows, transposed between the lane groups.
struct RkqMMArgs {
    RkqJob j[kRkqMaxJobs];
    int start[kRkqMaxJobs + 1];   // first workgroup of each job
    int n, B, seq_tiles;
};

// One weight, as the products multiply it.
__device__ __forceinline__ float dequant_at(const RkqJob& J, int row, int k, int blk) {
    if (blk < 0) return J.w[x16_at(row, k, (J.Kd + 15) / 16)];
    if (!blk) return J.w[(size_t)row * J.Kd + k];
    const int half = blk / 2, g = k / blk, e = k % blk;
    const uint8_t byte = J.q[(size_t)row * (J.Kd / 2) + (size_t)g * half + (e % half)];
    const float sc = J.sc[(size_t)row * (J.Kd / blk) + g];
    const int qv = e < half ? (byte & 0x0F) : (byte >> 4);
    return fmaf((float)qv, sc, -8.0f * sc);
}

// This workgroup's job (uniform selects: no dynamic index into the arguments).
// The first workgroup of the job is selected in the same pass as the job
// index: selecting it by index afterwards was folded back into an indexed
// read of a local copy of start[], which the compiler kept in scratch memory
// (a store and a dependent load at every launch).
__device__ __forceinline__ void rkq_job_at(const RkqMMArgs& A, int wg, RkqJob& J, int& u0) {
    int ji = 0, j0 = A.start[0];
#pragma unroll
    for (int i = 1; i < kRkqMaxJobs; ++i)
        if (i < A.n && wg >= A.start[i]) { ji = i; j0 = A.start[i]; }
    J = A.j[0];
#pragma unroll
    for (int i = 1; i < kRkqMaxJobs; ++i)
        if (i == ji) J = A.j[i];
    u0 = wg - j0;
}

__device__ __forceinline__ float rkq_epi(int epi, float y, float v) {
    switch (epi) {
    case RKQ_ADD: return y + v;
    case RKQ_RELU2: { const float r = v > 0.0f ? v : 0.0f; return r * r; }
    case RKQ_TANH: return refmath::tanhf(v);
    case RKQ_SIGMOID: return refmath::sigmoid(v);
    default: return v;
    }
}

// A lane's outputs out0 .. out0 + 3 (out0 % 4 == 0) of sequence sq: columns
// past the last multiple of 8 take the reference's scalar tail (acc + x * w,
// two roundings), then the epilogue. In x16 order the outputs that pad the last
// block of 16 are written as zeros.
__device__ __forceinline__ void rkq_finish(const RkqJob& J, int B, int blk, int sq, int out0, v4f acc) {
    if (sq >= B || out0 >= (J.M + 15) / 16 * 16) return;
    if (out0 + 4 > (J.M & ~7)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int out = out0 + i;
            if (out < (J.M & ~7) || out >= J.M) continue;
            float v = 0.0f;
            for (int k = 0; k < J.Kd; ++k)
                v = v + J.X[x16_at(sq, k, (J.Kd + 15) / 16)] * dequant_at(J, out, k, blk);
            acc[i] = v;
        }
    }
    if (J.y16) {   // never RKQ_ADD
        float* y = J.Y + x16_at(sq, out0, (J.M + 15) / 16);
#pragma unroll
        for (int i = 0; i < 4; ++i) y[64 * i] = out0 + i < J.M ? rkq_epi(J.epi, 0.0f, acc[i]) : 0.0f;
        return;
    }
    float* y = J.Y + (size_t)sq * J.ldy + out0;
    if (out0 + 4 <= J.M && ((reinterpret_cast<uintptr_t>(J.Y) | (uintptr_t)J.ldy * 4) & 15) == 0) {
        v4f old = v4f{0.f, 0.f, 0.f, 0.f};
        if (J.epi == RKQ_ADD) old = *reinterpret_cast<const v4f*>(y);
        v4f r;
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = rkq_epi(J.epi, old[i], acc[i]);
        *reinterpret_cast<v4f*>(y) = r;
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (out0 + i < J.M) y[i] = rkq_epi(J.epi, J.epi == RKQ_ADD ? y[i] : 0.0f, acc[i]);
}

// r[j] of lane group g <- r[g] of lane group j (groups of 16 lanes).
__device__ __forceinline__ void group_transpose(float (&r)[4]) {
    auto swap32 = [](float& a, float& b) {
        const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        a = __uint_as_float(p[0]);
        b = __uint_as_float(p[1]);
    };
    auto swap16 = [](float& a, float& b) {
        const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        a = __uint_as_float(p[0]);
        b = __uint_as_float(p[1]);
    };
    swap32(r[0], r[2]);
    swap32(r[1], r[3]);
    swap16(r[0], r[1]);
    swap16(r[2], r[3]);
}

// A copy the compiler cannot merge with its source: the swaps of the transpose
// work in place, and the copies it would make itself, of a loaded group's
// registers, it placed right behind the load, where they wait for it.
__device__ __forceinline__ float fresh(float v) {
    float r;
    asm("v_mov_b32 %0, %1" : "=v"(r) : "v"(v));
    return r;
}

// A unit's weights of a lane for one output tile: 16 inputs of fp32, or one
// INT4 group.
template <int BLK> struct RkqW { uint4 q[BLK / 32]; float sc; };
template <> struct RkqW<0> { float4 w; };
template <> struct RkqW<-1> { float4 w; };

template <int BLK, int O, int S, int PF>
__global__ __launch_bounds__(64) void k_rkq_mm(const RkqMMArgs A) {
    constexpr int U = BLK > 0 ? BLK : 16, UB = U / 16;   // inputs and 16-input blocks of a unit
    // Consecutive numbers run on one XCD (dispatch is round-robin over the 8):
    // an output tile's sequence tiles read its weights from one L2.
    const int T = (int)gridDim.x, b = (int)blockIdx.x, q8 = T / 8, r8 = T % 8, x8 = b % 8;
    RkqJob J;
    int u0;
    rkq_job_at(A, x8 * q8 + min(x8, r8) + b / 8, J, u0);
    const int ot = u0 / A.seq_tiles * O, st = u0 % A.seq_tiles * S;
    const int l = threadIdx.x, n = l & 15, g = l >> 4;
    const int Kd = J.Kd, nkb = (Kd + 15) / 16, nu = (Kd + U - 1) / U;
    const int mt = (J.M + 15) / 16, xt = (A.B + 15) / 16;   // output and sequence tiles there are
    // x (and tiled weights) through buffer resources: block kb of tile t is the
    // KiB at scalar offset (t nkb + kb) 1024, lane l's float4 at 16 l. Tiles
    // past the end read the last one; their results are never stored.
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(J.X), (short)0, (int)((uint32_t)xt * nkb * 1024u), 0x00020000);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(J.w), (short)0, (int)(BLK < 0 ? (uint32_t)mt * nkb * 1024u : 0u), 0x00020000);
    auto ldf = [&](const __amdgpu_buffer_rsrc_t& r, int so) -> float4 {
        const u32x4v v = __builtin_amdgcn_raw_buffer_load_b128(r, 16 * l, so, 0);
        return make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3]));
    };
    int xo[S], wo[O];
    const float* wr[O];
    const uint8_t* qr[O];
    const float* sr[O];
#pragma unroll
    for (int s = 0; s < S; ++s) xo[s] = min(st + s, xt - 1) * nkb * 1024;
#pragma unroll
    for (int o = 0; o < O; ++o) {
        wo[o] = min(ot + o, mt - 1) * nkb * 1024;
        const int row = min((ot + o) * 16 + n, J.M - 1);
        wr[o] = BLK == 0 ? J.w + (size_t)row * Kd : nullptr;
        qr[o] = BLK > 0 ? J.q + (size_t)row * (size_t)(Kd / 2) : nullptr;
        sr[o] = BLK > 0 ? J.sc + (size_t)row * (size_t)(Kd / U) : nullptr;
    }
    RkqW<BLK> w[PF][O];
    float4 x[PF][S][UB];
    auto load = [&](int p, int u_) {
        const int u = min(u_, nu - 1);               // past the end: the last unit again, never used
#pragma unroll
        for (int o = 0; o < O; ++o) {
            if constexpr (BLK < 0) {
                w[p][o].w = ldf(rw, wo[o] + u * 1024);
            } else if constexpr (BLK == 0) {
                w[p][o].w = *reinterpret_cast<const float4*>(wr[o] + min(u * U + 4 * g, Kd - 4));
            } else {
#pragma unroll
                for (int i = 0; i < BLK / 32; ++i)
                    w[p][o].q[i] = *reinterpret_cast<const uint4*>(qr[o] + u * (BLK / 2) + 16 * i);
                w[p][o].sc = sr[o][u];
            }
        }
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int i = 0; i < UB; ++i) x[p][s][i] = ldf(rx, xo[s] + (u * UB + i) * 1024);
    };
    v4f acc[O][S];
#pragma unroll
    for (int o = 0; o < O; ++o)
#pragma unroll
        for (int s = 0; s < S; ++s) acc[o][s] = v4f{0.f, 0.f, 0.f, 0.f};
    auto unit = [&](int p, int u) {
#pragma unroll
        for (int i = 0; i < UB; ++i) {
            float wv[O][4];
#pragma unroll
            for (int o = 0; o < O; ++o) {
                if constexpr (BLK < 0) {
                    const float4 v = w[p][o].w;
                    wv[o][0] = v.x; wv[o][1] = v.y; wv[o][2] = v.z; wv[o][3] = v.w;
                } else if constexpr (BLK == 0) {
                    const bool in = u * U + 4 * g < Kd;   // a short last unit is padded with zeros
                    const float4 v = w[p][o].w;
                    wv[o][0] = in ? fresh(v.x) : 0.0f; wv[o][1] = in ? fresh(v.y) : 0.0f;
                    wv[o][2] = in ? fresh(v.z) : 0.0f; wv[o][3] = in ? fresh(v.w) : 0.0f;
                    group_transpose(wv[o]);
                } else {
                    // step 4 i + j: dword 4 i + j of the low nibbles, then of the high
                    constexpr int HB = UB / 2;
                    const float sc = w[p][o].sc, m8 = -8.0f * sc;
                    const uint4 q = w[p][o].q[i % HB];
                    const uint32_t sh = 8 * g + (i < HB ? 0 : 4);
                    wv[o][0] = fmaf((float)((q.x >> sh) & 0xFu), sc, m8);
                    wv[o][1] = fmaf((float)((q.y >> sh) & 0xFu), sc, m8);
                    wv[o][2] = fmaf((float)((q.z >> sh) & 0xFu), sc, m8);
                    wv[o][3] = fmaf((float)((q.w >> sh) & 0xFu), sc, m8);
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int o = 0; o < O; ++o)
#pragma unroll
                    for (int s = 0; s < S; ++s) {
                        const float4 v = x[p][s][i];
                        const float xv = j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w;
                        acc[o][s] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[o][j], xv, acc[o][s], 0, 0, 0);
                    }
        }
    };
#pragma unroll
    for (int p = 0; p < PF; ++p) load(p, p);
    int ub = 0;
    for (; ub + PF <= nu; ub += PF) {
#pragma unroll
        for (int p = 0; p < PF; ++p) {
            unit(p, ub + p);
            load(p, ub + p + PF);
            __builtin_amdgcn_sched_barrier(0);       // a unit's loads stay with it
        }
    }
#pragma unroll
    for (int p = 0; p < PF; ++p)
        if (ub + p < nu) unit(p, ub + p);
#pragma unroll
    for (int o = 0; o < O; ++o)
#pragma unroll
        for (int s = 0; s < S; ++s)
            rkq_finish(J, A.B, BLK, (st + s) * 16 + n, (ot + o) * 16 + 4 * g, acc[o][s]);
}

// The tiled fp32 form of an M x Kd matrix: x16 order with the output in the
// row's place, each value the one the products use, zeros past Kd; rows past M
// repeat row M - 1.
__global__ __launch_bounds__(256) void k_rkq_tile(RkqJob J, int blk, float* out) {
    const int nkb = (J.Kd + 15) / 16;
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)((J.M + 15) / 16) * nkb * 256) return;
    const int j = i & 3, l = (i >> 2) & 63;
    const size_t t = i >> 8;
    const int k = (int)(t % nkb) * 16 + 4 * j + (l >> 4), row = min((int)(t / nkb) * 16 + (l & 15), J.M - 1);
    out[i] = k < J.Kd ? dequant_at(J, row, k, blk) : 0.0f;
}

// ---------------------------------------------------------------- heads
// One group of an INT4 row (BLK inputs; the codes in BLK / 32 chunks of 16
// bytes, scale sc) on top of acc: acc = fmaf(x[i], w[i], acc) for i in order,
// w[i] dequantized as fma(q, sc, -8 sc) (dequant_at's value). Input i is
// byte i % (BLK / 2) of the group, low nibble for the first half.
template <int BLK>
__device__ __forceinline__ float up_group(float acc, const uint4* qv, float sc, const float* x) {
    constexpr int HALF = BLK / 2;
    const float m8 = -8.0f * sc;
#pragma unroll
    for (int i = 0; i < BLK; ++i) {
        const int bi = i % HALF, ch = bi / 16, by = bi % 16;
        const uint32_t word = by < 4 ? qv[ch].x : by < 8 ? qv[ch].y : by < 12 ? qv[ch].z : qv[ch].w;
        const uint32_t bt = (word >> (8 * (by % 4))) & 0xFFu;
        const uint32_t q = i < HALF ? (bt & 0xFu) : (bt >> 4);
        acc = fmaf(x[i], fmaf((float)q, sc, m8), acc);
    }
    return acc;
}

// LoRA up-projection m of channel c for sequence b (see RkqHeadArgs): every
// code chunk is loaded first (up to 4, clamped so that no load depends on the
// rank), then the output is one sequential chain from 0 over its inputs, as
// the products compute it.
template <int BLK>
__device__ __forceinline__ float up_one(const RkqHeadArgs& A, int b, int c, int m) {
    constexpr int NQ = BLK / 32, CH = 4;   // chunks per group; chunks per matrix at most
    // rank 0 (layer 0's v2 slot, naming another matrix): one group's loads of
    // row c of that matrix, in bounds, never used
    const int Kr = A.up_k[m], K = Kr > 0 ? Kr : BLK, nch = K / 32;
    const uint4* q = reinterpret_cast<const uint4*>(A.up_q[m] + (size_t)c * (size_t)(K / 2));
    const float* sp = A.up_sc[m] + (size_t)c * (size_t)(K / BLK);
    uint4 qv[CH];
    float sc[CH / NQ];
#pragma unroll
    for (int j = 0; j < CH; ++j) qv[j] = q[min(j, nch - 1)];
#pragma unroll
    for (int g = 0; g < CH / NQ; ++g) sc[g] = sp[min(g, K / BLK - 1)];
    float acc = 0.0f;
    const float* x = A.up_x[m] + (size_t)b * (size_t)A.up_ldx;
#pragma unroll
    for (int g = 0; g < CH / NQ; ++g)
        if (g < Kr / BLK) acc = up_group<BLK>(acc, &qv[g * NQ], sc[g], x + g * BLK);
    return acc;
}

// NWV = 4 (the up-projections fused in): waves 1..3 compute them into LDS
// (wave 1: w2; wave 2: a2, then v2; wave 3: g2) while wave 0 loads its state
// row; after one workgroup barrier they end and wave 0 runs the rest alone.
// NWV = 1: one wave, the up-projections read from dw, da, g, dv.
template <int NWV>
__global__ __launch_bounds__(64 * NWV) void k_rkq_heads(RkqHeadArgs A) {
    __shared__ float w_[kHS], k_[kHS], v_[kHS], a_[kHS], kn_[kHS], r_[kHS], y_[kHS], dt_[kHS],
        sq_[kHS], part[8], stat[3];
    __shared__ float upv[NWV > 1 ? 4 : 1][kHS];
    const int h = blockIdx.x, b = blockIdx.y, t = threadIdx.x & 63;
    // The workgroup's syncs after the up-projections: with NWV > 1 wave 0 is
    // the only wave left, and its LDS operations complete in program order,
    // so a fence that keeps the compiler from moving them across is enough
    // (no barrier waits on the waves that have ended).
    auto sync = [] {
        if constexpr (NWV > 1) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        } else {
            __syncthreads();
        }
    };
    const size_t row = (size_t)b * A.D;
    const int c = h * kHS + t;
    if constexpr (NWV > 1) {
        const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        if (wv != 0) {
            auto one = [&](int m) {
                upv[m][t] = A.up_blk == 32 ? up_one<32>(A, b, c, m) : up_one<64>(A, b, c, m);
            };
            if (wv == 1) one(0);
            else if (wv == 2) { one(1); one(3); }
            else one(2);
            __syncthreads();
            return;
        }
    }
    // Every input of the wave is loaded before any is used: the state row,
    // the channel's products and parameters, and the epilogue's.
    float* Sr = A.S + (size_t)b * A.s_bstride + (size_t)h * kHS * kHS + (size_t)t * kHS;
    float s[kHS];
#pragma unroll
    for (int q = 0; q < kHS; q += 4) {
        const float4 v4 = *reinterpret_cast<const float4*>(Sr + q);
        s[q] = v4.x; s[q + 1] = v4.y; s[q + 2] = v4.z; s[q + 3] = v4.w;
    }
    float dw, da, dv, gv;
    if constexpr (NWV > 1) {
        __syncthreads();   // the up-projections in
        dw = upv[0][t]; da = upv[1][t]; gv = upv[2][t]; dv = A.first ? 0.0f : upv[3][t];
        A.g_out[row + c] = gv;
    } else {
        dw = A.dw[row + c]; da = A.da[row + c]; gv = A.g[row + c];
        dv = A.first ? 0.0f : A.dv[row + c];
    }
    const float w0 = A.w0[c], v_in = A.v[row + c];
    const float vf = A.first ? 0.0f : A.vfirst[row + c];
    const float v0 = A.v0[c], a0 = A.a0[c], kv = A.k[row + c];
    const float kkw = A.kk_w[c], kaw = A.ka_w[c], rv = A.r[row + c], rkw = A.rk_w[c];
    const float lnw = A.lnx_w[c], lnb = A.lnx_b[c];
    // Channel terms (rwkv7.c:236-260).
    const float ww = refmath::expf(-refmath::sigmoid(dw + w0) * kR2);
    float vv = v_in;
    if (A.first) {
        A.vfirst[row + c] = vv;
    } else {
        const float mix = refmath::sigmoid(dv + v0);
        vv = vv + (vf - vv) * mix;
    }
    const float av = refmath::sigmoid(da + a0);
    const float kkv = kv * kkw;
    const float k2 = kv + kv * (av - 1.0f) * kaw;
    if (A.dbg && b == 0) {
        A.dbg[(size_t)2 * A.D + c] = k2;
        A.dbg[(size_t)3 * A.D + c] = vv;
        A.dbg[(size_t)4 * A.D + c] = av;
        A.dbg[(size_t)6 * A.D + c] = ww;
    }
    w_[t] = ww; k_[t] = k2; v_[t] = vv; a_[t] = av; kn_[t] = kkv; r_[t] = rv;
    dt_[t] = rv * k2 * rkw;
    sync();
    // |kk|: eight stride-8 partial sums of squares (rwkv7.c:156-162).
    if (t < 8) {
        float ss = 0.0f;
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const float e = kn_[8 * m + t];
            ss = fmaf(e, e, ss);
        }
        part[t] = ss;
    }
    sync();
    if (t == 0) {
        float nrm = sqrtf(hsum8(part));
        if (!(nrm > 1e-12f)) nrm = 1e-12f;
        stat[0] = 1.0f / nrm;
    }
    sync();
    const float kn = kkv * stat[0];
    sync();
    kn_[t] = kn;
    sync();
    // State row t (rwkv7.c:165-187).
    float proj[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < kHS; j += 8)
#pragma unroll
        for (int q = 0; q < 8; ++q) proj[q] = fmaf(s[j + q], kn_[j + q], proj[q]);
    const float pv = hsum8(proj);
    float yacc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < kHS; j += 8)
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const float kka = kn_[j + q] * a_[j + q];
            const float vk = vv * k_[j + q];
            const float ns = fmaf(s[j + q], w_[j + q], vk - pv * kka);
            s[j + q] = ns;
            yacc[q] = fmaf(ns, r_[j + q], yacc[q]);
        }
#pragma unroll
    for (int q = 0; q < kHS; q += 4)
        *reinterpret_cast<float4*>(Sr + q) = make_float4(s[q], s[q + 1], s[q + 2], s[q + 3]);
    y_[t] = hsum8(yacc);
    sync();
    // Group norm, bonus, gate (rwkv7.c:266-288): the mean and the bonus dot
    // as sequential sums (lanes 0 and 1 side by side), then the variance.
    if (t < 2) {
        const float* src = t == 0 ? y_ : dt_;
        float acc = 0.0f;
#pragma unroll 8
        for (int i = 0; i < kHS; ++i) acc = acc + src[i];
        stat[1 + t] = acc;
    }
    sync();
    const float mean = stat[1] / (float)kHS, dot = stat[2];
    const float yy = y_[t];
    const float dd = yy - mean;
    sq_[t] = dd * dd;
    sync();
    if (t == 0) {
        float var = 0.0f;
#pragma unroll 8
        for (int i = 0; i < kHS; ++i) var = var + sq_[i];
        stat[0] = 1.0f / sqrtf(var / (float)kHS + kEpsGroup);
    }
    sync();
    const float n = (yy - mean) * stat[0] * lnw + lnb;
    const float yg = (n + dot * vv) * gv;
    A.y[x16_at(b, c, A.D / 16)] = yg;
    if (A.dbg && b == 0) A.dbg[(size_t)7 * A.D + c] = yg;
}

__global__ void k_refmath(const float* __restrict__ x, float* __restrict__ e, float* __restrict__ th,
                          int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        e[i] = refmath::expf(x[i]);
        th[i] = refmath::tanhf(x[i]);
    }
}

}  // namespace

snhip_status launch_rkq_ln(const RkqLnArgs& a, int B, hipStream_t st) {
    if (a.D <= 0 || a.D > kLnMax || a.D % 16 || B <= 0) return SNHIP_E_INVAL;
    hipLaunchKernelGGL(k_rkq_ln<kLnT>, dim3(B), dim3(kLnT), 0, st, a);
    SNHIP_CHECK(hipGetLastError());
    return SNHIP_OK;
}

snhip_status launch_rkq_heads(const RkqHeadArgs& a, int B, hipStream_t st) {
    if (a.D != a.NH * kHS || B <= 0) return SNHIP_E_INVAL;
    if (a.up_blk) {
        if ((a.up_blk != 32 && a.up_blk != 64) || !a.g_out) return SNHIP_E_INVAL;
        // every slot names a matrix the loads may read (an unused v2 slot in
        // layer 0: any of the others, rank 0, so its chain is empty)
        for (int m = 0; m < 4; ++m) {
            const int K = a.up_k[m];
            if (!a.up_q[m] || !a.up_sc[m] || !a.up_x[m] || K < 0 || K > 128 || K % a.up_blk ||
                (K == 0 && !(m == 3 && a.first)))
                return SNHIP_E_INVAL;
        }
    }
    if (a.up_blk) hipLaunchKernelGGL(k_rkq_heads<4>, dim3(a.NH, B), dim3(256), 0, st, a);
    else hipLaunchKernelGGL(k_rkq_heads<1>, dim3(a.NH, B), dim3(64), 0, st, a);
    SNHIP_CHECK(hipGetLastError());
    return SNHIP_OK;
}

// Compute units of the current device (queried once per device).
int cu_count() {
    static int cached[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (!cached[dev]) {
        int n = 0;
        cached[dev] = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0
                          ? n
                          : 256;
    }
    return cached[dev];
}

snhip_status launch_rkq_mm(const RkqJob* jobs, int n, int B, int block, hipStream_t st) {
    if (n <= 0 || n > kRkqMaxJobs || B <= 0 || (block != -1 && block != 0 && block != 32 && block != 64))
        return SNHIP_E_INVAL;
    RkqMMArgs a{};
    const long seqs = (B + 15) / 16;
    for (int i = 0; i < n; ++i) {
        const RkqJob& J = jobs[i];
        if (J.M <= 0 || J.Kd <= 0 || J.Kd % (block > 0 ? block : 4) || !J.X || !J.Y ||
            (block > 0 ? (!J.q || !J.sc) : !J.w) || (J.y16 && J.epi == RKQ_ADD) ||
            seqs * ((J.Kd + 15) / 16) >= (1 << 21))   // x within 32-bit offsets
            return SNHIP_E_INVAL;
        a.j[i] = J;
    }
    // Output x sequence tiles per wave: the fewest rounds of chains over the
    // SIMDs (four per CU; each runs its waves' chains at 8 cycles per input, a
    // lone chain at 9); where shapes come out even, the larger one reads its
    // operands less often.
    const long simds = 4L * cu_count();
    static constexpr int kShape[4][2] = {{1, 1}, {1, 2}, {2, 2}, {2, 4}};
    int shape = 0;
    double best = 0.0;
    auto waves = [&](int i) { return (jobs[i].M + 15) / 16; };
    for (int h = 0; h < 4; ++h) {
        const int O = kShape[h][0], S = kShape[h][1];
        long tiles = 0;
        for (int i = 0; i < n; ++i) tiles += (waves(i) + O - 1) / O;
        const long rounds = (tiles * ((seqs + S - 1) / S) + simds - 1) / simds;
        const double cost = rounds * O * S == 1 ? 1.125 : (double)(rounds * O * S);
        if (h == 0 || cost <= best) { shape = h; best = cost; }
    }
    // SNHIP_RKQ_SHAPE=0..3 pins one (tests).
    if (const char* e = getenv("SNHIP_RKQ_SHAPE")) shape = std::min(3u, (unsigned)atoi(e));
    const int O = kShape[shape][0], S = kShape[shape][1];
    a.n = n;
    a.B = B;
    a.seq_tiles = (int)((seqs + S - 1) / S);
    int total = 0;
    for (int i = 0; i < n; ++i) {
        a.start[i] = total;
        total += (waves(i) + O - 1) / O * a.seq_tiles;
    }
    for (int i = n; i <= kRkqMaxJobs; ++i) a.start[i] = total;
#define SNHIP_RKQ(B_, O_, S_, P_) hipLaunchKernelGGL((k_rkq_mm<B_, O_, S_, P_>), dim3(total), dim3(64), 0, st, a)
    // read-ahead: about 100 registers of operands per wave
#define SNHIP_RKQ4(B_, P0, P1, P2, P3)              \
    do {                                            \
        if (shape == 0) SNHIP_RKQ(B_, 1, 1, P0);    \
        else if (shape == 1) SNHIP_RKQ(B_, 1, 2, P1); \
        else if (shape == 2) SNHIP_RKQ(B_, 2, 2, P2); \
        else SNHIP_RKQ(B_, 2, 4, P3);               \
    } while (0)
    if (block < 0) SNHIP_RKQ4(-1, 16, 8, 6, 4);
    else if (block == 0) SNHIP_RKQ4(0, 12, 8, 6, 4);
    else if (block == 32) SNHIP_RKQ4(32, 8, 4, 3, 2);
    else SNHIP_RKQ4(64, 4, 3, 2, 1);
#undef SNHIP_RKQ4
#undef SNHIP_RKQ
    SNHIP_CHECK(hipGetLastError());
    return SNHIP_OK;
}

snhip_status launch_rkq_tile(const float* w, const uint8_t* q, const float* sc, int block, int M, int Kd,
                             float* out, hipStream_t st) {
    if (M <= 0 || Kd <= 0 || Kd % 4 || !out || (block != 0 && block != 32 && block != 64) ||
        (block ? (!q || !sc || Kd % block) : !w))
        return SNHIP_E_INVAL;
    RkqJob J{};
    J.w = w; J.q = q; J.sc = sc; J.M = M; J.Kd = Kd;
    hipLaunchKernelGGL(k_rkq_tile, dim3((unsigned)((x16_floats(M, Kd) + 255) / 256)), dim3(256), 0, st, J, block, out);
    SNHIP_CHECK(hipGetLastError());
    return SNHIP_OK;
}

}  // namespace snhip

extern "C" {

snhip_status snhip_refmath_host(const float* x, float* e, float* t, int32_t n) {
    if (!x || !e || !t || n <= 0) return SNHIP_E_INVAL;
    for (int32_t i = 0; i < n; ++i) {
        e[i] = snhip::refmath::expf(x[i]);
        t[i] = snhip::refmath::tanhf(x[i]);
    }
    return SNHIP_OK;
}

snhip_status snhip_refmath_dev(const float* x, float* e, float* t, int32_t n, void* stream) {
    if (!x || !e || !t || n <= 0) return SNHIP_E_INVAL;
    hipLaunchKernelGGL(snhip::k_refmath, dim3((n + 255) / 256), dim3(256), 0,
                       snhip::as_stream(stream), x, e, t, n);
    SNHIP_CHECK(hipGetLastError());
    return SNHIP_OK;
}

}  // extern "C"
