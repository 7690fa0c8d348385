// Chunked RWKV-7 prefill kernels (rkseq.h): a chunk of T consecutive tokens of
// one sequence as T rows, every rounding in the reference's order
// (sunnynet/runtime/rwkv7.c:127-320), so that the chunk leaves the bits that
// stepping its tokens one by one leaves.
//
// Of a layer only the 64 x 64 state recurrence runs token after token. The
// products take all T rows at once (launch_rkq_mm: each output keeps its own
// input-ordered chain), LayerNorm and token shift need only the row before, and
// everything of a head that does not read the state (decay, value residual,
// in-context rate, normalized kk, bonus dot; then group norm, bonus and gate) is
// one wave per (token, head). What is left for the recurrence is 8 multiply-adds
// of the read, one of the update and 8 of the read-out per state element.
//
// Measured (12 x 768, INT4 g32, 512-token prompt): 2.85 ms of kernels (products 1.31,
// recurrence 1.01, LayerNorms 0.34), 4.0 ms a call with the state read and the host's
// copy of the logits, where the token-by-token prefill took 345 ms (512 one-launch
// steps of 673 us).
#include <algorithm>
#include <type_traits>

#include "lanesum.h"
#include "refmath.h"
#include "rkseq.h"

namespace snhip {
namespace {

constexpr float kR2 = 0.6065306597126334f;   // 1/sqrt(e), rwkv7.c:38
constexpr float kEpsGroup = 6.4e-4f;          // rwkv7.c:39
constexpr int kHS = 64;
typedef unsigned int u32x4v __attribute__((ext_vector_type(4)));

// The wave's own LDS operations complete in order; this keeps the compiler
// from moving them across.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Row LayerNorm and token shift of kLnRows tokens per workgroup. Wave w
// normalizes row 3 blockIdx - 1 + w (wave 0's row belongs to the workgroup
// before and is normalized again here: its values are the first mix's previous
// token, and the sums are latency, not throughput), so a mix reads its
// neighbour from LDS and the layer needs no second pass. The row before the
// chunk is the carried shift vector; the chunk's last row goes to shift_next,
// not to the shift vector itself, which other workgroups of the launch read.
constexpr int kLnRows = 3;

// KL4: float4 per lane of the lane-sliced sums (rows of 256 KL4 values), 0 for
// any other length (one lane sums the row).
template <int KL4>
__global__ __launch_bounds__(64 * (kLnRows + 1)) void k_rkp_ln(RkpLnArgs A) {
    extern __shared__ float4 rows4[];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
    const int D = A.D, n4 = D / 4;
    const int row = (int)blockIdx.x * kLnRows - 1 + w;
    float4* own = rows4 + (size_t)w * n4;
    const float4* g4 = reinterpret_cast<const float4*>(A.g);
    const float4* c4 = reinterpret_cast<const float4*>(A.c);
    if (row < 0) {
        const float4* s4 = reinterpret_cast<const float4*>(A.shift);
        for (int q = l; q < n4; q += 64) own[q] = s4[q];
    } else if (row < A.T) {
        const float4* x4 = reinterpret_cast<const float4*>(A.x + (size_t)row * D);
        for (int q = l; q < n4; q += 64) own[q] = x4[q];
        wave_sync();
        float mean, rstd;
        if constexpr (KL4 > 0) {
            float v[4 * KL4];
#pragma unroll
            for (int q = 0; q < KL4; ++q) {
                const float4 x = own[l * KL4 + q];
                v[4 * q] = x.x; v[4 * q + 1] = x.y; v[4 * q + 2] = x.z; v[4 * q + 3] = x.w;
            }
            lane_ln_stats(v, D, A.eps, mean, rstd);
        } else {
            // every lane the same sums (reads of one address)
            float s = 0.0f;
            for (int q = 0; q < n4; ++q) {
                const float4 x = own[q];
                s = s + x.x; s = s + x.y; s = s + x.z; s = s + x.w;
            }
            mean = s / (float)D;
            s = 0.0f;
            for (int q = 0; q < n4; ++q) {
                const float4 x = own[q];
                float d = x.x - mean;
                s = s + d * d;
                d = x.y - mean;
                s = s + d * d;
                d = x.z - mean;
                s = s + d * d;
                d = x.w - mean;
                s = s + d * d;
            }
            rstd = 1.0f / sqrtf(s / (float)D + A.eps);
        }
        wave_sync();
        auto norm = [&](float x, float g, float c) { return (x - mean) * rstd * g + c; };
        for (int q = l; q < n4; q += 64) {
            const float4 x = own[q], g = g4[q], c = c4[q];
            own[q] = make_float4(norm(x.x, g.x, c.x), norm(x.y, g.y, c.y), norm(x.z, g.z, c.z),
                                 norm(x.w, g.w, c.w));
        }
    }
    __syncthreads();
    if (w == 0 || row >= A.T) return;
    const float4* prev = rows4 + (size_t)(w - 1) * n4;
    const float4* l4 = reinterpret_cast<const float4*>(A.lerp);
    const size_t mat = x16_floats(A.T, D);
    float4* nx = row == A.T - 1 ? reinterpret_cast<float4*>(A.shift_next) : nullptr;
    for (int q = l; q < n4; q += 64) {
        const float4 xn = own[q], p = prev[q];
        const float4 d = make_float4(p.x - xn.x, p.y - xn.y, p.z - xn.z, p.w - xn.w);
        for (int s = 0; s < A.mixes; ++s) {
            const float4 lp = l4[(size_t)s * n4 + q];
            float* o = A.out + s * mat + x16_at(row, 4 * q, D / 16);   // the four inputs are 64 floats apart
            o[0] = xn.x + lp.x * d.x;
            o[64] = xn.y + lp.y * d.y;
            o[128] = xn.z + lp.z * d.z;
            o[192] = xn.w + lp.w * d.w;
        }
        if (nx) nx[q] = xn;
    }
}

// Lane `lam` of a state row's eight (k_rkp_scan) owns columns 8 m + q, q = its
// partial sum's index: 0 1 2 3 7 6 5 4 over the lanes, so that the fold
// ((0+4)+(1+5))+((2+6)+(3+7)) is a half-row mirror and two quad permutes.
__device__ __forceinline__ int lam_of(int q) { return q < 4 ? q : 11 - q; }

// One wave per (token, head), four tokens per workgroup: everything of the
// head that does not read the state (the arithmetic of k_rkq_heads, channel j
// in lane j). w, kn, kn a, k and r go to `pack`, 64 values each with column
// 8 m + q at 8 lam_of(q) + m: a lane of the recurrence reads its eight columns
// as two float4.
__global__ __launch_bounds__(256) void k_rkp_prep(RkpHeadArgs A) {
    __shared__ float kk_[4][kHS], dt_[4][kHS], part_[4][8];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), t = threadIdx.x & 63;
    const int h = blockIdx.x, tok = (int)blockIdx.y * 4 + wv;
    if (tok >= A.T) return;   // no workgroup barrier below
    const int c = h * kHS + t;
    const size_t at = (size_t)tok * A.D + c;
    const float dw = A.dw[at], da = A.da[at], v_in = A.v[at], kv = A.k[at], rv = A.r[at];
    const float ww = refmath::expf(-refmath::sigmoid(dw + A.w0[c]) * kR2);
    float vv = v_in;
    if (A.first) {
        A.vfirst[at] = vv;
    } else {
        const float mix = refmath::sigmoid(A.dv[at] + A.v0[c]);
        vv = vv + (A.vfirst[at] - vv) * mix;
        A.v[at] = vv;
    }
    const float av = refmath::sigmoid(da + A.a0[c]);
    const float kkv = kv * A.kk_w[c];
    const float k2 = kv + kv * (av - 1.0f) * A.ka_w[c];
    kk_[wv][t] = kkv;
    dt_[wv][t] = rv * k2 * A.rk_w[c];
    wave_sync();
    // |kk| from eight stride-8 partial sums (rwkv7.c:156-162); the bonus dot as
    // one sequential sum, by lane 8
    if (t < 8) {
        float ss = 0.0f;
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const float e = kk_[wv][8 * m + t];
            ss = fmaf(e, e, ss);
        }
        part_[wv][t] = ss;
    } else if (t == 8) {
        float acc = 0.0f;
#pragma unroll 8
        for (int i = 0; i < kHS; ++i) acc = acc + dt_[wv][i];
        A.dot[(size_t)tok * A.NH + h] = acc;
    }
    wave_sync();
    const float* p = part_[wv];
    const float c0 = p[0] + p[4], c1 = p[1] + p[5], c2 = p[2] + p[6], c3 = p[3] + p[7];
    float nrm = sqrtf((c0 + c1) + (c2 + c3));
    if (!(nrm > 1e-12f)) nrm = 1e-12f;
    const float kn = kkv * (1.0f / nrm);
    float* o = A.pack + ((size_t)tok * A.NH + h) * kRkpPack + 8 * lam_of(t & 7) + (t >> 3);
    o[0] = ww;
    o[64] = kn;
    o[128] = kn * av;
    o[192] = k2;
    o[256] = rv;
}

// x + (x of the lane that the DPP control names), within groups of 8 lanes.
template <int CTRL>
__device__ __forceinline__ float dpp_add(float x) {
    return x + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float fold8(float x) {
    x = dpp_add<0x141>(x);   // row_half_mirror: q + (q ^ 4) in the lane order of lam_of
    x = dpp_add<0xB1>(x);    // quad_perm 1 0 3 2
    return dpp_add<0x4E>(x); // quad_perm 2 3 0 1
}

// The state recurrence of one layer over the chunk (rwkv7.c:165-187), one wave
// per eight state rows of a head: eight lanes per row, each with the eight
// columns of one of the reference's partial sums in registers. Rows never meet,
// so a head's eight waves run on eight CUs without an exchange (one wave per
// SIMD: a token costs its ~70 instructions' issue, and rows of one head on one
// CU would share it). The token's five packed vectors are read kAhead tokens
// early; block b works on head b % 8 + 8 (b / 64), so that one head's waves
// share an XCD's L2.
constexpr int kAhead = 5;
struct TokIn {
    float4 w[2], n[2], na[2], k[2], r[2];
    float v;
};
__global__ __launch_bounds__(64) void k_rkp_scan(RkpHeadArgs A) {
    const int b = blockIdx.x, h = (b & 7) + 8 * (b >> 6), rg = (b >> 3) & 7;
    if (h >= A.NH) return;
    const int l = threadIdx.x, lam = l & 7, row = rg * 8 + (l >> 3);
    const int q = lam < 4 ? lam : 11 - lam;
    float* Sr = A.S + (size_t)h * kHS * kHS + (size_t)row * kHS + q;
    float s[8];
#pragma unroll
    for (int m = 0; m < 8; ++m) s[m] = Sr[8 * m];
    // Through buffer resources: a token costs one scalar offset per array.
    const int D4 = A.D * 4, pbytes = A.NH * kRkpPack * 4;
    auto rsrc = [&](const float* base, int bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), (short)0, bytes, 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t rp = rsrc(A.pack, A.T * pbytes), rv = rsrc(A.v, A.T * D4), ry = rsrc(A.ys, A.T * D4);
    const int po = h * kRkpPack * 4 + 32 * lam, vo = (h * kHS + row) * 4;
    auto ld4 = [&](int so, int imm) -> float4 {
        const u32x4v v = __builtin_amdgcn_raw_buffer_load_b128(rp, po + imm, so, 0);
        return make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3]));
    };
    auto load = [&](TokIn& I, int tok) {
        const int t = min(tok, A.T - 1), so = t * pbytes;   // past the end: the last token again, never used
        I.n[0] = ld4(so, 256); I.n[1] = ld4(so, 272);
        I.na[0] = ld4(so, 512); I.na[1] = ld4(so, 528);
        I.w[0] = ld4(so, 0); I.w[1] = ld4(so, 16);
        I.k[0] = ld4(so, 768); I.k[1] = ld4(so, 784);
        I.r[0] = ld4(so, 1024); I.r[1] = ld4(so, 1040);
        I.v = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rv, vo, t * D4, 0));
    };
    // the row's eight lanes hold the same sum: all of them store it, no branch
    auto put = [&](int t, float y) {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y), ry, vo, t * D4, 0);
    };
    auto el = [](const float4 (&x)[2], int m) {
        const float4 v = x[m >> 2];
        return (m & 3) == 0 ? v.x : (m & 3) == 1 ? v.y : (m & 3) == 2 ? v.z : v.w;
    };
    // Step t reads the state before token t twice: for its own read and for
    // token t - 1's read-out, so the two chains of eight run interleaved (each
    // alone left the issue slot waiting: 125 us per 512-token layer). Step 0
    // writes to row 0 what step 1 then writes over.
    auto step = [&](const TokIn& X, const float4 (&r)[2], int t) {
        float pv = 0.0f, ya = 0.0f;
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            pv = fmaf(s[m], el(X.n, m), pv);
            ya = fmaf(s[m], el(r, m), ya);
        }
        pv = fold8(pv);
        ya = fold8(ya);
        put(max(t - 1, 0), ya);
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const float vk = X.v * el(X.k, m);
            s[m] = fmaf(s[m], el(X.w, m), vk - pv * el(X.na, m));
        }
    };
    TokIn I[kAhead];   // slot t % kAhead; a token's slot is refilled in the step after it, which reads its r
#pragma unroll
    for (int i = 0; i < kAhead; ++i) load(I[i], i);
    I[kAhead - 1].r[0] = I[kAhead - 1].r[1] = make_float4(0.f, 0.f, 0.f, 0.f);   // before token 0
    int t0 = 0;
    for (; t0 + kAhead <= A.T; t0 += kAhead) {
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            TokIn& P = I[(i + kAhead - 1) % kAhead];
            step(I[i], P.r, t0 + i);
            load(P, t0 + i + kAhead - 1);
            __builtin_amdgcn_sched_barrier(0);   // the loads stay with their token
        }
    }
#pragma unroll
    for (int i = 0; i < kAhead - 1; ++i)
        if (t0 + i < A.T) step(I[i], I[(i + kAhead - 1) % kAhead].r, t0 + i);
    // the last token's read-out; its r is read again (its slot is not a fixed one)
    const int sl = (A.T - 1) * pbytes;
    const float4 rl[2] = {ld4(sl, 1024), ld4(sl, 1040)};
    float ya = 0.0f;
#pragma unroll
    for (int m = 0; m < 8; ++m) ya = fmaf(s[m], el(rl, m), ya);
    put(A.T - 1, fold8(ya));
#pragma unroll
    for (int m = 0; m < 8; ++m) Sr[8 * m] = s[m];
}

// Group norm, bonus and gate (rwkv7.c:266-288): one wave per (token, head),
// four tokens per workgroup; the mean and the variance as sequential sums that
// every lane runs alike (reads of one LDS address).
__global__ __launch_bounds__(256) void k_rkp_gate(RkpHeadArgs A) {
    __shared__ float4 y_[4][kHS / 4];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), t = threadIdx.x & 63;
    const int h = blockIdx.x, tok = (int)blockIdx.y * 4 + wv;
    if (tok >= A.T) return;   // no workgroup barrier below
    const int c = h * kHS + t;
    const size_t at = (size_t)tok * A.D + c;
    const float yy = A.ys[at], vv = A.v[at], gv = A.g[at];
    const float lnw = A.lnx_w[c], lnb = A.lnx_b[c], dot = A.dot[(size_t)tok * A.NH + h];
    float* ys = reinterpret_cast<float*>(y_[wv]);
    ys[t] = yy;
    wave_sync();
    float4 v[kHS / 4];
#pragma unroll
    for (int i = 0; i < kHS / 4; ++i) v[i] = y_[wv][i];
    float acc = 0.0f;
#pragma unroll
    for (int i = 0; i < kHS / 4; ++i) {
        acc = acc + v[i].x; acc = acc + v[i].y; acc = acc + v[i].z; acc = acc + v[i].w;
    }
    const float mean = acc / (float)kHS;
    float var = 0.0f;
#pragma unroll
    for (int i = 0; i < kHS / 4; ++i) {
        float d = v[i].x - mean;
        var = var + d * d;
        d = v[i].y - mean;
        var = var + d * d;
        d = v[i].z - mean;
        var = var + d * d;
        d = v[i].w - mean;
        var = var + d * d;
    }
    const float rstd = 1.0f / sqrtf(var / (float)kHS + kEpsGroup);
    const float n = (yy - mean) * rstd * lnw + lnb;
    A.y[x16_at(tok, c, A.D / 16)] = (n + dot * vv) * gv;
}

}  // namespace

snhip_status launch_rkp_ln(const RkpLnArgs& a, hipStream_t st) {
    if (a.T <= 0 || a.D <= 0 || a.D > kRkpMaxDim || a.D % 16 || (a.mixes != 1 && a.mixes != 6)) return SNHIP_E_INVAL;
    const dim3 grid((a.T + kLnRows - 1) / kLnRows), blk(64 * (kLnRows + 1));
    const size_t shm = (size_t)(kLnRows + 1) * a.D * sizeof(float);   // at most 64 KiB
    switch (a.D % 256 ? 0 : a.D / 256) {
    case 1: hipLaunchKernelGGL(k_rkp_ln<1>, grid, blk, shm, st, a); break;
    case 2: hipLaunchKernelGGL(k_rkp_ln<2>, grid, blk, shm, st, a); break;
    case 3: hipLaunchKernelGGL(k_rkp_ln<3>, grid, blk, shm, st, a); break;
    case 4: hipLaunchKernelGGL(k_rkp_ln<4>, grid, blk, shm, st, a); break;
    default: hipLaunchKernelGGL(k_rkp_ln<0>, grid, blk, shm, st, a); break;
    }
    SNHIP_CHECK(hipGetLastError());
    return SNHIP_OK;
}

snhip_status launch_rkp_heads(const RkpHeadArgs& a, hipStream_t st) {
    if (a.T <= 0 || a.D != a.NH * kHS) return SNHIP_E_INVAL;
    const dim3 grid(a.NH, (a.T + 3) / 4);
    hipLaunchKernelGGL(k_rkp_prep, grid, dim3(256), 0, st, a);
    SNHIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_rkp_scan, dim3(64 * ((a.NH + 7) / 8)), dim3(64), 0, st, a);
    SNHIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_rkp_gate, grid, dim3(256), 0, st, a);
    SNHIP_CHECK(hipGetLastError());
    return SNHIP_OK;
}

}  // namespace snhip
