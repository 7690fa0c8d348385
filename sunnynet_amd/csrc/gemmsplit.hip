// Products of many rows on the fp16 matrix cores (see gemmsplit.h).
//
// Fragment order: rows in blocks of 32, k in blocks of 16; block (rb, kb) is 2 KiB,
// the h plane's 1 KiB and then the l plane's, each the 64 lanes' 16 bytes of one
// v_mfma_f32_32x32x16_f16 operand (lane l: row l % 32, k = 8 (l / 32) .. + 7). A
// stage of the product is then a run of whole KiB per row block in global memory,
// in LDS (loaded there directly, 16 bytes per lane) and per fragment read (one
// conflict-free ds_read_b128 per lane).
#include <algorithm>

#include "gemmsplit.h"
#include "gemmepi.h"

namespace snhip {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(1))) const void g_void;
typedef __attribute__((address_space(3))) void l_void;

// ---- planes. A block takes 8 rows, half a wave or one to a row; a lane splits 8 values at
// a time (16 bytes of each plane), so 8 neighbouring rows fill a 128-byte line.
// Rows of at most kSplitRegs values are held in registers between the search for
// the largest magnitude and the split; longer ones are loaded twice. Bound by HBM
// (8192 x 1024: 14 us for 67 MB); at 999 x 1024 by the latency of one pass (5 us).
// A row comes from memory (RowSrc), or from the kernel that would otherwise write it
// only for this pass to read it back: 8192 x 1024, conv and planes 53 -> 24 us,
// gates and planes 51 -> 41; 8192 x 1536, LayerNorm and planes 42 -> 28.
// Over the LPR lanes of a row.
template <int LPR, class F>
__device__ __forceinline__ float row_reduce(float v, F f) {
#pragma unroll
    for (int o = LPR / 2; o > 0; o >>= 1) v = f(v, __shfl_xor(v, o, 64));
    return v;
}
// The largest magnitude so far, infinite once there is an infinity or NaN.
__device__ __forceinline__ float row_look(float mx, const float (&x)[8]) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float a = fabsf(x[j]);
        mx = fmaxf(mx, a < __builtin_inff() ? a : __builtin_inff());
    }
    return mx;
}
__device__ __forceinline__ void split_store(const float (&y)[8], int s, bool bad, uint16_t* pl, int row, int k,
                                            int nk) {
    half8 h, l;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        float x = ldexpf(y[j], s);
        // such a row's products are all infinite or NaN: only those, signs and
        // zeros count
        if (bad && fabsf(x) < __builtin_inff()) x = x == 0.0f ? 0.0f : copysignf(1.0f, x);
        h[j] = (_Float16)x;
        l[j] = bad ? (_Float16)0.0f : (_Float16)(x - (float)h[j]);
        // too small for either plane, but not zero: the smallest value of its sign, so
        // that it times an infinity is one
        if ((float)h[j] == 0.0f && (float)l[j] == 0.0f && y[j] != 0.0f) l[j] = (_Float16)copysignf(0x1p-24f, y[j]);
    }
    half8* o = reinterpret_cast<half8*>(pl + (((size_t)(row >> 5) * nk + (k >> 4)) << 10)) + ((k >> 3) & 1) * 32 +
               (row & 31);
    o[0] = h;
    o[64] = l;
}
__device__ __forceinline__ void ld8(float (&v)[8], const float* p) {
    const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
__device__ __forceinline__ void st8(float* p, const float (&v)[8]) {
    reinterpret_cast<float4*>(p)[0] = make_float4(v[0], v[1], v[2], v[3]);
    reinterpret_cast<float4*>(p)[1] = make_float4(v[4], v[5], v[6], v[7]);
}
__device__ __forceinline__ float sgm(float x) { return 1.0f / (1.0f + expf(-x)); }

// Rows of X (with its shifted reads).
struct XSrc {
    GemmArgs g;
    __device__ __forceinline__ void load(float (&v)[8], int row, int k) const { ld8(v, gemm_xrow(g, row) + k); }
    template <int LPR, int NV> __device__ __forceinline__ void row(float (&)[NV][8], int, int) const {}
};
// Rows of W: fp32 (BLK 0), or INT4 groups of BLK, dequantized as quant.c:82-83.
template <int BLK>
struct WSrc {
    GemmArgs g;
    __device__ __forceinline__ void load(float (&v)[8], int row, int k) const {
        if constexpr (BLK == 0) {
            ld8(v, g.w + (long)row * g.K + k);
        } else {
            // byte j of a group: k = j (low nibble) and j + BLK / 2 (high)
            const int grp = k / BLK, in = k % BLK, sh = in >= BLK / 2 ? 4 : 0;
            const float sc = g.sc[(long)row * (g.K / BLK) + grp];
            const uint8_t* q = g.q + (long)row * (g.K / 2) + (long)grp * (BLK / 2) + in % (BLK / 2);
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = (float)((int)((q[j] >> sh) & 0xFu) - 8) * sc;
        }
    }
    template <int LPR, int NV> __device__ __forceinline__ void row(float (&)[NV][8], int, int) const {}
};
struct ConvSrc {
    SplitConv c;
    __device__ __forceinline__ void load(float (&v)[8], int row, int k) const {
        const int b = row / c.T, t = row - b * c.T;
        float r[8], d[8], p[8], acc[8];
        const float* x = c.raw + (size_t)row * c.D + k;
        ld8(r, x);
        ld8(d, c.dw + (size_t)(c.taps - 1) * c.D + k);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] = r[j] * d[j];
        for (int q = 0; q < c.taps - 1; ++q) {
            ld8(p, t - 1 - q >= 0 ? x - (size_t)(q + 1) * c.D
                                  : c.hist + (size_t)b * c.hist_bstride + (size_t)(q - t) * c.D + k);
            ld8(d, c.dw + (size_t)(c.taps - 2 - q) * c.D + k);
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[j] = acc[j] + p[j] * d[j];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = r[j] + acc[j];
    }
    template <int LPR, int NV> __device__ __forceinline__ void row(float (&)[NV][8], int, int) const {}
};
// A lane's 8 values are one group: its gate and u rows are 16 floats side by side.
struct GateSrc {
    SplitGate c;
    __device__ __forceinline__ void load(float (&v)[8], int row, int k) const {
        float u[8], gt[8], dl[8], a[8], b[8];
        const float* x = c.q + (size_t)row * 2 * c.D + 2 * k;
        ld8(u, x);
        ld8(gt, x + 8);
        ld8(dl, c.delta + k);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float gi = gt[j];
            v[j] = u[j] * (sgm(gi - gt[(j + 1) & 7]) * sgm(gi - gt[(j + 2) & 7]));
            float p = 1.0f - dl[j] * (1.0f - sgm(gi));
            if (c.clamp && p < c.p_floor) p = c.p_floor;
            a[j] = p;
            b[j] = (1.0f - p) * v[j];
        }
        st8(c.pa + (size_t)row * c.D + k, a);
        st8(c.pb + (size_t)row * c.D + k, b);
    }
    template <int LPR, int NV> __device__ __forceinline__ void row(float (&)[NV][8], int, int) const {}
};
struct LnSrc {
    SplitLn c;
    __device__ __forceinline__ void load(float (&v)[8], int row, int k) const { ld8(v, c.x + (size_t)row * c.n + k); }
    template <int LPR, int NV> __device__ __forceinline__ void row(float (&v)[NV][8], int lane, int K) const {
        auto add = [](float x, float y) { return x + y; };
        float g[NV][8], o[NV][8], t = 0.0f;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int k = min(lane * 8 + i * LPR * 8, K - 8);
            ld8(g[i], c.g + k);
            ld8(o[i], c.c + k);
#pragma unroll
            for (int j = 0; j < 8; ++j) t += v[i][j];                       // zeros past K
        }
        const float mean = row_reduce<LPR>(t, add) / (float)K;
        t = 0.0f;
#pragma unroll
        for (int i = 0; i < NV; ++i)
            if (lane * 8 + i * LPR * 8 < K)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float d = v[i][j] - mean;
                    t += d * d;
                }
        const float rstd = 1.0f / sqrtf(row_reduce<LPR>(t, add) / (float)K + c.eps);
#pragma unroll
        for (int i = 0; i < NV; ++i)
            if (lane * 8 + i * LPR * 8 < K)
#pragma unroll
                for (int j = 0; j < 8; ++j) v[i][j] = (v[i][j] - mean) * rstd * g[i][j] + o[i][j];
    }
};

template <class Src, bool REGS, int LPR>
__global__ __launch_bounds__(8 * LPR) void k_split_rows(Src src, int rows, int K, uint16_t* __restrict__ pl,
                                                    int* __restrict__ ex) {
    const int lane = threadIdx.x % LPR, nk = K / 16;
    const int row = blockIdx.x * 8 + threadIdx.x / LPR;
    if (row >= rows) return;
    constexpr int NV = REGS ? kSplitRegs / (LPR * 8) : 1;
    float v[NV][8], mx = 0.0f;
    auto most = [](float x, float y) { return fmaxf(x, y); };
    if constexpr (REGS) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int k = lane * 8 + i * LPR * 8;
            if (k < K) src.load(v[i], row, k);
            else
#pragma unroll
                for (int j = 0; j < 8; ++j) v[i][j] = 0.0f;
        }
        src.template row<LPR, NV>(v, lane, K);
#pragma unroll
        for (int i = 0; i < NV; ++i) mx = row_look(mx, v[i]);
    } else {
        for (int k = lane * 8; k < K; k += LPR * 8) {
            src.load(v[0], row, k);
            mx = row_look(mx, v[0]);
        }
    }
    mx = row_reduce<LPR>(mx, most);
    const bool bad = !(mx < __builtin_inff());
    int e = 0;
    (void)frexpf(mx, &e);                        // mx in [2^(e-1), 2^e)
    const int s = bad ? 0 : (mx > 0.0f ? 15 - e : 0);
    if constexpr (REGS) {
#pragma unroll
        for (int i = 0; i < NV; ++i)
            if (lane * 8 + i * LPR * 8 < K) split_store(v[i], s, bad, pl, row, lane * 8 + i * LPR * 8, nk);
    } else {
        for (int k = lane * 8; k < K; k += LPR * 8) {
            src.load(v[0], row, k);
            split_store(v[0], s, bad, pl, row, k, nk);
        }
    }
    if (lane == 0) ex[row] = bad ? kSplitNonFinite : s;
}

template <bool REGS, class Src>
snhip_status split_launch(const Src& src, int rows, int K, SplitMat out, hipStream_t st) {
    // us per call, 32 / 64 lanes to a row: 8192 rows of 1024, planes alone 14.4 / 17.6,
    // conv 24 / 30, gates 41 / 45; 999 rows (125 blocks) 6.0 / 5.1, 14.1 / 9.2, 14.3 / 11.2.
    if (rows >= 4096)
        hipLaunchKernelGGL((k_split_rows<Src, REGS, 32>), dim3((rows + 7) / 8), dim3(256), 0, st, src, rows, K, out.pl,
                           out.ex);
    else
        hipLaunchKernelGGL((k_split_rows<Src, REGS, 64>), dim3((rows + 7) / 8), dim3(512), 0, st, src, rows, K, out.pl,
                           out.ex);
    SNHIP_CHECK(hipGetLastError());
    return SNHIP_OK;
}

// One output of a row with an infinity or NaN in it.
__device__ float split_bad(const uint16_t* xp, const uint16_t* wp, int m, int n, int nk) {
    const half8* x = reinterpret_cast<const half8*>(xp) + (size_t)(m >> 5) * nk * 128 + (m & 31);
    const half8* w = reinterpret_cast<const half8*>(wp) + (size_t)(n >> 5) * nk * 128 + (n & 31);
    float acc = 0.0f;
    for (int c = 0; c < 2 * nk; ++c) {
        const size_t o = (size_t)(c >> 1) * 128 + (c & 1) * 32;
        const half8 xh = x[o], xl = x[o + 64], wh = w[o], wl = w[o + 64];
        for (int j = 0; j < 8; ++j)
            acc = fmaf((float)xh[j] + (float)xl[j], (float)wh[j] + (float)wl[j], acc);
    }
    return acc;
}

// ---- the product. Four waves stacked along m, each RB x CB blocks of 32 x 32
// outputs. A stage is KB blocks of 16 in k: a wave's X fragments are its own and come
// straight to registers, the W fragments are shared through LDS; the next stage of
// both is in flight while this one is multiplied. Three fp16 products per fp32 one:
// N = K = 1024 at 8192 rows takes 54 us, 960 TFLOP/s in fp16 (a large library
// product reaches 1156 on the same card) and 313 in fp32, where the fp32 matrix
// cores took 183; N = 32000 1.51 ms, 1070 and 357 (5.7 ms). 2 x 4 blocks per wave
// with half the W reads measured the same (58 us, 1.48 ms).
constexpr int kEpiPart = -1;     // a split-K partial instead of an epilogue
template <int RB, int CB, int KB, int EPI>
__global__ __launch_bounds__(256, 2) void k_gemm_split(GemmArgs g, SplitMat X, SplitMat W, int kchunk,
                                                       int mt, int nt, float* __restrict__ part) {
    constexpr int PW = CB * KB * 2 / 4;              // KiB of W a wave brings in
    __shared__ __align__(16) half8 sm0[CB * KB * 2 * 64], sm1[CB * KB * 2 * 64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    // consecutive tiles (n fastest) run on one XCD and share its L2
    const int G = mt * nt, id = (int)blockIdx.x, q8 = G / 8, r8 = G % 8, x8 = id % 8;
    const int tile = x8 * q8 + min(x8, r8) + id / 8;
    const int tm = tile / nt, tn = tile - tm * nt;
    const int nk = g.K / 16, kbeg = blockIdx.y * kchunk, kend = min(nk, kbeg + kchunk);
    const int rb0 = (tm * 4 + w) * RB, cb0 = tn * CB;
    const half8* xp = reinterpret_cast<const half8*>(X.pl) + (size_t)rb0 * nk * 128 + lane;
    const half8* wp = reinterpret_cast<const half8*>(W.pl) + (size_t)cb0 * nk * 128 + lane;
    // h h, and apart from it h l + l h, 2^-11 of it: the roundings of that sum do not
    // count, and the large one is rounded once per 16 values of k instead of three
    // times. The second accumulators cost about 2.5 % of a 16 x 512 forward (7.45 ->
    // 7.64 ms; all l h first, then all h h: 7.71).
    floatx16 acc[RB][CB], low[RB][CB];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j)
#pragma unroll
            for (int c = 0; c < 16; ++c) acc[i][j][c] = low[i][j][c] = 0.0f;

    struct AFrag {
        half8 v[RB][KB][2];
    };
    // (K is a multiple of two blocks: longer stages end with blocks past the end,
    // which load the last one and are not multiplied)
    auto at = [&](int k) { return KB == 2 ? k : min(k, kend - 1); };
    auto load = [&](half8* sm, AFrag& A, int kb) {
#pragma unroll
        for (int c = 0; c < PW; ++c) {
            const int ch = w * PW + c, j = ch / (KB * 2), sub = ch % (KB * 2);
            __builtin_amdgcn_global_load_lds((g_void*)(wp + ((size_t)j * nk + at(kb + sub / 2)) * 128 + sub % 2 * 64),
                                             (l_void*)&sm[ch * 64], 16, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int k = 0; k < KB; ++k)
#pragma unroll
                for (int p = 0; p < 2; ++p) A.v[i][k][p] = xp[((size_t)i * nk + at(kb + k)) * 128 + p * 64];
    };
    auto mul = [&](const half8* sm, const AFrag& A, int kb) {
#pragma unroll
        for (int k = 0; k < KB; ++k) {
            if (KB > 2 && kb + k >= kend) break;
            half8 b[CB][2];
#pragma unroll
            for (int j = 0; j < CB; ++j)
#pragma unroll
                for (int p = 0; p < 2; ++p) b[j][p] = sm[((j * KB + k) * 2 + p) * 64 + lane];
            auto mac = [](const half8& x, const half8& w, floatx16& c) {
                c = __builtin_amdgcn_mfma_f32_32x32x16_f16(x, w, c, 0, 0, 0);
            };
#pragma unroll
            for (int j = 0; j < CB; ++j)
#pragma unroll
                for (int i = 0; i < RB; ++i) {
                    mac(A.v[i][k][1], b[j][0], low[i][j]);
                    mac(A.v[i][k][0], b[j][0], acc[i][j]);
                }
#pragma unroll
            for (int j = 0; j < CB; ++j)
#pragma unroll
                for (int i = 0; i < RB; ++i) mac(A.v[i][k][0], b[j][1], low[i][j]);
        }
    };
    auto ready = [] {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    };
    AFrag A0, A1;
    load(sm0, A0, kbeg);
    for (int kb = kbeg;; kb += 2 * KB) {
        ready();
        const bool more = kb + KB < kend;
        if (more) load(sm1, A1, kb + KB);
        __builtin_amdgcn_sched_barrier(0);
        mul(sm0, A0, kb);
        if (!more) break;
        ready();
        const bool again = kb + 2 * KB < kend;
        if (again) load(sm0, A0, kb + 2 * KB);
        __builtin_amdgcn_sched_barrier(0);
        mul(sm1, A1, kb + KB);
        if (!again) break;
    }
    // Register c of lane (r, h) is row (c / 4) * 8 + h * 4 + c % 4, column r of its block.
    const int r = lane & 31, h = lane >> 5;
    bool bad = false;
#pragma unroll
    for (int i = 0; i < RB; ++i) {
        const int mb = (rb0 + i) * 32 + h * 4;
        int em[16];
#pragma unroll
        for (int c = 0; c < 16; c += 4) {
            const int4 e = *reinterpret_cast<const int4*>(X.ex + mb + c * 2);
            em[c] = e.x; em[c + 1] = e.y; em[c + 2] = e.z; em[c + 3] = e.w;
        }
#pragma unroll
        for (int j = 0; j < CB; ++j) {
            const int n = (cb0 + j) * 32 + r;
            if (n >= g.N) continue;
            const int en = W.ex[n];
            float v[16];
            bool ok[16];
#pragma unroll
            for (int c = 0; c < 16; ++c) {
                const bool in = mb + (c >> 2) * 8 + (c & 3) < g.M;
                ok[c] = in && em[c] != kSplitNonFinite && en != kSplitNonFinite;
                bad |= in && !ok[c];
                v[c] = ldexpf(acc[i][j][c] + low[i][j][c], -(em[c] + en));
            }
            float* y = EPI == kEpiPart ? part + (long)blockIdx.y * g.M * g.N : g.Y;
            const long ldy = EPI == kEpiPart ? g.N : g.ldy;
            float t[EPI == GEPI_RESID ? 3 : 1][16];
            if constexpr (EPI == GEPI_RESID) {
                // the three terms of 16 outputs in flight together
#pragma unroll
                for (int c = 0; c < 16; ++c) {
                    const long m = min(mb + (c >> 2) * 8 + (c & 3), g.M - 1);
                    t[0][c] = g.s[m * g.lds + n];
                    t[1][c] = g.sfb[m * g.ldf + n];
                    t[2][c] = y[m * ldy + n];
                }
            }
#pragma unroll
            for (int c = 0; c < 16; ++c) {
                float x = v[c];
                if constexpr (EPI == GEPI_WEDGE) x = x * (1.0f + 0.5f * g.a_tanh / (1.0f + fabsf(x)));   // sunnynet.c:270-271
                if constexpr (EPI == GEPI_RESID) x = x + (g.b_gain * t[0][c] + t[1][c] + t[2][c]);       // :276
                if (ok[c]) y[(long)(mb + (c >> 2) * 8 + (c & 3)) * ldy + n] = x;
            }
        }
    }
    if (__any(bad)) {
        for (int i = 0; i < RB * 16; ++i)
            for (int j = 0; j < CB; ++j) {
                const int m = (rb0 + i / 16) * 32 + h * 4 + ((i & 15) >> 2) * 8 + (i & 3), n = (cb0 + j) * 32 + r;
                if (m >= g.M || n >= g.N) continue;
                if (X.ex[m] != kSplitNonFinite && W.ex[n] != kSplitNonFinite) continue;
                const float x = blockIdx.y == 0 ? split_bad(X.pl, W.pl, m, n, nk) : 0.0f;
                if (EPI == kEpiPart) part[((long)blockIdx.y * g.M + m) * g.N + n] = x;
                else gemm_epilogue(g, m, n, x);
            }
    }
}

}  // namespace

snhip_status launch_split_x(const GemmArgs& g, SplitMat out, hipStream_t st) {
    return g.K <= kSplitRegs ? split_launch<true>(XSrc{g}, g.M, g.K, out, st)
                             : split_launch<false>(XSrc{g}, g.M, g.K, out, st);
}

snhip_status launch_split_w(const GemmArgs& g, SplitMat out, hipStream_t st) {
    if (!g.q) return split_launch<false>(WSrc<0>{g}, g.N, g.K, out, st);
    if (g.block == 32) return split_launch<false>(WSrc<32>{g}, g.N, g.K, out, st);
    return split_launch<false>(WSrc<64>{g}, g.N, g.K, out, st);
}

snhip_status launch_split_conv(const SplitConv& c, int rows, SplitMat out, hipStream_t st) {
    return split_launch<true>(ConvSrc{c}, rows, c.D, out, st);
}
snhip_status launch_split_gate(const SplitGate& c, int rows, SplitMat out, hipStream_t st) {
    return split_launch<true>(GateSrc{c}, rows, c.D, out, st);
}
snhip_status launch_split_ln(const SplitLn& c, int rows, SplitMat out, hipStream_t st) {
    return split_launch<true>(LnSrc{c}, rows, c.n, out, st);
}

snhip_status launch_gemm_split(const GemmArgs& g, SplitMat x, SplitMat w, float* work, size_t work_floats,
                               hipStream_t st) {
    if (g.M <= 0 || g.N <= 0 || g.K <= 0 || g.K % 32 || g.epi < GEPI_STORE || g.epi > GEPI_RESID) {
        set_last_error("split gemm: K must be a positive multiple of 32, the epilogue store, wedge or residual");
        return SNHIP_E_INVAL;
    }
    const int nk = g.K / 16;
    auto tiles = [&](int tm, int tn) { return ((g.M + tm - 1) / tm) * ((g.N + tn - 1) / tn); };
    // Tiles of 128 x 128, with more X per byte of W read, once they fill the chip
    // twice; else 128 x 64 with twice the k in flight. us, 8192 rows, 128 / 64
    // wide: N = K = 1024 55 / 64, N = 512 37 / 35; 999 rows, N = K = 1024 with
    // its reduction 25 / 18.
    const bool big = tiles(128, 128) >= 512;
    const int tm = 128, tn = big ? 128 : 64, kb = big ? 2 : 4;
    const int mt = (g.M + tm - 1) / tm, nt = (g.N + tn - 1) / tn;
    // Few tiles split K over the idle CUs, at least two stages each: 64 tiles of
    // 16 stages 20 us whole, 16 in 4; but 192 tiles 22.5 whole, 26 in 2 (the
    // partials' reduction).
    int splits = 1;
    if (work) {
        splits = std::max(1, std::min(256 / (mt * nt), nk / (2 * kb)));
        while (splits > 1 && (size_t)splits * g.M * g.N > work_floats) --splits;
    }
    const int stages = (nk + kb - 1) / kb;
    const int kchunk = (stages + splits - 1) / splits * kb;
    splits = (nk + kchunk - 1) / kchunk;
    float* part = splits > 1 ? work : nullptr;
    const dim3 grid(mt * nt, splits);
    const int epi = part ? kEpiPart : g.epi;
#define SNHIP_SPLIT(RB, CB, KB, E)                                                                              \
    if (epi == E)                                                                                           \
    hipLaunchKernelGGL((k_gemm_split<RB, CB, KB, E>), grid, dim3(256), 0, st, g, x, w, kchunk, mt, nt, part)
#define SNHIP_SPLIT_ALL(RB, CB, KB)                                                                             \
    do {                                                                                                    \
        SNHIP_SPLIT(RB, CB, KB, kEpiPart);                                                                      \
        SNHIP_SPLIT(RB, CB, KB, GEPI_STORE);                                                                    \
        SNHIP_SPLIT(RB, CB, KB, GEPI_WEDGE);                                                                    \
        SNHIP_SPLIT(RB, CB, KB, GEPI_RESID);                                                                    \
    } while (0)
    if (big) SNHIP_SPLIT_ALL(1, 4, 2);
    else SNHIP_SPLIT_ALL(1, 2, 4);
#undef SNHIP_SPLIT_ALL
#undef SNHIP_SPLIT
    SNHIP_CHECK(hipGetLastError());
    return part ? launch_gemm_reduce(g, splits, part, st) : SNHIP_OK;
}

}  // namespace snhip
