// First-order gated recurrence on gfx950: s_t = a_t * s_{t-1} + b'_t with
// b'_t = (1 - a_t) * u_t (gated) or b_t (FMA form), per channel, over (B,T,N)
// channel-major fp32 arrays.
//
// Semantics and rounding follow sunnynet/runtime/recur.c:13-48 (and the
// identical scan_f32, sunnynet/kernels/scan_avx2.c:12-45): b' is a separate
// multiply, the update is one fused multiply-add, and channels in the scalar
// tail [N & ~7, N) of the reference use a*s + b' with two roundings. The
// result is therefore bit-identical to the reference for every input.
//
// Design. A channel's recurrence is sequential in T, and cfg-sized inputs
// have only a few tens of thousands of channels, so one lane per channel would
// leave HBM idle (too few bytes in flight per CU). Each workgroup instead
// takes 64*CPL adjacent channels (one lane per CPL channels, vector loads
// along the contiguous N axis) and W waves. Time is cut into tiles of W*TC
// steps; wave w owns steps [w*TC, (w+1)*TC) of every tile and keeps them in
// VGPRs. The exact state is handed from wave to wave through LDS in W
// barrier-separated slots per tile; in its slot a wave runs its TC dependent
// FMAs from registers, passes the state on, and immediately issues the loads
// for its slot of the next tile, so every wave has a whole tile's worth of
// loads in flight while the others compute. HBM traffic is exactly one read
// of a and b and one write of out. The barrier orders LDS only, so the
// prefetches are never drained by it.
#include "bufio.h"

namespace snhip {

typedef float f32x2v __attribute__((ext_vector_type(2)));
typedef float f32x4v __attribute__((ext_vector_type(4)));
template <int CPL> struct VecT;
template <> struct VecT<1> { using T = float; };
template <> struct VecT<2> { using T = f32x2v; };
template <> struct VecT<4> { using T = f32x4v; };

// Streaming (non-temporal) vector load / store of CPL consecutive floats.
template <int CPL>
__device__ __forceinline__ void ld(float (&v)[CPL], const float* p) {
    using V = typename VecT<CPL>::T;
    const V x = __builtin_nontemporal_load(reinterpret_cast<const V*>(p));
    if constexpr (CPL == 1) { v[0] = x; }
    else {
#pragma unroll
        for (int c = 0; c < CPL; ++c) v[c] = x[c];
    }
}

template <int CPL>
__device__ __forceinline__ void st(float* p, const float (&v)[CPL]) {
    using V = typename VecT<CPL>::T;
    V x;
    if constexpr (CPL == 1) { x = v[0]; }
    else {
#pragma unroll
        for (int c = 0; c < CPL; ++c) x[c] = v[c];
    }
    __builtin_nontemporal_store(x, reinterpret_cast<V*>(p));
}

template <int CPL, int W, int TC, bool GATED, bool ALLFUSED>
__global__ __launch_bounds__(64 * W)
void k_recur_scan(const float* __restrict__ a, const float* __restrict__ b,
                  const float* __restrict__ s0, float* __restrict__ out,
                  float* __restrict__ send, int B, int T, int N, int N8) {
    static_assert(W >= 2, "the hand-off pipeline needs at least two waves");
    __shared__ float carry[CPL * 64];
    const int lane = threadIdx.x & 63;
    const int w = threadIdx.x >> 6;
    const long total = (long)B * N;
    const long flat_raw = ((long)blockIdx.x * 64 + lane) * CPL;
    const bool valid = flat_raw < total;
    // Lanes past the last channel load (but never store) the last valid
    // vector, so loads need no predicate.
    const long flat = valid ? flat_raw : total - CPL;
    const long bb = flat / N;
    const int n = (int)(flat - bb * N);
    const size_t base = (size_t)bb * T * N + n;
    bool fused[CPL];
#pragma unroll
    for (int c = 0; c < CPL; ++c) fused[c] = ALLFUSED || (n + c) < N8;

    constexpr int TILE = W * TC;
    const int ntiles = (T + TILE - 1) / TILE;
    const int nfull = T / TILE;
    float av[TC][CPL], bv[TC][CPL];

    // Time indices are clamped to T-1, so every prefetch is in bounds and
    // branch-free; only the final partial tile checks t < T when stepping.
    auto load_slot = [&](int tile) {
        const int t0 = tile * TILE + w * TC;
#pragma unroll
        for (int k = 0; k < TC; ++k) {
            const size_t off = base + (size_t)min(t0 + k, T - 1) * N;
            ld<CPL>(av[k], a + off);
            ld<CPL>(bv[k], b + off);
        }
    };
    // b' = (1 - a) * u, computed off the critical path (in the slot before
    // this wave's own), exactly once per loaded slot.
    auto prep = [&]() {
        if constexpr (GATED) {
#pragma unroll
            for (int k = 0; k < TC; ++k)
#pragma unroll
                for (int c = 0; c < CPL; ++c) bv[k][c] = mul_rn(sub_rn(1.0f, av[k][c]), bv[k][c]);
        }
    };
    auto step = [&](float (&s)[CPL], int k) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            if constexpr (ALLFUSED) s[c] = fmaf(av[k][c], s[c], bv[k][c]);
            else s[c] = fused[c] ? fmaf(av[k][c], s[c], bv[k][c])
                                 : add_rn(mul_rn(av[k][c], s[c]), bv[k][c]);
        }
    };

    // The initial state enters through the same LDS slot as every later
    // carry, so no slot ever waits on a global load into the state registers
    // (such a wait would also drain the slot's own output stores).
    if (w == 0) {
        float s[CPL];
        ld<CPL>(s, s0 + (size_t)bb * N + n);
#pragma unroll
        for (int c = 0; c < CPL; ++c) carry[c * 64 + lane] = s[c];
    }
    load_slot(0);
    if (w == 0) prep();
    __syncthreads();
    // Slot j of tile t: wave j steps its TC time steps; wave j+1 prepares
    // its own slot of tile t; at j = W-1 wave 0 prepares its slot of t+1.
    for (int tile = 0; tile < nfull; ++tile) {
        for (int j = 0; j < W; ++j) {
            if (w == j) {
                float s[CPL];
#pragma unroll
                for (int c = 0; c < CPL; ++c) s[c] = carry[c * 64 + lane];
                float* po = out + base + (size_t)(tile * TILE + j * TC) * N;
#pragma unroll
                for (int k = 0; k < TC; ++k) {
                    step(s, k);
                    if (valid) st<CPL>(po + (size_t)k * N, s);
                }
#pragma unroll
                for (int c = 0; c < CPL; ++c) carry[c * 64 + lane] = s[c];
                if (tile + 1 < ntiles) load_slot(tile + 1);
            } else if (w == j + 1 || (j == W - 1 && w == 0 && tile + 1 < ntiles)) {
                prep();
            }
            barrier_lds();
        }
    }
    if (nfull < ntiles) {
        for (int j = 0; j < W; ++j) {
            if (w == j) {
                float s[CPL];
#pragma unroll
                for (int c = 0; c < CPL; ++c) s[c] = carry[c * 64 + lane];
                const int t0 = nfull * TILE + j * TC;
#pragma unroll
                for (int k = 0; k < TC; ++k) {
                    if (t0 + k < T) {
                        step(s, k);
                        if (valid) st<CPL>(out + base + (size_t)(t0 + k) * N, s);
                    }
                }
#pragma unroll
                for (int c = 0; c < CPL; ++c) carry[c * 64 + lane] = s[c];
            } else if (w == j + 1) {
                prep();
            }
            barrier_lds();
        }
    }
    if (w == 0 && valid) {
        float s[CPL];
#pragma unroll
        for (int c = 0; c < CPL; ++c) s[c] = carry[c * 64 + lane];
        st<CPL>(send + (size_t)bb * N + n, s);
    }
}

// Fast path for the common layout: every workgroup's 64*CPL channels lie in
// one batch row (N % (64*CPL) == 0) and a row fits a 2 GiB buffer window.
// Same slot pipeline as above, but all global traffic goes through buffer
// resources: the per-step row offset t*N*4 is a scalar (SGPR) operand, so the
// active slot issues only its FMAs and stores (no per-access 64-bit address
// arithmetic), and the prefetch registers hold data only, which leaves room
// for deeper time chunks. Prefetches past T re-read step T - 1 (the scalar
// row offset is not range-checked by the hardware) and are never used.

template <int CPL, int W, int TC, bool GATED>
__global__ __launch_bounds__(64 * W)
void k_recur_scan_buf(const float* __restrict__ a, const float* __restrict__ b,
                      const float* __restrict__ s0, float* __restrict__ out,
                      float* __restrict__ send, int T, int N) {
    static_assert(W >= 2, "the hand-off pipeline needs at least two waves");
    using IO = BufIO<CPL>;
    __shared__ float carry[CPL * 64];
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wg_per_row = N / (64 * CPL);
    const int bb = blockIdx.x / wg_per_row;
    const int n0 = (blockIdx.x - bb * wg_per_row) * 64 * CPL;
    const size_t row = (size_t)bb * T * N;
    const uint32_t nbytes = (uint32_t)((size_t)T * N * 4);
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(a + row, nbytes);
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(b + row, nbytes);
    const __amdgpu_buffer_rsrc_t ro = make_rsrc(out + row, nbytes);
    const int voff = (n0 + lane * CPL) * 4;
    const int rowb = N * 4;

    constexpr int TILE = W * TC;
    const int ntiles = (T + TILE - 1) / TILE;
    const int nfull = T / TILE;
    // bv holds the loaded b; bp the step addend b' (prepared off the critical
    // path). Separate arrays keep the two lifetimes disjoint for the allocator.
    float av[TC][CPL], bv[TC][CPL], bp[TC][CPL];

    // Steps past T (the last tile's tail) load step T - 1 instead: the row
    // offset is the scalar operand, which the buffer range check does not
    // cover. Those values are never used.
    auto load_slot = [&](int tile) {
        const int t0 = tile * TILE + w * TC;
#pragma unroll
        for (int k = 0; k < TC; ++k) {
            const int so = min(t0 + k, T - 1) * rowb;
            IO::load(av[k], ra, voff, so);
            IO::load(bv[k], rb, voff, so);
        }
    };
    auto prep = [&]() {
        if constexpr (GATED) {
#pragma unroll
            for (int k = 0; k < TC; ++k)
#pragma unroll
                for (int c = 0; c < CPL; ++c) bp[k][c] = mul_rn(sub_rn(1.0f, av[k][c]), bv[k][c]);
        }
    };

    if (w == 0) {
        float s[CPL];
        ld<CPL>(s, s0 + (size_t)bb * N + n0 + lane * CPL);
#pragma unroll
        for (int c = 0; c < CPL; ++c) carry[c * 64 + lane] = s[c];
    }
    load_slot(0);
    if (w == 0) prep();
    __syncthreads();
    for (int tile = 0; tile < nfull; ++tile) {
        for (int j = 0; j < W; ++j) {
            if (w == j) {
                float s[CPL];
#pragma unroll
                for (int c = 0; c < CPL; ++c) s[c] = carry[c * 64 + lane];
                const int t0 = tile * TILE + j * TC;
#pragma unroll
                for (int k = 0; k < TC; ++k) {
#pragma unroll
                    for (int c = 0; c < CPL; ++c) s[c] = fmaf(av[k][c], s[c], GATED ? bp[k][c] : bv[k][c]);
                    IO::store(ro, voff, (t0 + k) * rowb, s);
                }
#pragma unroll
                for (int c = 0; c < CPL; ++c) carry[c * 64 + lane] = s[c];
                if (tile + 1 < ntiles) load_slot(tile + 1);
            } else if (w == j + 1 || (j == W - 1 && w == 0 && tile + 1 < ntiles)) {
                prep();
            }
            barrier_lds();
        }
    }
    if (nfull < ntiles) {
        for (int j = 0; j < W; ++j) {
            if (w == j) {
                float s[CPL];
#pragma unroll
                for (int c = 0; c < CPL; ++c) s[c] = carry[c * 64 + lane];
                const int t0 = nfull * TILE + j * TC;
#pragma unroll
                for (int k = 0; k < TC; ++k) {
                    if (t0 + k < T) {
#pragma unroll
                        for (int c = 0; c < CPL; ++c) s[c] = fmaf(av[k][c], s[c], GATED ? bp[k][c] : bv[k][c]);
                        IO::store(ro, voff, (t0 + k) * rowb, s);
                    }
                }
#pragma unroll
                for (int c = 0; c < CPL; ++c) carry[c * 64 + lane] = s[c];
            } else if (w == j + 1) {
                prep();
            }
            barrier_lds();
        }
    }
    if (w == 0) {
        float s[CPL];
#pragma unroll
        for (int c = 0; c < CPL; ++c) s[c] = carry[c * 64 + lane];
        st<CPL>(send + (size_t)bb * N + n0 + lane * CPL, s);
    }
}

// Ring form, for few channels: chains of T steps on so few lanes that their
// latency, not HBM, sets the time. One lane per channel, up to 64 channels (of
// any rows: flat index b N + n) per workgroup of W waves; wave w owns steps
// [w TC, (w + 1) TC) of every tile. On the ring's critical path a wave runs
// only its slot's chain from registers and hands the result on through LDS
// (value, then sequence word; LDS operations of a wave complete in order, so
// who sees the word sees the value); it then runs the chain again from the same
// start and stores, while the next waves are in their slots. Each wave holds
// two tiles of inputs: tile i + 1 is loaded before tile i is processed. Rows
// are uniform offsets: a step costs one scalar add. What is left bounds it by the
// loads a CU keeps in flight (63 per wave): 4 waves of 32 or 64 steps, and 32
// backward, measure the same as 8 of 32 (16 backward). A whole call on 4096
// channels of 2048 steps, forward 55 -> 30 us (one workgroup per 64 channels, a
// barrier per slot before), backward 961 -> 54 us (one lane per channel straight
// through time before); 2331 channels of 333 steps 19 -> 12 us forward.
//   SCAN_FMA, SCAN_GATED: x0 = a, x1 = b; y0 = out, end = send (steps forward)
//   SCAN_BWD: x0 = p, x1 = dout, x2 = nu, x3 = out; y0 = dp, y1 = dnu, end = ds0
//   SCAN_DS:  x0 = p, x1 = dstate; y0 = ds before each step's decay, end = ds0
// The last two walk time backwards from 0, in scan_avx2.c:50-99's and
// core_avx2.c:78-149's order: ds += x1; (outputs); ds *= p.
enum { SCAN_FMA, SCAN_GATED, SCAN_BWD, SCAN_DS };
struct RingArgs {
    const float *x0, *x1, *x2, *x3, *s0;
    float *y0, *y1, *end;
    int T, N, N8;      // channels from N8 on take two roundings (forward)
    size_t s0_stride;  // of a batch row of s0
    int total;         // B N
    int ch;            // channels of a workgroup (at most 64; the other lanes idle)
    int yT, yrow;      // y0: floats per batch row and per step
    unsigned bytes, ybytes;
};

typedef __attribute__((address_space(3))) volatile int lds_word;
typedef __attribute__((address_space(3))) volatile float lds_val;
constexpr int kRingPolls = 1 << 26;   // bounded all the same: the waves of a workgroup are resident together

template <int MODE, int TC>
struct RingBuf {
    float a[TC], b[TC];
    float c[MODE == SCAN_BWD ? TC : 1], d[MODE == SCAN_BWD ? TC : 1];
};

template <int MODE, bool ALLFUSED, int W, int TC>
__global__ __launch_bounds__(64 * W) void k_scan_ring(const RingArgs A) {
    constexpr bool BACK = MODE == SCAN_BWD || MODE == SCAN_DS;
    __shared__ float carry[64];
    __shared__ int seq;
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // consecutive numbers run on one XCD: neighbours share the lines of its L2
    const int G = (int)gridDim.x, g = (int)blockIdx.x, q8 = G / 8, r8 = G % 8, x8 = g % 8;
    const int raw = (x8 * q8 + min(x8, r8) + g / 8) * A.ch + lane;
    const bool valid = lane < A.ch && raw < A.total;
    // lanes without a channel load a neighbour's and store nothing
    const int ch = min(min(raw, raw - lane + A.ch - 1), A.total - 1);
    const int bb = ch / A.N, n = ch - bb * A.N;
    const int T = A.T, rowb = A.N * 4;
    const bool fused = ALLFUSED || n < A.N8;
    auto rsrc = [](const float* p, unsigned bytes) { return make_rsrc(p, bytes); };
    const __amdgpu_buffer_rsrc_t r0 = rsrc(A.x0, A.bytes), r1 = rsrc(A.x1, A.bytes);
    const __amdgpu_buffer_rsrc_t r2 = rsrc(MODE == SCAN_BWD ? A.x2 : A.x0, A.bytes);
    const __amdgpu_buffer_rsrc_t r3 = rsrc(MODE == SCAN_BWD ? A.x3 : A.x0, A.bytes);
    const __amdgpu_buffer_rsrc_t w0 = rsrc(A.y0, A.ybytes);
    const __amdgpu_buffer_rsrc_t w1 = rsrc(MODE == SCAN_BWD ? A.y1 : A.y0, A.ybytes);
    const int vo = (bb * T * A.N + n) * 4;
    // out of range for lanes without a channel: the store is dropped
    const int yo = valid ? (bb * A.yT + n) * 4 : 0x7fffffff;
    const int yrowb = A.yrow * 4;
    constexpr int TILE = W * TC;
    const int ntiles = (T + TILE - 1) / TILE;
    auto ld1 = [](const __amdgpu_buffer_rsrc_t& r, int v, int so) {
        return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, v, so, 0));
    };
    // Step k of this wave's slot of `tile` is time t_of; steps past the end load
    // a step within it and are not run.
    auto t_of = [&](int tile, int k) {
        const int i = tile * TILE + w * TC + k;
        return BACK ? T - 1 - i : i;
    };
    float sz = 0.0f;
    if (MODE == SCAN_BWD || !BACK) sz = A.s0[(size_t)bb * A.s0_stride + n];
    auto load = [&](RingBuf<MODE, TC>& X, int tile) {
#pragma unroll
        for (int k = 0; k < TC; ++k) {
            const int t = min(max(t_of(tile, k), 0), T - 1), so = t * rowb;
            X.a[k] = ld1(r0, vo, so);
            X.b[k] = ld1(r1, vo, so);
            if constexpr (MODE == SCAN_BWD) {
                X.c[k] = ld1(r2, vo, so);
                X.d[k] = ld1(r3, vo, max(t - 1, 0) * rowb);
            }
        }
    };
    auto prep = [&](RingBuf<MODE, TC>& X, int tile) {
        if constexpr (MODE == SCAN_GATED) {
#pragma unroll
            for (int k = 0; k < TC; ++k) {
                X.b[k] = mul_rn(sub_rn(1.0f, X.a[k]), X.b[k]);
                asm volatile("" : "+v"(X.b[k]));   // here, not after the wait for the carry
            }
        } else if constexpr (MODE == SCAN_BWD) {
#pragma unroll
            for (int k = 0; k < TC; ++k) {
                X.c[k] = sub_rn(t_of(tile, k) == 0 ? sz : X.d[k], X.c[k]);   // s_{-1} is s0
                X.d[k] = sub_rn(1.0f, X.a[k]);
                asm volatile("" : "+v"(X.c[k]), "+v"(X.d[k]));
            }
        } else {
            // (the chain's inputs are in before the wait)
#pragma unroll
            for (int k = 0; k < TC; ++k) asm volatile("" : "+v"(X.a[k]), "+v"(X.b[k]));
        }
    };
    auto step = [&](float s, const RingBuf<MODE, TC>& X, int k) {
        if constexpr (BACK) return mul_rn(add_rn(X.b[k], s), X.a[k]);
        else if constexpr (ALLFUSED) return fmaf(X.a[k], s, X.b[k]);
        else return fused ? fmaf(X.a[k], s, X.b[k]) : add_rn(mul_rn(X.a[k], s), X.b[k]);
    };
    auto emit = [&](float s, const RingBuf<MODE, TC>& X, int k, int t) {
        auto st1 = [&](const __amdgpu_buffer_rsrc_t& r, float v) {
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, yo, t * yrowb, 0);
        };
        if constexpr (MODE == SCAN_BWD) {
            const float ds = add_rn(X.b[k], s);
            st1(w1, mul_rn(ds, X.d[k]));
            st1(w0, mul_rn(ds, X.c[k]));
            return mul_rn(ds, X.a[k]);
        } else if constexpr (MODE == SCAN_DS) {
            const float ds = add_rn(X.b[k], s);
            st1(w0, ds);
            return mul_rn(ds, X.a[k]);
        } else {
            const float o = step(s, X, k);
            st1(w0, o);
            return o;
        }
    };
    auto run = [&](RingBuf<MODE, TC>& X, int tile) {
        prep(X, tile);
        const int want = tile * W + w, left = T - want * TC;   // steps from this slot's first on
        float s = 0.0f;
        for (int i = 0; i < kRingPolls; ++i) {
            const int q = __builtin_amdgcn_readfirstlane(*(lds_word*)&seq);
            s = *(lds_val*)&carry[lane];
            if (q == want) break;
            if (q + 1 < want) __builtin_amdgcn_s_sleep(1);   // not next: leave the issue slots alone
        }
        __builtin_amdgcn_s_setprio(3);   // the chain goes ahead of the SIMD's other wave
        __builtin_amdgcn_sched_barrier(0);
        float e = s;
        if (left >= TC) {
#pragma unroll
            for (int k = 0; k < TC; ++k) e = step(e, X, k);
        } else {
#pragma unroll
            for (int k = 0; k < TC; ++k)
                if (k < left) e = step(e, X, k);
        }
        *(lds_val*)&carry[lane] = e;
        *(lds_word*)&seq = want + 1;
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < TC; ++k)
            if (k < left) s = emit(s, X, k, t_of(tile, k));
    };
    // keeps a tile's loads where they are written, ahead of the tile before it
    auto issued = [] {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    if (w == 0) {
        carry[lane] = BACK ? 0.0f : sz;
        if (lane == 0) seq = 0;
    }
    __syncthreads();
    RingBuf<MODE, TC> P, Q;
    load(P, 0);
    int tile = 0;
    for (; tile + 2 <= ntiles; tile += 2) {
        load(Q, tile + 1);
        issued();
        run(P, tile);
        load(P, min(tile + 2, ntiles - 1));
        issued();
        run(Q, tile + 1);
    }
    if (tile < ntiles) run(P, tile);
    __syncthreads();
    if (w == 0 && valid && A.end) A.end[ch] = carry[lane];
}

template <bool GATED>
__global__ void k_recur_step(const float* __restrict__ a, const float* __restrict__ b,
                             float* __restrict__ s, long total, int N, int N8) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= total) return;
    const int n = (int)(i % N);
    const float x = a[i];
    const float bp = GATED ? mul_rn(sub_rn(1.0f, x), b[i]) : b[i];
    s[i] = (n < N8) ? fmaf(x, s[i], bp) : add_rn(mul_rn(x, s[i]), bp);
}

namespace {
template <int CPL, int W, int TC>
hipError_t launch_cfg(const float* a, const float* b, const float* s0, float* out,
                      float* send, int B, int T, int N, int gated, hipStream_t st) {
    const long lanes = ((long)B * N + CPL - 1) / CPL;
    const unsigned grid = (unsigned)((lanes + 63) / 64);
    const int N8 = N & ~7;
    const dim3 g(grid), blk(64 * W);
    if (N == N8) {
        if (gated)
            hipLaunchKernelGGL((k_recur_scan<CPL, W, TC, true, true>), g, blk, 0, st,
                               a, b, s0, out, send, B, T, N, N8);
        else
            hipLaunchKernelGGL((k_recur_scan<CPL, W, TC, false, true>), g, blk, 0, st,
                               a, b, s0, out, send, B, T, N, N8);
    } else {
        if (gated)
            hipLaunchKernelGGL((k_recur_scan<CPL, W, TC, true, false>), g, blk, 0, st,
                               a, b, s0, out, send, B, T, N, N8);
        else
            hipLaunchKernelGGL((k_recur_scan<CPL, W, TC, false, false>), g, blk, 0, st,
                               a, b, s0, out, send, B, T, N, N8);
    }
    return hipGetLastError();
}

bool aligned(const void* p, size_t n) { return (reinterpret_cast<uintptr_t>(p) % n) == 0; }

// When the ring form is taken (us a call, ring / the kernel of the layout). Its
// launch costs 1 to 2 us more than a small scan's, and past 1 us per 8192 channels
// it loads a whole tile however short T is, so it needs some length to win.
//
// Forward, layouts of the buffer kernels: below 16384 channels from more than 128
// steps (a tile of theirs) on. 1024 channels: 64 steps 5.8 / 5.1, 128 5.6 / 4.8, 192
// 5.3 / 7.9; 14336: 128 6.5 / 5.6, 192 6.9 / 9.8; at 2048 steps 4096 channels 30 /
// 58, 8192 35 / 62, 12288 64 / 66, 16384 85 / 74.
// Other layouts, one channel per lane: from 80 steps on below 4096 channels, 64
// below 12288, 48 below 24576, 32 beyond. 777 channels: 64 steps 6.4 / 6.0, 96 6.5 / 6.7; 6993: 48
// 6.9 / 6.2, 64 6.7 / 7.2; 12432: 32 6.7 / 6.0, 48 6.9 / 7.1; 32752: 24 12.3 / 11.9, 32
// 11.8 / 12.3; 2048 steps, 12012: 75 / 173.
// Two channels per lane (even widths, 24576 channels on): past one tile of 128
// steps. 32736 channels: 128 steps 16.9 / 13.3, 160 18.2 / 24.1, 2048 198 / 224; 130944:
// 128 57.8 / 55.3, 160 58.0 / 90.8, 2048 727 / 898. In the FMA form, where that
// kernel's workgroups come out even over the CUs, only to 256 steps: 32736
// channels: 256 22.0 / 23.8, 512 42.9 / 46.8, 1024 97.6 / 93.0; 65472: 256 41.1 / 48.8, 512
// 104 / 95.8; 130944: 256 97.1 / 96.2, 384 161 / 145; uneven, 49104: 512 68 / 85.
//
// Backward: up to 16384 channels from 24 steps on, in other layouts than the buffer
// kernel's beyond that too, from more steps the more channels. 128 channels: 16 steps
// 5.3 / 3.7, 24 5.1 / 4.8, 32 5.1 / 5.9; 8192: 16 5.5 / 4.5, 24 5.6 / 5.8; 32736: 32
// 10.3 / 8.9, 48 10.6 / 18.7; 98256: 64 37 / 28, 96 42 / 41, 128 63 / 96; 130944: 64
// 47 / 34, 96 62 / 80. At 2048 steps 4096 channels 54 / 961, 16384 165 / 230 (buffer
// kernel), 32768 269 / 262 (so not there).
constexpr long kRingChannels = 16384;
bool ring_pays(bool buf, int cpl, int B, int T, int N, bool gated) {
    const long chans = (long)B * N;
    if (buf) return chans < kRingChannels && T > 128;
    if (cpl == 1) return T >= (chans < 4096 ? 80 : chans < 12288 ? 64 : chans < 24576 ? 48 : 32);
    const long wgs = (long)B * ((N + 127) / 128);
    return T > 128 && (gated || T <= 256 || wgs % 256 != 0);
}
bool ring_pays_bwd(bool buf, int B, int T, int N) {
    const long chans = (long)B * N;
    if (chans <= kRingChannels) return T >= 24;
    return !buf && T >= std::min(96L, 24 + 24 * chans / 32768);
}
// Channels of a ring workgroup: half a wave where that still spreads the call over
// at most one workgroup per CU. 32 / 64 of them, us: 8192 channels backward 90 /
// 106, forward 35 / 36; 2331 channels of 333 steps backward 13 / 28; but 12288
// channels forward 73 / 64, backward 143 / 133.
int ring_ch(long chans) { return chans <= 32 * 256 ? 32 : 64; }
}  // namespace

template <int CPL, int W, int TC>
hipError_t launch_buf(const float* a, const float* b, const float* s0, float* out, float* send,
                      int B, int T, int N, int gated, hipStream_t st) {
    const unsigned grid = (unsigned)((long)B * N / (64 * CPL));
    if (gated)
        hipLaunchKernelGGL((k_recur_scan_buf<CPL, W, TC, true>), dim3(grid), dim3(64 * W), 0, st,
                           a, b, s0, out, send, T, N);
    else
        hipLaunchKernelGGL((k_recur_scan_buf<CPL, W, TC, false>), dim3(grid), dim3(64 * W), 0, st,
                           a, b, s0, out, send, T, N);
    return hipGetLastError();
}

// The ring form's 32-bit offsets: every array, with a tile past its end, below
// 2 GiB.
bool ring_scan_ok(int B, int T, int N, int row) {
    return ((long)B * T + 1024) * row * 4 < (1L << 31) && (long)B * N < (1L << 24);
}

template <int MODE, int TC>
hipError_t launch_ring(RingArgs a, int B, hipStream_t st) {
    constexpr int W = 8;
    a.total = B * a.N;
    const unsigned grid = (unsigned)((a.total + a.ch - 1) / a.ch);
    if (a.N8 == a.N) hipLaunchKernelGGL((k_scan_ring<MODE, true, W, TC>), dim3(grid), dim3(64 * W), 0, st, a);
    else hipLaunchKernelGGL((k_scan_ring<MODE, false, W, TC>), dim3(grid), dim3(64 * W), 0, st, a);
    return hipGetLastError();
}

RingArgs ring_args(const float* x0, const float* x1, const float* s0, float* y0, float* end, int B, int T, int N) {
    RingArgs a{};
    a.x0 = x0; a.x1 = x1; a.s0 = s0; a.y0 = y0; a.end = end;
    a.T = T; a.N = N; a.N8 = N; a.s0_stride = N;
    a.yT = T * N; a.yrow = N;
    a.bytes = a.ybytes = (unsigned)((size_t)B * T * N * 4);
    return a;
}

snhip_status launch_ring_gated(const float* p, const float* u, const float* s0, float* states, int B, int T,
                               int N, hipStream_t st) {
    RingArgs r = ring_args(p, u, s0, states, nullptr, B, T, N);
    r.ch = ring_ch((long)B * N);
    SNHIP_CHECK((launch_ring<SCAN_GATED, 32>(r, B, st)));
    return SNHIP_OK;
}

snhip_status launch_ring_rows(const float* p, const float* b, const float* s0, size_t s0_stride, float* states,
                              float* end, int B, int T, int N, hipStream_t st) {
    RingArgs r = ring_args(p, b, s0, states, end, B, T, N);
    r.N8 = 0;
    r.s0_stride = s0_stride;
    r.ch = ring_ch((long)B * N);
    SNHIP_CHECK((launch_ring<SCAN_FMA, 32>(r, B, st)));
    return SNHIP_OK;
}

snhip_status launch_ring_ds(const float* p, const float* dstate, float* out, int row, float* ds0, int B, int T,
                            int N, hipStream_t st) {
    RingArgs r = ring_args(p, dstate, nullptr, out, ds0, B, T, N);
    r.ch = ring_ch((long)B * N);
    r.yT = T * row;
    r.yrow = row;
    r.ybytes = (unsigned)(((size_t)B * T * row - (row - N)) * 4);   // `out` starts within its first row
    SNHIP_CHECK((launch_ring<SCAN_DS, 32>(r, B, st)));
    return SNHIP_OK;
}

// Launch-shape selection. SNHIP_SCAN_SHAPE="kind,cpl,w,tc" (kind "buf", "gen" or
// "ring"; for "ring" w is the channels of a workgroup) pins one compiled shape for
// the tuning sweep and tests; otherwise the ring form where it pays (ring_pays) and
// its 32-bit offsets reach, else the buffer kernel when the layout allows it, else
// the generic kernel.
snhip_status launch_recur_scan(const float* a, const float* b, const float* s0,
                               float* out, float* send, int B, int T, int N,
                               int gated, hipStream_t st) {
    const bool al8 = aligned(a, 8) && aligned(b, 8) && aligned(s0, 8) && aligned(out, 8) &&
                     aligned(send, 8);
    const bool al16 = aligned(a, 16) && aligned(b, 16) && aligned(s0, 16) &&
                      aligned(out, 16) && aligned(send, 16);
    const long chans = (long)B * N;
    auto buf_ok = [&](int cpl, int tile) {
        return N % (64 * cpl) == 0 && (cpl < 2 || al8) && (cpl < 4 || al16) &&
               (long)(T + tile) * N * 4 < (1L << 31);
    };
    char kind = 'g';
    int cpl = 1, w = 8, tc = 16;
    if (N % 2 == 0 && al8 && chans / 128 >= 192) cpl = 2;
    // Two channels per lane above 16384 channels, and at 16384 while one tile of it
    // holds every step; us, two / one: 16384 channels, 64 steps 5.1 / 5.6, 128 8.2 / 6.1,
    // 2048 89 / 74; 18432, 16 steps 4.1 / 5.5, 160 10.4 / 12.5, 2048 90 / 98.
    if (buf_ok(2, 2 * 32) && chans / 128 >= (T <= 64 ? 128 : 129)) { kind = 'b'; cpl = 2; w = 2; tc = 32; }
    else if (buf_ok(1, 4 * 32)) { kind = 'b'; cpl = 1; w = 4; tc = 32; }
    if (ring_pays(kind == 'b', cpl, B, T, N, gated) && ring_scan_ok(B, T, N, N)) {
        kind = 'r'; cpl = 1; w = ring_ch(chans); tc = 32;
    }
    if (const char* env = getenv("SNHIP_SCAN_SHAPE")) {
        char k[8] = {0};
        int c = 0, ww = 0, t = 0;
        if (sscanf(env, "%7[a-z],%d,%d,%d", k, &c, &ww, &t) == 4) {
            kind = k[0]; cpl = c; w = ww; tc = t;
        }
        if (kind == 'b' && !buf_ok(cpl, w * tc)) return SNHIP_E_INVAL;
        if (kind == 'r' && !ring_scan_ok(B, T, N, N)) return SNHIP_E_INVAL;
        if (kind == 'g' && ((cpl == 2 && (N % 2 || !al8)) || (cpl == 4 && (N % 4 || !al16))))
            return SNHIP_E_INVAL;
    }
    hipError_t e = hipErrorInvalidValue;
    if (kind == 'r' && cpl == 1 && w >= 1 && w <= 64 && tc == 32) {
        RingArgs r = ring_args(a, b, s0, out, send, B, T, N);
        r.N8 = N & ~7;
        r.ch = w;
        e = gated ? launch_ring<SCAN_GATED, 32>(r, B, st) : launch_ring<SCAN_FMA, 32>(r, B, st);
    } else
#define SNHIP_GEN_CASE(C, WW, TT)                                                   \
    if (kind == 'g' && cpl == C && w == WW && tc == TT)                             \
        e = launch_cfg<C, WW, TT>(a, b, s0, out, send, B, T, N, gated, st);         \
    else
#define SNHIP_BUF_CASE(C, WW, TT)                                                   \
    if (kind == 'b' && cpl == C && w == WW && tc == TT)                             \
        e = launch_buf<C, WW, TT>(a, b, s0, out, send, B, T, N, gated, st);         \
    else
    SNHIP_GEN_CASE(1, 8, 16)
    SNHIP_GEN_CASE(2, 8, 16)
    SNHIP_GEN_CASE(2, 2, 32)
    SNHIP_GEN_CASE(4, 4, 16)
    SNHIP_BUF_CASE(1, 4, 32)
    SNHIP_BUF_CASE(1, 4, 64)
    SNHIP_BUF_CASE(2, 2, 32)
    SNHIP_BUF_CASE(2, 2, 64)
    SNHIP_BUF_CASE(2, 4, 32)
    SNHIP_BUF_CASE(2, 4, 64)
    SNHIP_BUF_CASE(2, 8, 32)
    SNHIP_BUF_CASE(4, 2, 32)
    { set_last_error("SNHIP_SCAN_SHAPE names a shape that is not compiled"); return SNHIP_E_UNSUPPORTED; }
#undef SNHIP_GEN_CASE
#undef SNHIP_BUF_CASE
    if (e != hipSuccess) {
        set_last_error(std::string("recur_scan launch: ") + hipGetErrorString(e));
        return SNHIP_E_DEVICE;
    }
    return SNHIP_OK;
}

snhip_status launch_recur_step(const float* a, const float* b, float* s, int B, int N,
                               int gated, hipStream_t st) {
    const long total = (long)B * N;
    const unsigned grid = (unsigned)((total + 255) / 256);
    if (gated)
        hipLaunchKernelGGL((k_recur_step<true>), dim3(grid), dim3(256), 0, st, a, b, s, total, N, N & ~7);
    else
        hipLaunchKernelGGL((k_recur_step<false>), dim3(grid), dim3(256), 0, st, a, b, s, total, N, N & ~7);
    SNHIP_CHECK(hipGetLastError());
    return SNHIP_OK;
}

// ---------------------------------------------------------------------------
// Backward of the gated scan s_t = p_t s_{t-1} + (1 - p_t) nu_t
// (sunnynet/kernels/scan_avx2.c:50-99): per channel, in reverse time,
//   ds += dout_t;  dnu_t = ds (1 - p_t);  dp_t = ds (s_{t-1} - nu_t);  ds *= p_t
// with s_{-1} = s0, and ds0 = ds after t = 0. The reference's 8-wide path and
// scalar tail use these unfused operations in this order, so the result is
// bit-identical. Same slot pipeline as k_recur_scan_buf, walking time
// backwards: wave w owns reversed steps [w TC, (w + 1) TC) of every tile of
// W TC steps; while the active wave runs its TC dependent add/multiply pairs
// the next wave prepares s_{t-1} - nu_t and 1 - p_t, off the carried chain.
// HBM traffic per step: four reads (dout, p, nu, s_{t-1}), two writes.
template <int CPL, int W, int TC>
__global__ __launch_bounds__(64 * W)
void k_scan_bwd_buf(const float* __restrict__ p, const float* __restrict__ nu,
                    const float* __restrict__ s0, const float* __restrict__ out,
                    const float* __restrict__ dout, float* __restrict__ dp,
                    float* __restrict__ dnu, float* __restrict__ ds0, int T, int N) {
    static_assert(W >= 2, "the hand-off pipeline needs at least two waves");
    using IO = BufIO<CPL>;
    __shared__ float carry[CPL * 64];
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wg_per_row = N / (64 * CPL);
    const int bb = blockIdx.x / wg_per_row;
    const int n0 = (blockIdx.x - bb * wg_per_row) * 64 * CPL;
    const size_t row = (size_t)bb * T * N;
    const uint32_t nbytes = (uint32_t)((size_t)T * N * 4);
    const __amdgpu_buffer_rsrc_t rp = make_rsrc(p + row, nbytes);
    const __amdgpu_buffer_rsrc_t rn = make_rsrc(nu + row, nbytes);
    const __amdgpu_buffer_rsrc_t ro = make_rsrc(out + row, nbytes);
    const __amdgpu_buffer_rsrc_t rd = make_rsrc(dout + row, nbytes);
    const __amdgpu_buffer_rsrc_t rgp = make_rsrc(dp + row, nbytes);
    const __amdgpu_buffer_rsrc_t rgn = make_rsrc(dnu + row, nbytes);
    const int voff = (n0 + lane * CPL) * 4;
    const int rowb = N * 4;

    constexpr int TILE = W * TC;
    const int ntiles = (T + TILE - 1) / TILE;
    // pv: p; gv: dout; dv: nu, then s_{t-1} - nu; qv: s_{t-1}, then 1 - p.
    float pv[TC][CPL], gv[TC][CPL], dv[TC][CPL], qv[TC][CPL], sz[CPL];
    ld<CPL>(sz, s0 + (size_t)bb * N + n0 + lane * CPL);

    // Time step of reversed step k of this wave's slot in `tile`.
    auto t_of = [&](int tile, int k) { return T - 1 - (tile * TILE + w * TC + k); };
    // Steps before 0 (the last tile's tail) load step 0 (the scalar row offset
    // is not range-checked); they are never used.
    auto load_slot = [&](int tile) {
#pragma unroll
        for (int k = 0; k < TC; ++k) {
            const int t = max(t_of(tile, k), 0);
            const int so = t * rowb, sp = max(t - 1, 0) * rowb;
            IO::load(pv[k], rp, voff, so);
            IO::load(gv[k], rd, voff, so);
            IO::load(dv[k], rn, voff, so);
            IO::load(qv[k], ro, voff, sp);
        }
    };
    auto prep = [&](int tile) {
#pragma unroll
        for (int k = 0; k < TC; ++k) {
            const bool first = t_of(tile, k) == 0;           // s_{-1} is s0
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                dv[k][c] = sub_rn(first ? sz[c] : qv[k][c], dv[k][c]);
                qv[k][c] = sub_rn(1.0f, pv[k][c]);
            }
        }
    };
    auto run_slot = [&](int tile) {
        float ds[CPL];
#pragma unroll
        for (int c = 0; c < CPL; ++c) ds[c] = carry[c * 64 + lane];
#pragma unroll
        for (int k = 0; k < TC; ++k) {
            const int t = t_of(tile, k);
            if (t < 0) break;
            float gn[CPL], gp[CPL];
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                ds[c] = add_rn(gv[k][c], ds[c]);
                gn[c] = mul_rn(ds[c], qv[k][c]);
                gp[c] = mul_rn(ds[c], dv[k][c]);
                ds[c] = mul_rn(ds[c], pv[k][c]);
            }
            IO::store(rgn, voff, t * rowb, gn);
            IO::store(rgp, voff, t * rowb, gp);
        }
#pragma unroll
        for (int c = 0; c < CPL; ++c) carry[c * 64 + lane] = ds[c];
    };

    if (w == 0)
#pragma unroll
        for (int c = 0; c < CPL; ++c) carry[c * 64 + lane] = 0.0f;
    load_slot(0);
    if (w == 0) prep(0);
    __syncthreads();
    for (int tile = 0; tile < ntiles; ++tile) {
        for (int j = 0; j < W; ++j) {
            if (w == j) {
                run_slot(tile);
                if (tile + 1 < ntiles) load_slot(tile + 1);
            } else if (w == j + 1) {
                prep(tile);
            } else if (j == W - 1 && w == 0 && tile + 1 < ntiles) {
                prep(tile + 1);
            }
            barrier_lds();
        }
    }
    if (w == 0) {
        float ds[CPL];
#pragma unroll
        for (int c = 0; c < CPL; ++c) ds[c] = carry[c * 64 + lane];
        st<CPL>(ds0 + (size_t)bb * N + n0 + lane * CPL, ds);
    }
}

// Any layout: one lane per channel, straight through time.
__global__ void k_scan_bwd_gen(const float* __restrict__ p, const float* __restrict__ nu,
                               const float* __restrict__ s0, const float* __restrict__ out,
                               const float* __restrict__ dout, float* __restrict__ dp,
                               float* __restrict__ dnu, float* __restrict__ ds0, int B, int T, int N) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)B * N) return;
    const long bb = i / N;
    const int n = (int)(i - bb * N);
    const size_t rb = (size_t)bb * T * N + n;
    float ds = 0.0f;
    for (int t = T - 1; t >= 0; --t) {
        const size_t off = rb + (size_t)t * N;
        ds = add_rn(dout[off], ds);
        const float pv = p[off];
        const float sprev = t > 0 ? out[off - N] : s0[(size_t)bb * N + n];
        dnu[off] = mul_rn(ds, sub_rn(1.0f, pv));
        dp[off] = mul_rn(ds, sub_rn(sprev, nu[off]));
        ds = mul_rn(ds, pv);
    }
    ds0[(size_t)bb * N + n] = ds;
}

snhip_status launch_scan_bwd(const float* p, const float* nu, const float* s0, const float* out,
                             const float* dout, float* dp, float* dnu, float* ds0, int B, int T,
                             int N, hipStream_t st) {
    const bool al8 = aligned(p, 8) && aligned(nu, 8) && aligned(s0, 8) && aligned(out, 8) &&
                     aligned(dout, 8) && aligned(dp, 8) && aligned(dnu, 8) && aligned(ds0, 8);
    constexpr int C = 2, WW = 2, TT = 16;
    const bool buf_ok = N % (64 * C) == 0 && al8 && (long)T * N * 4 < (1L << 31);
    const bool ring_ok = ring_scan_ok(B, T, N, N);
    const bool buf = buf_ok && ((long)B * N >= kRingChannels || !ring_ok);
    if (ring_ok && ring_pays_bwd(buf_ok, B, T, N)) {
        RingArgs r = ring_args(p, dout, s0, dp, ds0, B, T, N);
        r.x2 = nu; r.x3 = out; r.y1 = dnu;
        r.ch = ring_ch((long)B * N);
        const hipError_t e = launch_ring<SCAN_BWD, 16>(r, B, st);
        if (e != hipSuccess) {
            set_last_error(std::string("scan_bwd launch: ") + hipGetErrorString(e));
            return SNHIP_E_DEVICE;
        }
    } else if (buf) {
        const unsigned grid = (unsigned)((long)B * N / (64 * C));
        hipLaunchKernelGGL((k_scan_bwd_buf<C, WW, TT>), dim3(grid), dim3(64 * WW), 0, st, p, nu, s0, out,
                           dout, dp, dnu, ds0, T, N);
    } else {
        const long total = (long)B * N;
        hipLaunchKernelGGL(k_scan_bwd_gen, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, p, nu,
                           s0, out, dout, dp, dnu, ds0, B, T, N);
    }
    SNHIP_CHECK(hipGetLastError());
    return SNHIP_OK;
}

// ---- achievable-bandwidth calibration: plain streaming kernels over the
// scan's byte pattern (two fp32 arrays read, one written) and over its reads
// alone, float4 per lane, non-temporal like the scan, grid-stride. They give
// the bandwidth a straightforward stream reaches on the device, beside the
// nominal HBM peak the scan is quoted against.
namespace {
typedef float v4f_ __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(256) void k_hbm_add(const v4f_* __restrict__ a, const v4f_* __restrict__ b,
                                                 v4f_* __restrict__ c, size_t n4) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i + stride < n4; i += 2 * stride) {
        const v4f_ x0 = __builtin_nontemporal_load(a + i), x1 = __builtin_nontemporal_load(a + i + stride);
        const v4f_ y0 = __builtin_nontemporal_load(b + i), y1 = __builtin_nontemporal_load(b + i + stride);
        __builtin_nontemporal_store(x0 + y0, c + i);
        __builtin_nontemporal_store(x1 + y1, c + i + stride);
    }
    for (; i < n4; i += stride) c[i] = a[i] + b[i];
}

__global__ __launch_bounds__(256) void k_hbm_read2(const v4f_* __restrict__ a, const v4f_* __restrict__ b,
                                                   v4f_* __restrict__ c, size_t n4) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    v4f_ acc = {0.f, 0.f, 0.f, 0.f};
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += stride)
        acc += __builtin_nontemporal_load(a + i) + __builtin_nontemporal_load(b + i);
    // one store per workgroup-sized slice of c keeps the sums live
    if (threadIdx.x == 0) c[blockIdx.x] = acc;
}
}  // namespace

}  // namespace snhip

extern "C" snhip_status snhip_abi_hbm_probe_dev(int32_t kind, const float* a, const float* b, float* c,
                                                 int64_t n, int32_t grid, void* stream) {
    using namespace snhip;
    if (!a || !b || !c || n <= 0 || n % 4 || grid <= 0 || (kind != 0 && kind != 1) ||
        !aligned(a, 16) || !aligned(b, 16) || !aligned(c, 16) || (kind == 1 && (int64_t)grid * 4 > n))
        return SNHIP_E_INVAL;
    const size_t n4 = (size_t)n / 4;
    if (kind == 0)
        hipLaunchKernelGGL(k_hbm_add, dim3((unsigned)grid), dim3(256), 0, as_stream(stream),
                           reinterpret_cast<const v4f_*>(a), reinterpret_cast<const v4f_*>(b),
                           reinterpret_cast<v4f_*>(c), n4);
    else
        hipLaunchKernelGGL(k_hbm_read2, dim3((unsigned)grid), dim3(256), 0, as_stream(stream),
                           reinterpret_cast<const v4f_*>(a), reinterpret_cast<const v4f_*>(b),
                           reinterpret_cast<v4f_*>(c), n4);
    SNHIP_CHECK(hipGetLastError());
    return SNHIP_OK;
}
