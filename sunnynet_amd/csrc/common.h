// Shared host/device helpers for the SunnyNet HIP backend (gfx950).
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <string>

#include "snhip_abi.h"
#include "streamorder.h"

namespace snhip {

// Per-thread text of the last HIP failure, exposed by snhip_abi_last_error.
void set_last_error(const std::string& msg);
const std::string& last_error();

// Records the failing call and returns SNHIP_E_DEVICE from the enclosing
// function (which must return snhip_status).
#define SNHIP_CHECK(expr)                                                     \
    do {                                                                      \
        hipError_t e_ = (expr);                                               \
        if (e_ != hipSuccess) {                                               \
            ::snhip::set_last_error(std::string(#expr) + ": " +               \
                                    hipGetErrorString(e_));                   \
            return SNHIP_E_DEVICE;                                            \
        }                                                                     \
    } while (0)

// Same, for functions returning a pointer (returns nullptr).
#define SNHIP_CHECK_NULL(expr)                                                \
    do {                                                                      \
        hipError_t e_ = (expr);                                               \
        if (e_ != hipSuccess) {                                               \
            ::snhip::set_last_error(std::string(#expr) + ": " +               \
                                    hipGetErrorString(e_));                   \
            return nullptr;                                                   \
        }                                                                     \
    } while (0)

inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

// Unsigned value of an environment variable (at least lo), or dflt if unset.
// Read at call time, so a test may change it between calls of one handle.
inline unsigned env_unsigned(const char* name, unsigned dflt, unsigned lo) {
    const char* e = getenv(name);
    if (!e) return dflt;
    const long v = atol(e);
    return v < (long)lo ? lo : (unsigned)v;
}

// Device memory of the handles. dev_alloc returns null when there is none, and
// leaves no error behind for the launches that follow; with SNHIP_MEM_LIMIT set
// (bytes, read per call) also when the handles of the process would hold more than
// that.
void* dev_alloc(size_t bytes);
void dev_free(void* p);

// A call that runs grid-synchronizing persistent kernels on `st`. enter() waits
// until what is queued on the stream is done and then for the device's gate;
// finish() waits for the call's kernels and opens the gate (so does the destructor).
// Whoever holds the gate thus waits for its own kernels only: nothing on a stream,
// of this library or not, that depends on another call's result is waited for under
// it.
class PersistCall {
public:
    explicit PersistCall(hipStream_t st) : st_(st) {}
    ~PersistCall() { (void)finish(); }
    // *alone: whether other processes are kept out too (see devgate.h); if not, the
    // gate is not held and the caller takes kernels that need no co-resident grid.
    hipError_t enter(bool* alone);
    hipError_t finish();
    PersistCall(const PersistCall&) = delete;
    PersistCall& operator=(const PersistCall&) = delete;

private:
    hipStream_t st_;
    class DeviceGate* gate_ = nullptr;   // held
};

// Launches a grid-synchronizing persistent kernel whose grid is sized to
// co-reside (checked against the kernel's occupancy when the handle is set up),
// inside a PersistCall on `st`. It is an ordinary launch: a cooperative one goes
// through a queue of its own with host-side waits on both ends, about 60 us per
// call (SunnyNet-100M fp32 B = 1 step 315 -> 258 us). What the cooperative queue
// also gave, that no two such kernels share the device, the gate keeps, among this
// process's threads and among the processes that see its files (in SNHIP_LOCK_DIR,
// by default /tmp: containers that share a card share that folder). Without the
// files a call takes the per-kernel step. SNHIP_COOP=1 launches cooperatively; the
// runtime gives the cooperative queue to one process at a time, and the launches
// of others fail.
hipError_t launch_persistent(const void* k, dim3 grid, dim3 block, void** args, hipStream_t st);

// Steps of one launch, or of the launches of one hold of the gate, so that other
// callers wait for a fraction of a second and not for a whole decode: giving the
// gate away and back costs a launch and a wait of the host, about 15 us.
constexpr int kPersistHoldSteps = 1024;

// StreamOrderT on the device.
struct HipEvents {
    using Stream = hipStream_t;
    using Event = hipEvent_t;
    using Error = hipError_t;
    static constexpr hipError_t ok = hipSuccess;
    static hipError_t capturing(Stream st, bool* c) {
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        const hipError_t e = hipStreamIsCapturing(st, &cs);
        *c = cs != hipStreamCaptureStatusNone;
        return e;
    }
    static unsigned long long id(Stream st) {
        // odd for the per-thread streams, which no handle (an address) is
        static std::atomic<unsigned long long> threads{0};
        thread_local const unsigned long long mine = 2 * ++threads + 1;
        return st == hipStreamPerThread ? mine : (unsigned long long)reinterpret_cast<uintptr_t>(st);
    }
    static hipError_t create(Event* ev) { return hipEventCreateWithFlags(ev, hipEventDisableTiming); }
    static void destroy(Event ev) { (void)hipEventDestroy(ev); }
    static hipError_t record(Event ev, Stream st) { return hipEventRecord(ev, st); }
    static hipError_t wait(Stream st, Event ev) { return hipStreamWaitEvent(st, ev, 0); }
    // also while this thread captures a stream (in the global mode such a call
    // ends the capture)
    static hipError_t host_wait(Event ev) {
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        hipError_t e = hipThreadExchangeStreamCaptureMode(&mode);
        if (e != hipSuccess) return e;
        e = hipEventSynchronize(ev);
        const hipError_t r = hipThreadExchangeStreamCaptureMode(&mode);
        return e != hipSuccess ? e : r;
    }
};
using StreamOrder = StreamOrderT<HipEvents>;

// Whether `st` may use every CU (a stream made with a CU mask may not, and a
// grid sized for the whole device would not co-reside on it).
bool stream_has_all_cus(hipStream_t st);

// Waits for this wave's outstanding LDS operations only (gfx9 s_waitcnt
// encoding: vmcnt = 63, expcnt = 7, lgkmcnt = 0); global loads stay in flight.
__device__ __forceinline__ void wait_lds() { __builtin_amdgcn_s_waitcnt(0xc07f); }

// Workgroup barrier that orders LDS traffic but does not drain outstanding
// global loads (a full __syncthreads() would wait for every prefetch).
__device__ __forceinline__ void barrier_lds() {
    wait_lds();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Reference-order arithmetic helpers. The library is compiled with
// -ffp-contract=off, so these stay separate roundings.
__device__ __forceinline__ float mul_rn(float a, float b) { return __fmul_rn(a, b); }
__device__ __forceinline__ float add_rn(float a, float b) { return __fadd_rn(a, b); }
__device__ __forceinline__ float sub_rn(float a, float b) { return __fsub_rn(a, b); }

}  // namespace snhip

// Internal launchers shared across translation units.
namespace snhip {
snhip_status launch_scan_bwd(const float* p, const float* nu, const float* s0, const float* out,
                             const float* dout, float* dp, float* dnu, float* ds0, int B, int T,
                             int N, hipStream_t st);
snhip_status launch_core_fwd(const float* q, const float* delta, const float* s0, float* states,
                             float* uo, float* po, int B, int T, int D, hipStream_t st);
snhip_status launch_core_bwd(const float* q, const float* delta, const float* s0, const float* states,
                             const float* uo, const float* po, const float* dstate, const float* du_in,
                             float* dq, float* ddelta, float* ds0, int B, int T, int D, hipStream_t st);
snhip_status launch_core_bwd_noalloc(const float* q, const float* delta, const float* s0,
                                     const float* states, const float* uo, const float* po,
                                     const float* dstate, const float* du_in, float* dq, float* ddelta,
                                     float* ds0, int B, int T, int D, hipStream_t st);
// The ring form of the recurrence (scan.hip) for arrays of `row` floats per step:
// whether its 32-bit offsets reach; states of the gated form; states and the last
// one of s = p s + b with two roundings, s0's batch rows s0_stride apart; and,
// walking time backwards from 0, ds += dstate, out = ds, ds *= p, with out's steps `row` apart
// and ds after the first step in ds0.
bool ring_scan_ok(int B, int T, int N, int row);
snhip_status launch_ring_gated(const float* p, const float* u, const float* s0, float* states, int B, int T,
                               int N, hipStream_t st);
snhip_status launch_ring_rows(const float* p, const float* b, const float* s0, size_t s0_stride, float* states,
                              float* end, int B, int T, int N, hipStream_t st);
snhip_status launch_ring_ds(const float* p, const float* dstate, float* out, int row, float* ds0, int B, int T,
                            int N, hipStream_t st);
snhip_status launch_recur_scan(const float* a, const float* b, const float* s0,
                               float* out, float* send, int B, int T, int N,
                               int gated, hipStream_t st);
snhip_status launch_recur_step(const float* a, const float* b, float* s, int B,
                               int N, int gated, hipStream_t st);
snhip_status launch_quant_i4(const float* x, uint8_t* q, float* scale, int rows,
                             int N, int block, hipStream_t st);
snhip_status launch_dequant_i4(const uint8_t* q, const float* scale, float* x,
                               int rows, int N, int block, hipStream_t st);
}  // namespace snhip
