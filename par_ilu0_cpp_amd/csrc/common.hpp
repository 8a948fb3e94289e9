// Shared host/device helpers for the gfx950 ILU(k)-GMRES library.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <stdexcept>
#include <string>

namespace pilu {

// ---------------------------------------------------------------------
// Error handling: every HIP call on the product path is checked and turns
// into std::runtime_error with the call site.
// ---------------------------------------------------------------------
[[noreturn]] void hip_fail(hipError_t e, const char* what, const char* file, int line);

// Device memory has run out: the one HIP failure that is answered by doing
// without a structure where there is another way.
struct OutOfDeviceMemory : std::runtime_error {
    using std::runtime_error::runtime_error;
};

#define PILU_HIP(call)                                                   \
    do {                                                                 \
        hipError_t pilu_e_ = (call);                                     \
        if (pilu_e_ != hipSuccess) ::pilu::hip_fail(pilu_e_, #call, __FILE__, __LINE__); \
    } while (0)

// Device allocation behind DevBuf.  Inside a SetupScope (per host thread)
// freed blocks are kept and handed out again (best fit, at most twice the
// request) instead of going back to the driver; the outermost scope's end
// synchronises its stream and frees them.  Blocks freed outside go to a bounded
// pool that all solvers allocate from.  All work on such blocks inside a
// scope must be ordered on that one stream.
void* dev_alloc(size_t bytes);
void dev_free(void* p, size_t bytes);

// The calling thread's dev_alloc call after the next `calls` ones fails as if
// device memory had run out; a negative number stops that.  For tests: no
// other code calls it.
extern "C" void par_ilu_fail_allocation(long calls);

class SetupScope {
public:
    explicit SetupScope(hipStream_t s);
    ~SetupScope();
    SetupScope(const SetupScope&) = delete;
    SetupScope& operator=(const SetupScope&) = delete;
};

// Owning device allocation (dev_alloc / dev_free).
template <typename T>
class DevBuf {
public:
    DevBuf() = default;
    explicit DevBuf(size_t count) { resize(count); }
    ~DevBuf() { release(); }
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    DevBuf(DevBuf&& o) noexcept : p_(o.p_), n_(o.n_) { o.p_ = nullptr; o.n_ = 0; }
    DevBuf& operator=(DevBuf&& o) noexcept {
        if (this != &o) { release(); p_ = o.p_; n_ = o.n_; o.p_ = nullptr; o.n_ = 0; }
        return *this;
    }
    // Grows (never shrinks) to at least `count` elements; contents are not kept.
    void reserve(size_t count) { if (count > n_) resize(count); }
    void resize(size_t count) {
        release();
        if (count) p_ = static_cast<T*>(dev_alloc(count * sizeof(T)));
        n_ = count;
    }
    void release() {
        if (p_) dev_free(p_, n_ * sizeof(T));
        p_ = nullptr;
        n_ = 0;
    }
    T* get() const { return p_; }
    size_t size() const { return n_; }
    size_t bytes() const { return n_ * sizeof(T); }

private:
    T* p_ = nullptr;
    size_t n_ = 0;
};

// ---------------------------------------------------------------------
// "Value as flag": a published FP64 value is stored with one 64-bit
// relaxed agent-scope atomic store; consumers spin with relaxed agent-scope
// atomic loads until the slot no longer holds kPending.  kPending is a
// signalling NaN; arithmetic never produces one and publish() turns any NaN
// into the canonical quiet NaN, so a published value can never look pending.
// On gfx950 these compile to plain global_load/store with sc1 (coherent at
// device scope across XCDs) and need no L2 writeback or invalidate.
// ---------------------------------------------------------------------
constexpr uint64_t kPending = 0x7FF4DEADBEEF0001ull;
constexpr uint64_t kQuietNan = 0x7FF8000000000000ull;

__device__ __forceinline__ uint64_t peek_bits(const double* p) {
    return __hip_atomic_load(reinterpret_cast<const uint64_t*>(p), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void publish(double* p, double v) {
    uint64_t b = __double_as_longlong(v);
    if (v != v) b = kQuietNan;
    __hip_atomic_store(reinterpret_cast<uint64_t*>(p), b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void publish_raw(uint64_t* p, uint64_t b) {
    __hip_atomic_store(p, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ uint64_t peek_raw(const uint64_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ int peek_int(const int* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void publish_int(int* p, int v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---------------------------------------------------------------------
// Work tickets.  Sync-free kernels hand out work in dependency order with
// one atomic ticket per workgroup: a workgroup can only wait on work held
// by a workgroup that took its ticket earlier and is therefore resident,
// so progress never depends on the hardware's dispatch order.  The last
// workgroup to finish puts the counters back to zero, so the kernel needs
// no host-side reset and can be replayed inside a graph.
// ctr[0] = next ticket, ctr[1] = finished workgroups.
// ---------------------------------------------------------------------
__device__ __forceinline__ int take_ticket(int* ctr) {
    __shared__ int s_ticket;
    if (threadIdx.x == 0)
        s_ticket = __hip_atomic_fetch_add(&ctr[0], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    return s_ticket;
}

// nblocks: workgroups that take tickets from ctr (the whole grid unless a
// launch splits its workgroups over several ticket counters).  True in thread
// 0 of the last one.
__device__ __forceinline__ bool retire_ticket(int* ctr, int nblocks = -1) {
    __syncthreads();
    if (threadIdx.x == 0) {
        int done = __hip_atomic_fetch_add(&ctr[1], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (done == (nblocks < 0 ? static_cast<int>(gridDim.x) : nblocks) - 1) {
            __hip_atomic_store(&ctr[0], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&ctr[1], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return true;
        }
    }
    return false;
}

// v of the lane K places up within the lane's row of 16 (DPP row shift; 0
// past the row's end).
template <int K>
__device__ __forceinline__ double dpp_row_shl(double v) {
    static_assert(K >= 1 && K <= 15, "row shift");
    const uint64_t b = static_cast<uint64_t>(__double_as_longlong(v));
    const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(b & 0xffffffffu), 0x100 | K, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(b >> 32), 0x100 | K, 0xf, 0xf, true);
    return __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(static_cast<uint32_t>(hi)) << 32) |
                                                       static_cast<uint32_t>(lo)));
}

// v of the lane K (16, 32) places up, in the lanes whose bit K is clear (the
// swap exchanges one operand's lanes with bit K set and the other's without).
template <int K>
__device__ __forceinline__ double upper_row(double v) {
    static_assert(K == 16 || K == 32, "row distance");
    const unsigned lo = static_cast<unsigned>(__double2loint(v)), hi = static_cast<unsigned>(__double2hiint(v));
    if constexpr (K == 32) {
        const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
        return __hiloint2double(static_cast<int>(h[1]), static_cast<int>(l[1]));
    } else {
        const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
        return __hiloint2double(static_cast<int>(h[1]), static_cast<int>(l[1]));
    }
}

// Sum over G adjacent lanes (G a power of two <= 64), valid in the group's
// first lane (the others hold partial sums).  Lane 0 adds lane G/2's value,
// then G/4's, ..., then lane 1's: the addition tree of the xor butterfly,
// so the result is deterministic for a given G.  Offsets below 16 are DPP
// row shifts, 16 and 32 row swaps: no LDS traffic.
// Every lane of the group must be active.
template <int G>
__device__ __forceinline__ double group_sum(double v) {
    if constexpr (G >= 64) v += upper_row<32>(v);
    if constexpr (G >= 32) v += upper_row<16>(v);
    if constexpr (G >= 16) v += dpp_row_shl<8>(v);
    if constexpr (G >= 8) v += dpp_row_shl<4>(v);
    if constexpr (G >= 4) v += dpp_row_shl<2>(v);
    if constexpr (G >= 2) v += dpp_row_shl<1>(v);
    return v;
}

// Sum over the wave, in every lane: within rows of 16 by DPP shifts, then the
// rows' sums in order (a fixed order; no LDS traffic, where a shuffle
// butterfly takes six dependent LDS round trips).
__device__ __forceinline__ double wave_total(double v) {
    v += dpp_row_shl<8>(v);
    v += dpp_row_shl<4>(v);
    v += dpp_row_shl<2>(v);
    v += dpp_row_shl<1>(v);
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < 64; k += 16) {
        const int lo = __builtin_amdgcn_readlane(__double2loint(v), k), hi = __builtin_amdgcn_readlane(__double2hiint(v), k);
        t += __hiloint2double(hi, lo);
    }
    return t;
}

template <int G>
__device__ __forceinline__ int group_max(int v) {
#pragma unroll
    for (int off = G / 2; off > 0; off >>= 1) {
        int o = __shfl_xor(v, off, G);
        v = o > v ? o : v;
    }
    return v;
}

// True for every lane whose G-lane group has `pred` set on all lanes.
template <int G>
__device__ __forceinline__ bool group_all(bool pred) {
    const uint64_t m = __ballot(pred);
    if constexpr (G == 64) {
        return m == ~0ull;
    } else {
        const int lane = threadIdx.x & 63;
        const int shift = lane & ~(G - 1);
        const uint64_t gm = (1ull << G) - 1ull;
        return ((m >> shift) & gm) == gm;
    }
}

// s / d with rc = 1 / d rounded to nearest: q = s rc, then one correction
// q + (s - q d) rc, correctly rounded (Markstein 1990, IBM J. Res. Dev. 34)
// as long as no intermediate leaves the normal range.  rc is 0 where d is
// outside 2^+-200 (recip_for); s outside 2^+-766 (zero, infinity and NaN
// included) in one of `lanes` takes the wave through the division itself.
__device__ __forceinline__ double recip_for(double d) {
    const unsigned e = (static_cast<unsigned>(__double2hiint(d)) >> 20) & 0x7ffu;
    return e - (1023u - 200u) <= 400u ? 1.0 / d : 0.0;
}

__device__ __forceinline__ double divide_by(double s, double d, double rc, uint64_t lanes) {
    const unsigned e = (static_cast<unsigned>(__double2hiint(s)) >> 20) & 0x7ffu;
    const uint64_t slow = (__ballot(e - 257u > 1532u) | __ballot(rc == 0.0)) & lanes;
    const double q = s * rc;
    double r = fma(fma(-q, d, s), rc, q);
    if (__builtin_expect(slow != 0, 0)) r = s / d;
    return r;
}

__device__ __forceinline__ void spin_pause() { __builtin_amdgcn_s_sleep(1); }

// Watchdog for sync-free waits: a wait that outlives `limit` ticks of the
// constant-rate device wall clock gives up, raises kErrTimeout in the
// kernel's error word and lets the kernel drain (the waiting row publishes
// NaN), so a scheduling fault turns into an error instead of a hang.
constexpr int kErrTimeout = 1 << 8;

struct Watchdog {
    uint64_t start;
    uint64_t limit;
    __device__ explicit Watchdog(uint64_t lim) : start(wall_clock64()), limit(lim) {}
    __device__ bool expired() const { return wall_clock64() - start > limit; }
};

// Back substitution of the (i + 1) x (i + 1) upper triangle hh (columns `ld`
// apart) by one wave, rs in place (src/gmres.cpp:265-272): the wave copies the
// triangle to `tri` (LDS, room for kBackMax columns) and its first lane solves
// row by row from there, in the same order; larger triangles are read where
// they are.  From memory a thread took 140 us for 50 columns.
constexpr int kBackMax = 64;
__device__ __forceinline__ void back_substitute(int i, const double* hh, long ld, double* rs, double* tri) {
    const int lane = threadIdx.x & 63;
    const bool staged = i < kBackMax;
    if (staged)
        for (int j = 0; j <= i; ++j)
            for (int k = lane; k <= j; k += 64) tri[j * kBackMax + k] = hh[j * ld + k];
    double* const x = tri + kBackMax * kBackMax;
    for (int k = lane; staged && k <= i; k += 64) x[k] = rs[k];
    __syncthreads();
    auto solve = [i](const double* t, long st, double* r) {
        r[i] = r[i] / t[i * st + i];
        for (int ii = i - 1; ii >= 0; --ii) {
            double v = r[ii];
            for (int j = ii + 1; j <= i; ++j) v -= t[j * st + ii] * r[j];
            r[ii] = v / t[ii * st + ii];
        }
    };
    if (lane == 0) {
        if (staged) solve(tri, kBackMax, x);  // apart, so that these are LDS reads
        else solve(hh, ld, rs);
    }
    __syncthreads();
    for (int k = lane; staged && k <= i; k += 64) rs[k] = x[k];
}
constexpr int kBackLds = kBackMax * (kBackMax + 1);  // doubles

// Ticks of the device wall clock in `seconds` (host side).
uint64_t watchdog_ticks(double seconds);

// Host-side phase times of the set-up path, printed to stderr when the
// environment holds PAR_ILU_TIMING (each mark first waits for `stream`).
bool phase_timing_enabled();
struct PhaseTimer {
    const char* scope;
    hipStream_t stream;
    bool on;
    double t0;
    PhaseTimer(const char* sc, hipStream_t s);
    void mark(const char* what);
};

inline int ceil_div(long a, long b) { return static_cast<int>((a + b - 1) / b); }

}  // namespace pilu
