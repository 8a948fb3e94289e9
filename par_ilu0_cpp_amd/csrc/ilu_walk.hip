// Level walk: a sweep in one workgroup, for deep and narrow schedules
// (ilu_walk.hpp).
//
// Such a sweep is bound by its chain of levels.  Level-scheduled rows over the
// whole GPU hand x on through memory, which costs a level about 1.9 us (a
// store, and the polls that find it); a barrier and LDS cost one workgroup a
// fraction of that, as long as a level is no more than its sixteen waves'
// work.  On 40k rows of 133 entries (ILU(2) of a random band: 3835 levels of
// 10 rows, FP32 factors) a sweep takes 2.7 ms here and 7.2 ms as level-scheduled
// rows.  Of a level's 0.7 us, about 0.2 go to bank conflicts of the x reads, 0.2 to
// the tree over the lanes, 0.15 to waits for the stream, the rest to the barrier
// and one step's latency.  Eight waves: four take 3.5 ms, sixteen 3.7.
//
// A task is up to 64 / G rows of one level, G lanes a row, and two rows with
// two sums per lane for G = 64, so that the tree over the lanes and the
// division are issued once for both.  Tasks go to the waves in turn, so every
// wave has its share of the stream to prefetch; rows of a level are taken by
// length, so that a task's are alike.  A step is P entries per lane and row of
// a task.  Lane t of a row sums entries t, t + G, ... in order and the lanes'
// sums are added as in k_sweep: the results are the same bits for the same G.
//
// x of the last kWalkRing schedule positions is kept in LDS; an older
// dependency is read from the output in memory.  Everything else (LDS slots,
// values, b, rows, diagonal) comes from the wave's own stream in step order,
// requested kWalkAhead steps ahead.
#include <algorithm>
#include <cstring>
#include <type_traits>

#include <rocprim/rocprim.hpp>

#include "ilu_walk.hpp"

namespace pilu {

using Ext = lljbash::IluSolver::Ext;

namespace {

constexpr int kWalkWaves = 8;
constexpr int kWalkAhead = 6;      // most steps requested ahead (k_walk); see kFacAhead for 4 and 8
constexpr int kWalkRing = 1 << 14;
constexpr unsigned kWalkFar = 0x80000000u;  // in an entry's slot: a row, to be read from memory
// step flags; the barriers before the step are counted above them
constexpr int kStepFirst = 1, kStepLast = 2, kStepFar = 4, kStepBits = 3;

// entries of a row in a direction
template <bool UPPER>
__device__ __forceinline__ int2 row_range(int row, const int* __restrict__ rp, const int* __restrict__ dg) {
    return UPPER ? make_int2(dg[row] + 1, rp[row + 1]) : make_int2(rp[row], dg[row]);
}

// Rows a lane sums for, and rows of a task; the sums of lane group h are those
// of rows h, or of both rows (G = 64).
__host__ __device__ constexpr int sums_of(int G) { return G == 64 ? 2 : 1; }
__host__ __device__ constexpr int rows_of(int G) { return G == 64 ? 2 : 64 / G; }

template <int M, int P, typename T>
struct WalkStep {
    unsigned at[M * P];  // LDS slots of the entries' x, or kWalkFar | row
    T v[M * P];
    double b[M];
    double2 d;   // u_ii, 1 / u_ii
    int row;     // the row of the lane's result, -1: none
    int2 ctl;    // flags and barriers; the task's first schedule position
};

__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Load from the L2, waited for here: a load whose wait the compiler places
// would have it wait for everything requested ahead in every step.
__device__ __forceinline__ double load_far(const double* p) {
    double v;
    asm volatile("global_load_dwordx2 %0, %1, off sc1\n\ts_waitcnt vmcnt(0)" : "=&v"(v) : "v"(p) : "memory");
    return v;
}

// N elements from an address aligned to the smaller of them all and 16 bytes.
template <int N, typename U>
__device__ __forceinline__ void load_all(const U* p, U (&v)[N]) {
    struct alignas(sizeof(U) * N < 16 ? sizeof(U) * N : 16) Pack {
        U x[N];
    };
    const Pack t = *reinterpret_cast<const Pack*>(p);
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = t.x[k];
}

// a[lane] + a[lane + 32] in the lower half, b[lane - 32] + b[lane] in the upper.
__device__ __forceinline__ double fold_two(double a, double b) {
    const unsigned al = static_cast<unsigned>(__double2loint(a)), ah = static_cast<unsigned>(__double2hiint(a));
    const unsigned bl = static_cast<unsigned>(__double2loint(b)), bh = static_cast<unsigned>(__double2hiint(b));
    const auto l = __builtin_amdgcn_permlane32_swap(al, bl, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(ah, bh, false, false);
    return __hiloint2double(static_cast<int>(h[0]), static_cast<int>(l[0])) +
           __hiloint2double(static_cast<int>(h[1]), static_cast<int>(l[1]));
}

// The rows' sums of a task, each added up as group_sum<G> does, in the first
// lane of the rows_of(G) lane groups.
template <int G>
__device__ __forceinline__ double task_sums(const double (&acc)[sums_of(G)]) {
    if constexpr (G == 64)
        return group_sum<32>(fold_two(acc[0], acc[1]));
    else
        return group_sum<G>(acc[0]);
}

// Every wave passes nlev - 1 barriers.  A far entry's row was solved at least
// 3/4 kWalkRing positions before the level (build_walk), which is 96 tasks of
// each wave or more; its wave has since consumed loads issued after the row's
// store, and a wave's vector memory operations complete in order: the store is
// in the L2 that the agent-scope load reads.
//
// A wave issues an instruction about every five cycles, so what stands between
// a barrier and the next is kept short: entries and b are converted before the
// barrier, the previous step's store and requests go out while the LDS reads
// are under way.
template <int G, int P, typename T, bool UPPER>
__global__ __launch_bounds__(kWalkWaves * 64) void k_walk(int nlev, const int* __restrict__ sbase,
                                                          const int2* __restrict__ ctl, const int* __restrict__ row,
                                                          const unsigned* __restrict__ ref, const T* __restrict__ val,
                                                          const double2* __restrict__ diag, const double* __restrict__ bt,
                                                          double* out, const int* gate) {
    extern __shared__ double xr[];  // ring, then a slot that stays 0
    if (gate && *gate == 0) return;
    constexpr int M = sums_of(G), E = M * P, R = rows_of(G);
    constexpr int D = E > 4 ? 4 : kWalkAhead;
    const int lane = threadIdx.x & 63;
    // in vector registers, so that no address is uniform: scalar loads share
    // LDS's counter and return out of order, and every LDS wait would wait for
    // the ones requested ahead
    int q = lane / (64 / R), h = lane / G, none = 0;
    asm("" : "+v"(q), "+v"(h), "+v"(none));
    const bool first = lane % G == 0, result = lane % (64 / R) == 0;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int s0 = sbase[wave], ns = sbase[wave + 1] - s0;
    if (threadIdx.x == 0) xr[kWalkRing] = 0.0;
    __syncthreads();
    int passed = 0;
    if (ns > 0) {
        // per array: this lane's element of step 0; past the wave's last step
        // (by up to 2 kWalkAhead) lie the next wave's, or unused ones
        const int2* pc = ctl + s0 + none;
        const int* pr = row + static_cast<long>(s0) * R + q;
        const unsigned* pf = ref + (static_cast<long>(s0) * 64 + lane) * E;
        const T* pv = val + (static_cast<long>(s0) * 64 + lane) * E;
        const double* pb = bt + static_cast<long>(s0) * R + h * M;
        const double2* pd = UPPER ? diag + static_cast<long>(s0) * R + q : nullptr;
        auto issue = [&](int u, WalkStep<M, P, T>& w) {
            w.ctl = pc[u];
            load_all<E>(pf + u * 64 * E, w.at);
            load_all<E>(pv + u * 64 * E, w.v);
            w.row = pr[u * R];
            load_all<M>(pb + u * R, w.b);
            if (UPPER) w.d = pd[u * R];
            // the steps' loads stay in step order: a wait is for the loads
            // before it, whichever way it was reached
            asm volatile("" ::: "memory");
        };
        WalkStep<M, P, T> ring[D];
#pragma unroll
        for (int u = 0; u < D - 1; ++u) issue(u, ring[u]);
        double acc[M], res = 0.0;
#pragma unroll
        for (int m = 0; m < M; ++m) acc[m] = 0.0;
        int done = -1;  // row of res, not stored yet
        for (int s = 0; s < ns; s += D) {
#pragma unroll
            for (int u = 0; u < D; ++u) {
                WalkStep<M, P, T>& w = ring[u];
                const bool on = s + u < ns;
                int c = 0;
                double v[E], x[E];
                if (on) {
                    unsigned at[E];
                    c = __builtin_amdgcn_readfirstlane(w.ctl.x);
#pragma unroll
                    for (int e = 0; e < E; ++e) {
                        v[e] = static_cast<double>(w.v[e]);
                        at[e] = (c & kStepFar) && (w.at[e] & kWalkFar) ? kWalkRing : w.at[e];
                    }
                    if (c & kStepFirst) {
#pragma unroll
                        for (int m = 0; m < M; ++m) acc[m] = first ? w.b[m] : 0.0;
                    }
                    for (int k = c >> kStepBits; k > 0; --k) lds_barrier();
                    passed += c >> kStepBits;
#pragma unroll
                    for (int e = 0; e < E; ++e) x[e] = xr[at[e]];
                }
                if (done >= 0) out[done] = res;
                done = -1;
                issue(u + D - 1, ring[(u + D - 1) % D]);  // outside the condition: the waits count it
                if (on) {
                    if (c & kStepFar) {
#pragma unroll
                        for (int e = 0; e < E; ++e)
                            if (w.at[e] & kWalkFar) x[e] = load_far(out + (w.at[e] & ~kWalkFar));
                    }
#pragma unroll
                    for (int e = 0; e < P; ++e)
#pragma unroll
                        for (int m = 0; m < M; ++m)
                            acc[m] = fma(-x[m * P + e], v[m * P + e], acc[m]);
                    if (c & kStepLast) {
                        res = task_sums<G>(acc);
                        if (UPPER) res = divide_by(res, w.d.x, w.d.y, __ballot(w.row >= 0));
                        done = result ? w.row : -1;
                        if (done >= 0) xr[(w.ctl.y + q) & (kWalkRing - 1)] = res;
                    }
                }
            }
            pc += D;
            pr += D * R;
            pf += D * 64 * E;
            pv += D * 64 * E;
            pb += D * R;
            if (UPPER) pd += D * R;
        }
        if (done >= 0) out[done] = res;
    }
    for (; passed < nlev - 1; ++passed) lds_barrier();
}

// b in step order.
__global__ void k_walk_b(long m, const int* __restrict__ row, const double* __restrict__ b, double* __restrict__ bt,
                         const int* gate) {
    if (gate && *gate == 0) return;
    const long i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
    if (i >= m) return;
    const int r = row[i];
    bt[i] = r >= 0 ? b[r] : 0.0;
}

__global__ void k_walk_arm(int n, uint64_t* p, const int* gate) {
    if (gate && *gate == 0) return;
    const int stride = static_cast<int>(gridDim.x * blockDim.x);
    for (long i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = kPending;
}

// ---- set-up ----

__global__ void k_walk_inv(int n, const int* __restrict__ perm, int* __restrict__ pos) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) pos[perm[k]] = k;
}

// Tasks of each level; the widest level.
__global__ void k_walk_count(int nlev, int R, const int* __restrict__ off, int* __restrict__ cnt, int* widest) {
    const int l = blockIdx.x * blockDim.x + threadIdx.x;
    if (l > nlev) return;
    const int w = l < nlev ? off[l + 1] - off[l] : 0;
    cnt[l] = (w + R - 1) / R;
    if (l < nlev) atomicMax(widest, w);
}

// Task k: level, first schedule position, rows.
struct Task {
    int lev, pos, rows;
};

__device__ __forceinline__ Task task_at(int k, int nlev, int R, const int* __restrict__ toff, const int* __restrict__ off) {
    int lo = 0, hi = nlev;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (toff[mid] <= k) lo = mid;
        else hi = mid;
    }
    const int p = off[lo] + (k - toff[lo]) * R, left = off[lo + 1] - p;
    return {lo, p, left < R ? left : R};
}

// Position of task k in wave order: the waves' tasks one wave after the other.
__device__ __forceinline__ int wave_order(int k, int per) { return k % kWalkWaves * per + k / kWalkWaves; }

// Steps of each task, in wave order.
template <bool UPPER>
__global__ void k_walk_steps(int ntask, int per, int nlev, int G, int P, const int* __restrict__ toff, const int* __restrict__ off,
                             const int* __restrict__ perm, const int* __restrict__ rp, const int* __restrict__ dg,
                             int* __restrict__ steps) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= ntask) return;
    const Task t = task_at(k, nlev, rows_of(G), toff, off);
    int most = 1;
    for (int j = 0; j < t.rows; ++j) {
        const int2 r = row_range<UPPER>(perm[t.pos + j], rp, dg);
        most = max(most, (r.y - r.x + G * P - 1) / (G * P));
    }
    steps[wave_order(k, per)] = most;
}

// The stream's pattern, one wave per task.
template <bool UPPER>
__global__ __launch_bounds__(256) void k_walk_fill(int ntask, int per, int nlev, int G, int P, const int* __restrict__ toff,
                                                   const int* __restrict__ off, const int* __restrict__ perm,
                                                   const int* __restrict__ pos, const int* __restrict__ rp,
                                                   const int* __restrict__ dg, const int* __restrict__ ci,
                                                   const int* __restrict__ first, int2* __restrict__ ctl,
                                                   int* __restrict__ row,
                                                   int* __restrict__ brow, unsigned* __restrict__ ref) {
    const int k = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (k >= ntask) return;
    const int lane = threadIdx.x & 63, t = lane % G, R = rows_of(G), M = sums_of(G);
    const Task me = task_at(k, nlev, R, toff, off);
    const int w = wave_order(k, per), s0 = first[w], n = first[w + 1] - s0;
    const int before = k < kWalkWaves ? me.lev : me.lev - task_at(k - kWalkWaves, nlev, R, toff, off).lev;
    const int end = off[me.lev + 1];
    auto row_of = [&](int j) { return j < me.rows ? perm[me.pos + j] : -1; };
    for (int s = 0; s < n; ++s) {
        const long g = s0 + s;
        bool far = false;
        for (int m = 0; m < M; ++m) {
            const int my = row_of(m * (64 / G) + lane / G);
            const int2 r = my >= 0 ? row_range<UPPER>(my, rp, dg) : make_int2(0, 0);
            for (int e = 0; e < P; ++e) {
                const int p = r.x + (s * P + e) * G + t;
                unsigned at = kWalkRing;
                if (p < r.y) {
                    const int c = ci[p], x = pos[c];
                    at = x + kWalkRing >= end ? static_cast<unsigned>(x & (kWalkRing - 1)) : kWalkFar | static_cast<unsigned>(c);
                }
                far = far || (at & kWalkFar);
                ref[((g * 64 + lane) * M + m) * P + e] = at;
            }
            if (t == 0) brow[g * R + lane / G * M + m] = my;
        }
        if (lane % (64 / R) == 0) row[g * R + lane / (64 / R)] = row_of(lane / (64 / R));
        far = __ballot(far) != 0;
        if (lane == 0)
            ctl[g] = make_int2((s == 0 ? kStepFirst | before << kStepBits : 0) | (s == n - 1 ? kStepLast : 0) |
                                   (far ? kStepFar : 0),
                               me.pos);
    }
}

// The stream's values, in the same order.
template <typename T, bool UPPER>
__global__ __launch_bounds__(256) void k_walk_gather(int ntask, int per, int nlev, int G, int P, const int* __restrict__ toff,
                                                     const int* __restrict__ off, const int* __restrict__ perm,
                                                     const int* __restrict__ rp, const int* __restrict__ dg,
                                                     const int* __restrict__ first, const T* __restrict__ fac,
                                                     T* __restrict__ val, double2* __restrict__ diag) {
    const int k = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (k >= ntask) return;
    const int lane = threadIdx.x & 63, t = lane % G, R = rows_of(G), M = sums_of(G);
    const Task me = task_at(k, nlev, R, toff, off);
    const int w = wave_order(k, per), s0 = first[w], n = first[w + 1] - s0;
    auto row_of = [&](int j) { return j < me.rows ? perm[me.pos + j] : -1; };
    for (int m = 0; m < M; ++m) {
        const int my = row_of(m * (64 / G) + lane / G);
        const int2 r = my >= 0 ? row_range<UPPER>(my, rp, dg) : make_int2(0, 0);
        for (int s = 0; s < n; ++s)
            for (int e = 0; e < P; ++e) {
                const int p = r.x + (s * P + e) * G + t;
                val[((static_cast<long>(s0 + s) * 64 + lane) * M + m) * P + e] = p < r.y ? fac[p] : T(0);
            }
    }
    if (UPPER && lane % (64 / R) == 0) {
        const int my = row_of(lane / (64 / R));
        const double d = my >= 0 ? static_cast<double>(fac[dg[my]]) : 1.0;
        for (int s = 0; s < n; ++s) diag[static_cast<long>(s0 + s) * R + lane / (64 / R)] = make_double2(d, recip_for(d));
    }
}

// Rows of a level by length: key of the row at each schedule position.
template <bool UPPER>
__global__ void k_walk_keys(int n, int nlev, int G, int P, const int* __restrict__ off, const int* __restrict__ perm,
                            const int* __restrict__ rp, const int* __restrict__ dg, unsigned* __restrict__ keys) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    int lo = 0, hi = nlev;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (off[mid] <= k) lo = mid;
        else hi = mid;
    }
    const int2 r = row_range<UPPER>(perm[k], rp, dg);
    keys[k] = static_cast<unsigned>(lo) << 4 | static_cast<unsigned>(min((r.y - r.x) / (G * P), 15));
}

inline int blocks_for(long n, int per) { return static_cast<int>(std::max<long>(1, (n + per - 1) / per)); }

template <int G, int P, typename T, bool UPPER>
void launch_walk(Ext* e, const WalkStream& w, const T* val, const double* b, double* out, const int* gate) {
    auto kern = k_walk<G, P, T, UPPER>;
    constexpr int lds = (kWalkRing + 1) * sizeof(double);
    PILU_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    const long m = w.steps * rows_of(G);
    k_walk_b<<<blocks_for(m, 256), 256, 0, e->stream>>>(m, w.brow.get(), b, w.bt.get(), gate);
    kern<<<1, kWalkWaves * 64, lds, e->stream>>>(w.nlev, w.sbase.get(), w.ctl.get(), w.row.get(), w.ref.get(), val,
                                                 reinterpret_cast<const double2*>(w.diag.get()), w.bt.get(), out, gate);
}

template <typename T, bool UPPER>
void walk_t(Ext* e, const WalkStream& w, const T* val, const double* b, double* out, const int* gate) {
    switch (w.g) {
        case 4: launch_walk<4, 2, T, UPPER>(e, w, val, b, out, gate); break;
        case 8: launch_walk<8, 2, T, UPPER>(e, w, val, b, out, gate); break;
        case 16: launch_walk<16, 2, T, UPPER>(e, w, val, b, out, gate); break;
        case 32: launch_walk<32, 2, T, UPPER>(e, w, val, b, out, gate); break;
        default:
            if (w.p == 2) launch_walk<64, 2, T, UPPER>(e, w, val, b, out, gate);
            else launch_walk<64, 4, T, UPPER>(e, w, val, b, out, gate);
    }
}

}  // namespace

bool build_walk(Ext* e, bool upper, int G, WalkStream& w) {
    w.steps = 0;
    const int n = e->n, nlev = upper ? e->nlev_u : e->nlev_l;
    if (G < 4 || n <= 0 || nlev >= (1 << 24)) return false;
    hipStream_t s = e->stream;
    const int* by_level = (upper ? e->perm_u : e->perm_l).get();
    const int* off = (upper ? e->lvoff_u : e->lvoff_l).get();
    const int R = rows_of(G);
    // rows of up to G entries on average need one step or two with two entries
    // per lane; for longer ones four save steps
    const int P = G == 64 && e->nnz - n > 2L * 96 * n ? 4 : 2;
    DevBuf<unsigned> keys(n), keys_out(n);
    w.perm.reserve(n);
    if (upper) k_walk_keys<true><<<blocks_for(n, 256), 256, 0, s>>>(n, nlev, G, P, off, by_level, e->rp.get(), e->dg.get(), keys.get());
    else k_walk_keys<false><<<blocks_for(n, 256), 256, 0, s>>>(n, nlev, G, P, off, by_level, e->rp.get(), e->dg.get(), keys.get());
    unsigned bits = 5;
    while (bits < 32 && (1u << (bits - 4)) < static_cast<unsigned>(nlev)) ++bits;
    size_t sort_bytes = 0;
    PILU_HIP(rocprim::radix_sort_pairs(nullptr, sort_bytes, keys.get(), keys_out.get(), by_level, w.perm.get(),
                                       static_cast<unsigned>(n), 0u, bits, s));
    e->sort_tmp.reserve(sort_bytes);
    PILU_HIP(rocprim::radix_sort_pairs(e->sort_tmp.get(), sort_bytes, keys.get(), keys_out.get(), by_level, w.perm.get(),
                                       static_cast<unsigned>(n), 0u, bits, s));
    const int* perm = w.perm.get();
    auto scan = [&](const int* in, int* out, size_t m) {
        size_t bytes = 0;
        PILU_HIP(rocprim::exclusive_scan(nullptr, bytes, in, out, 0, m, rocprim::plus<int>(), s));
        e->sort_tmp.reserve(bytes);
        PILU_HIP(rocprim::exclusive_scan(e->sort_tmp.get(), bytes, in, out, 0, m, rocprim::plus<int>(), s));
    };
    DevBuf<int> pos(n), cnt(static_cast<size_t>(nlev) + 1), widest(1);
    w.toff.reserve(static_cast<size_t>(nlev) + 1);
    PILU_HIP(hipMemsetAsync(widest.get(), 0, sizeof(int), s));
    k_walk_inv<<<blocks_for(n, 256), 256, 0, s>>>(n, perm, pos.get());
    k_walk_count<<<blocks_for(nlev + 1, 256), 256, 0, s>>>(nlev, R, off, cnt.get(), widest.get());
    scan(cnt.get(), w.toff.get(), static_cast<size_t>(nlev) + 1);
    int ntask = 0, wide = 0;
    PILU_HIP(hipMemcpyAsync(&ntask, w.toff.get() + nlev, sizeof(int), hipMemcpyDeviceToHost, s));
    PILU_HIP(hipMemcpyAsync(&wide, widest.get(), sizeof(int), hipMemcpyDeviceToHost, s));
    PILU_HIP(hipStreamSynchronize(s));
    if (wide > kWalkRing / 4) return false;
    const int per = (ntask + kWalkWaves - 1) / kWalkWaves;
    const size_t nt = static_cast<size_t>(per) * kWalkWaves + 1;
    DevBuf<int> steps(nt);
    w.first.reserve(nt);
    PILU_HIP(hipMemsetAsync(steps.get(), 0, nt * sizeof(int), s));
    if (upper)
        k_walk_steps<true><<<blocks_for(ntask, 256), 256, 0, s>>>(ntask, per, nlev, G, P, w.toff.get(), off, perm, e->rp.get(),
                                                                  e->dg.get(), steps.get());
    else
        k_walk_steps<false><<<blocks_for(ntask, 256), 256, 0, s>>>(ntask, per, nlev, G, P, w.toff.get(), off, perm, e->rp.get(),
                                                                   e->dg.get(), steps.get());
    scan(steps.get(), w.first.get(), nt);
    w.sbase.reserve(kWalkWaves + 1);
    PILU_HIP(hipMemcpy2DAsync(w.sbase.get(), sizeof(int), w.first.get(), sizeof(int) * per, sizeof(int), kWalkWaves + 1,
                              hipMemcpyDeviceToDevice, s));
    int total = 0;
    PILU_HIP(hipMemcpyAsync(&total, w.first.get() + nt - 1, sizeof(int), hipMemcpyDeviceToHost, s));
    PILU_HIP(hipStreamSynchronize(s));
    const size_t held = static_cast<size_t>(total) + 2 * kWalkAhead;
    // slots and values of the entries; per row its id, twice, b and the diagonal
    const size_t step_bytes = 64 * P * sums_of(G) * (sizeof(int) + sizeof(double)) + R * (2 * sizeof(int) + 3 * sizeof(double)) + sizeof(int2);
    if (held * step_bytes > e->stream_budget()) return false;
    w.ctl.reserve(held);
    w.row.reserve(held * R);
    w.brow.reserve(held * R);
    w.bt.reserve(held * R);
    w.ref.reserve(held * 64 * P * sums_of(G));
    if (upper)
        k_walk_fill<true><<<blocks_for(ntask, 4), 256, 0, s>>>(ntask, per, nlev, G, P, w.toff.get(), off, perm, pos.get(),
                                                               e->rp.get(), e->dg.get(), e->ci.get(), w.first.get(),
                                                               w.ctl.get(), w.row.get(), w.brow.get(), w.ref.get());
    else
        k_walk_fill<false><<<blocks_for(ntask, 4), 256, 0, s>>>(ntask, per, nlev, G, P, w.toff.get(), off, perm, pos.get(),
                                                                e->rp.get(), e->dg.get(), e->ci.get(), w.first.get(),
                                                                w.ctl.get(), w.row.get(), w.brow.get(), w.ref.get());
    PILU_HIP(hipGetLastError());
    w.g = G;
    w.p = P;
    w.nlev = nlev;
    w.ntask = ntask;
    w.per = per;
    w.factors = -1;
    w.steps = total;
    return true;
}

void gather_walk(Ext* e, bool upper, WalkStream& w) {
    refuse_if_no_alloc(e, "sweep stream values");
    const int* perm = w.perm.get();
    const int* off = (upper ? e->lvoff_u : e->lvoff_l).get();
    const size_t held = static_cast<size_t>(w.steps) + 2 * kWalkAhead;
    if (upper) w.diag.reserve(2 * held * rows_of(w.g));
    double2* diag = reinterpret_cast<double2*>(w.diag.get());
    auto run = [&](auto* fac, auto* val) {
        using T = std::remove_pointer_t<decltype(val)>;
        if (upper)
            k_walk_gather<T, true><<<blocks_for(w.ntask, 4), 256, 0, e->stream>>>(
                w.ntask, w.per, w.nlev, w.g, w.p, w.toff.get(), off, perm, e->rp.get(), e->dg.get(), w.first.get(), fac, val, diag);
        else
            k_walk_gather<T, false><<<blocks_for(w.ntask, 4), 256, 0, e->stream>>>(
                w.ntask, w.per, w.nlev, w.g, w.p, w.toff.get(), off, perm, e->rp.get(), e->dg.get(), w.first.get(), fac, val, diag);
    };
    const size_t cnt = held * 64 * w.p * sums_of(w.g);
    if (e->precision == 32) {
        w.val32.reserve(cnt);
        run(e->fac32.get(), w.val32.get());
    } else {
        w.val64.reserve(cnt);
        run(e->fac.get(), w.val64.get());
    }
    PILU_HIP(hipGetLastError());
    w.factors = e->factor_version;
}

void sweep_walk(Ext* e, bool upper, const WalkStream& w, const double* b, double* out, double* reset, const int* gate) {
    if (w.steps == 0 || w.factors != e->factor_version)
        throw std::runtime_error("level walk: stream missing (factorize before sweeping)");
    if (e->precision == 32) {
        if (upper) walk_t<float, true>(e, w, w.val32.get(), b, out, gate);
        else walk_t<float, false>(e, w, w.val32.get(), b, out, gate);
    } else {
        if (upper) walk_t<double, true>(e, w, w.val64.get(), b, out, gate);
        else walk_t<double, false>(e, w, w.val64.get(), b, out, gate);
    }
    if (reset)
        k_walk_arm<<<std::min(blocks_for(e->n, 256), 2048), 256, 0, e->stream>>>(e->n, reinterpret_cast<uint64_t*>(reset), gate);
}

}  // namespace pilu
