// Batched ILU(k)-GMRES(m): many independent systems, several right-hand
// sides each, solved together.  No counterpart in the reference, which
// solves one system per call (src/gmres.cpp:138-288); every (system, RHS)
// pair here runs exactly that iteration, with its own Krylov basis,
// Hessenberg matrix, tolerance and step count.
//
// Layout.  The systems are one block-diagonal CSR matrix (system s owns rows
// sys_ptr[s] .. sys_ptr[s+1]); ILU(k) of a block-diagonal matrix is the
// per-block ILU(k), so one symbolic pass, one factorization launch and one
// launch per sweep serve every system.  Vectors are stored RHS-interleaved,
// X[row * K + r], so the K values of a row are one 64-byte line at K = 8.
//
// Work decomposition.  Rows are cut into chunks of at most kChunkElems / K that
// never cross a system boundary; reductions are per chunk and per RHS, and
// an instance's total is the fixed-order sum over its system's chunks.  The
// scalar part (step condition, Givens, back-solve) runs one thread per
// instance.  One restart cycle is a fixed kernel sequence, captured once in
// a HIP graph and replayed until every instance has finished.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <stdexcept>
#include <string>
#include <vector>

#include "ilu_internal.hpp"
#include "par_ilu_ex.h"

namespace pilu {

namespace {

constexpr int kBThreads = 256;
constexpr int kBPer = 16;                       // vector elements per thread of a chunk
constexpr int kChunkElems = kBThreads * kBPer;  // rows x right-hand sides of a chunk

struct BCtl {
    int its, maxits, cycle_active, step_active, i, status, breakdown, done;
    double tol, beta, inv, pad;
};

// ---- multi-RHS sweep: one workgroup per system ----
// Workgroup s walks the (level, row) groups of system s in order (perm,
// sys_grp, grp_off from block_level_schedule with the systems as blocks);
// the K right-hand sides of a row are K adjacent lanes.  Rows of one level
// are independent and the levels are separated by a workgroup barrier, so
// no cross-workgroup waits are needed.  Each lane sums its row in entry
// order from b, one fma per entry, as the single-system sweep with one lane
// per row does.  A system with no instance running the current Arnoldi step
// returns at once.
//
// Software pipeline: everything a row needs except the x of its
// dependencies (its position, bounds, first kSsE columns and values, b and
// the diagonal) comes from the pattern, the factors or the input vector, so
// it is requested one level ahead for the first kSsSlots row slots of every
// thread; a level then waits only for its x reads, which hit the lines this
// workgroup wrote before the barrier.  Further slots and entries are read
// directly.
constexpr int kSThreads = 1024;
constexpr int kSsE = 4;
constexpr int kSsSlots = 2;

template <typename T>
struct SsRow {
    int row, e, end;
    int c[kSsE];
    T v[kSsE];
    T dv;
    double bv;
};

template <int K, typename T, bool UPPER>
__device__ __forceinline__ void ss_fetch(int p, int p1, int r, const int* __restrict__ perm, const int* __restrict__ rp,
                                         const int* __restrict__ ci, const int* __restrict__ dg,
                                         const T* __restrict__ val, const double* b, SsRow<T>& t) {
    t.row = -1;
    t.e = t.end = 0;
    if (p >= p1) return;
    t.row = perm[p];
    const int d = dg[t.row];
    t.e = UPPER ? d + 1 : rp[t.row];
    t.end = UPPER ? rp[t.row + 1] : d;
#pragma unroll
    for (int q = 0; q < kSsE; ++q)
        if (t.e + q < t.end) {
            t.c[q] = ci[t.e + q];
            t.v[q] = val[t.e + q];
        }
    if (UPPER) t.dv = val[d];
    t.bv = b[static_cast<long>(t.row) * K + r];
}

template <int K, typename T, bool UPPER>
__device__ __forceinline__ void ss_solve(const SsRow<T>& t, int r, const int* __restrict__ ci,
                                         const T* __restrict__ val, double* out) {
    if (t.row < 0) return;
    double acc = t.bv;
#pragma unroll
    for (int q = 0; q < kSsE; ++q)
        if (t.e + q < t.end) acc = fma(-out[static_cast<long>(t.c[q]) * K + r], static_cast<double>(t.v[q]), acc);
    for (int e = t.e + kSsE; e < t.end; ++e)
        acc = fma(-out[static_cast<long>(ci[e]) * K + r], static_cast<double>(val[e]), acc);
    out[static_cast<long>(t.row) * K + r] = UPPER ? acc / static_cast<double>(t.dv) : acc;
}

template <int K, typename T, bool UPPER>
__global__ __launch_bounds__(kSThreads) void k_ssweep(const int* __restrict__ sys_grp, const int* __restrict__ grp_off,
                                                      const int* __restrict__ perm, const int* __restrict__ rp,
                                                      const int* __restrict__ ci, const int* __restrict__ dg,
                                                      const T* __restrict__ val, const double* b, double* out,
                                                      const BCtl* ctl) {
    constexpr int kRowsPerPass = kSThreads / K;
    const int s = blockIdx.x;
    if (ctl) {
        bool any = false;
#pragma unroll
        for (int r = 0; r < K; ++r) any = any || ctl[s * K + r].step_active != 0;
        if (!any) return;
    }
    const int r = threadIdx.x % K;
    const int slot = static_cast<int>(threadIdx.x) / K;
    const int g0 = sys_grp[s], g1 = sys_grp[s + 1];
    SsRow<T> nxt[kSsSlots];
#pragma unroll
    for (int k = 0; k < kSsSlots; ++k) nxt[k].row = -1;
    if (g0 < g1) {
        const int q0 = grp_off[g0], q1 = grp_off[g0 + 1];
#pragma unroll
        for (int k = 0; k < kSsSlots; ++k)
            ss_fetch<K, T, UPPER>(q0 + slot + k * kRowsPerPass, q1, r, perm, rp, ci, dg, val, b, nxt[k]);
    }
    for (int g = g0; g < g1; ++g) {
        const int p0 = grp_off[g], p1 = grp_off[g + 1];
        SsRow<T> cur[kSsSlots];
#pragma unroll
        for (int k = 0; k < kSsSlots; ++k) cur[k] = nxt[k];
        if (g + 1 < g1) {
            const int n1 = grp_off[g + 2];
#pragma unroll
            for (int k = 0; k < kSsSlots; ++k)
                ss_fetch<K, T, UPPER>(p1 + slot + k * kRowsPerPass, n1, r, perm, rp, ci, dg, val, b, nxt[k]);
        }
#pragma unroll
        for (int k = 0; k < kSsSlots; ++k) ss_solve<K, T, UPPER>(cur[k], r, ci, val, out);
        for (int p = p0 + slot + kSsSlots * kRowsPerPass; p < p1; p += kRowsPerPass) {
            SsRow<T> t;
            ss_fetch<K, T, UPPER>(p, p1, r, perm, rp, ci, dg, val, b, t);
            ss_solve<K, T, UPPER>(t, r, ci, val, out);
        }
        __syncthreads();
    }
}

// ---- multi-RHS sweep over rounds ----
// The rows of a system in level order are cut into rounds of up to
// blockDim / KP rows of one level; a workgroup takes KP of a system's
// right-hand sides, KP adjacent lanes per row.  x of the last rows solved is
// kept in an LDS ring indexed by schedule position: the set-up checks that
// every dependency is still in the ring when its row is solved (in a banded
// or grid ordering a dependency lies a few levels back), so a level costs an
// LDS read, the row's fmas, an LDS write and an LDS-only barrier.  Everything
// else (columns as ring slots, values, row ids, {u_ii, 1 / u_ii}, b) is
// requested kBrAhead rounds ahead from a stream in round order.  Rows are
// summed in entry order from b, one fma per entry, as k_ssweep does.
//
// Bound by the level chain.  k_ssweep's x went through memory (a store, a
// barrier that waits for it, a load): 333 + 360 us per L + U pair on 40
// systems of 45^2 to 110^2 (219 levels at most), one workgroup per system.
// Rounds ahead for values, columns, diagonal and b, and for the row ids that give
// b's address (fetched before the former and replaced after).  40 systems x 8
// right-hand sides: 53.3 ms a solve, 59.4 with two.
constexpr int kBrAhead = 4;
constexpr int kBrAheadRow = 8;
static_assert(kBrAhead < kBrAheadRow && kBrAheadRow % kBrAhead == 0, "the ring indexes of k_bsweep");
constexpr size_t kBrMaxLds = 64 * 1024;

template <int S, typename T>
struct BrRow {
    int c[S];
    T v[S];
    double2 d;
    double b;
};

template <int KP, int S, typename T, bool UPPER>
__global__ __launch_bounds__(1024) void k_bsweep(const int* __restrict__ rptr, const int2* __restrict__ rid,
                                                 const int* __restrict__ col, const T* __restrict__ val,
                                                 const double2* __restrict__ diag, const double* b, double* out, int nsys,
                                                 int K, int ring, const BCtl* ctl) {
    extern __shared__ double xr[];  // ring slots, then one that stays 0
    // the workgroups of a system's right-hand sides run on one XCD (workgroup
    // w on XCD w % 8), whose L2 then holds the lines they share
    const int per = K / KP;
    const int s = static_cast<int>(blockIdx.x >> 3) / per * 8 + (blockIdx.x & 7);
    const int r0 = static_cast<int>(blockIdx.x >> 3) % per * KP;
    if (s >= nsys) return;
    if (ctl) {
        bool any = false;
#pragma unroll
        for (int r = 0; r < KP; ++r) any = any || ctl[s * K + r0 + r].step_active != 0;
        if (!any) return;
    }
    const int rr = threadIdx.x % KP, j = threadIdx.x / KP, rows = blockDim.x / KP;
    const int q0 = rptr[s], nr = rptr[s + 1] - q0;
    if (nr <= 0) return;
    if (j == 0) xr[ring * KP + rr] = 0.0;
    auto at = [&](int q) { return static_cast<long>(q0 + (q < nr ? q : nr - 1)) * rows + j; };
    auto issue = [&](int q, const int2& id, BrRow<S, T>& t) {
        const long k = at(q);
#pragma unroll
        for (int e = 0; e < S; ++e) {
            t.c[e] = col[k * S + e];
            t.v[e] = val[k * S + e];
        }
        if (UPPER) t.d = diag[k];
        t.b = b[static_cast<long>(id.x < 0 ? 0 : id.x) * K + r0 + rr];
    };
    int2 id[kBrAheadRow];
    BrRow<S, T> rec[kBrAhead];
#pragma unroll
    for (int u = 0; u < kBrAheadRow; ++u) id[u] = rid[at(u)];
#pragma unroll
    for (int u = 0; u < kBrAhead; ++u) issue(u, id[u], rec[u]);
    __syncthreads();
    for (int q = 0; q < nr; q += kBrAheadRow) {
#pragma unroll
        for (int u = 0; u < kBrAheadRow; ++u) {
            const int2 me = id[u];
            BrRow<S, T>& t = rec[u % kBrAhead];
            if (q + u < nr) {
                double acc = t.b;
#pragma unroll
                for (int e = 0; e < S; ++e) acc = fma(-xr[t.c[e] * KP + rr], static_cast<double>(t.v[e]), acc);
                if (UPPER) acc = divide_by(acc, t.d.x, t.d.y, ~0ull);
                if (me.x >= 0) {
                    xr[(me.y & 0x7fffffff) * KP + rr] = acc;
                    out[static_cast<long>(me.x) * K + r0 + rr] = acc;
                }
                if (__builtin_amdgcn_readfirstlane(me.y) < 0) {  // last round of its level
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
                    __builtin_amdgcn_s_barrier();
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
                }
            }
            issue(q + u + kBrAhead, id[(u + kBrAhead) % kBrAheadRow], t);
            id[u] = rid[at(q + u + kBrAheadRow)];
        }
    }
}

__global__ void k_br_inv(int n, const int* __restrict__ perm, int* __restrict__ kinv) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) kinv[perm[k]] = k;
}

// Longest way, in schedule positions, from a row's dependency to the end of
// the row's level.
template <bool UPPER>
__global__ void k_br_reach(int ngroups, const int* __restrict__ off, const int* __restrict__ perm,
                           const int* __restrict__ kinv, const int* __restrict__ rp, const int* __restrict__ dg,
                           const int* __restrict__ ci, int* reach) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= ngroups) return;
    int m = 0;
    for (int k = off[g]; k < off[g + 1]; ++k) {
        const int row = perm[k], e1 = UPPER ? rp[row + 1] : dg[row];
        for (int e = UPPER ? dg[row] + 1 : rp[row]; e < e1; ++e) m = max(m, off[g + 1] - kinv[ci[e]]);
    }
    atomicMax(reach, m);
}

// Stream of row j of every round {first position, rows, level ends, first
// position of the system}: (row or -1, ring slot | level end), the entries'
// ring slots and factor positions (-1: none, the slot that stays 0).
template <bool UPPER>
__global__ void k_br_fill(long total, int rows, int S, int ring, const int4* __restrict__ rounds,
                          const int* __restrict__ perm, const int* __restrict__ kinv, const int* __restrict__ rp,
                          const int* __restrict__ dg, const int* __restrict__ ci, int2* __restrict__ rid,
                          int* __restrict__ col, int* __restrict__ src) {
    const long i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
    if (i >= total) return;
    const int4 r = rounds[i / rows];
    const int j = static_cast<int>(i % rows);
    int row = -1, own = 0, e0 = 0, cnt = 0;
    if (j < r.y) {
        row = perm[r.x + j];
        own = (r.x + j - r.w) & (ring - 1);
        e0 = UPPER ? dg[row] + 1 : rp[row];
        cnt = (UPPER ? rp[row + 1] : dg[row]) - e0;
    }
    rid[i] = make_int2(row, own | (r.z ? static_cast<int>(0x80000000u) : 0));
    for (int e = 0; e < S; ++e) {
        col[i * S + e] = e < cnt ? (kinv[ci[e0 + e]] - r.w) & (ring - 1) : ring;
        src[i * S + e] = e < cnt ? e0 + e : -1;
    }
}

template <typename T>
__global__ void k_br_gather(long total, int S, const int* __restrict__ src, const T* __restrict__ fac,
                            T* __restrict__ val, const int2* __restrict__ rid, const int* __restrict__ dg,
                            double2* __restrict__ diag) {
    const long i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
    if (i >= total) return;
    for (int e = 0; e < S; ++e) {
        const int k = src[i * S + e];
        val[i * S + e] = k >= 0 ? fac[k] : T(0);
    }
    if (diag) {
        const int row = rid[i].x;
        const double d = row >= 0 ? static_cast<double>(fac[dg[row]]) : 1.0;
        diag[i] = make_double2(d, recip_for(d));
    }
}

// Sum over the threads of a block that share t % K; result valid in
// threads t < K (one per RHS).  Fixed order.
template <int K>
__device__ double rhs_reduce(double v, double* s_red) {
#pragma unroll
    for (int off = K; off < 64; off <<= 1) v += __shfl_xor(v, off, 64);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();
    if (lane < K) s_red[wave * K + lane] = v;
    __syncthreads();
    double t = 0.0;
    if (threadIdx.x < K)
        for (int w = 0; w < kBThreads / 64; ++w) t += s_red[w * K + threadIdx.x];
    return t;
}

// Instance total of chunk partials part[c*K + r] over the system's chunks.
__device__ __forceinline__ double system_sum(const double* part, const int* sys_chunk, int s, int r, int K) {
    double t = 0.0;
    for (int c = sys_chunk[s]; c < sys_chunk[s + 1]; ++c) t += part[static_cast<long>(c) * K + r];
    return t;
}

// True when some instance of system s still needs this chunk: with
// step == true, an instance running the current Arnoldi step; otherwise an
// instance not yet finished.  Uniform over the block, so a chunk of a system
// whose right-hand sides have all converged costs one small read.
template <int K>
__device__ __forceinline__ bool system_live(const BCtl* ctl, int s, bool step) {
    bool any = false;
#pragma unroll
    for (int r = 0; r < K; ++r) {
        const BCtl& q = ctl[s * K + r];
        any = any || (step ? q.step_active != 0 : q.done == 0);
    }
    return any;
}

// Y = alpha A X + beta Yin on one chunk per block; part[c*K+r] = partial of
// dotv.Y (dotv != null) or Y.Y (nrm).  With ctl, chunks of systems that
// need no work (system_live) are skipped.
template <int K>
__global__ __launch_bounds__(kBThreads) void k_bspmv(const int* __restrict__ chunk_beg, const int* __restrict__ rp,
                                                     const int* __restrict__ ci, const double* __restrict__ val,
                                                     double alpha, const double* __restrict__ x, double beta,
                                                     const double* yin, double* y, const double* __restrict__ dotv,
                                                     bool nrm, double* part, const int* __restrict__ chunk_sys,
                                                     const BCtl* ctl, bool step) {
    __shared__ double s_red[(kBThreads / 64) * K];
    const int c = blockIdx.x;
    if (ctl && !system_live<K>(ctl, chunk_sys[c], step)) return;
    const int r = threadIdx.x % K;
    const int rb = chunk_beg[c], re = chunk_beg[c + 1];
    double acc = 0.0;
    for (int row = rb + threadIdx.x / K; row < re; row += kBThreads / K) {
        // kSpE entries requested together, summed in entry order
        constexpr int kSpE = 5;
        double s = 0.0;
        const int e1 = rp[row + 1];
        for (int e = rp[row]; e < e1; e += kSpE) {
            double a[kSpE], xe[kSpE];
#pragma unroll
            for (int q = 0; q < kSpE; ++q) {
                const int k = e + q < e1 ? e + q : e1 - 1;
                a[q] = val[k];
                xe[q] = x[static_cast<long>(ci[k]) * K + r];
            }
#pragma unroll
            for (int q = 0; q < kSpE; ++q)
                if (e + q < e1) s = fma(a[q], xe[q], s);
        }
        const long o = static_cast<long>(row) * K + r;
        const double v = beta == 0.0 ? alpha * s : beta * yin[o] + alpha * s;
        y[o] = v;
        if (dotv) acc = fma(dotv[o], v, acc);
        else if (nrm) acc = fma(v, v, acc);
    }
    if (part) {
        const double t = rhs_reduce<K>(acc, s_red);
        if (threadIdx.x < K) part[static_cast<long>(c) * K + threadIdx.x] = t;
    }
}

// MGS term j of step i for every instance: h = (v_j, w); w -= h v_j; next partials.
template <int K>
__global__ __launch_bounds__(kBThreads) void k_bmgs(const int* __restrict__ list, const int* __restrict__ chunk_beg,
                                                    const int* __restrict__ chunk_sys,
                                                    const int* __restrict__ sys_chunk, const double* __restrict__ vj,
                                                    double* w, const double* __restrict__ vnext,
                                                    const double* part_in, double* part_out, double* hh, long hstride,
                                                    int hpos, const BCtl* ctl) {
    __shared__ double s_red[(kBThreads / 64) * K];
    const int c = list[blockIdx.x];
    const int s = chunk_sys[c];
    if (!system_live<K>(ctl, s, true)) return;
    const int r = threadIdx.x % K;
    const double h = system_sum(part_in, sys_chunk, s, r, K);
    if (c == sys_chunk[s] && threadIdx.x < K) hh[(static_cast<long>(s) * K + r) * hstride + hpos] = h;
    const int rb = chunk_beg[c], re = chunk_beg[c + 1];
    double acc = 0.0;
    for (long o = static_cast<long>(rb) * K + threadIdx.x; o < static_cast<long>(re) * K; o += kBThreads) {
        const double wr = fma(-h, vj[o], w[o]);
        w[o] = wr;
        acc = fma(vnext ? vnext[o] : wr, wr, acc);
    }
    const double t = rhs_reduce<K>(acc, s_red);
    if (threadIdx.x < K) part_out[static_cast<long>(c) * K + threadIdx.x] = t;
}

// End of Arnoldi step i of one instance (src/gmres.cpp:226-262) with ||w|| = t:
// breakdown test, earlier rotations on column i, new rotation, estimate.
// col holds h_0 .. h_i; c and s the rotations (their i-th is set); rs the
// right-hand side's two entries touched.
__device__ __forceinline__ void b_givens(BCtl& q, int i, double t, double* col, double* c, double* s, double* rs,
                                         int stride) {
    col[(i + 1) * stride] = t;
    if (t <= 1e-16) {
        q.breakdown = 1;
        q.cycle_active = 0;
        return;
    }
    q.inv = 1.0 / t;
    for (int k = 1; k <= i; ++k) {
        const int k1 = k - 1;
        const double tk = col[k1 * stride], tn = col[k * stride];
        col[k1 * stride] = c[k1 * stride] * tk + s[k1 * stride] * tn;
        col[k * stride] = -s[k1 * stride] * tk + c[k1 * stride] * tn;
    }
    const double a = col[i * stride], b = col[(i + 1) * stride];
    double gam = std::sqrt(a * a + b * b);
    if (gam == 0.0) gam = 1e-16;
    c[i * stride] = a / gam;
    s[i * stride] = b / gam;
    rs[1] = -s[i * stride] * rs[0];
    rs[0] = c[i * stride] * rs[0];
    col[i * stride] = c[i * stride] * a + s[i * stride] * b;
    q.beta = std::fabs(rs[1]);
    if (std::isnan(q.beta)) {
        q.status = 2;
        q.done = 1;
        q.cycle_active = 0;
    }
}

// Loop condition of the Krylov loop (src/gmres.cpp:199) for step i.
__device__ __forceinline__ void b_gate(BCtl& q, int i) {
    if (q.cycle_active && q.beta > q.tol) {
        const int before = q.its++;
        if (before < q.maxits) {
            q.step_active = 1;
            q.i = i;
            return;
        }
    }
    q.step_active = 0;
    q.cycle_active = 0;
}

// All MGS terms of step i, the scaling of w, the step's rotations and the next
// step's gate in one launch.  A workgroup keeps its chunk of w in registers
// and, per term, publishes its partial products as value-flags, waits for
// those of its system's other chunks and sums them in chunk order, so all of
// them hold the same h.  Basis vectors are read once, one term ahead.
//
// Workgroups take the chunks of `list` in order through tickets; a system's
// chunks have consecutive tickets.  So only the newest system can be partly
// started, and the launch drains as long as its chunks fit beside each other.
// A CU holds two workgroups (176 to 185 registers; 64 KiB of LDS at most), an XCD
// of 32 CUs 64: kBmaChunks fit wherever the hardware puts them, and as it deals
// workgroups to the eight XCDs in turn, several solves doing the same do.
// fused_chunks() asks for the occupancy: where a device is a smaller partition,
// twice the largest system's chunks have to fit.  Larger systems take one
// launch per term.  Partial slots come in two generations by step parity, each
// step re-arming the other one.
//
// One launch per term read v_j, v_j+1 and w and wrote w each time: 35 us per
// term on 40 systems x 8 right-hand sides, 147 of a solve's 379 ms.
constexpr int kBmaChunks = 64;

template <int K>
__global__ __launch_bounds__(kBThreads) void k_bmgs_all(int nchunks, int i, int m, const int* __restrict__ list,
                                                        const int* __restrict__ chunk_beg,
                                                        const int* __restrict__ chunk_sys,
                                                        const int* __restrict__ sys_chunk, const double* v, double* w,
                                                        long nk, const double* __restrict__ part0, double* pbuf,
                                                        double* hh, long hstride, BCtl* ctl, int* ctr, int* err,
                                                        uint64_t wd_limit, int max_nc) {
    extern __shared__ double s_dyn[];
    __shared__ double s_red[(kBThreads / 64) * K];
    __shared__ double s_h[K];
    double* s_p = s_dyn;                       // partials of the system's chunks
    double* s_col = s_dyn + max_nc * K;        // column i, (m + 2) per instance, strided by K
    double* s_c = s_col + (m + 2) * K;         // rotations
    double* s_s = s_c + (m + 1) * K;
    const int c = list[take_ticket(ctr)];
    const int s = chunk_sys[c], c0 = sys_chunk[s], nc = sys_chunk[s + 1] - c0;
    if (!system_live<K>(ctl, s, true)) {
        retire_ticket(ctr);
        return;
    }
    const Watchdog wd(wd_limit);
    bool timed_out = false;
    const int r = threadIdx.x % K;
    const bool lead = c == c0;
    const long gen = static_cast<long>(m + 1) * nchunks * K;
    double* pb = pbuf + (i & 1) * gen;
    double* pnext = pbuf + ((i + 1) & 1) * gen;
    for (int k = threadIdx.x; k < (m + 1) * K; k += kBThreads)
        publish_raw(reinterpret_cast<uint64_t*>(pnext + (static_cast<long>(k / K) * nchunks + c) * K + k % K), kPending);
    double* const hbase = hh + (static_cast<long>(s) * K + r) * hstride;  // r == threadIdx.x for the rotations
    if (lead)
        for (int k = threadIdx.x; k < i * K; k += kBThreads) {
            const double* q = hh + (static_cast<long>(s) * K + k % K) * hstride + static_cast<long>(m + 1) * m;
            s_c[k] = q[k / K];
            s_s[k] = q[m + 1 + k / K];
        }
    const bool on = ctl[s * K + r].step_active != 0;
    const long o0 = static_cast<long>(chunk_beg[c]) * K + threadIdx.x, o1 = static_cast<long>(chunk_beg[c + 1]) * K;
    double wr[kBPer], vn[kBPer], vq[kBPer];
#pragma unroll
    for (int k = 0; k < kBPer; ++k) {
        const long o = o0 + static_cast<long>(k) * kBThreads;
        wr[k] = o < o1 ? w[o] : 0.0;
        vn[k] = o < o1 ? v[o] : 0.0;
        vq[k] = o < o1 && i > 0 ? v[nk + o] : 0.0;
    }
    // h of the K instances from the partials in s_p
    auto total = [&]() {
        __syncthreads();
        if (threadIdx.x < K) {
            double t = 0.0;
            for (int k = 0; k < nc; ++k) t += s_p[k * K + threadIdx.x];
            s_h[threadIdx.x] = t;
        }
        __syncthreads();
        return s_h[r];
    };
    for (int k = threadIdx.x; k < nc * K; k += kBThreads) s_p[k] = part0[static_cast<long>(c0) * K + k];
    double h = total();
    for (int j = 0; j <= i; ++j) {
        if (lead && threadIdx.x < K) s_col[j * K + threadIdx.x] = h;
        const bool more = j < i;
        double acc = 0.0;
#pragma unroll
        for (int k = 0; k < kBPer; ++k) {
            wr[k] = fma(-h, vn[k], wr[k]);
            acc = more ? fma(vq[k], wr[k], acc) : fma(wr[k], wr[k], acc);
        }
        const double t = rhs_reduce<K>(acc, s_red);
        double* slot = pb + (static_cast<long>(j) * nchunks + c0) * K;
        if (threadIdx.x < K) publish(slot + (c - c0) * K + threadIdx.x, t);
        const double* v2 = v + (j + 2) * nk;
#pragma unroll
        for (int k = 0; k < kBPer; ++k) {
            vn[k] = vq[k];
            const long o = o0 + static_cast<long>(k) * kBThreads;
            vq[k] = j + 1 < i && o < o1 ? v2[o] : 0.0;
        }
        for (int k = threadIdx.x; k < nc * K; k += kBThreads) {
            uint64_t bits;
            while ((bits = peek_bits(slot + k)) == kPending) {
                if (timed_out || wd.expired()) {
                    timed_out = true;
                    bits = kQuietNan;
                    break;
                }
                spin_pause();
            }
            s_p[k] = __longlong_as_double(bits);
        }
        h = total();
    }
    const double t = std::sqrt(h);
    const double a = 1.0 / t;
#pragma unroll
    for (int k = 0; k < kBPer; ++k) {
        const long o = o0 + static_cast<long>(k) * kBThreads;
        if (o < o1) w[o] = on && !(t <= 1e-16) ? wr[k] * a : wr[k];
    }
    if (lead && threadIdx.x < K) {
        BCtl& q = ctl[s * K + r];
        if (on) {
            double* rs = hbase + static_cast<long>(m + 1) * m + 2 * (m + 1) + i;
            b_givens(q, i, t, s_col + r, s_c + r, s_s + r, rs, K);
            double* col = hbase + static_cast<long>(i) * (m + 1);
            for (int k = 0; k <= i + 1; ++k) col[k] = s_col[k * K + r];
            double* cs = hbase + static_cast<long>(m + 1) * m;
            if (!q.breakdown) {
                cs[i] = s_c[i * K + r];
                cs[m + 1 + i] = s_s[i * K + r];
            }
        }
        if (i + 1 < m) b_gate(q, i + 1);
    }
    if (timed_out && threadIdx.x == 0) atomicOr(err, kErrTimeout);
    retire_ticket(ctr);
}

__global__ void k_bpending(long words, uint64_t* p) {
    const long stride = static_cast<long>(gridDim.x) * blockDim.x;
    for (long k = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x; k < words; k += stride) p[k] = kPending;
}

// part[c*K+r] = partial sum of b^2 over chunk c, RHS r.
template <int K>
__global__ __launch_bounds__(kBThreads) void k_bnorm(const int* __restrict__ chunk_beg, const double* __restrict__ b,
                                                     double* part) {
    __shared__ double s_red[(kBThreads / 64) * K];
    const int c = blockIdx.x;
    double acc = 0.0;
    for (long o = static_cast<long>(chunk_beg[c]) * K + threadIdx.x; o < static_cast<long>(chunk_beg[c + 1]) * K;
         o += kBThreads)
        acc = fma(b[o], b[o], acc);
    const double t = rhs_reduce<K>(acc, s_red);
    if (threadIdx.x < K) part[static_cast<long>(c) * K + threadIdx.x] = t;
}

// v *= inv per instance (mode 0: cycle start, mode 1: after a step).
template <int K>
__global__ __launch_bounds__(kBThreads) void k_bscale(const int* __restrict__ list, const int* __restrict__ chunk_beg,
                                                      const int* __restrict__ chunk_sys, double* v, const BCtl* ctl,
                                                      int mode) {
    const int c = list ? list[blockIdx.x] : blockIdx.x;
    const int s = chunk_sys[c];
    const int r = threadIdx.x % K;
    const BCtl& q = ctl[s * K + r];
    const bool on = mode == 0 ? q.cycle_active != 0 : (q.step_active != 0 && q.breakdown == 0);
    if (!on) return;
    const double a = q.inv;
    for (long o = static_cast<long>(chunk_beg[c]) * K + threadIdx.x; o < static_cast<long>(chunk_beg[c + 1]) * K;
         o += kBThreads)
        v[o] *= a;
}

// sol += sum_j rs_j z_j per instance.
template <int K>
__global__ __launch_bounds__(kBThreads) void k_bupdate(const int* __restrict__ chunk_beg, const int* __restrict__ chunk_sys,
                                                       const double* __restrict__ z, long nk, const BCtl* ctl,
                                                       const double* hh, long hstride, int m, double* sol) {
    const int c = blockIdx.x;
    const int s = chunk_sys[c];
    const int r = threadIdx.x % K;
    const BCtl& q = ctl[s * K + r];
    if (q.status == 2 || q.i < 0) return;
    const double* rs = hh + (static_cast<long>(s) * K + r) * hstride + static_cast<long>(m + 1) * m + 2 * (m + 1);
    for (long o = static_cast<long>(chunk_beg[c]) * K + threadIdx.x; o < static_cast<long>(chunk_beg[c + 1]) * K;
         o += kBThreads) {
        double x = sol[o];
        for (int j = 0; j <= q.i; ++j) x = fma(rs[j], z[j * nk + o], x);
        sol[o] = x;
    }
}

// ---- one thread per instance ----
__global__ void k_bcycle_begin(int ni, int K, BCtl* ctl, const double* part, const int* sys_chunk, double* hh,
                               long hstride, int m) {
    const int inst = blockIdx.x * blockDim.x + threadIdx.x;
    if (inst >= ni) return;
    BCtl& q = ctl[inst];
    q.i = -1;
    q.breakdown = 0;
    q.step_active = 0;
    q.cycle_active = 0;
    if (q.done) return;
    const double beta = std::sqrt(system_sum(part, sys_chunk, inst / K, inst % K, K));
    q.beta = beta;
    if (beta <= q.tol) {
        q.status = 1;
        q.done = 1;
        return;
    }
    if (std::isnan(beta)) {
        q.status = 2;
        q.done = 1;
        return;
    }
    q.inv = 1.0 / beta;
    hh[static_cast<long>(inst) * hstride + static_cast<long>(m + 1) * m + 2 * (m + 1)] = beta;
    q.cycle_active = 1;
    b_gate(q, 0);
}

// (for the systems whose Gram-Schmidt is not k_bmgs_all's: big[s] != 0)
__global__ void k_bfinish(int ni, int K, const int* __restrict__ big, BCtl* ctl, const double* part, const int* sys_chunk, double* hh, long hstride,
                          int m) {
    const int inst = blockIdx.x * blockDim.x + threadIdx.x;
    if (inst >= ni) return;
    BCtl& q = ctl[inst];
    if (!big[inst / K] || !q.step_active) return;
    const double t = std::sqrt(system_sum(part, sys_chunk, inst / K, inst % K, K));
    const int im1 = m + 1, i = q.i;
    double* base = hh + static_cast<long>(inst) * hstride;
    double* cc = base + static_cast<long>(im1) * m;
    b_givens(q, i, t, base + static_cast<long>(i) * im1, cc, cc + im1, cc + 2 * im1 + i, 1);
}

// The next step's gate (after k_bscale, which still looks at this step's).
__global__ void k_bgate(int ni, int K, const int* __restrict__ big, BCtl* ctl, int i) {
    const int inst = blockIdx.x * blockDim.x + threadIdx.x;
    if (inst < ni && big[inst / K]) b_gate(ctl[inst], i);
}

// Back-solve and end-of-cycle decision (src/gmres.cpp:265-283).
__global__ __launch_bounds__(64) void k_bbacksolve(BCtl* ctl, double* hh, long hstride, int m) {
    __shared__ double s_tri[kBackLds];
    const BCtl& q = ctl[blockIdx.x];
    if (q.done || q.i < 0) return;
    double* base = hh + blockIdx.x * hstride;
    back_substitute(q.i, base, m + 1, base + static_cast<long>(m + 1) * m + 2 * (m + 1), s_tri);
}

__global__ void k_bend_cycle(int ni, BCtl* ctl, int* unfinished) {
    // single block: decide per instance, then count the unfinished ones
    __shared__ int s_cnt;
    if (threadIdx.x == 0) s_cnt = 0;
    __syncthreads();
    int cnt = 0;
    for (int inst = threadIdx.x; inst < ni; inst += blockDim.x) {
        BCtl& q = ctl[inst];
        if (!q.done) {
            if (q.beta <= q.tol) { q.status = 1; q.done = 1; }
            else if (q.its > q.maxits) { q.status = 3; q.done = 1; }
            else if (q.its >= q.maxits) { q.status = 4; q.done = 1; }  // exhausted at a restart boundary
        }
        cnt += q.done ? 0 : 1;
    }
    atomicAdd(&s_cnt, cnt);
    __syncthreads();
    if (threadIdx.x == 0) *unfinished = s_cnt;
}

__global__ void k_binit(int ni, BCtl* ctl, const double* part, const int* sys_chunk, int K, double rel_tol, int maxits) {
    const int inst = blockIdx.x * blockDim.x + threadIdx.x;
    if (inst >= ni) return;
    BCtl q{};
    q.maxits = maxits;
    q.tol = rel_tol * std::sqrt(system_sum(part, sys_chunk, inst / K, inst % K, K));
    ctl[inst] = q;
}

__global__ void k_bresult(int ni, int K, const BCtl* ctl, const double* part, const double* part_b, const int* sys_chunk,
                          int* its, int* conv, double* rel) {
    const int inst = blockIdx.x * blockDim.x + threadIdx.x;
    if (inst >= ni) return;
    const BCtl& q = ctl[inst];
    its[inst] = q.its;
    conv[inst] = (q.status == 1 || q.status == 4) ? 1 : 0;
    const double rb = std::sqrt(system_sum(part_b, sys_chunk, inst / K, inst % K, K));
    const double rr = std::sqrt(system_sum(part, sys_chunk, inst / K, inst % K, K));
    rel[inst] = rb > 0 ? rr / rb : rr;
}

}  // namespace

class BatchedGmres {
public:
    ~BatchedGmres() {
        drop_graph();
        if (stream_) (void)hipStreamDestroy(stream_);
    }

    int setup(const CsrMatrix* d_a, int lof, int nsys, const int* sys_ptr, int nrhs) {
        if (nrhs != 1 && nrhs != 2 && nrhs != 4 && nrhs != 8) throw std::runtime_error("nrhs must be 1, 2, 4 or 8");
        if (nsys <= 0 || sys_ptr[0] != 0 || sys_ptr[nsys] != d_a->size) throw std::runtime_error("bad sys_ptr");
        if (!stream_) PILU_HIP(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
        drop_graph();
        ready_ = set_up_ = false;  // from here on nothing fits the old factors, also if this set-up fails
        K_ = nrhs;
        nsys_ = nsys;
        n_ = d_a->size;
        // chunks
        std::vector<int> beg, sys, sc(nsys + 1), big(nsys), list_f, list_b;
        const int chunk_rows = kChunkElems / nrhs;
        max_nc_ = 0;
        for (int s = 0; s < nsys; ++s) {
            if (sys_ptr[s + 1] <= sys_ptr[s]) throw std::runtime_error("empty system");
            sc[s] = static_cast<int>(beg.size());
            for (int r = sys_ptr[s]; r < sys_ptr[s + 1]; r += chunk_rows) {
                beg.push_back(r);
                sys.push_back(s);
            }
            const int nc = static_cast<int>(beg.size()) - sc[s];
            big[s] = nc > kBmaChunks;
            if (!big[s]) max_nc_ = std::max(max_nc_, nc);
            for (int c = sc[s]; c < sc[s] + nc; ++c) (big[s] ? list_b : list_f).push_back(c);
        }
        sc[nsys] = static_cast<int>(beg.size());
        nchunks_ = static_cast<int>(beg.size());
        nfused_ = static_cast<int>(list_f.size());
        fused_m_ = -1;
        list_f.insert(list_f.end(), list_b.begin(), list_b.end());
        chunk_list_.resize(list_f.size());
        sys_big_.resize(big.size());
        PILU_HIP(hipMemcpy(chunk_list_.get(), list_f.data(), list_f.size() * sizeof(int), hipMemcpyHostToDevice));
        sys_all_.resize(big.size());
        PILU_HIP(hipMemcpy(sys_all_.get(), std::vector<int>(big.size(), 1).data(), big.size() * sizeof(int), hipMemcpyHostToDevice));
        PILU_HIP(hipMemcpy(sys_big_.get(), big.data(), big.size() * sizeof(int), hipMemcpyHostToDevice));
        beg.push_back(n_);
        chunk_beg_.resize(beg.size());
        chunk_sys_.resize(sys.size());
        sys_chunk_.resize(sc.size());
        PILU_HIP(hipMemcpy(chunk_beg_.get(), beg.data(), beg.size() * sizeof(int), hipMemcpyHostToDevice));
        PILU_HIP(hipMemcpy(chunk_sys_.get(), sys.data(), sys.size() * sizeof(int), hipMemcpyHostToDevice));
        PILU_HIP(hipMemcpy(sys_chunk_.get(), sc.data(), sc.size() * sizeof(int), hipMemcpyHostToDevice));
        // system of every row (the sweeps' schedule is per system)
        std::vector<int> rs(static_cast<size_t>(n_));
        for (int q = 0; q < nsys; ++q) std::fill(rs.begin() + sys_ptr[q], rs.begin() + sys_ptr[q + 1], q);
        row_sys_.resize(rs.size());
        PILU_HIP(hipMemcpy(row_sys_.get(), rs.data(), rs.size() * sizeof(int), hipMemcpyHostToDevice));
        // pattern: symbolic ILU(lof) of the block-diagonal matrix
        const int nnz_f = ilu_.SymbolicDevice(n_, d_a->row_ptr, d_a->col_idx, lof);
        if (nnz_f < 0) return nnz_f;
        // per-system level schedules of the sweeps
        Ext* ie = ilu_.DeviceState();
        block_level_schedule(ie, false, row_sys_.get(), nsys, sperm_l_, sgrp_l_, soff_l_);
        block_level_schedule(ie, true, row_sys_.get(), nsys, sperm_u_, sgrp_u_, soff_u_);
        build_rounds(ie);
        PILU_HIP(hipDeviceSynchronize());
        set_up_ = true;
        return nnz_f;
    }

    bool factorize(const double* d_avals) {
        if (!set_up_) throw std::runtime_error("batched: set up first");
        PILU_HIP(hipDeviceSynchronize());
        const bool ok = ilu_.FactorizeDeviceFromA(d_avals);
        if (br_kp_ > 0) gather_rounds(ilu_.DeviceState());
        PILU_HIP(hipDeviceSynchronize());
        ready_ = true;
        return ok;
    }

    void set_precision(int bits) { ilu_.SetFactorPrecision(bits); drop_graph(); }

    int solve(const CsrMatrix* d_a, const double* d_rhs, double* d_sol, double rel_tol, int m, int maxits, int* its,
              int* conv, double* rel) {
        // another precision than the factors' asks for a new factorization
        if (!ready_ || !ilu_.DeviceState()->factored) throw std::runtime_error("batched: factorize first");
        if (d_a->size != n_) throw std::runtime_error("batched: matrix size changed");
        PILU_HIP(hipDeviceSynchronize());  // caller's null-stream work is complete
        const int ni = nsys_ * K_;
        const long nk = static_cast<long>(n_) * K_;
        const long hstride = static_cast<long>(m + 1) * (m + 3);
        bool realloc = m != m_ || maxits != maxits_;
        v_.reserve(static_cast<size_t>(m + 1) * nk);
        z_.reserve(static_cast<size_t>(m) * nk);
        hh_.reserve(static_cast<size_t>(ni) * hstride);
        part_.reserve(3 * static_cast<size_t>(nchunks_) * K_);
        ctl_.reserve(ni);
        y_.reserve(nk);
        flags_.reserve(4);
        if (fused_chunks(m) > 0) {
            pbuf_.reserve(2 * static_cast<size_t>(m + 1) * nchunks_ * K_);
            if (tick_.size() < 2) {
                tick_.reserve(2);
                PILU_HIP(hipMemset(tick_.get(), 0, 2 * sizeof(int)));
            }
        }
        res_.reserve(nk);
        int_out_.reserve(2 * static_cast<size_t>(ni));
        dbl_out_.reserve(ni);
        if (v_.get() != gv_ || z_.get() != gz_ || pbuf_.get() != gpb_ || part_.get() != gpart_ || d_rhs != grhs_ || d_sol != gsol_ || d_a->value != gval_ ||
            d_a->row_ptr != grp_ || d_a->col_idx != gci_ || realloc)
            drop_graph();
        m_ = m;
        maxits_ = maxits;
        Ext* ie = ilu_.DeviceState();
        // tolerances: tol = rel_tol * ||b_inst||
        double* pb = part_.get() + 2L * nchunks_ * K_;
        norm_launch(d_rhs, pb);
        k_binit<<<ceil_div(ni, 256), 256, 0, stream_>>>(ni, ctl_.get(), pb, sys_chunk_.get(), K_, rel_tol, maxits);
        PILU_HIP(hipGetLastError());
        if (!graph_exec_) {
            PILU_HIP(hipStreamBeginCapture(stream_, hipStreamCaptureModeThreadLocal));
            enqueue_cycle(d_a, d_rhs, d_sol, ie, m, hstride, nk);
            hipGraph_t g;
            PILU_HIP(hipStreamEndCapture(stream_, &g));
            PILU_HIP(hipGraphInstantiate(&graph_exec_, g, nullptr, nullptr, 0));
            PILU_HIP(hipGraphDestroy(g));
            gpb_ = pbuf_.get(); gpart_ = part_.get();
            gv_ = v_.get(); gz_ = z_.get(); grhs_ = d_rhs; gsol_ = d_sol; gval_ = d_a->value;
            grp_ = d_a->row_ptr; gci_ = d_a->col_idx;
        }
        int unfinished = ni;
        cycles_ = 0;
        while (unfinished > 0) {
            PILU_HIP(hipGraphLaunch(graph_exec_, stream_));
            PILU_HIP(hipMemcpyAsync(&unfinished, flags_.get(), sizeof(int), hipMemcpyDeviceToHost, stream_));
            PILU_HIP(hipStreamSynchronize(stream_));
            ++cycles_;
            if (cycles_ > maxits + 2) throw std::runtime_error("batched GMRES: no progress");
        }
        int err = 0;
        PILU_HIP(hipMemcpy(&err, ie->err.get() + 1, sizeof(int), hipMemcpyDeviceToHost));
        if (err & kErrTimeout) throw std::runtime_error("batched solve: dependency wait timed out (watchdog)");
        // results: true residual per instance
        double* pr = part_.get();
        spmv_launch(d_a, -1.0, d_sol, 1.0, d_rhs, res_.get(), nullptr, true, pr);
        k_bresult<<<ceil_div(ni, 256), 256, 0, stream_>>>(ni, K_, ctl_.get(), pr, pb, sys_chunk_.get(), int_out_.get(),
                                                          int_out_.get() + ni, dbl_out_.get());
        PILU_HIP(hipMemcpyAsync(its, int_out_.get(), sizeof(int) * ni, hipMemcpyDeviceToHost, stream_));
        PILU_HIP(hipMemcpyAsync(conv, int_out_.get() + ni, sizeof(int) * ni, hipMemcpyDeviceToHost, stream_));
        PILU_HIP(hipMemcpyAsync(rel, dbl_out_.get(), sizeof(double) * ni, hipMemcpyDeviceToHost, stream_));
        PILU_HIP(hipStreamSynchronize(stream_));
        return cycles_;
    }

    lljbash::IluSolver& ilu() { return ilu_; }
    int cycles() const { return cycles_; }

private:
    using Ext = lljbash::IluSolver::Ext;

    void drop_graph() {
        if (graph_exec_) (void)hipGraphExecDestroy(graph_exec_);
        graph_exec_ = nullptr;
    }

    // gate: 0 every chunk, 1 chunks of unfinished systems, 2 chunks of systems running the current step
    void spmv_launch(const CsrMatrix* a, double alpha, const double* x, double beta, const double* yin, double* y,
                     const double* dotv, bool nrm, double* part, int gate = 0) {
        const BCtl* ctl = gate ? ctl_.get() : nullptr;
        switch (K_) {
#define PILU_CASE(KK)                                                                                                 \
    case KK:                                                                                                          \
        k_bspmv<KK><<<nchunks_, kBThreads, 0, stream_>>>(chunk_beg_.get(), a->row_ptr, a->col_idx, a->value, alpha, \
                                                          x, beta, yin, y, dotv, nrm, part, chunk_sys_.get(), ctl,    \
                                                          gate == 2);                                                 \
        break;
            PILU_CASE(1) PILU_CASE(2) PILU_CASE(4) PILU_CASE(8)
#undef PILU_CASE
        }
    }

    // partials of ||b||^2 per chunk and RHS
    void norm_launch(const double* b, double* part) {
        switch (K_) {
#define PILU_CASE(KK)                                                                                       \
    case KK:                                                                                                \
        k_bnorm<KK><<<nchunks_, kBThreads, 0, stream_>>>(chunk_beg_.get(), b, part);                        \
        break;
            PILU_CASE(1) PILU_CASE(2) PILU_CASE(4) PILU_CASE(8)
#undef PILU_CASE
        }
    }

    template <int K, typename T>
    void sweeps_t(Ext* e, const T* val, const double* b, double* x) {
        k_ssweep<K, T, false><<<nsys_, kSThreads, 0, stream_>>>(sgrp_l_.get(), soff_l_.get(), sperm_l_.get(),
                                                                e->rp.get(), e->ci.get(), e->dg.get(), val, b,
                                                                y_.get(), ctl_.get());
        k_ssweep<K, T, true><<<nsys_, kSThreads, 0, stream_>>>(sgrp_u_.get(), soff_u_.get(), sperm_u_.get(),
                                                               e->rp.get(), e->ci.get(), e->dg.get(), val, y_.get(),
                                                               x, ctl_.get());
    }

    // ---- sweeps over rounds (k_bsweep) ----

    // Stream of one direction.
    struct Rounds {
        DevBuf<int> rptr, rid, col, src;
        DevBuf<double> val64, diag;
        DevBuf<float> val32;
        int ring = 0;
        long total = 0;  // rounds x rows per round
    };

    // Decides whether the sweeps run over rounds and builds their streams:
    // short rows, and dependencies that stay in the LDS ring.  br_kp_ = 0
    // leaves the sweeps to k_ssweep.  A workgroup takes as many of a system's
    // right-hand sides as still give every CU one (k_bsweep's latency per
    // level does not depend on it, and coalescing favours many).
    void build_rounds(Ext* e) {
        br_kp_ = 0;
        const int widest = std::max(e->max_lo, e->max_up);
        if (widest > 4) return;
        br_s_ = widest <= 2 ? 2 : 4;
        int dev = 0, cus = 0;
        PILU_HIP(hipGetDevice(&dev));
        PILU_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        hipStream_t s = nullptr;
        std::vector<int> grp[2], off[2];
        DevBuf<int> kinv(2 * static_cast<size_t>(n_)), reach(2);
        PILU_HIP(hipMemsetAsync(reach.get(), 0, 2 * sizeof(int), s));
        int widest_level = 1;
        for (int d = 0; d < 2; ++d) {
            const DevBuf<int>& dg = d ? sgrp_u_ : sgrp_l_;
            const DevBuf<int>& df = d ? soff_u_ : soff_l_;
            const int* perm = (d ? sperm_u_ : sperm_l_).get();
            grp[d].resize(static_cast<size_t>(nsys_) + 1);
            PILU_HIP(hipMemcpy(grp[d].data(), dg.get(), grp[d].size() * sizeof(int), hipMemcpyDeviceToHost));
            const int ng = grp[d][nsys_];
            off[d].resize(static_cast<size_t>(ng) + 1);
            PILU_HIP(hipMemcpy(off[d].data(), df.get(), off[d].size() * sizeof(int), hipMemcpyDeviceToHost));
            for (int g = 0; g < ng; ++g) widest_level = std::max(widest_level, off[d][g + 1] - off[d][g]);
            int* ki = kinv.get() + static_cast<long>(d) * n_;
            k_br_inv<<<ceil_div(n_, 256), 256, 0, s>>>(n_, perm, ki);
            auto kern = d ? k_br_reach<true> : k_br_reach<false>;
            if (ng > 0)
                kern<<<ceil_div(ng, 256), 256, 0, s>>>(ng, df.get(), perm, ki, e->rp.get(), e->dg.get(), e->ci.get(),
                                                       reach.get() + d);
            PILU_HIP(hipGetLastError());
        }
        int far[2] = {0, 0};
        PILU_HIP(hipMemcpy(far, reach.get(), sizeof(far), hipMemcpyDeviceToHost));
        int kp = K_;
        while (kp > 1 && static_cast<long>(nsys_) * (K_ / kp) < cus) kp /= 2;
        for (Rounds* r : {&br_l_, &br_u_}) {
            r->ring = 64;
            while (r->ring < far[r == &br_u_] && r->ring < (1 << 20)) r->ring *= 2;
            while (kp > 1 && ring_bytes(*r, kp) > kBrMaxLds) kp /= 2;
            if (ring_bytes(*r, kp) > kBrMaxLds) return;
        }
        br_rows_ = std::max(64 / kp, 1);
        while (br_rows_ < widest_level && br_rows_ * kp < 1024 && br_rows_ < 256) br_rows_ *= 2;
        for (int d = 0; d < 2; ++d) {
            Rounds& r = d ? br_u_ : br_l_;
            std::vector<int> rptr(static_cast<size_t>(nsys_) + 1, 0);
            std::vector<int4> rounds;
            for (int q = 0; q < nsys_; ++q) {
                rptr[q] = static_cast<int>(rounds.size());
                const int k0 = grp[d][q] < grp[d][q + 1] ? off[d][grp[d][q]] : 0;
                for (int g = grp[d][q]; g < grp[d][q + 1]; ++g)
                    for (int k = off[d][g]; k < off[d][g + 1]; k += br_rows_)
                        rounds.push_back(make_int4(k, std::min(br_rows_, off[d][g + 1] - k),
                                                   k + br_rows_ >= off[d][g + 1] ? 1 : 0, k0));
            }
            rptr[nsys_] = static_cast<int>(rounds.size());
            r.total = static_cast<long>(rounds.size()) * br_rows_;
            if (r.total == 0 || r.total * br_s_ >= (1L << 31)) return;
            r.rptr.resize(rptr.size());
            PILU_HIP(hipMemcpy(r.rptr.get(), rptr.data(), rptr.size() * sizeof(int), hipMemcpyHostToDevice));
            DevBuf<int4> dr(rounds.size());
            PILU_HIP(hipMemcpy(dr.get(), rounds.data(), rounds.size() * sizeof(int4), hipMemcpyHostToDevice));
            r.rid.reserve(2 * r.total);
            r.col.reserve(r.total * br_s_);
            r.src.reserve(r.total * br_s_);
            auto fill = d ? k_br_fill<true> : k_br_fill<false>;
            fill<<<ceil_div(r.total, 256), 256, 0, s>>>(r.total, br_rows_, br_s_, r.ring, dr.get(),
                                                        (d ? sperm_u_ : sperm_l_).get(),
                                                        kinv.get() + static_cast<long>(d) * n_, e->rp.get(), e->dg.get(),
                                                        e->ci.get(), reinterpret_cast<int2*>(r.rid.get()), r.col.get(),
                                                        r.src.get());
            PILU_HIP(hipGetLastError());
            PILU_HIP(hipStreamSynchronize(s));  // dr goes out of scope
        }
        br_kp_ = kp;
    }

    static size_t ring_bytes(const Rounds& r, int kp) { return sizeof(double) * (static_cast<size_t>(r.ring) + 1) * kp; }

    // Values of the rounds from the factors (on the factorization's stream).
    void gather_rounds(Ext* e) {
        for (Rounds* r : {&br_l_, &br_u_}) {
            double2* diag = nullptr;
            if (r == &br_u_) {
                r->diag.reserve(2 * r->total);
                diag = reinterpret_cast<double2*>(r->diag.get());
            }
            const int2* rid = reinterpret_cast<const int2*>(r->rid.get());
            const int grid = ceil_div(r->total, 256);
            if (e->precision == 32) {
                r->val32.reserve(r->total * br_s_);
                k_br_gather<float><<<grid, 256, 0, e->stream>>>(r->total, br_s_, r->src.get(), e->fac32.get(),
                                                                r->val32.get(), rid, e->dg.get(), diag);
            } else {
                r->val64.reserve(r->total * br_s_);
                k_br_gather<double><<<grid, 256, 0, e->stream>>>(r->total, br_s_, r->src.get(), e->fac.get(),
                                                                 r->val64.get(), rid, e->dg.get(), diag);
            }
            PILU_HIP(hipGetLastError());
        }
    }

    template <int KP, int S, typename T, bool UPPER>
    void rounds_one(const T* val, const double* b, double* x) {
        const Rounds& r = UPPER ? br_u_ : br_l_;
        const int per = K_ / KP;
        // eight systems (one per XCD) x their groups of right-hand sides at a time
        const int grid = ceil_div(nsys_, 8) * per * 8;
        k_bsweep<KP, S, T, UPPER><<<grid, br_rows_ * KP, ring_bytes(r, KP), stream_>>>(
            r.rptr.get(), reinterpret_cast<const int2*>(r.rid.get()), r.col.get(), val,
            reinterpret_cast<const double2*>(r.diag.get()), b, x, nsys_, K_, r.ring, ctl_.get());
    }

    template <int KP, int S>
    void rounds_pair(Ext* e, const double* b, double* x) {
        if (e->precision == 32) {
            rounds_one<KP, S, float, false>(br_l_.val32.get(), b, y_.get());
            rounds_one<KP, S, float, true>(br_u_.val32.get(), y_.get(), x);
        } else {
            rounds_one<KP, S, double, false>(br_l_.val64.get(), b, y_.get());
            rounds_one<KP, S, double, true>(br_u_.val64.get(), y_.get(), x);
        }
    }

    template <int KP>
    void rounds_kp(Ext* e, const double* b, double* x) {
        if (br_s_ == 2) rounds_pair<KP, 2>(e, b, x);
        else rounds_pair<KP, 4>(e, b, x);
    }

    template <int K>
    void sweeps_k(Ext* e, const double* b, double* x) {
        if (e->precision == 32) sweeps_t<K, float>(e, e->fac32.get(), b, x);
        else sweeps_t<K, double>(e, e->fac.get(), b, x);
    }

    void sweeps(Ext* e, const double* b, double* x) {
        switch (br_kp_) {
            case 1: rounds_kp<1>(e, b, x); return;
            case 2: rounds_kp<2>(e, b, x); return;
            case 4: rounds_kp<4>(e, b, x); return;
            case 8: rounds_kp<8>(e, b, x); return;
            default: break;
        }
        switch (K_) {
            case 1: sweeps_k<1>(e, b, x); break;
            case 2: sweeps_k<2>(e, b, x); break;
            case 4: sweeps_k<4>(e, b, x); break;
            default: sweeps_k<8>(e, b, x); break;
        }
    }

    void mgs_launch(const int* list, int n, const double* vj, double* w, const double* vnext, const double* pin, double* pout, long hstride,
                    int hpos) {
        switch (K_) {
#define PILU_CASE(KK)                                                                                                \
    case KK:                                                                                                         \
        k_bmgs<KK><<<n, kBThreads, 0, stream_>>>(list, chunk_beg_.get(), chunk_sys_.get(), sys_chunk_.get(), vj, w, \
                                                         vnext, pin, pout, hh_.get(), hstride, hpos, ctl_.get());    \
        break;
            PILU_CASE(1) PILU_CASE(2) PILU_CASE(4) PILU_CASE(8)
#undef PILU_CASE
        }
    }

    size_t mgs_lds(int m) const { return sizeof(double) * K_ * (static_cast<size_t>(max_nc_) + 3 * (m + 2)); }

    // Chunks of k_bmgs_all (the first of chunk_list_): none where the rotations
    // of a long restart exceed the LDS, or where the device has no room for the
    // largest system's chunks twice (for another solve doing the same).
    int fused_chunks(int m) {
        if (fused_m_ == m) return fused_;
        fused_m_ = m;
        fused_ = 0;
        if (nfused_ == 0 || mgs_lds(m) > 64 * 1024) return 0;
        const void* kern = K_ == 1   ? reinterpret_cast<const void*>(k_bmgs_all<1>)
                           : K_ == 2 ? reinterpret_cast<const void*>(k_bmgs_all<2>)
                           : K_ == 4 ? reinterpret_cast<const void*>(k_bmgs_all<4>)
                                     : reinterpret_cast<const void*>(k_bmgs_all<8>);
        int dev = 0, cus = 0, per_cu = 0;
        PILU_HIP(hipGetDevice(&dev));
        PILU_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        PILU_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, kBThreads, mgs_lds(m)));
        if (2L * max_nc_ <= static_cast<long>(cus) * per_cu) fused_ = nfused_;
        return fused_;
    }

    void mgs_all_launch(int i, int m, const double* v, double* w, long nk, const double* part0, long hstride, Ext* ie) {
        const uint64_t wd = watchdog_ticks(ie->watchdog_s);
        switch (K_) {
#define PILU_CASE(KK)                                                                                                 \
    case KK:                                                                                                          \
        k_bmgs_all<KK><<<nfused_, kBThreads, mgs_lds(m), stream_>>>(                                                  \
            nchunks_, i, m, chunk_list_.get(), chunk_beg_.get(), chunk_sys_.get(), sys_chunk_.get(), v, w, nk, part0, pbuf_.get(),       \
            hh_.get(), hstride, ctl_.get(), tick_.get(), ie->err.get() + 1, wd, max_nc_);                             \
        break;
            PILU_CASE(1) PILU_CASE(2) PILU_CASE(4) PILU_CASE(8)
#undef PILU_CASE
        }
    }

    void scale_launch(const int* list, int n, double* v, int mode) {
        switch (K_) {
#define PILU_CASE(KK)                                                                                          \
    case KK:                                                                                                   \
        k_bscale<KK><<<n, kBThreads, 0, stream_>>>(list, chunk_beg_.get(), chunk_sys_.get(), v, ctl_.get(), mode); \
        break;
            PILU_CASE(1) PILU_CASE(2) PILU_CASE(4) PILU_CASE(8)
#undef PILU_CASE
        }
    }

    void update_launch(double* sol, long nk, long hstride) {
        switch (K_) {
#define PILU_CASE(KK)                                                                                              \
    case KK:                                                                                                       \
        k_bupdate<KK><<<nchunks_, kBThreads, 0, stream_>>>(chunk_beg_.get(), chunk_sys_.get(), z_.get(), nk,       \
                                                            ctl_.get(), hh_.get(), hstride, m_, sol);               \
        break;
            PILU_CASE(1) PILU_CASE(2) PILU_CASE(4) PILU_CASE(8)
#undef PILU_CASE
        }
    }

    void enqueue_cycle(const CsrMatrix* a, const double* rhs, double* sol, Ext* ie, int m, long hstride, long nk) {
        const int ni = nsys_ * K_;
        const int ib = ceil_div(ni, 256);
        double* p0 = part_.get();
        double* p1 = p0 + static_cast<long>(nchunks_) * K_;
        double* v = v_.get();
        double* z = z_.get();
        spmv_launch(a, -1.0, sol, 1.0, rhs, v, nullptr, true, p0, 1);
        k_bcycle_begin<<<ib, 256, 0, stream_>>>(ni, K_, ctl_.get(), p0, sys_chunk_.get(), hh_.get(), hstride, m);
        scale_launch(nullptr, nchunks_, v, 0);
        // k_bcycle_begin has set the first step's gate; each step sets the next one's
        const int nf = fused_chunks(m), nb = nchunks_ - nf;
        const int* list = chunk_list_.get() + nf;
        const int* big = nf > 0 ? sys_big_.get() : sys_all_.get();
        const long slots = static_cast<long>(nchunks_) * K_;  // the first term's, of step 0's generation
        if (nf > 0)
            k_bpending<<<std::min(ceil_div(slots, 256), 1024), 256, 0, stream_>>>(
                slots, reinterpret_cast<uint64_t*>(pbuf_.get()));
        for (int i = 0; i < m; ++i) {
            double* vi = v + i * nk;
            double* vi1 = v + (i + 1) * nk;
            double* zi = z + i * nk;
            sweeps(ie, vi, zi);
            spmv_launch(a, 1.0, zi, 0.0, nullptr, vi1, v, false, p0, 2);
            if (nf > 0) mgs_all_launch(i, m, v, vi1, nk, p0, hstride, ie);
            if (nb == 0) continue;
            double* pin = p0;
            double* pout = p1;
            for (int j = 0; j <= i; ++j) {
                mgs_launch(list, nb, v + j * nk, vi1, j < i ? v + (j + 1) * nk : nullptr, pin, pout, hstride,
                           i * (m + 1) + j);
                std::swap(pin, pout);
            }
            k_bfinish<<<ib, 256, 0, stream_>>>(ni, K_, big, ctl_.get(), pin, sys_chunk_.get(), hh_.get(), hstride, m);
            scale_launch(list, nb, vi1, 1);
            if (i + 1 < m) k_bgate<<<ib, 256, 0, stream_>>>(ni, K_, big, ctl_.get(), i + 1);
        }
        k_bbacksolve<<<ni, 64, 0, stream_>>>(ctl_.get(), hh_.get(), hstride, m);
        update_launch(sol, nk, hstride);
        k_bend_cycle<<<1, 1024, 0, stream_>>>(ni, ctl_.get(), flags_.get());
    }

    lljbash::IluSolver ilu_;
    hipStream_t stream_ = nullptr;
    hipGraphExec_t graph_exec_ = nullptr;
    const void *gv_ = nullptr, *gz_ = nullptr, *grhs_ = nullptr, *gsol_ = nullptr, *gval_ = nullptr,
               *grp_ = nullptr, *gci_ = nullptr, *gpb_ = nullptr, *gpart_ = nullptr;
    int br_kp_ = 0, br_s_ = 2, br_rows_ = 64;  // right-hand sides per workgroup (0: k_ssweep), entries and rows per round
    Rounds br_l_, br_u_;
    // Gram-Schmidt: chunks of the systems k_bmgs_all takes come first in
    // chunk_list_; most chunks of one of them
    int nfused_ = 0, max_nc_ = 0;
    int fused_m_ = -1, fused_ = 0;  // fused_chunks(fused_m_)
    DevBuf<int> chunk_list_, sys_big_, sys_all_;
    DevBuf<double> pbuf_;
    DevBuf<int> tick_;
    int K_ = 8, nsys_ = 0, n_ = 0, nchunks_ = 0, m_ = -1, maxits_ = -1, cycles_ = 0;
    bool set_up_ = false, ready_ = false;
    DevBuf<int> chunk_beg_, chunk_sys_, sys_chunk_, row_sys_, flags_, int_out_;
    DevBuf<int> sperm_l_, sgrp_l_, soff_l_, sperm_u_, sgrp_u_, soff_u_;  // per-system level schedules
    DevBuf<double> v_, z_, hh_, part_, y_, res_, dbl_out_;
    DevBuf<BCtl> ctl_;
};

}  // namespace pilu

// ---- C ABI (include/par_ilu_ex.h) ----
namespace {
template <typename F>
int bguard(const char* what, F&& f) {
    try {
        return f();
    } catch (const std::exception& e) {
        std::fprintf(stderr, "%s: %s\n", what, e.what());
        return std::string(e.what()) == "missing diag" ? -2 : -1;
    }
}
pilu::BatchedGmres* B(BatchGmresHdl h) { return static_cast<pilu::BatchedGmres*>(h); }
}  // namespace

extern "C" {

BatchGmresHdl BatchGmresCreateEx(void) { return new pilu::BatchedGmres; }

void BatchGmresDestroyEx(BatchGmresHdl h) { delete B(h); }

int BatchGmresSetupEx(BatchGmresHdl h, const CsrMatrix* d_a, int lof, int nsys, const int* sys_ptr, int nrhs) {
    return bguard("BatchGmresSetup", [&] { return B(h)->setup(d_a, lof, nsys, sys_ptr, nrhs); });
}

int BatchGmresSetFactorPrecisionEx(BatchGmresHdl h, int bits) {
    return bguard("BatchGmresSetFactorPrecision", [&] { B(h)->set_precision(bits); return 0; });
}

int BatchGmresFactorizeEx(BatchGmresHdl h, const double* d_avalues) {
    return bguard("BatchGmresFactorize", [&] { return B(h)->factorize(d_avalues) ? 0 : -1; });
}

int BatchGmresSolveEx(BatchGmresHdl h, const CsrMatrix* d_a, const double* d_rhs, double* d_sol, double rel_tol,
                      int m, int maxits, int* its, int* converged, double* true_rel_res) {
    return bguard("BatchGmresSolve",
                  [&] { return B(h)->solve(d_a, d_rhs, d_sol, rel_tol, m, maxits, its, converged, true_rel_res); });
}

}  // extern "C"
