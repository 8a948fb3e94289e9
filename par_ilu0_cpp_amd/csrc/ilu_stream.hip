// Block-local triangular sweep over a chunk stream (modes 2 and 3 where a
// row's entries fit its lanes).
//
// A block (tile or contiguous rows) is solved by one workgroup.  Its rows,
// in (local level, row) order, are cut into chunks of at most 64 / G rows of
// one level, dealt in turn to kStSolvers solver waves; a lane holds at most
// one entry of its row.  Per chunk the stream holds, lane by lane, the LDS
// slots of the entry's x and of the row's own x, where the row's result goes,
// and the value; for U also {u_ii, 1 / u_ii} per row.  The chunks of a block
// are consecutive, so a request is a scalar offset plus the lane's constant
// one.
//
// Synchronisation is by value only.  LDS holds the block's x and one slot
// per distinct out-of-block column ("import"), all kPending on entry.  A
// solver wave re-reads the LDS words of its chunk until none is pending:
// chunks are in level order, so the lowest unsolved level can always
// proceed.  A block's imports have consecutive mailbox words in global
// memory, in order of first use.  The wave that solves a row stores its x
// into the mailbox word of every block that imports it (one per lane of the
// row after the first), and an importer wave polls its block's words, 64
// neighbouring ones per request, and copies them to LDS.  So the solver
// waves' in-order memory counter never waits on a poll and no barrier
// follows the start.  Mailboxes come in two generations: a launch uses the
// one *gen names, arms the other with kPending for the next launch, and its
// last workgroup switches *gen.  `out` itself carries no flags.
//
// Row sums are k_sweep's for the same G: lane t takes entry t from 0 (b for
// lane 0) with one fma, then group_sum.  Unused lanes read a zero slot with
// value 0, which adds -0 and changes no bit.
//
// What bounds it is the dependency chain: at 128^3 ILU(1) 763 levels per
// sweep and about 83 tile crossings.  k_sweep_pp spent some 150 instructions
// per pass and wave and polled the out-of-block x in the solving waves: 1172
// us (FP64 factors) and 1202 us (FP32) per L+U apply on 128 x 4 x 8 tiles.
// Measured here on the way: 961 us with importer waves polling `out`, 733
// with mailboxes (a hand-off fell from 1.8 to 0.96 us at the median), 688
// with buffer requests and a written-out LDS poll (about 45 instructions per
// chunk), 630 with 8 solver waves instead of 4, so that the waves of one
// level issue their requests while the next level is solved, 609 (FP64) and
// 571 (FP32) without padding chunks; 12 solver waves 636, a second importer
// or more polls in flight 625 to 780, 8 / 4 chunks ahead 642.  One
// workgroup per CU is faster than two or three (609 against 773 us): the
// solver waves of blocks still waiting take issue slots from the others.
#include <rocprim/device/device_scan.hpp>

#include <algorithm>
#include <stdexcept>
#include <vector>

#include "ilu_internal.hpp"
#include "ilu_stream.hpp"
#include "ilu_stream_plan.hpp"

namespace pilu {

namespace {

using Ext = lljbash::IluSolver::Ext;

constexpr int kStThreads = 64 * (kStSolvers + 1);  // solver waves and one importer wave
constexpr size_t kStMinLds = 81 * 1024;  // one workgroup per CU

__device__ __forceinline__ void lds_put(double* xs, unsigned at, double v) {
    __hip_atomic_store(reinterpret_cast<uint64_t*>(reinterpret_cast<char*>(xs) + at),
                       static_cast<uint64_t>(__double_as_longlong(v)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// The lane's LDS word (byte address `at`) once no lane's is pending (a pending
// lane's NaN past the watchdog).  The poll is written out: a read, its wait
// and one branch, with a bound of kStSpins reads; compiled code added as much
// again on the way out of the loop, which every level pays.
constexpr int kStSpins = 512;
__device__ __forceinline__ uint64_t wait_lds(unsigned at, const Watchdog& wd, bool& timed_out) {
    uint64_t bits;
    int left;
    auto poll = [&]() {
        asm volatile(
            "s_movk_i32 %1, %4\n"
            "1:\n"
            "ds_read_b64 %0, %2\n"
            "s_waitcnt lgkmcnt(0)\n"
            "v_cmp_eq_u64 vcc, %3, %0\n"
            "s_cbranch_vccz 2f\n"
            "s_sub_i32 %1, %1, 1\n"
            "s_cmp_lg_u32 %1, 0\n"
            "s_cbranch_scc1 1b\n"
            "2:\n"
            : "=&v"(bits), "=&s"(left)
            : "v"(at), "s"(kPending), "n"(kStSpins)
            : "vcc", "scc", "memory");
    };
    poll();
    if (__builtin_expect(left == 0, 0)) {
        do {
            timed_out = timed_out || wd.expired();
            if (timed_out) {
                if (bits == kPending) bits = kQuietNan;
                break;
            }
            poll();
        } while (left == 0);
    }
    return bits;
}

// One lane of a chunk: where its x and its row's x sit in LDS (slots in bits
// 0..14 and 15..29), and a byte offset: lane 0 of a row: the row in b and
// out; the other lanes: a mailbox word the row's result goes to.
struct StA {
    uint2 p;
};
constexpr unsigned kStNone = 0xfffffff8u;  // past every buffer: loads give 0, stores are dropped

template <typename T>
struct StB {
    T v;
    double b;    // b of the row in its lane 0, 0 in the others
    double2 d;
};

// Raw buffer access: scalar base, one 32-bit byte offset per lane and a
// scalar offset, so a chunk's requests need no address arithmetic.  A lane
// offset past `bytes` (kStNone) reads 0 and stores nothing; scalar offsets stay
// inside the buffer (kStOverrun).
using Rsrc = __amdgpu_buffer_rsrc_t;
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ Rsrc st_rsrc(const void* p, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, static_cast<int>(bytes), 0x00027000);
}
__device__ __forceinline__ uint2 st_load2(Rsrc r, unsigned lane_off, unsigned off) {
    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, lane_off, off, 0);
    return make_uint2(v.x, v.y);
}
__device__ __forceinline__ double st_load_d(Rsrc r, unsigned lane_off, unsigned off) {
    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, lane_off, off, 0);
    return __hiloint2double(static_cast<int>(v.y), static_cast<int>(v.x));
}
__device__ __forceinline__ float st_load_f(Rsrc r, unsigned lane_off, unsigned off) {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, lane_off, off, 0));
}
__device__ __forceinline__ double2 st_load_d2(Rsrc r, unsigned lane_off, unsigned off) {
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, lane_off, off, 0);
    return make_double2(__hiloint2double(static_cast<int>(v.y), static_cast<int>(v.x)),
                        __hiloint2double(static_cast<int>(v.w), static_cast<int>(v.z)));
}
constexpr int kStPlain = 0, kStAgent = 16;  // cache policy: 16 = sc1, agent-coherent
template <int POLICY>
__device__ __forceinline__ void st_store(Rsrc r, unsigned lane_off, double v) {
    const u32x2 w = {static_cast<unsigned>(__double2loint(v)), static_cast<unsigned>(__double2hiint(v))};
    __builtin_amdgcn_raw_buffer_store_b64(w, r, lane_off, 0, POLICY);
}

// v of the first lane of every G adjacent lanes (2 <= G <= 16).
template <int G>
__device__ __forceinline__ double group_first(double v) {
    int lo = __double2loint(v), hi = __double2hiint(v);
    constexpr int quad = G == 2 ? 0xa0 : 0x00;  // quad_perm [0,0,2,2] or [0,0,0,0]
    lo = __builtin_amdgcn_update_dpp(lo, lo, quad, 0xf, 0xf, false);
    hi = __builtin_amdgcn_update_dpp(hi, hi, quad, 0xf, 0xf, false);
    if constexpr (G >= 8) {  // row_shr:4 into the odd banks
        lo = __builtin_amdgcn_update_dpp(lo, lo, 0x114, 0xf, 0xa, false);
        hi = __builtin_amdgcn_update_dpp(hi, hi, 0x114, 0xf, 0xa, false);
    }
    if constexpr (G >= 16) {  // row_shr:8 into the upper two banks
        lo = __builtin_amdgcn_update_dpp(lo, lo, 0x118, 0xf, 0xc, false);
        hi = __builtin_amdgcn_update_dpp(hi, hi, 0x118, 0xf, 0xc, false);
    }
    return __hiloint2double(hi, lo);
}

template <int G, typename T, bool UPPER>
__global__ __launch_bounds__(kStThreads) void k_sweep_st(int n, const int* __restrict__ kptr,
                                                         const int* __restrict__ cptr,
                                                         const int2* __restrict__ irange, uint64_t* mail,
                                                         unsigned mail_words, int* gen, unsigned held,
                                                         const uint2* __restrict__ scol, const T* __restrict__ sval,
                                                         const double2* __restrict__ sdiag, const double* b,
                                                         double* out, const int* gate, int* ctr, int* err,
                                                         uint64_t wd_limit) {
    extern __shared__ double xs[];
    if (gate && *gate == 0) return;
    constexpr int R = 64 / G;
    const int ticket = take_ticket(ctr);
    const Watchdog wd(wd_limit);
    const int nrows = kptr[ticket + 1] - kptr[ticket];
    const int c0 = cptr[ticket], c1 = cptr[ticket + 1];
    const int i0 = irange[ticket].x, nimp = irange[ticket].y;
    const int nslot = nrows + nimp;
    const int parity = peek_int(gen) & 1;
    uint64_t* const box = mail + static_cast<long>(parity) * mail_words;
    for (int i = threadIdx.x; i < nslot; i += kStThreads) xs[i] = __longlong_as_double(kPending);
    for (int i = threadIdx.x; i < nimp; i += kStThreads)
        mail[static_cast<long>(parity ^ 1) * mail_words + i0 + i] = kPending;
    if (threadIdx.x < 2) xs[nslot + threadIdx.x] = 0.0;  // read by unused lanes; written by unused rows
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    bool timed_out = false;
    if (wave >= kStSolvers) {
        // importer: lane l takes imports l, l + 64, ...; a lane moves on as
        // soon as its own value has arrived
        const uint64_t* const src = box + i0;
        int i = lane;
        unsigned rounds = 0;
        while (__ballot(i < nimp) != 0) {
            bool got = false;
            if (i < nimp) {
                uint64_t bits = peek_raw(src + i);
                if (bits == kPending && timed_out) bits = kQuietNan;
                if (bits != kPending) {
                    lds_put(xs, 8u * (nrows + i), __longlong_as_double(bits));
                    i += 64;
                    got = true;
                }
            }
            if ((++rounds & 63u) == 0) timed_out = timed_out || wd.expired();
            if (__ballot(got) == 0) spin_pause();
        }
    } else if (c0 < c1) {
        __builtin_amdgcn_s_setprio(3);
        const bool first = (lane & (G - 1)) == 0;
        const uint64_t first_lanes = __ballot(first);
        const unsigned lds0 =
            static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) double*)xs));
        const Rsrc r_col = st_rsrc(scol, held * 512u);
        const Rsrc r_val = st_rsrc(sval, held * static_cast<unsigned>(64 * sizeof(T)));
        const Rsrc r_diag = st_rsrc(sdiag, UPPER ? held * static_cast<unsigned>(16 * R) : 0u);
        const Rsrc r_b = st_rsrc(b, 8u * n), r_out = st_rsrc(out, 8u * n);
        const Rsrc r_box = st_rsrc(box, 8u * mail_words);
        const unsigned o_col = 8u * lane, o_val = sizeof(T) * lane, o_diag = 16u * (lane / G);
        // past a block's end the requests run into the next block's chunks
        // or the unused ones behind the last, whose values are not used
        unsigned ca = c0 + wave, cb = c0 + wave;  // next chunk of each kind to request
        auto issue_a = [&](StA& a) {
            a.p = st_load2(r_col, o_col, ca * 512u);
            ca += kStSolvers;
        };
        auto issue_b = [&](const StA& a, StB<T>& r) {
            if constexpr (sizeof(T) == 8) r.v = st_load_d(r_val, o_val, cb * 512u);
            else r.v = st_load_f(r_val, o_val, cb * 256u);
            r.b = st_load_d(r_b, first ? a.p.y : kStNone, 0);
            if (UPPER) r.d = st_load_d2(r_diag, o_diag, cb * (16u * R));
            cb += kStSolvers;
        };
        StA ra[kStAhead];
        StB<T> rb[kStAheadB];
#pragma unroll
        for (int u = 0; u < kStAhead; ++u) issue_a(ra[u]);
#pragma unroll
        for (int u = 0; u < kStAheadB; ++u) issue_b(ra[u], rb[u]);
        const int npass = (c1 - c0) / kStSolvers;
        for (int p = 0; p < npass; p += kStAhead) {
#pragma unroll
            for (int u = 0; u < kStAhead; ++u) {
                const StA a = ra[u];
                const StB<T> r = rb[u % kStAheadB];
                if (p + u < npass) {
                    const uint64_t bits = wait_lds(lds0 + (a.p.x & 0x7fffu) * 8u, wd, timed_out);
                    const double sum = group_sum<G>(fma(-__longlong_as_double(bits), static_cast<double>(r.v), r.b));
                    const double x = UPPER ? divide_by(sum, r.d.x, r.d.y, first_lanes) : sum;
                    if (first) lds_put(xs, (a.p.x >> 15) * 8u, x);
                    asm volatile("" ::: "memory");  // the LDS word first: the next level waits for it
                    const double xg = group_first<G>(x);
                    if (first) st_store<kStPlain>(r_out, a.p.y, x);
                    else st_store<kStAgent>(r_box, a.p.y, xg);
                }
                issue_b(ra[(u + kStAheadB) % kStAhead], rb[u % kStAheadB]);
                issue_a(ra[u]);
            }
        }
        __builtin_amdgcn_s_setprio(0);
    }
    if (timed_out) atomicOr(err, kErrTimeout);
    if (retire_ticket(ctr)) publish_int(gen, parity ^ 1);
}

__global__ void k_st_arm(long words, uint64_t* p, const int* gate) {
    if (gate && *gate == 0) return;
    const long stride = static_cast<long>(gridDim.x) * blockDim.x;
    for (long i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x; i < words; i += stride) p[i] = kPending;
}

// ---- stream construction (per pattern, partition and lanes per row) ----

int read_word(const int* d, hipStream_t s) {
    int h = 0;
    PILU_HIP(hipMemcpyAsync(&h, d, sizeof(int), hipMemcpyDeviceToHost, s));
    PILU_HIP(hipStreamSynchronize(s));
    return h;
}

inline int grid_for(long n, int per_block) { return std::max(1, ceil_div(n, per_block)); }

// First schedule position of every processed block.
__global__ void k_st_kptr(int nblk, const int* __restrict__ blev, const int* __restrict__ loff, int* __restrict__ kptr) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p <= nblk) kptr[p] = loff[blev[p]];
}

// Schedule position of every row, and the out-of-block entries of the row
// at every position (cnt[n] = 0, for the scan's total).
__global__ void k_st_count(int n, int upper, const int* __restrict__ perm, const int* __restrict__ rp,
                           const int* __restrict__ dg, const int* __restrict__ ci, const int* __restrict__ block_of,
                           int* __restrict__ kinv, int* __restrict__ cnt) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k == n) cnt[n] = 0;
    if (k >= n) return;
    const int row = perm[k], blk = block_of[row];
    kinv[row] = k;
    const int e1 = upper ? rp[row + 1] : dg[row];
    int c = 0;
    for (int e = upper ? dg[row] + 1 : rp[row]; e < e1; ++e) c += block_of[ci[e]] != blk;
    cnt[k] = c;
}

// Chunks of every block, a multiple of the solver waves (nch[nblk] = 0).
__global__ __launch_bounds__(256) void k_st_chunks(int nblk, int R, const int* __restrict__ blev,
                                                   const int* __restrict__ loff, int* __restrict__ nch) {
    __shared__ int s_sum;
    const int p = blockIdx.x;
    if (threadIdx.x == 0) s_sum = 0;
    __syncthreads();
    int c = 0;
    if (p < nblk)
        for (int g = blev[p] + threadIdx.x; g < blev[p + 1]; g += 256) c += (loff[g + 1] - loff[g] + R - 1) / R;
    if (c) atomicAdd(&s_sum, c);
    __syncthreads();
    if (threadIdx.x == 0) nch[p] = (s_sum + kStSolvers - 1) / kStSolvers * kStSolvers;
}

// Columns of the out-of-block entries, in (position, entry) order.
__global__ void k_st_refs(int n, int upper, const int* __restrict__ perm, const int* __restrict__ rp,
                          const int* __restrict__ dg, const int* __restrict__ ci, const int* __restrict__ block_of,
                          const int* __restrict__ escan, int* __restrict__ refs) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n || escan[k] == escan[k + 1]) return;
    const int row = perm[k], blk = block_of[row];
    const int e1 = upper ? rp[row + 1] : dg[row];
    int at = escan[k];
    for (int e = upper ? dg[row] + 1 : rp[row]; e < e1; ++e)
        if (block_of[ci[e]] != blk) refs[at++] = ci[e];
}

// The distinct out-of-block columns of every block in order of first use:
// imp[r0 + i] is the i-th of the block whose references start at r0,
// irange[p] = {r0, how many}, refs[] becomes the import index of every
// reference.  One workgroup per block with an open-addressed LDS table
// (column -> first reference, then -> import index); a block with more
// references than the table takes keeps one import per reference.
constexpr int kStTable = 1 << 14;
constexpr int kStMaxRefs = kStTable * 3 / 4;
constexpr size_t kStTableLds = static_cast<size_t>(kStTable) * 8;

__global__ __launch_bounds__(1024) void k_st_dedupe(int nblk, const int* __restrict__ kptr,
                                                    const int* __restrict__ escan, int* __restrict__ refs,
                                                    int* __restrict__ imp, int2* __restrict__ irange) {
    extern __shared__ int s_tab[];
    __shared__ int s_scan[16];
    int* key = s_tab;
    int* val = s_tab + kStTable;
    const int p = blockIdx.x, tid = threadIdx.x;
    const int r0 = escan[kptr[p]], m = escan[kptr[p + 1]] - r0;
    if (m > kStMaxRefs) {
        for (int i = tid; i < m; i += 1024) {
            imp[r0 + i] = refs[r0 + i];
            refs[r0 + i] = i;
        }
        if (tid == 0) irange[p] = make_int2(r0, m);
        return;
    }
    for (int i = tid; i < kStTable; i += 1024) {
        key[i] = -1;
        val[i] = 0x7fffffff;
    }
    __syncthreads();
    auto find = [&](int col, bool insert) {
        unsigned h = (static_cast<unsigned>(col) * 2654435761u) >> 18;  // top 14 bits
        while (true) {
            const int k = insert ? atomicCAS(&key[h], -1, col) : key[h];
            if (k == col || (insert && k == -1)) return h;
            h = (h + 1) & (kStTable - 1);
        }
    };
    for (int i = tid; i < m; i += 1024) atomicMin(&val[find(refs[r0 + i], true)], i);
    __syncthreads();
    int base = 0;
    for (int i0 = 0; i0 < m; i0 += 1024) {
        const int i = i0 + tid;
        const int col = i < m ? refs[r0 + i] : 0;
        const unsigned h = i < m ? find(col, false) : 0;
        const bool first = i < m && val[h] == i;
        const uint64_t mask = __ballot(first);
        if ((tid & 63) == 0) s_scan[tid >> 6] = __popcll(mask);
        __syncthreads();
        int before = base, all = 0;
        for (int w = 0; w < 16; ++w) {
            if (w < (tid >> 6)) before += s_scan[w];
            all += s_scan[w];
        }
        if (first) {
            const int at = before + __popcll(mask & ((1ull << (tid & 63)) - 1));
            imp[r0 + at] = col;
            val[h] = -1 - at;  // from here on the entry's import index
        }
        base += all;
        __syncthreads();
    }
    for (int i = tid; i < m; i += 1024) refs[r0 + i] = -1 - val[find(refs[r0 + i], false)];
    if (tid == 0) irange[p] = make_int2(r0, base);
}

// {first position, rows} of every chunk; the last few of a block may have no rows.
__global__ __launch_bounds__(256) void k_st_cut(int R, const int* __restrict__ blev, const int* __restrict__ loff,
                                                const int* __restrict__ cptr, int2* __restrict__ chunks) {
    __shared__ int s_scan[256];
    const int p = blockIdx.x, tid = threadIdx.x;
    const int g1 = blev[p + 1], c1 = cptr[p + 1];
    int base = cptr[p];
    for (int g0 = blev[p]; g0 < g1; g0 += 256) {
        const int g = g0 + tid;
        const int lo = g < g1 ? loff[g] : 0, hi = g < g1 ? loff[g + 1] : 0;
        const int m = (hi - lo + R - 1) / R;
        s_scan[tid] = m;
        __syncthreads();
        for (int o = 1; o < 256; o <<= 1) {
            const int v = tid >= o ? s_scan[tid - o] : 0;
            __syncthreads();
            s_scan[tid] += v;
            __syncthreads();
        }
        int at = base + s_scan[tid] - m;
        for (int k = lo; k < hi; k += R) chunks[at++] = make_int2(k, min(R, hi - k));
        base += s_scan[255];
        __syncthreads();
    }
    for (int c = base + tid; c < c1; c += 256) chunks[c] = make_int2(0, 0);
}

// Stream of one lane: its x address and the factor entry it holds (-1:
// none), and the row ids.  A chunk's block is found by bisection of cptr;
// the chunks past the last one hold nothing.
template <bool UPPER>
__global__ void k_st_fill(long nlanes, int nchunk, int G, int nblk, const int2* __restrict__ chunks, const int* __restrict__ cptr,
                          const int* __restrict__ kptr, const int2* __restrict__ irange,
                          const int* __restrict__ escan, const int* __restrict__ refs,
                          const int* __restrict__ perm, const int* __restrict__ kinv, const int* __restrict__ rp,
                          const int* __restrict__ dg, const int* __restrict__ ci, const int* __restrict__ block_of,
                          uint2* __restrict__ scol, int* __restrict__ ssrc, int* __restrict__ srow,
                          int* __restrict__ rowlane) {
    const long i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
    if (i >= nlanes) return;
    const int R = 64 / G;
    const int c = static_cast<int>(i >> 6), l = static_cast<int>(i & 63), j = l / G, t = l % G;
    if (c >= nchunk) {
        scol[i] = make_uint2(0, kStNone);
        ssrc[i] = -1;
        if (t == 0) srow[static_cast<long>(c) * R + j] = -1;
        return;
    }
    int lo = 0, hi = nblk;  // last block with cptr <= c
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (cptr[mid] <= c) lo = mid; else hi = mid;
    }
    const int k0 = kptr[lo], nrows = kptr[lo + 1] - k0;
    const int nimp = irange[lo].y;
    // unused lanes read the slot that holds 0, unused rows write the one after it
    unsigned xa = nrows + nimp, own = nrows + nimp + 1;
    int src = -1, row = -1;
    const int2 ch = chunks[c];
    if (j < ch.y) {
        const int k = ch.x + j;
        row = perm[k];
        own = k - k0;
        const int blk = block_of[row];
        const int e0 = UPPER ? dg[row] + 1 : rp[row], e1 = UPPER ? rp[row + 1] : dg[row];
        if (t < e1 - e0) {
            const int col = ci[e0 + t];
            src = e0 + t;
            if (block_of[col] == blk) {
                xa = kinv[col] - k0;
            } else {
                int at = escan[k];
                for (int e = e0; e < e0 + t; ++e) at += block_of[ci[e]] != blk;
                xa = nrows + refs[at];
            }
        }
    }
    scol[i] = make_uint2(xa | own << 15, t == 0 && row >= 0 ? 8u * row : kStNone);
    ssrc[i] = src;
    if (t == 0) {
        srow[static_cast<long>(c) * R + j] = row;
        if (row >= 0) rowlane[row] = static_cast<int>(i);
    }
}

// Mailbox words of every row's importers, one per lane of the row but the
// first (rowlane[row]); *over is set when a row has more than G - 1.
// irefs: where a block's imports are listed, irange: its mailbox words.
__global__ __launch_bounds__(256) void k_st_exports(int G, const int2* __restrict__ irefs,
                                                    const int2* __restrict__ irange, const int* __restrict__ imp,
                                                    const int* __restrict__ rowlane, int* __restrict__ cnt,
                                                    uint2* __restrict__ scol, int* __restrict__ over) {
    const int2 r = irefs[blockIdx.x];
    const int m0 = irange[blockIdx.x].x;
    for (int i = threadIdx.x; i < r.y; i += 256) {
        const int row = imp[r.x + i];
        const int at = 1 + atomicAdd(cnt + row, 1);
        if (at < G) scol[rowlane[row] + at].y = 8u * static_cast<unsigned>(m0 + i);
        else *over = 1;
    }
}

// Values of the stream from the factors, and {u_ii, 1 / u_ii} per row (U).
template <typename T>
__global__ void k_st_gather(long nlanes, const int* __restrict__ src, const T* __restrict__ fac, T* __restrict__ sval,
                            long nrow, const int* __restrict__ srow, const int* __restrict__ dg,
                            double2* __restrict__ sdiag) {
    const long stride = static_cast<long>(gridDim.x) * blockDim.x;
    const long i0 = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
    for (long i = i0; i < nlanes; i += stride) {
        const int s = src[i];
        sval[i] = s >= 0 ? fac[s] : T(0);
    }
    if (sdiag)
        for (long k = i0; k < nrow; k += stride) {
            const int row = srow[k];
            const double d = row >= 0 ? static_cast<double>(fac[dg[row]]) : 1.0;
            sdiag[k] = make_double2(d, recip_for(d));
        }
}

template <int G, typename T, bool UPPER>
void launch_st(Ext* e, const SweepStream& st, const T* sval, const double* b, double* out, const int* gate, int* ctr,
               int* err) {
    auto kern = k_sweep_st<G, T, UPPER>;
    PILU_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                 static_cast<int>(st.lds)));
    kern<<<st.nblk, kStThreads, st.lds, e->stream>>>(
        e->n, st.kptr.get(), st.cptr.get(), reinterpret_cast<const int2*>(st.irange.get()), st.mail.get(),
        static_cast<unsigned>(st.mail_words), st.gen.get(), static_cast<unsigned>(st.nchunk + kStOverrun),
        reinterpret_cast<const uint2*>(st.scol.get()), sval, reinterpret_cast<const double2*>(st.sdiag.get()), b, out,
        gate, ctr, err, watchdog_ticks(e->watchdog_s));
}

template <typename T, bool UPPER>
void sweep_st_t(Ext* e, const SweepStream& st, const T* sval, const double* b, double* out, const int* gate, int* ctr,
                int* err) {
    switch (st.g) {
        case 2: launch_st<2, T, UPPER>(e, st, sval, b, out, gate, ctr, err); break;
        case 4: launch_st<4, T, UPPER>(e, st, sval, b, out, gate, ctr, err); break;
        case 8: launch_st<8, T, UPPER>(e, st, sval, b, out, gate, ctr, err); break;
        default: launch_st<16, T, UPPER>(e, st, sval, b, out, gate, ctr, err); break;
    }
}

}  // namespace

bool stream_width_fits(const Ext* e, bool upper, int G) {
    return G >= 2 && G <= 16 && (upper ? e->max_up : e->max_lo) <= G;
}

bool build_stream(Ext* e, bool upper, int G, const StreamSchedule& sc, SweepStream& st) {
    refuse_if_no_alloc(e, "sweep stream");
    const int n = e->n, nblk = sc.nblk, R = 64 / G, up = upper ? 1 : 0;
    hipStream_t s = e->stream;
    const int *perm = sc.perm, *blev = sc.blev, *loff = sc.loff, *block_of = sc.block_of;
    st.g = G;
    st.nblk = nblk;
    st.factors = -1;
    st.lds = 0;
    DevBuf<int> irefs(2 * static_cast<size_t>(nblk));
    DevBuf<int> kinv(n), cnt(static_cast<size_t>(n) + 1), escan(static_cast<size_t>(n) + 1);
    DevBuf<int> nch(static_cast<size_t>(nblk) + 1);
    const size_t nb1 = static_cast<size_t>(nblk) + 1;
    st.kptr.reserve(nb1);
    st.cptr.reserve(nb1);
    st.irange.reserve(2 * nb1);
    k_st_kptr<<<grid_for(nblk + 1, 256), 256, 0, s>>>(nblk, blev, loff, st.kptr.get());
    k_st_count<<<grid_for(static_cast<long>(n) + 1, 256), 256, 0, s>>>(n, up, perm, e->rp.get(), e->dg.get(),
                                                                      e->ci.get(), block_of, kinv.get(),
                                                                      cnt.get());
    PILU_HIP(hipGetLastError());
    auto scan = [&](const int* in, int* out, size_t m) {
        size_t bytes = 0;
        PILU_HIP(rocprim::exclusive_scan(nullptr, bytes, in, out, 0, m, rocprim::plus<int>(), s));
        e->sort_tmp.reserve(bytes);
        PILU_HIP(rocprim::exclusive_scan(e->sort_tmp.get(), bytes, in, out, 0, m, rocprim::plus<int>(), s));
    };
    scan(cnt.get(), escan.get(), static_cast<size_t>(n) + 1);
    k_st_chunks<<<nblk + 1, 256, 0, s>>>(nblk, R, blev, loff, nch.get());
    PILU_HIP(hipGetLastError());
    scan(nch.get(), st.cptr.get(), nb1);
    // references per partition are bounded by the entries of one triangle
    const int nref = read_word(escan.get() + n, s);
    DevBuf<int> refs(std::max(nref, 1)), imp(std::max(nref, 1));
    k_st_refs<<<grid_for(n, 256), 256, 0, s>>>(n, up, perm, e->rp.get(), e->dg.get(), e->ci.get(),
                                              block_of, escan.get(), refs.get());
    PILU_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_st_dedupe),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(kStTableLds)));
    k_st_dedupe<<<nblk, 1024, kStTableLds, s>>>(nblk, st.kptr.get(), escan.get(), refs.get(), imp.get(),
                                               reinterpret_cast<int2*>(irefs.get()));
    PILU_HIP(hipGetLastError());
    std::vector<int> h(4 * nb1);
    PILU_HIP(hipMemcpyAsync(h.data(), st.kptr.get(), sizeof(int) * nb1, hipMemcpyDeviceToHost, s));
    PILU_HIP(hipMemcpyAsync(h.data() + nb1, st.cptr.get(), sizeof(int) * nb1, hipMemcpyDeviceToHost, s));
    PILU_HIP(hipMemcpyAsync(h.data() + 2 * nb1, irefs.get(), 2 * sizeof(int) * nblk, hipMemcpyDeviceToHost, s));
    PILU_HIP(hipStreamSynchronize(s));
    size_t lds = kStMinLds;
    st.max_chunks = 0;
    st.mail_words = 0;
    for (int p = 0; p < nblk; ++p) {
        const size_t rows = h[p + 1] - h[p], imps = h[2 * nb1 + 2 * p + 1];
        h[2 * nb1 + 2 * p] = static_cast<int>(st.mail_words);
        st.mail_words += static_cast<long>(imps);
        lds = std::max(lds, st_block_lds(rows, imps));
        st.max_chunks = std::max(st.max_chunks, h[nb1 + p + 1] - h[nb1 + p]);
    }
    st.nchunk = h[nb1 + nblk];
    // every buffer has 32-bit byte offsets and the block fits the LDS (so
    // its slots 15 bits); the packed factors take the partition otherwise
    if (lds > kStMaxLds || st.nchunk + kStOverrun > (1L << 31) / 512 || st.mail_words >= (1L << 28) || n >= (1 << 28))
        return false;
    const long held = st.nchunk + kStOverrun, nlanes = held * 64;
    // slots, source, value; per row its id and the diagonal; two generations of mailboxes
    const size_t lane_bytes = sizeof(uint2) + sizeof(int) + sizeof(double), row_bytes = sizeof(int) + 2 * sizeof(double);
    if (nlanes * lane_bytes + held * R * row_bytes + 2 * sizeof(uint64_t) * st.mail_words > e->stream_budget()) return false;
    PILU_HIP(hipMemcpyAsync(st.irange.get(), h.data() + 2 * nb1, 2 * sizeof(int) * nblk, hipMemcpyHostToDevice, s));
    int* rowlane = cnt.get();  // the counts have been scanned
    DevBuf<int> chunks(2 * static_cast<size_t>(std::max<long>(st.nchunk, 1)));
    st.scol.reserve(2 * nlanes);
    st.ssrc.reserve(nlanes);
    st.srow.reserve(held * R);
    k_st_cut<<<nblk, 256, 0, s>>>(R, blev, loff, st.cptr.get(), reinterpret_cast<int2*>(chunks.get()));
    auto fill = upper ? k_st_fill<true> : k_st_fill<false>;
    fill<<<grid_for(nlanes, 256), 256, 0, s>>>(
        nlanes, static_cast<int>(st.nchunk), G, nblk, reinterpret_cast<const int2*>(chunks.get()), st.cptr.get(),
        st.kptr.get(), reinterpret_cast<const int2*>(irefs.get()), escan.get(), refs.get(), perm, kinv.get(),
        e->rp.get(), e->dg.get(), e->ci.get(), block_of, reinterpret_cast<uint2*>(st.scol.get()), st.ssrc.get(),
        st.srow.get(), rowlane);
    // every import becomes a mailbox word its row's lanes store to
    DevBuf<int> exported(static_cast<size_t>(n) + 1);
    PILU_HIP(hipMemsetAsync(exported.get(), 0, sizeof(int) * (static_cast<size_t>(n) + 1), s));
    if (st.mail_words > 0)
        k_st_exports<<<nblk, 256, 0, s>>>(G, reinterpret_cast<const int2*>(irefs.get()),
                                          reinterpret_cast<const int2*>(st.irange.get()), imp.get(), rowlane,
                                          exported.get(), reinterpret_cast<uint2*>(st.scol.get()),
                                          exported.get() + n);
    st.mail.reserve(2 * static_cast<size_t>(std::max(st.mail_words, 1L)));
    st.gen.reserve(1);
    PILU_HIP(hipMemsetAsync(st.gen.get(), 0, sizeof(int), s));
    k_st_arm<<<grid_for(2 * st.mail_words, 256 * 8), 256, 0, s>>>(2 * st.mail_words, st.mail.get(), nullptr);
    PILU_HIP(hipGetLastError());
    if (read_word(exported.get() + n, s) != 0) return false;  // a row with more importing blocks than lanes
    st.lds = lds;
    return true;
}

void gather_stream(Ext* e, bool upper, SweepStream& st) {
    refuse_if_no_alloc(e, "sweep stream values");
    const long held = st.nchunk + kStOverrun, nlanes = held * 64, nrow = held * (64 / st.g);
    if (upper) st.sdiag.reserve(2 * nrow);
    double2* sdiag = upper ? reinterpret_cast<double2*>(st.sdiag.get()) : nullptr;
    const int grid = 2048;
    if (e->precision == 32) {
        st.sval32.reserve(nlanes);
        k_st_gather<float><<<grid, 256, 0, e->stream>>>(nlanes, st.ssrc.get(), e->fac32.get(), st.sval32.get(), nrow,
                                                        st.srow.get(), e->dg.get(), sdiag);
    } else {
        st.sval64.reserve(nlanes);
        k_st_gather<double><<<grid, 256, 0, e->stream>>>(nlanes, st.ssrc.get(), e->fac.get(), st.sval64.get(), nrow,
                                                         st.srow.get(), e->dg.get(), sdiag);
    }
    PILU_HIP(hipGetLastError());
    st.factors = e->factor_version;
}

void sweep_stream(Ext* e, bool upper, const SweepStream& st, const double* b, double* out, double* reset,
                  const int* gate, int* ctr, int* err) {
    if (st.lds == 0 || st.factors != e->factor_version)
        throw std::runtime_error("stream sweep: stream missing (factorize before sweeping)");
    if (e->precision == 32) {
        if (upper) sweep_st_t<float, true>(e, st, st.sval32.get(), b, out, gate, ctr, err);
        else sweep_st_t<float, false>(e, st, st.sval32.get(), b, out, gate, ctr, err);
    } else {
        if (upper) sweep_st_t<double, true>(e, st, st.sval64.get(), b, out, gate, ctr, err);
        else sweep_st_t<double, false>(e, st, st.sval64.get(), b, out, gate, ctr, err);
    }
    // the other direction's output, where that one waits on value-flags: this
    // sweep has read b, which may be the same vector
    if (reset)
        k_st_arm<<<grid_for(e->n, 256 * 8), 256, 0, e->stream>>>(e->n, reinterpret_cast<uint64_t*>(reset), gate);
}

}  // namespace pilu
