// Learned diagonal compensation: a 3-layer message-passing network over the
// matrix graph that predicts, for every row, the relaxation factor omega_i
// of the compensated factorization (IluSolver::SetDiagonalCompensation).
// No counterpart in the reference.
//
// Graph: rows are nodes, off-diagonal entries a_ij are edges with weight
// w_ij = a_ij / sqrt(|a_ii a_jj|).  Node features (16, eight used): scale-
// free row statistics (diagonal dominance, signed row sum, extreme
// couplings, degree, coupling energy, lower-triangle share).
// Layer l (input width D = 16, 32, 32; hidden 32):
//   M = W_graph H;  Z = [H | M] W_l + b_l;  H' = relu(Z)
// Head: omega = sigmoid(H_3 w_o + b_o).
// The dense products run on BF16 MFMA (v_mfma_f32_16x16x16_bf16) with FP32
// accumulation; gathers, head, loss and Adam are FP32.  Training minimises
// the mean squared error between omega and per-row targets.  All reductions
// over rows are two-level with a fixed order, so gradients are
// deterministic.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <stdexcept>
#include <vector>

#include "common.hpp"
#include "gmres.hpp"
#include "par_ilu_ex.h"

namespace pilu {
namespace gnn {

constexpr int kHid = 32;
constexpr int kFeat = 16;
constexpr int kLayers = 3;
constexpr int kInDim[kLayers] = {kFeat, kHid, kHid};
// parameter layout: W0 (32x32), b0, W1 (64x32), b1, W2 (64x32), b2, wo (32), bo
constexpr int kOffW[kLayers] = {0, 1024 + 32, 1024 + 32 + 2048 + 32};
constexpr int kOffB[kLayers] = {1024, 1024 + 32 + 2048, 1024 + 32 + 2048 + 32 + 2048};
constexpr int kOffWo = 1024 + 32 + 2 * (2048 + 32);
constexpr int kOffBo = kOffWo + kHid;
constexpr int kParams = kOffBo + 1;  // 5249

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ unsigned short f2bf(float f) {
    const uint32_t u = __float_as_uint(f);
    return static_cast<unsigned short>((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);  // round to nearest even
}

__device__ __forceinline__ short bits_bf(float f) { return static_cast<short>(f2bf(f)); }

// ---- features ----
__global__ void k_diag_values(int n, const int* __restrict__ rp, const int* __restrict__ ci,
                              const double* __restrict__ va, double* __restrict__ d) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double v = 0.0;
    for (int e = rp[i]; e < rp[i + 1]; ++e)
        if (ci[e] == i) v = va[e];
    d[i] = v;
}

// Row features and edge weights.  A workgroup's 256 rows are one contiguous
// range of entries: they are staged in LDS by coalesced reads, with the
// columns' diagonals, and the weights leave the same way; each thread then
// walks its own row in LDS (240 us at 128^3 when every thread read and wrote
// its row in memory).  Ranges past the LDS take the entries from memory.
constexpr int kFeatRows = 256;
constexpr int kFeatEntries = 2560;
__global__ __launch_bounds__(kFeatRows) void k_features(int n, const int* __restrict__ rp, const int* __restrict__ ci,
                                                        const double* __restrict__ va, const double* __restrict__ d,
                                                        float* __restrict__ feat, float* __restrict__ ew) {
    __shared__ double s_a[kFeatEntries], s_d[kFeatEntries];
    __shared__ int s_j[kFeatEntries];
    const int r0 = blockIdx.x * kFeatRows, r1 = min(n, r0 + kFeatRows);
    const int p0 = rp[r0], p1 = rp[r1];
    const bool staged = p1 - p0 <= kFeatEntries;
    if (staged) {
        for (int e = p0 + threadIdx.x; e < p1; e += kFeatRows) {
            const int j = ci[e];
            s_j[e - p0] = j;
            s_a[e - p0] = va[e];
            s_d[e - p0] = d[j];
        }
        __syncthreads();
    }
    const int i = r0 + threadIdx.x;
    if (i < n) {
        const double di = d[i];
        const double ai = fabs(di) > 0 ? fabs(di) : 1.0;
        double sabs = 0, ssum = 0, mx = 0, mn = 1e300, sw2 = 0, lower = 0;
        int cnt = 0;
        for (int e = rp[i]; e < rp[i + 1]; ++e) {
            const int j = staged ? s_j[e - p0] : ci[e];
            double w = 0.0;
            if (j != i) {
                const double a = staged ? s_a[e - p0] : va[e];
                const double dc = staged ? s_d[e - p0] : d[j];
                const double dj = fabs(dc) > 0 ? fabs(dc) : 1.0;
                w = a / sqrt(ai * dj);
                sabs += fabs(a);
                ssum += a;
                mx = fabs(a) > mx ? fabs(a) : mx;
                mn = fabs(a) < mn ? fabs(a) : mn;
                sw2 += w * w;
                if (j < i) lower += fabs(a);
                ++cnt;
            }
            if (staged) s_a[e - p0] = w;
            else ew[e] = static_cast<float>(w);
        }
        if (cnt == 0) mn = 0;
        f32x4* f = reinterpret_cast<f32x4*>(feat + static_cast<long>(i) * kFeat);
        f[0] = {1.f, static_cast<float>(sabs / ai), static_cast<float>(ssum / (di != 0 ? di : 1.0)),
                static_cast<float>(mx / ai)};
        f[1] = {static_cast<float>(mn / ai), cnt / 8.f, static_cast<float>(sw2),
                static_cast<float>(sabs > 0 ? lower / sabs : 0.0)};
        f[2] = f[3] = {0.f, 0.f, 0.f, 0.f};
    }
    if (staged) {
        __syncthreads();
        for (int e = p0 + threadIdx.x; e < p1; e += kFeatRows) ew[e] = static_cast<float>(s_a[e - p0]);
    }
}

__device__ __forceinline__ bf16x4 to_bf(const f32x4& v) {
    bf16x4 r;
#pragma unroll
    for (int t = 0; t < 4; ++t) r[t] = bits_bf(v[t]);
    return r;
}

// out[i] += sum_e w_e H[col_e]: D / 4 lanes per row, four features each, a
// row's edges read four at a time and summed in edge order.
template <int D>
__global__ __launch_bounds__(256) void k_aggregate(int n, const int* __restrict__ rp, const int* __restrict__ ci,
                                                   const float* __restrict__ w, const float* __restrict__ h,
                                                   float* __restrict__ out) {
    constexpr int L = D / 4;
    const long row = (static_cast<long>(blockIdx.x) * 256 + threadIdx.x) / L;
    if (row >= n) return;
    const int d = (threadIdx.x % L) * 4;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    int e = rp[row];
    const int e1 = rp[row + 1];
    for (; e < e1; e += 4) {
        float we[4];
        f32x4 he[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int k = e + q < e1 ? e + q : e1 - 1;
            we[q] = w[k];
            he[q] = *reinterpret_cast<const f32x4*>(h + static_cast<long>(ci[k]) * D + d);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (e + q < e1)
#pragma unroll
                for (int t = 0; t < 4; ++t) acc[t] = fmaf(we[q], he[q][t], acc[t]);
    }
    f32x4* o = reinterpret_cast<f32x4*>(out + row * D + d);
    f32x4 r = *o;
#pragma unroll
    for (int t = 0; t < 4; ++t) r[t] += acc[t];
    *o = r;
}

// One message-passing layer: M = W_graph H, hout = relu([H | M] W + b), and
// after the last layer (HEAD) omega = sigmoid(hout wo + bo).  A wave takes 16
// rows: four neighbouring lanes gather a row's messages, 16 bytes each per 16
// features, so a request touches 16 lines (one lane per row, as the MFMA
// operand has it, touched 64 and was bound by them: 340 us per 32-wide layer
// at 128^3); the rounded sums then move to their operand lanes and M never
// leaves registers.  The weights stay in registers over a wave's tiles.
// TRAIN also stores M (and the last layer's output) for the backward pass.
// Messages are summed in edge order, the products in ascending k.
//
// Bound by memory traffic: H in (with its neighbours, mostly from L2), edges,
// H out.  Rows are dealt to the XCDs in eight contiguous slabs (workgroup b
// runs on XCD b % 8), so a row's grid neighbours are in the same L2.  As
// separate aggregate, dense and head passes over M and an unused Z a forward
// pass at 128^3 took 2.72 ms (563 + 372 us per 32-wide layer).
template <int D, bool TRAIN, bool HEAD>
__global__ __launch_bounds__(256) void k_layer(int n, const int* __restrict__ rp, const int* __restrict__ ci,
                                               const float* __restrict__ w, const float* __restrict__ h,
                                               const unsigned short* __restrict__ wb, const float* __restrict__ b,
                                               float* __restrict__ hout, float* __restrict__ mout,
                                               const float* __restrict__ prm, float* __restrict__ omega) {
    constexpr int KH = D / 16;  // 16-wide steps over H, then as many over M
    constexpr int E = 8;        // edges requested together
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int ar = lane & 15, kq = lane >> 4;  // place in the MFMA operands
    const int gr = lane >> 2, gq = lane & 3;   // row and 16-byte piece while gathering
    bf16x4 w0[2 * KH], w1[2 * KH];
#pragma unroll
    for (int ks = 0; ks < 2 * KH; ++ks)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int k = ks * 16 + kq * 4 + t;
            w0[ks][t] = static_cast<short>(wb[k * kHid + ar]);
            w1[ks][t] = static_cast<short>(wb[k * kHid + 16 + ar]);
        }
    const float b0 = b[ar], b1 = b[16 + ar];
    float o0 = 0.f, o1 = 0.f, ob = 0.f;
    if constexpr (HEAD) {
        o0 = prm[kOffWo + ar];
        o1 = prm[kOffWo + 16 + ar];
        ob = prm[kOffBo];
    }
    const long tiles = (static_cast<long>(n) + 63) / 64, slab = (tiles + 7) / 8, step = gridDim.x >> 3;
    const long t1 = min(tiles, slab * ((blockIdx.x & 7) + 1));
    // the wave's row of tile t (clamped: lanes past n repeat the last row)
    auto row_of = [&](long t) {
        const long r = min(t, t1 - 1) * 64 + wave * 16 + gr;
        return r < n ? r : static_cast<long>(n) - 1;
    };
    // a row's entry range two tiles ahead, its first E entries one tile ahead
    int ea, eb, c[E];
    float we[E];
    auto fetch_entries = [&](int e, int e1) {
#pragma unroll
        for (int q = 0; q < E; ++q) {
            int k = e + q < e1 ? e + q : e1 - 1;
            k = k > 0 ? k : 0;
            we[q] = w[k];
            c[q] = ci[k];
        }
    };
    long tile = slab * (blockIdx.x & 7) + (blockIdx.x >> 3);
    if (tile >= t1) return;
    ea = rp[row_of(tile)];
    eb = rp[row_of(tile) + 1];
    fetch_entries(ea, eb);
    int na = rp[row_of(tile + step)], nb = rp[row_of(tile + step) + 1];
    for (; tile < t1; tile += step) {
        const long r0 = tile * 64 + wave * 16, row = row_of(tile);
        f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
        f32x4 m[KH], own[KH];
#pragma unroll
        for (int k = 0; k < KH; ++k) {
            m[k] = {0.f, 0.f, 0.f, 0.f};
            own[k] = *(reinterpret_cast<const f32x4*>(h + row * D) + k * 4 + gq);
        }
        int e = ea;
        const int e1 = eb;
        auto gather = [&](bool next) {
            f32x4 he[E][KH];
            float wq[E];
#pragma unroll
            for (int q = 0; q < E; ++q) {
                wq[q] = we[q];
                const f32x4* src = reinterpret_cast<const f32x4*>(h + static_cast<long>(c[q]) * D) + gq;
#pragma unroll
                for (int j = 0; j < KH; ++j) he[q][j] = src[j * 4];
            }
            if (next) {
                ea = na;
                eb = nb;
                fetch_entries(ea, eb);
                na = rp[row_of(tile + 2 * step)];
                nb = rp[row_of(tile + 2 * step) + 1];
            }
#pragma unroll
            for (int q = 0; q < E; ++q)
                if (e + q < e1)
#pragma unroll
                    for (int j = 0; j < KH; ++j)
#pragma unroll
                        for (int t = 0; t < 4; ++t) m[j][t] = fmaf(wq[q], he[q][j][t], m[j][t]);
            e += E;
        };
        // rows of more than E entries take further rounds before the next
        // tile's entries are requested
        while (__ballot(e1 - e > E) != 0) {
            gather(false);
            fetch_entries(e, e1);
        }
        gather(true);
        // own row first, then the messages: 16 columns at a time, rounded and
        // moved from lane 4 row + piece to lane row + 16 piece
        auto product = [&](const f32x4& v, int ks) {
            const int2 q = __builtin_bit_cast(int2, to_bf(v));
            const int2 p = make_int2(__shfl(q.x, ar * 4 + kq, 64), __shfl(q.y, ar * 4 + kq, 64));
            const bf16x4 x = __builtin_bit_cast(bf16x4, p);
            acc0 = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(x, w0[ks], acc0, 0, 0, 0);
            acc1 = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(x, w1[ks], acc1, 0, 0, 0);
        };
#pragma unroll
        for (int ks = 0; ks < KH; ++ks) product(own[ks], ks);
#pragma unroll
        for (int ks = 0; ks < KH; ++ks) {
            product(m[ks], KH + ks);
            if (TRAIN && r0 + gr < n) *(reinterpret_cast<f32x4*>(mout + row * D) + ks * 4 + gq) = m[ks];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const long r = r0 + kq * 4 + j;
            const float z0 = acc0[j] + b0, z1 = acc1[j] + b1;
            const float h0 = z0 > 0.f ? z0 : 0.f, h1 = z1 > 0.f ? z1 : 0.f;
            if ((TRAIN || !HEAD) && r < n) {
                hout[r * kHid + ar] = h0;
                hout[r * kHid + 16 + ar] = h1;
            }
            if constexpr (HEAD) {
                float u = fmaf(h0, o0, h1 * o1);
#pragma unroll
                for (int off = 1; off < 16; off <<= 1) u += __shfl_xor(u, off, 64);
                if (ar == 0 && r < n) omega[r] = 1.f / (1.f + expf(-(u + ob)));
            }
        }
    }
}

// dX = (dHout * [Hout > 0]) W^T, split into dH (first D columns) and dM
// (relu's output is positive exactly where its input is).
template <int D>
__global__ __launch_bounds__(256) void k_dense_bwd_x(int n, const float* __restrict__ dhout, const float* __restrict__ hout,
                                                     const unsigned short* __restrict__ wb, float* __restrict__ dh,
                                                     float* __restrict__ dm) {
    constexpr int K = 2 * D;
    const int lane = threadIdx.x & 63;
    const long r0 = (static_cast<long>(blockIdx.x) * 4 + (threadIdx.x >> 6)) * 16;
    if (r0 >= n) return;
    const int ar = lane & 15, kq = lane >> 4;
    const long arow = r0 + ar;
    f32x4 acc[K / 16];
#pragma unroll
    for (int t = 0; t < K / 16; ++t) acc[t] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < kHid / 16; ++ks) {
        const int k0 = ks * 16 + kq * 4;
        bf16x4 a;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            float g = 0.f;
            if (arow < n) {
                const long o = arow * kHid + k0 + t;
                g = hout[o] > 0.f ? dhout[o] : 0.f;
            }
            a[t] = bits_bf(g);
        }
#pragma unroll
        for (int ct = 0; ct < K / 16; ++ct) {
            bf16x4 bb;
#pragma unroll
            for (int t = 0; t < 4; ++t) bb[t] = static_cast<short>(wb[(ct * 16 + ar) * kHid + k0 + t]);
            acc[ct] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, bb, acc[ct], 0, 0, 0);
        }
    }
#pragma unroll
    for (int ct = 0; ct < K / 16; ++ct)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const long row = r0 + kq * 4 + j;
            if (row >= n) continue;
            const int c = ct * 16 + ar;
            if (c < D) dh[row * D + c] = acc[ct][j];
            else dm[row * D + (c - D)] = acc[ct][j];
        }
}

// Partials of dW = [H | M]^T dZ (K x 32) and db = sum dZ (32), one per
// workgroup: its waves take 16-row tiles in turn, their sums are added in
// wave order in LDS.  kWgradBlocks workgroups of four waves keep every CU
// busy; one wave per 512 rows and a serial sum of its partials by one thread
// per weight took 229 + 148 us per layer at 64^3.
constexpr int kWgradBlocks = 512;
template <int D>
__global__ __launch_bounds__(256) void k_dense_bwd_w(int n, const float* __restrict__ h, const float* __restrict__ m,
                                                     const float* __restrict__ dhout, const float* __restrict__ hout,
                                                     float* __restrict__ part) {
    constexpr int K = 2 * D;
    constexpr int LEN = K * kHid + kHid;
    __shared__ float s_sum[LEN];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int ar = lane & 15, kq = lane >> 4;
    f32x4 acc[K / 16][2];
#pragma unroll
    for (int ft = 0; ft < K / 16; ++ft) acc[ft][0] = acc[ft][1] = {0.f, 0.f, 0.f, 0.f};
    float db[2] = {0.f, 0.f};
    for (long r0 = (static_cast<long>(blockIdx.x) * 4 + wave) * 16; r0 < n; r0 += static_cast<long>(gridDim.x) * 64) {
        // B operand rows: data rows r0 + kq*4 + t; columns c = ct*16 + ar
        bf16x4 bz[2];
#pragma unroll
        for (int ct = 0; ct < 2; ++ct)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const long row = r0 + kq * 4 + t;
                float g = 0.f;
                if (row < n) {
                    const long o = row * kHid + ct * 16 + ar;
                    g = hout[o] > 0.f ? dhout[o] : 0.f;
                }
                db[ct] += g;
                bz[ct][t] = bits_bf(g);
            }
#pragma unroll
        for (int ft = 0; ft < K / 16; ++ft) {
            bf16x4 a;  // A[f][k] = X[row k][f], f = ft*16 + ar
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const long row = r0 + kq * 4 + t;
                const int f = ft * 16 + ar;
                float x = 0.f;
                if (row < n) x = f < D ? h[row * D + f] : m[row * D + (f - D)];
                a[t] = bits_bf(x);
            }
            acc[ft][0] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, bz[0], acc[ft][0], 0, 0, 0);
            acc[ft][1] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, bz[1], acc[ft][1], 0, 0, 0);
        }
    }
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
        db[ct] += __shfl_xor(db[ct], 16, 64);
        db[ct] += __shfl_xor(db[ct], 32, 64);
    }
    for (int wv = 0; wv < 4; ++wv) {
        if (wave == wv) {
#pragma unroll
            for (int ft = 0; ft < K / 16; ++ft)
#pragma unroll
                for (int ct = 0; ct < 2; ++ct)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        float* q = s_sum + (ft * 16 + kq * 4 + j) * kHid + ct * 16 + ar;
                        *q = wv == 0 ? acc[ft][ct][j] : *q + acc[ft][ct][j];
                    }
            if (kq < 2) {
                float* q = s_sum + K * kHid + kq * 16 + ar;
                const float v = kq == 0 ? db[0] : db[1];
                *q = wv == 0 ? v : *q + v;
            }
        }
        __syncthreads();
    }
    float* out = part + static_cast<long>(blockIdx.x) * LEN;
    for (int k = threadIdx.x; k < LEN; k += 256) out[k] = s_sum[k];
}

// out[j] = sum over parts: kSumSplit threads per j each add a contiguous
// share of the parts in order, then their sums are added in order.
constexpr int kSumSplit = 16;
__global__ __launch_bounds__(256) void k_sum_parts(int nparts, int len, const float* __restrict__ part,
                                                   float* __restrict__ out) {
    constexpr int J = 256 / kSumSplit;
    __shared__ float s_sum[kSumSplit][J];
    const int jl = threadIdx.x % J, sp = threadIdx.x / J;
    const int j = blockIdx.x * J + jl;
    const int share = (nparts + kSumSplit - 1) / kSumSplit;
    float s = 0.f;
    if (j < len)
        for (int p = sp * share; p < min(nparts, (sp + 1) * share); ++p) s += part[static_cast<long>(p) * len + j];
    s_sum[sp][jl] = s;
    __syncthreads();
    if (sp == 0 && j < len) {
        for (int k = 1; k < kSumSplit; ++k) s += s_sum[k][jl];
        out[j] = s;
    }
}

// MSE loss head backward; per-block partials of (dwo[32], dbo, loss).
__global__ __launch_bounds__(256) void k_head_bwd(int n, const float* __restrict__ h3, const float* __restrict__ omega,
                                                  const float* __restrict__ target, const float* __restrict__ prm,
                                                  float* __restrict__ dh3, float* __restrict__ part) {
    __shared__ float s[256][kHid + 2];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    float du = 0.f, l = 0.f;
    if (i < n) {
        const float w = omega[i];
        const float diff = w - target[i];
        du = 2.f / n * diff * w * (1.f - w);
        l = diff * diff / n;
        for (int d = 0; d < kHid; ++d) dh3[static_cast<long>(i) * kHid + d] = du * prm[kOffWo + d];
    }
    for (int d = 0; d < kHid; ++d) s[threadIdx.x][d] = i < n ? du * h3[static_cast<long>(i) * kHid + d] : 0.f;
    s[threadIdx.x][kHid] = du;
    s[threadIdx.x][kHid + 1] = l;
    __syncthreads();
    if (threadIdx.x < kHid + 2) {
        float t = 0.f;
        for (int r = 0; r < 256; ++r) t += s[r][threadIdx.x];
        part[static_cast<long>(blockIdx.x) * (kHid + 2) + threadIdx.x] = t;
    }
}

__global__ void k_adam(int np, float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m1,
                       float* __restrict__ m2, float lr, float b1, float b2, float eps, float c1, float c2) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= np) return;
    const float gj = g[j];
    const float a = b1 * m1[j] + (1.f - b1) * gj;
    const float v = b2 * m2[j] + (1.f - b2) * gj * gj;
    m1[j] = a;
    m2[j] = v;
    p[j] -= lr * (a / c1) / (sqrtf(v / c2) + eps);
}

__global__ void k_to_bf16(int count, const float* __restrict__ src, unsigned short* __restrict__ dst) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < count) dst[j] = f2bf(src[j]);
}

__global__ void k_gather_f(long count, const int* __restrict__ idx, const float* __restrict__ src,
                           float* __restrict__ dst) {
    const long j = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
    if (j < count) dst[j] = src[idx[j]];
}

}  // namespace gnn

class GnnModel {
public:
    GnnModel() {
        params_.resize(gnn::kParams);
        grads_.resize(gnn::kParams + 1);  // and the loss
        m1_.resize(gnn::kParams);
        m2_.resize(gnn::kParams);
        wb_.resize(gnn::kParams);
        PILU_HIP(hipMemset(m1_.get(), 0, sizeof(float) * gnn::kParams));
        PILU_HIP(hipMemset(m2_.get(), 0, sizeof(float) * gnn::kParams));
        // Glorot-style deterministic initialisation (splitmix sequence).
        std::vector<float> h(gnn::kParams, 0.f);
        uint64_t st = 0x9E3779B97F4A7C15ull;
        auto rnd = [&]() {
            st += 0x9E3779B97F4A7C15ull;
            uint64_t x = st;
            x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
            x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
            x ^= x >> 31;
            return static_cast<double>(x >> 11) * (1.0 / 9007199254740992.0) * 2.0 - 1.0;
        };
        for (int l = 0; l < gnn::kLayers; ++l) {
            const int k = 2 * gnn::kInDim[l];
            const double a = std::sqrt(6.0 / (k + gnn::kHid));
            for (int j = 0; j < k * gnn::kHid; ++j) h[gnn::kOffW[l] + j] = static_cast<float>(a * rnd());
        }
        const double ao = std::sqrt(6.0 / (gnn::kHid + 1));
        for (int j = 0; j < gnn::kHid; ++j) h[gnn::kOffWo + j] = static_cast<float>(ao * rnd());
        set_params(h.data());
    }

    void set_params(const float* host) {
        PILU_HIP(hipMemcpy(params_.get(), host, sizeof(float) * gnn::kParams, hipMemcpyHostToDevice));
        refresh_bf16();
    }
    void get_params(float* host) const {
        PILU_HIP(hipMemcpy(host, params_.get(), sizeof(float) * gnn::kParams, hipMemcpyDeviceToHost));
    }
    void get_grads(float* host) const {
        PILU_HIP(hipMemcpy(host, grads_.get(), sizeof(float) * gnn::kParams, hipMemcpyDeviceToHost));
    }

    // Forward pass; omega (device, n floats) receives the predictions.  train
    // also keeps what the backward pass reads.
    void forward(int n, const int* rp, const int* ci, const double* va, float* omega, bool train = false) {
        prepare(n, rp, ci, va, train);
        // k_layer reads an entry for rows that have none (and leaves it out): where
        // there is no entry at all, the caller's columns may be null
        const int* cols = ci;
        if (nnz_ == 0) {
            if (no_cols_.size() == 0) {
                no_cols_.resize(1);
                PILU_HIP(hipMemset(no_cols_.get(), 0, sizeof(int)));
            }
            cols = no_cols_.get();
        }
        // a multiple of the 8 XCDs, at most 8 workgroups per CU
        const int grid = std::min((ceil_div(n, 64) + 7) / 8 * 8, 2048);
        auto run = [&](auto kern, int l) {
            const float* hin = l == 0 ? feat_.get() : h_[l - 1].get();
            kern<<<grid, 256>>>(n, rp, cols, ew_.get(), hin, wb_.get() + gnn::kOffW[l], params_.get() + gnn::kOffB[l],
                                h_[l].get(), m_[l].get(), params_.get(), omega);
        };
        if (train) {
            run(gnn::k_layer<gnn::kFeat, true, false>, 0);
            run(gnn::k_layer<gnn::kHid, true, false>, 1);
            run(gnn::k_layer<gnn::kHid, true, true>, 2);
        } else {
            run(gnn::k_layer<gnn::kFeat, false, false>, 0);
            run(gnn::k_layer<gnn::kHid, false, false>, 1);
            run(gnn::k_layer<gnn::kHid, false, true>, 2);
        }
        PILU_HIP(hipGetLastError());
    }

    // Gradients of the MSE loss (into grads_); returns the loss.
    double backward(int n, const int* rp, const int* ci, const double* va, const int* rpt, const int* cit,
                    const int* tmap, const float* target) {
        omega_.reserve(n);
        forward(n, rp, ci, va, omega_.get(), true);
        ewt_.reserve(std::max<long>(nnz_, 1));
        gnn::k_gather_f<<<ceil_div(nnz_, 256), 256>>>(nnz_, tmap, ew_.get(), ewt_.get());
        // the partials' sums go straight to their places in grads_ (a layer's
        // weights and bias, and the head's, are neighbours there)
        auto sum = [](int parts, int len, const float* part, float* out) {
            constexpr int per = 256 / gnn::kSumSplit;
            gnn::k_sum_parts<<<ceil_div(len, per), 256>>>(parts, len, part, out);
        };
        // head
        const int hb = ceil_div(n, 256);
        part_.reserve(static_cast<size_t>(hb) * (gnn::kHid + 2));
        gnn::k_head_bwd<<<hb, 256>>>(n, h_[2].get(), omega_.get(), target, params_.get(), dh_.get(), part_.get());
        sum(hb, gnn::kHid + 2, part_.get(), grads_.get() + gnn::kOffWo);  // wo, bo and, past the gradients, the loss
        // layers, last to first; dh_ holds dL/dH_{l+1}
        const int wgs16 = ceil_div(n, 64);
        const int wgrad = std::min(wgs16, gnn::kWgradBlocks);
        for (int l = gnn::kLayers - 1; l >= 0; --l) {
            const int D = gnn::kInDim[l];
            const float* hin = l == 0 ? feat_.get() : h_[l - 1].get();
            const int len = 2 * D * gnn::kHid + gnn::kHid;
            wpart_.reserve(static_cast<size_t>(wgrad) * len);
            auto bwd_w = D == gnn::kFeat ? gnn::k_dense_bwd_w<gnn::kFeat> : gnn::k_dense_bwd_w<gnn::kHid>;
            bwd_w<<<wgrad, 256>>>(n, hin, m_[l].get(), dh_.get(), h_[l].get(), wpart_.get());
            sum(wgrad, len, wpart_.get(), grads_.get() + gnn::kOffW[l]);
            if (l == 0) break;
            // dH_l = dX[:, :D] + W_graph^T dX[:, D:]
            gnn::k_dense_bwd_x<gnn::kHid><<<wgs16, 256>>>(n, dh_.get(), h_[l].get(), wb_.get() + gnn::kOffW[l],
                                                          dh2_.get(), dm_.get());
            gnn::k_aggregate<gnn::kHid><<<ceil_div(n, 32), 256>>>(n, rpt, cit, ewt_.get(), dm_.get(), dh2_.get());
            std::swap(dh_, dh2_);
        }
        PILU_HIP(hipGetLastError());
        float loss = 0.f;
        PILU_HIP(hipMemcpy(&loss, grads_.get() + gnn::kParams, sizeof(float), hipMemcpyDeviceToHost));
        return loss;
    }

    double train_step(int n, const int* rp, const int* ci, const double* va, const int* rpt, const int* cit,
                      const int* tmap, const float* target, float lr) {
        const double loss = backward(n, rp, ci, va, rpt, cit, tmap, target);
        ++step_;
        const float b1 = 0.9f, b2 = 0.999f;
        const float c1 = 1.f - std::pow(b1, static_cast<float>(step_));
        const float c2 = 1.f - std::pow(b2, static_cast<float>(step_));
        gnn::k_adam<<<ceil_div(gnn::kParams, 256), 256>>>(gnn::kParams, params_.get(), grads_.get(), m1_.get(),
                                                         m2_.get(), lr, b1, b2, 1e-8f, c1, c2);
        refresh_bf16();
        PILU_HIP(hipDeviceSynchronize());
        return loss;
    }

private:
    static long host_nnz(const int* d_rp, int n) {
        int v = 0;
        PILU_HIP(hipMemcpy(&v, d_rp + n, sizeof(int), hipMemcpyDeviceToHost));
        return v;
    }

    void refresh_bf16() {
        gnn::k_to_bf16<<<ceil_div(gnn::kParams, 256), 256>>>(gnn::kParams, params_.get(), wb_.get());
        PILU_HIP(hipGetLastError());
    }

    void prepare(int n, const int* rp, const int* ci, const double* va, bool train) {
        nnz_ = host_nnz(rp, n);
        const long nnz = nnz_;
        const long nr = static_cast<long>(ceil_div(n, 64)) * 64;  // room for whole 16-row tiles
        dg_.reserve(n);
        feat_.reserve(nr * gnn::kFeat);
        ew_.reserve(std::max<long>(nnz, 1));
        for (int l = 0; l < gnn::kLayers; ++l)
            if (train || l + 1 < gnn::kLayers) h_[l].reserve(nr * gnn::kHid);
        if (train) {
            for (int l = 0; l < gnn::kLayers; ++l) m_[l].reserve(nr * gnn::kInDim[l]);
            dh_.reserve(nr * gnn::kHid);
            dh2_.reserve(nr * gnn::kHid);
            dm_.reserve(nr * gnn::kHid);
        }
        gnn::k_diag_values<<<ceil_div(n, 256), 256>>>(n, rp, ci, va, dg_.get());
        gnn::k_features<<<ceil_div(n, gnn::kFeatRows), gnn::kFeatRows>>>(n, rp, ci, va, dg_.get(), feat_.get(), ew_.get());
    }

    DevBuf<float> params_, grads_, m1_, m2_, feat_, ew_, ewt_, m_[gnn::kLayers], h_[gnn::kLayers], dh_, dh2_,
        dm_, part_, wpart_, omega_;
    long nnz_ = 0;
    DevBuf<unsigned short> wb_;
    DevBuf<double> dg_;
    DevBuf<int> no_cols_;
    long step_ = 0;
};

}  // namespace pilu

namespace {
template <typename F>
int gguard(const char* what, F&& f) {
    try {
        return f();
    } catch (const std::exception& e) {
        std::fprintf(stderr, "%s: %s\n", what, e.what());
        return -1;
    }
}
pilu::GnnModel* Gm(GnnHdl h) { return static_cast<pilu::GnnModel*>(h); }
}  // namespace

extern "C" {

GnnHdl GnnCreateEx(void) {
    try {
        return new pilu::GnnModel;
    } catch (const std::exception& e) {
        std::fprintf(stderr, "GnnCreate: %s\n", e.what());
        return nullptr;
    }
}

void GnnDestroyEx(GnnHdl h) { delete Gm(h); }

int GnnParameterCountEx(void) { return pilu::gnn::kParams; }

int GnnSetParametersEx(GnnHdl h, const float* host) {
    return gguard("GnnSetParameters", [&] { Gm(h)->set_params(host); return 0; });
}

int GnnGetParametersEx(GnnHdl h, float* host) {
    return gguard("GnnGetParameters", [&] { Gm(h)->get_params(host); return 0; });
}

int GnnPredictEx(GnnHdl h, const CsrMatrix* d_a, float* d_omega) {
    return gguard("GnnPredict", [&] {
        Gm(h)->forward(d_a->size, d_a->row_ptr, d_a->col_idx, d_a->value, d_omega);
        PILU_HIP(hipDeviceSynchronize());
        return 0;
    });
}

int GnnGradientsEx(GnnHdl h, const CsrMatrix* d_a, const CsrMatrix* d_at, const int* d_tmap, const float* d_target,
                   float* host_grads, double* loss) {
    return gguard("GnnGradients", [&] {
        const double l = Gm(h)->backward(d_a->size, d_a->row_ptr, d_a->col_idx, d_a->value, d_at->row_ptr,
                                         d_at->col_idx, d_tmap, d_target);
        if (loss) *loss = l;
        if (host_grads) Gm(h)->get_grads(host_grads);
        return 0;
    });
}

int GnnTrainStepEx(GnnHdl h, const CsrMatrix* d_a, const CsrMatrix* d_at, const int* d_tmap, const float* d_target,
                   float lr, double* loss) {
    return gguard("GnnTrainStep", [&] {
        const double l = Gm(h)->train_step(d_a->size, d_a->row_ptr, d_a->col_idx, d_a->value, d_at->row_ptr,
                                           d_at->col_idx, d_tmap, d_target, lr);
        if (loss) *loss = l;
        return 0;
    });
}

bool GmresSolveLearnedDeviceEx(GmresHdl gmres, IluSolverHdl ilu, GnnHdl gnn, const CsrMatrix* d_a,
                               const double* d_rhs, double* d_sol, int budget, int* iter, int* fallback) {
    auto* g = static_cast<lljbash::PreconditionedGmres*>(gmres);
    auto* s = static_cast<lljbash::IluSolver*>(ilu);
    if (fallback) *fallback = 0;
    if (iter) *iter = 0;
    try {
        const int n = d_a->size;
        pilu::DevBuf<float> omega(n);
        pilu::DevBuf<double> x0(n);
        PILU_HIP(hipMemcpy(x0.get(), d_sol, sizeof(double) * n, hipMemcpyDeviceToDevice));
        Gm(gnn)->forward(n, d_a->row_ptr, d_a->col_idx, d_a->value, omega.get());
        s->SetDiagonalCompensation(omega.get());
        bool fok = s->FactorizeDeviceFromA(d_a->value);
        s->SetDiagonalCompensation(nullptr);
        std::pair<bool, int> r{false, 0};
        if (fok) r = g->SolveDevice(d_a, d_rhs, d_sol);
        if (!fok || !r.first || r.second > budget) {
            PILU_HIP(hipMemcpy(d_sol, x0.get(), sizeof(double) * n, hipMemcpyDeviceToDevice));
            s->FactorizeDeviceFromA(d_a->value);
            r = g->SolveDevice(d_a, d_rhs, d_sol);
            if (fallback) *fallback = 1;
        }
        if (iter) *iter = r.second;
        return r.first;
    } catch (const std::exception& e) {
        s->SetDiagonalCompensation(nullptr);
        std::fprintf(stderr, "GmresSolveLearnedDevice: %s\n", e.what());
        return false;
    }
}

}  // extern "C"
