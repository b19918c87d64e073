// The nearest neighbour (k = 1) in L1/L2 spaces of up to 8 dimensions: a block
// of four waves serves Q queries, its lanes take consecutive tree nodes.
//
// What bounds it: instruction issue, 2 D + 4 vector instructions per pair of a
// query and a node.  The queries' coordinates sit in scalar registers, a row is
// read once for Q of them, and a lane keeps, per query, the smallest FP32 value,
// whose node it was, and the second smallest: no branch, no list.  The
// smallest value of the block gives the threshold below which the exact nearest
// must lie (knn_bound.hpp); a lane whose own smallest is under it measures that
// node exactly.  Where a lane's second smallest is under it too (nodes on a
// small circle seen from afar, as a tree of limited range begins, or a goal
// sampled often), one more pass over the rows lists those queries' pairs, and
// the block measures the list; past the list's end each lane measures its rows'
// pairs as it meets them (a query at a time over all rows, 8192 queries and
// 3000 nodes at 8 points took 176 us, 72 now; 66 in the scan).  (A lane per query over broadcast rows, chunk by
// chunk of the tree, took a list, a branch per four nodes, a seed bound and a
// merge, three launches: 256 queries and 2000 nodes of R^2 19.7 us then, 5.2
// now; 8192 and 16 000 93 and 39; 65 536 and 65 000 1050 and 800.)
#include <algorithm>
#include <climits>
#include <cmath>
#include <limits>

#include "knn_bound.hpp"
#include "wave_ops.hpp"

namespace mptg {
namespace {

constexpr int kOneBlock = 256, kOneWaves = kOneBlock / 64;
constexpr int kOneCand = 4096;

template <int D, int METRIC>
__device__ __forceinline__ float one_value(const float* q, const float* row) {
    float a = 0.0f;
#pragma unroll
    for (int i = 0; i < D; ++i) {
        const float t = q[i] - row[i];
        if constexpr (METRIC == MPTG_METRIC_L1) a = a + __builtin_fabsf(t);
        else a = __builtin_fmaf(t, t, a);
    }
    return a;
}

template <int D>
struct OneRow {
    static constexpr int DP = D <= 2 ? 2 : D <= 4 ? 4 : 8;
    float v[DP];
    __device__ __forceinline__ void load(const float* __restrict__ x32, int64_t j) {
        if constexpr (DP == 2) {
            const float2 a = *(const float2*)(x32 + j * 2);
            v[0] = a.x;
            v[1] = a.y;
        } else {
#pragma unroll
            for (int k = 0; k < DP; k += 4) {
                const float4 a = *(const float4*)(x32 + j * DP + k);
                v[k] = a.x;
                v[k + 1] = a.y;
                v[k + 2] = a.z;
                v[k + 3] = a.w;
            }
        }
    }
};

__device__ __forceinline__ bool one_better(double d, int32_t i, double bd, int32_t bi) {
    return d < bd || (d == bd && i < bi);
}

template <int D, int METRIC, int Q>
__global__ __launch_bounds__(kOneBlock) void knn_one(const double* __restrict__ x64, const float* __restrict__ x32,
                                                     int64_t n, const double* __restrict__ q, int64_t nq,
                                                     double radius, double pbound, double inf,
                                                     double* __restrict__ out_d, int32_t* __restrict__ out_i,
                                                     const int64_t* n_dev, const int32_t* skip,
                                                     const uint32_t* nq_dev) {
    __shared__ float min_s[kOneWaves][Q], thr_s[Q];
    __shared__ double best_d[kOneWaves][Q];
    __shared__ int32_t best_i[kOneWaves][Q];
    // pairs under the threshold of queries that a lane has two or more of
    __shared__ uint32_t cand_j[kOneCand];
    __shared__ uint8_t cand_c[kOneCand];
    __shared__ unsigned long long near_d[Q];
    __shared__ int near_i[Q], ncand;
    __shared__ uint32_t crowd_s;  // those queries, a bit each
    if (skip && *skip) return;  // block-uniform
    if (n_dev) n = *n_dev;
    const int64_t live = nq_dev ? (int64_t)*nq_dev : nq;
    const int64_t q0 = (int64_t)blockIdx.x * Q;
    if (q0 >= live) return;  // block-uniform
    const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
    float qv[Q][D];
#pragma unroll
    for (int c = 0; c < Q; ++c) {
        const int64_t qi = q0 + c < live ? q0 + c : live - 1;
#pragma unroll
        for (int i = 0; i < D; ++i)
            qv[c][i] = __uint_as_float(
                (uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint((float)q[qi * D + i])));
    }
    const float finf = __builtin_inff();
    float low[Q], second[Q];
    int32_t at[Q];
#pragma unroll
    for (int c = 0; c < Q; ++c) {
        low[c] = second[c] = finf;
        at[c] = -1;
    }
    constexpr int U = Q >= 8 ? 2 : 4;  // rows in flight
    for (int64_t j0 = 0; j0 < n; j0 += kOneBlock * U) {
        OneRow<D> row[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t j = j0 + u * kOneBlock + t;
            if (j < n) {
                row[u].load(x32, j);
            } else {
#pragma unroll
                for (int i = 0; i < D; ++i) row[u].v[i] = finf;  // value +inf: never the smallest
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int32_t j = (int32_t)(j0 + u * kOneBlock) + t;
#pragma unroll
            for (int c = 0; c < Q; ++c) {
                const float a = one_value<D, METRIC>(qv[c], row[u].v);
                at[c] = a < low[c] ? j : at[c];
                second[c] = __builtin_amdgcn_fmed3f(a, low[c], second[c]);
                low[c] = __builtin_fminf(a, low[c]);
            }
        }
    }
#pragma unroll
    for (int c = 0; c < Q; ++c) {
        const float m = wave_min_f32(low[c]);
        if (lane == 0) min_s[wid][c] = m;
    }
    __syncthreads();
    if (t < Q) {
        const int64_t qi = q0 + t < live ? q0 + t : live - 1;
        double mq = 0.0;
        for (int i = 0; i < D; ++i) mq = __builtin_fmax(mq, __builtin_fabs(q[qi * D + i]));
        const double S = mq + pbound;
        float m = min_s[0][t];
        for (int w = 1; w < kOneWaves; ++w) m = __builtin_fminf(m, min_s[w][t]);
        float thr = prefilter_threshold<D, METRIC>(radius, S);
        if (m < finf) thr = __builtin_fminf(thr, prefilter_threshold<D, METRIC>(prefilter_upper<D, METRIC>(m, S), S));
        thr_s[t] = thr;
        near_d[t] = bits_of(inf);
        near_i[t] = INT_MAX;
    }
    if (t == 0) {
        ncand = 0;
        crowd_s = 0;
    }
    __syncthreads();
    uint32_t crowd = 0;
#pragma unroll
    for (int c = 0; c < Q; ++c) crowd |= (second[c] <= thr_s[c] ? 1u : 0u) << c;
    if (crowd) atomicOr(&crowd_s, crowd);
    __syncthreads();
    crowd = (uint32_t)__builtin_amdgcn_readfirstlane((int)crowd_s);
    bool listed = false;  // the crowded queries have their nearest in near_d, near_i
    if (crowd) {
        // one more pass over the rows lists those queries' pairs
        float lim[Q];
#pragma unroll
        for (int c = 0; c < Q; ++c)
            lim[c] = (crowd >> c) & 1u
                         ? __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(thr_s[c])))
                         : -1.0f;
        for (int64_t j0 = 0; j0 < n; j0 += kOneBlock * U) {
            if (__builtin_amdgcn_readfirstlane(
                    __hip_atomic_load(&ncand, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) > kOneCand)
                break;  // too many already
            OneRow<D> row[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t j = j0 + u * kOneBlock + t;
                row[u].load(x32, j < n ? j : 0);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t j = j0 + u * kOneBlock + t;
                uint32_t in = 0;
#pragma unroll
                for (int c = 0; c < Q; ++c) in |= (one_value<D, METRIC>(qv[c], row[u].v) <= lim[c] ? 1u : 0u) << c;
                if (j >= n) in = 0;
                for (; in; in &= in - 1) {
                    const int slot = atomicAdd(&ncand, 1);
                    if (slot >= kOneCand) break;
                    cand_j[slot] = (uint32_t)j;
                    cand_c[slot] = (uint8_t)__builtin_ctz(in);
                }
            }
        }
        __syncthreads();
        const int found = ncand;
        listed = found <= kOneCand;
        if (listed) {
            auto exact = [&](int i) {
                return exact_dist<D, METRIC>(q + (q0 + cand_c[i]) * D, x64 + (int64_t)cand_j[i] * D);
            };
            for (int i = t; i < found; i += kOneBlock)
                if (q0 + cand_c[i] < live) {
                    const double d = exact(i);
                    if (d <= radius) atomicMin(&near_d[cand_c[i]], (unsigned long long)bits_of(d));
                }
            __syncthreads();
            for (int i = t; i < found; i += kOneBlock)
                if (q0 + cand_c[i] < live) {
                    const double d = exact(i);
                    if (d <= radius && bits_of(d) == near_d[cand_c[i]]) atomicMin(&near_i[cand_c[i]], (int)cand_j[i]);
                }
        } else {
            // More pairs than the list holds (many nodes at one place): a
            // lane measures the pairs of its rows as it meets them.  Its rows
            // come by ascending id, so none past a node at the query itself.
            double bd[Q];
            int32_t bi[Q];
#pragma unroll
            for (int c = 0; c < Q; ++c) {
                bd[c] = inf;
                bi[c] = INT_MAX;
            }
            uint32_t open = crowd;
            constexpr int R = Q == 1 ? 4 : Q == 4 ? 2 : 1;  // rows in flight
            for (int64_t j0 = t; j0 < n && open; j0 += kOneBlock * R) {
                OneRow<D> row[R];
                double x[R][D];
                uint32_t in[R];
#pragma unroll
                for (int u = 0; u < R; ++u) row[u].load(x32, j0 + u * kOneBlock < n ? j0 + u * kOneBlock : 0);
#pragma unroll
                for (int u = 0; u < R; ++u) {
                    in[u] = 0;
#pragma unroll
                    for (int c = 0; c < Q; ++c) in[u] |= (one_value<D, METRIC>(qv[c], row[u].v) <= lim[c] ? 1u : 0u) << c;
                    in[u] = j0 + u * kOneBlock < n ? in[u] & open : 0u;
                    if (in[u]) {
#pragma unroll
                        for (int i = 0; i < D; ++i) x[u][i] = x64[(j0 + u * kOneBlock) * D + i];
                    }
                }
#pragma unroll
                for (int u = 0; u < R; ++u) {
#pragma unroll
                    for (int c = 0; c < Q; ++c) {
                        if (!((in[u] & open) >> c & 1u)) continue;
                        const double d = exact_dist<D, METRIC>(q + (q0 + c < live ? q0 + c : live - 1) * D, x[u]);
                        const int32_t j = (int32_t)(j0 + u * kOneBlock);
                        if (d <= radius && one_better(d, j, bd[c], bi[c])) {  // (a distance may be infinite)
                            bd[c] = d;
                            bi[c] = j;
                            open &= ~((d == 0.0 ? 1u : 0u) << c);
                        }
                    }
                }
            }
#pragma unroll
            for (int c = 0; c < Q; ++c) {
                if (!((crowd >> c) & 1u)) continue;  // uniform
                double wd = bd[c];
                int32_t wi = bi[c];
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) {
                    const double d = __shfl_xor(wd, o);
                    const int32_t i = __shfl_xor(wi, o);
                    if (one_better(d, i, wd, wi)) {
                        wd = d;
                        wi = i;
                    }
                }
                if (lane == 0) {
                    best_d[wid][c] = wd;
                    best_i[wid][c] = wi;
                }
            }
        }
    }
#pragma unroll
    for (int c = 0; c < Q; ++c) {
        if ((crowd >> c) & 1u) continue;
        const float thr = thr_s[c];
        const double* qc = q + (q0 + c < live ? q0 + c : live - 1) * D;
        double bd = inf;
        int32_t bi = INT_MAX;
        if (low[c] <= thr) {  // (a threshold of +inf comes with a crowd)
            const double d = exact_dist<D, METRIC>(qc, x64 + (int64_t)at[c] * D);
            if (d <= radius) {
                bd = d;
                bi = at[c];
            }
        }
        // the wave's best, lane by lane: one lane has a node, nearly always
        double wd = inf;
        int32_t wi = INT_MAX;
        for (uint64_t m = __ballot(bi != INT_MAX); m; m &= m - 1) {
            const int src = __builtin_ctzll(m);
            const uint64_t b = bits_of(bd);
            const double d = double_of((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, src) |
                                       (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), src)
                                           << 32);
            const int32_t i = __builtin_amdgcn_readlane(bi, src);
            if (one_better(d, i, wd, wi)) {
                wd = d;
                wi = i;
            }
        }
        if (lane == 0) {
            best_d[wid][c] = wd;
            best_i[wid][c] = wi;
        }
    }
    __syncthreads();
    if (t < Q && q0 + t < live) {
        const bool mine = listed && ((crowd >> t) & 1u);
        double bd = mine ? double_of(near_d[t]) : best_d[0][t];
        int32_t bi = mine ? near_i[t] : best_i[0][t];
        for (int w = 1; w < kOneWaves && !mine; ++w)
            if (one_better(best_d[w][t], best_i[w][t], bd, bi)) {
                bd = best_d[w][t];
                bi = best_i[w][t];
            }
        out_d[q0 + t] = bi != INT_MAX ? bd : inf;
        out_i[q0 + t] = bi != INT_MAX ? bi : -1;
    }
}

template <int D, int METRIC, int Q>
void launch_one(mptg_ctx* ctx, const double* q, int64_t nq, double radius, double* out_d, int32_t* out_i, int64_t n,
                const int64_t* n_dev, const int32_t* skip, const uint32_t* nq_dev) {
    hipLaunchKernelGGL((knn_one<D, METRIC, Q>), dim3((unsigned)((nq + Q - 1) / Q)), dim3(kOneBlock), 0, ctx->stream,
                       ctx->x64, ctx->x32, n, q, nq, radius, ctx->coord_bound,
                       std::numeric_limits<double>::infinity(), out_d, out_i, n_dev, skip, nq_dev);
}

// Queries of a block once that leaves a block to every CU (coordinates and
// results in registers); fewer otherwise.
template <int D>
constexpr int one_queries() {
    return D <= 2 ? 16 : 8;
}

}  // namespace

// A block goes through the whole tree (0.45 us per 1000 nodes in two
// dimensions, 0.6 in seven), so few queries over a large tree take the scan,
// which splits it: at 65 000 nodes one query takes 24 us here and 36 there, at
// 10^6 450 and 101.  From 32 queries per CU on every block is resident, and
// the line depends on how much of a row it reads is padding, which the scan
// does not compare: in 2 to 4, 7 and 8 dimensions the scan gains on it slowly
// (8192 queries, L2: 0.24 ms there, 0.12 here in R^2 at 70 000, 1.72 and 1.57
// at 10^6; L1: 0.49 and 0.45 at 300 000, 1.28 and 1.43 at 10^6), with 5 or 6
// of 8 coordinates sooner (L2: 0.91 and 0.93 at 300 000; L1: 0.30 both at
// 100 000, 0.37 and 0.41 at 131 072), on the line too (0.20 and 0.14 ms at
// 100 000, 0.34 and 0.46 at 200 000).
// The byte prefilter of L1 in 8 dimensions (q8: the scan would use it) tests a
// pair in 2 instructions, not 20, behind two more launches: 8192 queries
// over 16 000 nodes 49 us, here 63; 1024 over 65 000 47 and 61; 16 384 over 500
// 21 and 26; but 2000 over 20 000 32 and 24, 256 over 65 000 78 and 34.  (Its
// bytes tell nothing apart in a tree that fills a thousandth of its box: 8192
// over 65 000 such nodes 1.4 ms, here 0.2.)
bool knn_one_applies(const mptg_ctx* ctx, int64_t nq, int64_t n, bool q8) {
    const bool l2 = ctx->metric == MPTG_METRIC_L2;
    if (ctx->dim < 1 || ctx->dim > 8 || (ctx->metric != MPTG_METRIC_L1 && !l2)) return false;
    if (nq <= 0 || nq >= ((int64_t)1 << 31)) return false;
    if (n <= (int64_t)1 << 16) return !(q8 && (nq >= (int64_t)ctx->cus * 64 || nq * n >= (int64_t)3 << 24));
    if (q8 || nq < (int64_t)ctx->cus * 32) return false;
    if (ctx->dim == 1) return n <= 100000;
    if (ctx->dim == 5 || ctx->dim == 6) return n <= (l2 ? (int64_t)1 << 18 : 100000);
    return n <= (l2 ? (int64_t)1 << 20 : (int64_t)1 << 19);
}

int knn_one_path(mptg_ctx* ctx, const double* d_q, int64_t nq, double radius, int32_t* d_idx, double* d_dist,
                 int64_t n, const int64_t* n_dev, const int32_t* skip, const uint32_t* nq_dev) {
    auto go = [&]<int D>() {
        constexpr int Q = one_queries<D>();
        auto metric = [&]<int M>() {
            if (nq >= (int64_t)ctx->cus * Q) launch_one<D, M, Q>(ctx, d_q, nq, radius, d_dist, d_idx, n, n_dev, skip, nq_dev);
            else if (nq >= (int64_t)ctx->cus * 4) launch_one<D, M, 4>(ctx, d_q, nq, radius, d_dist, d_idx, n, n_dev, skip, nq_dev);
            else launch_one<D, M, 1>(ctx, d_q, nq, radius, d_dist, d_idx, n, n_dev, skip, nq_dev);
        };
        if (ctx->metric == MPTG_METRIC_L1) metric.template operator()<MPTG_METRIC_L1>();
        else metric.template operator()<MPTG_METRIC_L2>();
    };
    switch (ctx->dim) {
        case 1: go.template operator()<1>(); break;
        case 2: go.template operator()<2>(); break;
        case 3: go.template operator()<3>(); break;
        case 4: go.template operator()<4>(); break;
        case 5: go.template operator()<5>(); break;
        case 6: go.template operator()<6>(); break;
        case 7: go.template operator()<7>(); break;
        default: go.template operator()<8>(); break;
    }
    MPTG_HIP(ctx, hipGetLastError());
    return MPTG_OK;
}

}  // namespace mptg
