// k-nearest neighbours for k > 1 (up to 64) in L1/L2 spaces: a block of W
// waves serves Q queries.  Lanes take consecutive tree nodes, every wave
// keeps each query's k best as a wave list (one entry per lane,
// wave_list.hpp), and the W waves' lists meet in LDS.
//
// What bounds it: the lists.  A lane that keeps a k-list of its own needs
// 5 k registers and inserts by moving all of them, and merging such lists
// over S chunks of the tree is one lane walking S k entries: on 5 000 nodes
// of R^2 with 1 024 queries and k = 45 that took 315 + 5 010 us (scan +
// merge; 8 waves per SIMD in the grid, 2 resident).  With the list spread
// over the wave an insert is 12 VALU instructions, lists need no memory until
// the end, and a wave's expected inserts are k (1 + ln(n / (W k))).
//
// Reading the tree: the FP32 shadow rows (contiguous 16-byte loads of
// consecutive lanes) with the proven FP32 bound of knn_bound.hpp in front of the
// exact distance; in up to 2 dimensions an FP64 row is one 16-byte load and
// the distance cheaper than a bound, so the exact distance is taken at once.
// The next rows are loaded before the present ones are used.  A row is
// tested against Q queries: at Q = 1 the loads, not the arithmetic, set the
// pace once there are enough queries to fill the chip.
#include <algorithm>
#include <climits>
#include <cmath>
#include <limits>

#include "knn_bound.hpp"
#include "wave_list.hpp"

namespace mptg {
namespace {

// A node's row as the scan reads it: FP64 coordinates (direct) or the FP32
// shadow, DP floats.
template <int D>
struct ScanRow {
    static constexpr bool kDirect = D <= 2;
    static constexpr int DP = (D <= 2) ? 2 : (D <= 4 ? 4 : (D <= 8 ? 8 : ((D + 3) / 4) * 4));
    using T = std::conditional_t<kDirect, double, float>;
    T v[kDirect ? D : DP];
    __device__ __forceinline__ void load(const double* __restrict__ x64, const float* __restrict__ x32, int64_t p) {
        if constexpr (kDirect) {
#pragma unroll
            for (int i = 0; i < D; ++i) v[i] = x64[p * D + i];
        } else {
#pragma unroll
            for (int i = 0; i < DP; i += 4) {
                const float4 f = *reinterpret_cast<const float4*>(x32 + p * DP + i);
                v[i] = f.x;
                v[i + 1] = f.y;
                v[i + 2] = f.z;
                v[i + 3] = f.w;
            }
        }
    }
};

template <int D, int METRIC, int W, int Q>
__global__ __launch_bounds__(64 * W) void knn_wave(const float* __restrict__ x32, const double* __restrict__ x64,
                                                   int64_t n, const double* __restrict__ q, int64_t nq, int k,
                                                   double radius, double pbound, double inf,
                                                   double* __restrict__ out_d, int32_t* __restrict__ out_i) {
    using Row = ScanRow<D>;
    constexpr bool kDirect = Row::kDirect;
    using T = typename Row::T;
    __shared__ double sd[W > 1 ? W * kWaveListMax : 1];
    __shared__ int32_t si[W > 1 ? W * kWaveListMax : 1];
    const int lane = threadIdx.x & 63;
    const int w = W > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
    const int64_t q0 = (int64_t)blockIdx.x * Q;
    T qv[Q][D];
    double S[Q];
    WaveList wl[Q];
    T thr[Q];  // rows beyond it cannot enter the list: squared sums (L2) or sums (L1)
    auto threshold = [&](int u) -> T {
        const double t = __builtin_fmin(wl[u].kd, radius);
        if constexpr (!kDirect) return prefilter_threshold<D, METRIC>(t, S[u]);
        else if constexpr (METRIC == MPTG_METRIC_L1) return t;
        // sqrt(s) <= t implies s <= t^2 (1 + 2^-51); tiny t: no test
        else return t < 1e-140 ? inf : t * t * (1.0 + 0x1.0p-40);
    };
#pragma unroll
    for (int u = 0; u < Q; ++u) {
        const int64_t qi = q0 + u < nq ? q0 + u : nq - 1;  // a short last block repeats a query
        double m = 0.0;
#pragma unroll
        for (int i = 0; i < D; ++i) {
            const double x = q[qi * D + i];
            qv[u][i] = (T)x;
            m = __builtin_fmax(m, __builtin_fabs(x));
        }
        S[u] = m + pbound;
        wl[u].init(k, inf);
        thr[u] = threshold(u);
    }
    const int64_t step = 64 * W;
    Row row;
    int64_t p = (int64_t)w * 64 + lane;
    if (p < n) row.load(x64, x32, p);
    for (int64_t base = (int64_t)w * 64; base < n; base += step, p += step) {
        const Row cur = row;
        if (p + step < n) row.load(x64, x32, p + step);
        const bool in = p < n;
#pragma unroll
        for (int u = 0; u < Q; ++u) {
            T s = 0;
#pragma unroll
            for (int i = 0; i < D; ++i) {
                const T t = qv[u][i] - cur.v[i];
                if constexpr (METRIC == MPTG_METRIC_L1) s = s + __builtin_elementwise_abs(t);
                else if constexpr (kDirect) s = s + t * t;
                else s = __builtin_fmaf(t, t, s);
            }
            bool pass = in && s <= thr[u];
            if (__ballot(pass)) {
                double dq = 0.0;
                if (pass) {
                    if constexpr (!kDirect) dq = exact_dist<D, METRIC>(q + (q0 + u < nq ? q0 + u : nq - 1) * D, x64 + p * D);
                    else if constexpr (METRIC == MPTG_METRIC_L1) dq = s;
                    else dq = __builtin_sqrt(s);
                    pass = dq <= radius && wl_before(dq, (int32_t)p, wl[u].kd, wl[u].ki);
                }
                if (__ballot(pass)) {
                    wl[u].offer(pass, dq, (int32_t)p, lane);
                    thr[u] = threshold(u);
                }
            }
        }
    }
#pragma unroll
    for (int u = 0; u < Q; ++u) {
        const int64_t qi = q0 + u;
        if (qi >= nq) break;  // block-uniform
        if constexpr (W == 1) {
            if (lane < k) {
                const bool have = wl[u].li != INT_MAX;
                out_d[qi * k + lane] = have ? wl[u].ld : inf;
                out_i[qi * k + lane] = have ? wl[u].li : -1;
            }
        } else {
            // an entry's rank among the W sorted lists -- (distance, id) keys
            // are distinct, empty entries sort last -- is its output position
            if (u > 0) __syncthreads();
            sd[w * kWaveListMax + lane] = wl[u].ld;
            si[w * kWaveListMax + lane] = wl[u].li;
            __syncthreads();
            int rank = lane;
            const bool real = lane < k && wl[u].li != INT_MAX;
            int total = 0;
#pragma unroll
            for (int v = 0; v < W; ++v) {
                // entries of wave v before this one: its list is sorted, k long
                int lo = 0, hi = k;
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (wl_before(sd[v * kWaveListMax + mid], si[v * kWaveListMax + mid], wl[u].ld, wl[u].li)) lo = mid + 1;
                    else hi = mid;
                }
                if (v != w) rank += lo;
                total += __popcll(__ballot(lane < k && si[v * kWaveListMax + lane] != INT_MAX));
            }
            if (real && rank < k) {
                out_d[qi * k + rank] = wl[u].ld;
                out_i[qi * k + rank] = wl[u].li;
            }
            if (w == 0 && lane < k && lane >= total) {
                out_d[qi * k + lane] = inf;
                out_i[qi * k + lane] = -1;
            }
        }
    }
}

template <int D, int METRIC>
void launch_wave(mptg_ctx* ctx, int W, int Q, int64_t n, const double* q, int64_t nq, int k, double radius,
                 double* out_d, int32_t* out_i) {
    const double inf = std::numeric_limits<double>::infinity();
#define MPTG_KNN_WAVE(WW, QQ)                                                                                       \
    hipLaunchKernelGGL((knn_wave<D, METRIC, WW, QQ>), dim3((unsigned)((nq + QQ - 1) / QQ)), dim3(64 * WW), 0,       \
                       ctx->stream, (const float*)ctx->x32, (const double*)ctx->x64, n, q, nq, k, radius,           \
                       ctx->coord_bound, inf, out_d, out_i)
    if constexpr (D <= 8) {
        if (Q == 4) {
            MPTG_KNN_WAVE(1, 4);
            return;
        }
    }
    if (W == 1) MPTG_KNN_WAVE(1, 1);
    else if (W == 4) MPTG_KNN_WAVE(4, 1);
    else MPTG_KNN_WAVE(16, 1);
#undef MPTG_KNN_WAVE
}

}  // namespace

bool knn_wave_dim_ok(int dim) { return (dim >= 1 && dim <= 8) || dim == 10 || dim == 12 || dim == 16 || dim == 20; }

int knn_wave_path(mptg_ctx* ctx, const double* d_q, int64_t nq, int k, double radius, int32_t* d_idx,
                  double* d_dist, int64_t n) {
    if (k < 1 || k > kWaveListMax) return fail(ctx, MPTG_E_RANGE, "k must be 1..64");
    if (!knn_wave_dim_ok(ctx->dim)) return fail(ctx, MPTG_E_ARG, "unsupported dimension for the nearest-neighbour kernel");
    if (nq >= ((int64_t)1 << 31)) return fail(ctx, MPTG_E_RANGE, "at most 2^31 - 1 queries");
    if (nq == 0) return MPTG_OK;
    // waves per query: about 8 waves per SIMD in all, and at least 4 rounds
    // of 64 nodes per wave (below that the merge of the lists costs more than
    // the split saves); queries per wave: 4 once the queries alone fill the
    // chip four times over.  Sixteen waves is the most: one query over 10^6
    // nodes keeps one CU busy for 0.57 ms (R^12, k = 20) to 1.3 (R^20, L1, k =
    // 48), where the k-list scan spread over the chip took 2.4 and 7.4 for its
    // lists' merge; at 256 queries it is 0.58 against 6.4 and 1.4 against 40.
    const int64_t fill = (int64_t)ctx->cus * 32, rounds = (n + 63) / 64;
    const int Q = ctx->dim <= 8 && nq >= 4 * fill ? 4 : 1;
    int W = 1;
    while (W < 16 && 4 * W * nq <= fill * 2 && 16 * W <= rounds) W *= 4;
    auto go = [&]<int D>() {
        if (ctx->metric == MPTG_METRIC_L1) launch_wave<D, MPTG_METRIC_L1>(ctx, W, Q, n, d_q, nq, k, radius, d_dist, d_idx);
        else launch_wave<D, MPTG_METRIC_L2>(ctx, W, Q, n, d_q, nq, k, radius, d_dist, d_idx);
    };
    switch (ctx->dim) {
        case 1: go.template operator()<1>(); break;
        case 2: go.template operator()<2>(); break;
        case 3: go.template operator()<3>(); break;
        case 4: go.template operator()<4>(); break;
        case 5: go.template operator()<5>(); break;
        case 6: go.template operator()<6>(); break;
        case 7: go.template operator()<7>(); break;
        case 8: go.template operator()<8>(); break;
        case 10: go.template operator()<10>(); break;
        case 12: go.template operator()<12>(); break;
        case 16: go.template operator()<16>(); break;
        default: go.template operator()<20>(); break;
    }
    MPTG_HIP(ctx, hipGetLastError());
    return MPTG_OK;
}

}  // namespace mptg
