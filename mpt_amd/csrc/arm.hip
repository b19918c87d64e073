// Planar-arm link() on the GPU: a kernel for every edge, and
// one for the few it leaves.
//
// Reference semantics (demo/link_manipulator_scenario.hpp:118-138): valid(a),
// valid(b), then the pre-order of recursive midpoints (a+b)/2 down to
// L-inf(a-b) < tol; the verdict is the AND over that fixed set, the check
// count is the position of the first failing waypoint in the visiting order.
//
// Regular trees.  Each midpoint step moves an endpoint by at most 2^-53 M
// (M = max |coordinate|), so after d levels every interval width is within
// d 2^-52 M of w_max / 2^d.  When
//     w_max / 2^(h-1) - e >= tol   and   w_max / 2^h + e < tol,
//     e = (h + 1) 2^-50 M,
// every node above depth h splits and every node at depth h is a leaf: the
// tree is perfect with 2^h - 1 waypoints and pre-order ordinal -> path is a
// closed form.  Lanes take consecutive ranks of the chosen order, rebuild
// their midpoint from (a, b) along the path (bit-identical to the
// reference's recursion), run valid() and ballot for the first failure.
// Edges whose widths fall within e of tol at depth h-1 or h (never
// observed; kept exact anyway) are walked by one lane with the stackless
// exact walk.
//
// A check takes L = D/5 lanes (arm_near.hpp: FP32 clearance bounds), so a
// round of a wave is R = 64/L ranks.
//
// Schedule (arm_link).  Wave w of a block sets its edge up (height, prefix
// sums of the end states' angles, in LDS) and checks its first R ranks: most
// colliding edges fail there, and giving them more than one wave would only
// add rounds whose answers are not needed.  Then all P waves of the block
// take the rounds of each edge still open, wave p rounds 1 + p, 1 + p + P, ...
// A wave leaves an edge when its first certain failure (a minimum in LDS over
// the waves) is below its next round, so that minimum ends at exactly the
// first certainly failing rank of the chosen order: the rank lies in one
// wave's rounds, and the wave cannot leave before it.  Few edges (E = 1): a
// block has one edge and its P waves take rounds p, p + P, ... from the
// start, since a chip with idle waves gains from every round that starts
// early.
//
// A check the bounds leave in doubt goes to a list and counts as passed;
// arm_link_rest gives each listed check the exact test, a wave per check, and
// lowers the edge's result where it fails.  The exact test inline held every
// wave of arm_link at 140 VGPRs for a handful of checks in a million (8192
// planner edges: 110 us against 50).  Past the list's end the edge itself is
// listed, and arm_link_rest walks it with the exact check behind the bounds.
// Edges whose trees are not perfect go to a third list and are walked node by
// node.
//
// The kernels this replaced (64 ranks per round, a lane per exact FP64 check)
// took 81 + 278 + 6 us for 8192 planner edges of the 20-link arm among 200
// disks, and 75 + 85 + 5 us for 64.
#include <algorithm>

#include "arm_near.hpp"
#include "wave_list.hpp"

namespace mptg {
namespace {

constexpr int kWave = 64;

// Counters and lists of one link call (ctx->scratch[10]): zero at the start
// of a call, cleared by the last block of arm_link_rest.
struct ArmLists {
    uint32_t n_open, n_irregular, n_doubt, ticket;
};
constexpr size_t kArmListsBytes = 256;

__device__ __forceinline__ int lane_id() { return (int)(threadIdx.x & 63); }

// Waypoint at `rank` of the chosen order (tree of h levels): the reference
// pre-order, or the surrogate order -- the edge's kPicks picks (best-scored
// nodes of its top tree, from the scoring kernel) at ranks 0..3, then every
// other waypoint in reference order.  `sorted` holds the picks in ascending
// ordinal order, `picks` as scored.
template <int ORD>
__device__ __forceinline__ uint32_t ordinal_at(uint32_t rank, const uint32_t (&sorted)[kPicks],
                                               const uint16_t* __restrict__ picks) {
    if constexpr (ORD == MPTG_ORDER_SURROGATE)
        return rank < (uint32_t)kPicks ? (uint32_t)picks[rank] : skip_picks(rank - kPicks, sorted);
    return rank;
}

// The 4 picks of edge e in ascending ordinal order (wave-uniform loads).
__device__ __forceinline__ void sorted_picks(const uint16_t* __restrict__ picks, int64_t e, uint32_t (&p)[kPicks]) {
#pragma unroll
    for (int i = 0; i < kPicks; ++i) p[i] = picks[e * kPicks + i];
    // 5-comparator sorting network
    auto cs = [&](int i, int j) {
        const uint32_t lo = p[i] < p[j] ? p[i] : p[j], hi = p[i] < p[j] ? p[j] : p[i];
        p[i] = lo;
        p[j] = hi;
    };
    cs(0, 1);
    cs(2, 3);
    cs(0, 2);
    cs(1, 3);
    cs(1, 2);
}

// Dyadic positions of a perfect tree's waypoints in pre-order: entry
// 2^h - 1 + ordinal for the trees of h <= kPosLevels levels.
constexpr int kPosLevels = 9;
struct TreePos {
    float t[2 << kPosLevels];
    constexpr TreePos() : t{} {
        for (int h = 1; h <= kPosLevels; ++h)
            for (uint32_t o = 0; o < (1u << h) - 1u; ++o) {
                float lo = 0.0f, width = 1.0f;
                uint32_t k = o, sub = (1u << h) - 1u;
                while (k != 0) {
                    k -= 1;
                    width *= 0.5f;
                    const uint32_t half = (sub - 1u) >> 1;
                    if (k >= half) {
                        k -= half;
                        lo += width;
                    }
                    sub = half;
                }
                t[(1u << h) - 1u + o] = lo + 0.5f * width;
            }
    }
};
__device__ const TreePos kTreePos{};

// An edge's data for its rounds, set up by one wave.
template <int D>
struct ArmEdge {
    double2 turn[D];          // absolute link angles at `from` (turns), and their change to `to`
    uint32_t sorted[kPicks];  // surrogate order: its picks by ordinal
    int64_t e;
    uint32_t W;               // waypoints
    uint32_t first, open;     // keys of the first certain failure and of the first check in doubt
                              // that found its list full: 0 = from, 1 = to, 2 + rank
    uint32_t status;
};
enum : uint32_t { kEdgeNone = 0, kEdgeLive = 1, kEdgeOverLimit = 2 };
constexpr uint32_t kNoKey = 0xffffffffu;

__device__ __forceinline__ double wave_max_f64(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = __builtin_fmax(v, __shfl_xor(v, o));
    return v;
}

// Inclusive prefix sum over lanes 0 .. 31.
__device__ __forceinline__ double prefix32(double v, int lane) {
    v += row_up<1>(v);
    v += row_up<2>(v);
    v += row_up<4>(v);
    v += row_up<8>(v);
    const double r = wl_readlane(v, 15);
    return (lane & 16) ? v + r : v;
}

struct ArmLinkArgs {
    const double *from, *to;
    int64_t n;
    int known_valid;
    const uint8_t* mask;
    double tol;
    SceneArgs sc;
    const uint16_t* picks;
    uint8_t* verdict;
    uint32_t* checks;
    ArmLists* lists;
    int64_t *open, *irregular;  // edges, n at most each
    uint64_t* doubt;            // checks: edge << 32 | key
    uint32_t doubt_cap;
    unsigned long long* work;
};

// The edges [e0, e0 + E) of one block of P waves; EXACT: checks in doubt take
// the exact check here, else they are listed.  Ends with a barrier
// before its last reads of `edges` only: callers that loop add their own.
template <int D, bool COUNT, int ORD, int P, int E, bool EXACT>
__device__ __forceinline__ void arm_block(const ArmLinkArgs& A, ArmEdge<D>* edges, int64_t e0) {
    static_assert(E == P || E == 1, "an edge per wave, or one per block");
    constexpr int L = near_lanes<D>(), R = kWave / L;  // ranks per round
    const int lane = lane_id(), u = lane % L, slot = lane / L;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    NearWork nw{0, 0};
    uint32_t n_calls = 0, n_exact = 0;

    if (w < E) {  // set up edge w
        const int64_t e = e0 + w;
        ArmEdge<D>& ed = edges[w];
        uint32_t status = kEdgeNone, W = 0;
        if (e < A.n && (!A.mask || A.mask[e])) {
            const double a = lane < D ? A.from[e * D + lane] : 0.0, b = lane < D ? A.to[e * D + lane] : 0.0;
            const double t0 = prefix32(a * kInv2Pi, lane), dt = prefix32((b - a) * kInv2Pi, lane);
            if (lane < D) ed.turn[lane] = make_double2(t0, dt);
            int h = 0;
            bool regular = false;
            if (!bisect_height(wave_max_f64(__builtin_fabs(a - b)),
                               wave_max_f64(__builtin_fmax(__builtin_fabs(a), __builtin_fabs(b))), A.tol, &h,
                               &regular)) {
                status = kEdgeOverLimit;
            } else if (!regular || (ORD == MPTG_ORDER_SURROGATE && h > kMaxPickDepth)) {
                if (lane == 0) A.irregular[atomicAdd(&A.lists->n_irregular, 1u)] = e;
            } else {
                status = kEdgeLive;
                W = (1u << h) - 1u;
            }
            if constexpr (ORD == MPTG_ORDER_SURROGATE) {
                uint32_t sp[kPicks] = {0, 0, 0, 0};
                if (W > (uint32_t)kPicks) sorted_picks(A.picks, e, sp);
                if (lane < kPicks) ed.sorted[lane] = lane == 0 ? sp[0] : (lane == 1 ? sp[1] : (lane == 2 ? sp[2] : sp[3]));
            }
        }
        if (lane == 0) {
            ed.e = e;
            ed.W = W;
            ed.first = ed.open = kNoKey;
            ed.status = status;
        }
    }
    __syncthreads();

    float len[kNearLinks];
#pragma unroll
    for (int k = 0; k < kNearLinks; ++k) len[k] = (float)A.sc.lengths[u * kNearLinks + k];

    // Checks this wave's R slots of edge i, keys k0 .. k0 + R - 1.  ends:
    // slots 0 and 1 are the end states (keys 0 and 1), else slot j is rank
    // k0 - 2 + j.
    auto round = [&](int i, uint32_t k0, bool ends) {
        ArmEdge<D>& ed = edges[i];
        const int64_t e = ed.e;
        const uint32_t W = ed.W;
        const uint32_t key = k0 + (uint32_t)slot;
        const bool active = ends ? slot < 2 : key - 2u < W;
        const int h = 32 - __builtin_clz(W | 1u);
        double t = ends && slot == 1 ? 1.0 : 0.0;
        uint32_t o = 0;
        if (!ends) {
            uint32_t sp[kPicks] = {0, 0, 0, 0};
            if constexpr (ORD == MPTG_ORDER_SURROGATE) {
#pragma unroll
                for (int q = 0; q < kPicks; ++q) sp[q] = ed.sorted[q];
            }
            o = active ? ordinal_at<ORD>(key - 2u, sp, A.picks + e * kPicks) : 0u;
            if (h <= kPosLevels) {
                t = (double)kTreePos.t[W + o];
            } else {
                uint32_t path = 0;
                int depth = 0;
                preorder_path(h, o, &path, &depth);
                // (2 steps + 1) / 2^(depth + 1), the first step the highest bit
                const uint32_t steps = depth ? __brev(path) >> (32 - depth) : 0u;
                t = __builtin_ldexp((double)(2u * steps + 1u), -(depth + 1));
            }
        }
        double turn[kNearLinks];
#pragma unroll
        for (int k = 0; k < kNearLinks; ++k) {
            const double2 td = ed.turn[u * kNearLinks + k];
            turn[k] = __builtin_fma(t, td.y, td.x);
        }
        bool bad, doubt;
        if constexpr (EXACT) {
            uint32_t path = 0;
            int depth = -1;
            if (!ends) preorder_path(h, o, &path, &depth);
            const double* a = A.from + e * D;
            const double* b = A.to + e * D;
            bad = !arm_ok_near<D, COUNT>(A.sc, turn, len, ends && slot == 1 ? b : a, b, path, depth, active, &nw,
                                         &n_exact);
            doubt = false;
        } else {
            const int f = near_links<D, COUNT>(A.sc, turn, len, active, &nw);
            bad = group_any<L>(f & 1);
            doubt = group_any<L>(f & 2) && !bad;
        }
        if constexpr (COUNT) n_calls += active && u == 0 ? 1 : 0;
        const uint64_t m = __ballot(active && bad);
        if (m && lane == 0) atomicMin(&ed.first, k0 + (uint32_t)(__builtin_ctzll(m) / L));
        if constexpr (!EXACT) {
            const bool lead = active && doubt && u == 0 &&
                              key < __hip_atomic_load(&ed.first, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            const uint64_t d = __ballot(lead);
            if (d) {
                const uint32_t cnt = (uint32_t)__popcll(d);
                uint32_t base = 0;
                if (lane == 0) base = atomicAdd(&A.lists->n_doubt, cnt);
                base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
                const uint32_t at = base + (uint32_t)__popcll(d & ((1ull << lane) - 1ull));
                if (lead && at < A.doubt_cap) A.doubt[at] = ((uint64_t)e << 32) | key;
                if (lead && at >= A.doubt_cap) atomicMin(&ed.open, key);
            }
        }
    };

    // One call site for every round (inlined once).  Stage 0: the end states
    // of the wave's own edge; 1: its own first round; 2: the open edges.
    const bool own = w < E && edges[w].status != kEdgeNone;  // (over the limit: W = 0, the end states alone)
    int stage = A.known_valid ? 1 : 0, i = w;
    uint32_t key = 0;
    const uint32_t key0 = 2u + (uint32_t)R * (uint32_t)((E == P ? 1 : 0) + w);
    while (true) {
        bool run = own;
        if (stage == 0) {
            key = 0;
        } else if (stage == 1) {
            key = 2;
            run = run && E == P && edges[w].W > 0 && edges[w].first == kNoKey;
        } else {
            if (i >= E) break;
            run = edges[i].status == kEdgeLive && key - 2u < edges[i].W &&
                  __hip_atomic_load(&edges[i].first, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) >= key;
        }
        if (run) round(i, key, stage == 0);
        if (stage < 2) {
            if (++stage == 2) {
                if constexpr (E == P) __syncthreads();  // every wave gets here once
                i = 0;
                key = key0;
            }
        } else if (run) {
            key += (uint32_t)R * P;
        } else {
            ++i;
            key = key0;
        }
    }
    __syncthreads();
    if (threadIdx.x < E) {
        const ArmEdge<D>& ed = edges[threadIdx.x];
        const int64_t e = ed.e;
        if (ed.status != kEdgeNone) {
            if (!EXACT && ed.open < ed.first) {
                A.open[atomicAdd(&A.lists->n_open, 1u)] = e;
            } else if (ed.first != kNoKey) {
                A.verdict[e] = 0;
                A.checks[e] = ed.first + 1u;
            } else {
                A.verdict[e] = ed.status == kEdgeLive;
                A.checks[e] = ed.status == kEdgeLive ? 2u + ed.W : MPTG_CHECKS_OVER_LIMIT;
            }
        }
    }
    if constexpr (COUNT) {
        atomicAdd(&A.work[0], (unsigned long long)n_calls);
        atomicAdd(&A.work[1], (unsigned long long)n_calls * D);
        atomicAdd(&A.work[2], (unsigned long long)nw.lookups);
        atomicAdd(&A.work[3], (unsigned long long)nw.tests);
        atomicAdd(&A.work[4], (unsigned long long)(u == 0 ? n_exact : 0u));
    }
}

template <int D, bool COUNT, int ORD, int P, int E>
__global__ __launch_bounds__(kWave* P) void arm_link(ArmLinkArgs A) {
    __shared__ ArmEdge<D> edges[E];
    arm_block<D, COUNT, ORD, P, E, false>(A, edges, (int64_t)blockIdx.x * E);
}

// |hi - lo| of one coordinate over the interval of the node at (path, depth).
__device__ __forceinline__ double coord_width(double lo, double hi, uint32_t path, int depth) {
    for (int k = 0; k < depth; ++k) {
        const double m = (lo + hi) / 2;
        const bool right = (path >> k) & 1u;
        lo = right ? m : lo;
        hi = right ? hi : m;
    }
    return __builtin_fabs(lo - hi);
}

// Edges whose trees are not perfect: a group of L lanes walks each node by
// node as the reference's recursion does.  Every lane of the wave calls it;
// e < 0: no edge.
template <int D>
__device__ __forceinline__ void irregular_walk(const ArmLinkArgs& A, int64_t e) {
    constexpr int L = near_lanes<D>();
    bool live = e >= 0;
    const double* a = A.from + (live ? e : 0) * D;
    const double* b = A.to + (live ? e : 0) * D;
    uint32_t path = 0, c = 1, result = 0;
    int depth = 0, stage = 0;  // 0: from, 1: to, 2: the tree
    bool ok = true;
    while (__ballot(live)) {
        bool check = live && !A.known_valid;
        if (live && stage == 2) {
            double m = 0.0;
#pragma unroll 1
            for (int j = 0; j < D; ++j) m = __builtin_fmax(m, coord_width(a[j], b[j], path, depth));
            check = !(m < A.tol);
            c += check ? 1u : 0u;
        }
        const bool pass = arm_ok_split<D, L>(
            A.sc, [&](int j) { return stage == 0 ? a[j] : (stage == 1 ? b[j] : coord_mid(a[j], b[j], path, depth)); },
            check);
        if (!live) {
            // done; this group's lanes only take part in the others' checks
        } else if (!pass) {
            ok = live = false;
            result = c;
        } else if (stage < 2) {
            c += stage == 0 ? 1u : 0u;
            ++stage;
        } else if (check) {
            if (depth >= kMaxArmDepth) {
                ok = live = false;
                result = MPTG_CHECKS_OVER_LIMIT;
            }
            ++depth;  // descend left (bit stays 0)
        } else {
            while (depth > 0 && ((path >> (depth - 1)) & 1u)) {
                path &= ~(1u << (depth - 1));
                --depth;
            }
            if (depth == 0) {
                live = false;
                result = c;
            } else {
                path |= 1u << (depth - 1);
            }
        }
    }
    if (e >= 0 && threadIdx.x % L == 0) {
        A.verdict[e] = ok ? 1 : 0;
        A.checks[e] = result;
    }
}

// The exact check of one state by a whole wave: the midpoint of (a, b) at
// (path, depth), or a at depth -1 (wave-uniform).  Lane i < D takes link i:
// its coordinate, then the angle and the joints as the same left-to-right
// sums arm_valid makes, then its link against the disks listed for its cell
// (every other disk is clear of it by more than the bounds' margin).
template <int D>
__device__ __forceinline__ bool arm_exact_wave(const SceneArgs& sc, const double* a, const double* b, uint32_t path,
                                               int depth) {
    const int lane = lane_id();
    const bool mine = lane < D;
    const int j = mine ? lane : 0;
    const double q = depth < 0 ? a[j] : coord_mid(a[j], b[j], path, depth);
    double angle = 0.0, fx = 0.0, fy = 0.0;
#pragma unroll
    for (int i = 0; i < D; ++i) {
        const double v = wl_readlane(q, i);
        angle = i <= lane ? angle + v : angle;
    }
    double s, c;
    pm::sincos(angle, &s, &c);
    const double L = sc.lengths[j];
    const double lx = L * c, ly = L * s;
#pragma unroll
    for (int i = 0; i < D; ++i) {
        const double vx = wl_readlane(lx, i), vy = wl_readlane(ly, i);
        fx = i < lane ? fx + vx : fx;
        fy = i < lane ? fy + vy : fy;
    }
    const double tx = fx + lx, ty = fy + ly;
    if (__ballot(mine && joint_lost(tx, ty))) return sc.ndisks == 0;
    const float inv = sc.near_inv, mid = sc.near_extent * inv;
    const int nc = sc.near_n;
    int ix = (int)__builtin_fmaf(0.5f * ((float)fx + (float)tx), inv, mid);
    int iy = (int)__builtin_fmaf(0.5f * ((float)fy + (float)ty), inv, mid);
    ix = ix < 0 ? 0 : (ix >= nc ? nc - 1 : ix);
    iy = iy < 0 ? 0 : (iy >= nc ? nc - 1 : iy);
    const uint2 run = mine ? sc.near_cells[iy * nc + ix] : make_uint2(0u, 0u);
    bool ok = true;
    for (uint32_t k = 0; k < run.y; ++k) {
        const ArmDisk dk = sc.arm_disks[sc.near_ids[run.x + k]];
        if (!(seg_dist_sq(dk.cx, dk.cy, fx, fy, tx, ty) > dk.rr2)) ok = false;
    }
    return __ballot(!ok) == 0;
}

// A listed check: an exact failure lowers the edge's result (its provisional
// check count is at least the key's).
template <int D, int ORD>
__device__ __forceinline__ void settle_doubt(const ArmLinkArgs& A, uint64_t entry) {
    const int lane = lane_id();
    const int64_t e = (int64_t)(entry >> 32);
    const uint32_t key = (uint32_t)entry;
    const double* a = A.from + e * D;
    const double* b = A.to + e * D;
    uint32_t path = 0;
    int depth = -1;
    if (key >= 2u) {
        const double x = lane < D ? a[lane] : 0.0, y = lane < D ? b[lane] : 0.0;
        int h = 0;
        bool regular = false;
        bisect_height(wave_max_f64(__builtin_fabs(x - y)),
                      wave_max_f64(__builtin_fmax(__builtin_fabs(x), __builtin_fabs(y))), A.tol, &h, &regular);
        uint32_t sp[kPicks] = {0, 0, 0, 0};
        if constexpr (ORD == MPTG_ORDER_SURROGATE) sorted_picks(A.picks, e, sp);
        preorder_path(h, ordinal_at<ORD>(key - 2u, sp, A.picks + e * kPicks), &path, &depth);
    }
    if (!arm_exact_wave<D>(A.sc, key == 1u ? b : a, b, path, depth) && lane == 0) {
        A.verdict[e] = 0;
        atomicMin(&A.checks[e], key + 1u);
    }
}

// all: every edge with the exact check behind the bounds, or alone in scenes
// without bounds.  Else what arm_link (or `all`) left: checks in doubt, edges
// past that list's end, and edges with irregular trees; the last block to end
// clears the counters for the next call.  (A listed edge's checks in doubt
// may be settled before or after its walk writes its result: the walk finds
// the first failure itself, so neither order changes it.)  (Nothing listed, the usual case, ends at once: every
// block sees the same counts, since the clearing block is the last of them
// to leave.)
constexpr int kRestWaves = 4;
template <int D, bool COUNT, int ORD>
__global__ __launch_bounds__(kWave* kRestWaves) void arm_link_rest(ArmLinkArgs A, int all) {
    __shared__ ArmEdge<D> edge;
    const int64_t n_open = all ? A.n : (int64_t)A.lists->n_open;
    const int64_t n_irr = all ? 0 : (int64_t)A.lists->n_irregular;
    uint32_t n_doubt = all ? 0u : A.lists->n_doubt;
    n_doubt = n_doubt < A.doubt_cap ? n_doubt : A.doubt_cap;
    for (uint32_t i = blockIdx.x + gridDim.x * __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); i < n_doubt;
         i += gridDim.x * kRestWaves)
        settle_doubt<D, ORD>(A, A.doubt[i]);
    for (int64_t i = blockIdx.x; i < n_open; i += gridDim.x) {  // block-uniform
        arm_block<D, COUNT, ORD, kRestWaves, 1, true>(A, &edge, all ? i : A.open[i]);
        __syncthreads();
    }
    if (n_open + n_irr + (int64_t)n_doubt == 0 || all) return;
    constexpr int L = near_lanes<D>();
    const int64_t groups = (int64_t)gridDim.x * (kWave * kRestWaves / L);
    const int64_t g = ((int64_t)blockIdx.x * (kWave * kRestWaves) + threadIdx.x) / L;
    for (int64_t i0 = 0; i0 < n_irr; i0 += groups) irregular_walk<D>(A, i0 + g < n_irr ? A.irregular[i0 + g] : -1);
    __syncthreads();
    if (threadIdx.x == 0 && atomicAdd(&A.lists->ticket, 1u) == gridDim.x - 1) {
        A.lists->n_open = 0;
        A.lists->n_irregular = 0;
        A.lists->n_doubt = 0;
        A.lists->ticket = 0;
    }
}

}  // namespace

template <int D, bool COUNT, int ORD>
static int launch_arm(mptg_ctx* ctx, ArmLinkArgs A) {
    int rc;
    if constexpr (ORD == MPTG_ORDER_SURROGATE) {
        if ((rc = ensure(ctx, ctx->scratch[9], sizeof(uint16_t) * kPicks * A.n))) return rc;
        if ((rc = surrogate_picks(ctx, A.from, A.to, A.n, A.mask, (uint16_t*)ctx->scratch[9].p))) return rc;
        A.picks = (const uint16_t*)ctx->scratch[9].p;
    }
    phase_mark(ctx, 1);
    const unsigned rest = (unsigned)std::min<int64_t>(A.n, ctx->cus);
    if (A.sc.near_n > 0) {
#define MPTG_ARM_LINK(P, E)                                                                                     \
    hipLaunchKernelGGL((arm_link<D, COUNT, ORD, P, E>), dim3((unsigned)((A.n + E - 1) / E)), dim3(kWave * P), 0, \
                       ctx->stream, A)
        // a block per edge up to the waves that fill the chip (8 per edge, 32
        // per CU): 2000 edges 46 -> 38 us, 3000 the same either way.  Blocks of
        // many edges: 8 (20 links: 8192 edges 98 us with 4, 92 with 8, 95 with
        // 16); arms of fewer links have fewer rounds to share, 4.
        constexpr int PE = D >= 20 ? 8 : 4;
        if (A.n < (int64_t)ctx->cus * 8) MPTG_ARM_LINK(8, 1);
        else MPTG_ARM_LINK(PE, PE);
#undef MPTG_ARM_LINK
    } else {
        hipLaunchKernelGGL((arm_link_rest<D, COUNT, ORD>), dim3((unsigned)std::min<int64_t>(A.n, (int64_t)ctx->cus * 8)),
                           dim3(kWave * kRestWaves), 0, ctx->stream, A, 1);
    }
    phase_mark(ctx, 2);
    phase_mark(ctx, 3);
    hipLaunchKernelGGL((arm_link_rest<D, COUNT, ORD>), dim3(rest), dim3(kWave * kRestWaves), 0, ctx->stream, A, 0);
    phase_mark(ctx, 4);
    phase_mark(ctx, 5);
    return MPTG_OK;
}

template <int D>
static int launch_arm_d(mptg_ctx* ctx, int order, const ArmLinkArgs& A) {
    if (order == MPTG_ORDER_SURROGATE)
        return A.work ? launch_arm<D, true, MPTG_ORDER_SURROGATE>(ctx, A) : launch_arm<D, false, MPTG_ORDER_SURROGATE>(ctx, A);
    return A.work ? launch_arm<D, true, MPTG_ORDER_REFERENCE>(ctx, A) : launch_arm<D, false, MPTG_ORDER_REFERENCE>(ctx, A);
}

int launch_arm_link(mptg_ctx* ctx, const double* from, const double* to, int64_t n, int known_valid,
                    const uint8_t* mask, uint8_t* verdict, uint32_t* checks, unsigned long long* work, int order) {
    if (ctx->dim != ctx->scene.nlinks) return MPTG_E_STATE;
    if (ctx->dim != 5 && ctx->dim != 10 && ctx->dim != 20) return MPTG_E_STATE;
    if (n <= 0) return MPTG_OK;
    int rc;
    DevBuf& buf = ctx->scratch[10];
    const int64_t cap = n + 4096;  // checks in doubt
    const size_t need = kArmListsBytes + sizeof(int64_t) * (size_t)(2 * n + cap);
    if (!buf.p || buf.bytes < need) ctx->link_lists_clean = false;
    if ((rc = ensure(ctx, buf, need))) return rc;
    ArmLinkArgs A{from, to, n, known_valid, mask, ctx->link_param, scene_args(ctx), nullptr, verdict, checks,
                  (ArmLists*)buf.p, (int64_t*)((char*)buf.p + kArmListsBytes), nullptr, nullptr, (uint32_t)cap, work};
    A.irregular = A.open + n;
    A.doubt = (uint64_t*)(A.irregular + n);
    if (!ctx->link_lists_clean && (rc = launch_zero_u32(ctx, (uint32_t*)A.lists, kArmListsBytes / 4))) return rc;
    const bool was_clean = ctx->link_lists_clean;
    ctx->link_lists_clean = false;  // until both kernels are enqueued
    phase_mark(ctx, 0);
    switch (ctx->dim) {
        case 5: rc = launch_arm_d<5>(ctx, order, A); break;
        case 10: rc = launch_arm_d<10>(ctx, order, A); break;
        default: rc = launch_arm_d<20>(ctx, order, A); break;
    }
    if (rc) return rc;
    MPTG_HIP(ctx, hipGetLastError());
    ctx->link_lists_clean = was_clean || !stream_capturing(ctx);
    return MPTG_OK;
}

}  // namespace mptg
