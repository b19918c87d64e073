// Arm validity with FP32 clearance bounds in front of the exact test, L = D/5
// lanes per state (five links each).
//
// What bounded the exact check: arm_ok_lane issues ~7 400 wave instructions
// for 64 states of the 20-link arm among 200 disks -- per link the fdlibm
// sine and cosine and, on an edge, the midpoint recursion of one coordinate
// (~130 FP64 instructions), then group and link tests over divergent disk
// runs.  Nearly every (link, disk) pair clears or hits by far more than the
// rounding of a cheaper evaluation, so:
//   * angles come as turns; a waypoint's are A_j + t (B_j - A_j), one FP64
//     FMA per link, from the edge's prefix sums (t is the waypoint's dyadic
//     position), reduced to [-1/2, 1/2] and rounded to FP32;
//   * v_sin_f32 / v_cos_f32 (arguments in turns) and FP32 joints;
//   * a link is tested against the disks listed for the cell of its midpoint
//     (every disk within half the longest link + its own r + R of the cell);
//   * the test is certain when the FP32 distance is farther than a margin
//     from r + R.  A state with a certain hit is invalid, one with every pair
//     certainly clear is valid, any other takes the exact check
//     (arm_ok_split), so verdicts are the exact check's.
// Planner edges of the scene above: 0.12 tests per link, and one check in
// 20 000 is left to the exact one.
//
// Margin.  With T = the sum of the link lengths, Lm the longest link and rm
// the disk's r + R, the FP32 distance differs from the exact expression's by
// less than the sum of
//   directions: the angle's rounding 2^-26 turns = 9.4e-8 rad and the
//     instructions' error, at most 1.26e-7 each on gfx950 over every FP32
//     argument in [-1/2, 1/2] (measured exhaustively): 2.8e-7 T over the
//     chain; angles below kMaxTurns turns in FP64, and the exact test's own
//     sums and midpoints of them, add under 1.5e-7 T;
//   joints: lengths rounded to FP32, five links summed per lane, at most
//     three prefix sums and one addition, each 2^-24 T, both axes: 8.3e-7 T;
//   the centre's rounding, |centre| below T + Lm + 2 rm where it matters:
//     8.5e-8 (T + Lm + 2 rm);
//   the distance itself, a dozen FP32 operations on values below Lm + rm:
//     8e-7 (Lm + rm);
//   the exact expression's own FP64 rounding: below 1e-11 T.
// The sum is below 1.35e-6 T + 9e-7 Lm + 1e-6 rm; the disk's margin is
// kNearMargin (T + Lm + rm) with kNearMargin = 2^-18 = 3.8e-6, 2.8 times that.
// (A margin from the scene's largest disk left the checks near every disk in
// doubt: 8192 edges beside a wall of radius 1e5 took 700 us, 37 now.  Angles
// above 1024 turns left to the exact test took 1 450 us, 31 now.)
#pragma once
#include "bisect_dev.hpp"

namespace mptg {

constexpr int kNearLinks = 5;  // links per lane
constexpr double kMaxTurns = 131072.0;  // half of what pm::sincos takes
constexpr double kInv2Pi = 0.15915494309189533577;

template <int D>
constexpr int near_lanes() {
    static_assert(D % kNearLinks == 0 && 64 % (D / kNearLinks) == 0, "five links per lane, whole groups per wave");
    return D / kNearLinks;
}

// Lane l's value moved to lane l + O within its row of 16 lanes (0 enters).
template <int O>
__device__ __forceinline__ double row_up(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x110 + O, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x110 + O, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

template <int O>
__device__ __forceinline__ float row_up(float v) {
    return float_of((uint32_t)__builtin_amdgcn_update_dpp(0, (int)bits_of(v), 0x110 + O, 0xf, 0xf, false));
}

// Exclusive prefix sum over the L lanes of an aligned group (L = 1, 2, 4).
template <int L, typename T>
__device__ __forceinline__ T group_before(T v, int u) {
    if constexpr (L == 1) return T(0);
    T x = row_up<1>(v);
    x = u >= 1 ? x : T(0);
    if constexpr (L > 2) {
        const T y = row_up<1>(x), z = row_up<2>(x);
        x = x + (u >= 2 ? y : T(0)) + (u >= 3 ? z : T(0));
    }
    return x;
}

// The flags of this lane's group of L lanes, ORed.
template <int L>
__device__ __forceinline__ bool group_any(bool f) {
    if constexpr (L == 1) return f;
    const uint64_t m = __ballot(f);
    return ((m >> (threadIdx.x & 63u & ~(unsigned)(L - 1))) & ((1ull << L) - 1ull)) != 0;
}

struct NearWork {
    uint32_t lookups, tests;
};

// This lane's five links against the disks near them: bit 0 = certain hit,
// bit 1 = some pair not certainly clear (a hit sets both).  turn[k] = the
// link's absolute angle in turns, len[k] its length.  Every lane of the wave
// calls it (the joints are a prefix sum over the group); lanes that are not
// active look at no disk and return 0.
template <int D, bool COUNT = false>
__device__ __forceinline__ int near_links(const SceneArgs& sc, const double (&turn)[kNearLinks],
                                          const float (&len)[kNearLinks], bool active, NearWork* wk = nullptr) {
    constexpr int L = near_lanes<D>(), N = kNearLinks;
    const int u = (int)(threadIdx.x & (L - 1));
    float px[N], py[N], ux[N], uy[N];
    float x = 0.0f, y = 0.0f;
    bool sane = true;
#pragma unroll
    for (int k = 0; k < N; ++k) {
        sane = sane && __builtin_fabs(turn[k]) < kMaxTurns;  // false for NaN
        const float f = (float)(turn[k] - __builtin_rint(turn[k]));
        ux[k] = __builtin_amdgcn_cosf(f);
        uy[k] = __builtin_amdgcn_sinf(f);
        px[k] = x;
        py[k] = y;
        x = __builtin_fmaf(len[k], ux[k], x);
        y = __builtin_fmaf(len[k], uy[k], y);
    }
    const float bx = group_before<L>(x, u), by = group_before<L>(y, u);
    if (!group_any<L>(!sane)) {
        const float inv = sc.near_inv, mid = sc.near_extent * inv;
        const int nc = sc.near_n;
        uint2 run[N];
        uint32_t most = 0;
#pragma unroll
        for (int k = 0; k < N; ++k) {
            px[k] += bx;
            py[k] += by;
            const float h = 0.5f * len[k];
            int ix = (int)__builtin_fmaf(__builtin_fmaf(h, ux[k], px[k]), inv, mid);
            int iy = (int)__builtin_fmaf(__builtin_fmaf(h, uy[k], py[k]), inv, mid);
            ix = ix < 0 ? 0 : (ix >= nc ? nc - 1 : ix);
            iy = iy < 0 ? 0 : (iy >= nc ? nc - 1 : iy);
            run[k] = active ? sc.near_cells[iy * nc + ix] : make_uint2(0u, 0u);
            if constexpr (COUNT) wk->lookups += active ? 1 : 0;
        }
#pragma unroll
        for (int k = 0; k < N; ++k) most = run[k].y > most ? run[k].y : most;
        bool hit = false, open = false;
        // the j-th disk of each link's list together: five loads in flight
        for (uint32_t j = 0; j < most; ++j) {
#pragma unroll
            for (int k = 0; k < N; ++k) {
                if (j < run[k].y) {
                    const float4 d = sc.near_disks[run[k].x + j];
                    const float wx = d.x - px[k], wy = d.y - py[k];
                    float t = __builtin_fmaf(wx, ux[k], wy * uy[k]);
                    t = __builtin_fminf(__builtin_fmaxf(t, 0.0f), len[k]);
                    const float ex = __builtin_fmaf(-t, ux[k], wx), ey = __builtin_fmaf(-t, uy[k], wy);
                    const float d2 = __builtin_fmaf(ex, ex, ey * ey);
                    hit = hit || d2 < d.z;
                    open = open || !(d2 > d.w);
                    if constexpr (COUNT) wk->tests += 1;
                }
            }
            if (hit) break;
        }
        return (hit ? 1 : 0) | (open ? 2 : 0);
    }
    return active ? 2 : 0;
}

// valid() of the state of this lane's group: the midpoint of the interval
// (a, b) at (path, depth), or a itself at depth -1; turn / len: this lane's
// links, as near_links takes them.  Every lane of the wave calls it; inactive
// groups return true.  The result is the same on all lanes of a group.
template <int D, bool COUNT = false>
__device__ __forceinline__ bool arm_ok_near(const SceneArgs& sc, const double (&turn)[kNearLinks],
                                            const float (&len)[kNearLinks], const double* a, const double* b,
                                            uint32_t path, int depth, bool active, NearWork* wk = nullptr,
                                            uint32_t* exact = nullptr) {
    constexpr int L = near_lanes<D>();
    bool bad = false, open = active;
    if (sc.near_n > 0) {  // uniform
        const int f = near_links<D, COUNT>(sc, turn, len, active, wk);
        bad = group_any<L>(f & 1);
        open = group_any<L>(f & 2) && !bad;
    }
    if (__ballot(open)) {
        if constexpr (COUNT) *exact += open ? 1 : 0;
        if (!arm_ok_split<D, L>(
                sc, [&](int j) { return depth < 0 ? a[j] : coord_mid(a[j], b[j], path, depth); }, open))
            bad = true;
    }
    return !bad;
}

// This lane's links of a state with coordinates coord(i): absolute angles in
// turns (prefix sums over the group) and lengths.
template <int D, typename Coord>
__device__ __forceinline__ void state_turns(const SceneArgs& sc, Coord&& coord, double (&turn)[kNearLinks],
                                            float (&len)[kNearLinks]) {
    constexpr int L = near_lanes<D>();
    const int u = (int)(threadIdx.x & (L - 1));
    double a = 0.0;
#pragma unroll
    for (int k = 0; k < kNearLinks; ++k) {
        a = __builtin_fma(coord(u * kNearLinks + k), kInv2Pi, a);
        turn[k] = a;
        len[k] = (float)sc.lengths[u * kNearLinks + k];
    }
    const double before = group_before<L>(a, u);
#pragma unroll
    for (int k = 0; k < kNearLinks; ++k) turn[k] += before;
}

}  // namespace mptg
