// SE(3) rigid body among triangle meshes: the reference's valid(q) =
// !fcl::collide(robot at pose(q), env) (demo/se3_rigid_body_scenario.hpp:288-312)
// and its DiscreteMotionValidator link (:330-334), on the device.
//
// The predicate is mesh_hd.hpp's: posed robot triangle a and environment
// triangle b collide iff their boxes overlap and the separating-axis test
// finds no separating axis.  Culling below only skips pairs whose boxes are
// apart, so the verdict is the predicate's exactly.
//
// Layout in HBM (built on the host at upload):
//   env BVH   binned-SAH binary tree (<= 4 triangles per leaf, depth <= 38)
//             collapsed to MeshNode16[nnodes]: 512 B per node holding the
//             boxes and references of up to sixteen nodes four levels below
//             it, 32 B each, so sixteen lanes read one node
//   env tris  16 floats (64 B) per triangle in leaf order: v0 v1 v2, box lo, hi
//   robot     9 floats per triangle, Morton-sorted by centroid so that the
//             consecutive triangles of a lane's group are close together;
//             after them the groups' boxes (centre, half-sides)
// Kernels (one 64-lane wave per block, one item per wave at a time):
//   mesh_valid  one state per wave
//   mesh_link   one waypoint of one edge per wave at a time (reference
//               checks_done counts), nothing past an edge's first hit
// See mesh_collides for the check of one state.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <vector>

#include "mesh_hd.hpp"
#include "space_dev.hpp"
#include "wave_ops.hpp"

namespace mptg {

namespace {

constexpr int kGroupShift = 3;                  // a lane's group: up to 2^3 robot triangles
constexpr int kBuildDepth = 38;                 // BVH depth bound
constexpr int kMaxDmvWaypointsMesh = 1 << 24;   // same limit as the other DMV kernels
constexpr int kTableMaxMesh = 255;

// ---------------------------------------------------------------------------
// host: BVH build
// ---------------------------------------------------------------------------
struct BuildRef {
    float lo[3], hi[3], c[3];
    int32_t id;
};

struct BvhBuilder {
    std::vector<BuildRef> refs;
    std::vector<MeshNode> nodes;

    static void grow(float* lo, float* hi, const float* blo, const float* bhi) {
        for (int i = 0; i < 3; ++i) {
            lo[i] = std::min(lo[i], blo[i]);
            hi[i] = std::max(hi[i], bhi[i]);
        }
    }
    static float area(const float* lo, const float* hi) {
        const float dx = hi[0] - lo[0], dy = hi[1] - lo[1], dz = hi[2] - lo[2];
        if (!(dx >= 0)) return 0.0f;
        return dx * dy + dy * dz + dz * dx;
    }

    int build(int begin, int end, int depth) {
        const int id = (int)nodes.size();
        nodes.push_back(MeshNode{});
        float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
        float clo[3] = {INFINITY, INFINITY, INFINITY}, chi[3] = {-INFINITY, -INFINITY, -INFINITY};
        for (int i = begin; i < end; ++i) {
            grow(lo, hi, refs[i].lo, refs[i].hi);
            grow(clo, chi, refs[i].c, refs[i].c);
        }
        auto set_box = [&](MeshNode& n) {
            for (int i = 0; i < 3; ++i) {
                n.lo[i] = lo[i];
                n.hi[i] = hi[i];
            }
        };
        const int count = end - begin;
        if (count <= kLeafTris) {
            MeshNode& n = nodes[id];
            set_box(n);
            n.a = begin;
            n.b = -count;
            return id;
        }
        int axis = 0;
        for (int i = 1; i < 3; ++i)
            if (chi[i] - clo[i] > chi[axis] - clo[axis]) axis = i;
        int mid = -1;
        const float ext = chi[axis] - clo[axis];
        if (depth < 20 && ext > 0) {
            constexpr int kBins = 16;
            int bn[kBins] = {};
            float blo[kBins][3], bhi[kBins][3];
            for (int b = 0; b < kBins; ++b)
                for (int i = 0; i < 3; ++i) {
                    blo[b][i] = INFINITY;
                    bhi[b][i] = -INFINITY;
                }
            auto bin_of = [&](const BuildRef& r) {
                int b = (int)((r.c[axis] - clo[axis]) / ext * kBins);
                return std::min(std::max(b, 0), kBins - 1);
            };
            for (int i = begin; i < end; ++i) {
                int b = bin_of(refs[i]);
                bn[b]++;
                grow(blo[b], bhi[b], refs[i].lo, refs[i].hi);
            }
            float best = INFINITY;
            int best_split = -1;
            for (int s = 1; s < kBins; ++s) {
                float llo[3] = {INFINITY, INFINITY, INFINITY}, lhi[3] = {-INFINITY, -INFINITY, -INFINITY};
                float rlo[3] = {INFINITY, INFINITY, INFINITY}, rhi[3] = {-INFINITY, -INFINITY, -INFINITY};
                int nl = 0, nr = 0;
                for (int b = 0; b < s; ++b) {
                    nl += bn[b];
                    if (bn[b]) grow(llo, lhi, blo[b], bhi[b]);
                }
                for (int b = s; b < kBins; ++b) {
                    nr += bn[b];
                    if (bn[b]) grow(rlo, rhi, blo[b], bhi[b]);
                }
                if (nl == 0 || nr == 0) continue;
                const float cost = area(llo, lhi) * nl + area(rlo, rhi) * nr;
                if (cost < best) {
                    best = cost;
                    best_split = s;
                }
            }
            if (best_split > 0) {
                auto it = std::partition(refs.begin() + begin, refs.begin() + end,
                                         [&](const BuildRef& r) { return bin_of(r) < best_split; });
                mid = (int)(it - refs.begin());
            }
        }
        if (mid <= begin || mid >= end) {  // median split: depth stays logarithmic
            mid = begin + count / 2;
            std::nth_element(refs.begin() + begin, refs.begin() + mid, refs.begin() + end,
                             [&](const BuildRef& x, const BuildRef& y) {
                                 return x.c[axis] < y.c[axis] || (x.c[axis] == y.c[axis] && x.id < y.id);
                             });
        }
        const int left = build(begin, mid, depth + 1);
        const int right = build(mid, end, depth + 1);
        MeshNode& n = nodes[id];
        set_box(n);
        n.a = left;
        n.b = right;
        return id;
    }
};

int bvh_depth(const std::vector<MeshNode>& nodes, int n, int d) {
    if (nodes[n].b <= 0) return d;
    return std::max(bvh_depth(nodes, nodes[n].a, d + 1), bvh_depth(nodes, nodes[n].b, d + 1));
}

// Sixteen-wide node: its slots hold the boxes and references of the binary
// nodes four levels below (a leaf above that level takes one slot, and the
// slots that such leaves leave free go to one more level of the first of the
// others).  b > 0: a is a MeshNode16 index; b <= 0: triangles [a, a - b); an
// unused slot has an empty box (lo > hi).
constexpr int kWide = 16, kWideLevels = 4;
struct MeshSlot {
    float lo[3];
    int32_t a;
    float hi[3];
    int32_t b;
};
struct MeshNode16 {
    MeshSlot slot[kWide];
};
static_assert(sizeof(MeshNode16) == 512, "sixteen-wide node is 512 bytes");

// Collapse the binary subtree under id (an internal node, or a leaf root) into
// out (pre-order).
int collapse16(const std::vector<MeshNode>& n2, int id, std::vector<MeshNode16>& out) {
    const int me = (int)out.size();
    out.push_back(MeshNode16{});
    int slot[kWide] = {id}, above[kWide], n = 1;
    for (int level = 0; level <= kWideLevels; ++level) {  // the last one as far as there is room
        const int m = n;
        std::copy(slot, slot + m, above);
        n = 0;
        for (int i = 0; i < m; ++i) {
            const MeshNode& g = n2[(size_t)above[i]];
            if (g.b > 0 && n + (m - i) < kWide) {
                slot[n++] = g.a;
                slot[n++] = g.b;
            } else {
                slot[n++] = above[i];
            }
        }
    }
    MeshNode16 node;
    for (MeshSlot& o : node.slot) o = {{INFINITY, INFINITY, INFINITY}, 0, {-INFINITY, -INFINITY, -INFINITY}, 0};
    for (int k = 0; k < n; ++k) {
        const MeshNode& g = n2[(size_t)slot[k]];
        MeshSlot& o = node.slot[k];
        for (int i = 0; i < 3; ++i) {
            o.lo[i] = g.lo[i];
            o.hi[i] = g.hi[i];
        }
        o.a = g.b > 0 ? collapse16(n2, slot[k], out) : g.a;
        o.b = g.b > 0 ? 1 : g.b;
    }
    out[(size_t)me] = node;
    return me;
}

uint32_t spread10(uint32_t v) {
    v &= 1023u;
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

// ---------------------------------------------------------------------------
// device
// ---------------------------------------------------------------------------
struct MeshArgs {
    const float4* slots;   // 16 slots of 2 float4 per node
    const float4* tris;    // 4 float4 per triangle
    const float* robot;    // 9 floats per triangle
    const float4* groups;  // 2 float4 per group: centre, half-sides
    int nnodes, nrobot;
    int shift;    // a group is 2^shift robot triangles
    float reach, env_reach;  // largest coordinate in magnitude
};

// Below this magnitude no coordinate's products overflow: an axis from a
// normal is at most 2^5 kTameReach^3, its dot product 2^7 kTameReach^4.
constexpr float kTameReach = 0x1p29f;

// One wave's work lists in a check: BVH nodes to open, leaves met, (lane's
// group, environment triangle) pairs and (robot triangle, environment
// triangle) pairs whose boxes overlap.
constexpr int kOpenNodes = 64 / kWide;  // nodes opened at a time, sixteen lanes each
constexpr int kStackSoft = 64;          // above it one node at a time
struct MeshLists {
    // kStackSoft + 60 after the last step of several nodes, and then fifteen
    // more per level of a depth-first descent
    int32_t stack[kStackSoft + 60 + (kWide - 1) * (kBuildDepth / kWideLevels + 2)];
    uint32_t leaf[128];  // first triangle | (count - 1) << 20
    uint32_t pair[128];  // lane | environment triangle << 6
    uint32_t sat[128];   // robot triangle of the chunk | environment triangle << 9
};

// Slots of the lanes with `want` in a list that holds `at` entries; `at` grows.
__device__ __forceinline__ int take_slot(bool want, int& at) {
    const uint64_t b = __ballot(want);
    const int mine = at + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0));
    at += __popcll(b);
    return mine;
}

__device__ __forceinline__ void load_posed(const MeshArgs& m, const Pose32& pose, int i, float* tri) {
    const float* src = m.robot + (size_t)i * 9;
#pragma unroll
    for (int v = 0; v < 3; ++v) xform(pose, src + 3 * v, tri + 3 * v);
}

// Box of robot triangles [first, first + cnt) as posed, vertex by vertex.
__device__ __forceinline__ void posed_box(const MeshArgs& m, const Pose32& pose, int first, int cnt, float* lo, float* hi) {
    for (int i = 0; i < 3; ++i) {
        lo[i] = INFINITY;
        hi[i] = -INFINITY;
    }
#pragma unroll 1
    for (int t = 0; t < cnt; ++t) {
        float tri[9], tlo[3], thi[3];
        load_posed(m, pose, first + t, tri);
        tri_box(tri, tlo, thi);
        for (int i = 0; i < 3; ++i) {
            lo[i] = tlo[i] < lo[i] ? tlo[i] : lo[i];
            hi[i] = thi[i] > hi[i] ? thi[i] : hi[i];
        }
    }
}

// tri_tri_overlap without its early returns: some lane of 64 pairs nearly
// always needs the last axis, and seventeen nested exits hold as many masks.
// For coordinates whose products cannot overflow there is no NaN, and the
// minima and maxima are single instructions.
__device__ __forceinline__ int apart_on_tame(const float* ax, const float* p, const float* q) {
    const float p0 = dot3(ax, p), p1 = dot3(ax, p + 3), p2 = dot3(ax, p + 6);
    const float q0 = dot3(ax, q), q1 = dot3(ax, q + 3), q2 = dot3(ax, q + 6);
    const float pmax = __builtin_fmaxf(__builtin_fmaxf(p0, p1), p2), pmin = __builtin_fminf(__builtin_fminf(p0, p1), p2);
    const float qmax = __builtin_fmaxf(__builtin_fmaxf(q0, q1), q2), qmin = __builtin_fminf(__builtin_fminf(q0, q1), q2);
    return (int)(pmax < qmin) | (int)(qmax < pmin);
}
__device__ __forceinline__ bool tri_tri_overlap_wave(const float* p, const float* q, bool tame) {
    float ep[3][3], eq[3][3], np[3], nq[3], ax[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        sub3(p + 3 * ((i + 1) % 3), p + 3 * i, ep[i]);
        sub3(q + 3 * ((i + 1) % 3), q + 3 * i, eq[i]);
    }
    cross3(ep[0], ep[1], np);
    cross3(eq[0], eq[1], nq);
    if (!tame) {
        // any coordinates: axis by axis in a loop, to hold few registers
        int apart = (int)apart_on(np, p, q) | (int)apart_on(nq, p, q);
#pragma unroll 1
        for (int k = 0; k < 15; ++k) {
            const int i = k / 5, j = k % 5;
            float u[3], v[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const float epi = i == 0 ? ep[0][c] : i == 1 ? ep[1][c] : ep[2][c];
                const float eqi = i == 0 ? eq[0][c] : i == 1 ? eq[1][c] : eq[2][c];
                const float eqj = j == 0 ? eq[0][c] : j == 1 ? eq[1][c] : eq[2][c];
                u[c] = j < 3 ? epi : j == 3 ? np[c] : nq[c];
                v[c] = j < 3 ? eqj : j == 3 ? epi : eqi;
            }
            cross3(u, v, ax);
            apart |= (int)apart_on(ax, p, q);
        }
        return !apart;
    }
    int apart = apart_on_tame(np, p, q) | apart_on_tame(nq, p, q);
    if (__ballot(!apart) == 0) return false;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            cross3(ep[i], eq[j], ax);
            apart |= apart_on_tame(ax, p, q);
        }
        cross3(np, ep[i], ax);
        apart |= apart_on_tame(ax, p, q);
        cross3(nq, eq[i], ax);
        apart |= apart_on_tame(ax, p, q);
    }
    return !apart;
}

// Does the robot at `pose` collide with the environment?  Whole wave; the
// pose is the same on every lane.
//
// A lane owns a group of 2^shift robot triangles and takes a box around it:
// the group's own box moved by the pose (centre R c + t, half-sides |R| h),
// wide enough for every rounding here and in the posed vertices.  Per chunk of
// 64 groups the wave opens BVH nodes that meet the box of them all, four nodes
// at a time, a slot a lane; keeps the environment triangles of the
// leaves that meet it, a triangle a lane; pairs each of those with the groups
// whose boxes it meets; tests the boxes of the pairs' triangles, a triangle a
// lane, which is the predicate's own test; and gives the pairs left to the
// separating-axis test, 64 at a time.  Each of the lists passes its entries on
// when it holds a wave's worth, and in the end.
//
// Bounds: instruction issue (1 370 vector and 920 scalar instructions per
// counted check, 500 robot triangles among 50 000) and, for half of a wave's
// time, the latency of dependent loads; sixteen-wide nodes make four or five
// of them on the way to a leaf, four-wide ones took nine (142 -> 126 us for
// the 4096 edges of mesh_link).  One four-wide node at a time, depth first,
// with scalar loads and a ballot per slot over the lanes' boxes, took 75 nodes,
// 3 300 vector and 2 400 scalar instructions per check (197 us), where 13
// environment triangles lie in the robot's box.
__device__ bool mesh_collides(const MeshArgs& m, const Pose32& pose, MeshLists& w) {
    const int lane = threadIdx.x & 63;
    if (m.nnodes == 0 || m.nrobot == 0) return false;
    const int sh = m.shift;
    const int per = 64 >> sh;  // pairs whose triangles fill the wave
    for (int c0 = 0; c0 < m.nrobot; c0 += 64 << sh) {
        const int first = c0 + (lane << sh);
        const int cnt = max(0, min(1 << sh, m.nrobot - first));
        float llo[3] = {INFINITY, INFINITY, INFINITY}, lhi[3] = {-INFINITY, -INFINITY, -INFINITY};
        bool odd = false;
        if (cnt > 0) {
            const float4 c = m.groups[2 * (first >> sh)], h = m.groups[2 * (first >> sh) + 1];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const float r0 = pose.r[3 * i], r1 = pose.r[3 * i + 1], r2 = pose.r[3 * i + 2], t = pose.t[i];
                const float a0 = __builtin_fabsf(r0), a1 = __builtin_fabsf(r1), a2 = __builtin_fabsf(r2);
                const float mid = __builtin_fmaf(r0, c.x, __builtin_fmaf(r1, c.y, __builtin_fmaf(r2, c.z, t)));
                // 32 roundings of the largest magnitude on the way: the sums
                // here and in a posed vertex take 15 between them
                const float slop = 0x1p-19f * (__builtin_fmaf(a0 + a1 + a2, m.reach, __builtin_fabsf(t)) + 0x1p-100f);
                const float half =
                    __builtin_fmaf(a0, h.x, __builtin_fmaf(a1, h.y, __builtin_fmaf(a2, h.z, slop)));
                llo[i] = mid - half;
                lhi[i] = mid + half;
                odd |= !(__builtin_isfinite(llo[i]) && __builtin_isfinite(lhi[i]));
            }
        }
        if (__ballot(odd)) posed_box(m, pose, first, cnt, llo, lhi);  // a pose without finite bounds
        float blo[3], bhi[3];
        bool tame = m.env_reach < kTameReach;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            blo[i] = wave_min_f32(llo[i]);
            bhi[i] = -wave_min_f32(-lhi[i]);
            tame = tame && blo[i] > -kTameReach && bhi[i] < kTameReach;
        }
        int nopen = 1, nleaf = 0, npair = 0, nsat = 0;  // wave-uniform
        if (lane == 0) w.stack[0] = 0;
        int et = 0;  // this lane's environment triangle and its box; `tris`: the lanes that have one
        float elo[3] = {}, ehi[3] = {};
        uint64_t tris = 0;
        for (;;) {
            __syncthreads();
            const bool found = nopen == 0 && nleaf == 0 && tris == 0;  // no more pairs to come
            if (nsat >= 64 || (nsat > 0 && found && npair == 0)) {
                const int n = min(nsat, 64);
                bool hit = false;
                if (lane < n) {
                    const uint32_t e = w.sat[nsat - 1 - lane];
                    float tri[9], ev[9];
                    load_posed(m, pose, c0 + (int)(e & 511u), tri);
                    const float4* src = m.tris + 4 * (size_t)(e >> 9);
                    const float4 a = src[0], b = src[1];
                    ev[0] = a.x; ev[1] = a.y; ev[2] = a.z; ev[3] = a.w;
                    ev[4] = b.x; ev[5] = b.y; ev[6] = b.z; ev[7] = b.w;
                    ev[8] = src[2].x;
                    hit = tri_tri_overlap_wave(tri, ev, tame);
                }
                if (__ballot(hit)) return true;
                nsat -= n;
            } else if (npair >= per || (npair > 0 && found)) {
                const int n = min(npair, per);
                const int p = lane >> sh;
                bool meet = false;
                uint32_t e = 0;
                int t = 0;
                if (p < n) {
                    e = w.pair[npair - 1 - p];
                    t = (int)((e & 63u) << sh) + (lane & ((1 << sh) - 1));
                    if (c0 + t < m.nrobot) {
                        float tri[9], tlo[3], thi[3];
                        load_posed(m, pose, c0 + t, tri);
                        tri_box(tri, tlo, thi);
                        const float4* src = m.tris + 4 * (size_t)(e >> 6);
                        const float4 c = src[2], d = src[3];
                        const float blo_e[3] = {c.y, c.z, c.w}, bhi_e[3] = {d.x, d.y, d.z};
                        meet = boxes_overlap(tlo, thi, blo_e, bhi_e);
                    }
                }
                npair -= n;
                const int at = take_slot(meet, nsat);
                if (meet) w.sat[at] = (uint32_t)t | (e >> 6) << 9;
            } else if (tris) {
                do {
                    const int src = __builtin_ctzll(tris);
                    tris &= tris - 1;
                    const float tlo[3] = {lane_f32(elo[0], src), lane_f32(elo[1], src), lane_f32(elo[2], src)};
                    const float thi[3] = {lane_f32(ehi[0], src), lane_f32(ehi[1], src), lane_f32(ehi[2], src)};
                    const bool meet = boxes_overlap(tlo, thi, llo, lhi);
                    const uint32_t tri = (uint32_t)__builtin_amdgcn_readlane(et, src);
                    const int at = take_slot(meet, npair);
                    if (meet) w.pair[at] = (uint32_t)lane | tri << 6;
                } while (tris && npair < per);
            } else if (nleaf > 64 || (nleaf > 0 && nopen == 0)) {
                const int n = min(nleaf, 16);
                bool meet = false;
                if ((lane >> 2) < n) {
                    const uint32_t e = w.leaf[nleaf - 1 - (lane >> 2)];
                    if ((uint32_t)(lane & 3) <= e >> 20) {
                        et = (int)(e & 0xfffffu) + (lane & 3);
                        const float4 c = m.tris[4 * (size_t)et + 2], d = m.tris[4 * (size_t)et + 3];
                        elo[0] = c.y; elo[1] = c.z; elo[2] = c.w;
                        ehi[0] = d.x; ehi[1] = d.y; ehi[2] = d.z;
                        meet = boxes_overlap(elo, ehi, blo, bhi);
                    }
                }
                nleaf -= n;
                tris = __ballot(meet);
            } else if (nopen > 0) {
                do {
                    const int n = nopen > kStackSoft ? 1 : min(nopen, kOpenNodes);
                    bool inner = false, leaf = false;
                    int a = 0, b = 0;
                    const int o = lane / kWide;
                    if (o < n) {
                        const float4* src =
                            m.slots + 2 * (kWide * (size_t)w.stack[nopen - 1 - o] + (lane & (kWide - 1)));
                        const float4 lo = src[0], hi = src[1];
                        a = (int)__float_as_uint(lo.w);
                        b = (int)__float_as_uint(hi.w);
                        const float slo[3] = {lo.x, lo.y, lo.z}, shi[3] = {hi.x, hi.y, hi.z};
                        const bool meet = boxes_overlap(slo, shi, blo, bhi);
                        inner = meet && b > 0;
                        leaf = meet && b < 0;
                    }
                    __syncthreads();  // the entries are read before new ones take their places
                    nopen -= n;
                    const int at = take_slot(inner, nopen);
                    if (inner) w.stack[at] = a;
                    const int al = take_slot(leaf, nleaf);
                    if (leaf) w.leaf[al] = (uint32_t)a | (uint32_t)(-b - 1) << 20;
                    __syncthreads();
                } while (nopen > 0 && nleaf <= 64);
            } else {
                break;
            }
        }
    }
    return false;
}

__global__ __launch_bounds__(64) void mesh_valid(MeshArgs m, const double* __restrict__ q, int64_t n,
                                                 uint8_t* __restrict__ ok) {
    __shared__ MeshLists lists;
    for (int64_t i = blockIdx.x; i < n; i += gridDim.x) {
        double s[7];
#pragma unroll
        for (int j = 0; j < 7; ++j) s[j] = q[i * 7 + j];
        const bool hit = mesh_collides(m, pose_from_state(s), lists);
        if (threadIdx.x == 0) ok[i] = hit ? 0 : 1;
    }
}

__global__ __launch_bounds__(64) void mesh_filter(MeshArgs m, const double* __restrict__ q, int64_t n,
                                                  uint8_t* __restrict__ mask, uint8_t* __restrict__ status,
                                                  int invalid_code) {
    __shared__ MeshLists lists;
    for (int64_t i = blockIdx.x; i < n; i += gridDim.x) {
        if (!mask[i]) continue;
        double s[7];
#pragma unroll
        for (int j = 0; j < 7; ++j) s[j] = q[i * 7 + j];
        const bool hit = mesh_collides(m, pose_from_state(s), lists);
        if (threadIdx.x == 0 && hit) {
            mask[i] = 0;
            status[i] = (uint8_t)invalid_code;
        }
    }
}

// DMV link (src/mpt/discrete_motion_validator.hpp:71-130) of n edges: one wave
// checks one waypoint at a time.  The check sequence of an edge is valid(to)
// at position 0 (counted even when vouched for, as the reference's validator
// counts it), then the DMV waypoints in table order at positions 1..mw.
//
// mesh_link_prepare lists the live edges with their waypoint counts and sets
// their slots in `checks` to ~0.  mesh_link deals (position, edge) items,
// positions before edges, to its waves in turn; a wave tests 64 of its items
// at once (not past the edge's last waypoint, nor past a position that has
// failed already), each lane interpolates the pose of its own item, and the
// wave checks those left one by one.  A failure lowers the edge's slot to its
// position with atomicMin; every position below the final slot has been
// checked, so it ends at exactly the first failing one.  No wave waits for
// another.  mesh_link_finish turns the slots into verdicts and
// check counts.
//
// Dealt this way a wave meets other edges from item to item.  When P waves
// shared an edge's waypoints (2 of 8192 waves for 4096 edges), the waves of
// the few long free edges checked up to a dozen waypoints in series while the
// other waves had ended, and a larger P checked waypoints past failures; and
// every lane of a wave computed the one pose, which was half of the registers.
// 4096 edges, 19 700 counted checks against 50 000 triangles: 315 us that way,
// 197 dealt out, 111 with the present mesh_collides (64 waves dealt to each CU:
// 128, 111 and 123 us for 32, 64 and 128).  Storing the poses in the prepare
// kernel instead took no less (its atomics, one wave per four edges, were as
// long as the interpolation).
//
// Edges beyond 255 waypoints replay the 256-slot ring on one wave, 64 indices
// at a time.
struct MeshWork {
    uint32_t n_live, max_mw;  // zero between calls (mesh_link_finish clears them)
};
constexpr size_t kMeshWorkBytes = 256;

__device__ __forceinline__ int64_t mesh_waypoints(const SpaceArgs& sp, const double* a, const double* b, double inv) {
    const double x = __builtin_ceil(space_dist(sp, a, b) * inv);
    int64_t steps = 0;
    if (x >= 2.0) steps = x < 0x1.0p62 ? (int64_t)x : ((int64_t)1 << 62);
    return steps > 0 ? steps - 1 : 0;
}

__global__ __launch_bounds__(256) void mesh_link_prepare(SpaceArgs sp, double inv, const double* __restrict__ from,
                                                         const double* __restrict__ to, int64_t n,
                                                         int known_valid, const uint8_t* __restrict__ mask,
                                                         uint32_t* __restrict__ slot, MeshWork* __restrict__ work, uint2* __restrict__ live) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int lane = threadIdx.x & 63;
    int mw = -1;
    if (e < n) {
        slot[e] = 0xffffffffu;
        if (!mask || mask[e]) {
            double a[7], b[7];
#pragma unroll
            for (int j = 0; j < 7; ++j) {
                a[j] = from[e * 7 + j];
                b[j] = to[e * 7 + j];
            }
            const int64_t w = mesh_waypoints(sp, a, b, inv);
            // over the limit: valid(to) alone is checked; if it holds, the
            // finish kernel reports the edge
            if (w <= kMaxDmvWaypointsMesh) mw = (int)w;
            else if (!known_valid) mw = 0;
        }
    }
    const uint64_t m = __ballot(mw >= 0);
    if (m == 0) return;
    int most = mw;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) most = max(most, __shfl_xor(most, o));
    uint32_t base = 0;
    if (lane == 0) {
        base = atomicAdd(&work->n_live, (uint32_t)__popcll(m));
        atomicMax(&work->max_mw, (uint32_t)min(most, kTableMaxMesh));  // a ring edge is one item
    }
    base = __builtin_amdgcn_readfirstlane(base);
    if (mw >= 0) live[base + __popcll(m & ((1ull << lane) - 1ull))] = make_uint2((uint32_t)e, (uint32_t)mw);
}

// The next indices of an edge's 256-slot ring, in check order (lane 0).
struct MeshRing {
    uint64_t rmin[256], rmax[256], emitted[64];
    uint64_t qs, qe, seq_cur, seq_end;
    int seq, count, mw;

    __device__ void start(int waypoints) {
        mw = waypoints;
        rmin[0] = 1;
        rmax[0] = (uint64_t)waypoints;
        qs = 0;
        qe = 1;
        seq = 0;
    }
    __device__ void emit() {
        int c = 0;
        while (c < 64 && (seq || qs != qe)) {
            if (seq) {
                emitted[c++] = seq_cur;
                if (seq_cur == seq_end) seq = 0;
                else ++seq_cur;
                continue;
            }
            const uint64_t mn = rmin[qs % 256], mx = rmax[qs % 256];
            ++qs;
            if (mn == mx) {
                emitted[c++] = mn;
            } else if (qe + 2 < qs + 256) {
                const uint64_t mid = (mn + mx) / 2;
                emitted[c++] = mid;
                if (mn < mid) {
                    rmin[qe % 256] = mn;
                    rmax[qe % 256] = mid - 1;
                    ++qe;
                }
                if (mid < mx) {
                    rmin[qe % 256] = mid + 1;
                    rmax[qe % 256] = mx;
                    ++qe;
                }
            } else {
                seq = 1;
                seq_cur = mn;
                seq_end = mx;
            }
        }
        count = c;
    }
};

__device__ __forceinline__ Pose32 lane_pose(const Pose32& p, int src) {
    Pose32 o;
#pragma unroll
    for (int i = 0; i < 9; ++i) o.r[i] = lane_f32(p.r[i], src);
#pragma unroll
    for (int i = 0; i < 3; ++i) o.t[i] = lane_f32(p.t[i], src);
    return o;
}

// Four waves per SIMD: 127 registers, none spilled (five waves spill 32).
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) void mesh_link(
    SpaceArgs sp, MeshArgs m, const uint8_t* __restrict__ table, const double* __restrict__ from,
    const double* __restrict__ to, int known_valid, const MeshWork* __restrict__ work,
    const uint2* __restrict__ live, uint32_t* __restrict__ slot) {
    __shared__ MeshLists lists;
    __shared__ MeshRing ring;
    const int lane = threadIdx.x;
    const uint32_t pos0 = known_valid ? 1u : 0u;  // the first position checked
    uint64_t first = blockIdx.x;
    // this lane's item of the batch: edge, waypoint count, position
    uint32_t my_e = 0, my_pos = 0;
    int my_mw = 0;
    uint64_t rings = 0;  // the batch's items that are whole edges with a ring
    bool in_ring = false;
    uint32_t ring_e = 0, ring_at = 0;  // the edge in the ring, and its next position
    while (true) {
        // a batch of up to 64 positions, a lane each: `todo`
        bool want = false;
        uint32_t e = 0, pos = 0;
        int mw = 0;
        uint64_t index = 0;  // the waypoint, 0: valid(to)
        if (in_ring) {
            __syncthreads();  // the indices emitted last have been read
            if (lane == 0) ring.emit();
            __syncthreads();
            const int c = ring.count;
            if (c == 0) {
                in_ring = false;
                continue;
            }
            want = lane < c;
            e = ring_e;
            mw = ring.mw;
            pos = ring_at + (uint32_t)lane;
            index = want ? ring.emitted[lane] : 0;
            ring_at += (uint32_t)c;
        } else if (rings) {
            const int src = __builtin_ctzll(rings);
            rings &= rings - 1;
            in_ring = true;
            ring_e = (uint32_t)__builtin_amdgcn_readlane((int)my_e, src);
            ring_at = 1;
            __syncthreads();
            if (lane == src) ring.start(my_mw);
            __syncthreads();
            if (known_valid) continue;
            want = lane == 0;  // valid(to) first
            e = ring_e;
            mw = ring.mw;
        } else {
            const uint64_t n_live = work->n_live;
            const uint64_t items = n_live * ((uint64_t)work->max_mw + 1u - pos0);
            if (first >= items) break;
            const uint64_t it = first + (uint64_t)lane * gridDim.x;
            first += (uint64_t)gridDim.x * 64;
            bool whole = false;
            if (it < items) {
                const uint64_t row = items < (1ull << 32) ? (uint64_t)((uint32_t)it / (uint32_t)n_live) : it / n_live;
                const uint2 le = live[it - row * n_live];
                my_e = le.x;
                my_mw = (int)le.y;
                my_pos = (uint32_t)row + pos0;
                whole = my_mw > kTableMaxMesh && my_pos == pos0;
                want = my_mw <= kTableMaxMesh && my_pos <= (uint32_t)my_mw && slot[my_e] >= my_pos;
            }
            rings = __ballot(whole);
            e = my_e;
            mw = my_mw;
            pos = my_pos;
            if (want && pos > 0) index = table[((int64_t)mw * (mw - 1)) / 2 + pos - 1];
        }
        Pose32 pose{};
        if (want) {
            double a[7], b[7], q[7];
#pragma unroll
            for (int j = 0; j < 7; ++j) {
                a[j] = from[(int64_t)e * 7 + j];
                b[j] = to[(int64_t)e * 7 + j];
                q[j] = b[j];
            }
            if (index > 0) space_interp(sp, a, b, (double)index * (1.0 / (double)(mw + 1)), q);
            pose = pose_from_state(q);
        }
        for (uint64_t todo = __ballot(want); todo; todo &= todo - 1) {  // wave-uniform, in position order
            const int src = __builtin_ctzll(todo);
            const uint32_t ee = (uint32_t)__builtin_amdgcn_readlane((int)e, src);
            const uint32_t pp = (uint32_t)__builtin_amdgcn_readlane((int)pos, src);
            // an earlier position has failed meanwhile
            if ((uint32_t)__builtin_amdgcn_readfirstlane(
                    (int)__hip_atomic_load(&slot[ee], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) < pp)
                continue;
            if (mesh_collides(m, lane_pose(pose, src), lists)) {
                if (lane == 0) atomicMin(&slot[ee], pp);
                if (in_ring) {
                    in_ring = false;
                    break;
                }
            }
        }
    }
}

// Verdicts and check counts of the edges from their slots.
__global__ __launch_bounds__(256) void mesh_link_finish(SpaceArgs sp, double inv, const double* __restrict__ from,
                                                        const double* __restrict__ to, int64_t n,
                                                        const uint8_t* __restrict__ mask,
                                                        uint8_t* __restrict__ verdict, uint32_t* __restrict__ checks,
                                                        MeshWork* __restrict__ work) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e == 0) work->n_live = work->max_mw = 0;
    if (e >= n || (mask && !mask[e])) return;
    const uint32_t s = checks[e];
    if (s != 0xffffffffu) {
        verdict[e] = 0;
        checks[e] = s + 1u;
        return;
    }
    double a[7], b[7];
#pragma unroll
    for (int j = 0; j < 7; ++j) {
        a[j] = from[e * 7 + j];
        b[j] = to[e * 7 + j];
    }
    const int64_t mw = mesh_waypoints(sp, a, b, inv);
    if (mw > kMaxDmvWaypointsMesh) {
        verdict[e] = 0;
        checks[e] = MPTG_CHECKS_OVER_LIMIT;
    } else {
        verdict[e] = 1;
        checks[e] = (uint32_t)(1 + mw);
    }
}

}  // namespace

// Triangles of a lane's group: as few as give every lane a group, and at most
// eight (their box is then that of the best part of a box of the robot's).
static int group_shift(int nrobot) {
    int sh = 0;
    while (sh < kGroupShift && (64 << sh) < nrobot) ++sh;
    return sh;
}
// The groups' boxes follow the robot's triangles, 16-byte aligned (floats).
static size_t group_offset(int nrobot) { return ((size_t)nrobot * 9 + 3) / 4 * 4; }

MeshArgs mesh_args(const mptg_ctx* ctx) {
    const SceneDev& s = ctx->scene;
    return MeshArgs{(const float4*)s.mesh_nodes.p, (const float4*)s.mesh_tris.p,
                    (const float*)s.mesh_robot.p,  (const float4*)((const float*)s.mesh_robot.p + group_offset(s.mesh_nrobot)),
                    s.mesh_nnodes, s.mesh_nrobot, group_shift(s.mesh_nrobot), s.mesh_reach, s.mesh_env_reach};
}

int launch_mesh_valid(mptg_ctx* ctx, const double* d_q, int64_t n, uint8_t* d_ok) {
    if (n <= 0) return MPTG_OK;
    const unsigned g = (unsigned)std::min<int64_t>(n, (int64_t)ctx->cus * ctx->tune.mesh_waves_per_cu);
    hipLaunchKernelGGL(mesh_valid, dim3(g), dim3(64), 0, ctx->stream, mesh_args(ctx), d_q, n, d_ok);
    MPTG_HIP(ctx, hipGetLastError());
    return MPTG_OK;
}

int launch_mesh_filter(mptg_ctx* ctx, const double* d_states, int64_t n, uint8_t* d_mask, uint8_t* d_status,
                       int invalid_code) {
    if (n <= 0) return MPTG_OK;
    const unsigned g = (unsigned)std::min<int64_t>(n, (int64_t)ctx->cus * ctx->tune.mesh_waves_per_cu);
    hipLaunchKernelGGL(mesh_filter, dim3(g), dim3(64), 0, ctx->stream, mesh_args(ctx), d_states, n, d_mask, d_status,
                       invalid_code);
    MPTG_HIP(ctx, hipGetLastError());
    return MPTG_OK;
}

int launch_mesh_link(mptg_ctx* ctx, const uint8_t* d_table, const double* d_from, const double* d_to, int64_t n,
                     int known_valid, const uint8_t* d_mask, uint8_t* d_verdict, uint32_t* d_checks) {
    if (n <= 0) return MPTG_OK;
    int rc;
    DevBuf& buf = ctx->scratch[10];
    const size_t need = kMeshWorkBytes + sizeof(uint2) * (size_t)n;
    if (!buf.p || buf.bytes < need) ctx->link_lists_clean = false;
    if ((rc = ensure(ctx, buf, need))) return rc;
    MeshWork* work = (MeshWork*)buf.p;
    uint2* live = (uint2*)((char*)buf.p + kMeshWorkBytes);
    if (!ctx->link_lists_clean && (rc = launch_zero_u32(ctx, (uint32_t*)work, kMeshWorkBytes / 4))) return rc;
    const bool was_clean = ctx->link_lists_clean;
    ctx->link_lists_clean = false;  // until every kernel is enqueued
    const unsigned g1 = (unsigned)((n + 255) / 256);
    hipLaunchKernelGGL(mesh_link_prepare, dim3(g1), dim3(256), 0, ctx->stream, space_args(ctx), 1.0 / ctx->link_param,
                       d_from, d_to, n, known_valid, d_mask, d_checks, work, live);
    // waves: as many as the device holds, or 256 per edge (every waypoint of
    // a short edge at once) in a batch too small for that (the rewire pass's
    // late batches hold a few edges)
    const unsigned gp = (unsigned)std::min<int64_t>(n * 256, (int64_t)ctx->cus * ctx->tune.mesh_waves_per_cu);
    hipLaunchKernelGGL(mesh_link, dim3(gp), dim3(64), 0, ctx->stream, space_args(ctx), mesh_args(ctx), d_table,
                       d_from, d_to, known_valid, (const MeshWork*)work, (const uint2*)live, d_checks);
    hipLaunchKernelGGL(mesh_link_finish, dim3(g1), dim3(256), 0, ctx->stream, space_args(ctx), 1.0 / ctx->link_param,
                       d_from, d_to, n, d_mask, d_verdict, d_checks, work);
    MPTG_HIP(ctx, hipGetLastError());
    ctx->link_lists_clean = was_clean || !stream_capturing(ctx);
    return MPTG_OK;
}

}  // namespace mptg

using namespace mptg;

extern "C" int mptg_scene_mesh(mptg_ctx* ctx, const float* h_robot, int nrobot, const float* h_env, int nenv) {
    int rc = check_device_ready(ctx);
    if (rc) return rc;
    if (ctx->metric != MPTG_METRIC_SE3) return fail(ctx, MPTG_E_STATE, "mesh scenes need the SE3 space");
    if (nrobot < 0 || nenv < 0 || (nrobot > 0 && !h_robot) || (nenv > 0 && !h_env))
        return fail(ctx, MPTG_E_ARG, "bad mesh arrays");
    if (nenv > (1 << 20)) return fail(ctx, MPTG_E_RANGE, "at most 2^20 environment triangles");
    if (nrobot > (1 << 16)) return fail(ctx, MPTG_E_RANGE, "at most 2^16 robot triangles");
    auto finite = [](const float* v, int64_t n) {  // without a branch per value
        int bad = 0;
        for (int64_t i = 0; i < n; ++i) bad |= !(std::fabs(v[i]) < INFINITY);
        return !bad;
    };
    if (!finite(h_robot, (int64_t)nrobot * 9)) return fail(ctx, MPTG_E_ARG, "non-finite robot vertex");
    if (!finite(h_env, (int64_t)nenv * 9)) return fail(ctx, MPTG_E_ARG, "non-finite environment vertex");
    // environment BVH
    BvhBuilder bb;
    bb.refs.resize((size_t)nenv);
    for (int t = 0; t < nenv; ++t) {
        BuildRef& r = bb.refs[(size_t)t];
        tri_box(h_env + (size_t)t * 9, r.lo, r.hi);
        for (int i = 0; i < 3; ++i) r.c[i] = 0.5f * (r.lo[i] + r.hi[i]);
        r.id = t;
    }
    bb.nodes.reserve((size_t)nenv + 1);
    if (nenv > 0) bb.build(0, nenv, 0);
    if (nenv > 0 && bvh_depth(bb.nodes, 0, 0) > kBuildDepth)
        return fail(ctx, MPTG_E_STATE, "environment BVH deeper than the traversal stack");
    std::vector<float> tris((size_t)nenv * kTriFloats, 0.0f);
    for (int i = 0; i < nenv; ++i) {
        const BuildRef& r = bb.refs[(size_t)i];
        float* d = &tris[(size_t)i * kTriFloats];
        std::memcpy(d, h_env + (size_t)r.id * 9, 9 * sizeof(float));
        for (int k = 0; k < 3; ++k) {
            d[9 + k] = r.lo[k];
            d[12 + k] = r.hi[k];
        }
    }
    // robot: Morton order of triangle centroids
    std::vector<float> robot((size_t)nrobot * 9);
    {
        float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
        std::vector<float> cen((size_t)nrobot * 3);
        for (int t = 0; t < nrobot; ++t)
            for (int i = 0; i < 3; ++i) {
                const float* v = h_robot + (size_t)t * 9;
                float c = (v[i] + v[3 + i] + v[6 + i]) / 3.0f;
                cen[(size_t)t * 3 + i] = c;
                lo[i] = std::min(lo[i], c);
                hi[i] = std::max(hi[i], c);
            }
        std::vector<std::pair<uint32_t, int>> key((size_t)nrobot);
        for (int t = 0; t < nrobot; ++t) {
            uint32_t code = 0;
            for (int i = 0; i < 3; ++i) {
                float ext = hi[i] - lo[i];
                uint32_t qv = ext > 0 ? (uint32_t)std::min(1023.0f, (cen[(size_t)t * 3 + i] - lo[i]) / ext * 1023.0f) : 0;
                code |= spread10(qv) << i;
            }
            key[(size_t)t] = {code, t};
        }
        std::sort(key.begin(), key.end());
        for (int t = 0; t < nrobot; ++t)
            std::memcpy(&robot[(size_t)t * 9], h_robot + (size_t)key[(size_t)t].second * 9, 9 * sizeof(float));
    }
    // the groups' boxes, 8 floats each
    const int sh = group_shift(nrobot);
    const int ngroup = (nrobot + (1 << sh) - 1) >> sh;
    robot.resize(group_offset(nrobot) + 8 * (size_t)ngroup, 0.0f);
    float reach = 0.0f;
    for (int g = 0; g < ngroup; ++g) {
        const int t1 = std::min(nrobot, (g + 1) << sh);
        float* o = &robot[group_offset(nrobot) + 8 * (size_t)g];
        float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
        for (int v = 3 * (g << sh); v < 3 * t1; ++v) BvhBuilder::grow(lo, hi, &robot[3 * (size_t)v], &robot[3 * (size_t)v]);
        for (int i = 0; i < 3; ++i) {
            reach = std::max({reach, std::fabs(lo[i]), std::fabs(hi[i])});
            const float c = 0.5f * lo[i] + 0.5f * hi[i];
            o[i] = c;
            o[4 + i] = std::nextafter(std::max(hi[i] - c, c - lo[i]), INFINITY);
        }
    }
    SceneDev& s = ctx->scene;
    MPTG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    std::vector<MeshNode16> wide;
    wide.reserve(bb.nodes.size() / 8 + 1);
    if (!bb.nodes.empty()) collapse16(bb.nodes, 0, wide);
    if ((rc = ensure(ctx, s.mesh_nodes, sizeof(MeshNode16) * std::max<size_t>(1, wide.size())))) return rc;
    if ((rc = ensure(ctx, s.mesh_tris, sizeof(float) * std::max<size_t>(16, tris.size())))) return rc;
    if ((rc = ensure(ctx, s.mesh_robot, sizeof(float) * std::max<size_t>(9, robot.size())))) return rc;
    if (!wide.empty())
        MPTG_HIP(ctx, hipMemcpy(s.mesh_nodes.p, wide.data(), sizeof(MeshNode16) * wide.size(),
                                hipMemcpyHostToDevice));
    if (!tris.empty())
        MPTG_HIP(ctx, hipMemcpy(s.mesh_tris.p, tris.data(), sizeof(float) * tris.size(), hipMemcpyHostToDevice));
    if (!robot.empty())
        MPTG_HIP(ctx, hipMemcpy(s.mesh_robot.p, robot.data(), sizeof(float) * robot.size(), hipMemcpyHostToDevice));
    s.mesh_nnodes = (int)wide.size();
    s.mesh_nrobot = nrobot;
    s.mesh_reach = reach;
    s.mesh_env_reach = 0;
    if (!bb.nodes.empty())
        for (int i = 0; i < 3; ++i)
            s.mesh_env_reach = std::max({s.mesh_env_reach, std::fabs(bb.nodes[0].lo[i]), std::fabs(bb.nodes[0].hi[i])});
    s.kind = MPTG_SCENE_MESH;
    ctx->valid_upto = 0;  // valid() changed: every node is checked again
    ctx->some_invalid = false;
    return MPTG_OK;
}
