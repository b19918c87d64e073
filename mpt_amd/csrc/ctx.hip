// Context lifecycle, space/tree/scene state and the host-pointer entry points.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "internal.hpp"
#include "space_dev.hpp"

namespace mptg {

thread_local std::string g_create_err;
void prrt_free(mptg_ctx* ctx);
void surrogate_free(mptg_ctx* ctx);

namespace {
__global__ __launch_bounds__(256) void zero_u32_kernel(uint32_t* __restrict__ p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0u;
}
}  // namespace

int launch_zero_u32(mptg_ctx* ctx, uint32_t* p, int64_t n) {
    if (n <= 0) return MPTG_OK;
    hipLaunchKernelGGL(zero_u32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream, p, n);
    MPTG_HIP(ctx, hipGetLastError());
    return MPTG_OK;
}

int ensure(mptg_ctx* ctx, DevBuf& b, size_t bytes) {
    if (b.bytes >= bytes && b.p) return MPTG_OK;
    if (ctx->capturing) return fail(ctx, MPTG_E_STATE, "device buffer would grow during graph capture");
    if (b.p) {
        MPTG_HIP(ctx, hipStreamSynchronize(ctx->stream));
        MPTG_HIP(ctx, hipFree(b.p));
        b.p = nullptr;
        b.bytes = 0;
    }
    ++ctx->epoch;
    size_t want = std::max<size_t>(bytes, 256);
    MPTG_HIP(ctx, hipMalloc(&b.p, want));
    b.bytes = want;
    return MPTG_OK;
}

bool stream_capturing(const mptg_ctx* ctx) {
    if (ctx->capturing) return true;
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(ctx->stream, &st) == hipSuccess && st != hipStreamCaptureStatusNone;
}

int ensure_pinned(mptg_ctx* ctx, size_t bytes) {
    if (ctx->pinned_bytes >= bytes) return MPTG_OK;
    if (ctx->pinned) {
        MPTG_HIP(ctx, hipStreamSynchronize(ctx->stream));
        MPTG_HIP(ctx, hipHostFree(ctx->pinned));
        ctx->pinned = nullptr;
        ctx->pinned_bytes = 0;
    }
    size_t want = std::max<size_t>(bytes, 1 << 16);
    MPTG_HIP(ctx, hipHostMalloc(&ctx->pinned, want, hipHostMallocDefault));
    ctx->pinned_bytes = want;
    return MPTG_OK;
}

int check_device(mptg_ctx* ctx) {
    if (!ctx) return fail(nullptr, MPTG_E_ARG, "null context");
    MPTG_HIP(ctx, hipSetDevice(ctx->device));
    return MPTG_OK;
}

int check_device_ready(mptg_ctx* ctx) {
    if (ctx) ++ctx->epoch;  // the entry point may change what a captured graph holds
    return check_device(ctx);
}

static void free_tree(mptg_ctx* ctx) {
    (void)hipFree(ctx->x64);
    (void)hipFree(ctx->x32);
    (void)hipFree(ctx->parent);
    (void)hipFree(ctx->cost);
    (void)hipFree(ctx->child);
    ctx->x64 = nullptr;
    ctx->x32 = nullptr;
    ctx->parent = nullptr;
    ctx->cost = nullptr;
    ctx->child = ctx->next = ctx->prev = nullptr;
    ctx->cap = 0;
}

static int grow_tree(mptg_ctx* ctx, int64_t cap) {
    if (cap <= ctx->cap) return MPTG_OK;
    ++ctx->epoch;
    int d = ctx->dim, dp = pitch32(d);
    double* x64 = nullptr;
    float* x32 = nullptr;
    int32_t* par = nullptr;
    double* cost = nullptr;
    int32_t* links = nullptr;
    MPTG_HIP(ctx, hipMalloc(&x64, sizeof(double) * d * cap));
    MPTG_HIP(ctx, hipMalloc(&x32, sizeof(float) * dp * cap));
    MPTG_HIP(ctx, hipMalloc(&par, sizeof(int32_t) * cap));
    MPTG_HIP(ctx, hipMalloc(&cost, sizeof(double) * cap));
    MPTG_HIP(ctx, hipMalloc(&links, sizeof(int32_t) * 3 * cap));
    // zero the FP32 pad columns once so every row is fully defined
    MPTG_HIP(ctx, hipMemsetAsync(x32, 0, sizeof(float) * dp * cap, ctx->stream));
    if (ctx->size > 0) {
        const size_t n = (size_t)ctx->size;
        MPTG_HIP(ctx, hipMemcpyAsync(x64, ctx->x64, sizeof(double) * d * n, hipMemcpyDeviceToDevice, ctx->stream));
        MPTG_HIP(ctx, hipMemcpyAsync(x32, ctx->x32, sizeof(float) * dp * n, hipMemcpyDeviceToDevice, ctx->stream));
        MPTG_HIP(ctx, hipMemcpyAsync(par, ctx->parent, sizeof(int32_t) * n, hipMemcpyDeviceToDevice, ctx->stream));
        MPTG_HIP(ctx, hipMemcpyAsync(cost, ctx->cost, sizeof(double) * n, hipMemcpyDeviceToDevice, ctx->stream));
        for (int l = 0; l < 3; ++l)
            MPTG_HIP(ctx, hipMemcpyAsync(links + l * cap, ctx->child + l * ctx->cap, sizeof(int32_t) * n,
                                         hipMemcpyDeviceToDevice, ctx->stream));
    }
    MPTG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    free_tree(ctx);
    ctx->x64 = x64;
    ctx->x32 = x32;
    ctx->parent = par;
    ctx->cost = cost;
    ctx->child = links;
    ctx->next = links + cap;
    ctx->prev = links + 2 * cap;
    ctx->cap = cap;
    return MPTG_OK;
}

int tree_reserve(mptg_ctx* ctx, int64_t cap) {
    if (ctx->dim <= 0) return fail(ctx, MPTG_E_STATE, "mptg_space must be called before the tree is used");
    if (cap < 0 || cap > (int64_t)INT32_MAX) return fail(ctx, MPTG_E_RANGE, "tree capacity must be < 2^31");
    if (cap <= ctx->cap) return MPTG_OK;
    int64_t c = std::max<int64_t>(cap, std::min<int64_t>((int64_t)INT32_MAX, ctx->cap * 2));
    return grow_tree(ctx, c);
}

// Disk lists of the arm's FP32 clearance bounds (arm_near.hpp): per cell of an
// n x n grid over the square the joints can reach, every disk a link whose
// midpoint lies in the cell may touch, with the squared distances below and
// above which the FP32 test is certain.  A cell inside a disk by more than the
// margins needs that disk alone: every such link hits it.
//
// A wave per cell, sixteen to a block: one pass over the disks counts (or finds
// a disk around the cell), an atomic add takes the block's place in the lists
// (one per cell, on the one address, took 30 us), a second pass writes the
// entries.  Built on the host and copied in three pieces the lists took two
// thirds of a scene's upload (20 links, 200 disks: 60 us without them, 180
// with; 5000 disks 0.62 and 2.2 ms; 3000 disks that each reach most cells 0.31
// and 13 ms; now, with one copy for the rest and a counting sort, 41 us, 0.27
// and 0.11 ms).
struct NearBuild {
    const ArmDisk* disks;
    int ndisks, n;
    double T, longest;  // all links, the longest
    uint32_t cap;       // entries there is room for
    uint32_t* total;    // entries there are
    uint2* cells;
    float4* out;
    int32_t* ids;
};

constexpr int kNearWaves = 16;
__global__ __launch_bounds__(64 * kNearWaves) void near_lists(NearBuild B) {
    __shared__ uint32_t counts[kNearWaves], first;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int cell = (int)blockIdx.x * kNearWaves + w;
    const bool have = cell < B.n * B.n;
    const int ndisks = have ? B.ndisks : 0;
    const double size = 2.0 * B.T / B.n;
    const double lx = -B.T + (cell % B.n) * size, ly = -B.T + (cell / B.n) * size;
    auto margin = [&](const ArmDisk& d) { return kNearMargin * (B.T + B.longest + d.rt); };
    auto near = [&](const ArmDisk& d, bool* around) {
        // the midpoint's error is a joint's; its cell coordinate's FP32
        // rounding is within 1e-6 T; rounding here and in the exact
        // expression is below 1e-12 r
        const double slack = 2.0 * margin(d) + 8e-6 * B.T;
        const double reach = B.longest / 2 + d.rt + slack, inside = d.rt - slack;
        const double x0 = lx - d.cx, x1 = d.cx - (lx + size), y0 = ly - d.cy, y1 = d.cy - (ly + size);
        const double gx = __builtin_fmax(__builtin_fmax(x0, x1), 0.0), gy = __builtin_fmax(__builtin_fmax(y0, y1), 0.0);
        const double fx = __builtin_fmax(-x0, -x1), fy = __builtin_fmax(-y0, -y1);  // to the farthest corner
        *around = inside > 0.0 && fx * fx + fy * fy < inside * inside;
        return gx * gx + gy * gy <= reach * reach;
    };
    auto entry = [&](uint32_t at, int i, const ArmDisk& d) {
        const double lo = __builtin_fmax(d.rt - margin(d), 0.0), hi = d.rt + margin(d);
        B.ids[at] = i;
        B.out[at] = make_float4((float)d.cx, (float)d.cy, __double2float_rd(lo * lo), __double2float_ru(hi * hi));
    };
    uint32_t count = 0;
    int alone = -1;
    for (int i0 = 0; i0 < ndisks && alone < 0; i0 += 64) {
        const int i = i0 + lane;
        bool around = false;
        const bool take = i < ndisks && near(B.disks[i], &around);
        const uint64_t a = __ballot(around);
        if (a) alone = i0 + (int)__builtin_ctzll(a);
        count += (uint32_t)__popcll(__ballot(take));
    }
    if (alone >= 0) count = 1;
    if (lane == 0) counts[w] = count;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t sum = 0;
        for (int v = 0; v < kNearWaves; ++v) sum += counts[v];
        first = atomicAdd(B.total, sum);
    }
    __syncthreads();
    uint32_t base = first;
    for (int v = 0; v < w; ++v) base += counts[v];
    base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
    if (lane == 0 && have) B.cells[cell] = make_uint2(base, count);
    if (base + count > B.cap) return;  // no room: the caller reads the total
    if (alone >= 0) {
        if (lane == 0) entry(base, alone, B.disks[alone]);
        return;
    }
    for (int i0 = 0; i0 < ndisks; i0 += 64) {
        const int i = i0 + lane;
        bool around = false;
        const ArmDisk d = B.disks[i < ndisks ? i : 0];
        const bool take = i < ndisks && near(d, &around);
        const uint64_t m = __ballot(take);
        if (take) entry(base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull)), i, d);
        base += (uint32_t)__popcll(m);
    }
}

// Builds the lists; *more: they did not fit, call again with the *entries there
// are.  near_n = 0 (no lists) for arms and disks outside the bounds'
// assumptions, and for lists past kNearMaxEntries.
static int build_near(mptg_ctx* ctx, const double* len, int nlinks, const double* disks, int ndisks,
                      uint32_t* entries, bool* more) {
    SceneDev& s = ctx->scene;
    *more = false;
    s.near_n = 0;
    double T = 0.0, longest = 0.0, rmax = 0.0;
    for (int i = 0; i < nlinks; ++i) {
        if (!(len[i] >= 0.0) || !std::isfinite(len[i])) return MPTG_OK;
        T += len[i];
        longest = std::max(longest, len[i]);
    }
    for (int i = 0; i < ndisks; ++i) {
        const double* d = &disks[4 * (size_t)i];
        if (!std::isfinite(d[0]) || !std::isfinite(d[1]) || !(d[3] >= 0.0) || !std::isfinite(d[3])) return MPTG_OK;
        rmax = std::max(rmax, d[3]);
    }
    // the FP32 squares stay clear of overflow and of denormals
    if (!(T > kNearLeast) || !(T + rmax < kNearMost)) return MPTG_OK;
    // cells half a link wide: the lists are then within a third of the
    // shortest possible, and 64 x 64 cells of the 20-link arm stay in L2
    const int n = std::max(1, std::min(kNearCells, (int)std::ceil(4.0 * T / longest)));
    // room for 64 cells a disk at first, then for the entries there are
    constexpr size_t kEntry = sizeof(float4) + sizeof(int32_t);
    const size_t cells = 256, out = cells + sizeof(uint2) * kNearCells * kNearCells;
    if (*entries > (uint32_t)kNearMaxEntries) return MPTG_OK;
    uint32_t cap = std::max<uint32_t>(*entries, (uint32_t)std::min<int64_t>(kNearMaxEntries, std::max<int64_t>(1 << 12, (int64_t)ndisks * 64)));
    if (s.near.bytes > out + kEntry * cap)
        cap = (uint32_t)std::min<size_t>((s.near.bytes - out) / kEntry, (size_t)kNearMaxEntries);
    const size_t ids = out + sizeof(float4) * (size_t)cap;
    int rc;
    if ((rc = ensure(ctx, s.near, ids + sizeof(int32_t) * (size_t)cap))) return rc;
    char* p = (char*)s.near.p;
    if ((rc = launch_zero_u32(ctx, (uint32_t*)p, 1))) return rc;
    NearBuild B{(const ArmDisk*)s.arm_disks, ndisks, n, T, longest, cap, (uint32_t*)p,
                (uint2*)(p + cells), (float4*)(p + out), (int32_t*)(p + ids)};
    hipLaunchKernelGGL(near_lists, dim3((unsigned)((n * n + kNearWaves - 1) / kNearWaves)), dim3(64 * kNearWaves), 0,
                       ctx->stream, B);
    MPTG_HIP(ctx, hipGetLastError());
    MPTG_HIP(ctx, hipMemcpyAsync(entries, p, sizeof(uint32_t), hipMemcpyDeviceToHost, ctx->stream));
    MPTG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (*entries > cap) {
        *more = true;
        return MPTG_OK;
    }
    s.near_n = n;
    s.near_extent = (float)T;
    s.near_inv = (float)(n / (2.0 * T));
    s.near_cells = B.cells;
    s.near_disks = B.out;
    s.near_ids = B.ids;
    return MPTG_OK;
}

}  // namespace mptg

using namespace mptg;

extern "C" {

int mptg_create(int device, mptg_ctx** out) {
    if (!out) return fail(nullptr, MPTG_E_ARG, "null output pointer");
    *out = nullptr;
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n == 0)
        return fail(nullptr, MPTG_E_HIP, std::string("no HIP device: ") + hipGetErrorString(e));
    if (device < 0 || device >= n) return fail(nullptr, MPTG_E_ARG, "device index out of range");
    e = hipSetDevice(device);
    if (e != hipSuccess) return fail(nullptr, MPTG_E_HIP, hipGetErrorString(e));
    mptg_ctx* ctx = new mptg_ctx();
    ctx->device = device;
    e = hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking);
    if (e != hipSuccess) {
        delete ctx;
        return fail(nullptr, MPTG_E_HIP, std::string("hipStreamCreate: ") + hipGetErrorString(e));
    }
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) == hipSuccess) ctx->cus = prop.multiProcessorCount;
    if (ctx->cus <= 0) ctx->cus = 256;
    *out = ctx;
    return MPTG_OK;
}

void mptg_destroy(mptg_ctx* ctx) {
    if (!ctx) return;
    (void)hipSetDevice(ctx->device);
    (void)hipStreamSynchronize(ctx->stream);
    for (hipEvent_t e : ctx->phase_ev)
        if (e) (void)hipEventDestroy(e);
    free_tree(ctx);
    (void)hipFree(ctx->scene.boxes);
    (void)hipFree(ctx->scene.grid);
    (void)hipFree(ctx->scene.circles);
    (void)hipFree(ctx->scene.arm.p);
    (void)hipFree(ctx->scene.near.p);
    (void)hipFree(ctx->scene.mesh_nodes.p);
    (void)hipFree(ctx->scene.mesh_tris.p);
    (void)hipFree(ctx->scene.mesh_robot.p);
    for (auto& b : ctx->scratch) (void)hipFree(b.p);
    (void)hipFree(ctx->dmv_table16.p);
    (void)hipFree(ctx->rnn_buf.p);
    (void)hipFree(ctx->rnn_pairs.p);
    (void)hipFree(ctx->rnn_q.p);
    (void)hipFree(ctx->rnn_out.p);
    for (auto& b : ctx->knn_sel) (void)hipFree(b.p);
    for (auto& b : ctx->knn_grid) (void)hipFree(b.p);
    prrt_free(ctx);
    surrogate_free(ctx);
    if (ctx->pinned) (void)hipHostFree(ctx->pinned);
    if (ctx->ev_start) (void)hipEventDestroy(ctx->ev_start);
    if (ctx->ev_stop) (void)hipEventDestroy(ctx->ev_stop);
    (void)hipStreamDestroy(ctx->stream);
    delete ctx;
}

const char* mptg_last_error(const mptg_ctx* ctx) {
    return ctx ? ctx->err.c_str() : g_create_err.c_str();
}

int mptg_sync(mptg_ctx* ctx) {
    int rc = check_device(ctx);
    if (rc) return rc;
    MPTG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return MPTG_OK;
}

void* mptg_stream(mptg_ctx* ctx) { return ctx ? (void*)ctx->stream : nullptr; }

int mptg_dev_alloc(mptg_ctx* ctx, uint64_t bytes, void** d_out) {
    int rc = check_device(ctx);
    if (rc) return rc;
    if (!d_out) return fail(ctx, MPTG_E_ARG, "null output pointer");
    *d_out = nullptr;
    MPTG_HIP(ctx, hipMalloc(d_out, bytes ? bytes : 1));
    return MPTG_OK;
}

int mptg_dev_free(mptg_ctx* ctx, void* d_ptr) {
    int rc = check_device(ctx);
    if (rc) return rc;
    MPTG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    MPTG_HIP(ctx, hipFree(d_ptr));
    return MPTG_OK;
}

int mptg_dev_upload(mptg_ctx* ctx, void* d_dst, const void* h_src, uint64_t bytes) {
    int rc = check_device(ctx);
    if (rc) return rc;
    if (bytes == 0) return MPTG_OK;
    MPTG_HIP(ctx, hipMemcpyAsync(d_dst, h_src, bytes, hipMemcpyHostToDevice, ctx->stream));
    MPTG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return MPTG_OK;
}

int mptg_dev_download(mptg_ctx* ctx, void* h_dst, const void* d_src, uint64_t bytes) {
    int rc = check_device(ctx);
    if (rc) return rc;
    if (bytes == 0) return MPTG_OK;
    MPTG_HIP(ctx, hipMemcpyAsync(h_dst, d_src, bytes, hipMemcpyDeviceToHost, ctx->stream));
    MPTG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return MPTG_OK;
}

int mptg_dev_memset(mptg_ctx* ctx, void* d_dst, int value, uint64_t bytes) {
    int rc = check_device(ctx);
    if (rc) return rc;
    if (bytes == 0) return MPTG_OK;
    MPTG_HIP(ctx, hipMemsetAsync(d_dst, value, bytes, ctx->stream));
    return MPTG_OK;
}

int mptg_timer_start(mptg_ctx* ctx) {
    int rc = check_device(ctx);
    if (rc) return rc;
    if (!ctx->ev_start) MPTG_HIP(ctx, hipEventCreate(&ctx->ev_start));
    if (!ctx->ev_stop) MPTG_HIP(ctx, hipEventCreate(&ctx->ev_stop));
    MPTG_HIP(ctx, hipEventRecord(ctx->ev_start, ctx->stream));
    return MPTG_OK;
}

int mptg_timer_stop(mptg_ctx* ctx, float* ms) {
    int rc = check_device(ctx);
    if (rc) return rc;
    if (!ctx->ev_start || !ms) return fail(ctx, MPTG_E_STATE, "mptg_timer_start was not called");
    MPTG_HIP(ctx, hipEventRecord(ctx->ev_stop, ctx->stream));
    MPTG_HIP(ctx, hipEventSynchronize(ctx->ev_stop));
    MPTG_HIP(ctx, hipEventElapsedTime(ms, ctx->ev_start, ctx->ev_stop));
    return MPTG_OK;
}

int mptg_space(mptg_ctx* ctx, int metric, int dim, double w0, double w1) {
    int rc = check_device_ready(ctx);
    if (rc) return rc;
    if (metric != MPTG_METRIC_L2 && metric != MPTG_METRIC_L1 && metric != MPTG_METRIC_SE3)
        return fail(ctx, MPTG_E_ARG, "unknown metric");
    if (metric == MPTG_METRIC_SE3 && dim != 7) return fail(ctx, MPTG_E_ARG, "SE3 states have 7 coordinates");
    if (dim < 1 || dim > kMaxDim) return fail(ctx, MPTG_E_ARG, "dimension must be in 1..32");
    if (metric == MPTG_METRIC_SE3 && !(w0 > 0 && w1 > 0)) return fail(ctx, MPTG_E_ARG, "SE3 weights must be > 0");
    if (ctx->size > 0 && (dim != ctx->dim || metric != ctx->metric))
        return fail(ctx, MPTG_E_STATE, "cannot change the space of a non-empty tree");
    if (dim != ctx->dim && ctx->x64) {
        MPTG_HIP(ctx, hipStreamSynchronize(ctx->stream));
        free_tree(ctx);
    }
    ctx->metric = metric;
    ctx->dim = dim;
    ctx->w_so3 = metric == MPTG_METRIC_SE3 ? w0 : 1.0;
    ctx->w_l2 = metric == MPTG_METRIC_SE3 ? w1 : 1.0;
    return MPTG_OK;
}

int mptg_tree_reserve(mptg_ctx* ctx, int64_t capacity) {
    int rc = check_device_ready(ctx);
    if (rc) return rc;
    return tree_reserve(ctx, capacity);
}

int mptg_tree_clear(mptg_ctx* ctx) {
    int rc = check_device_ready(ctx);
    if (rc) return rc;
    MPTG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    ctx->size = 0;
    ctx->star_ok = true;
    ctx->valid_upto = 0;
    ctx->some_invalid = false;
    // the prefilter's coordinate bound: the planner's sampling box and goal
    // (every node a planner adds lies within them), grown again by inserts
    ctx->coord_bound = planner_coord_bound(ctx);
    ctx->prrt.iteration = 0;
    ctx->prrt.goals = 0;
    ctx->prrt.goal_ids.clear();
    ctx->prrt.goal_cost0.clear();
    ctx->prrt.goal_parent0.clear();
    ctx->prrt.stats = mptg_prrt_stats{};
    ctx->prrt.counters_valid = false;
    return MPTG_OK;
}

int mptg_tree_insert(mptg_ctx* ctx, const double* h_states, const int32_t* h_parents, int64_t n) {
    int rc = check_device_ready(ctx);
    if (rc) return rc;
    if (n < 0 || (n > 0 && !h_states)) return fail(ctx, MPTG_E_ARG, "bad states");
    if (n == 0) return MPTG_OK;
    rc = tree_reserve(ctx, ctx->size + n);
    if (rc) return rc;
    int d = ctx->dim, dp = pitch32(d);
    std::vector<float> x32((size_t)n * dp, 0.0f);
    double bound = ctx->coord_bound;
    for (int64_t i = 0; i < n; ++i)
        for (int j = 0; j < d; ++j) {
            double v = h_states[i * d + j];
            if (!std::isfinite(v)) return fail(ctx, MPTG_E_ARG, "non-finite state coordinate");
            x32[i * dp + j] = (float)v;
            bound = std::max(bound, std::fabs(v));
        }
    std::vector<int32_t> par((size_t)n, -1);
    if (h_parents)
        for (int64_t i = 0; i < n; ++i) {
            if (h_parents[i] < -1 || h_parents[i] >= ctx->size + i)
                return fail(ctx, MPTG_E_ARG, "parent id must be -1 or an earlier node");
            par[i] = h_parents[i];
        }
    int64_t s = ctx->size;
    MPTG_HIP(ctx, hipMemcpyAsync(ctx->x64 + s * d, h_states, sizeof(double) * d * n, hipMemcpyHostToDevice,
                                 ctx->stream));
    MPTG_HIP(ctx, hipMemcpyAsync(ctx->x32 + s * dp, x32.data(), sizeof(float) * dp * n, hipMemcpyHostToDevice,
                                 ctx->stream));
    MPTG_HIP(ctx, hipMemcpyAsync(ctx->parent + s, par.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice,
                                 ctx->stream));
    MPTG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    ctx->size += n;
    ctx->coord_bound = bound;
    ctx->star_ok = false;  // no path costs or child lists for these nodes
    return MPTG_OK;
}

int64_t mptg_tree_size(const mptg_ctx* ctx) { return ctx ? ctx->size : -1; }

int mptg_tree_read(mptg_ctx* ctx, int64_t first, int64_t n, double* h_states, int32_t* h_parents) {
    int rc = check_device(ctx);
    if (rc) return rc;
    if (first < 0 || n < 0 || first + n > ctx->size) return fail(ctx, MPTG_E_RANGE, "read beyond tree size");
    if (n == 0) return MPTG_OK;
    int d = ctx->dim;
    if (h_states)
        MPTG_HIP(ctx, hipMemcpyAsync(h_states, ctx->x64 + first * d, sizeof(double) * d * n,
                                     hipMemcpyDeviceToHost, ctx->stream));
    if (h_parents)
        MPTG_HIP(ctx, hipMemcpyAsync(h_parents, ctx->parent + first, sizeof(int32_t) * n, hipMemcpyDeviceToHost,
                                     ctx->stream));
    MPTG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return MPTG_OK;
}

// ---- scenes ---------------------------------------------------------------
static int upload(mptg_ctx* ctx, void** dst, const void* src, size_t bytes) {
    if (*dst) {
        MPTG_HIP(ctx, hipStreamSynchronize(ctx->stream));
        MPTG_HIP(ctx, hipFree(*dst));
        *dst = nullptr;
    }
    if (bytes == 0) return MPTG_OK;
    MPTG_HIP(ctx, hipMalloc(dst, bytes));
    MPTG_HIP(ctx, hipMemcpyAsync(*dst, src, bytes, hipMemcpyHostToDevice, ctx->stream));
    MPTG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return MPTG_OK;
}

int mptg_scene_boxes(mptg_ctx* ctx, const double* h_boxes, int n) {
    int rc = check_device_ready(ctx);
    if (rc) return rc;
    if (n < 0 || (n > 0 && !h_boxes)) return fail(ctx, MPTG_E_ARG, "bad boxes");
    if (n > 4096) return fail(ctx, MPTG_E_RANGE, "at most 4096 boxes");
    rc = upload(ctx, (void**)&ctx->scene.boxes, h_boxes, sizeof(double) * 4 * n);
    if (rc) return rc;
    ctx->scene.kind = MPTG_SCENE_BOXES;
    ctx->valid_upto = 0;  // valid() changed: every node is checked again
    ctx->some_invalid = false;
    ctx->scene.nboxes = n;
    return MPTG_OK;
}

int mptg_scene_shapes(mptg_ctx* ctx, const double* h_circles, int ncircles, const double* h_rects, int nrects) {
    int rc = check_device_ready(ctx);
    if (rc) return rc;
    if (ncircles < 0 || nrects < 0 || (ncircles > 0 && !h_circles) || (nrects > 0 && !h_rects))
        return fail(ctx, MPTG_E_ARG, "bad circles or rectangles");
    if (ncircles > 4096 || nrects > 4096) return fail(ctx, MPTG_E_RANGE, "at most 4096 circles and 4096 rectangles");
    std::vector<double> c((size_t)4 * ncircles);
    for (int i = 0; i < ncircles; ++i) {
        const double r = h_circles[3 * i + 2];
        if (!std::isfinite(h_circles[3 * i]) || !std::isfinite(h_circles[3 * i + 1]) || !std::isfinite(r))
            return fail(ctx, MPTG_E_ARG, "circles must be finite");
        c[4 * i] = h_circles[3 * i];
        c[4 * i + 1] = h_circles[3 * i + 1];
        c[4 * i + 2] = r * r;  // radius_ * radius_, as Circle compares
        c[4 * i + 3] = r;
    }
    if ((rc = upload(ctx, (void**)&ctx->scene.circles, c.data(), sizeof(double) * c.size()))) return rc;
    if ((rc = upload(ctx, (void**)&ctx->scene.boxes, h_rects, sizeof(double) * 4 * nrects))) return rc;
    ctx->scene.kind = MPTG_SCENE_SHAPES;
    ctx->scene.ncircles = ncircles;
    ctx->scene.nboxes = nrects;
    ctx->valid_upto = 0;  // valid() changed: every node is checked again
    ctx->some_invalid = false;
    return MPTG_OK;
}

int mptg_scene_grid(mptg_ctx* ctx, const uint8_t* h_cells, int width, int height) {
    int rc = check_device_ready(ctx);
    if (rc) return rc;
    if (width <= 0 || height <= 0 || !h_cells) return fail(ctx, MPTG_E_ARG, "bad grid");
    if ((int64_t)width * height > ((int64_t)1 << 31)) return fail(ctx, MPTG_E_RANGE, "grid larger than 2^31 cells");
    // one bit per cell in 8 x 8 tiles (the layout grid_valid reads); cells of
    // the last tile row / column beyond the grid stay 0 and are never read
    // (grid_valid rejects them by the bounds check first)
    const int tx = (width + 7) / 8, ty = (height + 7) / 8;
    std::vector<uint64_t> bits((size_t)tx * ty, 0);
    for (int y = 0; y < height; ++y) {
        const uint8_t* row = h_cells + (size_t)width * y;
        uint64_t* trow = bits.data() + (size_t)(y >> 3) * tx;
        const int sh = (y & 7) << 3;
        for (int x = 0; x < width; ++x)
            if (row[x]) trow[x >> 3] |= 1ull << (sh | (x & 7));
    }
    rc = upload(ctx, (void**)&ctx->scene.grid, bits.data(), bits.size() * sizeof(uint64_t));
    if (rc) return rc;
    ctx->scene.kind = MPTG_SCENE_GRID;
    ctx->valid_upto = 0;  // valid() changed: every node is checked again
    ctx->some_invalid = false;
    ctx->scene.width = width;
    ctx->scene.height = height;
    ctx->scene.grid_tx = tx;
    return MPTG_OK;
}

int mptg_scene_arm(mptg_ctx* ctx, const double* h_lengths, int nlinks, double robot_radius,
                   const double* h_disks, int ndisks) {
    int rc = check_device_ready(ctx);
    if (rc) return rc;
    if (nlinks < 1 || nlinks > kMaxDim || !h_lengths) return fail(ctx, MPTG_E_ARG, "arm needs 1..32 links");
    if (ndisks < 0 || ndisks > 65536 || (ndisks > 0 && !h_disks)) return fail(ctx, MPTG_E_ARG, "bad disks");
    // reference order: [cx, cy, (r+R)^2, r+R]
    std::vector<double> dk((size_t)ndisks * 4);
    for (int i = 0; i < ndisks; ++i) {
        dk[4 * i + 0] = h_disks[3 * i + 0];
        dk[4 * i + 1] = h_disks[3 * i + 1];
        double rr = h_disks[3 * i + 2] + robot_radius;  // (radius_ + robotRadius), squared as the reference
        dk[4 * i + 2] = rr * rr;
        dk[4 * i + 3] = rr;
    }
    // kernel layout: [cx, cy, (r+R)^2, r+R] and a per-link segment-length
    // bound L (1 + 2^-30) + 1e-12 for the far-disk skip
    // then per group of kArmGroup links a bound on its half-length,
    // S_g/2 (1 + 2^-30) + 1e-12
    constexpr int kGroup = 5;
    const int ngroups = (nlinks + kGroup - 1) / kGroup;
    std::vector<double> ad((size_t)std::max(1, ndisks) * 4, 0.0), lim((size_t)(nlinks + ngroups));
    for (int i = 0; i < ndisks; ++i) {
        double rt = h_disks[3 * i + 2] + robot_radius;
        ad[4 * i + 0] = h_disks[3 * i + 0];
        ad[4 * i + 1] = h_disks[3 * i + 1];
        ad[4 * i + 2] = rt * rt;
        ad[4 * i + 3] = rt;
    }
    // disk grid: about one disk per cell on average (at most kArmGridMax per
    // axis) over the disk centres' bounding box; disks stored by cell,
    // row-major, ties by index.  The verdict is an AND over disks, so their
    // order changes nothing.
    int gnx = 1, gny = 1;
    double gx0 = 0.0, gy0 = 0.0, gix = 0.0, giy = 0.0, rtmax = 0.0;
    if (ndisks > 0) {
        double xmin = ad[0], xmax = ad[0], ymin = ad[1], ymax = ad[1];
        for (int i = 0; i < ndisks; ++i) {
            xmin = std::min(xmin, ad[4 * (size_t)i]);
            xmax = std::max(xmax, ad[4 * (size_t)i]);
            ymin = std::min(ymin, ad[4 * (size_t)i + 1]);
            ymax = std::max(ymax, ad[4 * (size_t)i + 1]);
            rtmax = std::max(rtmax, ad[4 * (size_t)i + 3]);
        }
        const int side = std::max(1, std::min(kArmGridMax, (int)std::lround(std::sqrt((double)ndisks))));
        gnx = xmax > xmin ? side : 1;
        gny = ymax > ymin ? side : 1;
        gx0 = xmin;
        gy0 = ymin;
        gix = xmax > xmin ? (double)gnx / (xmax - xmin) : 0.0;
        giy = ymax > ymin ? (double)gny / (ymax - ymin) : 0.0;
    }
    const int ncells = gnx * gny;
    std::vector<double> index(8 + (ncells + 1 + 1) / 2, 0.0);
    index[0] = gx0;
    index[1] = gy0;
    index[2] = gix;
    index[3] = giy;
    index[4] = rtmax;
    index[5] = gnx;
    index[6] = gny;
    {
        // counting sort by cell; starts[c]: the disks in cells below c
        int32_t* starts = reinterpret_cast<int32_t*>(index.data() + 8);
        std::vector<int> key((size_t)ndisks);
        for (int i = 0; i < ndisks; ++i) {
            key[(size_t)i] = arm_cell(ad[4 * (size_t)i + 1], gy0, giy, gny) * gnx + arm_cell(ad[4 * (size_t)i], gx0, gix, gnx);
            starts[key[(size_t)i] + 1]++;
        }
        for (int c = 0; c < ncells; ++c) starts[c + 1] += starts[c];
        std::vector<int> next(starts, starts + ncells);
        std::vector<double> sorted(ad.size(), 0.0);
        for (int i = 0; i < ndisks; ++i)
            std::memcpy(&sorted[4 * (size_t)next[(size_t)key[(size_t)i]]++], &ad[4 * (size_t)i], 4 * sizeof(double));
        ad.swap(sorted);
    }
    for (int i = 0; i < nlinks; ++i) lim[i] = h_lengths[i] * (1.0 + 0x1.0p-30) + 1e-12;
    for (int g = 0; g < ngroups; ++g) {
        double S = 0.0;
        for (int i = g * kGroup; i < (g + 1) * kGroup && i < nlinks; ++i) S += h_lengths[i];
        lim[nlinks + g] = S / 2 * (1.0 + 0x1.0p-30) + 1e-12;
    }
    // one block, one copy (16-byte aligned pieces first)
    std::vector<double> len(h_lengths, h_lengths + nlinks);
    std::vector<double> all;
    size_t at[5], k = 0;
    for (const std::vector<double>* v : {&ad, &dk, &index, &lim, &len}) {
        at[k++] = all.size();
        all.insert(all.end(), v->begin(), v->end());
    }
    MPTG_HIP(ctx, hipStreamSynchronize(ctx->stream));  // nothing reads the old scene any more
    if ((rc = ensure(ctx, ctx->scene.arm, sizeof(double) * all.size()))) return rc;
    double* base = (double*)ctx->scene.arm.p;
    MPTG_HIP(ctx, hipMemcpyAsync(base, all.data(), sizeof(double) * all.size(), hipMemcpyHostToDevice, ctx->stream));
    ctx->scene.arm_disks = base + at[0];
    ctx->scene.disks = base + at[1];
    ctx->scene.arm_index = base + at[2];
    ctx->scene.arm_lim = base + at[3];
    ctx->scene.lengths = base + at[4];
    uint32_t entries = 0;
    for (bool more = true; more;)
        if ((rc = build_near(ctx, h_lengths, nlinks, ad.data(), ndisks, &entries, &more))) return rc;
    MPTG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    ctx->scene.kind = MPTG_SCENE_ARM;
    ctx->valid_upto = 0;  // valid() changed: every node is checked again
    ctx->some_invalid = false;
    ctx->scene.total_length = 0;
    for (int i = 0; i < nlinks; ++i) ctx->scene.total_length += h_lengths[i];
    ctx->scene.nlinks = nlinks;
    ctx->scene.ndisks = ndisks;
    ctx->scene.robot_radius = robot_radius;
    return MPTG_OK;
}

int mptg_set_link(mptg_ctx* ctx, int mode, double param) {
    int rc = check_device_ready(ctx);
    if (rc) return rc;
    if (mode != MPTG_LINK_DMV && mode != MPTG_LINK_BISECT && mode != MPTG_LINK_BISECT_L2)
        return fail(ctx, MPTG_E_ARG, "unknown link mode");
    if (!(param > 0) || !std::isfinite(param)) return fail(ctx, MPTG_E_ARG, "link parameter must be > 0");
    ctx->link_mode = mode;
    ctx->link_param = param;
    return MPTG_OK;
}

// ---- host-pointer wrappers --------------------------------------------------
int mptg_knn(mptg_ctx* ctx, const double* h_q, int64_t nq, int k, double radius, int32_t* h_idx,
             double* h_dist) {
    int rc = check_device(ctx);
    if (rc) return rc;
    if (nq < 0 || (nq > 0 && (!h_q || !h_idx || !h_dist))) return fail(ctx, MPTG_E_ARG, "bad knn buffers");
    if (k < 1 || k > kMaxK) return fail(ctx, MPTG_E_ARG, "k must be in 1..64");
    if (nq == 0) return MPTG_OK;
    int d = ctx->dim;
    size_t qb = sizeof(double) * d * nq, ib = sizeof(int32_t) * k * nq, db = sizeof(double) * k * nq;
    if ((rc = ensure(ctx, ctx->scratch[0], qb))) return rc;
    if ((rc = ensure(ctx, ctx->scratch[1], ib))) return rc;
    if ((rc = ensure(ctx, ctx->scratch[2], db))) return rc;
    MPTG_HIP(ctx, hipMemcpyAsync(ctx->scratch[0].p, h_q, qb, hipMemcpyHostToDevice, ctx->stream));
    rc = launch_knn(ctx, (const double*)ctx->scratch[0].p, nq, k, radius, (int32_t*)ctx->scratch[1].p,
                    (double*)ctx->scratch[2].p, ctx->size);
    if (rc) return rc;
    MPTG_HIP(ctx, hipMemcpyAsync(h_idx, ctx->scratch[1].p, ib, hipMemcpyDeviceToHost, ctx->stream));
    MPTG_HIP(ctx, hipMemcpyAsync(h_dist, ctx->scratch[2].p, db, hipMemcpyDeviceToHost, ctx->stream));
    MPTG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return MPTG_OK;
}

int mptg_knn_dev(mptg_ctx* ctx, const double* d_q, int64_t nq, int k, double radius, int32_t* d_idx,
                 double* d_dist) {
    int rc = check_device(ctx);
    if (rc) return rc;
    if (nq < 0 || (nq > 0 && (!d_q || !d_idx || !d_dist))) return fail(ctx, MPTG_E_ARG, "bad knn buffers");
    if (k < 1 || k > kMaxK) return fail(ctx, MPTG_E_ARG, "k must be in 1..64");
    if (nq == 0) return MPTG_OK;
    return launch_knn(ctx, d_q, nq, k, radius, d_idx, d_dist, ctx->size);
}

int mptg_valid(mptg_ctx* ctx, const double* h_q, int64_t n, uint8_t* h_ok) {
    int rc = check_device(ctx);
    if (rc) return rc;
    if (n < 0 || (n > 0 && (!h_q || !h_ok))) return fail(ctx, MPTG_E_ARG, "bad valid buffers");
    if (n == 0) return MPTG_OK;
    size_t qb = sizeof(double) * ctx->dim * n;
    if ((rc = ensure(ctx, ctx->scratch[0], qb))) return rc;
    if ((rc = ensure(ctx, ctx->scratch[1], n))) return rc;
    MPTG_HIP(ctx, hipMemcpyAsync(ctx->scratch[0].p, h_q, qb, hipMemcpyHostToDevice, ctx->stream));
    rc = launch_valid(ctx, (const double*)ctx->scratch[0].p, n, (uint8_t*)ctx->scratch[1].p);
    if (rc) return rc;
    MPTG_HIP(ctx, hipMemcpyAsync(h_ok, ctx->scratch[1].p, n, hipMemcpyDeviceToHost, ctx->stream));
    MPTG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return MPTG_OK;
}

int mptg_link(mptg_ctx* ctx, const double* h_from, const double* h_to, int64_t n, int order,
              int endpoints_known_valid, uint8_t* h_verdict, uint32_t* h_checks) {
    int rc = check_device(ctx);
    if (rc) return rc;
    if (n < 0 || (n > 0 && (!h_from || !h_to || !h_verdict || !h_checks)))
        return fail(ctx, MPTG_E_ARG, "bad link buffers");
    if (n == 0) return MPTG_OK;
    size_t qb = sizeof(double) * ctx->dim * n;
    if ((rc = ensure(ctx, ctx->scratch[0], qb))) return rc;
    if ((rc = ensure(ctx, ctx->scratch[1], qb))) return rc;
    if ((rc = ensure(ctx, ctx->scratch[2], n))) return rc;
    if ((rc = ensure(ctx, ctx->scratch[3], sizeof(uint32_t) * n))) return rc;
    MPTG_HIP(ctx, hipMemcpyAsync(ctx->scratch[0].p, h_from, qb, hipMemcpyHostToDevice, ctx->stream));
    MPTG_HIP(ctx, hipMemcpyAsync(ctx->scratch[1].p, h_to, qb, hipMemcpyHostToDevice, ctx->stream));
    rc = launch_link(ctx, (const double*)ctx->scratch[0].p, (const double*)ctx->scratch[1].p, n, order,
                     endpoints_known_valid, (uint8_t*)ctx->scratch[2].p, (uint32_t*)ctx->scratch[3].p);
    if (rc) return rc;
    MPTG_HIP(ctx, hipMemcpyAsync(h_verdict, ctx->scratch[2].p, n, hipMemcpyDeviceToHost, ctx->stream));
    MPTG_HIP(ctx, hipMemcpyAsync(h_checks, ctx->scratch[3].p, sizeof(uint32_t) * n, hipMemcpyDeviceToHost,
                                 ctx->stream));
    MPTG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    for (int64_t i = 0; i < n; ++i)
        if (h_checks[i] == MPTG_CHECKS_OVER_LIMIT)
            return fail(ctx, MPTG_E_RANGE, "an edge exceeds the link() work limits (2^24 waypoints / 30 levels)");
    return MPTG_OK;
}

int mptg_link_dev(mptg_ctx* ctx, const double* d_from, const double* d_to, int64_t n, int order,
                  int endpoints_known_valid, uint8_t* d_verdict, uint32_t* d_checks) {
    int rc = check_device(ctx);
    if (rc) return rc;
    if (n < 0 || (n > 0 && (!d_from || !d_to || !d_verdict || !d_checks)))
        return fail(ctx, MPTG_E_ARG, "bad link buffers");
    if (n == 0) return MPTG_OK;
    return launch_link(ctx, d_from, d_to, n, order, endpoints_known_valid, d_verdict, d_checks);
}

int mptg_link_dev_noalloc(mptg_ctx* ctx, const double* d_from, const double* d_to, int64_t n, int order,
                          int endpoints_known_valid, uint8_t* d_verdict, uint32_t* d_checks) {
    int rc = check_device(ctx);
    if (rc) return rc;
    if (n < 0 || (n > 0 && (!d_from || !d_to || !d_verdict || !d_checks)))
        return fail(ctx, MPTG_E_ARG, "bad link buffers");
    return link_dev_noalloc(ctx, d_from, d_to, n, order, endpoints_known_valid, d_verdict, d_checks);
}

}  // extern "C"
