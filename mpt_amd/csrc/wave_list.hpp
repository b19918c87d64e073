// A wave's sorted k-list of (distance, node id) candidates, one entry per
// lane: lane j < k holds the j-th best in ascending (distance, id) order.
// Shared by the kernels that give one query a whole wave (grid queries, the
// SE(3) scan).
#pragma once
#include <climits>

#include <hip/hip_runtime.h>

namespace mptg {

constexpr int kWaveListMax = 64;  // one entry per lane

__device__ __forceinline__ bool wl_before(double a, int ia, double b, int ib) {
    return a < b || (a == b && ia < ib);
}

__device__ __forceinline__ double wl_readlane(double v, int l) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
    return __hiloint2double(hi, lo);
}

// Lane l's value moved to lane l + 1 (lane 0 keeps its own): one DPP move.
__device__ __forceinline__ int32_t wl_up(int32_t v) {
    return __builtin_amdgcn_update_dpp(v, v, 0x138 /* wave_shr:1 */, 0xf, 0xf, false);
}

// (kd, ki) mirror lane k - 1's entry (the k-th best) as wave-uniform values.
// +inf comes in as a value (a kernel argument), not a constant: this
// toolchain encodes a 64-bit scalar move of the constant 0x7ff0000000000000
// with a 32-bit literal holding its low half, so a uniform +inf held in
// scalar registers would read as 0.0.
struct WaveList {
    double ld;
    int32_t li;
    double kd;
    int32_t ki;
    int k;
    __device__ __forceinline__ void init(int k_, double inf) {
        ld = inf;
        li = INT_MAX;
        kd = inf;
        ki = INT_MAX;
        k = k_;
    }
    // Inserts a wave-uniform candidate that beats (kd, ki): the first entry
    // it beats and every one after it move one lane up (wl_up, a DPP move in
    // the VALU; a shuffle is an LDS round trip).
    __device__ __forceinline__ void insert(double cd, int32_t ci, int lane) {
        const double pd = __hiloint2double(wl_up(__double2hiint(ld)), wl_up(__double2loint(ld)));
        const int32_t pi = wl_up(li);
        const int pos = __builtin_ctzll(__ballot(wl_before(cd, ci, ld, li)));  // never empty: lane k - 1 is beaten
        ld = lane > pos ? pd : (lane == pos ? cd : ld);
        li = lane > pos ? pi : (lane == pos ? ci : li);
        kd = wl_readlane(ld, k - 1);
        ki = __builtin_amdgcn_readlane(li, k - 1);
    }
    // Offers every lane's (d, id) where `pass` holds, in lane order; after
    // each insert only those that still beat the k-th best stay.
    __device__ __forceinline__ void offer(bool pass, double d, int32_t id, int lane) {
        unsigned long long m = __ballot(pass && wl_before(d, id, kd, ki));
        while (m) {
            const int b = __builtin_ctzll(m);
            insert(wl_readlane(d, b), __builtin_amdgcn_readlane(id, b), lane);
            m = __ballot(pass && lane > b && wl_before(d, id, kd, ki));
        }
    }
};

}  // namespace mptg
