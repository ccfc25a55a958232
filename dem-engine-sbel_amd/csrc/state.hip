// Owner state and contact records between their device layout (one record per owner or contact) and the caller's arrays
// (one per field): packed and unpacked here, so the host moves plain contiguous ranges (it used to walk the records, a
// third of the time of reading 1M owners back).
#include "deme_internal.h"

namespace deme_int {
using namespace deme_dev;
namespace {

// Each array that is asked for (non-null) from the owner records; accelerations from their own arrays.
__global__ __launch_bounds__(256) void k_state_get(const OwnerRec* __restrict__ own, const float* __restrict__ acc,
                                                   uint32_t nO, StateArrays a) {
    const uint32_t o = blockIdx.x * blockDim.x + threadIdx.x;
    if (o >= nO) return;
    const OwnerRec r = load_owner(own, o);
    if (a.voxel) a.voxel[o] = r.voxel;
    const uint16_t loc[3] = {r.lx, r.ly, r.lz};
    const float f[10] = {r.qw, r.qx, r.qy, r.qz, r.vx, r.vy, r.vz, r.wx, r.wy, r.wz};
#pragma unroll
    for (int k = 0; k < 3; k++)
        if (a.loc[k]) a.loc[k][o] = loc[k];
#pragma unroll
    for (int k = 0; k < 10; k++)
        if (a.f[k]) a.f[k][o] = f[k];
#pragma unroll
    for (int k = 0; k < 6; k++)
        if (a.acc[k]) a.acc[k][o] = acc[(uint64_t)k * nO + o];
    if (a.fam) a.fam[o] = r.fam;
}

// The given arrays into the owner records (fresh: no records yet, the others take their defaults and mass and scene
// come along). pos0: the build positions of the candidate lists in force, or null. They tell every finite state whether
// the lists still hold; an orientation that is not finite would pass unseen (no comparison holds for a NaN displacement),
// so it marks the lists stale.
__global__ __launch_bounds__(256) void k_state_put(OwnerRec* __restrict__ own, float* __restrict__ acc, uint32_t nO,
                                                   StateArrays a, const float* __restrict__ mass,
                                                   const uint32_t* __restrict__ scene, bool fresh,
                                                   BuildPos* __restrict__ pos0) {
    const uint32_t o = blockIdx.x * blockDim.x + threadIdx.x;
    if (o >= nO) return;
    OwnerRec r{};
    if (fresh) {
        r.qw = 1.f;
        r.mass = mass[o];
        r.scene = scene[o];
    } else {
        r = load_owner(own, o);
    }
    r.pad0 = 0;
    if (a.voxel) r.voxel = a.voxel[o];
    uint16_t* loc[3] = {&r.lx, &r.ly, &r.lz};
    float* f[10] = {&r.qw, &r.qx, &r.qy, &r.qz, &r.vx, &r.vy, &r.vz, &r.wx, &r.wy, &r.wz};
#pragma unroll
    for (int k = 0; k < 3; k++)
        if (a.loc[k]) *loc[k] = a.loc[k][o];
#pragma unroll
    for (int k = 0; k < 10; k++)
        if (a.f[k]) *f[k] = a.f[k][o];
#pragma unroll
    for (int k = 0; k < 6; k++)
        if (a.acc[k]) acc[(uint64_t)k * nO + o] = a.acc[k][o];
    if (a.fam) r.fam = a.fam[o];
    if (pos0 && !(isfinite(r.qw) && isfinite(r.qx) && isfinite(r.qy) && isfinite(r.qz))) pos0[0].x = INT32_MIN;
    uint4* dst = reinterpret_cast<uint4*>(own + o);
    const uint4* src = reinterpret_cast<const uint4*>(&r);
    dst[0] = src[0];
    dst[1] = src[1];
    dst[2] = src[2];
    dst[3] = src[3];
}

// Three floats at float column `col` of each 48-byte contact record, packed.
__global__ __launch_bounds__(256) void k_record_columns(const float* __restrict__ rec, uint64_t n, int col,
                                                        float* __restrict__ out) {
    const uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= 3 * n) return;
    const uint64_t i = k / 3;
    out[k] = rec[i * 12 + (uint64_t)col + (k - 3 * i)];
}

// Histories (float4 per contact) component-major; map: contact i's history is prev[map[i]] (none: zero).
__global__ __launch_bounds__(256) void k_history_columns(const float4* __restrict__ hist,
                                                         const uint32_t* __restrict__ map, uint64_t nPrev, uint64_t n,
                                                         float* __restrict__ out) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 h = make_float4(0.f, 0.f, 0.f, 0.f);
    if (!map) {
        h = hist[i];
    } else {
        const uint32_t m = map[i];
        if (m != DEME_NULL_MAPPING_PARTNER && m < nPrev) h = hist[m];
    }
    out[i] = h.x;
    out[n + i] = h.y;
    out[2 * n + i] = h.z;
    out[3 * n + i] = h.w;
}

inline uint32_t blocks(uint64_t n) { return (uint32_t)((n + 255) / 256); }

}  // namespace

hipError_t launch_state_get(const OwnerRec* own, const float* acc, uint32_t nO, const StateArrays& a, hipStream_t st) {
    if (nO == 0) return hipSuccess;
    k_state_get<<<blocks(nO), 256, 0, st>>>(own, acc, nO, a);
    return hipGetLastError();
}

hipError_t launch_state_put(OwnerRec* own, float* acc, uint32_t nO, const StateArrays& a, const float* mass,
                            const uint32_t* scene, bool fresh, BuildPos* pos0, hipStream_t st) {
    if (nO == 0) return hipSuccess;
    k_state_put<<<blocks(nO), 256, 0, st>>>(own, acc, nO, a, mass, scene, fresh, pos0);
    return hipGetLastError();
}

hipError_t launch_record_columns(const ForceRec* rec, uint64_t n, int col, float* out, hipStream_t st) {
    if (n == 0) return hipSuccess;
    k_record_columns<<<blocks(3 * n), 256, 0, st>>>(reinterpret_cast<const float*>(rec), n, col, out);
    return hipGetLastError();
}

hipError_t launch_history_columns(const float4* hist, const uint32_t* map, uint64_t nPrev, uint64_t n, float* out,
                                  hipStream_t st) {
    if (n == 0) return hipSuccess;
    k_history_columns<<<blocks(n), 256, 0, st>>>(hist, map, nPrev, n, out);
    return hipGetLastError();
}

}  // namespace deme_int
