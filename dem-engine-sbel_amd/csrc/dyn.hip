// Dynamics for gfx950: frictional Hertz-Mindlin contact force with tangential history, owner-keyed force/torque
// reduction without global atomics, and clump integration.
//
// Reference: src/DEM/dT.cpp:1349-1432 and the kernels it launches (DEMPrepForceKernels.cu, DEMCalcForceKernels.cu +
// DEMCustomizablePolicies/FullHertzianForceModel.cu, DEMCollectForceKernels.cu + DEMCubForceCollection.cu,
// DEMIntegrationKernels.cu + IntegrationVelPassOn*.cu).
//
// Every float/double promotion of the reference's expressions is kept (e.g. `2. * E_cnt * sqrt_Rd` is evaluated in
// double and rounded to float), and the device code is compiled without contraction.
#include "deme_internal.h"

// Rows a14-a15, the contact force kernel: generated at build time from jit/force_kernel.tpl with the default
// frictional Hertz-Mindlin model (jit/hertz_frictional.model), the same source the runtime hipRTC path specialises.
#include "force_aot.hip"
// Rows a16 (clump owners) + a17, the owner update: generated at build time from jit/owner_kernel.tpl with no motion
// strategies (numeric prescriptions from the family rule table).
#include "owner_aot.hip"

namespace deme_int {
using namespace deme_dev;
namespace {

// The simulation time read by the owner update's motion rules (a kernel, not a copy: it may sit in a captured graph).
__global__ void k_set_clock(double* clock, double t) {
    if (threadIdx.x == 0) clock[0] = t;
}

__global__ void k_advance_clock(double* clock, float h) {
    if (threadIdx.x == 0) clock[0] += (double)h;
}

// ChangeFamily (APIPublic.cpp:184-207): every owner of family `from` moves to family `to`.
__global__ __launch_bounds__(256) void k_change_family(OwnerRec* own, uint32_t nO, uint8_t from, uint8_t to) {
    const uint32_t o = blockIdx.x * blockDim.x + threadIdx.x;
    if (o < nO && own[o].fam == from) own[o].fam = to;
}

__global__ __launch_bounds__(256) void k_material_pairs(const deme_material* __restrict__ mats, uint32_t nM,
                                                        MatPair* __restrict__ pairs) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < nM * nM) pairs[k] = materialPair(mats[k / nM], mats[k % nM]);
}

inline uint32_t blocks(uint64_t n, uint32_t b) { return (uint32_t)((n + b - 1) / b); }

}  // namespace

hipError_t launch_material_pairs(const deme_material* mats, uint32_t nM, MatPair* pairs, hipStream_t st) {
    if (nM == 0) return hipSuccess;
    k_material_pairs<<<blocks((uint64_t)nM * nM, 256), 256, 0, st>>>(mats, nM, pairs);
    return hipGetLastError();
}

hipError_t launch_force(const KParams& P, uint32_t nC, const uint32_t* idA, const uint32_t* idB, const uint8_t* ctype,
                        const SphereRec* sph, const OwnerRec* own, const float4* moi, const deme_anal_obj* anal,
                        const PlanePose* pose, const deme_material* mats, const float4* histIn, const uint32_t* map,
                        float4* histOut, const uint32_t* mirror, float* aTerm, float* bTerm,
                        const PlaneSums& sums, uint8_t* aOn, uint8_t* bOn, ForceRec* out, hipStream_t st, SpecGuard guard, ForceKind kind) {
    if (nC == 0) return hipSuccess;
    if (out)
        deme_force_full<<<blocks(nC, 256), 256, 0, st>>>(P, nC, idA, idB, ctype, sph, own, moi, anal, pose, mats, histIn,
                                                       map, histOut, mirror, aTerm, bTerm, sums, aOn, bOn, out,
                                                       guard, kind == FORCE_KIND_SETTLED);
    else if (kind != FORCE_KIND_ALL)
        deme_force_margin<<<blocks(nC, 1024), 256, 0, st>>>(P, nC, idA, idB, ctype, sph, own, moi, anal, pose, mats,
                                                            histIn, map, histOut, mirror, aTerm, bTerm, sums, aOn,
                                                            bOn, nullptr, guard, kind == FORCE_KIND_SETTLED);
    else
        deme_force_terms<<<blocks(nC, 256), 256, 0, st>>>(P, nC, idA, idB, ctype, sph, own, moi, anal, pose, mats,
                                                        histIn, map, histOut, mirror, aTerm, bTerm, sums, aOn, bOn,
                                                        nullptr, guard, kind == FORCE_KIND_SETTLED);
    return hipGetLastError();
}

hipError_t launch_force_direct(const KParams& P, const DirectList& D, const SphereRec* sph, const OwnerRec* own,
                               const float4* moi, const deme_anal_obj* anal, const PlanePose* pose,
                               const deme_material* mats, float* aTerm, float* bTerm, const PlaneSums& sums,
                               hipStream_t st) {
    deme_force_direct<<<direct_force_blocks(D), 256, 0, st>>>(P, D, sph, own, moi, anal, pose, mats, aTerm, bTerm, sums);
    return hipGetLastError();
}

hipError_t launch_owner_update(const KParams& P, uint32_t nO, uint32_t nClumps, const uint32_t* ownerSphStart,
                               const uint32_t* rowStart, const uint32_t* bRowStart, const float* aTerm,
                               const float* bTerm, const uint8_t* aOn, const uint8_t* bOn, const PlaneSums& sums,
                               const PlaneRefresh& planes, const deme_family_rule* rules, OwnerRec* own, float* acc,
                               int doIntegrate, const double* clock, hipStream_t st, OwnerRec* ownOut,
                               SpecGuard guard, const DirectList& direct, const DirectCheck& check) {
    if (nO == 0) return hipSuccess;
    if (sums.nOwners > MAX_ANAL_OWNERS) return hipErrorInvalidValue;
    deme_owner_update<<<owner_blocks(nClumps, sums.nOwners), 256, 0, st>>>(
        P, nO, nClumps, ownerSphStart, rowStart, bRowStart, aTerm, bTerm, aOn, bOn, sums, planes, rules, own,
        ownOut ? ownOut : own, acc, doIntegrate, clock, guard, direct, check);
    return hipGetLastError();
}

hipError_t launch_set_clock(double* clock, double t, hipStream_t st) {
    k_set_clock<<<1, 64, 0, st>>>(clock, t);
    return hipGetLastError();
}

hipError_t launch_advance_clock(double* clock, float h, hipStream_t st) {
    k_advance_clock<<<1, 64, 0, st>>>(clock, h);
    return hipGetLastError();
}

hipError_t launch_change_family(OwnerRec* own, uint32_t nO, uint8_t from, uint8_t to, hipStream_t st) {
    if (nO == 0) return hipSuccess;
    k_change_family<<<blocks(nO, 256), 256, 0, st>>>(own, nO, from, to);
    return hipGetLastError();
}

}  // namespace deme_int
