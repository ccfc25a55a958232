// Stepping on the candidates of a list build (deme_step with detection every step and no drift margin).
//
// Detecting every step, the passes of the contact-list path mostly renumber: of 1M clumps' 2.97M candidates all but a
// few touch from one step to the next, yet each pass forms flags, row counts, two scans, the rows, the mirror links and
// the history map (220 of 400 us a step), and small systems pay the launches. Between builds the candidates' own order
// already is the canonical order, so the force kernel can take them directly: history and owner terms live in the
// candidate's slots, a flag says whether it touched, and the owner update sums the flagged terms of the candidate rows
// -- the same terms in the same order, bit for bit. Only the plane owners' sums are folded in another order; an owner that
// they would move is left to the host, which folds that step's terms in the list's order (k_direct_plane_sums) and goes on
// with passes. A step is then two kernels (force, owner update), and the host reads one status per batch of steps.
//
// This file holds what connects the two forms: the plane candidates (spheres near a plane, which the pair lists do not
// hold), histories carried from the contact list to the candidates and back, and from one build's candidates to the
// next.
#include "deme_internal.h"

namespace deme_int {
using namespace deme_dev;
namespace {

// Planes within `margin` of touching each sphere (no family mask: families may change from step to step).
__global__ __launch_bounds__(256) void k_direct_near(KParams P, const SphereRec* __restrict__ sph,
                                                     const OwnerRec* __restrict__ own, uint32_t nS,
                                                     const PlanePose* __restrict__ pose, uint32_t nA, double margin,
                                                     unsigned long long* __restrict__ nearBits,
                                                     uint32_t* __restrict__ nearCnt) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nS) return;
    const SphereRec sr = load_sphere(sph, s);
    const OwnerRec o = load_owner(own, sr.owner);
    double X, Y, Z;
    sphere_position(P, o, sr, X, Y, Z);
    const double reach = (double)sr.r + (double)P.beta + margin;
    unsigned long long bits = 0;
    uint32_t a0, a1;
    scene_planes(P, o.scene, a0, a1);
    for (uint32_t a = a0; a < a1 && a < nA && a - a0 < 64; a++)
        if (plane_cd(P, pose[a], X, Y, Z, reach)) bits |= 1ull << (a - a0);
    nearBits[s] = bits;
    nearCnt[s] = (uint32_t)__popcll(bits);
}

__global__ __launch_bounds__(256) void k_direct_plane_rows(KParams P, const SphereRec* __restrict__ sph,
                                                           const OwnerRec* __restrict__ own, uint32_t nS,
                                                           const unsigned long long* __restrict__ nearBits,
                                                           const uint32_t* __restrict__ pStart,
                                                           uint32_t* __restrict__ pSph, uint32_t* __restrict__ pPlane,
                                                           const PlanePose* __restrict__ pose, uint32_t nA,
                                                           PlanePose* __restrict__ pose0) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (blockIdx.x == 0)
        for (uint32_t a = threadIdx.x; a < nA; a += 256) pose0[a] = pose[a];
    if (s >= nS) return;
    unsigned long long bits = nearBits[s];
    if (!bits) return;
    uint32_t a0 = 0, a1 = 0;
    scene_planes(P, own[sph[s].owner].scene, a0, a1);
    for (uint32_t q = pStart[s]; bits; q++) {
        pSph[q] = s;
        pPlane[q] = a0 + (uint32_t)(__ffsll(bits) - 1);
        bits &= bits - 1;
    }
}

// The contact list's histories to the candidates: pairs through their contact index (cidx, valid where on), planes by
// looking their component up at the head of the sphere's row. One lane per candidate, planes after the pairs.
__global__ __launch_bounds__(256) void k_direct_enter(DirectList D, uint32_t pairBlocks,
                                                      const uint32_t* __restrict__ cidx,
                                                      const uint32_t* __restrict__ rowStart,
                                                      const uint32_t* __restrict__ idB,
                                                      const uint8_t* __restrict__ ctype,
                                                      const float4* __restrict__ listHist) {
    if (blockIdx.x < pairBlocks) {
        const uint32_t c = blockIdx.x * 256u + threadIdx.x;
        if (c >= D.nPair) return;
        const uint8_t f = D.on[c];
        D.bOn[D.tPos[c]] = f;
        if (f) D.hist[c] = listHist[cidx[c]];
        return;
    }
    const uint32_t q = (blockIdx.x - pairBlocks) * 256u + threadIdx.x;
    if (q >= D.nPlane) return;
    const uint32_t s = D.pSph[q], p = D.pPlane[q], e = rowStart[s + 1];
    uint8_t f = 0;
    for (uint32_t i = rowStart[s]; i < e && ctype[i] == DEME_SPHERE_PLANE_CONTACT && idB[i] <= p; i++)
        if (idB[i] == p) {
            f = 1;
            D.pHist[q] = listHist[i];
        }
    D.pOn[q] = f;
}

// One sphere's row of new candidates matched against its old row (both ascending in partner): flags and histories of
// the partners found. Rows are short: the old row's first entries are held in registers.
constexpr uint32_t JOIN_REG = 8;
__device__ __forceinline__ void join_row(uint32_t o0, uint32_t o1, const uint32_t* __restrict__ oldB,
                                         const uint8_t* __restrict__ oldOn, const float4* __restrict__ oldHist,
                                         uint32_t n0, uint32_t n1, const uint32_t* __restrict__ newB,
                                         const uint32_t* __restrict__ tPos, uint8_t* __restrict__ on,
                                         uint8_t* __restrict__ bOn, float4* __restrict__ hist) {
    const uint32_t no = o1 - o0;
    uint32_t ob[JOIN_REG];
    uint8_t of[JOIN_REG];
#pragma unroll
    for (uint32_t k = 0; k < JOIN_REG; k++) {
        ob[k] = k < no ? oldB[o0 + k] : 0xFFFFFFFFu;
        of[k] = k < no ? oldOn[o0 + k] : (uint8_t)0;
    }
    for (uint32_t c = n0; c < n1; c++) {
        const uint32_t b = newB[c];
        uint32_t m = 0xFFFFFFFFu;
        uint8_t f = 0;
#pragma unroll
        for (uint32_t k = 0; k < JOIN_REG; k++)
            if (k < no && ob[k] == b) {
                m = o0 + k;
                f = of[k];
            }
        for (uint32_t j = o0 + JOIN_REG; j < o1 && m == 0xFFFFFFFFu; j++)
            if (oldB[j] == b) {
                m = j;
                f = oldOn[j];
            }
        on[c] = f;
        if (bOn) bOn[tPos[c]] = f;
        if (f) hist[c] = oldHist[m];
    }
}

__global__ __launch_bounds__(256) void k_direct_join(uint32_t nS, const uint32_t* __restrict__ oldStart,
                                                     const uint32_t* __restrict__ oldB,
                                                     const uint32_t* __restrict__ newStart,
                                                     const uint32_t* __restrict__ newB,
                                                     const uint32_t* __restrict__ oldPStart,
                                                     const uint32_t* __restrict__ oldPlane, DirectList O, DirectList D) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nS) return;
    join_row(oldStart[s], oldStart[s + 1], oldB, O.on, O.hist, newStart[s], newStart[s + 1], newB, D.tPos, D.on, D.bOn,
             D.hist);
    const uint32_t p0 = D.pStart[s], p1 = D.pStart[s + 1];
    if (p0 < p1)
        join_row(oldPStart[s], oldPStart[s + 1], oldPlane, O.pOn, O.pHist, p0, p1, D.pPlane, nullptr, D.pOn, nullptr,
                 D.pHist);
}

// An owner's pose at a candidate build (coordinates in fixed point as the spheres' build positions); returns a bound of
// its spheres' speed.
__device__ __forceinline__ float owner_build(const KParams& P, const SphereRec* __restrict__ sph,
                                             const OwnerRec* __restrict__ own,
                                             const uint32_t* __restrict__ ownerSphStart, uint32_t o, double scale,
                                             OwnerBuild* __restrict__ own0) {
    const OwnerRec r = load_owner(own, o);
    double X, Y, Z;
    owner_position(P, r.voxel, r.lx, r.ly, r.lz, X, Y, Z);
    float rel2 = 0.f;
    for (uint32_t s = ownerSphStart[o]; s < ownerSphStart[o + 1]; s++) {
        const SphereRec sr = load_sphere(sph, s);
        rel2 = fmaxf(rel2, sr.rx * sr.rx + sr.ry * sr.ry + sr.rz * sr.rz);
    }
    OwnerBuild b;
    b.x = build_fix(X, scale);
    b.y = build_fix(Y, scale);
    b.z = build_fix(Z, scale);
    b.relMax = rel2 > 0.f ? sqrtf(rel2) * 1.000001f : 0.f;  // (rounded up)
    b.qw = r.qw;
    b.qx = r.qx;
    b.qy = r.qy;
    b.qz = r.qz;
    uint4* dst = reinterpret_cast<uint4*>(own0 + o);
    const uint4* src = reinterpret_cast<const uint4*>(&b);
    dst[0] = src[0];
    dst[1] = src[1];
    const float v = sqrtf(r.vx * r.vx + r.vy * r.vy + r.vz * r.vz);
    const float w = sqrtf(r.wx * r.wx + r.wy * r.wy + r.wz * r.wz);
    return v + w * b.relMax;
}

__global__ __launch_bounds__(256) void k_owner_build(KParams P, const SphereRec* __restrict__ sph,
                                                     const OwnerRec* __restrict__ own,
                                                     const uint32_t* __restrict__ ownerSphStart, uint32_t nClumps,
                                                     double scale, OwnerBuild* __restrict__ own0,
                                                     SkinStats* __restrict__ stats) {
    const uint32_t o = blockIdx.x * blockDim.x + threadIdx.x;
    // the largest speed of a sphere (bounded by |v| + |w| relMax), for the choice of the skin
    float speed = 0.f;
    if (o < nClumps) speed = owner_build(P, sph, own, ownerSphStart, o, scale, own0);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) speed = fmaxf(speed, __shfl_xor(speed, off, 64));
    // (only a wave above what stands there already goes to the one address: every wave of 1M owners did, 274 us)
    const uint32_t bits = __float_as_uint(speed);
    if ((threadIdx.x & 63u) == 0 && bits > __hip_atomic_load(&stats->speedBits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMax(&stats->speedBits, bits);
}

// How the candidates' gaps are spread over the skin: a sample of them (every stride-th), gaps in sixteenths of the skin.
__global__ __launch_bounds__(256) void k_gap_hist(KParams P, const SphereRec* __restrict__ sph,
                                                  const OwnerRec* __restrict__ own, const uint32_t* __restrict__ candA,
                                                  const uint32_t* __restrict__ candB, uint32_t nK, uint32_t stride,
                                                  double skin, SkinStats* __restrict__ stats) {
    __shared__ uint32_t h[SKIN_BUCKETS];
    if (threadIdx.x < SKIN_BUCKETS) h[threadIdx.x] = 0;
    __syncthreads();
    const uint64_t c = ((uint64_t)blockIdx.x * 256u + threadIdx.x) * stride;
    if (c < nK) {
        const SphereRec a = load_sphere(sph, candA[c]), b = load_sphere(sph, candB[c]);
        const OwnerRec oa = load_owner(own, a.owner), ob = load_owner(own, b.owner);
        double ax, ay, az, bx, by, bz;
        sphere_position(P, oa, a, ax, ay, az);
        sphere_position(P, ob, b, bx, by, bz);
        const double dx = ax - bx, dy = ay - by, dz = az - bz;
        const double gap = sqrt(dx * dx + dy * dy + dz * dz) - ((double)a.r + (double)b.r + 2.0 * (double)P.beta);
        const double k = gap / skin * SKIN_BUCKETS;
        atomicAdd(&h[k > 0.0 ? (k < SKIN_BUCKETS ? (uint32_t)k : SKIN_BUCKETS - 1) : 0u], 1u);
    }
    __syncthreads();
    if (threadIdx.x < SKIN_BUCKETS && h[threadIdx.x]) atomicAdd(&stats->gaps[threadIdx.x], h[threadIdx.x]);
}

// The check of a state the owner update did not leave itself (a call's first step on the candidates).
__global__ __launch_bounds__(256) void k_direct_check(KParams P, DirectCheck C, const OwnerRec* __restrict__ own,
                                                      uint32_t nClumps, const PlanePose* __restrict__ pose, uint32_t nA,
                                                      DirectState* st) {
    const uint32_t o = blockIdx.x * blockDim.x + threadIdx.x;
    double disp = 0.0;
    uint32_t bad = 0;
    if (o < nClumps) bad = direct_check_owner(P, C, load_owner(own, o), o, disp);
    if (blockIdx.x == 0)
        for (uint32_t a = threadIdx.x; a < nA; a += 256)
            if (direct_plane_moved(C, pose[a], C.pose0[a])) bad |= ERRBIT_STALE;
    direct_report(st, C.limit, disp, bad);
}

// Back to the contact list, first: the plane contacts of the last step per sphere (count and bits within the scene's
// components), and the pass's counters cleared.
__global__ __launch_bounds__(256) void k_direct_plane_bits(KParams P, const SphereRec* __restrict__ sph,
                                                           const OwnerRec* __restrict__ own, uint32_t nS, DirectList D,
                                                           uint32_t* __restrict__ numAnal,
                                                           unsigned long long* __restrict__ planeBits,
                                                           uint32_t* __restrict__ clear, uint32_t nClear) {
    if (blockIdx.x == 0)
        for (uint32_t k = threadIdx.x; k < nClear; k += 256) clear[k] = 0u;
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nS) return;
    unsigned long long bits = 0;
    const uint32_t q0 = D.pStart[s], q1 = D.pStart[s + 1];
    if (q0 < q1) {
        uint32_t a0 = 0, a1 = 0;
        scene_planes(P, own[sph[s].owner].scene, a0, a1);
        for (uint32_t q = q0; q < q1; q++)
            if (D.pOn[q]) bits |= 1ull << (D.pPlane[q] - a0);
    }
    planeBits[s] = bits;
    numAnal[s] = (uint32_t)__popcll(bits);
}

// ... last: the candidates' histories to the list (contact indices in cidx; a sphere's plane contacts head its row).
__global__ __launch_bounds__(256) void k_direct_leave(DirectList D, uint32_t pairBlocks,
                                                      const uint32_t* __restrict__ cidx,
                                                      const uint32_t* __restrict__ rowStart,
                                                      float4* __restrict__ listHist, SpecGuard guard) {
    if (spec_skip(guard)) return;
    if (blockIdx.x < pairBlocks) {
        const uint32_t c = blockIdx.x * 256u + threadIdx.x;
        if (c < D.nPair && D.on[c]) listHist[cidx[c]] = D.hist[c];
        return;
    }
    const uint32_t q = (blockIdx.x - pairBlocks) * 256u + threadIdx.x;
    if (q >= D.nPlane || !D.pOn[q]) return;
    const uint32_t s = D.pSph[q];
    uint32_t k = 0;
    for (uint32_t j = D.pStart[s]; j < q; j++) k += D.pOn[j];
    listHist[rowStart[s] + k] = D.pHist[q];
}

// The plane owners' partial sums of the last step on the candidates by the places of the contact list (idA, idB, ctype; as
// the force kernel over the list folds them), from the terms that the step left per plane candidate.
__global__ __launch_bounds__(256) void k_direct_plane_sums(DirectList D, uint32_t nC, const uint32_t* __restrict__ idA,
                                                           const uint32_t* __restrict__ idB,
                                                           const uint8_t* __restrict__ ctype,
                                                           const deme_anal_obj* __restrict__ anal, PlaneSums sums) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    int gOwner = -1;
    float g[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (i < nC && ctype[i] == DEME_SPHERE_PLANE_CONTACT) {
        const uint32_t s = idA[i], p = idB[i];
        for (uint32_t q = D.pStart[s]; q < D.pStart[s + 1]; q++)
            if (D.pPlane[q] == p) {
                gOwner = (int)(anal[p].owner - sums.first);
#pragma unroll
                for (int k = 0; k < 6; k++) g[k] = D.pTerm[((uint64_t)D.nPlane + q) * 6 + k];
            }
    }
    fold_plane_terms(sums, gOwner, g);
}

inline uint32_t blocks(uint64_t n) { return (uint32_t)((n + 255) / 256); }

}  // namespace

hipError_t launch_direct_near(const KParams& P, const SphereRec* sph, const OwnerRec* own, uint32_t nS,
                              const PlanePose* pose, uint32_t nA, double margin, unsigned long long* nearBits,
                              uint32_t* nearCnt, hipStream_t st) {
    if (nS == 0) return hipSuccess;
    k_direct_near<<<blocks(nS), 256, 0, st>>>(P, sph, own, nS, pose, nA, margin, nearBits, nearCnt);
    return hipGetLastError();
}

hipError_t launch_direct_plane_rows(const KParams& P, const SphereRec* sph, const OwnerRec* own, uint32_t nS,
                                    const unsigned long long* nearBits, const uint32_t* pStart, uint32_t* pSph,
                                    uint32_t* pPlane, const PlanePose* pose, uint32_t nA, PlanePose* pose0,
                                    hipStream_t st) {
    if (nS == 0) return hipSuccess;
    k_direct_plane_rows<<<blocks(nS), 256, 0, st>>>(P, sph, own, nS, nearBits, pStart, pSph, pPlane, pose, nA, pose0);
    return hipGetLastError();
}

hipError_t launch_direct_enter(const DirectList& D, const uint32_t* cidx, const uint32_t* rowStart, const uint32_t* idB,
                               const uint8_t* ctype, const float4* listHist, hipStream_t st) {
    const uint32_t pb = blocks(D.nPair), g = pb + blocks(D.nPlane);
    if (g == 0) return hipSuccess;
    k_direct_enter<<<g, 256, 0, st>>>(D, pb, cidx, rowStart, idB, ctype, listHist);
    return hipGetLastError();
}

hipError_t launch_direct_join(uint32_t nS, const uint32_t* oldStart, const uint32_t* oldB, const uint32_t* newStart,
                              const uint32_t* newB, const uint32_t* oldPStart, const uint32_t* oldPlane,
                              const DirectList& O, const DirectList& D, hipStream_t st) {
    if (nS == 0) return hipSuccess;
    k_direct_join<<<blocks(nS), 256, 0, st>>>(nS, oldStart, oldB, newStart, newB, oldPStart, oldPlane, O, D);
    return hipGetLastError();
}

hipError_t launch_owner_build(const KParams& P, const SphereRec* sph, const OwnerRec* own,
                              const uint32_t* ownerSphStart, uint32_t nClumps, double scale, OwnerBuild* own0,
                              SkinStats* stats, hipStream_t st) {
    if (nClumps == 0) return hipSuccess;
    k_owner_build<<<blocks(nClumps), 256, 0, st>>>(P, sph, own, ownerSphStart, nClumps, scale, own0, stats);
    return hipGetLastError();
}

hipError_t launch_gap_hist(const KParams& P, const SphereRec* sph, const OwnerRec* own, const uint32_t* candA,
                           const uint32_t* candB, uint32_t nK, double skin, SkinStats* stats, hipStream_t st) {
    if (nK == 0) return hipSuccess;
    const uint32_t stride = (nK + SKIN_SAMPLES - 1) / SKIN_SAMPLES;
    k_gap_hist<<<blocks((nK + stride - 1) / stride), 256, 0, st>>>(P, sph, own, candA, candB, nK, stride, skin, stats);
    return hipGetLastError();
}

hipError_t launch_direct_check(const KParams& P, const DirectCheck& C, const OwnerRec* own, uint32_t nClumps,
                               const PlanePose* pose, uint32_t nA, DirectState* state, hipStream_t st) {
    if (nClumps == 0) return hipSuccess;
    k_direct_check<<<blocks(nClumps), 256, 0, st>>>(P, C, own, nClumps, pose, nA, state);
    return hipGetLastError();
}

hipError_t launch_direct_plane_bits(const KParams& P, const SphereRec* sph, const OwnerRec* own, uint32_t nS,
                                    const DirectList& D, uint32_t* numAnal, unsigned long long* planeBits,
                                    uint32_t* clear, uint32_t nClear, hipStream_t st) {
    if (nS == 0) return hipSuccess;
    k_direct_plane_bits<<<blocks(nS), 256, 0, st>>>(P, sph, own, nS, D, numAnal, planeBits, clear, nClear);
    return hipGetLastError();
}

hipError_t launch_direct_plane_sums(const DirectList& D, uint32_t nC, const uint32_t* idA, const uint32_t* idB,
                                    const uint8_t* ctype, const deme_anal_obj* anal, const PlaneSums& sums,
                                    hipStream_t st) {
    if (nC == 0) return hipSuccess;
    k_direct_plane_sums<<<blocks(nC), 256, 0, st>>>(D, nC, idA, idB, ctype, anal, sums);
    return hipGetLastError();
}

hipError_t launch_direct_leave(const DirectList& D, const uint32_t* cidx, const uint32_t* rowStart, float4* listHist,
                               hipStream_t st, SpecGuard guard) {
    const uint32_t pb = blocks(D.nPair), g = pb + blocks(D.nPlane);
    if (g == 0) return hipSuccess;
    k_direct_leave<<<g, 256, 0, st>>>(D, pb, cidx, rowStart, listHist, guard);
    return hipGetLastError();
}

}  // namespace deme_int
