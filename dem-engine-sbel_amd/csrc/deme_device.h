// Device-side records and arithmetic helpers for the DEM hot path on gfx950.
//
// All device code is compiled with -ffp-contract=off and IEEE division/sqrt, so every double/float operation rounds
// exactly like the reference's arithmetic (no fused multiply-adds are introduced).
#pragma once

#ifndef __HIPCC_RTC__
#include <hip/hip_runtime.h>
#include <stdint.h>
#endif

#include "../../include/deme/deme_types.h"

namespace deme_dev {

// --------------------------------------------------------------------------------------------------------------
// HBM-resident records. Owner state is kept as one 64-byte record per owner so that the force kernel's random
// owner gathers touch a single 64-byte segment instead of a dozen SoA cache lines.
// --------------------------------------------------------------------------------------------------------------
struct __attribute__((aligned(16))) OwnerRec {
    uint64_t voxel;       // voxelID_t
    uint16_t lx, ly, lz;  // subVoxelPos_t
    uint8_t fam;          // family_t
    uint8_t pad0;
    float qw, qx, qy, qz;  // oriQ
    float vx, vy, vz;      // linear velocity
    float wx, wy, wz;      // body-frame angular velocity (omgBar)
    float mass;
    uint32_t scene;  // independent scene of a batch (0 for a single scene)
};
static_assert(sizeof(OwnerRec) == 64, "OwnerRec must be 64 bytes");

// Sphere component template, flattened per sphere (ClumpCompAcqStratAllFlatten.cu).
struct __attribute__((aligned(16))) SphereRec {
    uint32_t owner;
    float r;
    float rx, ry, rz;
    uint32_t mat;
    uint32_t pad0, pad1;
};
static_assert(sizeof(SphereRec) == 32, "SphereRec must be 32 bytes");

// Per-sphere contact-detection record written once per detection pass: world position (relative to the world's
// left-bottom-front corner) in double, the sphere radius in float, and the sphere id.
struct __attribute__((aligned(16))) CdRec {
    double x, y, z;
    float r;
    uint32_t id;
};
static_assert(sizeof(CdRec) == 32, "CdRec must be 32 bytes");

// A sphere's position at a candidate build, in fixed point: coordinate = q * unit, unit a power of two chosen so that
// +-2^31 units cover twice the bin grid's extent (rounding error at most unit / 2 per axis). INT32_MIN on an axis marks
// a position that did not fit (or was not a number).
struct BuildPos {
    int32_t x, y, z;
};
static_assert(sizeof(BuildPos) == 12, "BuildPos must be 12 bytes");

// Per-contact outputs of the force kernel (contactForces, contactTorque_convToForce, contactPointGeometryA/B).
struct __attribute__((aligned(16))) ForceRec {
    float fx, fy, fz;
    float tx, ty, tz;
    float ax, ay, az;
    float bx, by, bz;
};
static_assert(sizeof(ForceRec) == 48, "ForceRec must be 48 bytes");

// World pose of one analytical component, recomputed whenever owner states change.
struct __attribute__((aligned(16))) PlanePose {
    double px, py, pz;
    float nx, ny, nz;
    uint32_t owner;
    uint32_t fam;
    uint32_t type;
};
static_assert(sizeof(PlanePose) == 48, "PlanePose must be 48 bytes");

// Inspector quantities (DEMInspector::switch_quantity_type, AuxClasses.cpp:58-103) and reductions; the tile of the
// inspection kernels (256 threads, 8 coalesced strides each).
enum { INSPECT_CLUMP_MAX_Z = 0, INSPECT_CLUMP_MIN_Z = 1, INSPECT_CLUMP_MAX_ABSV = 2, INSPECT_CLUMP_VOLUME = 3 };
enum { INSPECT_MAX = 0, INSPECT_MIN = 1, INSPECT_SUM = 2 };
constexpr int INSPECT_BLOCK = 256, INSPECT_ITEMS = 8;

// Kernel-visible simulation constants.
struct KParams {
    double l, voxelSize, binSize;
    uint32_t nbX, nbY, nbZ;
    uint32_t nBins;  // nbX * nbY * nbZ (< 2^32, checked on the host)
    uint32_t nvX, nvY;
    float beta, h;
    float Gx, Gy, Gz;
    uint32_t integrator;
    uint32_t nS, nA;  // sphere and analytical-component counts (bounds of data-dependent gathers)
    // Analytical components are grouped by scene: scene k owns components planeStart[k] .. planeStart[k + 1] - 1
    // (at most 64). A single scene has planeStart = {0, nA}.
    const uint32_t* planeStart;
    uint32_t nScenes;
    // what the frictional model makes of each pair of materials (a, b), at pairs[a * nM + b]
    uint32_t nM;
    const struct MatPair* pairs;
    uint32_t oneSphere;  // 1: clump o is sphere o alone (its row bounds need no look-up of its spheres)
};

// Effective parameters of a pair of materials and the damping ratio of its restitution (0 to 1, negative).
struct alignas(16) MatPair {
    float E, G, mu, Crr, beta, pad[3];
};
__device__ __forceinline__ MatPair load_pair(const KParams& P, uint32_t a, uint32_t b) {
    const float4* q = reinterpret_cast<const float4*>(P.pairs + a * P.nM + b);
    const float4 v = q[0];
    MatPair m;
    m.E = v.x;
    m.G = v.y;
    m.mu = v.z;
    m.Crr = v.w;
    m.beta = reinterpret_cast<const float*>(q)[4];
    return m;
}

// Range of analytical components a body of the given scene can touch.
__device__ __forceinline__ void scene_planes(const KParams& P, uint32_t scene, uint32_t& a0, uint32_t& a1) {
    if (P.nScenes == 1) {
        // one scene: every component (no table lookup on the dependent-load chain)
        a0 = 0;
        a1 = scene == 0 ? P.nA : 0;
    } else if (scene < P.nScenes) {
        a0 = P.planeStart[scene];
        a1 = P.planeStart[scene + 1];
    } else {
        a0 = a1 = 0;
    }
}

// --------------------------------------------------------------------------------------------------------------
// Saturating float->integer conversions (the reference's device conversions saturate; NaN -> 0).
// --------------------------------------------------------------------------------------------------------------
__device__ __forceinline__ uint32_t sat_u32(double x) {
    if (!(x > 0.0)) return 0u;
    if (x >= 4294967295.0) return 0xFFFFFFFFu;
    return (uint32_t)x;
}
__device__ __forceinline__ uint16_t sat_u16(double x) {
    if (!(x > 0.0)) return 0;
    if (x >= 65535.0) return 65535;
    return (uint16_t)(uint32_t)x;
}
__device__ __forceinline__ uint64_t sat_u64(double x) {
    if (!(x > 0.0)) return 0ull;
    if (x >= 18446744073709551616.0) return ~0ull;
    return (uint64_t)x;
}

// voxelIDToPosition<double, voxelID_t, subVoxelPos_t> (DEMHelperKernels.cu:93-110)
__device__ __forceinline__ void owner_position(const KParams& P, uint64_t id, uint16_t lx, uint16_t ly, uint16_t lz,
                                               double& X, double& Y, double& Z) {
    const uint64_t vx = id & (((uint64_t)1 << P.nvX) - 1);
    const uint64_t vy = (id >> P.nvX) & (((uint64_t)1 << P.nvY) - 1);
    const uint64_t vz = id >> (P.nvX + P.nvY);
    X = (double)vx * P.voxelSize + (double)lx * P.l;
    Y = (double)vy * P.voxelSize + (double)ly * P.l;
    Z = (double)vz * P.voxelSize + (double)lz * P.l;
}

// positionToVoxelID<voxelID_t, subVoxelPos_t, double> (DEMHelperKernels.cu:113-135)
__device__ __forceinline__ void position_to_voxel(const KParams& P, double X, double Y, double Z, uint64_t& id,
                                                  uint16_t& lx, uint16_t& ly, uint16_t& lz) {
    const uint64_t nx = sat_u64(X / P.voxelSize), ny = sat_u64(Y / P.voxelSize), nz = sat_u64(Z / P.voxelSize);
    lx = sat_u16((X - (double)nx * P.voxelSize) / P.l);
    ly = sat_u16((Y - (double)ny * P.voxelSize) / P.l);
    lz = sat_u16((Z - (double)nz * P.voxelSize) / P.l);
    id = nx + (ny << P.nvX) + (nz << (P.nvX + P.nvY));
}

// applyOriQToVector3<float, float> (DEMHelperKernels.cu:137-148)
__device__ __forceinline__ void rotate(float& X, float& Y, float& Z, float Qw, float Qx, float Qy, float Qz) {
    const float oX = X, oY = Y, oZ = Z;
    X = (2.0f * (Qw * Qw + Qx * Qx) - 1.0f) * oX + (2.0f * (Qx * Qy - Qw * Qz)) * oY + (2.0f * (Qx * Qz + Qw * Qy)) * oZ;
    Y = (2.0f * (Qx * Qy + Qw * Qz)) * oX + (2.0f * (Qw * Qw + Qy * Qy) - 1.0f) * oY + (2.0f * (Qy * Qz - Qw * Qx)) * oZ;
    Z = (2.0f * (Qx * Qz - Qw * Qy)) * oX + (2.0f * (Qy * Qz + Qw * Qx)) * oY + (2.0f * (Qw * Qw + Qz * Qz) - 1.0f) * oZ;
}

// locateMaskPair (DEMHelperKernels.cu:51-56)
__device__ __forceinline__ uint32_t mask_index(uint32_t i, uint32_t j) {
    if (i > j) {
        const uint32_t t = i;
        i = j;
        j = t;
    }
    return (1 + j) * j / 2 + i;
}

// Sphere world position as every reference kernel derives it: owner position in double plus the float-rotated
// component offset (DEMBinSphereKernels.cu:39-51).
__device__ __forceinline__ void sphere_position(const KParams& P, const OwnerRec& o, const SphereRec& s, double& X,
                                                double& Y, double& Z) {
    double ox, oy, oz;
    owner_position(P, o.voxel, o.lx, o.ly, o.lz, ox, oy, oz);
    float rx = s.rx, ry = s.ry, rz = s.rz;
    rotate(rx, ry, rz, o.qw, o.qx, o.qy, o.qz);
    X = ox + (double)rx;
    Y = oy + (double)ry;
    Z = oz + (double)rz;
}

__device__ __forceinline__ OwnerRec load_owner(const OwnerRec* __restrict__ p, uint32_t i) {
    // four 16-byte loads
    const uint4* q = reinterpret_cast<const uint4*>(p + i);
    uint4 a = q[0], b = q[1], c = q[2], d = q[3];
    OwnerRec r;
    uint4* w = reinterpret_cast<uint4*>(&r);
    w[0] = a;
    w[1] = b;
    w[2] = c;
    w[3] = d;
    return r;
}

__device__ __forceinline__ SphereRec load_sphere(const SphereRec* __restrict__ p, uint32_t i) {
    const uint4* q = reinterpret_cast<const uint4*>(p + i);
    uint4 a = q[0], b = q[1];
    SphereRec r;
    uint4* w = reinterpret_cast<uint4*>(&r);
    w[0] = a;
    w[1] = b;
    return r;
}

__device__ __forceinline__ CdRec load_cd(const CdRec* __restrict__ p, uint32_t i) {
    const uint4* q = reinterpret_cast<const uint4*>(p + i);
    uint4 a = q[0], b = q[1];
    CdRec r;
    uint4* w = reinterpret_cast<uint4*>(&r);
    w[0] = a;
    w[1] = b;
    return r;
}

// ERRBIT_STALE: a sphere moved too far since the candidate lists were built; they must be rebuilt and the pass redone
// ERRBIT_EDGE: a sphere too near the bin grid's upper ends for stepping on the candidates
// ERRBIT_DRIVEN: a plane owner that its contacts' forces move (see DirectList), whose update was left out
enum : uint32_t {
    ERRBIT_CAPACITY = 1u,
    ERRBIT_PAIR_OVERFLOW = 2u,
    ERRBIT_OUTSIDE = 4u,
    ERRBIT_STALE = 8u,
    ERRBIT_EDGE = 16u,
    ERRBIT_DRIVEN = 32u
};

// --------------------------------------------------------------------------------------------------------------
// The contact predicate of detection: expanded overlap, plane distance, and the contact-point bin rule.
// --------------------------------------------------------------------------------------------------------------
struct BinRange {
    uint32_t x0, x1, y0, y1, z0, z1;
};

// DEMBinSphereKernels.cu:52-64 (double position and radius span, truncating conversions)
__device__ __forceinline__ BinRange bin_range(const KParams& P, double X, double Y, double Z, double rCD) {
    const double bx = X / P.binSize, by = Y / P.binSize, bz = Z / P.binSize, span = rCD / P.binSize;
    BinRange r;
    r.x0 = sat_u32(bx - span);
    r.x1 = sat_u32(bx + span);
    r.y0 = sat_u32(by - span);
    r.y1 = sat_u32(by + span);
    r.z0 = sat_u32(bz - span);
    r.z1 = sat_u32(bz + span);
    return r;
}

// checkSphereEntityOverlap<double> without contact point (DEMHelperKernels.cu:356-391); rCD already holds r + beta.
__device__ __forceinline__ bool plane_cd(const KParams& P, const PlanePose& pp, double X, double Y, double Z,
                                         double rCD) {
    if (pp.type != DEME_ANAL_OBJ_TYPE_PLANE) return false;
    const double dx = X - pp.px, dy = Y - pp.py, dz = Z - pp.pz;
    const double dist = dx * (double)pp.nx + dy * (double)pp.ny + dz * (double)pp.nz;
    return !(dist > rCD + (double)P.beta);
}

__device__ __forceinline__ bool range_in_grid(const KParams& P, const BinRange& r) {
    return r.x1 < P.nbX && r.y1 < P.nbY && r.z1 < P.nbZ;
}

// Membership of a linear bin id in the linear ids of a range (the reference's bins may alias when a range crosses
// the grid's upper faces; this enumerates exactly the ids the reference would form).
// (Out of line: the rare path. Arguments by value, so the caller's ranges stay in registers.)
static __device__ __noinline__ bool range_has_linear(uint32_t nbX, uint32_t nbY, BinRange r, uint32_t lin) {
    const uint32_t nbXY = nbX * nbY;
    for (uint32_t k = 0; k <= r.z1 - r.z0; k++)
        for (uint32_t j = 0; j <= r.y1 - r.y0; j++)
            for (uint32_t i = 0; i <= r.x1 - r.x0; i++)
                if ((r.x0 + i) + (r.y0 + j) * nbX + (r.z0 + k) * nbXY == lin) return true;
    return false;
}

// Expanded radius as the reference's detection kernel forms it: float(r + beta), widened to double.
__device__ __forceinline__ double expanded_radius(const KParams& P, float r) {
    float rf = r;
    rf += P.beta;
    return (double)rf;
}

// First half of the reference's sphere-pair test (checkSpheresOverlap<double>, DEMHelperKernels.cu:195-205): the
// expanded spheres overlap.
__device__ __forceinline__ bool expanded_overlap(double ra, const CdRec& A, double rb, const CdRec& B) {
    const double dx = A.x - B.x, dy = A.y - B.y, dz = A.z - B.z;
    const double d2 = dx * dx + dy * dy + dz * dz;
    return !(d2 > (ra + rb) * (ra + rb));
}

// Second half, for a pair that overlaps: the contact point (DEMHelperKernels.cu:206-222) computed with A the lower id,
// and its bin inside both spheres' AABB bin ranges.
struct RuleBins {
    uint32_t ix, iy, iz;
    BinRange ga, gb;
};

__device__ __forceinline__ void contact_point(const KParams& P, const CdRec& A, const CdRec& B, double& cx, double& cy,
                                              double& cz) {
    const double ra = expanded_radius(P, A.r), rb = expanded_radius(P, B.r);
    const double dx = A.x - B.x, dy = A.y - B.y, dz = A.z - B.z;
    const double d2 = dx * dx + dy * dy + dz * dz;
    float nX = (float)dx, nY = (float)dy, nZ = (float)dz;
    const float mag = sqrtf(nX * nX + nY * nY + nZ * nZ);
    nX /= mag;
    nY /= mag;
    nZ /= mag;
    const double half = (ra + rb - sqrt(d2)) / 2.0;
    cx = B.x + (rb - half) * (double)nX;
    cy = B.y + (rb - half) * (double)nY;
    cz = B.z + (rb - half) * (double)nZ;
}

__device__ __forceinline__ double cd_radius(const KParams& P, float r) {
    double v = (double)r;
    v += (double)P.beta;
    return v;
}

// The reference's bin indices, with its divisions by binSize.
__device__ __forceinline__ void rule_bins_exact(const KParams& P, const CdRec& A, const CdRec& B, double cx, double cy,
                                                double cz, RuleBins& R) {
    R.ix = sat_u32(cx / P.binSize);
    R.iy = sat_u32(cy / P.binSize);
    R.iz = sat_u32(cz / P.binSize);
    R.ga = bin_range(P, A.x, A.y, A.z, cd_radius(P, A.r));
    R.gb = bin_range(P, B.x, B.y, B.z, cd_radius(P, B.r));
}

// The same bin indices from multiplications by the reciprocal of the bin size, used when every floor input lies
// farther from an integer than the product and the quotient can differ (a few ulps; the margin is 2^-40 relative):
// then each floor, and so the rule, equals the division's. Returns false when a value is too close to call.
__device__ __forceinline__ bool far_from_int(double t, double scale) {
    const double f = t - floor(t);
    const double eps = 0x1p-40 * (scale + 1.0);
    return f > eps && f < 1.0 - eps;
}

__device__ __forceinline__ bool range_fast(const KParams& P, double inv, double X, double Y, double Z, double rCD,
                                           BinRange& r) {
    const double bx = X * inv, by = Y * inv, bz = Z * inv, span = rCD * inv;
    const double ax = fabs(bx) + span, ay = fabs(by) + span, az = fabs(bz) + span;
    const double x0 = bx - span, x1 = bx + span, y0 = by - span, y1 = by + span, z0 = bz - span, z1 = bz + span;
    if (!(far_from_int(x0, ax) && far_from_int(x1, ax) && far_from_int(y0, ay) && far_from_int(y1, ay) &&
          far_from_int(z0, az) && far_from_int(z1, az)))
        return false;
    r.x0 = sat_u32(x0);
    r.x1 = sat_u32(x1);
    r.y0 = sat_u32(y0);
    r.y1 = sat_u32(y1);
    r.z0 = sat_u32(z0);
    r.z1 = sat_u32(z1);
    return true;
}

__device__ __forceinline__ bool rule_bins_fast(const KParams& P, double inv, const CdRec& A, const CdRec& B, double cx,
                                               double cy, double cz, RuleBins& R) {
    const double qx = cx * inv, qy = cy * inv, qz = cz * inv;
    if (!(far_from_int(qx, fabs(qx)) && far_from_int(qy, fabs(qy)) && far_from_int(qz, fabs(qz)))) return false;
    R.ix = sat_u32(qx);
    R.iy = sat_u32(qy);
    R.iz = sat_u32(qz);
    return range_fast(P, inv, A.x, A.y, A.z, cd_radius(P, A.r), R.ga) &&
           range_fast(P, inv, B.x, B.y, B.z, cd_radius(P, B.r), R.gb);
}

__device__ __forceinline__ bool rule_member(const KParams& P, const RuleBins& R) {
    if (range_in_grid(P, R.ga) && range_in_grid(P, R.gb)) {
        // no aliasing: a linear id is one (i, j, k) -- unless the point itself lies past the grid, where the
        // reference's linear id aliases; fall through to the exact enumeration then
        if (R.ix < P.nbX && R.iy < P.nbY && R.iz < P.nbZ)
            return R.ix >= R.ga.x0 && R.ix <= R.ga.x1 && R.iy >= R.ga.y0 && R.iy <= R.ga.y1 && R.iz >= R.ga.z0 &&
                   R.iz <= R.ga.z1 && R.ix >= R.gb.x0 && R.ix <= R.gb.x1 && R.iy >= R.gb.y0 && R.iy <= R.gb.y1 &&
                   R.iz >= R.gb.z0 && R.iz <= R.gb.z1;
    }
    const uint32_t lin = R.ix + R.iy * P.nbX + R.iz * P.nbX * P.nbY;
    return range_has_linear(P.nbX, P.nbY, R.ga, lin) && range_has_linear(P.nbX, P.nbY, R.gb, lin);
}

// True only when the bin rule of an overlapping pair must hold. The exact contact point lies inside both expanded
// spheres, ra - half from A's centre and rb - half from B's (half: half the overlap, at most the smaller radius), so its
// bin lies in both spheres' bin ranges as soon as half exceeds what rounding can move: the float-rounded direction
// moves the point by under 6e-7 (ra + rb), float(r + beta) differs from r + beta by under 6e-8 (ra + rb), and the
// double positions and quotients add a few 2^-52 of the coordinates. Floors and saturation are monotone, and a triple
// inside both ranges is among the linear ids of both, so the aliasing cases agree. Everything else (grazing pairs,
// near-coincident centres, one sphere deep inside another, NaN) answers false and takes the full rule.
__device__ __forceinline__ bool bin_rule_certain(double ra, const CdRec& A, double rb, const CdRec& B) {
    const double dx = A.x - B.x, dy = A.y - B.y, dz = A.z - B.z;
    const double sum = ra + rb, dist = sqrt(dx * dx + dy * dy + dz * dz), half = 0.5 * (sum - dist);
    const double reach = fabs(A.x) + fabs(A.y) + fabs(A.z) + sum;
    return half > 1e-6 * sum + 0x1p-46 * reach && half <= fmin(ra, rb) && dist > 1e-3 * sum && sum > 1e-12;
}

// A: the lower id of an overlapping pair. inv: 1 / binSize.
__device__ __forceinline__ bool bin_rule_point(const KParams& P, double inv, const CdRec& A, const CdRec& B) {
    if (bin_rule_certain(expanded_radius(P, A.r), A, expanded_radius(P, B.r), B)) return true;
    double cx, cy, cz;
    contact_point(P, A, B, cx, cy, cz);
    RuleBins R;
    if (!rule_bins_fast(P, inv, A, B, cx, cy, cz, R)) rule_bins_exact(P, A, B, cx, cy, cz, R);
    return rule_member(P, R);
}

// The rule for pairs whose spheres' ranges lie inside the grid on every axis, the contact point with them (no linear id
// aliases then, so membership is per axis), one axis at a time: the force kernel's registers are taken, and the general
// form inlined there costs it a wave per SIMD (140 registers; out of line, 150). A: the lower id.
__device__ __forceinline__ bool axis_in_ranges(double binSize, double c, double xa, double ra, double xb, double rb) {
    const uint32_t i = sat_u32(c / binSize);
    const double ba = xa / binSize, sa = ra / binSize;
    if (i < sat_u32(ba - sa) || i > sat_u32(ba + sa)) return false;
    const double bb = xb / binSize, sb = rb / binSize;
    return !(i < sat_u32(bb - sb) || i > sat_u32(bb + sb));
}
__device__ __forceinline__ bool bin_rule_inside(const KParams& P, const CdRec& A, const CdRec& B) {
    if (bin_rule_certain(expanded_radius(P, A.r), A, expanded_radius(P, B.r), B)) return true;
    double cx, cy, cz;
    contact_point(P, A, B, cx, cy, cz);
    const double ra = cd_radius(P, A.r), rb = cd_radius(P, B.r);
    if (!axis_in_ranges(P.binSize, cx, A.x, ra, B.x, rb)) return false;
    __builtin_amdgcn_sched_barrier(0);
    if (!axis_in_ranges(P.binSize, cy, A.y, ra, B.y, rb)) return false;
    __builtin_amdgcn_sched_barrier(0);
    return axis_in_ranges(P.binSize, cz, A.z, ra, B.z, rb);
}

// The bin-range check of a sphere's detection record: ERRBIT_CAPACITY when it touches more bins than the reference can
// count, ERRBIT_OUTSIDE when a bin of its range lies past the grid, 0 when neither.
__device__ __forceinline__ uint32_t bin_range_err(const KParams& P, const BinRange& r) {
    const uint32_t nx = r.x1 - r.x0 + 1, ny = r.y1 - r.y0 + 1, nz = r.z1 - r.z0 + 1;
    if ((uint64_t)nx * ny * nz > 65535u) return ERRBIT_CAPACITY;
    // The linear id grows with each of i, j, k, so without 32-bit wrap the range's largest id is its last corner.
    const uint32_t nbXY = P.nbX * P.nbY;
    const uint64_t last = (uint64_t)r.x1 + (uint64_t)r.y1 * P.nbX + (uint64_t)r.z1 * nbXY;
    bool outside = last >= P.nBins;
    if (last > 0xFFFFFFFFull) {
        // ids wrap: enumerate them as the reference forms them
        outside = false;
        for (uint32_t dk = 0; dk < nz; dk++)
            for (uint32_t dj = 0; dj < ny; dj++)
                for (uint32_t di = 0; di < nx; di++)
                    outside |= ((r.x0 + di) + (r.y0 + dj) * P.nbX + (r.z0 + dk) * nbXY) >= P.nBins;
    }
    return outside ? ERRBIT_OUTSIDE : 0u;
}

// World pose of an analytical component from its owner's state.
__device__ __forceinline__ PlanePose plane_pose_of(const KParams& P, const deme_anal_obj& ob, const OwnerRec& o) {
    double ox, oy, oz;
    owner_position(P, o.voxel, o.lx, o.ly, o.lz, ox, oy, oz);
    float px = ob.relPos[0], py = ob.relPos[1], pz = ob.relPos[2];
    float nx = ob.rot[0], ny = ob.rot[1], nz = ob.rot[2];
    rotate(px, py, pz, o.qw, o.qx, o.qy, o.qz);
    rotate(nx, ny, nz, o.qw, o.qx, o.qy, o.qz);
    PlanePose pp;
    pp.px = ox + (double)px;
    pp.py = oy + (double)py;
    pp.pz = oz + (double)pz;
    pp.nx = nx;
    pp.ny = ny;
    pp.nz = nz;
    pp.owner = ob.owner;
    pp.fam = o.fam;
    pp.type = ob.type;
    return pp;
}

// Sums over the sphere-plane contacts per analytical owner, passed from the force kernel to the owner update. Each
// force workgroup (ANAL_TILE contacts) marks the owners that it has terms for (a bit each, mark[block]) and writes their 6
// partial sums at part[(block * nOwners + owner) * 6]; the owner update folds those of nPart blocks (PART_FROM_COUNTERS:
// the number of blocks of the guard's contact count).
constexpr uint32_t PART_FROM_COUNTERS = 0xFFFFFFFFu;
constexpr uint32_t PLANES_BY_LIST = 0x100u;  // (see DirectList)
constexpr uint32_t MAX_ANAL_OWNERS = 8;
struct PlaneSums {
    float* part = nullptr;
    uint8_t* mark = nullptr;
    uint32_t first = 0, nOwners = 0;  // owner numbers first .. first + nOwners - 1
    uint32_t nPart = 0;
    uint32_t flags = 0;  // a bit for each owner that the update leaves as it is, and PLANES_BY_LIST
};
// The workgroup's partial sums of the plane owners' terms (gOwner < 0: the lane has none): per owner, wave butterflies
// and the four waves in order, a fixed tree. Every lane of the workgroup calls this. Folding here instead of storing a
// term per contact and launching two more kernels over the list saves those launches (6-9 us each at any size).
__device__ __forceinline__ void fold_plane_terms(const PlaneSums& sums, int gOwner, const float (&g)[6]) {
    if (sums.nOwners == 0) return;
    __shared__ float waveSum[4][6];
    __shared__ uint32_t waveMark[4];
    static_assert(MAX_ANAL_OWNERS <= 8, "a bit of mark[] per owner");
    uint32_t mine = 0;
    for (uint32_t k = 0; k < sums.nOwners; k++) mine |= __any(gOwner == (int)k) ? 1u << k : 0u;
    if ((threadIdx.x & 63u) == 0) waveMark[threadIdx.x >> 6] = mine;
    __syncthreads();
    const uint32_t mark = waveMark[0] | waveMark[1] | waveMark[2] | waveMark[3];
    if (threadIdx.x == 0) sums.mark[blockIdx.x] = (uint8_t)mark;
    float* dst = sums.part + (uint64_t)blockIdx.x * sums.nOwners * 6;
    for (uint32_t k = 0; k < sums.nOwners; k++) {
        if (!(mark >> k & 1u)) continue;
        if (mine >> k & 1u) {
#pragma unroll
            for (int c = 0; c < 6; c++) {
                float v = gOwner == (int)k ? g[c] : 0.f;
#pragma unroll
                for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
                if ((threadIdx.x & 63u) == 0) waveSum[threadIdx.x >> 6][c] = v;
            }
        } else if ((threadIdx.x & 63u) < 6) {
            waveSum[threadIdx.x >> 6][threadIdx.x & 63u] = 0.f;
        }
        __syncthreads();
        if (threadIdx.x < 6) {
            const uint32_t c = threadIdx.x;
            dst[k * 6 + c] = ((waveSum[0][c] + waveSum[1][c]) + waveSum[2][c]) + waveSum[3][c];
        }
        __syncthreads();
    }
}
// What the owner update refreshes after moving the analytical owners: the poses of all nA components (pose null: none).
struct PlaneRefresh {
    const deme_anal_obj* anal = nullptr;
    PlanePose* pose = nullptr;
    uint32_t nA = 0;
};

// Device-side counters read back by the host after a detection pass.
struct DevCounters {
    uint32_t pairCount;
    uint32_t err;
    uint32_t maxOcc;
    uint32_t pad;
    unsigned long long nActive;
    unsigned long long total[4];
    uint32_t pad1[18];
    // of the contacts listed with a drift margin, a sample (every 64th workgroup of candidates) and those that touch; on a
    // line of their own, since every wave that counts them reads err first
    uint32_t sampled, touching, pad2[30];
    // largest squared displacement (bits of a non-negative double) of a sphere since the candidate lists were built,
    // spread over DISP_SLOTS words (workgroup b folds into word b % DISP_SLOTS: one address per workgroup would
    // serialize the atomics); the largest word is the maximum
    unsigned long long disp2[64];
    // per axis, the extremes of the spheres' displacements since the build (same slots; order-preserving integer
    // images of the doubles, the minima complemented, so every word folds with atomicMax from a cleared zero)
    unsigned long long dispLo[3][64], dispHi[3][64];
};
static_assert(__builtin_offsetof(DevCounters, sampled) == 128 && __builtin_offsetof(DevCounters, disp2) == 256,
              "the sample's counters have a cache line of their own");
constexpr uint32_t DISP_SLOTS = 64;
// The host reads the counters up to the displacement extremes (the device alone uses those).
constexpr size_t DEV_COUNTERS_HOST_BYTES = __builtin_offsetof(DevCounters, dispLo);

// Order-preserving image of a double as an unsigned 64-bit integer (and back).
__host__ __device__ inline unsigned long long ordered_bits(double x) {
    unsigned long long b;
    __builtin_memcpy(&b, &x, sizeof(b));
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}
__host__ __device__ inline double from_ordered_bits(unsigned long long b) {
    b = (b >> 63) ? (b & 0x7FFFFFFFFFFFFFFFull) : ~b;
    double x;
    __builtin_memcpy(&x, &b, sizeof(x));
    return x;
}

__host__ __device__ inline double max_disp2(const DevCounters& c) {
    unsigned long long m = 0;
    for (uint32_t k = 0; k < DISP_SLOTS; k++) m = c.disp2[k] > m ? c.disp2[k] : m;
    double d;
    __builtin_memcpy(&d, &m, sizeof(d));
    return d;
}

// Kernels enqueued before the host has read a detection pass's counters (so the GPU does not wait for the host, or
// the whole step sits in a captured graph) exit at once, writing nothing, when the pass failed, a slab row
// overflowed, or the contact / mirror-row totals exceed the buffers they were given; the host then redoes them.
// Kernels over contacts then take the contact count from ctr->total[1]. ctr == nullptr: no guard.
struct SpecGuard {
    const DevCounters* ctr = nullptr;
    uint32_t slabCap = 0;
    unsigned long long capC = 0, capP = 0;
};
__device__ __forceinline__ bool spec_skip(const SpecGuard& g) {
    return g.ctr && (g.ctr->err || g.ctr->maxOcc > g.slabCap || g.ctr->total[1] > g.capC || g.ctr->total[2] > g.capP);
}

// --------------------------------------------------------------------------------------------------------------
// Stepping on the candidates: between list builds, the force kernel takes the build's candidates themselves (one lane
// each: the predicate, then the force of those that touch), with histories and owner terms kept by candidate, and the
// owner update sums over the candidate rows. No contact list is formed in between.
// --------------------------------------------------------------------------------------------------------------
// err: set by the checks of a state (ERRBIT_*), sticky; the force kernel copies it to skip, which the owner update of
// the same step obeys (that kernel itself checks the state it leaves, so it cannot read err); steps: owner updates
// done; held: the plane owners left where they are (a bit each); disp: the largest displacements since the build (bits of
// doubles, spread over DISP_SLOTS words).
struct DirectState {
    // lines of their own: a word read by every wave beside one that atomics change misses the caches
    uint32_t err, pad0[31], skip, pad1[31], steps, held, pad2[30];
    unsigned long long disp[64];
};
// The candidates: pairs c < nPair (candA < candB, tPos: slot of c in the transposed rows) and planes q < nPlane (sphere
// pSph, component pPlane; rows pStart by sphere). on / pOn: touched in the last step, whose history then stands in hist /
// pHist; bOn: on by transposed slot. aTerm: A's owner terms; bTerm: B's, by transposed slot; pTerm: A's of the planes, and
// behind them, from 6 nPlane on, the plane owners'. A clump's terms are summed in the list's order. The plane owners' sums
// are folded by the places of the plane candidates, which depend on the lists: their last bits may reach an owner's
// accelerations (which the last step of a call, a pass's, writes anew) but not its motion. Where the forces would move one
// (its velocities not prescribed) the owner update leaves it where it is and reports ERRBIT_DRIVEN; the host then sums that
// step's terms by the contact list's places and moves it. PLANES_BY_LIST: so with any plane owner (family change rules that
// read the accelerations).
// (No more fields than these: three more words of kernel arguments cost 600 spheres 0.35 us a step.)
struct DirectList {
    uint32_t nPair, nPlane;
    const uint32_t *candA, *candB, *tPos, *pSph, *pPlane, *pStart;
    uint8_t *on, *pOn, *bOn;
    float4 *hist, *pHist;
    float* pTerm;
    const uint8_t* mask;  // family mask, null when every pair is allowed
    DirectState* st;      // null: not stepping on candidates
};
// An owner's pose at a candidate build: its position in fixed point (as BuildPos), its orientation, and the largest
// distance of its spheres' centres from it.
struct __attribute__((aligned(16))) OwnerBuild {
    int32_t x, y, z;
    float relMax;
    float qw, qx, qy, qz;
};
static_assert(sizeof(OwnerBuild) == 32, "OwnerBuild must be 32 bytes");
// What the owner update checks of the state it leaves: no sphere farther than limit from its position at the build
// (bounded by its owner's motion since, own0, positions in units of unit), every sphere clear of the bin grid's upper ends
// (its upper corner below hiX, hiY, hiZ: its bin range, and the contact point of any pair, then lie inside the grid; the
// host's limits are minus infinity where a sphere could touch too many bins; an owner more than past below them needs no
// look at its spheres), and no component moved by more than planeLimit since the plane candidates were made (pose0; reach
// bounds a sphere's distance from the origin). A state that fails is left to the contact-list path: its pass reports an
// error, or goes on.
struct DirectCheck {
    const OwnerBuild* own0;
    const SphereRec* sph;
    const uint32_t* ownerSphStart;
    double unit, limit;
    double hiX, hiY, hiZ, past;
    const PlanePose* pose0;
    double planeLimit, reach;
};

// The spheres of an owner near the grid's upper ends, one by one (in the general case an upper wall's layer: a clump's
// bound past it would send a third of all worlds to the contact-list path).
__device__ __forceinline__ uint32_t direct_edge(const KParams& P, const DirectCheck& C, const OwnerRec& r, uint32_t o) {
    for (uint32_t s = C.ownerSphStart[o]; s < C.ownerSphStart[o + 1]; s++) {
        const SphereRec sr = load_sphere(C.sph, s);
        double X, Y, Z;
        sphere_position(P, r, sr, X, Y, Z);
        const double rCD = cd_radius(P, sr.r);
        if (!(X + rCD < C.hiX && Y + rCD < C.hiY && Z + rCD < C.hiZ)) return ERRBIT_EDGE;
    }
    return 0;
}

// One owner's part of the check: ERRBIT_* bits, disp raised to the bound of its spheres' displacement. A sphere moves by
// at most |dX| + |R(q) - R(q0)| relMax, and R is quadratic: R(q) - R(q0) = 2 M(q - q0, q + q0) with M symmetric and
// bilinear, |M(a, b)| at most |a| |b| / 2 for orthogonal a, b and |a| |b| else, so with a = q - q0, b = q + q0
// |R(q) - R(q0)| <= |a| |b| + 2 ||q|^2 - |q0|^2| (the tight bound for unit quaternions, whatever the drift of their
// norms). 1e-6 covers the float rounding of the four products. Per owner, not per sphere: 32 bytes instead of 44 for each
// of its spheres (1M three-sphere clumps, 4.98M candidates: the owner update 150 -> 140 us).
__device__ __forceinline__ uint32_t direct_check_owner(const KParams& P, const DirectCheck& C, const OwnerRec& r,
                                                       uint32_t o, double& disp) {
    const uint4* b4 = reinterpret_cast<const uint4*>(C.own0 + o);
    OwnerBuild b;
    uint4* w = reinterpret_cast<uint4*>(&b);
    w[0] = b4[0];
    w[1] = b4[1];
    double X, Y, Z;
    owner_position(P, r.voxel, r.lx, r.ly, r.lz, X, Y, Z);
    uint32_t bad = 0;
    if (!(X + C.past < C.hiX && Y + C.past < C.hiY && Z + C.past < C.hiZ)) bad = direct_edge(P, C, r, o);
    constexpr int32_t unfit = -2147483647 - 1;  // INT32_MIN (hipRTC has no limits)
    const double dx = X - (double)b.x * C.unit, dy = Y - (double)b.y * C.unit, dz = Z - (double)b.z * C.unit;
    double m = sqrt(dx * dx + dy * dy + dz * dz);
    if (b.relMax > 0.f) {
        const float aw = r.qw - b.qw, ax = r.qx - b.qx, ay = r.qy - b.qy, az = r.qz - b.qz;
        const float sw = r.qw + b.qw, sx = r.qx + b.qx, sy = r.qy + b.qy, sz = r.qz + b.qz;
        const float aa = aw * aw + ax * ax + ay * ay + az * az, bb = sw * sw + sx * sx + sy * sy + sz * sz;
        const float par = aw * sw + ax * sx + ay * sy + az * sz;  // |q|^2 - |q0|^2
        m += (double)(sqrtf(aa * bb) + 2.f * fabsf(par) + 1e-6f * (1.f + bb)) * (double)b.relMax;
    }
    if (b.x == unfit || b.y == unfit || b.z == unfit || !(m == m)) m = __builtin_huge_val();
    disp = m > disp ? m : disp;
    return bad;
}

// Whether component a's plane moved too far since its near spheres were listed: the signed distance of any point within
// reach of the origin changes by at most |n.p - n0.p0| + |n - n0| reach.
__device__ __forceinline__ bool direct_plane_moved(const DirectCheck& C, const PlanePose& a, const PlanePose& b) {
    const double oa = a.px * (double)a.nx + a.py * (double)a.ny + a.pz * (double)a.nz;
    const double ob = b.px * (double)b.nx + b.py * (double)b.ny + b.pz * (double)b.nz;
    const double dx = (double)a.nx - (double)b.nx, dy = (double)a.ny - (double)b.ny, dz = (double)a.nz - (double)b.nz;
    return !(fabs(oa - ob) + sqrt(dx * dx + dy * dy + dz * dz) * C.reach <= C.planeLimit);
}

// A workgroup's (256 lanes) displacements and error bits into the state; every lane calls it.
__device__ __forceinline__ void direct_report(DirectState* st, double limit, double disp, uint32_t bad) {
    if (disp > limit) bad |= ERRBIT_STALE;
    // the common case needs no fold: no error, and displacements below an eighth of the limit decide nothing
    if (!__any(bad != 0 || disp > limit * 0.125)) return;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        disp = fmax(disp, __shfl_xor(disp, off, 64));
        bad |= (uint32_t)__shfl_xor((int)bad, off, 64);
    }
    if ((threadIdx.x & 63u) == 0) {
        if (bad) atomicOr(&st->err, bad);
        atomicMax(&st->disp[(blockIdx.x * 4u + (threadIdx.x >> 6)) % DISP_SLOTS],
                  (unsigned long long)__double_as_longlong(disp));
    }
}

}  // namespace deme_dev
