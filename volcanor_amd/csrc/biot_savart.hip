// Biot-Savart N-body kernels for MI355X (gfx950).
//
// Velocity induced by straight vortex segments with the Vatistas n=2 core,
// the leaf vf_vind of the reference (classdef.f90:476-503):
//   v = gam/(4 pi) * (r1 x r2) * [r0 . (r1/|r1| - r2/|r2|)]
//       / sqrt((rc |r0|)^4 + |r1 x r2|^4),
// zero when |r1 x r2|^2 <= eps^2, r/|r| = 0 when |r| <= eps
// (unitVec, libMath.f90:249-262).  Per segment the library precomputes
// r0 = b - a, g = gam/(4 pi) and q = rc^2 |r0|^2; per pair r1 = p - a,
// r2 = r1 - r0 and r1 x r2 = r0 x r1.
//
// Work decomposition: segments come in groups of 32 consecutive records
// with a centre and a far radius (write_group_records); a wave takes 64 or
// 128 targets and one chunk of groups, and runs a shorter pair on every
// group that all its targets are far from (pair64_far, pair32_far).  Each
// (tile, chunk) item writes its own partial sums, which are reduced in a
// fixed order afterwards: results are bitwise repeatable.
//
// What bounds it: vector issue.  No MFMA: n1 and d1 are contractions of
// depth 4, but FP64 and FP32 MFMA run no faster than the vector units here
// (64 and 32 cycles per 16x16x4) and do not overlap with them (16 FMAs and
// one MFMA take the sum of both times).  Measured against pair64 for every
// pair with LDS broadcasts: 4.0e9 pairs on helices 6.5 -> 5.15 ms, a
// quad-rotor wake pass (1.58e10 pairs) 25.4 -> 19.9 ms (8.0e11 pairs/s);
// mixed, 2e10 pairs on helices 14.7 -> 11.3 ms (1.78e12 pairs/s), a rotor
// wake pass (2.2e9 pairs) 2.00 -> 1.46 ms.
//
// Precision modes
//   FP64  : FP64 throughout; 1/sqrt via v_rsq_f64 plus one third-order
//           correction.
//   MIXED : FP32 pair arithmetic, v_rsq_f32, the sums of each group folded
//           into FP64.  Far groups use coordinates relative to the group's
//           centre, the others hi/lo-split coordinates (r1 = (p_hi - a_hi)
//           + (p_lo - a_lo), accurate to FP32 relative precision of r1
//           itself).  Pairs with the target inside the core (within one
//           core radius of the segment) are recomputed in FP64 (the
//           regularised core and target-on-filament terms, where the
//           reference's exact-zero guards act).
//           Launches with fewer than 1024 targets (collocation points, judge
//           samples) run in FP64 in both modes.
#include <algorithm>

#include "vlm_internal.h"

namespace vlm {
namespace {

constexpr int BS_BLOCK = 256;
// constant address space: a load from a wave-uniform address becomes a
// scalar load.  The records are written by earlier launches only.
typedef const double __attribute__((address_space(4))) *cdptr;
typedef const long long __attribute__((address_space(4))) *clptr;
// Whole FP64 records as vectors: one s_load_dwordx16 per eight doubles
// (field by field the compiler issues five smaller loads: 5.38 against
// 5.12 ms for 4.0e9 pairs).
typedef double d8 __attribute__((ext_vector_type(8)));
typedef const d8 __attribute__((address_space(4))) *cd8ptr;


constexpr double EPS2 = kEps * kEps;
constexpr float EPS2F = 4.93038065763132e-32f;
constexpr float NEAR_CORE2 = 1.0f;  // h < rc, and |r1|^2 + |r2|^2 < 4 |r0|^2 (stored)

__device__ __forceinline__ double rsq64(double x)
{
    // v_rsq_f64 is accurate to about 2^-24; one third-order correction
    // y (1 + e/2 + 3 e^2/8) with e = 1 - x y^2 brings it to FP64 rounding
    // (the dropped 5 e^3/16 term is below 2^-69).
    const double y = __builtin_amdgcn_rsq(x);
    const double h = x * y;
    const double e = __builtin_fma(-h, y, 1.0);
    const double c = __builtin_fma(e, 0.375, 0.5);
    return __builtin_fma(y, e * c, y);
}

// x where c holds, else a value that acts as zero here: only the high dword
// (sign, exponent, top of the mantissa) is cleared, one select instead of
// two.  What is left is a positive number below 2^-1042.  It only enters
// products with the components of c = r0 x r1, below 2^-51 when
// |r1 x r2| <= eps, which underflow to exactly 0, so the sums are bitwise
// those of a true zero.
__device__ __forceinline__ double zero_unless(bool c, double x)
{
    const int hi = __double2hiint(x);
    return __hiloint2double(c ? hi : 0, __double2loint(x));
}

// FP64 pair; qq = (rc |r0|)^4, n0 = |r0|^2 (so r0 . r2 = r0 . r1 - n0).
// The reference's r0 . (r1/|r1| - r2/|r2|) / sqrt(qq + c2^2) is evaluated as
// d1 / sqrt(n1 den) - d2 / sqrt(n2 den): two reciprocal square roots per
// pair instead of three.  The pair guard |r1 x r2|^2 <= eps^2 is exact.  The
// unitVec guard (|r| <= eps -> that term 0) is a clamp n >= eps^2, one
// v_max instead of a compare and a select: on an end point (r = 0) the term
// is d * j = 0 exactly, as in the reference; for 0 < |r| <= eps,
// |r1 x r2| <= |r0| |r| lets the pair guard zero the pair whenever
// |r0| <= 1, and for longer segments the term left over is of the order of
// the pair's own (eps-sized) contribution.
__device__ __forceinline__ void pair64(double px, double py, double pz, double ax, double ay,
                                       double az, double g, double r0x, double r0y, double r0z,
                                       double qq, double n0, double &vx, double &vy, double &vz)
{
    const double r1x = px - ax, r1y = py - ay, r1z = pz - az;
    const double r2x = r1x - r0x, r2y = r1y - r0y, r2z = r1z - r0z;
    const double cx = r0y * r1z - r0z * r1y;
    const double cy = r0z * r1x - r0x * r1z;
    const double cz = r0x * r1y - r0y * r1x;
    const double c2 = cx * cx + cy * cy + cz * cz;
    const double n1 = r1x * r1x + r1y * r1y + r1z * r1z;
    const double n2 = r2x * r2x + r2y * r2y + r2z * r2z;
    const double d1 = r0x * r1x + r0y * r1y + r0z * r1z;
    const double d2 = d1 - n0;
    const double den = __builtin_fma(c2, c2, qq);
    const double j1 = rsq64(__builtin_fmax(n1, EPS2) * den);
    const double j2 = rsq64(__builtin_fmax(n2, EPS2) * den);
    const double s = zero_unless(c2 > EPS2, g * (d1 * j1 - d2 * j2));
    vx += cx * s;
    vy += cy * s;
    vz += cz * s;
}

// FP32 pair on split coordinates (a, b: near32; r: r0 and qq, n0).  Returns
// true for near-singular pairs, whose contribution is left to the FP64
// recompute (zero here): targets inside the core and, for segments without a
// core, every target nearby (c2^2 underflows in FP32 long before the exact
// guard acts, and den with it).  Same evaluation order as pair64:
// d1 / sqrt(n1 den) - d2 / sqrt(n2 den).
__device__ __forceinline__ bool pair32(const float *ph, const float *pl, float4 a, float4 b,
                                       float4 r, float n0, float *v)
{
    const float r1x = (ph[0] - a.x) + (pl[0] - b.x);
    const float r1y = (ph[1] - a.y) + (pl[1] - b.y);
    const float r1z = (ph[2] - a.z) + (pl[2] - b.z);
    const float r0x = r.x, r0y = r.y, r0z = r.z, q = b.w;
    const float r2x = r1x - r0x, r2y = r1y - r0y, r2z = r1z - r0z;
    const float cx = r0y * r1z - r0z * r1y;
    const float cy = r0z * r1x - r0x * r1z;
    const float cz = r0x * r1y - r0y * r1x;
    const float c2 = cx * cx + cy * cy + cz * cz;
    const float n1 = r1x * r1x + r1y * r1y + r1z * r1z;
    const float n2 = r2x * r2x + r2y * r2y + r2z * r2z;
    const bool nearp = (c2 < NEAR_CORE2 * q) && (n1 + n2 < 4.0f * n0);
    const float d1 = r0x * r1x + r0y * r1y + r0z * r1z;
    const float d2 = d1 - n0;
    const float den = __builtin_fmaf(c2, c2, r.w);
    const float j1 = __builtin_amdgcn_rsqf(__builtin_fmaxf(n1, EPS2F) * den);
    const float j2 = __builtin_amdgcn_rsqf(__builtin_fmaxf(n2, EPS2F) * den);
    float s = a.w * (d1 * j1 - d2 * j2);
    s = (c2 > EPS2F && !nearp) ? s : 0.0f;
    v[0] += cx * s;
    v[1] += cy * s;
    v[2] += cz * s;
    return nearp;
}

// FP64 pair of a group that every target of the wave is far from and within
// 2^24 core radii of (see write_group_records): |r1| >= 2 |r0| and qq > 0, so
// the clamps of pair64 and a zero denominator cannot occur, and
//   n2 = n1 + n0 - 2 d1        (terms at most 2.25 n1, n2 >= n1 / 4)
//   c2 = n0 n1 - d1^2          (Lagrange's identity)
//   sum of s c = (sum of s r0) x q - sum of s r0 x (a - c)
// with q = p - c, the target relative to the group's centre c: the pair
// accumulates S += w g r0 and T += w g r0 x (a - c) and the cross product is
// taken once per group.  35 vector instructions (two of them v_rsq_f64, four
// issue slots each) instead of pair64's 51.  The rounding of n1 and of the
// cancelling d1 j1 - d2 j2 is shared by n2, so the error against 64-bit
// references is no larger (quad-precision emulation, relative 2-norm over 60
// targets: 1.6e-15 against 6.3e-15 on a rotor wake, 2.2e-15 against 6.7e-15
// on helices).  pair64's zero for |r1 x r2| <= eps has no counterpart: near
// the axis the pair gives rounding (over a denominator of at least 32 eps
// n0 n1), and segments so short that |r0| |r1| is of the order of eps keep
// their value.
__device__ __forceinline__ void pair64_far(double px, double py, double pz, const d8 &u,
                                           const d8 &v, double &Sx, double &Sy, double &Sz,
                                           double &Tx, double &Ty, double &Tz)
{
    const double r1x = px - u[0], r1y = py - u[1], r1z = pz - u[2];
    const double n0 = u[7];
    const double n1 = r1x * r1x + r1y * r1y + r1z * r1z;
    const double d1 = u[4] * r1x + u[5] * r1y + u[6] * r1z;
    const double n2 = __builtin_fma(-2.0, d1, n1 + n0);
    const double c2 = __builtin_fma(-d1, d1, n0 * n1);
    const double d2 = d1 - n0;
    const double den = __builtin_fma(c2, c2, v[3]);
    const double j1 = rsq64(n1 * den);
    const double j2 = rsq64(n2 * den);
    const double w = d1 * j1 - d2 * j2;
    Sx += w * v[0];
    Sy += w * v[1];
    Sz += w * v[2];
    Tx += w * v[4];
    Ty += w * v[5];
    Tz += w * v[6];
}

// The same pair in FP32 on centred coordinates (q = p - c formed in FP64
// once per group): rounding q and a - c costs eps (|p - c| + |a - c|) <=
// eps (|r1| + 2 R) for a group of radius R, and groups wider than 64 of
// their longest segments are never far.  25 vector instructions, two of
// them v_rsq_f32.  For targets within 2^10 core radii.
__device__ __forceinline__ void pair32_far(const float *q, float4 a, float4 b, float4 c, float4 d,
                                           float *S, float *T)
{
    const float r1x = q[0] - a.x, r1y = q[1] - a.y, r1z = q[2] - a.z;
    const float n0 = a.w;
    const float n1 = r1x * r1x + r1y * r1y + r1z * r1z;
    const float d1 = b.x * r1x + b.y * r1y + b.z * r1z;
    const float n2 = __builtin_fmaf(-2.0f, d1, n1 + n0);
    const float c2 = __builtin_fmaf(-d1, d1, n0 * n1);
    const float d2 = d1 - n0;
    const float den = __builtin_fmaf(c2, c2, b.w);
    const float j1 = __builtin_amdgcn_rsqf(n1 * den);
    const float j2 = __builtin_amdgcn_rsqf(n2 * den);
    const float w = d1 * j1 - d2 * j2;
    S[0] += w * c.x;
    S[1] += w * c.y;
    S[2] += w * c.z;
    T[0] += w * d.x;
    T[1] += w * d.y;
    T[2] += w * d.z;
}

// The far pair at any distance: c2 from the cross product, the velocity
// summed directly (32 vector instructions).
__device__ __forceinline__ void pair32_cross(const float *q, float4 a, float4 b, float g, float *v)
{
    const float r1x = q[0] - a.x, r1y = q[1] - a.y, r1z = q[2] - a.z;
    const float n0 = a.w;
    const float cx = b.y * r1z - b.z * r1y;
    const float cy = b.z * r1x - b.x * r1z;
    const float cz = b.x * r1y - b.y * r1x;
    const float c2 = cx * cx + cy * cy + cz * cz;
    const float n1 = r1x * r1x + r1y * r1y + r1z * r1z;
    const float d1 = b.x * r1x + b.y * r1y + b.z * r1z;
    const float n2 = __builtin_fmaf(-2.0f, d1, n1 + n0);
    const float d2 = d1 - n0;
    const float den = __builtin_fmaf(c2, c2, b.w);
    const float j1 = __builtin_amdgcn_rsqf(n1 * den);
    const float j2 = __builtin_amdgcn_rsqf(n2 * den);
    const float w = g * (d1 * j1 - d2 * j2);
    v[0] += cx * w;
    v[1] += cy * w;
    v[2] += cz * w;
}

// One group for NK targets per lane, all far: records from the wave's LDS
// copy (broadcast reads), sums folded into FP64 once per group.
template <int NK>
__device__ __forceinline__ void group32_far(const float4 *buf, const float (&q)[NK][3],
                                            double (&v)[NK][3])
{
    float S[NK][3] = {}, T[NK][3] = {};
#pragma unroll 2
    for (int j = 0; j < GRP; ++j) {
        const float4 a = buf[4 * j], b = buf[4 * j + 1], c = buf[4 * j + 2], d = buf[4 * j + 3];
#pragma unroll
        for (int k = 0; k < NK; ++k) pair32_far(q[k], a, b, c, d, S[k], T[k]);
    }
#pragma unroll
    for (int k = 0; k < NK; ++k) {
        v[k][0] += (double)((S[k][1] * q[k][2] - S[k][2] * q[k][1]) - T[k][0]);
        v[k][1] += (double)((S[k][2] * q[k][0] - S[k][0] * q[k][2]) - T[k][1]);
        v[k][2] += (double)((S[k][0] * q[k][1] - S[k][1] * q[k][0]) - T[k][2]);
    }
}

// The same where a target may be past the distance that pair32_far is
// accurate to.
template <int NK>
__device__ __forceinline__ void group32_cross(const float4 *buf, const float (&q)[NK][3],
                                              double (&v)[NK][3])
{
    float s[NK][3] = {};
#pragma unroll 2
    for (int j = 0; j < GRP; ++j) {
        const float4 a = buf[4 * j], b = buf[4 * j + 1];
        const float g = buf[4 * j + 2].w;
#pragma unroll
        for (int k = 0; k < NK; ++k) pair32_cross(q[k], a, b, g, s[k]);
    }
#pragma unroll
    for (int k = 0; k < NK; ++k)
#pragma unroll
        for (int d = 0; d < 3; ++d) v[k][d] += (double)s[k][d];
}

// One group that is not far: the split coordinates from the wave's second LDS
// copy, then the flagged pairs in FP64 from the records rec64 in memory.
template <int NK>
__device__ __forceinline__ void group32_near(const float4 *buf, const float4 *nbuf,
                                             const double *rec64, const double (&p)[NK][3],
                                             double (&v)[NK][3])
{
    float ph[NK][3], pl[NK][3], s[NK][3] = {};
    unsigned mask[NK] = {};
#pragma unroll
    for (int k = 0; k < NK; ++k)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            ph[k][d] = (float)p[k][d];
            pl[k][d] = (float)(p[k][d] - (double)ph[k][d]);
        }
#pragma unroll 4
    for (int j = 0; j < GRP; ++j) {
        const float4 a = nbuf[2 * j], b = nbuf[2 * j + 1], r = buf[4 * j + 1];
        const float n0 = buf[4 * j].w;
#pragma unroll
        for (int k = 0; k < NK; ++k)
            mask[k] |= (pair32(ph[k], pl[k], a, b, r, n0, s[k]) ? 1u : 0u) << j;
    }
#pragma unroll
    for (int k = 0; k < NK; ++k) {
#pragma unroll
        for (int d = 0; d < 3; ++d) v[k][d] += (double)s[k][d];
        while (mask[k]) {
            const int j = __builtin_ctz(mask[k]);
            mask[k] &= mask[k] - 1u;
            const double *r = rec64 + j * REC64_N;
            pair64(p[k][0], p[k][1], p[k][2], r[0], r[1], r[2], r[3], r[4], r[5], r[6], r[11],
                   r[7], v[k][0], v[k][1], v[k][2]);
        }
    }
}

struct BsArgs {
    const double *rec64, *grp;
    const float *rec32, *near32;
    const long long *nseg;
    const double *t;
    double *part;
    int *counter;
    int64_t m, tstride;
    int nchunks, ntiles, nitems, nwaves, round_robin;
};

// Work items of both kernels: a wave takes 64 NT targets (NT per lane) and
// one chunk of groups; no LDS and no barrier, the records are wave-uniform
// and reach the vector instructions as scalar operands.
struct Item {
    int chunk, tile;
    int64_t g0, g1;
};

__device__ __forceinline__ Item item_of(const BsArgs &a, int item, int64_t ngroups)
{
    Item r;
    r.chunk = item / a.ntiles;
    r.tile = item - r.chunk * a.ntiles;
    const int64_t len = (ngroups + a.nchunks - 1) / a.nchunks;
    r.g0 = (int64_t)r.chunk * len;
    r.g1 = min(ngroups, r.g0 + len);
    return r;
}

// A wave's first item is its own index; later ones come from the counter,
// or, in launches of short items (chunks of fewer than LEN_MID groups),
// round robin: atomics on the one counter complete every 11 ns or so, which
// bounded those launches (3.4e7 pairs: 258 us with the counter, 107 without).
// Long launches need the counter: dealing out only their first quarter round
// robin cost 3-6%, three quarters 15%.
__device__ __forceinline__ int first_item()
{
    return __builtin_amdgcn_readfirstlane((int)blockIdx.x * (BS_BLOCK / 64) +
                                          ((int)threadIdx.x >> 6));
}
__device__ __forceinline__ int next_item(const BsArgs &a, int item)
{
    if (a.round_robin) return item + a.nwaves;
    int next = 0;
    if ((threadIdx.x & 63) == 0) next = atomicAdd(a.counter, 1);
    return a.nwaves + __builtin_amdgcn_readfirstlane(next);
}

__global__ __launch_bounds__(BS_BLOCK, 8) void bs_fp64_kernel(BsArgs a)
{
    const int lane = threadIdx.x & 63;
    const int64_t ngroups = (*(clptr)a.nseg + GRP - 1) / GRP;
    for (int item = first_item(); item < a.nitems; item = next_item(a, item)) {
        const Item it = item_of(a, item, ngroups);
        const int64_t t = (int64_t)it.tile * 64 + lane;
        const int64_t tc = t < a.m ? t : a.m - 1;   // idle lanes repeat the last target
        const double px = a.t[tc], py = a.t[a.tstride + tc], pz = a.t[2 * a.tstride + tc];
        double vx = 0.0, vy = 0.0, vz = 0.0;
        for (int64_t g = it.g0; g < it.g1; ++g) {
            const d8 h = *(cd8ptr)(a.grp + g * GRPH_N);
            const double qx = px - h[0], qy = py - h[1], qz = pz - h[2];
            const double d2 = qx * qx + qy * qy + qz * qz;
            if (__ballot(!((d2 > h[3]) & (d2 <= h[4]))) == 0) {
                cd8ptr r = (cd8ptr)(a.rec64 + g * (GRP * REC64_N));
                double Sx = 0, Sy = 0, Sz = 0, Tx = 0, Ty = 0, Tz = 0;
#pragma unroll 2
                for (int j = 0; j < GRP; ++j, r += 2) {
                    const d8 u = r[0], w = r[1];
                    pair64_far(px, py, pz, u, w, Sx, Sy, Sz, Tx, Ty, Tz);
                }
                vx += (Sy * qz - Sz * qy) - Tx;
                vy += (Sz * qx - Sx * qz) - Ty;
                vz += (Sx * qy - Sy * qx) - Tz;
            } else {
                cdptr r = (cdptr)a.rec64 + g * (GRP * REC64_N);
                for (int j = 0; j < GRP; ++j, r += REC64_N)
                    pair64(px, py, pz, r[0], r[1], r[2], r[3], r[4], r[5], r[6], r[11], r[7], vx,
                           vy, vz);
            }
        }
        if (t < a.m) {
            double *o = a.part + (size_t)it.chunk * 3 * a.m;
            o[t] = vx;
            o[a.m + t] = vy;
            o[2 * a.m + t] = vz;
        }
    }
}

// FP32 instructions run at half rate with a scalar operand (4.2 against 2.4
// cycles per wave instruction, measured), so here the wave copies each
// group's records to its own 2 KB of LDS (the next group's are loaded while
// this one is evaluated) and reads them back as broadcasts, each shared by
// the NT targets of a lane.  Groups that are not far for all 64 NT targets
// are tested again per 64; for the near ones the split coordinates follow
// into another 1 KB, and the lanes recompute their flagged pairs in FP64
// after the group.  With pair32 on scalar operands, one 64 at a time, a list
// in no spatial order (every group near, 4.8e9 pairs) took 5.26 ms; so 4.44.
template <int NT>
__global__ __launch_bounds__(BS_BLOCK, 5) void bs_mixed_kernel(BsArgs a)
{
    __shared__ float4 lds[BS_BLOCK / 64][GRP * 4], nlds[BS_BLOCK / 64][GRP * 2];
    const int lane = threadIdx.x & 63;
    float4 *buf = lds[threadIdx.x >> 6], *nbuf = nlds[threadIdx.x >> 6];
    const int64_t ngroups = (*(clptr)a.nseg + GRP - 1) / GRP;
    for (int item = first_item(); item < a.nitems; item = next_item(a, item)) {
        const Item it = item_of(a, item, ngroups);
        double p[NT][3], v[NT][3];
#pragma unroll
        for (int k = 0; k < NT; ++k) {
            const int64_t t = ((int64_t)it.tile * NT + k) * 64 + lane;
            const int64_t tc = t < a.m ? t : a.m - 1;   // idle lanes repeat the last target
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                p[k][d] = a.t[d * a.tstride + tc];
                v[k][d] = 0.0;
            }
        }
        const float4 *src = reinterpret_cast<const float4 *>(a.rec32) + lane;
        float4 n0, n1;
        if (it.g0 < it.g1) {
            n0 = src[it.g0 * (GRP * 4)];
            n1 = src[it.g0 * (GRP * 4) + 64];
        }
        for (int64_t g = it.g0; g < it.g1; ++g) {
            __builtin_amdgcn_wave_barrier();
            buf[lane] = n0;
            buf[lane + 64] = n1;
            __builtin_amdgcn_wave_barrier();
            const int64_t gn = min(g + 1, it.g1 - 1);
            n0 = src[gn * (GRP * 4)];
            n1 = src[gn * (GRP * 4) + 64];
            const cdptr h = (cdptr)a.grp + g * GRPH_N;
            float q[NT][3];
            unsigned odd = 0;   // bit k: the k-th 64 targets cannot all take the short pair
#pragma unroll
            for (int k = 0; k < NT; ++k) {
                double d2 = 0.0;
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    const double x = p[k][d] - h[d];
                    d2 += x * x;
                    q[k][d] = (float)x;
                }
                if (__ballot(!((d2 > h[3]) & (d2 <= h[5]))) != 0) odd |= 1u << k;
            }
            if (odd == 0) {
                group32_far<NT>(buf, q, v);
                continue;
            }
            unsigned near = 0;   // bit k: one of them is not far
#pragma unroll
            for (int k = 0; k < NT; ++k) {
                double d2 = 0.0;
#pragma unroll
                for (int d = 0; d < 3; ++d) d2 += (p[k][d] - h[d]) * (p[k][d] - h[d]);
                if (__ballot(!(d2 > h[3])) != 0) near |= 1u << k;
            }
            if (near == 0) {
                group32_cross<NT>(buf, q, v);
                continue;
            }
            nbuf[lane] = reinterpret_cast<const float4 *>(a.near32)[g * (GRP * 2) + lane];
            __builtin_amdgcn_wave_barrier();
            const double *r64 = a.rec64 + g * (GRP * REC64_N);
            if (near == (1u << NT) - 1u) {
                group32_near<NT>(buf, nbuf, r64, p, v);
                continue;
            }
#pragma unroll
            for (int k = 0; k < NT; ++k) {
                const float qk[1][3] = {{q[k][0], q[k][1], q[k][2]}};
                const double pk[1][3] = {{p[k][0], p[k][1], p[k][2]}};
                double vk[1][3] = {{v[k][0], v[k][1], v[k][2]}};
                if (near >> k & 1u) group32_near<1>(buf, nbuf, r64, pk, vk);
                else if (odd >> k & 1u) group32_cross<1>(buf, qk, vk);
                else group32_far<1>(buf, qk, vk);
                for (int d = 0; d < 3; ++d) v[k][d] = vk[0][d];
            }
        }
        double *o = a.part + (size_t)it.chunk * 3 * a.m;
#pragma unroll
        for (int k = 0; k < NT; ++k) {
            const int64_t t = ((int64_t)it.tile * NT + k) * 64 + lane;
            if (t < a.m) {
                o[t] = v[k][0];
                o[a.m + t] = v[k][1];
                o[2 * a.m + t] = v[k][2];
            }
        }
    }
}

// Few targets or short lists (few_pairs): each block
// takes SM_T targets and one segment chunk; its 256 lanes stride over the
// chunk (coalesced SoA loads, each record shared by the SM_T targets) and
// the partial sums are reduced in a fixed order (butterfly within the wave,
// waves in order).  Always FP64: these launches are a small fraction of the
// pairs.
constexpr int SM_T = 4;
constexpr int SM_BLOCK = 256;
constexpr int LEN_MID = 8;
constexpr int MIXED_NT = 2;       // targets per lane of the mixed kernel
constexpr int MIXED_MIN = 1024;   // fewer targets than this: FP64 in both modes

__device__ __forceinline__ double wave_sum(double v)
{
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// Chunks of the lists of one launch: list k has chunks chunk0[k] to
// chunk0[k + 1] - 1.
struct TermTab {
    int n, neg;   // neg: bit k set where the sum is negated before list k
    int chunk0[TERM_MAX + 1];
    int64_t off[TERM_MAX];
};

// The only list of a launch, from segment 0.
struct OneList {
    int nchunks;
};

// The list that a block works on, its first chunk, its chunks and its start.
struct ListChunks {
    int k, first, n;
    int64_t off;
};

__device__ __forceinline__ ListChunks chunks_of(const OneList &l, int)
{
    return {0, 0, l.nchunks, 0};
}

__device__ __forceinline__ ListChunks chunks_of(const TermTab &tt, int blk)
{
    int k = 0;
    while (k + 1 < tt.n && blk >= tt.chunk0[k + 1]) ++k;
    return {k, tt.chunk0[k], tt.chunk0[k + 1] - tt.chunk0[k], tt.off[k]};
}

// Lists: OneList or TermTab.  One list has a kernel of its own for its short
// argument block, which the host writes across the bus at each launch: with
// the table, and with the grid's size taken from the implicit arguments (256
// bytes more), 50 segments at 1000 points took 8.4 us a call, so 6.1.
template <typename Lists>
__global__ __launch_bounds__(SM_BLOCK) void bs_small_kernel(const double *s64, int64_t S,
                                                            const long long *counts, Lists lists,
                                                            const double *t, int64_t m,
                                                            int64_t tstride, double *part)
{
    __shared__ double red[3 * SM_T][SM_BLOCK / 64];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const ListChunks c = chunks_of(lists, (int)blockIdx.x);
    const int64_t nseg = counts[c.k];
    const int64_t len = (nseg + c.n - 1) / c.n;
    const int64_t s0 = (int64_t)((int)blockIdx.x - c.first) * len;
    const int64_t s1 = min(nseg, s0 + len);
    const int64_t g0 = (int64_t)blockIdx.y * SM_T;
    s64 += c.off;
    double px[SM_T], py[SM_T], pz[SM_T], vx[SM_T], vy[SM_T], vz[SM_T];
#pragma unroll
    for (int q = 0; q < SM_T; ++q) {
        const int64_t tq = g0 + q < m ? g0 + q : m - 1;
        px[q] = t[tq];
        py[q] = t[tstride + tq];
        pz[q] = t[2 * tstride + tq];
        vx[q] = vy[q] = vz[q] = 0.0;
    }
    for (int64_t sg = s0 + tid; sg < s1; sg += SM_BLOCK) {
        double r[SOA_N];
#pragma unroll
        for (int i = 0; i < SOA_N; ++i) r[i] = s64[i * S + sg];
#pragma unroll
        for (int q = 0; q < SM_T; ++q)
            pair64(px[q], py[q], pz[q], r[0], r[1], r[2], r[3], r[4], r[5], r[6], r[7], r[8],
                   vx[q], vy[q], vz[q]);
    }
#pragma unroll
    for (int q = 0; q < SM_T; ++q) {
        const double a = wave_sum(vx[q]), b = wave_sum(vy[q]), c = wave_sum(vz[q]);
        if (lane == 0) {
            red[3 * q][w] = a;
            red[3 * q + 1][w] = b;
            red[3 * q + 2][w] = c;
        }
    }
    __syncthreads();
    if (tid < 3 * SM_T) {
        const int q = tid / 3, d = tid % 3;
        if (g0 + q < m) {
            double v = 0.0;
            for (int k = 0; k < SM_BLOCK / 64; ++k) v += red[tid][k];
            part[((size_t)blockIdx.x * 3 + d) * m + g0 + q] = v;
        }
    }
}

// Component d of target t lies at out[d ds + t ts]: SoA (stride, 1) or the
// host's order (1, 3).
struct OutMap {
    int64_t ds, ts;
};

// Sum of the lists' chunk partials at one component of 64 targets, then the
// term recurrence (TermLists): RT_S slices of a list's chunks side by side,
// each in increasing order, the slices and then the lists added in order, so
// that a list contributes the same bits however many share the launch.
constexpr int RT_S = 8, RT_W = 16;

__global__ __launch_bounds__(64 * RT_W) void bs_reduce_terms_kernel(const double *part,
                                                                    TermTab tt, int64_t m,
                                                                    double *out, OutMap o, int acc)
{
    __shared__ double sh[TERM_MAX * RT_S][64];
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t t = (int64_t)blockIdx.x * 64 + l;
    const int d = blockIdx.y;
    const size_t cs = 3 * (size_t)m;
    for (int u = w; u < tt.n * RT_S; u += RT_W) {
        const int k = u / RT_S, q = u % RT_S;
        const int nc = tt.chunk0[k + 1] - tt.chunk0[k], len = (nc + RT_S - 1) / RT_S;
        const int c1 = min(nc, (q + 1) * len);
        double s = 0.0;
        if (t < m) {
            const double *p = part + (size_t)tt.chunk0[k] * cs + (size_t)d * m + t;
            int c = q * len;
            for (; c + 8 <= c1; c += 8) {
                double v[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = p[(size_t)(c + i) * cs];
#pragma unroll
                for (int i = 0; i < 8; ++i) s += v[i];
            }
            for (; c < c1; ++c) s += p[(size_t)c * cs];
        }
        sh[u][l] = s;
    }
    __syncthreads();
    if (w > 0 || t >= m) return;
    out += d * o.ds + t * o.ts;
    double v = acc ? *out : 0.0;
    for (int k = 0; k < tt.n; ++k) {
        double s = sh[k * RT_S][l];
        for (int q = 1; q < RT_S; ++q) s += sh[k * RT_S + q][l];
        v = (tt.neg >> k & 1 ? -v : v) + s;
    }
    *out = v;
}

// Fixed-order sum of the per-chunk partials: T targets of one component per
// workgroup, S slices of the chunk range side by side (each in increasing
// order, loads eight chunks ahead of the adds), the slices added in order.
// Bound by the dependent round trips to memory of one slice: a lane that
// walked all chunks alone waited once per eight loads, so many chunks take
// many slices.  Workgroup 0 clears the work counter for the next launch.
template <int T, int S>
__global__ __launch_bounds__(T * S) void bs_reduce_kernel(const double *part, int nchunks,
                                                          int64_t m, double *out, OutMap o,
                                                          int acc, int *counter)
{
    __shared__ double sh[S][T];
    const int l = threadIdx.x % T, w = threadIdx.x / T;
    const int64_t t = (int64_t)blockIdx.x * T + l;
    const int d = blockIdx.y;
    if (counter && blockIdx.x == 0 && d == 0 && threadIdx.x == 0) *counter = 0;
    const int len = (nchunks + S - 1) / S;
    const int c1 = min(nchunks, (w + 1) * len);
    double s = 0.0;
    if (t < m) {
        const double *p = part + (size_t)d * m + t;
        const size_t cs = 3 * (size_t)m;
        int c = w * len;
        for (; c + 8 <= c1; c += 8) {
            double v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = p[(size_t)(c + k) * cs];
#pragma unroll
            for (int k = 0; k < 8; ++k) s += v[k];
        }
        for (; c < c1; ++c) s += p[(size_t)c * cs];
    }
    if constexpr (S > 1) {
        sh[w][l] = s;
        __syncthreads();
        if (w > 0) return;
        for (int k = 1; k < S; ++k) s += sh[k][l];
    }
    if (t < m) {
        double *q = out + d * o.ds + t * o.ts;
        *q = acc ? *q + s : s;
    }
}

template <int T, int S>
void reduce_as(vlm_ctx *ctx, const double *part, int nchunks, int64_t m, double *out, OutMap o,
               int acc, int *counter)
{
    hipLaunchKernelGGL((bs_reduce_kernel<T, S>), dim3((unsigned)((m + T - 1) / T), 3), dim3(T * S),
                       0, ctx->stream, part, nchunks, m, out, o, acc, counter);
}

int launch_reduce(vlm_ctx *ctx, const double *part, int nchunks, int64_t m, double *out,
                  OutMap o, int acc, int *counter)
{
    if (nchunks >= 256) reduce_as<16, 64>(ctx, part, nchunks, m, out, o, acc, counter);
    else if (nchunks >= 32) reduce_as<64, 8>(ctx, part, nchunks, m, out, o, acc, counter);
    else if (nchunks >= 8) reduce_as<64, 4>(ctx, part, nchunks, m, out, o, acc, counter);
    else reduce_as<64, 1>(ctx, part, nchunks, m, out, o, acc, counter);
    VLM_HIP(hipGetLastError());
    return VLM_OK;
}

__global__ void zero_int_kernel(int *p) { *p = 0; }

template <typename K>
int resident_blocks(vlm_ctx *ctx, K kernel, int block, int *cache)
{
    if (*cache > 0) return *cache;
    int per_cu = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, block, 0) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device) !=
            hipSuccess)
        return -1;
    *cache = (per_cu > 0 ? per_cu : 1) * (cus > 0 ? cus : 1);
    return *cache;
}

// Records one profiled launch: the pair count is m times the device
// segment count, copied to the pinned slot of this record without a stream
// synchronisation and resolved at read-out (vlm_profile_get).
int profile_count(vlm_ctx *ctx, const long long *nseg_dev, int64_t m, int kind, const Timer *tm)
{
    Timer r{};
    if (tm) r = *tm;
    r.kind = kind;
    r.pairs = -1.0;
    const size_t slot = ctx->timers.size();
    if (slot < ctx->prof_cap) {
        VLM_HIP(hipMemcpyAsync(ctx->prof_nseg + slot, nseg_dev, sizeof(long long),
                               hipMemcpyDeviceToHost, ctx->stream));
        r.pairs = (double)m;
    }
    ctx->timers.push_back(r);
    if (kind == 0) ctx->prof_launches += 1;
    return VLM_OK;
}

}  // namespace

// bs_small_kernel has segments on its lanes, so no lane idles however few the
// targets and short lists spread over the device, but every pair is the long
// one.  Sums over resident sets, us, small against 64 targets per wave, on
// helices and on a rotor wake with a grid of points through it:
//                 helices      wake                    helices      wake
//   m   200 x 80000   48  54   48  54    200 x 200000   112 116  115 118
//   m   200 x 400000 220 219  223 213    300 x 133333   100  93  100  94
//   m   500 x 32000   42  47   45  45    500 x  80000    94  81  102  85
//   m  1000 x  9000   26  30   28  28   1000 x  24000    56  66   59  65
//   m  1000 x 40000   86  80   95  86   2048 x  11719    54  66   55  61
//   m  2048 x 19531   84  88   88  81   2048 x  39063   158 143  170 149
// Whole calls on host arrays, 20 x 2e5: 54 against 92, 90 x 2e5: 92, 108.
// From 2048 targets on every launch is a grouped (and so a timed) one.
static bool few_pairs(int64_t m, int64_t nseg)
{
    if (m < 192 && 5 * m < 4 * 64 * ((m + 63) / 64)) return true;   // waves not 4/5 full
    return m < 2048 && nseg <= 60000000 && m * nseg <= (m <= 256 ? 60000000 : 30000000);
}

int bs_formats(const vlm_ctx *ctx, int64_t m, int64_t nseg)
{
    if (ctx->precision == VLM_MIXED && m >= MIXED_MIN) return SEG_REC | SEG_F32;
    return few_pairs(m, nseg) ? SEG_SOA : SEG_REC;
}

int bs_eval_terms(vlm_ctx *ctx, const SegPtrs &seg, const TermLists &terms, const double *t,
                  int64_t m, int64_t tstride, double *out, int accumulate, const BsWork *ws,
                  bool aos)
{
    if (m <= 0) return VLM_OK;
    if (terms.n < 1 || terms.n > TERM_MAX) return fail(ctx, VLM_ERR_ARG, "bad term count");
    const int64_t max_chunks = ws ? (int64_t)(ws->part_cap / (3 * (size_t)m)) : INT32_MAX;
    if (max_chunks < terms.n) return fail(ctx, VLM_ERR_ARG, "workspace too small for the targets");
    // per list about 2048 blocks of at least 8 segments per lane; short
    // lists are split down to 2 per lane (their loads wait on each other), up
    // to 16 chunks (more only feed the reduction) and 512 blocks (2 per CU:
    // 600 targets x 6666 segments 17 us with 450 blocks, 21 with 1950)
    const int64_t groups = (m + SM_T - 1) / SM_T;
    TermTab tt;
    tt.n = terms.n;
    tt.neg = 0;
    tt.chunk0[0] = 0;
    for (int k = 0; k < terms.n; ++k) {
        int64_t nc = (2048 + groups - 1) / groups;
        const int64_t c2 = terms.est[k] / (2 * SM_BLOCK), c8 = terms.est[k] / (8 * SM_BLOCK);
        const int64_t maxc = std::max(c8, std::min<int64_t>({16, c2, 512 / groups}));
        if (nc > maxc) nc = maxc;
        if (nc > max_chunks / terms.n) nc = max_chunks / terms.n;
        if (nc < 1) nc = 1;
        tt.chunk0[k + 1] = tt.chunk0[k] + (int)nc;
        tt.off[k] = terms.off[k];
        if (terms.neg[k]) tt.neg |= 1 << k;
    }
    const int nchunks = tt.chunk0[tt.n];
    double *part = ws ? ws->part : nullptr;
    if (!ws) {
        VLM_HIP(ctx->part.reserve(ws_size<double>((size_t)nchunks * 3 * (size_t)m)));
        part = ctx->part.p;
    }
    const dim3 grid(nchunks, (unsigned)groups);
    const OutMap o = aos ? OutMap{1, 3} : OutMap{tstride, 1};
    if (tt.n == 1 && tt.off[0] == 0 && !tt.neg) {
        hipLaunchKernelGGL(bs_small_kernel<OneList>, grid, dim3(SM_BLOCK), 0, ctx->stream, seg.soa,
                           seg.cap, seg.count, OneList{nchunks}, t, m, tstride, part);
        // the sums of bs_reduce_terms_kernel
        if (nchunks > RT_S)
            reduce_as<64, RT_S>(ctx, part, nchunks, m, out, o, accumulate, nullptr);
        else
            reduce_as<64, 1>(ctx, part, nchunks, m, out, o, accumulate, nullptr);
    } else {
        hipLaunchKernelGGL(bs_small_kernel<TermTab>, grid, dim3(SM_BLOCK), 0, ctx->stream,
                           seg.soa, seg.cap, seg.count, tt, t, m, tstride, part);
        hipLaunchKernelGGL(bs_reduce_terms_kernel, dim3((unsigned)((m + 63) / 64), 3),
                           dim3(64 * RT_W), 0, ctx->stream, part, tt, m, out, o, accumulate);
    }
    VLM_HIP(hipGetLastError());
    if (ctx->profile && !ws)
        for (int k = 0; k < terms.n; ++k)
            VLM_TRY(profile_count(ctx, seg.count + k, m, 1, nullptr));
    return VLM_OK;
}

int bs_eval(vlm_ctx *ctx, const SegPtrs &seg, int64_t nseg_est, const double *t, int64_t m,
            int64_t tstride, double *out, int accumulate, const BsWork *ws, bool aos)
{
    if (m <= 0) return VLM_OK;
    const OutMap o = aos ? OutMap{1, 3} : OutMap{tstride, 1};
    // chunk partial sums: the context's growing buffer, or a fixed
    // workspace that caps the chunk count
    const int64_t max_chunks = ws ? (int64_t)(ws->part_cap / (3 * (size_t)m)) : INT32_MAX;
    if (ws && max_chunks < 1) return fail(ctx, VLM_ERR_ARG, "workspace too small for the targets");
    const bool prof = ctx->profile && !ws;
    if (nseg_est <= 0) return launch_reduce(ctx, nullptr, 0, m, out, o, accumulate, nullptr);
    const int fmt = bs_formats(ctx, m, nseg_est);
    if (((fmt & SEG_SOA) && !seg.soa) || ((fmt & SEG_REC) && !seg.rec64) ||
        ((fmt & SEG_F32) && !seg.rec32))
        return fail(ctx, VLM_ERR_STATE, "segment list lacks the records of this launch");
    if (fmt == SEG_SOA) {
        TermLists one;
        one.n = 1;
        one.off[0] = 0;
        one.est[0] = nseg_est;
        one.neg[0] = 0;
        return bs_eval_terms(ctx, seg, one, t, m, tstride, out, accumulate, ws, aos);
    }
    const bool mixed = (fmt & SEG_F32) != 0;
    const int tile = mixed ? 64 * MIXED_NT : 64;
    const int ntiles = (int)((m + tile - 1) / tile);
    const int cap = mixed ? resident_blocks(ctx, bs_mixed_kernel<MIXED_NT>, BS_BLOCK, &ctx->occ[1])
                          : resident_blocks(ctx, bs_fp64_kernel, BS_BLOCK, &ctx->occ[0]);
    if (cap <= 0) return fail(ctx, VLM_ERR_HIP, "occupancy query failed");
    const int64_t W = (int64_t)cap * (BS_BLOCK / 64);   // resident waves
    const int64_t ngroups = (nseg_est + GRP - 1) / GRP;
    const int64_t P = ngroups * ntiles;
    // groups per chunk: two items per wave while that makes chunks shorter
    // than LEN_MID groups (launches that barely fill the device: an item
    // costs its latency, not its work), then LEN_MID until there are 16
    // items per wave (the queue needs them to even out the end: 4 per wave
    // cost 5% on 4.0e9 pairs, 32 gained nothing), then longer chunks (fewer
    // partial sums)
    int64_t len = P / (2 * W);
    if (len > LEN_MID) len = LEN_MID;
    if (P / (16 * W) > len) len = P / (16 * W);
    if (len < 1) len = 1;
    if ((ngroups + len - 1) / len > max_chunks) len = (ngroups + max_chunks - 1) / max_chunks;
    const int nchunks = (int)((ngroups + len - 1) / len);
    double *part = ws ? ws->part : nullptr;
    int *counter = ws ? ws->counter : nullptr;
    if (!ws) {
        VLM_HIP(ctx->part.reserve(ws_size<double>((size_t)nchunks * 3 * (size_t)m)));
        if (!ctx->counter.p) {
            VLM_HIP(ctx->counter.reserve(1));
            hipLaunchKernelGGL(zero_int_kernel, dim3(1), dim3(1), 0, ctx->stream, ctx->counter.p);
        }
        part = ctx->part.p;
        counter = ctx->counter.p;
    }
    BsArgs a;
    a.rec64 = seg.rec64;
    a.grp = seg.grp;
    a.rec32 = seg.rec32;
    a.near32 = seg.near32;
    a.nseg = seg.count;
    a.t = t;
    a.part = part;
    a.counter = counter;
    a.m = m;
    a.tstride = tstride;
    a.nchunks = nchunks;
    a.ntiles = ntiles;
    const int64_t nitems = (int64_t)ntiles * nchunks;
    if (nitems > INT32_MAX - W) return fail(ctx, VLM_ERR_ARG, "too many work items");
    a.nitems = (int)nitems;
    const int64_t need = (nitems + BS_BLOCK / 64 - 1) / (BS_BLOCK / 64);
    const int grid = (int)(need < cap ? need : cap);
    a.nwaves = grid * (BS_BLOCK / 64);
    a.round_robin = len < LEN_MID || need <= cap;
    Timer tm{};
    if (prof) {
        VLM_HIP(hipEventCreate(&tm.a));
        VLM_HIP(hipEventCreate(&tm.b));
        VLM_HIP(hipEventRecord(tm.a, ctx->stream));
    }
    if (mixed)
        hipLaunchKernelGGL(bs_mixed_kernel<MIXED_NT>, dim3(grid), dim3(BS_BLOCK), 0, ctx->stream, a);
    else
        hipLaunchKernelGGL(bs_fp64_kernel, dim3(grid), dim3(BS_BLOCK), 0, ctx->stream, a);
    VLM_HIP(hipGetLastError());
    const hipError_t e = prof ? hipEventRecord(tm.b, ctx->stream) : hipSuccess;
    // before any return: the reduction leaves the work counter at 0
    VLM_TRY(launch_reduce(ctx, part, nchunks, m, out, o, accumulate, counter));
    VLM_HIP(e);
    return prof ? profile_count(ctx, seg.count, m, 0, &tm) : VLM_OK;
}

}  // namespace vlm
