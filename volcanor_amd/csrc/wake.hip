// Device-resident free wake: rotor objects, segment builders, the N-body
// wake pass and the fused wake-update passes (convection, continuity, age,
// dissipation, strain, shed, rollup, shift, scheme algebra).
//
// HBM layout per rotor (see vlm_c.h for the exported lattice layout):
//   * Near wake as a node lattice: node(b, p, j) with p the PHYSICAL row of
//     a ring buffer; logical row i lives in p = (head + i) mod nNwake.  The
//     reference shifts every near-wake ring down one row per step
//     (rotor_shiftwake, classdef.f90:4481-4498); here the shift is a head
//     move plus one row copy.  Shared ring corners exist once, so the
//     corner copies of blade_wake_continuity (classdef.f90:1609-1702) are
//     implicit.
//   * Velocity arrays keep LOGICAL rows, exactly like velNwake/velNwake1 in
//     the reference, which are not shifted with the wake.
//   * Far wake: per-filament end points (fc1 = trailing end, fc2 = leading).
//
// Sources are built per pass as unique segments: the two ring filaments
// that share a lattice edge are merged into one segment with net
// circulation when their core radii are equal (the common case), otherwise
// both are kept.  Rings with |gam| <= eps are skipped as in
// blade_vind_bywake (classdef.f90:1450-1456).
#include <algorithm>
#include <cmath>
#include <cstring>

#include "vlm_internal.h"

namespace vlm {

int points_to_device(vlm_ctx *ctx, int64_t m, const double *p, double *soa, int64_t stride);
int points_to_host(vlm_ctx *ctx, int64_t m, const double *soa, int64_t stride, double *p,
                   bool deferred = false);

namespace {

unsigned nblk(int64_t n) { return (unsigned)((n + 255) / 256); }

constexpr double EPS = kEps;

struct RV {  // raw views of a rotor's device state
    int nb, nc, ns, nN, nF, nbc, head, rn, rf;  // rn, rf 0-based
    double *node, *pnode, *le, *ple, *gam, *rc4, *age;
    double *ffc, *pffc, *fgam, *frc, *frc0, *fl0, *flc, *fage;
    double *wc, *wrc, *wg;
    double *vel[4], *velF[4];
};

RV view(Rotor &r)
{
    RV v;
    v.nb = r.d.nb;
    v.nc = r.d.nc;
    v.ns = r.d.ns;
    v.nN = r.d.nNwake;
    v.nF = r.d.nFwake;
    v.nbc = r.d.nbConvect;
    v.head = r.head;
    v.rn = r.rowNear - 1;
    v.rf = r.rowFar - 1;
    v.node = r.node.p;
    v.pnode = r.pnode.p;
    v.le = r.le.p;
    v.ple = r.ple.p;
    v.gam = r.gam.p;
    v.rc4 = r.rc4.p;
    v.age = r.age.p;
    v.ffc = r.ffc.p;
    v.pffc = r.pffc.p;
    v.fgam = r.fgam.p;
    v.frc = r.frc.p;
    v.frc0 = r.frc0.p;
    v.fl0 = r.fl0.p;
    v.flc = r.flc.p;
    v.fage = r.fage.p;
    v.wc = r.wc.p;
    v.wrc = r.wrc.p;
    v.wg = r.wg.p;
    for (int k = 0; k < 4; ++k) {
        v.vel[k] = r.velN[k].p;
        v.velF[k] = r.velF[k].p;
    }
    return v;
}

__device__ __forceinline__ int phys(const RV &v, int i)
{
    int p = v.head + i;
    return p >= v.nN ? p - v.nN : p;
}
__device__ __forceinline__ size_t nidx(const RV &v, int b, int p, int j)
{
    return ((size_t)b * v.nN + p) * (v.ns + 1) + j;
}
__device__ __forceinline__ size_t ridx(const RV &v, int b, int p, int j)
{
    return ((size_t)b * v.nN + p) * v.ns + j;
}
__device__ __forceinline__ size_t vidx(const RV &v, int b, int i, int j)
{
    return ((size_t)b * v.nN + i) * (v.ns + 1) + j;
}

// Entry k of a lattice of rows x cols walked in patches of PATCH rows: each
// patch column by column, every second patch backwards, so that any run of
// entries is compact in space whatever the number of columns.  Sources and
// targets take this order because the Biot-Savart kernel runs its shorter
// pair on a (wave of 64 targets, group of 32 segments) whose distance
// exceeds the group's radius: with whole spanwise rows (patch of one row)
// 54% of them are far on a 3 x 30 rotor after 360 steps of 5 degrees, with
// 4 rows 96% (8 rows 94%, 2 rows 93%).
constexpr int PATCH = 4;

__device__ __forceinline__ void patch_entry(int64_t k, int rows, int cols, int *i, int *j)
{
    const int b = (int)(k / (PATCH * cols));
    const int w = (int)(k - (int64_t)b * (PATCH * cols));
    const int h = min(PATCH, rows - PATCH * b);
    const int c = w / h;
    *i = PATCH * b + (w - c * h);
    *j = (b & 1) ? cols - 1 - c : c;
}

__device__ __forceinline__ bool put(Slot &q, const double *A, const double *B, double g, double rc)
{
    q.ax = A[0];
    q.ay = A[1];
    q.az = A[2];
    q.bx = B[0];
    q.by = B[1];
    q.bz = B[2];
    q.gam = g;
    q.rc = rc;
    return g != 0.0;
}

__device__ __forceinline__ double skipg(double g) { return fabs(g) > EPS ? g : 0.0; }

// One source set of a rotor, as the staging kernel sees it: items of at
// most two segments.
//   SRC_WING   ring form, items 2k and 2k+1 hold filaments 0-1 and 2-3 of ring k
//   SRC_BOUND  bound vortices vf4 and vf2 of ring k, without vf2 of the
//              trailing row (blade_vind_bywing_boundVortices,
//              classdef.f90:1376-1395)
//   SRC_WAKE   lattice edges (below); SRC_PRESC prescribed far-wake
//              filaments (classdef.f90:1471-1476, 1501-1507)
enum { SRC_WING, SRC_BOUND, SRC_WAKE, SRC_PRESC };

struct SrcDesc {
    // wing: wc wrc wg; wake: node le gam rc4 ffc fgam frc; prescribed: pf ps
    const double *p[7];
    int kind, nc, ns, nN, nF, head, rn, rf, far_exists;
    int64_t first, count;      // its items, among those of the launch
    int64_t per_blade;         // items per blade (wake)
};

constexpr int SRC_MAX = 20;            // descriptors per launch (kernel argument space)
constexpr int STAGE_BLOCKS = 4096;     // staging blocks of one list

// The N-body targets of a rotor, written as SoA by blocks of their own in the
// staging launch: near-wake nodes of rows rn..nN-1 then far trailing ends,
// for its nbc convected blades.
struct TgtDesc {
    const double *node, *ffc;
    int ns, nN, nF, head, rn, rf, nbc;
    int block0;                // first target block of the launch
    int64_t off;               // of its targets
};

constexpr int TGT_MAX = 12;

struct StageArgs {
    SrcDesc d[SRC_MAX];
    TgtDesc t[TGT_MAX];
    int n, nt, iters, block0, tblock0;
    int64_t total, tstride;
    Slot *slots;
    int *counts;
    double *tgt;
};
static_assert(sizeof(StageArgs) <= 4096, "kernel argument space");

__device__ void gather_target(const TgtDesc &d, int64_t e, double *t, int64_t stride)
{
    const int R = d.nN - d.rn, F = max(d.nF - d.rf, 0), cols = d.ns + 1;
    const int64_t nnear = (int64_t)R * cols, per = nnear + F;
    if (e >= per * d.nbc) return;
    const int b = (int)(e / per);
    const int64_t k = e - b * per;
    const double *P;
    if (k < nnear) {
        int i, j;
        patch_entry(k, R, cols, &i, &j);
        int p = d.head + d.rn + i;
        if (p >= d.nN) p -= d.nN;
        P = d.node + 3 * (((size_t)b * d.nN + p) * cols + j);
    } else {
        P = d.ffc + 6 * ((size_t)b * d.nF + d.rf + (k - nnear));
    }
    t += d.off + e;
    t[0] = P[0];
    t[stride] = P[1];
    t[2 * stride] = P[2];
}

// Near- and far-wake unique segments of every blade.  Edge enumeration per
// blade (R active rows, F active far filaments; rows and columns in patch
// order):
//   [0, R*ns)            trailing spanwise edge of row i: T(i,j) -> T(i,j+1)
//   [.., + ns)           leading edge of the newest row:  LE(j+1) -> LE(j)
//   [.., + R*(ns+1))     streamwise edge: U(i,j) -> T(i,j)
//   [.., + F)            far filament fc1 -> fc2
__device__ __forceinline__ void wake_edge(const SrcDesc &d, int64_t e, Slot (&s)[2], bool (&f)[2])
{
    const int b = (int)(e / d.per_blade);
    int64_t k = e - (int64_t)b * d.per_blade;
    const int ns = d.ns, nN = d.nN;
    const double *N = d.p[0] + 3 * (size_t)b * nN * (ns + 1);
    const double *L = d.p[1] + 3 * (size_t)b * (ns + 1);
    const double *gam = d.p[2] + (size_t)b * nN * ns, *rc4 = d.p[3] + 4 * (size_t)b * nN * ns;
    const int R = nN - d.rn;
    auto phys = [&](int i) {
        const int p = d.head + i;
        return p >= nN ? p - nN : p;
    };
    if (k < (int64_t)R * ns) {
        int i, j;
        patch_entry(k, R, ns, &i, &j);
        i += d.rn;
        const int p = phys(i);
        const double *A = N + 3 * (p * (ns + 1) + j);
        const double ga = skipg(gam[p * ns + j]);
        const double rca = rc4[4 * (p * ns + j) + 1];
        double gb = 0.0, rcb = rca;
        bool hasb = false;
        if (i + 1 < nN) {
            const int q = phys(i + 1);
            gb = -skipg(gam[q * ns + j]);
            rcb = rc4[4 * (q * ns + j) + 3];
            hasb = true;
        } else if (d.far_exists) {
            // open horseshoe (classdef.f90:1458-1463): not |gam|-guarded
            gb = -gam[p * ns + j];
            hasb = true;
        }
        if (!hasb || rca == rcb) {
            f[0] = put(s[0], A, A + 3, ga + gb, rca);
        } else {
            f[0] = put(s[0], A, A + 3, ga, rca);
            f[1] = put(s[1], A, A + 3, gb, rcb);
        }
        return;
    }
    k -= (int64_t)R * ns;
    if (k < ns) {
        const int j = (int)k, r = phys(d.rn) * ns + j;
        f[0] = put(s[0], L + 3 * (j + 1), L + 3 * j, skipg(gam[r]), rc4[4 * r + 3]);
        return;
    }
    k -= ns;
    if (k < (int64_t)R * (ns + 1)) {
        int i, j;
        patch_entry(k, R, ns + 1, &i, &j);
        i += d.rn;
        const int p = phys(i);
        const double *T = N + 3 * (p * (ns + 1) + j);
        const double *U = (i == d.rn) ? L + 3 * j : N + 3 * (phys(i - 1) * (ns + 1) + j);
        double ga = 0.0, rca = 0.0, gb = 0.0, rcb = 0.0;
        const bool hasa = j < ns, hasb = j >= 1;
        if (hasa) {
            ga = skipg(gam[p * ns + j]);
            rca = rc4[4 * (p * ns + j) + 0];
        }
        if (hasb) {
            gb = -skipg(gam[p * ns + j - 1]);
            rcb = rc4[4 * (p * ns + j - 1) + 2];
        }
        if (hasa && hasb && rca == rcb) {
            f[0] = put(s[0], U, T, ga + gb, rca);
        } else {
            if (hasa) f[0] = put(s[0], U, T, ga, rca);
            if (hasb) f[1] = put(s[1], U, T, gb, rcb);
        }
        return;
    }
    k -= (int64_t)R * (ns + 1);
    const size_t q = (size_t)b * d.nF + d.rf + k;
    f[0] = put(s[0], d.p[4] + 6 * q, d.p[4] + 6 * q + 3, skipg(d.p[5][q]), d.p[6][q]);
}

// Segments of the items of up to SRC_MAX source sets, compacted within each
// block (item order) into the block's own slots, and their count.  Bound by
// latency (a few dependent loads per item); with emit_records_kernel the
// list of a pass takes two launches, where one launch per set, a device
// scan and a scatter took 2 nr + 3.
__global__ __launch_bounds__(256) void stage_kernel(StageArgs a)
{
    __shared__ int wsum[4];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    if ((int)blockIdx.x >= a.tblock0) {
        const int tb = (int)blockIdx.x - a.tblock0;
        int q = 0;
        while (q + 1 < a.nt && tb >= a.t[q + 1].block0) ++q;
        gather_target(a.t[q], (int64_t)(tb - a.t[q].block0) * 256 + tid, a.tgt, a.tstride);
        return;
    }
    const int blk = a.block0 + blockIdx.x;
    Slot *dst = a.slots + (size_t)blk * a.iters * 512;
    int run = 0;
    for (int it = 0; it < a.iters; ++it) {
        const int64_t e = ((int64_t)blockIdx.x * a.iters + it) * 256 + tid;
        Slot s[2];
        bool f[2] = {false, false};
        if (e < a.total) {
            int q = 0;
            while (q + 1 < a.n && e >= a.d[q + 1].first) ++q;
            const SrcDesc &d = a.d[q];
            const int64_t k = e - d.first;
            if (k >= d.count) {
                // between the last set of a list and the next list's block
            } else if (d.kind == SRC_WAKE) {
                wake_edge(d, k, s, f);
            } else if (d.kind == SRC_PRESC) {
                const int b = (int)(k / PF_N);
                f[0] = put(s[0], d.p[0] + 6 * k, d.p[0] + 6 * k + 3, skipg(d.p[1][4 * b]),
                           d.p[1][4 * b + 1]);
            } else {
                const int64_t r = d.kind == SRC_WING ? k >> 1 : k;
                const double *c = d.p[0] + 12 * r, *rc = d.p[1] + 4 * r;
                const double g = d.p[2][r];
                if (d.kind == SRC_WING) {
                    const int h = 2 * (int)(k & 1);
                    f[0] = put(s[0], c + 3 * h, c + 3 * h + 3, g, rc[h]);
                    f[1] = put(s[1], c + 3 * h + 3, c + 3 * ((h + 2) & 3), g, rc[h + 1]);
                } else {
                    f[0] = put(s[0], c + 9, c, g, rc[3]);
                    f[1] = put(s[1], c + 3, c + 6, (int)(r % d.nc) < d.nc - 1 ? g : 0.0, rc[1]);
                }
            }
        }
        const unsigned long long b0 = __ballot(f[0]), b1 = __ballot(f[1]);
        const unsigned long long lt = (1ull << lane) - 1;
        if (lane == 0) wsum[w] = __popcll(b0) + __popcll(b1);
        __syncthreads();
        int pos = run + __popcll(b0 & lt) + __popcll(b1 & lt);
        for (int q = 0; q < 4; ++q) {
            if (q < w) pos += wsum[q];
            run += wsum[q];
        }
        __syncthreads();
        if (f[0]) dst[pos++] = s[0];
        if (f[1]) dst[pos] = s[1];
    }
    if (tid == 0) a.counts[blk] = run;
}

// The staged segments in order, as records: each block forms the prefix sum
// of its list's staging counts, and each lane finds the block its record
// comes from by bisection.  List t was staged in blocks sb[t] to sb[t+1]-1,
// is emitted by the blocks from eb[t] and starts at record off[t].
struct EmitTab {
    int n, stride;
    int sb[TERM_MAX + 1], eb[TERM_MAX + 1];
    int64_t off[TERM_MAX];
};

__global__ __launch_bounds__(256) void emit_records_kernel(const Slot *slots, const int *counts,
                                                           EmitTab tab, SegPtrs L)
{
    __shared__ int pre[STAGE_BLOCKS + 1];
    __shared__ int wsum[4];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    int t = 0;
    while (t + 1 < tab.n && (int)blockIdx.x >= tab.eb[t + 1]) ++t;
    const int blk = (int)blockIdx.x - tab.eb[t];
    const int nblocks = tab.sb[t + 1] - tab.sb[t];
    counts += tab.sb[t];
    slots += (size_t)tab.sb[t] * tab.stride;
    const int per = (nblocks + 255) / 256;
    int mine = 0;
    for (int q = 0; q < per; ++q) {
        const int b = tid * per + q;
        if (b < nblocks) mine += counts[b];
    }
    int incl = mine;
    for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(incl, o);
        if (lane >= o) incl += v;
    }
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    int excl = incl - mine, total = 0;
    for (int q = 0; q < 4; ++q) {
        if (q < w) excl += wsum[q];
        total += wsum[q];
    }
    for (int q = 0; q < per; ++q) {
        const int b = tid * per + q;
        if (b < nblocks) {
            pre[b] = excl;
            excl += counts[b];
        }
    }
    if (blk == 0 && tid == 0) L.count[t] = total;
    __syncthreads();
    const int k = blk * 256 + tid;
    if ((k & ~(GRP - 1)) >= total) return;   // whole groups leave together
    const bool valid = k < total;
    const int kk = valid ? k : total - 1;
    int lo = 0, hi = nblocks;   // last block with pre[lo] <= kk
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (pre[mid] <= kk) lo = mid;
        else hi = mid;
    }
    const Slot s = slots[(size_t)lo * tab.stride + (kk - pre[lo])];
    write_group_records(s, valid, tab.off[t] + k, L);
}

// pFwake_update (classdef.f90:998-1066) for blade blockIdx.x of wake type
// pred, from the far filaments start .. start+n-1 (0-based):
//   radius = mean over them of |(y, x)| of the TE end, pitch = |sum of the
//   z steps between consecutive TE ends| (-2 pi / dpsi) / (n - 1), both
//   relaxed by half against the blade's previous values;
//   a 10-revolution helix of PF_N filaments, clockwise whatever the rotor
//   (isClockwiseRotor is never set, 231 and 1048), turned to the TE end of
//   the last filament (the anchor) and lifted to its height over the hub;
//   filament i joins helix points i (LE end) and i+1 (TE end), filament 0
//   starts at the anchor; every filament takes the last far filament's
//   circulation and core radius.
// The sums run in one lane in the reference's order.
__global__ __launch_bounds__(256) void presc_update_kernel(RV v, int pred, int start, int n,
                                                           double hx, double hy, double hz,
                                                           double dpsi, double *pf, double *ps)
{
    __shared__ double sh[4];
    const int b = blockIdx.x;
    const double *FC = (pred ? v.pffc : v.ffc) + 6 * ((size_t)b * v.nF + start);
    const double *anc = FC + 6 * (size_t)(n - 1);
    constexpr double twoPi = 2.0 * kPi;
    if (threadIdx.x == 0) {
        double pitch = 0.0, radius = 0.0;
        for (int i = 0; i < n; ++i) {
            const double *a = FC + 6 * (size_t)i;
            radius += sqrt(a[1] * a[1] + a[0] * a[0]);
            if (i < n - 1) pitch += a[2] - a[6 + 2];
        }
        pitch = fabs(pitch) * (-twoPi / dpsi) / (n - 1);
        radius = radius / n;
        double *S = ps + 4 * b;
        const size_t q = (size_t)b * v.nF + start + n - 1;
        S[0] = v.fgam[q];
        S[1] = v.frc[q];
        S[2] = 0.5 * pitch + (1 - 0.5) * S[2];
        S[3] = 0.5 * radius + (1 - 0.5) * S[3];
        sh[0] = S[2];
        sh[1] = S[3];
        sh[2] = atan2(anc[1], anc[0]);
        sh[3] = anc[2] - hz;
    }
    __syncthreads();
    const double pitch = sh[0], radius = sh[1], dth = sh[2], dz = sh[3];
    const double dx = (twoPi * 10.0 - 0.0) / (PF_N + 1 - 1);
    double *W = pf + 6 * (size_t)b * PF_N;
    for (int k = threadIdx.x; k <= PF_N; k += blockDim.x) {
        const double th = -(k * dx + 0.0);
        const double c0 = radius * cos(th + dth), c1 = radius * sin(th + dth);
        const double c2 = pitch * fabs(th) / twoPi + dz;
        if (k < PF_N) {   // LE end of filament k (filament 0: the anchor)
            W[6 * k + 3] = k == 0 ? anc[0] : hx + c0;
            W[6 * k + 4] = k == 0 ? anc[1] : hy + c1;
            W[6 * k + 5] = k == 0 ? anc[2] : hz + c2;
        }
        if (k > 0) {      // TE end of filament k-1
            W[6 * (k - 1) + 0] = hx + c0;
            W[6 * (k - 1) + 1] = hy + c1;
            W[6 * (k - 1) + 2] = hz + c2;
        }
    }
}

// Everything a velocity pass leads to, per lattice node and far filament and
// for all rotors of the launch: the pass's velocity (SoA, target order) into
// its array, the initial wake velocity, the predicted wake as a copy of the
// current one (main.f90:1028-1035), the scheme algebra and the convection.
// Bound by launches (about 5 us each): these were six to ten kernels per
// rotor and pass, each of a few kB to a few MB.
//
// Scheme algebra over whole velocity arrays of the convected blades, rows
// outside the wake included, as the reference has it (main.f90:968-1404):
// v = velNwake, v1..v3 = velNwake1..3, p = velNwakePredicted,
// s = velNwakeStep; statements after the bar follow the convection.
enum AdvOp {
    ADV_NONE,
    ADV_AB2,         // s = (3 v - v1) / 2; v1 = s; v = s
    ADV_AM2_PRED,    // s = v; v = (3 v - v1) / 2
    ADV_AM2_CORR,    // v = (p + s) / 2                           | v1 = s
    ADV_AM3_PRED,    // 1160-1171
    ADV_AM3_CORR,    // 1219-1235                                 | v1 = v2; v2 = s
    ADV_AM4_PRED,    // 1307-1320
    ADV_AM4_CORR,    // 1365-1385                                 | v1 = v2; v2 = v3; v3 = s
    ADV_KEEP1, ADV_KEEP2, ADV_KEEP3   //                          | v1, v2 or v3 = v
};

struct AdvRotor {
    double *node, *pnode, *le, *ple, *ffc, *pffc, *vel[NVEL], *velF[NVEL];
    double un[3], uf[3];             // initial wake velocity, near and far
    int ns, nN, nF, nbc, head, rn, rf;
    int i0, i1;                      // near rows convected
    int scatter, init, copy;
    int block0;                      // first block of the launch
    int64_t off;                     // of its targets
};

constexpr int ADV_MAX = 12;

struct AdvArgs {
    AdvRotor r[ADV_MAX];
    int n, slot, op, convect;        // slot: VLM_VEL or VLM_VEL_PRED;
                                     // convect: -1 none, 0 current, 1 predicted wake
    double dt;
    const double *o;
    int64_t stride;
};
static_assert(sizeof(AdvArgs) <= 4096, "kernel argument space");

// Nodes, far filaments and (copy) shed line points per blade.
__host__ __device__ __forceinline__ int64_t adv_per(const AdvRotor &r)
{
    return (int64_t)r.nN * (r.ns + 1) + r.nF + (r.copy ? r.ns + 1 : 0);
}

__global__ __launch_bounds__(256) void advance_kernel(AdvArgs a)
{
    int q = 0;
    while (q + 1 < a.n && (int)blockIdx.x >= a.r[q + 1].block0) ++q;
    const AdvRotor &r = a.r[q];
    const int64_t e = (int64_t)((int)blockIdx.x - r.block0) * 256 + threadIdx.x;
    const int64_t per = adv_per(r);
    if (e >= per * r.nbc) return;
    const int b = (int)(e / per);
    int64_t k = e - b * per;
    // per blade: the targets in their order, the rows and filaments outside
    // the wake, the shed line
    const int cols = r.ns + 1, R = max(r.nN - r.rn, 0), F = max(r.nF - r.rf, 0);
    const int64_t nnear = (int64_t)R * cols, nwin = nnear + F;
    const int64_t nout = (int64_t)(r.nN - R) * cols;
    const bool win = k < nwin;
    bool near;
    int i, j = 0;
    if (win) {
        near = k < nnear;
        if (near) {
            patch_entry(k, R, cols, &i, &j);
            i += r.rn;
        } else {
            i = r.rf + (int)(k - nnear);
        }
    } else if (k - nwin < nout) {
        near = true;
        i = (int)((k - nwin) / cols);
        j = (int)((k - nwin) % cols);
    } else if (k - nwin - nout < r.nF - F) {
        near = false;
        i = (int)(k - nwin - nout);
    } else {
        const size_t n = 3 * ((size_t)b * cols + (k - nwin - nout - (r.nF - F)));
        for (int d = 0; d < 3; ++d) r.ple[n + d] = r.le[n + d];
        return;
    }
    const size_t iv = near ? ((size_t)b * r.nN + i) * cols + j : (size_t)b * r.nF + i;
    auto arr = [&](int s) { return (near ? r.vel[s] : r.velF[s]) + 3 * iv; };
    double *V = arr(VLM_VEL), *X = arr(a.slot);
    double x[3], v[3];
    for (int d = 0; d < 3; ++d) {
        x[d] = win && r.scatter ? a.o[d * a.stride + r.off + b * nwin + k] : X[d];
        if (win && r.init) x[d] += near ? r.un[d] : r.uf[d];
        if (win && (r.scatter || r.init)) X[d] = x[d];
        v[d] = x[d];   // with slot VLM_VEL
    }
    if (a.op == ADV_NONE && a.convect < 0) return;
    double *V1 = arr(VLM_VEL_PREV), *V2 = arr(VEL_H2), *V3 = arr(VEL_H3), *S = arr(VLM_VEL_STEP);
    for (int d = 0; d < 3; ++d) {
        switch (a.op) {
        case ADV_AB2: {
            const double s = 0.5 * (3.0 * v[d] - V1[d]);
            S[d] = s;
            V1[d] = s;
            v[d] = s;
            break;
        }
        case ADV_AM2_PRED:
            S[d] = v[d];
            v[d] = 0.5 * (3.0 * v[d] - V1[d]);
            break;
        case ADV_AM3_PRED:
            S[d] = v[d];
            v[d] = (23.0 * v[d] - 16.0 * V2[d] + 5.0 * V1[d]) / 12.0;
            break;
        case ADV_AM4_PRED:
            S[d] = v[d];
            v[d] = (55.0 * v[d] - 59.0 * V3[d] + 37.0 * V2[d] - 9.0 * V1[d]) / 24.0;
            break;
        case ADV_AM2_CORR: {
            const double s = S[d];
            v[d] = (x[d] + s) * 0.5;
            V1[d] = s;
            break;
        }
        case ADV_AM3_CORR: {
            const double s = S[d], v2 = V2[d];
            v[d] = (5.0 * x[d] + 8.0 * s - v2) / 12.0;
            V1[d] = v2;
            V2[d] = s;
            break;
        }
        case ADV_AM4_CORR: {
            const double s = S[d], v2 = V2[d], v3 = V3[d];
            v[d] = (9.0 * x[d] + 19.0 * s - 5.0 * v3 + v2) / 24.0;
            V1[d] = v2;
            V2[d] = v3;
            V3[d] = s;
            break;
        }
        case ADV_KEEP1:
            V1[d] = v[d];
            break;
        case ADV_KEEP2:
            V2[d] = v[d];
            break;
        case ADV_KEEP3:
            V3[d] = v[d];
            break;
        default:
            break;
        }
        if (a.op >= ADV_AB2 && a.op <= ADV_AM4_CORR) V[d] = v[d];
    }
    if (a.convect < 0) return;
    // blade_convectwake (classdef.f90:1515-1575): nodes of rows [i0, i1) and
    // far trailing ends move by v dt; both wakes use velNwake, as the
    // reference does.  Far-wake continuity: fc2(i+1) <- fc1(i).
    const bool copied = win && r.copy;
    if (near) {
        const bool moves = i >= r.i0 && i < r.i1;
        if (!moves && !copied) return;
        int p = r.head + i;
        if (p >= r.nN) p -= r.nN;
        const size_t n = 3 * (((size_t)b * r.nN + p) * cols + j);
        double *P = (a.convect ? r.pnode : r.node) + n;
        const double *B = copied ? r.node + n : P;
        for (int d = 0; d < 3; ++d) {
            const double p0 = B[d];
            P[d] = moves ? p0 + v[d] * a.dt : p0;
        }
    } else if (win) {
        double *P = (a.convect ? r.pffc : r.ffc) + 6 * iv;
        const double *B = copied ? r.ffc + 6 * iv : P;
        for (int d = 0; d < 3; ++d) {
            const double p1 = B[d] + v[d] * a.dt;
            P[d] = p1;
            if (i + 1 < r.nF) P[9 + d] = p1;
            if (copied && i == r.rf) P[3 + d] = B[3 + d];
        }
    }
}

struct RotMats {
    double T[16][9];  // column-major getTransformAxis per blade
};

__device__ __forceinline__ void rotp(const double *T, const double *o, const double *p, double *q)
{
    const double x = p[0] - o[0], y = p[1] - o[1], z = p[2] - o[2];
    q[0] = T[0] * x + T[3] * y + T[6] * z + o[0];
    q[1] = T[1] * x + T[4] * y + T[7] * z + o[1];
    q[2] = T[2] * x + T[5] * y + T[8] * z + o[2];
}

// Axisymmetric copy of blade 1's wake to blades 2..nb rotated by
// 2 pi (ib-1)/nb about the shaft (rotor_convectwake, classdef.f90:4801-4823).
__global__ void axisym_kernel(RV v, int pred, RotMats M, double ox, double oy, double oz)
{
    const int R = v.nN - v.rn, F = v.nF - v.rf;
    const int64_t per = (int64_t)R * (v.ns + 1) + (v.ns + 1) + F + (int64_t)R * v.ns;
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= per * (v.nb - 1)) return;
    const int b = 1 + (int)(e / per);
    int64_t k = e - (int64_t)(b - 1) * per;
    const double o[3] = {ox, oy, oz};
    const double *T = M.T[b];
    if (k < (int64_t)R * (v.ns + 1)) {
        const int i = v.rn + (int)(k / (v.ns + 1)), j = (int)(k % (v.ns + 1));
        const int p = phys(v, i);
        double *N = pred ? v.pnode : v.node;
        rotp(T, o, N + 3 * nidx(v, 0, p, j), N + 3 * nidx(v, b, p, j));
        return;
    }
    k -= (int64_t)R * (v.ns + 1);
    if (k < v.ns + 1) {
        double *L = pred ? v.ple : v.le;
        rotp(T, o, L + 3 * k, L + 3 * ((size_t)b * (v.ns + 1) + k));
        return;
    }
    k -= v.ns + 1;
    if (k < F) {
        const int i = v.rf + (int)k;
        double *FC = pred ? v.pffc : v.ffc;
        const size_t q0 = (size_t)i, qb = (size_t)b * v.nF + i;
        rotp(T, o, FC + 6 * q0, FC + 6 * qb);
        rotp(T, o, FC + 6 * q0 + 3, FC + 6 * qb + 3);
        if (!pred) {
            v.fgam[qb] = v.fgam[q0];
            v.frc[qb] = v.frc[q0];
            v.frc0[qb] = v.frc0[q0];
            v.fl0[qb] = v.fl0[q0];
            v.flc[qb] = v.flc[q0];
            v.fage[qb] = v.fage[q0];
        }
        return;
    }
    k -= F;
    if (!pred) {
        const int i = v.rn + (int)(k / v.ns), j = (int)(k % v.ns);
        const int p = phys(v, i);
        const size_t r0 = ridx(v, 0, p, j), rb = ridx(v, b, p, j);
        v.gam[rb] = v.gam[r0];
        v.age[rb] = v.age[r0];
        for (int q = 0; q < 4; ++q) v.rc4[4 * rb + q] = v.rc4[4 * r0 + q];
    }
}

// Axisymmetric blades take blade 1's prescribed wake turned by
// 2 pi (b-1)/nb about the shaft (rotor_updatePrescribedWake,
// classdef.f90:5203-5215, pFwake_rot_wake_axis 1068-1086).
__global__ void presc_axisym_kernel(int nb, RotMats M, double ox, double oy, double oz,
                                    double *pf, double *ps)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (nb - 1) * PF_N) return;
    const int b = 1 + e / PF_N, i = e % PF_N;
    const double o[3] = {ox, oy, oz};
    const double *src = pf + 6 * (size_t)i;
    double *dst = pf + 6 * ((size_t)b * PF_N + i);
    rotp(M.T[b], o, src, dst);
    rotp(M.T[b], o, src + 3, dst + 3);
    if (i < 4) ps[4 * b + i] = ps[i];
}

// rotor_assignshed (classdef.f90:4297-4325).  LE: shed line of row rowNear
// from the wing trailing vortex ring corners 2/3, circulation of the wing
// trailing row.  TE: trailing nodes of row max(rowNear-1, 1).
__global__ void assignshed_kernel(RV v, int te, int row)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= v.nb * (v.ns + 1)) return;
    const int b = e / (v.ns + 1), j = e % (v.ns + 1);
    const int js = j < v.ns ? j : v.ns - 1;
    const size_t ring = ((size_t)b * v.ns + js) * v.nc + (v.nc - 1);
    const double *W = v.wc + 12 * ring + (j < v.ns ? 3 : 6);
    const int p = phys(v, row);
    double *dst = te ? v.node + 3 * nidx(v, b, p, j) : v.le + 3 * ((size_t)b * (v.ns + 1) + j);
    dst[0] = W[0];
    dst[1] = W[1];
    dst[2] = W[2];
    if (!te && j < v.ns) v.gam[ridx(v, b, p, j)] = v.wg[ring];
}

// rotor_age_wake (classdef.f90:4331-4354); ageAzimuthal is output-only.
__global__ void age_kernel(RV v, double dt)
{
    const int R = v.nN - v.rn, F = v.nF - v.rf;
    const int64_t per = (int64_t)R * v.ns + F;
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= per * v.nb) return;
    const int b = (int)(e / per);
    const int64_t k = e - b * per;
    if (k < (int64_t)R * v.ns) {
        const int i = v.rn + (int)(k / v.ns), j = (int)(k % v.ns);
        v.age[ridx(v, b, phys(v, i), j)] += dt;
    } else {
        v.fage[(size_t)b * v.nF + v.rf + (k - (int64_t)R * v.ns)] += dt;
    }
}

// rotor_dissipate_wake (classdef.f90:4356-4408): every ring grows vf1
// (copied to vf3) and vf2 and decays gam, far filaments grow and decay; vf4
// of every row but the newest takes the grown vf2 of the row upstream, whose
// lane writes it.
__global__ void dissipate_kernel(RV v, double inc, double decay)
{
    const int R = v.nN - v.rn, F = v.nF - v.rf;
    const int64_t per = (int64_t)R * v.ns + F;
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= per * v.nb) return;
    const int b = (int)(e / per);
    const int64_t k = e - b * per;
    if (k < (int64_t)R * v.ns) {
        const int i = v.rn + (int)(k / v.ns), j = (int)(k % v.ns);
        const size_t r = ridx(v, b, phys(v, i), j);
        double *rc = v.rc4 + 4 * r;
        rc[0] = sqrt(rc[0] * rc[0] + inc);
        rc[2] = rc[0];
        v.gam[r] = v.gam[r] * decay;
        const double rc2 = sqrt(rc[1] * rc[1] + inc);
        rc[1] = rc2;
        if (i + 1 < v.nN) v.rc4[4 * ridx(v, b, phys(v, i + 1), j) + 3] = rc2;
    } else {
        const size_t q = (size_t)b * v.nF + v.rf + (k - (int64_t)R * v.ns);
        v.frc[q] = sqrt(v.frc[q] * v.frc[q] + inc);
        v.fgam[q] = v.fgam[q] * decay;
    }
}

// rotor_strain_wake (classdef.f90:4410-4422): far filaments only.
__global__ void strain_kernel(RV v)
{
    const int F = v.nF - v.rf;
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (F <= 0 || e >= v.nb * F) return;
    const size_t q = (size_t)(e / F) * v.nF + v.rf + e % F;
    const double *fc = v.ffc + 6 * q;
    const double dx = fc[0] - fc[3], dy = fc[1] - fc[4], dz = fc[2] - fc[5];
    v.flc[q] = sqrt(dx * dx + dy * dy + dz * dz);
    v.frc[q] = v.frc0[q] * sqrt(v.fl0[q] / v.flc[q]);
}

// Skew of the far-wake pair (i, i+1): the angle between filament i
// (fc1 -> fc2) and filament i+1 reversed, as |acos(cos) - pi| / pi
// (blade_burst_wake, classdef.f90:2322-2338; getAngleCos, libMath.f90:238-247).
__device__ double far_pair_skew(const double *ffc, size_t q)
{
    const double *f = ffc + 6 * q, *g = ffc + 6 * (q + 1);
    const double ax = f[3] - f[0], ay = f[4] - f[1], az = f[5] - f[2];
    const double bx = g[0] - g[3], by = g[1] - g[4], bz = g[2] - g[5];
    const double d = ax * bx + ay * by + az * bz;
    const double n = sqrt((ax * ax + ay * ay + az * az) * (bx * bx + by * by + bz * bz));
    return fabs(acos(d / n) - kPi) / kPi;
}

// rotor_burst_wake (classdef.f90:4911-4917): a far filament takes the large
// core radius when the pair with either neighbour reaches the skew limit.
// One thread per filament, so no two threads write one core radius.
__global__ void burst_kernel(RV v, double skew_limit, double large_core)
{
    const int F = v.nF - v.rf;
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (F <= 0 || e >= v.nb * F) return;
    const int i = v.rf + e % F;
    const size_t q = (size_t)(e / F) * v.nF + i;
    bool burst = false;
    if (i > v.rf) burst = far_pair_skew(v.ffc, q - 1) >= skew_limit;
    if (i + 1 < v.nF) burst = burst || far_pair_skew(v.ffc, q) >= skew_limit;
    if (burst) v.frc[q] = large_core;
}

// The end of a step on a full near wake, one workgroup per blade:
//   shift_far  rotor_shiftFwake (classdef.f90:4500-4513) when no far
//              filament is free; blocks of 256 from the oldest down, each
//              read whole before it is written
//   rollup     rotor_rollup (4515-4597): the circulation-weighted centroid
//              of the oldest near row becomes the far filament fi; one lane
//              per sum, in the reference's order over the span
//   shift      rotor_shiftwake (4481-4498): the head moves back one slot,
//              the new logical row 0 duplicates row 1 with its age reset.
// Bound by launches: as four kernels it took four times 4 to 5 us.
__global__ __launch_bounds__(256) void rollup_kernel(RV v, int rs, int re, int rollup_min,
                                                     int suppress, int fi, int shift_far)
{
    const int b = blockIdx.x, tid = threadIdx.x;
    if (shift_far) {
        const size_t q0 = (size_t)b * v.nF;
        for (int c = (v.nF - 1) / 256 * 256; c >= 0; c -= 256) {
            const int i = c + tid;
            double t[12];
            const bool on = i > 0 && i < v.nF;
            if (on) {
                const size_t q = q0 + i - 1;
                for (int d = 0; d < 6; ++d) t[d] = v.ffc[6 * q + d];
                t[6] = v.fgam[q];
                t[7] = v.frc[q];
                t[8] = v.frc0[q];
                t[9] = v.fl0[q];
                t[10] = v.flc[q];
                t[11] = v.fage[q];
            }
            __syncthreads();
            if (on) {
                const size_t q = q0 + i;
                for (int d = 0; d < 6; ++d) v.ffc[6 * q + d] = t[d];
                v.fgam[q] = t[6];
                v.frc[q] = t[7];
                v.frc0[q] = t[8];
                v.fl0[q] = t[9];
                v.flc[q] = t[10];
                v.fage[q] = t[11];
            } else if (i == 0) {
                v.fage[q0] = 0.0;
            }
        }
        __syncthreads();
    }
    const int last = v.nN - 1;
    const int p = phys(v, last);
    if (tid < 64) {
        const double *N = v.node;
        const double *L = v.le + 3 * (size_t)b * (v.ns + 1);
        // corner 4 of ring (last, j) = node(last-1, j+1) or the shed line
        const double *c4 = last == v.rn ? L + 3 : N + 3 * nidx(v, b, phys(v, last - 1), 1);
        const double *c3 = N + 3 * nidx(v, b, p, 1);
        const double *G = v.gam + ridx(v, b, p, 0), *RC = v.rc4 + 4 * ridx(v, b, p, 0);
        // lanes 0-2 leading centroid, 3-5 trailing, 6 radius, 7 circulation,
        // 8 its extremum
        double acc = tid == 8 ? G[v.ns - 1] : 0.0;
        const double *w = tid < 3 ? c4 + tid : tid < 6 ? c3 + tid - 3 : RC + 2;
        const int ws = tid < 6 ? 3 : 4;
        for (int j = rs; j <= re; ++j) {
            const double g = G[j];
            if (tid < 7) acc += w[ws * j] * g;
            else if (tid == 7) acc += g;
            else if (rollup_min ? g < acc : g > acc) acc = g;
        }
        double s[9];
        for (int k = 0; k < 9; ++k) s[k] = __shfl(acc, k);
        if (tid == 0 && v.nF > 0) {
            if (fabs(s[7]) > EPS) {
                for (int k = 0; k < 7; ++k) s[k] /= s[7];
            } else {
                for (int d = 0; d < 3; ++d) {
                    s[d] = c3[3 * (re - 1) + d];
                    s[3 + d] = c3[3 * re + d];
                }
                s[6] = RC[4 * re + 2];
            }
            const size_t q = (size_t)b * v.nF + fi;
            double *fc = v.ffc + 6 * q;
            for (int d = 0; d < 3; ++d) {
                fc[3 + d] = s[d];
                fc[d] = s[3 + d];
            }
            v.fgam[q] = suppress ? 0.0 : s[8];
            v.fage[q] = v.age[ridx(v, b, p, v.ns - 1)];
            v.frc0[q] = s[6];
            v.frc[q] = s[6];
            const double dx = s[3] - s[0], dy = s[4] - s[1], dz = s[5] - s[2];
            v.flc[q] = v.fl0[q] = sqrt(dx * dx + dy * dy + dz * dz);
            if (fi + 1 < v.nF)
                for (int d = 0; d < 3; ++d) v.ffc[6 * (q + 1) + 3 + d] = s[3 + d];
        }
    }
    __syncthreads();
    // the slot of the oldest row becomes the new row 0
    const int p1 = phys(v, 0);
    for (int j = tid; j <= v.ns; j += 256) {
        const double *s = v.node + 3 * nidx(v, b, p1, j);
        double *d = v.node + 3 * nidx(v, b, p, j);
        d[0] = s[0];
        d[1] = s[1];
        d[2] = s[2];
        if (j < v.ns) {
            const size_t r0 = ridx(v, b, p, j), r1 = ridx(v, b, p1, j);
            v.gam[r0] = v.gam[r1];
            for (int q = 0; q < 4; ++q) v.rc4[4 * r0 + q] = v.rc4[4 * r1 + q];
            v.age[r0] = 0.0;
        }
    }
}

// Part of a wake for the host: the doubles [c0, c0 + n) of its arrays one
// after the other, near rows in logical order, written straight to pinned
// memory.
struct WakePack {
    const double *src[7];      // nodes le gam rc4 | far ends, circulations, radii
    int64_t end[7];            // of each array, in doubles
    int64_t c0, n;
    int nN, head, row[7];      // doubles per near row, 0 where there are none
    double *dst;
};

__global__ __launch_bounds__(256) void wake_pack_kernel(WakePack a)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= a.n) return;
    int64_t k = a.c0 + e;
    int q = 0;
    while (k >= a.end[q]) ++q;
    if (q > 0) k -= a.end[q - 1];
    if (a.row[q]) {
        const int64_t r = k / a.row[q], b = r / a.nN;
        int64_t p = r - b * a.nN + a.head;
        if (p >= a.nN) p -= a.nN;
        k = (b * a.nN + p) * a.row[q] + (k - r * a.row[q]);
    }
    a.dst[e] = a.src[q][k];
}

// vel_order2_Nwake / vel_order2_Fwake (libCommon.f90:213-258) on the
// active window, written to `out` (logical rows).
__global__ void order2_kernel(const double *vn, const double *vnp1, double *out, int nbc,
                              int rows, int stride, int cols, int base)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (int64_t)nbc * rows * cols * 3) return;
    const int d = (int)(e % 3);
    int64_t r = e / 3;
    const int i = (int)(r % rows);
    r /= rows;
    const int j = (int)(r % cols);
    const int b = (int)(r / cols);
    auto at = [&](int ii) { return (((size_t)b * stride + base + ii) * cols + j) * 3 + d; };
    double val;
    if (i == 0 || i == rows - 1) val = (vnp1[at(i)] + vn[at(i)]) * 0.5;
    else val = (vnp1[at(i)] + vnp1[at(i - 1)] + vn[at(i + 1)] + vn[at(i)]) * 0.25;
    out[at(i)] = val;
}

__global__ void copy_window_kernel(const double *src, double *dst, int nbc, int rows, int stride,
                                   int cols, int base)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (int64_t)nbc * rows * cols * 3) return;
    const int d = (int)(e % 3);
    int64_t r = e / 3;
    const int i = (int)(r % rows);
    r /= rows;
    const int j = (int)(r % cols);
    const int b = (int)(r / cols);
    const size_t k = (((size_t)b * stride + base + i) * cols + j) * 3 + d;
    dst[k] = src[k];
}

__global__ void negate_kernel(double *p, int64_t n)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < n) p[e] = -p[e];
}

__global__ void fill_kernel(double *p, int64_t n, double val)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) p[k] = val;
}

// rotor_mirrorWake (classdef.f90:5024-5131) with vr_mirror / Fwake_mirror
// (722-735, 982-993): image d takes source s's wake on every blade, with
// coordinate ax and the circulation negated.  mode 0 (C): current near
// rows from i0 and far filaments from f0; 1 (P): predicted positions over
// the same rows, with the circulation, cores and ages, which the predicted
// wake shares with the current one (the reference copies them inside its
// predicted rings; the current rows get the same values again at the C
// mirror that follows); 2 (A): every row, i0 = f0 = 0.  Rows are logical
// on both sides (each rotor has its own ring head).  One thread per near node, leading-edge
// node, near ring or far filament of a blade.
__global__ void mirror_wake_kernel(RV d, RV s, int mode, int ax, int i0, int f0)
{
    const int ns = d.ns, R = d.nN - i0, F = d.nF - f0;
    const int64_t per = (int64_t)R * (ns + 1) + (ns + 1) + (int64_t)R * ns + F;
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= per * d.nb) return;
    const int b = (int)(e / per);
    int64_t k = e - b * per;
    const bool pred = mode == 1;
    auto copy3 = [ax](const double *src, double *dst) {
        dst[0] = src[0];
        dst[1] = src[1];
        dst[2] = src[2];
        dst[ax] = -src[ax];
    };
    if (k < (int64_t)R * (ns + 1)) {
        const int i = i0 + (int)(k / (ns + 1)), j = (int)(k % (ns + 1));
        copy3((pred ? s.pnode : s.node) + 3 * nidx(s, b, phys(s, i), j),
              (pred ? d.pnode : d.node) + 3 * nidx(d, b, phys(d, i), j));
        return;
    }
    k -= (int64_t)R * (ns + 1);
    if (k < ns + 1) {
        const size_t q = 3 * ((size_t)b * (ns + 1) + k);
        copy3((pred ? s.ple : s.le) + q, (pred ? d.ple : d.le) + q);
        return;
    }
    k -= ns + 1;
    if (k < (int64_t)R * ns) {
        const int i = i0 + (int)(k / ns), j = (int)(k % ns);
        const size_t rs = ridx(s, b, phys(s, i), j), rd = ridx(d, b, phys(d, i), j);
        d.gam[rd] = -s.gam[rs];
        d.age[rd] = s.age[rs];
        for (int q = 0; q < 4; ++q) d.rc4[4 * rd + q] = s.rc4[4 * rs + q];
        return;
    }
    k -= (int64_t)R * ns;
    const size_t q = (size_t)b * d.nF + f0 + k;
    const double *FS = pred ? s.pffc : s.ffc;
    double *FD = pred ? d.pffc : d.ffc;
    copy3(FS + 6 * q, FD + 6 * q);
    copy3(FS + 6 * q + 3, FD + 6 * q + 3);
    d.fgam[q] = -s.fgam[q];
    d.frc[q] = s.frc[q];
    d.frc0[q] = s.frc0[q];
    d.fl0[q] = s.fl0[q];
    d.flc[q] = s.flc[q];
    d.fage[q] = s.fage[q];
}

// rotor_mirrorGamma + rotor_map_gam: the image's wing circulation is the
// negated source's, ring for ring.
__global__ void mirror_gamma_kernel(const double *src, double *dst, int n)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e < n) dst[e] = -src[e];
}

}  // namespace

// ---------------------------------------------------------------------
// host-side helpers
// ---------------------------------------------------------------------
static int64_t wake_edges_per_blade(const Rotor &r)
{
    const int64_t R = r.d.nNwake - (r.rowNear - 1);
    const int64_t F = r.d.nFwake - (r.rowFar - 1);
    if (r.d.nNwake <= 0 || R <= 0) return F > 0 ? F : 0;
    return R * r.d.ns + r.d.ns + R * (r.d.ns + 1) + (F > 0 ? F : 0);
}

// prescribed far-wake sources: one slot per filament while a far wake exists
static int64_t presc_slots(const Rotor &r)
{
    return (r.presc_nt > 0 && r.rowFar <= r.d.nFwake) ? (int64_t)PF_N * r.d.nb : 0;
}

namespace {

int64_t target_count(const Rotor &r)
{
    if (r.d.nNwake <= 0 || r.image_of >= 0) return 0;
    const int64_t R = r.d.nNwake - (r.rowNear - 1);
    const int64_t F = r.d.nFwake - (r.rowFar - 1);
    if (R <= 0) return 0;
    return (R * (r.d.ns + 1) + (F > 0 ? F : 0)) * r.d.nbConvect;
}

Rotor *get_rotor(vlm_ctx *ctx, int ir)
{
    if (!ctx || ir < 0 || ir >= (int)ctx->rotors.size()) return nullptr;
    return ctx->rotors[ir];
}

// Source sets of (rotor, set) pairs as staging descriptors; total receives
// the number of items, est the expected number of segments (two per wing
// item, one per wake edge: edges whose two ring filaments differ in core
// radius are the exception).
void source_descs(vlm_ctx *ctx, const std::vector<std::pair<int, int>> &src,
                  std::vector<SrcDesc> &ds, int64_t *total, int64_t *est)
{
    int64_t n = 0, wing = 0;
    for (auto &q : src) {
        Rotor &r = *ctx->rotors[q.first];
        SrcDesc d;
        std::memset(&d, 0, sizeof(d));
        d.nc = r.d.nc;
        d.ns = r.d.ns;
        d.first = n;
        if (q.second == VLM_SET_WING || q.second == VLM_SET_WING_BOUND) {
            d.kind = q.second == VLM_SET_WING ? SRC_WING : SRC_BOUND;
            d.p[0] = r.wc.p;
            d.p[1] = r.wrc.p;
            d.p[2] = r.wg.p;
            const int64_t items = (int64_t)r.nring * (d.kind == SRC_WING ? 2 : 1);
            d.count = items;
            n += items;
            wing += items;
            ds.push_back(d);
            continue;
        }
        const int64_t per = wake_edges_per_blade(r);
        // no active near-wake row yet: no wake
        if (r.d.nNwake <= 0 || r.rowNear - 1 >= r.d.nNwake || per <= 0) continue;
        const int pred = q.second == VLM_SET_WAKE_PRED ? 1 : 0;
        d.kind = SRC_WAKE;
        d.p[0] = pred ? r.pnode.p : r.node.p;
        d.p[1] = pred ? r.ple.p : r.le.p;
        d.p[2] = r.gam.p;
        d.p[3] = r.rc4.p;
        d.p[4] = pred ? r.pffc.p : r.ffc.p;
        d.p[5] = r.fgam.p;
        d.p[6] = r.frc.p;
        d.nN = r.d.nNwake;
        d.nF = r.d.nFwake;
        d.head = r.head;
        d.rn = r.rowNear - 1;
        d.rf = r.rowFar - 1;
        d.far_exists = r.rowFar <= r.d.nFwake ? 1 : 0;
        d.per_blade = per;
        d.count = per * r.d.nb;
        n += d.count;
        ds.push_back(d);
        const int64_t np = presc_slots(r);
        if (np > 0) {
            std::memset(&d, 0, sizeof(d));
            d.kind = SRC_PRESC;
            d.p[0] = r.pf[pred].p;
            d.p[1] = r.ps[pred].p;
            d.first = n;
            d.count = np;
            n += np;
            ds.push_back(d);
        }
    }
    *total = n;
    *est = n + wing;
}

typedef std::vector<std::pair<int, int>> Sources;   // (rotor, set) pairs

// Build up to TERM_MAX source lists into ctx->seg, in the given formats:
// where each starts and its expected number of segments go to *lists (empty
// sets give lists of no segments).
// With pred >= 0 the staging launches also gather the N-body targets on the
// current (0) or predicted (1) wake, m in total, into ctx->tgt.
int build_lists(vlm_ctx *ctx, const std::vector<Sources> &terms, int formats, TermLists *lists,
                int pred = -1, int64_t m = 0)
{
    const int nt = (int)terms.size();
    std::vector<std::vector<SrcDesc>> ds(nt);
    std::vector<int64_t> total(nt);
    int64_t all = 0, nd = 0, cap = 0;
    lists->n = nt;
    for (int t = 0; t < nt; ++t) {
        source_descs(ctx, terms[t], ds[t], &total[t], &lists->est[t]);
        lists->off[t] = cap;
        cap += (2 * total[t] + GRP - 1) / GRP * GRP;
        all += total[t];
        nd += (int64_t)ds[t].size();
    }
    if (all > INT32_MAX / 4) return fail(ctx, VLM_ERR_ARG, "segment list too large");
    // items per staging block; a list starts on a block of its own, and a
    // launch (SRC_MAX sets) ends with one
    const int64_t spare = nt + nd / SRC_MAX + 1;
    StageArgs a;
    a.iters = (int)((all + 256 * (STAGE_BLOCKS - spare) - 1) / (256 * (STAGE_BLOCKS - spare)));
    if (a.iters < 1) a.iters = 1;
    const int64_t bi = 256 * (int64_t)a.iters;   // items per block
    VLM_HIP(ctx->slots.reserve(ws_size<Slot>((size_t)(all / bi + spare + 1) * a.iters * 512)));
    VLM_HIP(ctx->seg_counts.reserve(STAGE_BLOCKS));
    VLM_HIP(ctx->seg.reserve(std::max<int64_t>(cap, 4096), formats, &ctx->seg_view));
    a.slots = ctx->slots.p;
    a.counts = ctx->seg_counts.p;
    a.n = 0;
    a.nt = 0;
    a.block0 = 0;
    a.total = 0;
    int tblocks = 0;
    auto flush = [&]() {
        const int nb = (int)((a.total + bi - 1) / bi);
        a.tblock0 = nb;
        if (nb + tblocks > 0)
            hipLaunchKernelGGL(stage_kernel, dim3(nb + tblocks), dim3(256), 0, ctx->stream, a);
        a.block0 += nb;
        a.n = 0;
        a.nt = 0;
        a.total = 0;
        tblocks = 0;
    };
    if (pred >= 0) {
        VLM_HIP(ctx->tgt.reserve(ws_size<double>((size_t)3 * m)));
        a.tgt = ctx->tgt.p;
        a.tstride = m;
        int64_t off = 0;
        for (auto *r : ctx->rotors) {
            const int64_t n = target_count(*r);
            if (n == 0) continue;
            if (a.nt == TGT_MAX) flush();
            TgtDesc &d = a.t[a.nt++];
            d.node = pred ? r->pnode.p : r->node.p;
            d.ffc = pred ? r->pffc.p : r->ffc.p;
            d.ns = r->d.ns;
            d.nN = r->d.nNwake;
            d.nF = r->d.nFwake;
            d.head = r->head;
            d.rn = r->rowNear - 1;
            d.rf = r->rowFar - 1;
            d.nbc = r->d.nbConvect;
            d.block0 = tblocks;
            d.off = off;
            tblocks += (int)nblk(n);
            off += n;
        }
    }
    EmitTab tab;
    tab.n = nt;
    tab.stride = a.iters * 512;
    int eb = 0;
    for (int t = 0; t < nt; ++t) {
        a.total = (a.total + bi - 1) / bi * bi;
        tab.sb[t] = a.block0 + (int)(a.total / bi);
        tab.eb[t] = eb;
        tab.off[t] = lists->off[t];
        for (auto &d : ds[t]) {
            if (a.n == SRC_MAX) flush();
            a.d[a.n] = d;
            a.d[a.n++].first = a.total;
            a.total += d.count;
        }
        // at least one block writes the count
        eb += (int)std::max<int64_t>(1, (2 * total[t] + 255) / 256);
    }
    a.total = (a.total + bi - 1) / bi * bi;
    tab.sb[nt] = a.block0 + (int)(a.total / bi);
    flush();
    tab.eb[nt] = eb;
    hipLaunchKernelGGL(emit_records_kernel, dim3(eb), dim3(256), 0, ctx->stream, ctx->slots.p,
                       ctx->seg_counts.p, tab, ctx->seg_view);
    VLM_HIP(hipGetLastError());
    return VLM_OK;
}

// The expected number of segments of a list.
int64_t expected(vlm_ctx *ctx, const Sources &src)
{
    std::vector<SrcDesc> ds;
    int64_t n = 0, est = 0;
    source_descs(ctx, src, ds, &n, &est);
    return est;
}

// One list; *est receives its expected number of segments.
int build_sources(vlm_ctx *ctx, const Sources &src, int formats, int64_t *est, int pred = -1,
                  int64_t m = 0)
{
    TermLists one;
    VLM_TRY(build_lists(ctx, {src}, formats, &one, pred, m));
    *est = one.est[0];
    return VLM_OK;
}

int eval_sources(vlm_ctx *ctx, const double *t, int64_t m, int64_t tstride, double *out, int acc,
                 int64_t est)
{
    return bs_eval(ctx, ctx->seg_view, est, t, m, tstride, out, acc);
}

// getTransformAxis, libMath.f90:695-726 (column-major)
void transform_axis(double theta, const double *ax, double *T)
{
    const double n = std::sqrt(ax[0] * ax[0] + ax[1] * ax[1] + ax[2] * ax[2]);
    const double a0 = ax[0] / n, a1 = ax[1] / n, a2 = ax[2] / n;
    const double ct = std::cos(theta), st = std::sin(theta), om = 1.0 - ct;
    T[0] = ct + a0 * a0 * om;
    T[1] = a2 * st + a1 * a0 * om;
    T[2] = -a1 * st + a2 * a0 * om;
    T[3] = -a2 * st + a0 * a1 * om;
    T[4] = ct + a1 * a1 * om;
    T[5] = a0 * st + a2 * a1 * om;
    T[6] = a1 * st + a0 * a2 * om;
    T[7] = -a0 * st + a1 * a2 * om;
    T[8] = ct + a2 * a2 * om;
}

}  // namespace

// rotor_updatePrescribedWake, classdef.f90:5172-5217: the far filaments
// from rowFar (prescWakeGenNt = 0) or the last prescWakeGenNt + 1.
static int presc_update(vlm_ctx *ctx, Rotor &r, int pred)
{
    const int nF = r.d.nFwake;
    const int start = r.presc_gen_nt == 0 ? r.rowFar - 1 : nF - r.presc_gen_nt - 1;
    const int n = nF - start;
    if (start < 0 || n < 1) return VLM_OK;  // no far filament to anchor to
    if (std::fabs(r.shaft[0]) > kEps || std::fabs(r.shaft[1]) > kEps)
        return fail(ctx, VLM_ERR_ARG, "Prescribed far wake only implemented for shaft along Z-axis");
    const int t = pred ? 1 : 0;
    hipLaunchKernelGGL(presc_update_kernel, dim3(r.d.nbConvect), dim3(256), 0, ctx->stream,
                       view(r), pred, start, n, r.hub[0], r.hub[1], r.hub[2], r.presc_dpsi,
                       r.pf[t].p, r.ps[t].p);
    VLM_HIP(hipGetLastError());
    if (r.d.nbConvect == 1 && r.d.nb > 1) {
        if (r.d.nb > 16) return fail(ctx, VLM_ERR_ARG, "axisymmetric copy supports <= 16 blades");
        RotMats M;
        std::memset(&M, 0, sizeof(M));
        for (int b = 1; b < r.d.nb; ++b) transform_axis(2.0 * kPi / r.d.nb * b, r.shaft, M.T[b]);
        hipLaunchKernelGGL(presc_axisym_kernel, dim3(nblk((int64_t)(r.d.nb - 1) * PF_N)),
                           dim3(256), 0, ctx->stream, r.d.nb, M, r.hub[0], r.hub[1], r.hub[2],
                           r.pf[t].p, r.ps[t].p);
        VLM_HIP(hipGetLastError());
    }
    r.presc_built[t] = 1;
    return VLM_OK;
}

// rotor_mirrorWake of image r from its source (mode 0 C, 1 P, 2 A).
int mirror_wake(vlm_ctx *ctx, Rotor &r, int mode)
{
    if (r.image_of < 0 || r.image_of >= (int)ctx->rotors.size())
        return fail(ctx, VLM_ERR_STATE, "rotor is not an image (vlm_rotor_set_image)");
    Rotor &s = *ctx->rotors[r.image_of];
    if (r.d.nNwake <= 0) return VLM_OK;
    const int i0 = mode == 2 ? 0 : r.rowNear - 1, f0 = mode == 2 ? 0 : r.rowFar - 1;
    const int R = r.d.nNwake - i0, F = r.d.nFwake - f0;
    if (R < 0 || F < 0) return fail(ctx, VLM_ERR_STATE, "wake cursors out of range");
    const int64_t per = (int64_t)R * (r.d.ns + 1) + (r.d.ns + 1) + (int64_t)R * r.d.ns + F;
    hipLaunchKernelGGL(mirror_wake_kernel, dim3(nblk(per * r.d.nb)), dim3(256), 0, ctx->stream,
                       view(r), view(s), mode, r.image_axis, i0, f0);
    VLM_HIP(hipGetLastError());
    return VLM_OK;
}

// What follows the convection of a rotor of its own: the axisymmetric copy
// of blade 1's wake and the prescribed far wake (classdef.f90:4826-4829).
static int after_convect(vlm_ctx *ctx, Rotor &r, int pred)
{
    if (r.d.nbConvect == 1 && r.d.nb > 1) {
        if (r.d.nb > 16) return fail(ctx, VLM_ERR_ARG, "axisymmetric copy supports <= 16 blades");
        RotMats M;
        std::memset(&M, 0, sizeof(M));
        for (int b = 1; b < r.d.nb; ++b) {
            const double theta = 2.0 * kPi / r.d.nb * b;
            transform_axis(theta, r.shaft, M.T[b]);
        }
        const int64_t R = r.d.nNwake - (r.rowNear - 1), F = r.d.nFwake - (r.rowFar - 1);
        const int64_t per2 = (R > 0 ? R : 0) * (r.d.ns + 1) + (r.d.ns + 1) + (F > 0 ? F : 0) +
                             (R > 0 ? R : 0) * r.d.ns;
        hipLaunchKernelGGL(axisym_kernel, dim3(nblk(per2 * (r.d.nb - 1))), dim3(256), 0,
                           ctx->stream, view(r), pred, M, r.hub[0], r.hub[1], r.hub[2]);
        VLM_HIP(hipGetLastError());
    }
    if (r.presc_nt > 0 && r.iter > r.presc_nt) VLM_TRY(presc_update(ctx, r, pred));
    return VLM_OK;
}

// One advance of every rotor, or of rotor `only`.
struct Advance {
    int slot = VLM_VEL, op = ADV_NONE, convect = -1;
    bool scatter = false;   // ctx->out holds the pass's velocities, m targets
    bool init = false;      // add the initial wake velocity of step iter
    bool copy = false;      // predicted wake := current wake before it moves
    double dt = 0.0;
    int iter = 0;
    int64_t m = 0;
    const Rotor *only = nullptr;
};

static int advance(vlm_ctx *ctx, const Advance &p)
{
    AdvArgs a;
    a.n = 0;
    a.slot = p.slot;
    a.op = p.op;
    a.convect = p.convect;
    a.dt = p.dt;
    a.o = ctx->out.p;
    a.stride = p.m;
    int blocks = 0;
    Rotor *batch[ADV_MAX];
    auto flush = [&]() -> int {
        if (blocks > 0)
            hipLaunchKernelGGL(advance_kernel, dim3(blocks), dim3(256), 0, ctx->stream, a);
        VLM_HIP(hipGetLastError());
        if (p.convect >= 0)
            for (int q = 0; q < a.n; ++q) VLM_TRY(after_convect(ctx, *batch[q], p.convect));
        a.n = 0;
        blocks = 0;
        return VLM_OK;
    };
    int64_t off = 0;
    for (auto *r : ctx->rotors) {
        const int64_t nt = p.scatter ? target_count(*r) : 0, toff = off;
        off += nt;
        if ((p.only && r != p.only) || r->d.nNwake <= 0) continue;
        if (r->image_of >= 0) {
            // an image mirrors its source's wake at its place in the order
            if (p.convect < 0) continue;
            VLM_TRY(flush());
            VLM_TRY(mirror_wake(ctx, *r, p.convect));
            continue;
        }
        if (a.n == ADV_MAX) VLM_TRY(flush());
        batch[a.n] = r;
        AdvRotor &d = a.r[a.n++];
        d.node = r->node.p;
        d.pnode = r->pnode.p;
        d.le = r->le.p;
        d.ple = r->ple.p;
        d.ffc = r->ffc.p;
        d.pffc = r->pffc.p;
        for (int k = 0; k < NVEL; ++k) {
            d.vel[k] = r->velN[k].p;
            d.velF[k] = r->velF[k].p;
        }
        // initWakeVel of pass 1 (main.f90:829-838: + near, - far) or of pass
        // 2 (902-913 and the AM blocks: - near, - far)
        const double u = r->init_wake_vel, un = p.slot == VLM_VEL ? u : -u;
        d.init = p.init && p.iter < r->init_wake_vel_nt && u != 0.0;
        for (int k = 0; k < 3; ++k) {
            d.un[k] = un * r->shaft[k];
            d.uf[k] = -u * r->shaft[k];
        }
        d.ns = r->d.ns;
        d.nN = r->d.nNwake;
        d.nF = r->d.nFwake;
        d.nbc = r->d.nbConvect;
        d.head = r->head;
        d.rn = r->rowNear - 1;
        d.rf = r->rowFar - 1;
        d.i0 = d.rn;
        d.i1 = d.nN;
        if (p.convect == 1 && ctx->bug_compat) {
            d.i0 = 0;  // `do i = 1, rowNear, nNwake` runs for row 1 only
            d.i1 = 1;
        }
        d.scatter = nt > 0;
        d.copy = p.copy && d.nN > d.rn;
        d.block0 = blocks;
        d.off = toff;
        blocks += (int)nblk(adv_per(d) * d.nbc);
    }
    return flush();
}

// Velocities of all targets on the current or predicted wake into ctx->out;
// *m receives their number.
static int wake_pass(vlm_ctx *ctx, int pred, int64_t *mp)
{
    Sources src;
    int64_t m = 0;
    for (int ir = 0; ir < (int)ctx->rotors.size(); ++ir) {
        src.push_back({ir, VLM_SET_WING});
        src.push_back({ir, pred ? VLM_SET_WAKE_PRED : VLM_SET_WAKE});
        m += target_count(*ctx->rotors[ir]);
    }
    *mp = m;
    if (m == 0) return VLM_OK;
    int64_t nest = 0;
    VLM_TRY(build_sources(ctx, src, bs_formats(ctx, m, expected(ctx, src)), &nest, pred, m));
    VLM_HIP(ctx->out.reserve(ws_size<double>((size_t)3 * m)));
    return eval_sources(ctx, ctx->tgt.p, m, m, ctx->out.p, 0, nest);
}


// ---------------------------------------------------------------------
// Learned pass 2 (AM2 predictor stage): the MLP proposes the velocity on
// the predicted wake; a strided sample of targets is evaluated by the full
// Biot-Savart sum every step as judge and training data, and the whole
// pass is recomputed when the sampled error exceeds the tolerance.
// ---------------------------------------------------------------------
namespace {

__constant__ int kNbr[12][2] = {{-1, 0}, {1, 0}, {0, -1}, {0, 1}, {-1, -1}, {-1, 1},
                                {1, -1}, {1, 1}, {-2, 0}, {2, 0}, {0, -2}, {0, 2}};

// 45 features per P-pass target in gather order: 12 neighbour offsets on
// the predicted lattice (scaled by 1/lref) and three velocities scaled by
// 1/vref: pass-1 velocity, previous step's velocity, AB2 predictor velocity.
__global__ void features_kernel(RV v, float *X, int64_t off, double lref_inv,
                                const double *vref)
{
    const int R = v.nN - v.rn, F = v.nF - v.rf;
    const int64_t per = (int64_t)R * (v.ns + 1) + F;
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= per * v.nbc) return;
    const int b = (int)(e / per);
    const int64_t k = e - b * per;
    float *x = X + (off + e) * 45;
    const double vinv = 1.0 / vref[0];
    const double *vs, *vp, *va;
    if (k < (int64_t)R * (v.ns + 1)) {
        int i, j;
        patch_entry(k, R, v.ns + 1, &i, &j);
        i += v.rn;
        const double *P = v.pnode + 3 * nidx(v, b, phys(v, i), j);
        for (int q = 0; q < 12; ++q) {
            const int ii = i + kNbr[q][0], jj = j + kNbr[q][1];
            float ox = 0.f, oy = 0.f, oz = 0.f;
            if (jj >= 0 && jj <= v.ns && ii >= v.rn - 1 && ii < v.nN) {
                const double *Q = (ii == v.rn - 1) ? v.ple + 3 * ((size_t)b * (v.ns + 1) + jj)
                                                   : v.pnode + 3 * nidx(v, b, phys(v, ii), jj);
                ox = (float)((Q[0] - P[0]) * lref_inv);
                oy = (float)((Q[1] - P[1]) * lref_inv);
                oz = (float)((Q[2] - P[2]) * lref_inv);
            }
            x[3 * q] = ox;
            x[3 * q + 1] = oy;
            x[3 * q + 2] = oz;
        }
        const size_t vi = 3 * vidx(v, b, i, j);
        vs = v.vel[VLM_VEL_STEP] + vi;
        vp = v.vel[VLM_VEL_PREV] + vi;
        va = v.vel[VLM_VEL] + vi;
    } else {
        const int i = v.rf + (int)(k - (int64_t)R * (v.ns + 1));
        for (int q = 0; q < 36; ++q) x[q] = 0.f;
        const size_t vi = 3 * ((size_t)b * v.nF + i);
        vs = v.velF[VLM_VEL_STEP] + vi;
        vp = v.velF[VLM_VEL_PREV] + vi;
        va = v.velF[VLM_VEL] + vi;
    }
    for (int d = 0; d < 3; ++d) {
        x[36 + d] = (float)(vs[d] * vinv);
        x[39 + d] = (float)(vp[d] * vinv);
        x[42 + d] = (float)(va[d] * vinv);
    }
}

// Pass-1 velocity of every P-pass target (gather order), SoA.
__global__ void gather_step_vel_kernel(RV v, double *o, int64_t stride, int64_t off)
{
    const int R = v.nN - v.rn, F = v.nF - v.rf;
    const int64_t per = (int64_t)R * (v.ns + 1) + F;
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= per * v.nbc) return;
    const int b = (int)(e / per);
    const int64_t k = e - b * per;
    const double *V;
    if (k < (int64_t)R * (v.ns + 1)) {
        int i, j;
        patch_entry(k, R, v.ns + 1, &i, &j);
        i += v.rn;
        V = v.vel[VLM_VEL_STEP] + 3 * vidx(v, b, i, j);
    } else {
        V = v.velF[VLM_VEL_STEP] + 3 * ((size_t)b * v.nF + v.rf + (k - (int64_t)R * (v.ns + 1)));
    }
    o[off + e] = V[0];
    o[stride + off + e] = V[1];
    o[2 * stride + off + e] = V[2];
}

// vref = RMS of the pass-1 speed over all targets (single block).
__global__ __launch_bounds__(1024) void vref_kernel(const double *vn, int64_t m, double *vref)
{
    __shared__ double sh[1024];
    double s = 0.0;
    for (int64_t k = threadIdx.x; k < m; k += blockDim.x)
        s += vn[k] * vn[k] + vn[m + k] * vn[m + k] + vn[2 * m + k] * vn[2 * m + k];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int w = 512; w > 0; w >>= 1) {
        if (threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) vref[0] = fmax(sqrt(sh[0] / (double)(m > 0 ? m : 1)), 1e-12);
}

// v = v_pass1 + y * sigma * vref for every target, sigma = scal[4] the RMS
// of the replay buffer's targets: the network predicts the correction in
// units of its typical size.  With sigma = 0 (every recorded pass 2 equal
// to pass 1) the prediction is the pass-1 velocity itself.
__global__ void apply_mlp_kernel(const double *vn, const float *Y, int64_t m, const double *scal,
                                 double *out)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= m) return;
    const double s = scal[0] * scal[4];
    for (int d = 0; d < 3; ++d)
        out[d * m + e] = vn[d * m + e] + (s > 0.0 ? (double)Y[3 * e + d] * s : 0.0);
}

// sigma = RMS of the n x 3 buffer targets (single block, fixed order) into
// scal[4]; 0 for an empty buffer.
__global__ __launch_bounds__(1024) void target_scale_kernel(const float *bt, int64_t n,
                                                            double *scal)
{
    __shared__ double sh[1024];
    double s = 0.0;
    for (int64_t k = threadIdx.x; k < 3 * n; k += blockDim.x) s += (double)bt[k] * bt[k];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int w = 512; w > 0; w >>= 1) {
        if (threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) scal[4] = n > 0 ? sqrt(sh[0] / (double)(3 * n)) : 0.0;
}

// Minibatch targets in units of sigma (zero when sigma is zero).
__global__ void scale_targets_kernel(const float *bt, int64_t n3, const double *scal, float *out)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n3) return;
    const double sg = scal[4];
    out[k] = sg > 0.0 ? (float)((double)bt[k] / sg) : 0.f;
}

// Sampled targets: e = phase + k*stride.  Gather their positions.
__global__ void gather_sample_kernel(const double *t, int64_t m, int64_t phase, int64_t stride,
                                     int64_t ms, double *ts)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= ms) return;
    const int64_t e = phase + k * stride;
    ts[k] = t[e];
    ts[ms + k] = t[m + e];
    ts[2 * ms + k] = t[2 * m + e];
}

// Judge: per-sample squared error and squared exact speed; then write the
// exact values into the output and the training pair into the buffer.
// The same sample also scores the network-free substitute for pass 2, the
// linear extrapolation 2 v_n - v_(n-1) of the pass-1 velocity (with it the
// AM2 corrector reduces to AB2), so that the network's gain is measured on
// identical targets.
__global__ void judge_kernel(const double *vs, int64_t ms, const double *out, int64_t m,
                             int64_t phase, int64_t stride, const double *vn, const float *X,
                             const double *vref, double *err2, double *ref2, double *base2,
                             float *bx, float *bt, int64_t bcap, int64_t bhead)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= ms) return;
    const int64_t e = phase + k * stride;
    double se = 0.0, sr = 0.0, sb = 0.0;
    const double inv = 1.0 / vref[0];
    const int64_t slot = (bhead + k) % bcap;
    for (int d = 0; d < 3; ++d) {
        const double a = vs[d * ms + k], p = out[d * m + e];
        const double ex = 2.0 * vn[d * m + e] - (double)X[45 * e + 39 + d] * vref[0];
        se += (a - p) * (a - p);
        sr += a * a;
        sb += (a - ex) * (a - ex);
        bt[3 * slot + d] = (float)((a - vn[d * m + e]) * inv);
    }
    for (int q = 0; q < 45; ++q) bx[45 * slot + q] = X[45 * e + q];
    err2[k] = se;
    ref2[k] = sr;
    base2[k] = sb;
}

__global__ void put_sample_kernel(const double *vs, int64_t ms, double *out, int64_t m,
                                  int64_t phase, int64_t stride)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= ms) return;
    const int64_t e = phase + k * stride;
    for (int d = 0; d < 3; ++d) out[d * m + e] = vs[d * ms + k];
}

// Sums of three length-n arrays a, a+n, a+2n (one block, fixed order).
__global__ void sum3_kernel(const double *a, int64_t n, double *out)
{
    __shared__ double sh[3][256];
    double x[3] = {0.0, 0.0, 0.0};
    for (int64_t k = threadIdx.x; k < n; k += blockDim.x)
        for (int c = 0; c < 3; ++c) x[c] += a[c * n + k];
    for (int c = 0; c < 3; ++c) sh[c][threadIdx.x] = x[c];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w)
            for (int c = 0; c < 3; ++c) sh[c][threadIdx.x] += sh[c][threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int c = 0; c < 3; ++c) out[c] = sh[c][0];
}

// Training pairs from a full pass: every stride-th target.
__global__ void full_pairs_kernel(const double *vexact, const double *vn, int64_t m,
                                  const float *X, const double *vref, int64_t stride, int64_t np,
                                  float *bx, float *bt, int64_t bcap, int64_t bhead)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= np) return;
    const int64_t e = k * stride;
    const int64_t slot = (bhead + k) % bcap;
    const double inv = 1.0 / vref[0];
    for (int d = 0; d < 3; ++d) bt[3 * slot + d] = (float)((vexact[d * m + e] - vn[d * m + e]) * inv);
    for (int q = 0; q < 45; ++q) bx[45 * slot + q] = X[45 * e + q];
}

}  // namespace

// Full Biot-Savart pass 2 of the learned mode, plus training pairs from it
// (every stride-th target, a quarter of the replay buffer).
static int full_pass(vlm_ctx *ctx, int64_t m, int64_t nest)
{
    Predictor &P = ctx->pred;
    VLM_TRY(eval_sources(ctx, ctx->tgt.p, m, m, ctx->out.p, 0, nest));
    P.full += 1;
    const int64_t stride = (m + P.buf_cap / 4 - 1) / (P.buf_cap / 4);
    const int64_t np = (m + stride - 1) / stride;
    hipLaunchKernelGGL(full_pairs_kernel, dim3(nblk(np)), dim3(256), 0, ctx->stream, ctx->out.p,
                       P.vn.p, m, P.X.p, P.scal.p, stride, np, P.bx.p, P.bt.p, P.buf_cap,
                       P.buf_head);
    VLM_HIP(hipGetLastError());
    P.buf_head = (P.buf_head + np) % P.buf_cap;
    P.buf_n = P.buf_n + np < P.buf_cap ? P.buf_n + np : P.buf_cap;
    return VLM_OK;
}

int learned_pass(vlm_ctx *ctx, int64_t *mp)
{
    Predictor &P = ctx->pred;
    Sources src;
    int64_t m = 0;
    for (int ir = 0; ir < (int)ctx->rotors.size(); ++ir) {
        src.push_back({ir, VLM_SET_WING});
        src.push_back({ir, VLM_SET_WAKE_PRED});
        m += target_count(*ctx->rotors[ir]);
    }
    *mp = m;
    if (m == 0) return VLM_OK;
    int64_t nest = 0;
    // the full pass reads m targets, the judge about m / stride of them
    const int64_t stride0 = P.stride < 1 ? 1 : P.stride;
    const int64_t est = expected(ctx, src);
    int formats = bs_formats(ctx, m, est) | bs_formats(ctx, (m + stride0 - 1) / stride0, est) |
                  bs_formats(ctx, std::max<int64_t>(1, (m - stride0) / stride0), est);
    VLM_TRY(build_sources(ctx, src, formats, &nest, 1, m));
    VLM_HIP(ctx->out.reserve(ws_size<double>((size_t)3 * m)));
    VLM_HIP(P.vn.reserve((size_t)3 * m));
    VLM_HIP(P.X.reserve((size_t)45 * m));
    VLM_HIP(P.Y.reserve((size_t)3 * m));
    VLM_HIP(P.scal.reserve(8));
    VLM_HIP(P.tb.reserve((size_t)3 * P.batch));
    if (P.bx.n < (size_t)45 * P.buf_cap) {
        VLM_HIP(P.bx.reserve((size_t)45 * P.buf_cap));
        VLM_HIP(P.bt.reserve((size_t)3 * P.buf_cap));
    }
    int64_t off = 0;
    for (auto *rp : ctx->rotors) {
        const int64_t n = target_count(*rp);
        if (n == 0) continue;
        hipLaunchKernelGGL(gather_step_vel_kernel, dim3(nblk(n)), dim3(256), 0, ctx->stream,
                           view(*rp), P.vn.p, m, off);
        off += n;
    }
    hipLaunchKernelGGL(vref_kernel, dim3(1), dim3(1024), 0, ctx->stream, P.vn.p, m, P.scal.p);
    off = 0;
    for (auto *rp : ctx->rotors) {
        const int64_t n = target_count(*rp);
        if (n == 0) continue;
        hipLaunchKernelGGL(features_kernel, dim3(nblk(n)), dim3(256), 0, ctx->stream, view(*rp),
                           P.X.p, off, 1.0 / P.lref, P.scal.p);
        off += n;
    }
    // scale of the corrections seen so far (the buffer before this step)
    hipLaunchKernelGGL(target_scale_kernel, dim3(1), dim3(1024), 0, ctx->stream, P.bt.p,
                       P.buf_n, P.scal.p);
    VLM_HIP(hipGetLastError());
    const bool warm = P.steps < P.warmup;
    P.steps += 1;
    int64_t ms = 0, phase = 0, stride = 1;
    const double *judged_sums = nullptr;
    if (!warm) {
        VLM_TRY(mlp_forward_dev(ctx, m, P.X.p, P.Y.p));
        hipLaunchKernelGGL(apply_mlp_kernel, dim3(nblk(m)), dim3(256), 0, ctx->stream, P.vn.p,
                           P.Y.p, m, P.scal.p, ctx->out.p);
        // judge on a strided sample with a rotating phase
        stride = P.stride < 1 ? 1 : P.stride;
        phase = (P.steps * 7) % stride < m ? (P.steps * 7) % stride : 0;
        ms = (m - phase + stride - 1) / stride;
        VLM_HIP(P.ts.reserve((size_t)3 * ms));
        VLM_HIP(P.vs.reserve((size_t)3 * ms));
        VLM_HIP(P.e2.reserve((size_t)3 * ms));
        hipLaunchKernelGGL(gather_sample_kernel, dim3(nblk(ms)), dim3(256), 0, ctx->stream,
                           ctx->tgt.p, m, phase, stride, ms, P.ts.p);
        VLM_TRY(eval_sources(ctx, P.ts.p, ms, ms, P.vs.p, 0, nest));
        const int64_t take = ms < P.buf_cap ? ms : P.buf_cap;
        hipLaunchKernelGGL(judge_kernel, dim3(nblk(take)), dim3(256), 0, ctx->stream, P.vs.p,
                           take, ctx->out.p, m, phase, stride, P.vn.p, P.X.p, P.scal.p, P.e2.p,
                           P.e2.p + take, P.e2.p + 2 * take, P.bx.p, P.bt.p, P.buf_cap,
                           P.buf_head);
        hipLaunchKernelGGL(sum3_kernel, dim3(1), dim3(256), 0, ctx->stream, P.e2.p, take,
                           P.scal.p + 1);
        VLM_HIP(hipGetLastError());
        // the sums travel to pinned memory behind an event; the host waits
        // for them only after the training below is enqueued, so the GPU
        // trains while the host decides
        if (!ctx->judge_ev)
            VLM_HIP(hipEventCreateWithFlags(&ctx->judge_ev, hipEventDisableTiming));
        if (!ctx->judge_pin)
            VLM_HIP(hipHostMalloc(reinterpret_cast<void **>(&ctx->judge_pin), 4 * sizeof(double)));
        VLM_HIP(hipMemcpyAsync(ctx->judge_pin, P.scal.p + 1, 3 * sizeof(double),
                               hipMemcpyDeviceToHost, ctx->stream));
        VLM_HIP(hipEventRecord(ctx->judge_ev, ctx->stream));
        judged_sums = ctx->judge_pin;
        P.buf_head = (P.buf_head + take) % P.buf_cap;
        P.buf_n = P.buf_n + take < P.buf_cap ? P.buf_n + take : P.buf_cap;
    } else {
        VLM_TRY(full_pass(ctx, m, nest));
    }
    // Adam on minibatches: contiguous windows of the replay buffer at a
    // rotating offset (on a judged step before the decision, so the pairs
    // of a fallback pass are trained on from the next step)
    for (int it = 0; it < P.train_iters && P.buf_n > 0; ++it) {
        const int64_t B = P.buf_n < P.batch ? P.buf_n : P.batch;
        const int64_t start = (P.train_calls * 7919) % (P.buf_n - B + 1);
        P.train_calls += 1;
        hipLaunchKernelGGL(scale_targets_kernel, dim3(nblk(3 * B)), dim3(256), 0, ctx->stream,
                           P.bt.p + 3 * start, 3 * B, P.scal.p, P.tb.p);
        VLM_HIP(hipGetLastError());
        VLM_TRY(mlp_train_dev(ctx, B, P.bx.p + 45 * start, P.tb.p, 1, P.lr, nullptr,
                              it == P.train_iters - 1));
    }
    if (judged_sums) {
        VLM_HIP(hipEventSynchronize(ctx->judge_ev));
        const double h0 = judged_sums[0], h1 = judged_sums[1], h2 = judged_sums[2];
        P.last_err = h1 > 0 ? std::sqrt(h0 / h1) : 0.0;
        P.sum_err2 += h0;
        P.sum_ref2 += h1;
        P.sum_base2 += h2;
        P.judged += 1;
        if (P.last_err > P.tol) {
            P.fallbacks += 1;
            VLM_TRY(full_pass(ctx, m, nest));
        } else {
            hipLaunchKernelGGL(put_sample_kernel, dim3(nblk(ms)), dim3(256), 0, ctx->stream,
                               P.vs.p, ms, ctx->out.p, m, phase, stride);
            VLM_HIP(hipGetLastError());
            P.learned += 1;
        }
    }
    return VLM_OK;
}

}  // namespace vlm

using namespace vlm;

extern "C" {

int vlm_rotor_create(vlm_ctx *ctx, const vlm_rotor_desc *d, double spanwiseCore,
                     const double *scv, int *ir)
{
    if (!ctx || !d || !ir) return VLM_ERR_ARG;
    if (d->nb <= 0 || d->nc <= 0 || d->ns <= 0 || d->nNwake < 0 || d->nFwake < 0)
        return fail(ctx, VLM_ERR_ARG, "rotor sizes must be positive");
    if (d->nbConvect != 1 && d->nbConvect != d->nb)
        return fail(ctx, VLM_ERR_ARG, "nbConvect must be 1 or nb");
    if (d->nNwake > 0 && d->nNwake < 2)
        return fail(ctx, VLM_ERR_ARG, "at least 2 near wake rows are mandatory");
    if (d->nNwake > 0 && (d->rollupStart < 1 || d->rollupEnd > d->ns || d->rollupStart > d->rollupEnd + 1))
        return fail(ctx, VLM_ERR_ARG, "rollup span range outside 1..ns");
    if (d->nNwake > 0 && !scv) return fail(ctx, VLM_ERR_ARG, "streamwiseCoreVec missing");
    VLM_HIP(hipSetDevice(ctx->device));
    Rotor *r = new Rotor();
    r->d = *d;
    r->nring = d->nb * d->nc * d->ns;
    const size_t nb = d->nb, nN = d->nNwake, ns = d->ns, nF = d->nFwake;
    hipError_t e = hipSuccess;
    auto R = [&](DBuf<double> &b, size_t n) {
        if (e == hipSuccess) e = b.reserve(n);
    };
    R(r->wc, 12 * (size_t)r->nring);
    R(r->wrc, 4 * (size_t)r->nring);
    R(r->wg, r->nring);
    R(r->node, 3 * nb * nN * (ns + 1));
    R(r->pnode, 3 * nb * nN * (ns + 1));
    R(r->le, 3 * nb * (ns + 1));
    R(r->ple, 3 * nb * (ns + 1));
    R(r->gam, nb * nN * ns);
    R(r->rc4, 4 * nb * nN * ns);
    R(r->age, nb * nN * ns);
    R(r->ffc, 6 * nb * nF);
    R(r->pffc, 6 * nb * nF);
    R(r->fgam, nb * nF);
    R(r->frc, nb * nF);
    R(r->frc0, nb * nF);
    R(r->fl0, nb * nF);
    R(r->flc, nb * nF);
    R(r->fage, nb * nF);
    for (int k = 0; k < NVEL; ++k) {
        R(r->velN[k], r->nvn());
        R(r->velF[k], r->nvf());
    }
    for (int t = 0; t < 2; ++t) {
        R(r->pf[t], 6 * nb * PF_N);
        R(r->ps[t], 4 * nb);
    }
    R(r->pan, (size_t)PANEL_N * r->nring);
    R(r->sec, (size_t)SECTION_N * nb * ns);
    R(r->bla, (size_t)BLADE_N * nb);
    R(r->cps, 3 * (size_t)r->nring);
    R(r->vcp, 6 * (size_t)r->nring);
    R(r->rhs, r->nring);
    R(r->vld, 3 * (size_t)r->nring);
    R(r->gprev, r->nring);
    R(r->lout, (size_t)LOADS_SEC_N * nb * ns + LOADS_ROTOR_N);
    if (e != hipSuccess) {
        delete r;
        return hip_fail(ctx, e, "rotor allocation");
    }
    // zero everything (the reference zero-initialises every velocity array,
    // classdef.f90:3737-3820, and all wake circulations, 3830-3831)
    std::vector<DBuf<double> *> all = {&r->wc,   &r->wrc,  &r->wg,   &r->node, &r->pnode,
                                       &r->le,   &r->ple,  &r->gam,  &r->rc4,  &r->age,
                                       &r->ffc,  &r->pffc, &r->fgam, &r->frc,  &r->frc0,
                                       &r->fl0,  &r->flc,  &r->fage};
    for (int k = 0; k < NVEL; ++k) {
        all.push_back(&r->velN[k]);
        all.push_back(&r->velF[k]);
    }
    for (int t = 0; t < 2; ++t) {
        all.push_back(&r->pf[t]);
        all.push_back(&r->ps[t]);
    }
    for (auto *b : {&r->pan, &r->sec, &r->bla, &r->cps, &r->vcp, &r->rhs, &r->vld, &r->gprev,
                    &r->lout})
        all.push_back(b);
    for (auto *b : all)
        hipLaunchKernelGGL(fill_kernel, dim3(nblk((int64_t)b->n)), dim3(256), 0, ctx->stream,
                           b->p, (int64_t)b->n, 0.0);
    // initial core radii, classdef.f90:3826-3850
    if (nN > 0) {
        std::vector<double> rc4(4 * nb * nN * ns);
        for (size_t b = 0; b < nb; ++b)
            for (size_t i = 0; i < nN; ++i)
                for (size_t j = 0; j < ns; ++j) {
                    double *q = &rc4[4 * ((b * nN + i) * ns + j)];
                    q[0] = scv[j];
                    q[1] = spanwiseCore;
                    q[2] = scv[j + 1];
                    q[3] = spanwiseCore;
                }
        VLM_HIP(hipMemcpyAsync(r->rc4.p, rc4.data(), rc4.size() * sizeof(double),
                               hipMemcpyHostToDevice, ctx->stream));
        if (nF > 0) {
            std::vector<double> frc(nb * nF, scv[ns]);
            VLM_HIP(hipMemcpyAsync(r->frc.p, frc.data(), frc.size() * sizeof(double),
                                   hipMemcpyHostToDevice, ctx->stream));
            VLM_HIP(hipMemcpyAsync(r->frc0.p, frc.data(), frc.size() * sizeof(double),
                                   hipMemcpyHostToDevice, ctx->stream));
        }
        VLM_TRY(sync_stream(ctx));
    }
    r->rowNear = (int)nN + 1;
    r->rowFar = (int)nF + 1;
    ctx->rotors.push_back(r);
    ctx->aic.push_back(nullptr);
    ctx->lu.push_back(nullptr);
    ctx->piv.push_back(nullptr);
    ctx->aic_n.push_back(0);
    *ir = (int)ctx->rotors.size() - 1;
    return VLM_OK;
}

int vlm_rotor_set_wing(vlm_ctx *ctx, int ir, const double *corners, const double *rc,
                       const double *gam)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor") : VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    if (corners) VLM_TRY(h2d(ctx, r->wc.p, corners, sizeof(double) * 12 * r->nring));
    if (rc) VLM_TRY(h2d(ctx, r->wrc.p, rc, sizeof(double) * 4 * r->nring));
    if (gam) VLM_TRY(h2d(ctx, r->wg.p, gam, sizeof(double) * r->nring));
    return VLM_OK;
}

int vlm_rotor_set_axis(vlm_ctx *ctx, int ir, const double *shaft, const double *hub)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r || !shaft || !hub) return ctx ? fail(ctx, VLM_ERR_ARG, "bad rotor axis") : VLM_ERR_ARG;
    std::memcpy(r->shaft, shaft, sizeof(r->shaft));
    std::memcpy(r->hub, hub, sizeof(r->hub));
    return VLM_OK;
}

int vlm_rotor_set_init_wake_vel(vlm_ctx *ctx, int ir, double initWakeVel, int initWakeVelNt)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor") : VLM_ERR_ARG;
    if (!std::isfinite(initWakeVel)) return fail(ctx, VLM_ERR_ARG, "initWakeVel not finite");
    r->init_wake_vel = initWakeVel;
    r->init_wake_vel_nt = initWakeVelNt;
    return VLM_OK;
}

int vlm_rotor_init_cursors(vlm_ctx *ctx, int ir)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor") : VLM_ERR_ARG;
    r->rowFar = r->d.nFwake + 1;
    r->rowNear = r->d.nNwake + 1;
    return VLM_OK;
}

int vlm_rotor_begin_step(vlm_ctx *ctx, int ir, int iter)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor") : VLM_ERR_ARG;
    r->iter = iter;
    r->rowNear = r->rowNear - 1 > 1 ? r->rowNear - 1 : 1;
    if (iter > r->d.nNwake) r->rowFar = r->rowFar - 1 > 1 ? r->rowFar - 1 : 1;
    return VLM_OK;
}

int vlm_rotor_cursors(vlm_ctx *ctx, int ir, int *rowNear, int *rowFar)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor") : VLM_ERR_ARG;
    if (rowNear) *rowNear = r->rowNear;
    if (rowFar) *rowFar = r->rowFar;
    return VLM_OK;
}

int vlm_rotor_assignshed(vlm_ctx *ctx, int ir, int edge)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor") : VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    if (r->d.nNwake <= 0) return VLM_OK;
    if (edge != VLM_EDGE_LE && edge != VLM_EDGE_TE)
        return fail(ctx, VLM_ERR_ARG, "edge must be VLM_EDGE_LE or VLM_EDGE_TE");
    int row;
    if (edge == VLM_EDGE_LE) {
        if (r->rowNear > r->d.nNwake) return fail(ctx, VLM_ERR_STATE, "assignshed LE before first step");
        row = r->rowNear - 1;
    } else {
        row = (r->rowNear - 1 > 1 ? r->rowNear - 1 : 1) - 1;
    }
    hipLaunchKernelGGL(assignshed_kernel, dim3(nblk((int64_t)r->d.nb * (r->d.ns + 1))), dim3(256),
                       0, ctx->stream, view(*r), edge == VLM_EDGE_TE ? 1 : 0, row);
    VLM_HIP(hipGetLastError());
    return VLM_OK;
}

int vlm_rotor_age_wake(vlm_ctx *ctx, int ir, double dt)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor") : VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    if (r->d.nNwake <= 0 || r->rowNear > r->d.nNwake) return VLM_OK;
    const int64_t R = r->d.nNwake - (r->rowNear - 1);
    const int64_t F = r->d.nFwake - (r->rowFar - 1);
    const int64_t n = (R * r->d.ns + (F > 0 ? F : 0)) * r->d.nb;
    hipLaunchKernelGGL(age_kernel, dim3(nblk(n)), dim3(256), 0, ctx->stream, view(*r), dt);
    VLM_HIP(hipGetLastError());
    return VLM_OK;
}

int vlm_rotor_dissipate_wake(vlm_ctx *ctx, int ir, double dt, double kinematicVisc,
                             double apparentViscCoeff, double decayCoeff)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor") : VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    if (r->d.nNwake <= 0 || r->rowNear > r->d.nNwake) return VLM_OK;
    const double oseen = 1.2564;
    const double inc = 4.0 * oseen * apparentViscCoeff * kinematicVisc * dt;
    const double decay = std::exp(-decayCoeff * dt);
    const int64_t R = r->d.nNwake - (r->rowNear - 1);
    const int64_t F = r->d.nFwake - (r->rowFar - 1);
    const int64_t n = (R * r->d.ns + (F > 0 ? F : 0)) * r->d.nb;
    hipLaunchKernelGGL(dissipate_kernel, dim3(nblk(n)), dim3(256), 0, ctx->stream, view(*r), inc,
                       decay);
    VLM_HIP(hipGetLastError());
    return VLM_OK;
}

int vlm_rotor_strain_wake(vlm_ctx *ctx, int ir)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor") : VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    const int64_t F = r->d.nFwake - (r->rowFar - 1);
    if (r->d.nNwake <= 0 || F <= 0) return VLM_OK;
    hipLaunchKernelGGL(strain_kernel, dim3(nblk(F * r->d.nb)), dim3(256), 0, ctx->stream,
                       view(*r));
    VLM_HIP(hipGetLastError());
    return VLM_OK;
}

// Every device array of a rotor's state, in a fixed order (restart files).
static std::vector<DBuf<double> *> state_bufs(Rotor &r)
{
    std::vector<DBuf<double> *> v = {&r.wc,  &r.wrc, &r.wg,  &r.node, &r.pnode, &r.le,
                                     &r.ple, &r.gam, &r.rc4, &r.age,  &r.ffc,   &r.pffc,
                                     &r.fgam, &r.frc, &r.frc0, &r.fl0, &r.flc,  &r.fage};
    for (int k = 0; k < NVEL; ++k) {
        v.push_back(&r.velN[k]);
        v.push_back(&r.velF[k]);
    }
    for (int t = 0; t < 2; ++t) {
        v.push_back(&r.pf[t]);
        v.push_back(&r.ps[t]);
    }
    v.push_back(&r.gprev);  // gamPrev of the loads (blade_calc_force)
    return v;
}

static int64_t state_bytes(Rotor &r)
{
    int64_t n = 4 * (int64_t)sizeof(int64_t);
    for (auto *b : state_bufs(r)) n += (int64_t)(b->n * sizeof(double));
    return n;
}

int vlm_rotor_state_bytes(vlm_ctx *ctx, int ir, int64_t *bytes)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r || !bytes) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor or null pointer")
                                 : VLM_ERR_ARG;
    *bytes = state_bytes(*r);
    return VLM_OK;
}

int vlm_rotor_get_state(vlm_ctx *ctx, int ir, void *buf, int64_t bytes)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r || !buf) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor or null buffer")
                               : VLM_ERR_ARG;
    if (bytes != state_bytes(*r)) return fail(ctx, VLM_ERR_ARG, "state size mismatch");
    VLM_DEVICE(ctx);
    VLM_TRY(sync_stream(ctx));
    int64_t *h = static_cast<int64_t *>(buf);
    h[0] = r->rowNear;
    h[1] = r->rowFar;
    h[2] = r->head;
    h[3] = r->presc_built[0] | (r->presc_built[1] << 1);
    char *p = static_cast<char *>(buf) + 4 * sizeof(int64_t);
    for (auto *b : state_bufs(*r)) {
        if (b->n) VLM_HIP(hipMemcpy(p, b->p, b->n * sizeof(double), hipMemcpyDeviceToHost));
        p += b->n * sizeof(double);
    }
    return VLM_OK;
}

int vlm_rotor_set_state(vlm_ctx *ctx, int ir, const void *buf, int64_t bytes)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r || !buf) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor or null buffer")
                               : VLM_ERR_ARG;
    if (bytes != state_bytes(*r)) return fail(ctx, VLM_ERR_ARG, "state size mismatch");
    const int64_t *h = static_cast<const int64_t *>(buf);
    if (h[0] < 1 || h[0] > r->d.nNwake + 1 || h[1] < 1 || h[1] > r->d.nFwake + 1 || h[2] < 0 ||
        h[2] >= (r->d.nNwake > 0 ? r->d.nNwake : 1))
        return fail(ctx, VLM_ERR_ARG, "state cursors out of range");
    VLM_DEVICE(ctx);
    VLM_TRY(sync_stream(ctx));
    const char *p = static_cast<const char *>(buf) + 4 * sizeof(int64_t);
    for (auto *b : state_bufs(*r)) {
        if (b->n) VLM_HIP(hipMemcpy(b->p, p, b->n * sizeof(double), hipMemcpyHostToDevice));
        p += b->n * sizeof(double);
    }
    r->rowNear = (int)h[0];
    r->rowFar = (int)h[1];
    r->head = (int)h[2];
    r->presc_built[0] = (int)(h[3] & 1);
    r->presc_built[1] = (int)((h[3] >> 1) & 1);
    return VLM_OK;
}

int vlm_rotor_burst_wake(vlm_ctx *ctx, int ir, double skewLimit, double largeCoreRadius)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor") : VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    const int64_t F = r->d.nFwake - (r->rowFar - 1);
    if (r->d.nNwake <= 0 || F <= 0) return VLM_OK;
    hipLaunchKernelGGL(burst_kernel, dim3(nblk(F * r->d.nb)), dim3(256), 0, ctx->stream,
                       view(*r), skewLimit, largeCoreRadius);
    VLM_HIP(hipGetLastError());
    return VLM_OK;
}

int vlm_rotor_rollup(vlm_ctx *ctx, int ir)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor") : VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    if (r->d.nNwake <= 0) return VLM_OK;
    int fi = r->rowFar - 2;  // rowFarNext - 1, 0-based
    const int shift_far = r->d.nFwake > 0 && fi < 0;
    if (shift_far) fi = 0;
    hipLaunchKernelGGL(rollup_kernel, dim3(r->d.nb), dim3(256), 0, ctx->stream, view(*r),
                       r->d.rollupStart - 1, r->d.rollupEnd - 1, r->d.rollupMin,
                       r->d.suppressFwake, fi, shift_far);
    VLM_HIP(hipGetLastError());
    // logical row i+1 <- row i
    r->head = (r->head + r->d.nNwake - 1) % r->d.nNwake;
    return VLM_OK;
}

int vlm_rotor_convectwake(vlm_ctx *ctx, int ir, double dt, int wakeType)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor") : VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    if (wakeType != VLM_WAKE_C && wakeType != VLM_WAKE_P)
        return fail(ctx, VLM_ERR_ARG, "wakeType must be VLM_WAKE_C or VLM_WAKE_P");
    Advance p;
    p.convect = wakeType == VLM_WAKE_P;
    p.dt = dt;
    p.only = r;
    return advance(ctx, p);
}

int vlm_rotor_induced_velocity(vlm_ctx *ctx, int ir, int set, int64_t m, const double *p,
                               double *v, int accumulate)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor") : VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    if (set < VLM_SET_WING || set > VLM_SET_WAKE_PRED) return fail(ctx, VLM_ERR_ARG, "bad set");
    if (m <= 0) return VLM_OK;
    if (!p || !v) return fail(ctx, VLM_ERR_ARG, "null buffer");
    const Trim trim{ctx};
    Sources src = {{ir, set}};
    int64_t nest = 0;
    VLM_TRY(build_sources(ctx, src, bs_formats(ctx, m, expected(ctx, src)), &nest));
    VLM_HIP(ctx->tgt.reserve(ws_size<double>((size_t)3 * m)));
    VLM_HIP(ctx->out.reserve(ws_size<double>((size_t)3 * m)));
    VLM_TRY(points_to_device(ctx, m, p, ctx->tgt.p, m));
    if (accumulate) VLM_TRY(points_to_device(ctx, m, v, ctx->out.p, m));
    VLM_TRY(eval_sources(ctx, ctx->tgt.p, m, m, ctx->out.p, accumulate, nest));
    return points_to_host(ctx, m, ctx->out.p, m, v);
}

// The ordered term sum at m device targets (SoA, stride m) into out: with
// few targets TERM_MAX lists share four launches, otherwise each list gets
// its own.  A list of a few thousand segments is about 5 us per launch
// whatever the launch does: a step of four rotors, 32 lists of right-hand
// sides and 20 of loads, took 6194 us with four launches per list and takes
// 5370 us.  With many targets the pairs of one list fill the chip.
static int ordered_terms(vlm_ctx *ctx, int nterms, const int *ir, const int *set,
                         const int *flags, int64_t m, const double *tgt, double *out,
                         int accumulate)
{
    if (nterms == 0 && !accumulate) {
        hipLaunchKernelGGL(fill_kernel, dim3(nblk(3 * m)), dim3(256), 0, ctx->stream, out, 3 * m,
                           0.0);
        VLM_HIP(hipGetLastError());
    }
    int acc = accumulate;
    for (int k = 0; k < nterms;) {
        int fmt = 0, n = 0;
        std::vector<Sources> src;
        TermLists lists;
        for (; n < TERM_MAX && k + n < nterms; ++n) {
            const Sources s = {{ir[k + n], set[k + n]}};
            const int f = bs_formats(ctx, m, expected(ctx, s));
            if (n > 0 && (f != SEG_SOA || fmt != SEG_SOA)) break;
            fmt = f;
            src.push_back(s);
        }
        VLM_TRY(build_lists(ctx, src, fmt, &lists));
        for (int q = 0; q < n; ++q) lists.neg[q] = (flags[k + q] & VLM_TERM_NEGATE) != 0;
        if (fmt == SEG_SOA) {
            VLM_TRY(bs_eval_terms(ctx, ctx->seg_view, lists, tgt, m, m, out, acc));
        } else {
            if (lists.neg[0] && acc) {
                hipLaunchKernelGGL(negate_kernel, dim3(nblk(3 * m)), dim3(256), 0, ctx->stream,
                                   out, 3 * m);
                VLM_HIP(hipGetLastError());
            }
            VLM_TRY(bs_eval(ctx, ctx->seg_view, lists.est[0], tgt, m, m, out, acc));
        }
        acc = 1;
        k += n;
    }
    return VLM_OK;
}

static int induced_terms(vlm_ctx *ctx, int nterms, const int *ir, const int *set,
                         const int *flags, int64_t m, const double *p, double *v,
                         int accumulate, bool deferred)
{
    if (!ctx) return VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    if (nterms < 0 || (nterms > 0 && (!ir || !set || !flags)))
        return fail(ctx, VLM_ERR_ARG, "bad term list");
    for (int k = 0; k < nterms; ++k) {
        if (!get_rotor(ctx, ir[k])) return fail(ctx, VLM_ERR_ARG, "unknown rotor");
        if (set[k] < VLM_SET_WING || set[k] > VLM_SET_WAKE_PRED)
            return fail(ctx, VLM_ERR_ARG, "bad set");
    }
    if (m <= 0) return VLM_OK;
    if (!p || !v) return fail(ctx, VLM_ERR_ARG, "null buffer");
    const Trim trim{ctx};
    VLM_HIP(ctx->tgt.reserve(ws_size<double>((size_t)3 * m)));
    VLM_HIP(ctx->out.reserve(ws_size<double>((size_t)3 * m)));
    VLM_TRY(points_to_device(ctx, m, p, ctx->tgt.p, m));
    if (accumulate) VLM_TRY(points_to_device(ctx, m, v, ctx->out.p, m));
    VLM_TRY(ordered_terms(ctx, nterms, ir, set, flags, m, ctx->tgt.p, ctx->out.p, accumulate));
    return points_to_host(ctx, m, ctx->out.p, m, v, deferred);
}

}  // extern "C"

// The ordered term sum of induced_terms at m device targets (SoA, stride
// m) into a device SoA buffer out (overwritten): the right-hand side and
// the loads keep their collocation velocities on the device.
int vlm::induced_terms_soa(vlm_ctx *ctx, int nterms, const int *ir, const int *set,
                           const int *flags, int64_t m, const double *tgt, double *out)
{
    for (int k = 0; k < nterms; ++k) {
        if (!get_rotor(ctx, ir[k])) return fail(ctx, VLM_ERR_ARG, "unknown rotor");
        if (set[k] < VLM_SET_WING || set[k] > VLM_SET_WAKE_PRED)
            return fail(ctx, VLM_ERR_ARG, "bad set");
    }
    if (m <= 0) return VLM_OK;
    return ordered_terms(ctx, nterms, ir, set, flags, m, tgt, out, 0);
}

vlm::Rotor *vlm::rotor_of(vlm_ctx *ctx, int ir) { return get_rotor(ctx, ir); }

extern "C" {

int vlm_induced_velocity_terms(vlm_ctx *ctx, int nterms, const int *ir, const int *set,
                               const int *flags, int64_t m, const double *p, double *v,
                               int accumulate)
{
    return induced_terms(ctx, nterms, ir, set, flags, m, p, v, accumulate, false);
}

int vlm_induced_velocity_terms_deferred(vlm_ctx *ctx, int nterms, const int *ir,
                                        const int *set, const int *flags, int64_t m,
                                        const double *p, double *v, int accumulate)
{
    return induced_terms(ctx, nterms, ir, set, flags, m, p, v, accumulate, true);
}

int vlm_wake_velocity(vlm_ctx *ctx, int wakeType)
{
    if (!ctx) return VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    if (wakeType != VLM_WAKE_C && wakeType != VLM_WAKE_P)
        return fail(ctx, VLM_ERR_ARG, "wakeType must be VLM_WAKE_C or VLM_WAKE_P");
    Advance p;
    VLM_TRY(wake_pass(ctx, wakeType == VLM_WAKE_P, &p.m));
    p.slot = wakeType == VLM_WAKE_P ? VLM_VEL_PRED : VLM_VEL;
    p.scatter = true;
    return advance(ctx, p);
}

int vlm_convect(vlm_ctx *ctx, int scheme, int iter, double dt)
{
    if (!ctx) return VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    if (scheme < VLM_SCHEME_FT1 || scheme > VLM_SCHEME_AM4)
        return fail(ctx, VLM_ERR_ARG, "fdScheme must be 0..5");
    Advance p1, p2;
    VLM_TRY(wake_pass(ctx, 0, &p1.m));
    p1.scatter = p1.init = true;
    p1.iter = iter;
    p1.dt = dt;
    p1.convect = 0;
    // pass 1 alone: explicit schemes and start-up steps, which convect with
    // pass 1 and keep it as history.  AM3's first start-up branch tests
    // iter == 0, which the time loop never reaches (main.f90:1118), so its
    // step 1 runs the full scheme on the zero-initialised histories.
    bool start = true;
    if (scheme == VLM_SCHEME_AM3 && iter == 2) p1.op = ADV_KEEP2;
    else if (scheme == VLM_SCHEME_AM4 && iter >= 1 && iter <= 3) p1.op = ADV_KEEP1 + (iter - 1);
    else if ((scheme == VLM_SCHEME_AB2 || scheme == VLM_SCHEME_AM2) && iter == 1) p1.op = ADV_KEEP1;
    else if (scheme == VLM_SCHEME_AB2) p1.op = ADV_AB2;
    else start = scheme == VLM_SCHEME_FT1;
    if (start) return advance(ctx, p1);
    // predictor, then pass 2 on the predicted wake and the corrector
    p1.convect = 1;
    p1.copy = true;
    if (scheme == VLM_SCHEME_AM2) p1.op = ADV_AM2_PRED;
    if (scheme == VLM_SCHEME_AM3) p1.op = ADV_AM3_PRED;
    if (scheme == VLM_SCHEME_AM4) p1.op = ADV_AM4_PRED;
    VLM_TRY(advance(ctx, p1));
    if (scheme == VLM_SCHEME_AM2 && ctx->pred.mode == 1) VLM_TRY(learned_pass(ctx, &p2.m));
    else VLM_TRY(wake_pass(ctx, 1, &p2.m));
    p2.slot = VLM_VEL_PRED;
    p2.scatter = p2.init = true;
    p2.iter = iter;
    p2.dt = dt;
    p2.convect = 0;
    if (scheme == VLM_SCHEME_AM2) p2.op = ADV_AM2_CORR;
    if (scheme == VLM_SCHEME_AM3) p2.op = ADV_AM3_CORR;
    if (scheme == VLM_SCHEME_AM4) p2.op = ADV_AM4_CORR;
    if (scheme != VLM_SCHEME_PC2) return advance(ctx, p2);
    // PC2 averages the two passes over neighbouring rows before it convects
    p2.convect = -1;
    VLM_TRY(advance(ctx, p2));
    for (auto *r : ctx->rotors) {
        if (r->d.nNwake <= 0 || r->image_of >= 0) continue;
        const int rows = r->d.nNwake - (r->rowNear - 1);
        const int frows = r->d.nFwake - (r->rowFar - 1);
        const int nbc = r->d.nbConvect;
        if (rows > 0) {
            const int64_t n = (int64_t)nbc * rows * (r->d.ns + 1) * 3;
            hipLaunchKernelGGL(order2_kernel, dim3(nblk(n)), dim3(256), 0, ctx->stream,
                               r->velN[VLM_VEL].p, r->velN[VLM_VEL_PRED].p,
                               r->velN[VLM_VEL_STEP].p, nbc, rows, r->d.nNwake, r->d.ns + 1,
                               r->rowNear - 1);
            hipLaunchKernelGGL(copy_window_kernel, dim3(nblk(n)), dim3(256), 0, ctx->stream,
                               r->velN[VLM_VEL_STEP].p, r->velN[VLM_VEL].p, nbc, rows,
                               r->d.nNwake, r->d.ns + 1, r->rowNear - 1);
        }
        if (frows > 0) {
            const int64_t n = (int64_t)nbc * frows * 3;
            hipLaunchKernelGGL(order2_kernel, dim3(nblk(n)), dim3(256), 0, ctx->stream,
                               r->velF[VLM_VEL].p, r->velF[VLM_VEL_PRED].p,
                               r->velF[VLM_VEL_STEP].p, nbc, frows, r->d.nFwake, 1,
                               r->rowFar - 1);
            hipLaunchKernelGGL(copy_window_kernel, dim3(nblk(n)), dim3(256), 0, ctx->stream,
                               r->velF[VLM_VEL_STEP].p, r->velF[VLM_VEL].p, nbc, frows,
                               r->d.nFwake, 1, r->rowFar - 1);
        }
        VLM_HIP(hipGetLastError());
    }
    Advance p3;
    p3.convect = 0;
    p3.dt = dt;
    return advance(ctx, p3);
}

int vlm_rotor_set_image(vlm_ctx *ctx, int ir, int source, int imagePlane)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor") : VLM_ERR_ARG;
    Rotor *s = get_rotor(ctx, source);
    if (!s || source == ir) return fail(ctx, VLM_ERR_ARG, "bad source rotor of the image");
    if (imagePlane < 1 || imagePlane > 3) return fail(ctx, VLM_ERR_ARG, "imagePlane must be 1..3");
    if (s->image_of >= 0) return fail(ctx, VLM_ERR_ARG, "the source of an image is an image");
    for (auto *q : ctx->rotors)
        if (q->image_of == ir) return fail(ctx, VLM_ERR_ARG, "rotor is the source of an image");
    if (r->d.nb != s->d.nb || r->d.nc != s->d.nc || r->d.ns != s->d.ns ||
        r->d.nNwake != s->d.nNwake || r->d.nFwake != s->d.nFwake)
        return fail(ctx, VLM_ERR_ARG, "an image needs its source's nb, nc, ns, nNwake and nFwake");
    r->image_of = source;
    r->image_axis = imagePlane - 1;
    return VLM_OK;
}

int vlm_rotor_mirror_gamma(vlm_ctx *ctx, int ir)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor") : VLM_ERR_ARG;
    if (r->image_of < 0) return fail(ctx, VLM_ERR_STATE, "rotor is not an image (vlm_rotor_set_image)");
    VLM_DEVICE(ctx);
    const Rotor &s = *ctx->rotors[r->image_of];
    if (r->nring > 0) {
        hipLaunchKernelGGL(mirror_gamma_kernel, dim3(nblk(r->nring)), dim3(256), 0, ctx->stream,
                           s.wg.p, r->wg.p, r->nring);
        VLM_HIP(hipGetLastError());
    }
    return VLM_OK;
}

int vlm_rotor_mirror_wake(vlm_ctx *ctx, int ir, int wakeType)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor") : VLM_ERR_ARG;
    if (wakeType != VLM_WAKE_C && wakeType != VLM_WAKE_P && wakeType != VLM_WAKE_A)
        return fail(ctx, VLM_ERR_ARG, "wakeType must be VLM_WAKE_C, VLM_WAKE_P or VLM_WAKE_A");
    VLM_DEVICE(ctx);
    return mirror_wake(ctx, *r, wakeType == VLM_WAKE_A ? 2 : wakeType == VLM_WAKE_P ? 1 : 0);
}

int vlm_rotor_set_prescribed_wake(vlm_ctx *ctx, int ir, int prescWakeNt, int prescWakeGenNt,
                                  double deltaPsi)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor") : VLM_ERR_ARG;
    if (prescWakeNt < 0 || prescWakeGenNt < 0)
        return fail(ctx, VLM_ERR_ARG, "prescWakeNt and prescWakeGenNt must be >= 0");
    if (prescWakeNt > 0 && (r->d.nFwake < 1 || prescWakeGenNt >= r->d.nFwake))
        return fail(ctx, VLM_ERR_ARG,
                    "the prescribed far wake needs a far wake longer than prescWakeGenNt");
    r->presc_nt = prescWakeNt;
    r->presc_gen_nt = prescWakeGenNt;
    r->presc_dpsi = deltaPsi;
    return VLM_OK;
}

int vlm_rotor_get_prescribed_wake(vlm_ctx *ctx, int ir, int wakeType, double *fc, double *gam,
                                  double *rc, int *built)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor") : VLM_ERR_ARG;
    if (wakeType != 0 && wakeType != 1) return fail(ctx, VLM_ERR_ARG, "wakeType must be 0 or 1");
    VLM_DEVICE(ctx);
    VLM_TRY(sync_stream(ctx));
    const size_t nb = (size_t)r->d.nb;
    if (fc)
        VLM_HIP(hipMemcpy(fc, r->pf[wakeType].p, 6 * nb * PF_N * sizeof(double),
                          hipMemcpyDeviceToHost));
    if (gam || rc) {
        std::vector<double> S(4 * nb);
        VLM_HIP(hipMemcpy(S.data(), r->ps[wakeType].p, 4 * nb * sizeof(double),
                          hipMemcpyDeviceToHost));
        for (size_t b = 0; b < nb; ++b)
            for (int i = 0; i < PF_N; ++i) {
                if (gam) gam[b * PF_N + i] = S[4 * b];
                if (rc) rc[b * PF_N + i] = S[4 * b + 1];
            }
    }
    if (built) *built = r->presc_built[wakeType];
    return VLM_OK;
}

int vlm_rotor_get_wake(vlm_ctx *ctx, int ir, int wakeType, double *nodes, double *le,
                       double *gam, double *rc4, double *far_fc, double *far_gam, double *far_rc)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor") : VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    const int pred = wakeType == VLM_WAKE_P;
    const int64_t nb = r->d.nb, nN = r->d.nNwake, ns = r->d.ns, nF = r->d.nFwake;
    // Seven copies from device to unpinned memory and a reordering of the
    // near rows on the host took 130 us for 0.1 MB; the rows are put in order
    // by one kernel into pinned memory instead, in pieces of its arena.
    const double *src[7] = {pred ? r->pnode.p : r->node.p, pred ? r->ple.p : r->le.p, r->gam.p,
                            r->rc4.p, pred ? r->pffc.p : r->ffc.p, r->fgam.p, r->frc.p};
    const int64_t rows[7] = {3 * (ns + 1), 0, ns, 4 * ns, 0, 0, 0};
    const int64_t len[7] = {nb * nN * rows[0], nN > 0 ? 3 * nb * (ns + 1) : 0, nb * nN * rows[2],
                            nb * nN * rows[3], 6 * nb * nF, nb * nF, nb * nF};
    double *dst[7] = {nodes, le, gam, rc4, far_fc, far_gam, far_rc};
    WakePack a;
    int64_t total = 0;
    for (int q = 0; q < 7; ++q) {
        total += dst[q] && len[q] > 0 ? len[q] : 0;
        a.end[q] = total;
        a.src[q] = src[q];
        a.row[q] = (int)rows[q];
    }
    a.nN = (int)nN;
    a.head = r->head;
    VLM_TRY(sync_stream(ctx));
    constexpr int64_t kPiece = 1 << 19;   // doubles: half of the arena's 8 MB
    for (a.c0 = 0; a.c0 < total; a.c0 += a.n) {
        a.n = std::min(kPiece, total - a.c0);
        char *p = nullptr;
        VLM_TRY(pin_take(ctx, sizeof(double) * a.n, &p));
        a.dst = reinterpret_cast<double *>(p);
        hipLaunchKernelGGL(wake_pack_kernel, dim3(nblk(a.n)), dim3(256), 0, ctx->stream, a);
        VLM_HIP(hipGetLastError());
        VLM_TRY(sync_stream(ctx));
        for (int q = 0; q < 7; ++q) {
            const int64_t s0 = q > 0 ? a.end[q - 1] : 0;
            const int64_t lo = std::max(s0, a.c0), hi = std::min(a.end[q], a.c0 + a.n);
            if (lo < hi)
                std::memcpy(dst[q] + (lo - s0), a.dst + (lo - a.c0), sizeof(double) * (hi - lo));
        }
    }
    return VLM_OK;
}

int vlm_rotor_set_wake(vlm_ctx *ctx, int ir, const double *nodes, const double *le,
                       const double *gam, const double *rc4, const double *far_fc,
                       const double *far_gam, const double *far_rc, int rowNear, int rowFar)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor") : VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    const size_t nb = r->d.nb, nN = r->d.nNwake, ns = r->d.ns, nF = r->d.nFwake;
    if (rowNear < 1 || rowNear > (int)nN + 1 || rowFar < 1 || rowFar > (int)nF + 1)
        return fail(ctx, VLM_ERR_ARG, "cursor out of range");
    if (nN > 0 && (!nodes || !le || !gam || !rc4)) return fail(ctx, VLM_ERR_ARG, "null buffer");
    if (nF > 0 && (!far_fc || !far_gam || !far_rc)) return fail(ctx, VLM_ERR_ARG, "null buffer");
    VLM_TRY(sync_stream(ctx));
    r->head = 0;
    r->rowNear = rowNear;
    r->rowFar = rowFar;
    if (nN > 0) {
        std::vector<double> age(nb * nN * ns, 0.0);
        VLM_HIP(hipMemcpy(r->node.p, nodes, 3 * nb * nN * (ns + 1) * sizeof(double),
                          hipMemcpyHostToDevice));
        VLM_HIP(hipMemcpy(r->le.p, le, 3 * nb * (ns + 1) * sizeof(double), hipMemcpyHostToDevice));
        VLM_HIP(hipMemcpy(r->gam.p, gam, nb * nN * ns * sizeof(double), hipMemcpyHostToDevice));
        VLM_HIP(hipMemcpy(r->rc4.p, rc4, 4 * nb * nN * ns * sizeof(double), hipMemcpyHostToDevice));
        VLM_HIP(hipMemcpy(r->age.p, age.data(), age.size() * sizeof(double), hipMemcpyHostToDevice));
    }
    if (nF > 0) {
        std::vector<double> l(nb * nF), z(nb * nF, 0.0);
        for (size_t k = 0; k < nb * nF; ++k) {
            const double *f = far_fc + 6 * k;
            const double dx = f[0] - f[3], dy = f[1] - f[4], dz = f[2] - f[5];
            l[k] = std::sqrt(dx * dx + dy * dy + dz * dz);
        }
        VLM_HIP(hipMemcpy(r->ffc.p, far_fc, 6 * nb * nF * sizeof(double), hipMemcpyHostToDevice));
        VLM_HIP(hipMemcpy(r->fgam.p, far_gam, nb * nF * sizeof(double), hipMemcpyHostToDevice));
        VLM_HIP(hipMemcpy(r->frc.p, far_rc, nb * nF * sizeof(double), hipMemcpyHostToDevice));
        VLM_HIP(hipMemcpy(r->frc0.p, far_rc, nb * nF * sizeof(double), hipMemcpyHostToDevice));
        VLM_HIP(hipMemcpy(r->fl0.p, l.data(), nb * nF * sizeof(double), hipMemcpyHostToDevice));
        VLM_HIP(hipMemcpy(r->flc.p, l.data(), nb * nF * sizeof(double), hipMemcpyHostToDevice));
        VLM_HIP(hipMemcpy(r->fage.p, z.data(), nb * nF * sizeof(double), hipMemcpyHostToDevice));
    }
    return VLM_OK;
}

int vlm_rotor_get_velocity(vlm_ctx *ctx, int ir, int which, double *velN, double *velF)
{
    Rotor *r = get_rotor(ctx, ir);
    if (!r) return ctx ? fail(ctx, VLM_ERR_ARG, "unknown rotor") : VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    if (which < VLM_VEL || which > VLM_VEL_STEP) return fail(ctx, VLM_ERR_ARG, "bad which");
    VLM_TRY(sync_stream(ctx));
    if (velN && r->nvn() > 0)
        VLM_HIP(hipMemcpy(velN, r->velN[which].p, r->nvn() * sizeof(double), hipMemcpyDeviceToHost));
    if (velF && r->nvf() > 0)
        VLM_HIP(hipMemcpy(velF, r->velF[which].p, r->nvf() * sizeof(double), hipMemcpyDeviceToHost));
    return VLM_OK;
}

}  // extern "C"

extern "C" {

int vlm_predictor_errors(vlm_ctx *ctx, double *mlp_rel_rms, double *base_rel_rms,
                         int64_t *judged_steps)
{
    if (!ctx) return VLM_ERR_ARG;
    const Predictor &P = ctx->pred;
    const double r = P.sum_ref2 > 0 ? P.sum_ref2 : 1.0;
    if (mlp_rel_rms) *mlp_rel_rms = std::sqrt(P.sum_err2 / r);
    if (base_rel_rms) *base_rel_rms = std::sqrt(P.sum_base2 / r);
    if (judged_steps) *judged_steps = P.judged;
    return VLM_OK;
}

int vlm_set_predictor(vlm_ctx *ctx, int mode, double tol, int sample_stride, int warmup_steps,
                      int train_iters, double lref)
{
    if (!ctx) return VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    if (mode != 0 && mode != 1) return fail(ctx, VLM_ERR_ARG, "predictor mode must be 0 or 1");
    if (sample_stride < 1 || warmup_steps < 0 || train_iters < 0 || !(lref > 0) || !(tol > 0))
        return fail(ctx, VLM_ERR_ARG, "bad predictor settings");
    Predictor &P = ctx->pred;
    P.mode = mode;
    P.tol = tol;
    P.stride = sample_stride;
    P.warmup = warmup_steps;
    P.train_iters = train_iters;
    P.lref = lref;
    P.sum_err2 = P.sum_base2 = P.sum_ref2 = 0.0;
    P.judged = 0;
    return VLM_OK;
}

int vlm_predictor_stats(vlm_ctx *ctx, int64_t *full, int64_t *learned, int64_t *fallbacks,
                        double *last_err, double *last_loss)
{
    if (!ctx) return VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    Predictor &P = ctx->pred;
    if (full) *full = P.full;
    if (learned) *learned = P.learned;
    if (fallbacks) *fallbacks = P.fallbacks;
    if (last_err) *last_err = P.last_err;
    if (last_loss) {
        float l = 0.f;
        VLM_TRY(mlp_read_loss(ctx, &l));
        *last_loss = l;
    }
    return VLM_OK;
}

}  // extern "C"
