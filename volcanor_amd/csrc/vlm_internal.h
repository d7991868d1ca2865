// Internal declarations of libvlm (MI355X free-wake hot path).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "vlm_c.h"

namespace vlm {

// Device buffer owned by the library.  reserve() grows and discards the
// contents; growth is geometric (at least doubling) because buffers sized
// by the wake grow every step and hipFree synchronises the device.
template <typename T>
struct DBuf {
    T *p = nullptr;
    size_t n = 0;
    DBuf() = default;
    DBuf(const DBuf &) = delete;
    DBuf &operator=(const DBuf &) = delete;
    ~DBuf() { release(); }
    void release()
    {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    hipError_t reserve(size_t k)
    {
        if (k <= n && p) return hipSuccess;
        size_t want = k == 0 ? 1 : k;
        if (p && want < 2 * n) want = 2 * n;
        release();
        hipError_t e = hipMalloc(reinterpret_cast<void **>(&p), want * sizeof(T));
        if (e == hipSuccess) n = want;
        else p = nullptr;
        return e;
    }
};

// Elements to reserve for a workspace that grows with a run: at least 256 kB,
// so that a short list grows it once and not at each doubling (hipFree waits
// for the device).
template <typename T>
inline size_t ws_size(size_t n)
{
    const size_t least = ((size_t)256 << 10) / sizeof(T);
    return n > least ? n : least;
}

// Compacted straight-segment list, in groups of GRP consecutive segments.
// Every segment has one record that a wave reads through the scalar cache
// (16 values = two or one s_load_dwordx16), so the records are arrays of
// structures:
//   rec64 (16 doubles): a(3) g | r0(3) n0 | g r0(3) qq | g r0 x (a - c)(3) -
//   rec32 (16 floats):  a - c(3) n0 | r0(3) qq | g r0(3) g | g r0 x (a - c)(3) q
//   near32 (8 floats):  a_hi(3) g | a_lo(3) q'   (a = a_hi + a_lo; q' = q, or
//                       infinity for q <= 1e-18)
//   grp (8 doubles per group): centre c, squared far radius, the squared
//                       distances up to which the far pair's c2 is accurate
//                       in FP64 and in FP32 (below), -, -
// Launches of few pairs put segments on lanes instead and read one
// structure of arrays (stride cap):
//   soa (9): ax ay az g | r0x r0y r0z qq | n0
// with g = gam / (4 pi), r0 = b - a, n0 = |r0|^2, q = rc^2 n0, qq = q^2 and
// c the centre of the group's bounding box.  The last group is padded with
// records of zero circulation and length that start where its last segment
// does (qq = 1): the distance to that point is positive wherever the group is
// far, so that they give 0 for every target.
// count: device int64 with the number of valid segments.
constexpr int GRP = 32;
constexpr int SOA_N = 9, REC64_N = 16, REC32_N = 16, NEAR32_N = 8, GRPH_N = 8;
// |r1| up to rc times these: see write_group_records.
constexpr double FAR_CORE64 = 16777216.0, FAR_CORE32 = 1024.0;   // 2^24, 2^10

// What a list holds; a launch with m targets needs bs_formats(m, its segments).
enum { SEG_SOA = 1, SEG_REC = 2, SEG_F32 = 4, SEG_ALL = 7 };

// Device pointers of a list (null where a format is absent).
struct SegPtrs {
    double *soa = nullptr, *rec64 = nullptr, *grp = nullptr;
    float *rec32 = nullptr, *near32 = nullptr;
    long long *count = nullptr;
    int64_t cap = 0;  // segments, a multiple of GRP (stride of soa)
};

struct SegList {
    DBuf<double> soa, rec64, grp;
    DBuf<float> rec32, near32;
    DBuf<long long> count;
    void release()
    {
        soa.release();
        rec64.release();
        grp.release();
        rec32.release();
        near32.release();
    }
    size_t bytes() const
    {
        return sizeof(double) * (soa.n + rec64.n + grp.n) + sizeof(float) * (rec32.n + near32.n);
    }
    // Room for n segments in the given formats.
    hipError_t reserve(int64_t n, int formats, SegPtrs *out)
    {
        const size_t k = (size_t)((n + GRP - 1) / GRP) * GRP;
        hipError_t e = count.reserve(16);
        if (e == hipSuccess && (formats & SEG_SOA)) e = soa.reserve(k * SOA_N);
        if (e == hipSuccess && (formats & SEG_REC)) e = rec64.reserve(k * REC64_N);
        if (e == hipSuccess && (formats & SEG_REC)) e = grp.reserve(k / GRP * GRPH_N);
        if (e == hipSuccess && (formats & SEG_F32)) e = rec32.reserve(k * REC32_N);
        if (e == hipSuccess && (formats & SEG_F32)) e = near32.reserve(k * NEAR32_N);
        out->soa = formats & SEG_SOA ? soa.p : nullptr;
        out->rec64 = formats & SEG_REC ? rec64.p : nullptr;
        out->grp = formats & SEG_REC ? grp.p : nullptr;
        out->rec32 = formats & SEG_F32 ? rec32.p : nullptr;
        out->near32 = formats & SEG_F32 ? near32.p : nullptr;
        out->count = count.p;
        out->cap = (int64_t)k;
        return e;
    }
};

// Staging slots written by the segment builders before compaction.
struct Slot {
    double ax, ay, az, bx, by, bz, gam, rc;
};


// velocity arrays per rotor: the four of include/vlm_c.h, then two more
// histories used only by AM3 and AM4
constexpr int VEL_H2 = 4, VEL_H3 = 5, NVEL = 6;

constexpr int PF_N = 240;  // prescribed far-wake filaments per blade (classdef.f90:225)

// Records of vlm_rotor_set_panels and vlm_rotor_loads (include/vlm_c.h).
constexpr int PANEL_N = 15, SECTION_N = 16, BLADE_N = 9, LOADS_SEC_N = 19, LOADS_ROTOR_N = 9;

struct Rotor {
    vlm_rotor_desc d{};
    int rowNear = 0, rowFar = 0;  // 1-based, as in the reference
    int head = 0;                 // physical slot of logical near-wake row 0
    double shaft[3] = {0, 0, 1}, hub[3] = {0, 0, 0};
    double init_wake_vel = 0.0;   // initWakeVel, applied while iter < init_wake_vel_nt
    int init_wake_vel_nt = 0;
    int nring = 0;                // nb*nc*ns wing rings
    // wing (uploaded by the host after every rigid motion)
    DBuf<double> wc, wrc, wg;     // 12*nring, 4*nring, nring
    // near wake, physical rows
    DBuf<double> node, pnode;     // 3*nb*nN*(ns+1)
    DBuf<double> le, ple;         // 3*nb*(ns+1)
    DBuf<double> gam, rc4, age;   // nb*nN*ns, 4*nb*nN*ns, nb*nN*ns
    // far wake
    DBuf<double> ffc, pffc;       // 6*nb*nF
    DBuf<double> fgam, frc, frc0, fl0, flc, fage;  // nb*nF
    // velocities, logical rows: [VLM_VEL, PREV, PRED, STEP] and the older
    // histories of AM3/AM4 (velNwake2, velNwake3; PREV is velNwake1)
    DBuf<double> velN[NVEL], velF[NVEL];
    // prescribed far wake, per wake type (0 current, 1 predicted): PF_N
    // filaments per blade, end points pf[6*(b*PF_N + i) + (0..2 TE, 3..5 LE)],
    // and per blade ps[4*b + (0 gam, 1 core radius, 2 helix pitch, 3 radius)]
    DBuf<double> pf[2], ps[2];
    int presc_nt = 0, presc_gen_nt = 0;  // 0: no prescribed far wake
    double presc_dpsi = 0.0;             // omegaSlow * dt
    int presc_built[2] = {0, 0};
    int iter = 0;                        // step of the last vlm_rotor_begin_step
    // image rotor: index of the rotor it mirrors (-1: a lifting rotor of its
    // own) and the coordinate negated by the mirror (0 x, 1 y, 2 z)
    int image_of = -1, image_axis = 0;
    // right-hand side and loads on the device (vlm_rotor_set_panels,
    // vlm_rotor_rhs, vlm_rotor_loads): panel, section and blade geometry
    // after the last rigid motion (PANEL_N, SECTION_N, BLADE_N doubles
    // each), collocation points SoA, velCP and velCPm (6 per panel), the
    // RHS, the load velocities (SoA), gamPrev (restart state) and the
    // packed load results
    DBuf<double> pan, sec, bla, cps, vcp, rhs, vld, gprev, lout;
    int panels_set = 0;
    size_t nvn() const { return 3u * d.nb * (size_t)d.nNwake * (d.ns + 1); }
    size_t nvf() const { return 3u * d.nb * (size_t)(d.nFwake > 0 ? d.nFwake : 0); }
};

// One profiled Biot-Savart launch: events around the grouped kernel (a, b;
// null for launches of few pairs, which are counted but not timed: bs_formats)
// and the target count; pairs = targets x the device segment count, which
// is copied to the pinned slot of the same index without a synchronisation.
struct Timer {
    hipEvent_t a, b;
    double pairs;
    int kind = 0;  // 0 grouped kernel (timed), 1 kernel of few pairs
};

struct Mlp;

// Learned pass-2 predictor settings, statistics and training buffer.
struct Predictor {
    int mode = 0;          // 0 full Biot-Savart pass 2, 1 learned
    double tol = 1e-4;     // judge tolerance: RMS error / RMS speed on the sample
    int stride = 32;       // judge sample: every stride-th target
    int warmup = 8;        // first AM2 steps always run the full pass
    int train_iters = 4;   // Adam iterations per step on the buffer
    float lr = 1e-3f;
    double lref = 1.0;     // length scale of the neighbour offsets
    int64_t batch = 2048;  // minibatch of each Adam iteration
    int64_t steps = 0, full = 0, learned = 0, fallbacks = 0, judged = 0, train_calls = 0;
    double last_err = 0.0;
    // accumulated over judged steps: squared error of the network, of the
    // network-free substitute, and squared exact speed
    double sum_err2 = 0.0, sum_base2 = 0.0, sum_ref2 = 0.0;
    int64_t buf_cap = 16384, buf_n = 0, buf_head = 0;
    DBuf<float> X, Y, bx, bt, tb;  // tb: minibatch targets in units of the buffer RMS
    DBuf<double> vn, ts, vs, e2, scal;
};

struct FSet {
    SegList seg;
    SegPtrs view;
    int64_t n = 0;
};

struct PSet {
    DBuf<double> p;   // SoA 3*m
    DBuf<double> v;   // SoA 3*m
    int64_t m = 0;
};

}  // namespace vlm

struct vlm_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    int precision = VLM_FP64;
    int bug_compat = 1;
    std::string err;
    std::vector<vlm::Rotor *> rotors;
    std::vector<vlm::FSet *> fsets;
    std::vector<vlm::PSet *> psets;
    // scratch
    vlm::SegList seg;
    vlm::SegPtrs seg_view;       // the list built last
    vlm::DBuf<vlm::Slot> slots;
    vlm::DBuf<int> seg_counts;   // segments of each staging block
    vlm::DBuf<double> tgt, out, part;
    vlm::DBuf<int> counter;  // work counter of the Biot-Savart launches, 0 between them
    int occ[2] = {0, 0};     // resident workgroups per kernel (FP64, mixed)
    vlm::DBuf<double> hostio;  // device copy of host filament lists and matrices
    vlm::DBuf<int> hostio_i;
    hipEvent_t io_ev[2] = {nullptr, nullptr};  // pieces of a copy in flight (h2d, d2h)
    // pinned host arena for host<->device copies: truly asynchronous copies,
    // reset whenever the stream has been synchronised
    char *pin = nullptr;
    size_t pin_cap = 0, pin_off = 0;
    // profiling
    int profile = 0;
    std::vector<vlm::Timer> timers;
    std::vector<vlm::Timer> lu_timers;  // LU factorisations (pairs = flops)
    double prof_ms = 0.0, prof_pairs = 0.0;
    long long *prof_nseg = nullptr;  // pinned, one slot per timed launch
    size_t prof_cap = 0;
    int64_t prof_launches = 0;
    // dense solve state per rotor (AIC, LU, pivots)
    std::vector<double *> aic, lu;
    std::vector<int *> piv;
    std::vector<int> aic_n;
    vlm::DBuf<double> solve_tmp;
    vlm::DBuf<int> lu_work;   // row-move lists of the blocked LU
    vlm::Mlp *mlp = nullptr;
    vlm::Predictor pred;
    hipEvent_t judge_ev = nullptr;  // learned pass: the judge sums reached judge_pin
    double *judge_pin = nullptr;    // pinned, 4 doubles
    // deferred downloads: device -> pinned arena copies already enqueued,
    // copied to the caller's buffers at vlm_wait or at any stream sync
    struct Deferred {
        void *dst;
        const char *src;
        size_t bytes;
    };
    std::vector<Deferred> deferred;
    hipEvent_t defer_ev = nullptr;  // recorded after the last deferred copy
};

namespace vlm {

int fail(vlm_ctx *ctx, int code, const std::string &msg);
int hip_fail(vlm_ctx *ctx, hipError_t e, const char *what);

#define VLM_HIP(call)                                          \
    do {                                                       \
        hipError_t e_ = (call);                                \
        if (e_ != hipSuccess) return vlm::hip_fail(ctx, e_, #call); \
    } while (0)

// Every entry point that touches the GPU makes the context's device current.
#define VLM_DEVICE(ctx) VLM_HIP(hipSetDevice((ctx)->device))

#define VLM_TRY(call)                 \
    do {                              \
        int rc_ = (call);             \
        if (rc_ != VLM_OK) return rc_; \
    } while (0)

constexpr double kPi = 3.141592653589793238462643383279502884;
constexpr double kInv4Pi = 0.25 / kPi;
constexpr double kEps = 2.220446049250313080847263336181640625e-16;  // epsilon(1._dp)

// Writes the records of one group's GRP consecutive segments: lane l of a
// 32-lane half wave (every lane active) holds segment k (the group's first
// plus l); lanes with valid = false hold the last valid segment and write the
// padding record (none in the structure of arrays).  The far radius: a target further than |a - c| + 2 |r0|
// from the centre, for every segment, has |r1| >= 2 |r0| for all of them.
// It is infinite (never far) for a group that holds a segment with
// q <= 1e-18 (the far pair has no zero-denominator guard) or an infinite
// circulation (the moments would turn it into NaN), or is wider than
// 64 of its longest segments (32 consecutive records can jump between wake
// rows; a chain of 32 connected segments spans 34), whose centred
// coordinates would lose accuracy against |r1|.
__device__ __forceinline__ void write_group_records(const Slot &s, bool valid, int64_t k,
                                                    const SegPtrs &L)
{
    const double r0x = s.bx - s.ax, r0y = s.by - s.ay, r0z = s.bz - s.az;
    const double g = s.gam * (0.25 / 3.141592653589793238462643383279502884);
    const double n0 = r0x * r0x + r0y * r0y + r0z * r0z;
    const double q = s.rc * s.rc * n0;
    if (L.soa && valid) {
        const double v[SOA_N] = {s.ax, s.ay, s.az, g, r0x, r0y, r0z, q * q, n0};
#pragma unroll
        for (int i = 0; i < SOA_N; ++i) L.soa[i * L.cap + k] = v[i];
    }
    if (!L.rec64) return;
    float lo[3], hi[3];
    const float inf = __builtin_inff();
    lo[0] = valid ? (float)fmin(s.ax, s.bx) : inf;
    lo[1] = valid ? (float)fmin(s.ay, s.by) : inf;
    lo[2] = valid ? (float)fmin(s.az, s.bz) : inf;
    hi[0] = valid ? (float)fmax(s.ax, s.bx) : -inf;
    hi[1] = valid ? (float)fmax(s.ay, s.by) : -inf;
    hi[2] = valid ? (float)fmax(s.az, s.bz) : -inf;
#pragma unroll
    for (int o = 16; o > 0; o >>= 1)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            lo[d] = fminf(lo[d], __shfl_xor(lo[d], o, 32));
            hi[d] = fmaxf(hi[d], __shfl_xor(hi[d], o, 32));
        }
    const double cx = 0.5 * ((double)lo[0] + hi[0]), cy = 0.5 * ((double)lo[1] + hi[1]),
                 cz = 0.5 * ((double)lo[2] + hi[2]);
    const double lx = s.ax - cx, ly = s.ay - cy, lz = s.az - cz;
    const double l2 = 2.0 * sqrt(n0);
    float ex = valid ? (float)((sqrt(lx * lx + ly * ly + lz * lz) + l2) * 1.000001) : 0.f;
    float lmax = valid ? (float)l2 : 0.f;
    float rmin = valid ? (float)(fabs(s.rc) * 0.999999) : inf;
    if (valid && !(q > 1e-18 && fabs(g) < __builtin_inf())) ex = inf;
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) {
        ex = fmaxf(ex, __shfl_xor(ex, o, 32));
        lmax = fmaxf(lmax, __shfl_xor(lmax, o, 32));
        rmin = fminf(rmin, __shfl_xor(rmin, o, 32));
    }
    if (!(ex <= 32.0f * lmax)) ex = inf;
    double v[REC64_N] = {s.ax, s.ay, s.az, g, r0x, r0y, r0z, n0, g * r0x, g * r0y, g * r0z, q * q,
                         g * (r0y * lz - r0z * ly), g * (r0z * lx - r0x * lz),
                         g * (r0x * ly - r0y * lx), 0.0};
    if (!valid)
        for (int i = 3; i < REC64_N; ++i) v[i] = i == 11 ? 1.0 : 0.0;
    double2 *o64 = reinterpret_cast<double2 *>(L.rec64 + (size_t)k * REC64_N);
#pragma unroll
    for (int i = 0; i < REC64_N / 2; ++i) o64[i] = make_double2(v[2 * i], v[2 * i + 1]);
    if ((k & (GRP - 1)) == 0) {
        double2 *h = reinterpret_cast<double2 *>(L.grp + (size_t)(k / GRP) * GRPH_N);
        h[0] = make_double2(cx, cy);
        h[1] = make_double2(cz, (double)ex * (double)ex);
        const double l64 = fmax(rmin * FAR_CORE64 - ex, 0.0), l32 = fmax(rmin * FAR_CORE32 - ex, 0.0);
        h[2] = make_double2(l64 * l64, l32 * l32);
    }
    if (!L.rec32) return;
    const float hx = (float)s.ax, hy = (float)s.ay, hz = (float)s.az, qf = (float)q;
    float4 *o32 = reinterpret_cast<float4 *>(L.rec32 + (size_t)k * REC32_N);
    float4 *on = reinterpret_cast<float4 *>(L.near32 + (size_t)k * NEAR32_N);
    if (valid) {
        o32[0] = make_float4((float)lx, (float)ly, (float)lz, (float)n0);
        o32[1] = make_float4((float)r0x, (float)r0y, (float)r0z, qf * qf);
        o32[2] = make_float4((float)v[8], (float)v[9], (float)v[10], (float)g);
        o32[3] = make_float4((float)v[12], (float)v[13], (float)v[14], qf);
        on[0] = make_float4(hx, hy, hz, (float)g);
        on[1] = make_float4((float)(s.ax - (double)hx), (float)(s.ay - (double)hy),
                            (float)(s.az - (double)hz), q > 1e-18 ? qf : inf);
    } else {
        const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
        o32[0] = o32[2] = on[0] = on[1] = z;
        o32[1] = make_float4(0.f, 0.f, 0.f, 1.f);
        o32[3] = make_float4(0.f, 0.f, 0.f, 1.f);
    }
}

// Biot-Savart evaluation of a compacted segment list at m targets stored
// as SoA (x at t[0..], y at t[tstride..], z at t[2*tstride..]).  Result
// goes to out (SoA of stride tstride, or with aos xyz per target, also in
// pinned host memory); accumulate adds into it.  nseg_est is the
// expected count (0: the list is empty): it sets the number of chunks, and
// the kernel divides the device count evenly among them.
// A fixed workspace for bs_eval instead of the context's growing buffers
// (no allocation): room for part_cap doubles of chunk partial sums (at
// least 3 m, the chunk count is capped by it) and one int counter, which is
// 0 before the call.  Such launches are not profiled.
struct BsWork {
    double *part;
    size_t part_cap;
    int *counter;
};
int bs_eval(vlm_ctx *ctx, const SegPtrs &seg, int64_t nseg_est, const double *t, int64_t m,
            int64_t tstride, double *out, int accumulate, const BsWork *ws = nullptr,
            bool aos = false);
// The list formats that a launch with m targets and (about) nseg segments
// reads.
int bs_formats(const vlm_ctx *ctx, int64_t m, int64_t nseg);

// Short work (bs_formats == SEG_SOA), up to TERM_MAX lists in one
// structure of arrays: list k starts at segment off[k] and has seg.count[k]
// segments (about est[k]).
//   u = accumulate ? out : 0;  for k: u = (neg[k] ? -u : u) + velocity of k;
//   out = u
constexpr int TERM_MAX = 16;
struct TermLists {
    int n = 0;
    int64_t off[TERM_MAX], est[TERM_MAX];
    int neg[TERM_MAX];
};
int bs_eval_terms(vlm_ctx *ctx, const SegPtrs &seg, const TermLists &terms, const double *t,
                  int64_t m, int64_t tstride, double *out, int accumulate,
                  const BsWork *ws = nullptr, bool aos = false);

// Records of an explicit list (every filament kept, at its own index) from
// 3 x n device arrays, and its count.
int explicit_records(vlm_ctx *ctx, int64_t n, const double *a, const double *b, const double *g,
                     const double *rc, const SegPtrs &L);

// Rotor ir of the context (nullptr when out of range).
Rotor *rotor_of(vlm_ctx *ctx, int ir);
// The ordered sum of source-set terms (vlm_induced_velocity_terms) at m
// device targets, SoA with stride m, into the device SoA buffer out.
int induced_terms_soa(vlm_ctx *ctx, int nterms, const int *ir, const int *set,
                      const int *flags, int64_t m, const double *tgt, double *out);
void mlp_release(vlm_ctx *ctx);

// Host<->device copies through the pinned arena (ctx->pin): h2d copies the
// host bytes into the arena and enqueues an asynchronous copy, so the
// caller's buffer is free on return without a stream synchronisation;
// sync_stream waits for the stream and recycles the arena; d2h enqueues the
// copy, synchronises and copies out of the arena.  Copies above PIN_PIECE
// go piece by piece, the host's copy of one piece beside the transfer of the
// other (38 MB: 1.4 ms from and 2.2 ms to unpinned memory, 1.3 ms so).
// Kernels may read and write the arena themselves, which spares a small
// call the copies' launches.
constexpr size_t PIN_PIECE = (size_t)2 << 20;
// What a call on host data leaves in the context for the next one (copies of
// its filaments, points, results and matrices, its segment list and partial
// sums) is given back above this size, buffer by buffer, when the call ends
// with or without an error (hipFree waits for the device).
constexpr size_t KEEP_BYTES = (size_t)256 << 20;
struct Trim {
    vlm_ctx *ctx;
    ~Trim();
};
int pin_take(vlm_ctx *ctx, size_t bytes, char **out);
int h2d(vlm_ctx *ctx, void *dst, const void *src, size_t bytes);
int d2h(vlm_ctx *ctx, void *dst, const void *src, size_t bytes);
int sync_stream(vlm_ctx *ctx);
// Deferred download: the copy is enqueued now, dst is written at
// wait_deferred or at the next sync_stream (whichever comes first).
int d2h_deferred(vlm_ctx *ctx, void *dst, const void *src, size_t bytes);
// The same for pinned memory (pin_take) that work already enqueued writes.
int defer(vlm_ctx *ctx, std::initializer_list<vlm_ctx::Deferred> d);
int wait_deferred(vlm_ctx *ctx);
int mlp_forward_dev(vlm_ctx *ctx, int64_t m, const float *X, float *Y);
// Training step on a batch in device or pinned memory; the loss goes to
// loss_pin (a pinned slot: the call then synchronises), or with keep_loss
// only to the device for mlp_read_loss.
int mlp_train_dev(vlm_ctx *ctx, int64_t m, const float *X, const float *T, int adam, float lr,
                  float *loss_pin, int keep_loss = 0);
int mlp_read_loss(vlm_ctx *ctx, float *loss);

}  // namespace vlm
