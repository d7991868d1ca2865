// Context, error handling, segment compaction, explicit filament sets and
// kernel timing for libvlm.
#include <algorithm>
#include <cstring>

#include "vlm_internal.h"

namespace vlm {

int fail(vlm_ctx *ctx, int code, const std::string &msg)
{
    if (ctx) ctx->err = msg;
    return code;
}

int hip_fail(vlm_ctx *ctx, hipError_t e, const char *what)
{
    std::string m = std::string(what) + ": " + hipGetErrorString(e);
    return fail(ctx, e == hipErrorOutOfMemory ? VLM_ERR_ALLOC : VLM_ERR_HIP, m);
}

namespace {

unsigned nblk(int64_t n) { return (unsigned)((n + 255) / 256); }

constexpr size_t CALL_BYTES = (size_t)4 << 20;

// Records of an explicit list (every filament kept, at its own index), one
// lane per segment of the padded list, and its count.
__device__ void explicit_record(int64_t n, int64_t k, const double *a, const double *b, double g,
                                double rc, const SegPtrs &L)
{
    if (k == 0) *L.count = (long long)n;
    if ((k & ~(int64_t)(GRP - 1)) >= n) return;   // whole groups leave together
    Slot s;
    s.ax = a[0];
    s.ay = a[1];
    s.az = a[2];
    s.bx = b[0];
    s.by = b[1];
    s.bz = b[2];
    s.gam = g;
    s.rc = rc;
    write_group_records(s, k < n, k, L);
}

__global__ __launch_bounds__(256) void explicit_records_kernel(int64_t n, const double *a,
                                                               const double *b, const double *g,
                                                               const double *rc, SegPtrs L)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t i = k < n ? k : n - 1;
    if (n > 0) explicit_record(n, k, a + 3 * i, b + 3 * i, g[i], rc[i], L);
    else if (k == 0) *L.count = 0;
}

// 256 points of a host list (xyz per point) on their way to LDS, so that
// reads of pinned memory are whole lines; the loads issue together (a round
// trip to the host takes some 2 us).
struct Triples {
    double x[3];
    __device__ Triples(const double *p, int64_t i0, int64_t m)
    {
#pragma unroll
        for (int q = 0; q < 3; ++q) x[q] = p[min(3 * i0 + q * 256 + threadIdx.x, 3 * m - 1)];
    }
    __device__ void put(double *sh) const
    {
#pragma unroll
        for (int q = 0; q < 3; ++q) sh[q * 256 + threadIdx.x] = x[q];
    }
};

__device__ void points_block(const double *p, int64_t blk, int64_t m, double *soa, int64_t stride,
                             double *sh)
{
    const int64_t i0 = blk * 256, i = i0 + threadIdx.x;
    const Triples t(p, i0, m);
    t.put(sh);
    __syncthreads();
    if (i >= m) return;
    for (int d = 0; d < 3; ++d) soa[d * stride + i] = sh[3 * threadIdx.x + d];
}

// xyz per point -> SoA
__global__ __launch_bounds__(256) void aos_to_soa_kernel(int64_t m, const double *aos,
                                                         double *soa, int64_t stride)
{
    __shared__ double sh[768];
    points_block(aos, blockIdx.x, m, soa, stride, sh);
}

// SoA -> xyz per point
__global__ __launch_bounds__(256) void soa_to_aos_kernel(int64_t m, const double *soa,
                                                         int64_t stride, double *aos)
{
    __shared__ double sh[768];
    const int64_t i0 = (int64_t)blockIdx.x * 256, i = i0 + threadIdx.x;
    if (i < m)
        for (int d = 0; d < 3; ++d) sh[3 * threadIdx.x + d] = soa[d * stride + i];
    __syncthreads();
    const int64_t left = 3 * (m - i0);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const int e = q * 256 + threadIdx.x;
        if (e < left) aos[3 * i0 + e] = sh[e];
    }
}

// The filaments (a | b | circulations | radii) and points of one call, in
// pinned memory, as records and SoA targets: blocks below fblocks take 256
// filaments each.
__global__ __launch_bounds__(256) void call_inputs_kernel(const double *h, int64_t n, SegPtrs L,
                                                          int fblocks, const double *p, int64_t m,
                                                          double *t)
{
    __shared__ double sa[768], sb[768];
    if ((int)blockIdx.x >= fblocks) {
        points_block(p, (int)blockIdx.x - fblocks, m, t, m, sa);
        return;
    }
    const int64_t i0 = (int64_t)blockIdx.x * 256, k = i0 + threadIdx.x;
    const int64_t i = k < n ? k : n - 1;
    const Triples a(h, i0, n), b(h + 3 * n, i0, n);
    const double g = h[6 * n + i], rc = h[7 * n + i];
    a.put(sa);
    b.put(sb);
    __syncthreads();
    explicit_record(n, k, sa + 3 * (i - i0), sb + 3 * (i - i0), g, rc, L);
}

}  // namespace

int explicit_records(vlm_ctx *ctx, int64_t n, const double *a, const double *b, const double *g,
                     const double *rc, const SegPtrs &L)
{
    hipLaunchKernelGGL(explicit_records_kernel, dim3(n > 0 ? nblk(n) : 1), dim3(256), 0,
                       ctx->stream, n, a, b, g, rc, L);
    VLM_HIP(hipGetLastError());
    return VLM_OK;
}

namespace {

int upload_fset(vlm_ctx *ctx, int64_t nfil, const double *a, const double *b,
                const double *gam, const double *rc, int formats, SegList &seg, SegPtrs *view)
{
    VLM_HIP(ctx->hostio.reserve((size_t)8 * nfil));
    double *raw = ctx->hostio.p;
    VLM_TRY(h2d(ctx, raw, a, sizeof(double) * 3 * nfil));
    VLM_TRY(h2d(ctx, raw + 3 * nfil, b, sizeof(double) * 3 * nfil));
    VLM_TRY(h2d(ctx, raw + 6 * nfil, gam, sizeof(double) * nfil));
    VLM_TRY(h2d(ctx, raw + 7 * nfil, rc, sizeof(double) * nfil));
    VLM_HIP(seg.reserve(nfil, formats, view));
    return explicit_records(ctx, nfil, raw, raw + 3 * nfil, raw + 6 * nfil, raw + 7 * nfil, *view);
}

}  // namespace

static void flush_deferred(vlm_ctx *ctx)
{
    for (const auto &d : ctx->deferred) std::memcpy(d.dst, d.src, d.bytes);
    ctx->deferred.clear();
}

int sync_stream(vlm_ctx *ctx)
{
    VLM_HIP(hipStreamSynchronize(ctx->stream));
    flush_deferred(ctx);
    ctx->pin_off = 0;
    return VLM_OK;
}

int defer(vlm_ctx *ctx, std::initializer_list<vlm_ctx::Deferred> d)
{
    if (!ctx->defer_ev) VLM_HIP(hipEventCreateWithFlags(&ctx->defer_ev, hipEventDisableTiming));
    VLM_HIP(hipEventRecord(ctx->defer_ev, ctx->stream));
    ctx->deferred.insert(ctx->deferred.end(), d);
    return VLM_OK;
}

int d2h_deferred(vlm_ctx *ctx, void *dst, const void *src, size_t bytes)
{
    if (bytes == 0) return VLM_OK;
    char *p = nullptr;
    VLM_TRY(pin_take(ctx, bytes, &p));
    VLM_HIP(hipMemcpyAsync(p, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
    return defer(ctx, {{dst, p, bytes}});
}

// Waits only for the work enqueued up to the last deferred copy; the arena
// is not recycled here because later work on the stream may still use it.
int wait_deferred(vlm_ctx *ctx)
{
    if (ctx->deferred.empty()) return VLM_OK;
    VLM_HIP(hipEventSynchronize(ctx->defer_ev));
    flush_deferred(ctx);
    return VLM_OK;
}

// Reserve bytes of the pinned arena (64-byte aligned), synchronising and
// recycling it when full, growing it when a request exceeds its size.
int pin_take(vlm_ctx *ctx, size_t bytes, char **out)
{
    const size_t need = (bytes + 63) & ~(size_t)63;
    if (ctx->pin_off + need > ctx->pin_cap) {
        VLM_TRY(sync_stream(ctx));
        if (need > ctx->pin_cap) {
            if (ctx->pin) VLM_HIP(hipHostFree(ctx->pin));
            ctx->pin = nullptr;
            ctx->pin_cap = 0;
            size_t cap = need > ((size_t)8 << 20) ? need : ((size_t)8 << 20);
            VLM_HIP(hipHostMalloc(reinterpret_cast<void **>(&ctx->pin), cap,
                                  hipHostMallocDefault));
            ctx->pin_cap = cap;
        }
    }
    *out = ctx->pin + ctx->pin_off;
    ctx->pin_off += need;
    return VLM_OK;
}

Trim::~Trim()
{
    for (auto *b : {&ctx->hostio, &ctx->tgt, &ctx->out})
        if (b->n * sizeof(double) > KEEP_BYTES) b->release();
    // (wake passes have partial sums of up to 400 MB)
    if (ctx->part.n * sizeof(double) > 4 * KEEP_BYTES) ctx->part.release();
    if (ctx->seg.bytes() > KEEP_BYTES) {
        ctx->seg.release();
        ctx->seg_view = SegPtrs();
    }
}

static int piece_event(vlm_ctx *ctx, int slot)
{
    if (!ctx->io_ev[slot])
        VLM_HIP(hipEventCreateWithFlags(&ctx->io_ev[slot], hipEventDisableTiming));
    VLM_HIP(hipEventRecord(ctx->io_ev[slot], ctx->stream));
    return VLM_OK;
}

int h2d(vlm_ctx *ctx, void *dst, const void *src, size_t bytes)
{
    if (bytes == 0) return VLM_OK;
    char *p = nullptr;
    const size_t piece = bytes < PIN_PIECE ? bytes : PIN_PIECE;
    VLM_TRY(pin_take(ctx, bytes <= piece ? bytes : 2 * piece, &p));
    int k = 0;
    for (size_t o = 0; o < bytes; o += piece, ++k) {
        const size_t n = std::min(piece, bytes - o);
        char *q = p + (k & 1) * piece;
        if (k >= 2) VLM_HIP(hipEventSynchronize(ctx->io_ev[k & 1]));
        std::memcpy(q, (const char *)src + o, n);
        VLM_HIP(hipMemcpyAsync((char *)dst + o, q, n, hipMemcpyHostToDevice, ctx->stream));
        if (bytes > piece) VLM_TRY(piece_event(ctx, k & 1));
    }
    return VLM_OK;
}

int d2h(vlm_ctx *ctx, void *dst, const void *src, size_t bytes)
{
    if (bytes == 0) return sync_stream(ctx);
    char *p = nullptr;
    const size_t piece = bytes < PIN_PIECE ? bytes : PIN_PIECE;
    VLM_TRY(pin_take(ctx, bytes <= piece ? bytes : 2 * piece, &p));
    if (bytes <= piece) {
        VLM_HIP(hipMemcpyAsync(p, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
        VLM_TRY(sync_stream(ctx));
        std::memcpy(dst, p, bytes);
        return VLM_OK;
    }
    const size_t np = (bytes + piece - 1) / piece;
    for (size_t k = 0; k <= np; ++k) {
        if (k < np) {
            VLM_HIP(hipMemcpyAsync(p + (k & 1) * piece, (const char *)src + k * piece,
                                   std::min(piece, bytes - k * piece), hipMemcpyDeviceToHost,
                                   ctx->stream));
            VLM_TRY(piece_event(ctx, k & 1));
        }
        if (k > 0) {
            VLM_HIP(hipEventSynchronize(ctx->io_ev[(k - 1) & 1]));
            std::memcpy((char *)dst + (k - 1) * piece, p + ((k - 1) & 1) * piece,
                        std::min(piece, bytes - (k - 1) * piece));
        }
    }
    return sync_stream(ctx);
}

// Points of a piece: whole workgroups, and whole 64-byte lines.
constexpr int64_t PIECE_POINTS = (int64_t)(PIN_PIECE / (3 * sizeof(double))) / 256 * 256;

int points_to_device(vlm_ctx *ctx, int64_t m, const double *p, double *soa, int64_t stride)
{
    const int64_t piece = std::min(m, PIECE_POINTS);
    char *hp = nullptr;
    VLM_TRY(pin_take(ctx, sizeof(double) * 3 * (m > piece ? 2 * piece : m), &hp));
    for (int64_t k = 0, i = 0; i < m; ++k, i += piece) {
        const int64_t n = std::min(piece, m - i);
        double *h = reinterpret_cast<double *>(hp) + (k & 1) * 3 * piece;
        if (k >= 2) VLM_HIP(hipEventSynchronize(ctx->io_ev[k & 1]));
        std::memcpy(h, p + 3 * i, sizeof(double) * 3 * n);
        hipLaunchKernelGGL(aos_to_soa_kernel, dim3(nblk(n)), dim3(256), 0, ctx->stream, n, h,
                           soa + i, stride);
        VLM_HIP(hipGetLastError());
        if (m > piece) VLM_TRY(piece_event(ctx, k & 1));
    }
    return VLM_OK;
}

int points_to_host(vlm_ctx *ctx, int64_t m, const double *soa, int64_t stride, double *p,
                   bool deferred = false)
{
    // a deferred result waits in the arena as a whole
    const int64_t piece = deferred ? m : std::min(m, PIECE_POINTS);
    const int64_t np = m > 0 ? (m + piece - 1) / piece : 0;
    char *hp = nullptr;
    VLM_TRY(pin_take(ctx, sizeof(double) * 3 * (m > piece ? 2 * piece : m), &hp));
    double *h = reinterpret_cast<double *>(hp);
    for (int64_t k = 0; k <= np; ++k) {
        if (k < np) {
            const int64_t n = std::min(piece, m - k * piece);
            hipLaunchKernelGGL(soa_to_aos_kernel, dim3(nblk(n)), dim3(256), 0, ctx->stream, n,
                               soa + k * piece, stride, h + (k & 1) * 3 * piece);
            VLM_HIP(hipGetLastError());
            if (deferred) return defer(ctx, {{p, hp, sizeof(double) * 3 * m}});
            if (np > 1) VLM_TRY(piece_event(ctx, k & 1));
        }
        if (k > 0) {
            if (np > 1) VLM_HIP(hipEventSynchronize(ctx->io_ev[(k - 1) & 1]));
            else VLM_TRY(sync_stream(ctx));
            std::memcpy(p + 3 * (k - 1) * piece, h + ((k - 1) & 1) * 3 * piece,
                        sizeof(double) * 3 * std::min(piece, m - (k - 1) * piece));
        }
    }
    return np > 1 ? sync_stream(ctx) : VLM_OK;
}

}  // namespace vlm

using namespace vlm;

extern "C" {

int vlm_create(vlm_ctx **out, int device)
{
    if (!out) return VLM_ERR_ARG;
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return VLM_ERR_HIP;
    if (device < 0 || device >= ndev) return VLM_ERR_ARG;
    if (hipSetDevice(device) != hipSuccess) return VLM_ERR_HIP;
    vlm_ctx *ctx = new vlm_ctx();
    ctx->device = device;
    if (hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking) != hipSuccess) {
        delete ctx;
        return VLM_ERR_HIP;
    }
    ctx->prof_cap = 1 << 16;
    if (hipHostMalloc(reinterpret_cast<void **>(&ctx->prof_nseg),
                      ctx->prof_cap * sizeof(long long), hipHostMallocDefault) != hipSuccess) {
        ctx->prof_nseg = nullptr;
        ctx->prof_cap = 0;
    }
    *out = ctx;
    return VLM_OK;
}

int vlm_destroy(vlm_ctx *ctx)
{
    if (!ctx) return VLM_OK;
    (void)hipSetDevice(ctx->device);
    (void)hipStreamSynchronize(ctx->stream);
    flush_deferred(ctx);
    mlp_release(ctx);
    for (auto *r : ctx->rotors) delete r;
    for (auto *f : ctx->fsets) delete f;
    for (auto *p : ctx->psets) delete p;
    for (auto *p : ctx->aic) (void)hipFree(p);
    for (auto *p : ctx->lu) (void)hipFree(p);
    for (auto *p : ctx->piv) (void)hipFree(p);
    for (auto *v : {&ctx->timers, &ctx->lu_timers})
        for (auto &t : *v) {
            if (t.a) (void)hipEventDestroy(t.a);
            if (t.b) (void)hipEventDestroy(t.b);
        }
    if (ctx->prof_nseg) (void)hipHostFree(ctx->prof_nseg);
    if (ctx->pin) (void)hipHostFree(ctx->pin);
    if (ctx->judge_ev) (void)hipEventDestroy(ctx->judge_ev);
    if (ctx->defer_ev) (void)hipEventDestroy(ctx->defer_ev);
    for (auto e : ctx->io_ev)
        if (e) (void)hipEventDestroy(e);
    if (ctx->judge_pin) (void)hipHostFree(ctx->judge_pin);
    (void)hipStreamDestroy(ctx->stream);
    delete ctx;
    return VLM_OK;
}

const char *vlm_last_error(const vlm_ctx *ctx)
{
    if (!ctx) return "null context";
    return ctx->err.c_str();
}

int vlm_set_precision(vlm_ctx *ctx, int precision)
{
    if (!ctx) return VLM_ERR_ARG;
    if (precision != VLM_FP64 && precision != VLM_MIXED)
        return fail(ctx, VLM_ERR_ARG, "precision must be VLM_FP64 or VLM_MIXED");
    ctx->precision = precision;
    return VLM_OK;
}

int vlm_set_bug_compat(vlm_ctx *ctx, int bug_compat)
{
    if (!ctx) return VLM_ERR_ARG;
    ctx->bug_compat = bug_compat ? 1 : 0;
    return VLM_OK;
}

int vlm_synchronize(vlm_ctx *ctx)
{
    if (!ctx) return VLM_ERR_ARG;
    VLM_TRY(sync_stream(ctx));
    return VLM_OK;
}

int vlm_wait(vlm_ctx *ctx)
{
    if (!ctx) return VLM_ERR_ARG;
    return wait_deferred(ctx);
}

int vlm_filament_vind(vlm_ctx *ctx, int64_t nfil, const double *a, const double *b,
                      const double *gam, const double *rc, int64_t m, const double *p,
                      double *v, int accumulate)
{
    if (!ctx) return VLM_ERR_ARG;
    if (nfil < 0 || m < 0) return fail(ctx, VLM_ERR_ARG, "negative size");
    if (m == 0) return VLM_OK;
    if (!p || !v || (nfil > 0 && (!a || !b || !gam || !rc)))
        return fail(ctx, VLM_ERR_ARG, "null buffer");
    VLM_HIP(hipSetDevice(ctx->device));
    const Trim trim{ctx};
    const int formats = bs_formats(ctx, m, nfil);
    VLM_HIP(ctx->tgt.reserve(ws_size<double>((size_t)3 * m)));
    VLM_HIP(ctx->seg.reserve(std::max<int64_t>(nfil, 4096), formats, &ctx->seg_view));
    // Inputs of up to CALL_BYTES are read, and the result is written, by
    // kernels in pinned memory: three launches and one wait (300 points,
    // 2000 filaments: 39 us a call, against 88 with allocations and four
    // copies).  Larger ones are copied first (a kernel that gathers them from the host loses what the
    // copy of one piece beside the host's copy of the next gains).
    const size_t fil = (size_t)8 * nfil, pts = (size_t)3 * m;
    if (sizeof(double) * (fil + 2 * pts) <= CALL_BYTES) {
        char *hp = nullptr;
        VLM_TRY(pin_take(ctx, sizeof(double) * (fil + 2 * pts), &hp));
        double *h = reinterpret_cast<double *>(hp), *ph = h + fil, *vh = ph + pts;
        if (nfil > 0) {
            std::memcpy(h, a, sizeof(double) * 3 * nfil);
            std::memcpy(h + 3 * nfil, b, sizeof(double) * 3 * nfil);
            std::memcpy(h + 6 * nfil, gam, sizeof(double) * nfil);
            std::memcpy(h + 7 * nfil, rc, sizeof(double) * nfil);
        }
        std::memcpy(ph, p, sizeof(double) * pts);
        if (accumulate) std::memcpy(vh, v, sizeof(double) * pts);
        const unsigned fb = nblk(nfil);
        hipLaunchKernelGGL(call_inputs_kernel, dim3(fb + nblk(m)), dim3(256), 0, ctx->stream, h,
                           nfil, ctx->seg_view, (int)fb, ph, m, ctx->tgt.p);
        VLM_HIP(hipGetLastError());
        VLM_TRY(bs_eval(ctx, ctx->seg_view, nfil, ctx->tgt.p, m, m, vh, accumulate, nullptr,
                        true));
        VLM_TRY(sync_stream(ctx));
        std::memcpy(v, vh, sizeof(double) * pts);
        return VLM_OK;
    }
    if (nfil > 0)
        VLM_TRY(upload_fset(ctx, nfil, a, b, gam, rc, formats, ctx->seg, &ctx->seg_view));
    VLM_HIP(ctx->out.reserve(ws_size<double>(pts)));
    VLM_TRY(points_to_device(ctx, m, p, ctx->tgt.p, m));
    if (accumulate) VLM_TRY(points_to_device(ctx, m, v, ctx->out.p, m));
    VLM_TRY(bs_eval(ctx, ctx->seg_view, nfil, ctx->tgt.p, m, m, ctx->out.p, accumulate));
    return points_to_host(ctx, m, ctx->out.p, m, v);
}

int vlm_fset_create(vlm_ctx *ctx, int64_t nfil, const double *a, const double *b,
                    const double *gam, const double *rc, int *fset)
{
    if (!ctx || !fset) return VLM_ERR_ARG;
    if (nfil <= 0 || !a || !b || !gam || !rc) return fail(ctx, VLM_ERR_ARG, "empty filament set");
    VLM_HIP(hipSetDevice(ctx->device));
    const Trim trim{ctx};
    FSet *fs = new FSet();
    int rc_ = upload_fset(ctx, nfil, a, b, gam, rc, SEG_ALL, fs->seg, &fs->view);
    if (rc_ != VLM_OK) {
        delete fs;
        return rc_;
    }
    fs->n = nfil;
    ctx->fsets.push_back(fs);
    *fset = (int)ctx->fsets.size() - 1;
    return VLM_OK;
}

int vlm_pset_create(vlm_ctx *ctx, int64_t m, const double *p, int *pset)
{
    if (!ctx || !pset) return VLM_ERR_ARG;
    if (m <= 0 || !p) return fail(ctx, VLM_ERR_ARG, "empty point set");
    VLM_HIP(hipSetDevice(ctx->device));
    PSet *ps = new PSet();
    if (ps->p.reserve((size_t)3 * m) != hipSuccess || ps->v.reserve((size_t)3 * m) != hipSuccess) {
        delete ps;
        return fail(ctx, VLM_ERR_ALLOC, "point set allocation failed");
    }
    ps->m = m;
    int rc_ = points_to_device(ctx, m, p, ps->p.p, m);
    if (rc_ != VLM_OK) {
        delete ps;
        return rc_;
    }
    ctx->psets.push_back(ps);
    *pset = (int)ctx->psets.size() - 1;
    return VLM_OK;
}

int vlm_fset_vind(vlm_ctx *ctx, int fset, int pset)
{
    if (!ctx) return VLM_ERR_ARG;
    if (fset < 0 || fset >= (int)ctx->fsets.size() || pset < 0 ||
        pset >= (int)ctx->psets.size())
        return fail(ctx, VLM_ERR_ARG, "unknown filament or point set");
    VLM_HIP(hipSetDevice(ctx->device));
    FSet *fs = ctx->fsets[fset];
    PSet *ps = ctx->psets[pset];
    return bs_eval(ctx, fs->view, fs->n, ps->p.p, ps->m, ps->m, ps->v.p, 0);
}

int vlm_pset_velocity(vlm_ctx *ctx, int pset, double *v)
{
    if (!ctx || !v) return VLM_ERR_ARG;
    if (pset < 0 || pset >= (int)ctx->psets.size())
        return fail(ctx, VLM_ERR_ARG, "unknown point set");
    VLM_HIP(hipSetDevice(ctx->device));
    PSet *ps = ctx->psets[pset];
    return points_to_host(ctx, ps->m, ps->v.p, ps->m, v);
}

int vlm_profile_enable(vlm_ctx *ctx, int enable)
{
    if (!ctx) return VLM_ERR_ARG;
    ctx->profile = enable ? 1 : 0;
    return VLM_OK;
}

int vlm_profile_reset(vlm_ctx *ctx)
{
    if (!ctx) return VLM_ERR_ARG;
    VLM_TRY(sync_stream(ctx));
    for (auto &t : ctx->timers) {
        if (t.a) (void)hipEventDestroy(t.a);
        if (t.b) (void)hipEventDestroy(t.b);
    }
    ctx->timers.clear();
    for (auto &t : ctx->lu_timers) {
        (void)hipEventDestroy(t.a);
        (void)hipEventDestroy(t.b);
    }
    ctx->lu_timers.clear();
    ctx->prof_ms = 0.0;
    ctx->prof_pairs = 0.0;
    ctx->prof_launches = 0;
    return VLM_OK;
}

int vlm_profile_get(vlm_ctx *ctx, double *bs_ms, int64_t *bs_launches, double *pairs)
{
    if (!ctx) return VLM_ERR_ARG;
    VLM_TRY(sync_stream(ctx));
    double ms = 0.0, pr = 0.0;
    int64_t n = 0;
    for (size_t i = 0; i < ctx->timers.size(); ++i) {
        if (ctx->timers[i].kind != 0) continue;
        float e = 0.f;
        VLM_HIP(hipEventElapsedTime(&e, ctx->timers[i].a, ctx->timers[i].b));
        ms += e;
        ++n;
        if (i < ctx->prof_cap && ctx->timers[i].pairs > 0)
            pr += ctx->timers[i].pairs * (double)ctx->prof_nseg[i];
    }
    if (bs_ms) *bs_ms = ms;
    if (bs_launches) *bs_launches = n;
    if (pairs) *pairs = pr;
    return VLM_OK;
}

int vlm_profile_get_all(vlm_ctx *ctx, double *pairs, int64_t *launches)
{
    if (!ctx) return VLM_ERR_ARG;
    VLM_TRY(sync_stream(ctx));
    double pr = 0.0;
    for (size_t i = 0; i < ctx->timers.size(); ++i)
        if (i < ctx->prof_cap && ctx->timers[i].pairs > 0)
            pr += ctx->timers[i].pairs * (double)ctx->prof_nseg[i];
    if (pairs) *pairs = pr;
    if (launches) *launches = (int64_t)ctx->timers.size();
    return VLM_OK;
}

int vlm_profile_get_lu(vlm_ctx *ctx, double *ms, int64_t *factorisations, double *flops)
{
    if (!ctx) return VLM_ERR_ARG;
    VLM_TRY(sync_stream(ctx));
    double t = 0.0, f = 0.0;
    for (auto &tm : ctx->lu_timers) {
        float e = 0.f;
        VLM_HIP(hipEventElapsedTime(&e, tm.a, tm.b));
        t += e;
        f += tm.pairs;
    }
    if (ms) *ms = t;
    if (factorisations) *factorisations = (int64_t)ctx->lu_timers.size();
    if (flops) *flops = f;
    return VLM_OK;
}

}  // extern "C"

// Calibration streams for vlm_fp64_issue_rate: every lane runs 8 independent
// chains of CALIB_ITERS dependent operations (FMA, or v_rsq_f64) and stores
// one value at its global index, so the output holds exactly one double per
// launched lane.
namespace {
constexpr int CALIB_ITERS = 4096;
constexpr int CALIB_CHAINS = 8;

__global__ void __launch_bounds__(256) calib_fma_kernel(double *out, double s)
{
    double a[CALIB_CHAINS];
    for (int c = 0; c < CALIB_CHAINS; ++c) a[c] = s + c + threadIdx.x * 1e-9;
    for (int i = 0; i < CALIB_ITERS; ++i)
#pragma unroll
        for (int c = 0; c < CALIB_CHAINS; ++c) a[c] = __builtin_fma(a[c], 0.999999, 1e-7);
    double t = 0.0;
    for (int c = 0; c < CALIB_CHAINS; ++c) t += a[c];
    out[blockIdx.x * blockDim.x + threadIdx.x] = t;
}

__global__ void __launch_bounds__(256) calib_rsq_kernel(double *out, double s)
{
    double a[CALIB_CHAINS];
    for (int c = 0; c < CALIB_CHAINS; ++c) a[c] = s + c + threadIdx.x * 1e-9;
    for (int i = 0; i < CALIB_ITERS; ++i)
#pragma unroll
        for (int c = 0; c < CALIB_CHAINS; ++c) a[c] = __builtin_amdgcn_rsq(a[c]);
    double t = 0.0;
    for (int c = 0; c < CALIB_CHAINS; ++c) t += a[c];
    out[blockIdx.x * blockDim.x + threadIdx.x] = t;
}
}  // namespace

extern "C" {

int vlm_fp64_issue_rate(vlm_ctx *ctx, double *fma_tflops, double *rsq_over_fma)
{
    if (!ctx || !fma_tflops || !rsq_over_fma) return VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    VLM_TRY(sync_stream(ctx));
    int cus = 0;
    VLM_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device));
    const int threads = 256, blocks = cus * 16;
    double *out = nullptr;
    hipEvent_t ev[3] = {nullptr, nullptr, nullptr};
    float ms_f = 0.f, ms_r = 0.f;
    hipError_t err = hipMalloc(&out, sizeof(double) * (size_t)blocks * threads);
    for (int i = 0; i < 3 && err == hipSuccess; ++i) err = hipEventCreate(&ev[i]);
    // the first round is untimed (clocks ramp up), the second is timed
    for (int round = 0; round < 2 && err == hipSuccess; ++round) {
        err = hipEventRecord(ev[0], ctx->stream);
        if (err != hipSuccess) break;
        hipLaunchKernelGGL(calib_fma_kernel, dim3(blocks), dim3(threads), 0, ctx->stream, out, 1.5);
        err = hipEventRecord(ev[1], ctx->stream);
        if (err != hipSuccess) break;
        hipLaunchKernelGGL(calib_rsq_kernel, dim3(blocks), dim3(threads), 0, ctx->stream, out, 1.5);
        err = hipEventRecord(ev[2], ctx->stream);
        if (err == hipSuccess) err = hipGetLastError();
        if (err == hipSuccess) err = hipEventSynchronize(ev[2]);
    }
    if (err == hipSuccess) err = hipEventElapsedTime(&ms_f, ev[0], ev[1]);
    if (err == hipSuccess) err = hipEventElapsedTime(&ms_r, ev[1], ev[2]);
    for (int i = 0; i < 3; ++i)
        if (ev[i]) (void)hipEventDestroy(ev[i]);
    if (out) (void)hipFree(out);
    if (err != hipSuccess) return vlm::hip_fail(ctx, err, "vlm_fp64_issue_rate");
    const double fmas = 64.0 * (double)blocks * (threads / 64) * CALIB_ITERS * CALIB_CHAINS;
    *fma_tflops = 2.0 * fmas / (ms_f * 1e-3) / 1e12;
    *rsq_over_fma = (double)ms_r / (double)ms_f;
    return VLM_OK;
}

}  // extern "C"
