// vlm_filament_vind_noalloc: the filament sum of vlm_filament_vind on
// device-resident inputs, for callers that cannot allocate device memory
// (code under HIP graph capture, tight serving loops).
//
// Every intermediate buffer of the call lives in one file-scope device
// array, `scratch`, of NOALLOC_SCRATCH_BYTES: the segment records (FP64
// and FP32 formats, the count), the targets in
// structure-of-arrays form, the chunk partial sums of the Biot-Savart
// launch and its work counter.  The call enqueues kernels on the context's
// stream and returns; it calls no hipMalloc, no hipFree, no allocating
// library routine and no hipMemsetAsync (counters are cleared by kernels).
// The array's device address is taken with hipGetSymbolAddress once per
// device, at the first call on that device, and kept per device.
//
// Every call on a GPU shares that GPU's array, which keeps the last call's
// contents: calls that overlap on one GPU (two contexts, two streams, or
// two host threads) race and must be serialised by the caller.
#include <mutex>

#include "vlm_internal.h"

namespace vlm {
// Inputs are accepted up to 64 MiB at 120 B per filament and 72 B per point
// (the sizes of an earlier layout, kept as the limit of the call).  The
// records take 226 B per filament, so the array is 64 MiB x 226 / 120 plus
// room for chunks.
constexpr size_t NOALLOC_ACCEPTED_BYTES = (size_t)64 << 20;
constexpr size_t NOALLOC_SCRATCH_BYTES = (size_t)192 << 20;
}

static __device__ __align__(256) unsigned char scratch[vlm::NOALLOC_SCRATCH_BYTES];

namespace vlm {
namespace {

constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
unsigned char *g_scratch_ptr[MAX_DEVICES] = {};

// The device address of `scratch` on the context's device (which is
// current), looked up on the first call per device.
int scratch_address(vlm_ctx *ctx, unsigned char **ptr)
{
    if (ctx->device < 0 || ctx->device >= MAX_DEVICES)
        return fail(ctx, VLM_ERR_ARG, "device index out of range for the scratch table");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[ctx->device]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) return hip_fail(ctx, e, "hipGetSymbolAddress(scratch)");
        g_scratch_ptr[ctx->device] = static_cast<unsigned char *>(p);
    }
    *ptr = g_scratch_ptr[ctx->device];
    return VLM_OK;
}

size_t up256(size_t b) { return (b + 255) & ~(size_t)255; }

unsigned nblk(int64_t n) { return (unsigned)((n + 255) / 256); }

// AoS device arrays to SoA targets; the first workgroup also clears the
// work counter of the launch that follows.
__global__ void aos_to_soa3_kernel(int64_t m, const double *aos, double *soa, int *counter)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) *counter = 0;
    if (i >= m) return;
    soa[i] = aos[3 * i];
    soa[m + i] = aos[3 * i + 1];
    soa[2 * m + i] = aos[3 * i + 2];
}

}  // namespace
}  // namespace vlm

using namespace vlm;

extern "C" {

int vlm_filament_vind_noalloc(vlm_ctx *ctx, int64_t nfil, const double *a, const double *b,
                              const double *gam, const double *rc, int64_t m, const double *p,
                              double *v, int accumulate)
{
    if (!ctx) return VLM_ERR_ARG;
    if (nfil < 0 || m < 0) return fail(ctx, VLM_ERR_ARG, "negative size");
    if (m == 0) return VLM_OK;
    if (!p || !v || (nfil > 0 && (!a || !b || !gam || !rc)))
        return fail(ctx, VLM_ERR_ARG, "null buffer");
    // workspace layout: soa | rec64 | grp | rec32 | near32 (the formats that
    // m targets need) | count | counter |
    // targets | partials.  The sizes accepted are those of the
    // documented 64 MiB at 120 B per filament and 72 B per point; the array
    // itself is larger (226 B per filament, group records included).
    const int64_t cap = nfil > 0 ? nfil : 1, gcap = (cap + GRP - 1) / GRP, rcap = gcap * GRP;
    const int fmt = bs_formats(ctx, m, nfil);
    const size_t osoa = 0;
    const size_t o64 = osoa + (fmt & SEG_SOA ? up256((size_t)SOA_N * rcap * sizeof(double)) : 0);
    const size_t ogrp = o64 + (fmt & SEG_REC ? up256((size_t)REC64_N * rcap * sizeof(double)) : 0);
    const size_t o32 = ogrp + (fmt & SEG_REC ? up256((size_t)GRPH_N * gcap * sizeof(double)) : 0);
    const size_t onear = o32 + (fmt & SEG_F32 ? up256((size_t)REC32_N * rcap * sizeof(float)) : 0);
    const size_t ocnt = onear + (fmt & SEG_F32 ? up256((size_t)NEAR32_N * rcap * sizeof(float)) : 0);
    const size_t octr = ocnt + 256;
    const size_t otgt = octr + 256;
    const size_t opart = otgt + up256((size_t)3 * m * sizeof(double));
    const size_t accepted = up256((size_t)9 * cap * sizeof(double)) +
                            up256((size_t)12 * cap * sizeof(float)) + 512 +
                            2 * up256((size_t)3 * m * sizeof(double)) +
                            (size_t)3 * m * sizeof(double);
    if (nfil > ((int64_t)1 << 32) || m > ((int64_t)1 << 32) ||
        accepted > NOALLOC_ACCEPTED_BYTES)
        return fail(ctx, VLM_ERR_ARG,
                    "vlm_filament_vind_noalloc: " + std::to_string(nfil) + " filaments and " +
                        std::to_string(m) + " points exceed the " +
                        std::to_string(NOALLOC_ACCEPTED_BYTES >> 20) +
                        " MiB workspace (about 120 B per filament and 72 B per point, plus "
                        "24 B per point for each chunk of partial sums)");
    VLM_DEVICE(ctx);
    unsigned char *w = nullptr;
    VLM_TRY(scratch_address(ctx, &w));
    SegPtrs seg;
    if (fmt & SEG_SOA) seg.soa = reinterpret_cast<double *>(w + osoa);
    if (fmt & SEG_REC) seg.rec64 = reinterpret_cast<double *>(w + o64);
    if (fmt & SEG_REC) seg.grp = reinterpret_cast<double *>(w + ogrp);
    if (fmt & SEG_F32) seg.rec32 = reinterpret_cast<float *>(w + o32);
    if (fmt & SEG_F32) seg.near32 = reinterpret_cast<float *>(w + onear);
    seg.count = reinterpret_cast<long long *>(w + ocnt);
    seg.cap = rcap;
    double *tgt = reinterpret_cast<double *>(w + otgt);
    BsWork ws;
    ws.part = reinterpret_cast<double *>(w + opart);
    ws.part_cap = (NOALLOC_SCRATCH_BYTES - opart) / sizeof(double);
    ws.counter = reinterpret_cast<int *>(w + octr);
    if (nfil > 0) VLM_TRY(explicit_records(ctx, nfil, a, b, gam, rc, seg));
    hipLaunchKernelGGL(aos_to_soa3_kernel, dim3(nblk(m)), dim3(256), 0, ctx->stream, m, p, tgt,
                       ws.counter);
    VLM_HIP(hipGetLastError());
    VLM_TRY(bs_eval(ctx, seg, nfil, tgt, m, m, v, accumulate, &ws, true));
    return VLM_OK;
}

}  // extern "C"
