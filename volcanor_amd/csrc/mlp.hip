// Learned wake-velocity predictor: a 45 -> 64 -> 64 -> 64 -> 3 MLP (tanh
// hidden layers, FP32), with hand-written inference, backward and Adam
// kernels.  No reference counterpart: it stands in for pass 2 of the AM2
// predictor-corrector (the Biot-Savart pass on the predicted wake,
// main.f90:1052-1086) and is trained online on the pairs that full passes
// produce.
//
// Parameter packing (row-major W[out][in]):
//   W1 64x45 | b1 64 | W2 64x64 | b2 64 | W3 64x64 | b3 64 | W4 3x64 | b4 3
//
// Every layer is a small matrix product on the matrix cores (FP32 MFMA).  A
// workgroup takes tiles of 16 samples; each of its four waves owns 16
// columns of every layer and keeps their weights (and, for training, the
// weight gradients) in registers, and activations and deltas pass between
// the waves through LDS.  Both kernels are bound by the latency of that chain
// (six products, six barriers), so tiles are small and many: with 64 samples
// per workgroup, weights staged in LDS and a gradient row per tile, a batch
// of 2048 took 50 us on 32 CUs and its reduction and loss 14 us.
// Training writes one partial gradient per workgroup; a second kernel adds
// them in a fixed order (deterministic, no atomics) and applies Adam.
#include <cmath>
#include <cstring>
#include <vector>

#include "vlm_internal.h"

namespace vlm {

constexpr int MLP_IN = 45, MLP_H = 64, MLP_OUT = 3;
constexpr int OFF_W1 = 0;
constexpr int OFF_B1 = OFF_W1 + MLP_H * MLP_IN;
constexpr int OFF_W2 = OFF_B1 + MLP_H;
constexpr int OFF_B2 = OFF_W2 + MLP_H * MLP_H;
constexpr int OFF_W3 = OFF_B2 + MLP_H;
constexpr int OFF_B3 = OFF_W3 + MLP_H * MLP_H;
constexpr int OFF_W4 = OFF_B3 + MLP_H;
constexpr int OFF_B4 = OFF_W4 + MLP_OUT * MLP_H;
constexpr int MLP_NP = OFF_B4 + MLP_OUT;  // 11459
// Host batches up to this size are read by the kernels in pinned memory.
constexpr size_t MLP_DIRECT = (size_t)4 << 20;

namespace {

// Matrix-core layout of v_mfma_f32_16x16x4f32 (checked on gfx950): lane l
// supplies A[l%16][l/16] and B[l/16][l%16] of the 16x16x4 step; result
// register r of lane l is D[4*(l/16) + r][l%16].
typedef float fx4 __attribute__((ext_vector_type(4)));

constexpr int TS = 16;            // samples per tile (one workgroup, four waves)
constexpr int LX = 52;            // LDS row strides: multiples of 4 (b128 reads) that
constexpr int LH = 68;            // spread the 16 rows of a fragment over all banks
constexpr int LDY = 20;
constexpr int XE = 3;             // X elements per lane: TS x MLP_IN / 256, rounded up
constexpr int MLP_ROWS = 512;     // workgroups (partial gradients) of a training launch

// A product over K values runs as K / 4 steps in any order that A and B
// share: step t takes k = lk K/4 + t, so that a lane's values are contiguous.
template <int NT>
__device__ __forceinline__ fx4 product(const float *row, const float (&b)[NT], fx4 acc)
{
    float a[NT];
#pragma unroll
    for (int t = 0; t < NT; t += 4) {
        const float4 v = *reinterpret_cast<const float4 *>(row + t);
        a[t] = v.x;
        a[t + 1] = v.y;
        a[t + 2] = v.z;
        a[t + 3] = v.w;
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t], b[t], acc, 0, 0, 0);
    return acc;
}

// D^T Act over the tile's samples: A[o][s] = D[s][o], B[s][i] = Act[s][i].
__device__ __forceinline__ fx4 outer(const float (&d)[4], const float *act, int la, fx4 acc)
{
#pragma unroll
    for (int t = 0; t < 4; ++t)
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(d[t], act[t * la], acc, 0, 0, 0);
    return acc;
}

__device__ __forceinline__ void load16(const float *p, float (&w)[16])
{
#pragma unroll
    for (int t = 0; t < 16; t += 4) {
        const float4 v = *reinterpret_cast<const float4 *>(p + t);
        w[t] = v.x;
        w[t + 1] = v.y;
        w[t + 2] = v.z;
        w[t + 3] = v.w;
    }
}

// The forward weights of a lane: column 16 w + li of layers 1 to 3, column li
// of layer 4 (zero beyond the third).
struct Forward {
    float w1[12], w2[16], w3[16], w4[16], b1, b2, b3, b4;
    __device__ Forward(const float *P, int w, int li, int lk)
    {
        const int c = 16 * w + li;
#pragma unroll
        for (int t = 0; t < 12; ++t) {
            const int k = 12 * lk + t;
            const float v = P[OFF_W1 + c * MLP_IN + min(k, MLP_IN - 1)];
            w1[t] = k < MLP_IN ? v : 0.f;
        }
        load16(P + OFF_W2 + c * MLP_H + 16 * lk, w2);
        load16(P + OFF_W3 + c * MLP_H + 16 * lk, w3);
        load16(P + OFF_W4 + min(li, MLP_OUT - 1) * MLP_H + 16 * lk, w4);
        b1 = P[OFF_B1 + c];
        b2 = P[OFF_B2 + c];
        b3 = P[OFF_B3 + c];
        b4 = P[OFF_B4 + min(li, MLP_OUT - 1)];
#pragma unroll
        for (int t = 0; t < 16; ++t) w4[t] = li < MLP_OUT ? w4[t] : 0.f;
    }
};

// The tile's elements of X (row-major), for LDS: requested one tile ahead.
__device__ __forceinline__ void fetch_x(const float *X, int64_t s0, int64_t m, float (&x)[XE])
{
    const int64_t left = (m - s0) * MLP_IN;   // may be <= 0 past the last tile
#pragma unroll
    for (int q = 0; q < XE; ++q) {
        const int e = q * 256 + threadIdx.x;
        x[q] = e < TS * MLP_IN && e < left ? X[s0 * MLP_IN + e] : 0.f;
    }
}

__device__ __forceinline__ void put_x(const float (&x)[XE], float *Xs)
{
#pragma unroll
    for (int q = 0; q < XE; ++q) {
        const int e = q * 256 + threadIdx.x;
        if (e < TS * MLP_IN) Xs[e / MLP_IN * LX + e % MLP_IN] = x[q];
    }
}

// Zero padding of the input rows (columns 45 to 47).
__device__ __forceinline__ void pad_x(float *Xs)
{
    if (threadIdx.x < 3 * TS) Xs[threadIdx.x / 3 * LX + MLP_IN + threadIdx.x % 3] = 0.f;
}

// tanh layer: the lane's values are samples 4 lk + r of column c.
template <int NT>
__device__ __forceinline__ void layer(const float *row, const float (&w)[NT], float b, float *O,
                                      int c, int lk, float (&h)[4])
{
    const fx4 acc = product<NT>(row, w, fx4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        h[r] = tanhf(acc[r] + b);
        O[(4 * lk + r) * LH + c] = h[r];
    }
}

__global__ __launch_bounds__(256) void mlp_forward_kernel(const float *params, int64_t m,
                                                          const float *X, float *Y)
{
    __shared__ __align__(16) float Xs[TS * LX], Ha[TS * LH], Hb[TS * LH];
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63, li = l & 15, lk = l >> 4;
    const int c = 16 * w + li;
    const int64_t ntiles = (m + TS - 1) / TS;
    float x[XE], h[4];
    fetch_x(X, (int64_t)blockIdx.x * TS, m, x);
    const Forward f(params, w, li, lk);
    pad_x(Xs);
    for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
        const int64_t s0 = t * TS;
        put_x(x, Xs);
        fetch_x(X, s0 + (int64_t)gridDim.x * TS, m, x);
        __syncthreads();
        layer<12>(Xs + li * LX + 12 * lk, f.w1, f.b1, Ha, c, lk, h);
        __syncthreads();
        layer<16>(Ha + li * LH + 16 * lk, f.w2, f.b2, Hb, c, lk, h);
        __syncthreads();
        layer<16>(Hb + li * LH + 16 * lk, f.w3, f.b3, Ha, c, lk, h);
        __syncthreads();
        if (w == 0) {
            const fx4 y = product<16>(Ha + li * LH + 16 * lk, f.w4, fx4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t s = s0 + 4 * lk + r;
                if (li < MLP_OUT && s < m) Y[s * MLP_OUT + li] = y[r] + f.b4;
            }
        }
    }
}

// Tiles of a training batch: forward, loss 0.5 |y - t|^2 / m, backward deltas
// and the workgroup's partial gradient (row blockIdx.x of part).
__global__ __launch_bounds__(256) void mlp_train_tile_kernel(const float *params, int64_t m,
                                                             const float *X, const float *T,
                                                             float *part, float *loss)
{
    __shared__ __align__(16) float Xs[TS * LX], H1[TS * LH], H2[TS * LH], H3[TS * LH];
    __shared__ __align__(16) float D1[TS * LH], D2[TS * LH], D3[TS * LH], DYs[4][TS * LDY];
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63, li = l & 15, lk = l >> 4;
    const int c = 16 * w + li;
    const int64_t ntiles = (m + TS - 1) / TS;
    const float inv_m = 1.0f / (float)m;
    const fx4 zero = {0.f, 0.f, 0.f, 0.f};
    float x[XE], y[4];
    fetch_x(X, (int64_t)blockIdx.x * TS, m, x);
    auto fetch_t = [&](int64_t s0) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t s = s0 + 4 * lk + r;
            y[r] = li < MLP_OUT && s < m ? T[s * MLP_OUT + li] : 0.f;
        }
    };
    fetch_t((int64_t)blockIdx.x * TS);
    const Forward f(params, w, li, lk);
    // backward weights: rows k of W_{l+1} at the lane's column
    float u2[16], u3[16], u4[4];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        u2[t] = params[OFF_W2 + (16 * lk + t) * MLP_H + c];
        u3[t] = params[OFF_W3 + (16 * lk + t) * MLP_H + c];
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int o = 4 * lk + t;
        const float v = params[OFF_W4 + min(o, MLP_OUT - 1) * MLP_H + c];
        u4[t] = o < MLP_OUT ? v : 0.f;
    }
    fx4 g1[3] = {zero, zero, zero}, g2[4] = {zero, zero, zero, zero};
    fx4 g3[4] = {zero, zero, zero, zero}, g4 = zero;
    float gb1 = 0.f, gb2 = 0.f, gb3 = 0.f, gb4 = 0.f, lsum = 0.f;
    float *DY = DYs[w];   // each wave has the output deltas for itself
    pad_x(Xs);
    for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int64_t s0 = tile * TS, s1 = s0 + (int64_t)gridDim.x * TS;
        float h1[4], h2[4], h3[4], d[4];
        put_x(x, Xs);
        fetch_x(X, s1, m, x);
        __syncthreads();
        layer<12>(Xs + li * LX + 12 * lk, f.w1, f.b1, H1, c, lk, h1);
        __syncthreads();
        layer<16>(H1 + li * LH + 16 * lk, f.w2, f.b2, H2, c, lk, h2);
        __syncthreads();
        layer<16>(H2 + li * LH + 16 * lk, f.w3, f.b3, H3, c, lk, h3);
        __syncthreads();
        // dy = (y - t) / m on real samples and outputs, zero elsewhere
        fx4 acc = product<16>(H3 + li * LH + 16 * lk, f.w4, zero);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float e = 0.f;
            if (li < MLP_OUT && s0 + 4 * lk + r < m) {
                const float err = acc[r] + f.b4 - y[r];
                lsum += 0.5f * err * err * inv_m;
                e = err * inv_m;
            }
            DY[(4 * lk + r) * LDY + li] = e;
            gb4 += e;
        }
        fetch_t(s1);
        // layer 4: gradient of the wave's 16 columns, delta of layer 3
#pragma unroll
        for (int t = 0; t < 4; ++t) d[t] = DY[(4 * lk + t) * LDY + li];
        g4 = outer(d, H3 + 4 * lk * LH + c, LH, g4);
        auto delta = [&](const fx4 &p, const float (&h)[4], float *D, float &gb) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float v = p[r] * (1.f - h[r] * h[r]);
                D[(4 * lk + r) * LH + c] = v;
                gb += v;
            }
            // the wave's columns, as the other factor of its gradients
#pragma unroll
            for (int t = 0; t < 4; ++t) d[t] = D[(4 * lk + t) * LH + c];
        };
        delta(product<4>(DY + li * LDY + 4 * lk, u4, zero), h3, D3, gb3);
        __syncthreads();
#pragma unroll
        for (int ib = 0; ib < 4; ++ib)
            g3[ib] = outer(d, H2 + 4 * lk * LH + 16 * ib + li, LH, g3[ib]);
        delta(product<16>(D3 + li * LH + 16 * lk, u3, zero), h2, D2, gb2);
        __syncthreads();
#pragma unroll
        for (int ib = 0; ib < 4; ++ib)
            g2[ib] = outer(d, H1 + 4 * lk * LH + 16 * ib + li, LH, g2[ib]);
        delta(product<16>(D2 + li * LH + 16 * lk, u2, zero), h1, D1, gb1);
#pragma unroll
        for (int ib = 0; ib < 3; ++ib)
            g1[ib] = outer(d, Xs + 4 * lk * LX + 16 * ib + li, LX, g1[ib]);
        __syncthreads();
    }
    // gradients: lane l holds outputs 16 w + 4 lk + r of input 16 ib + li
    float *g = part + (size_t)blockIdx.x * MLP_NP;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int o = 16 * w + 4 * lk + r;
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) {
            const int i = 16 * ib + li;
            if (ib < 3 && i < MLP_IN) g[OFF_W1 + o * MLP_IN + i] = g1[ib < 3 ? ib : 0][r];
            g[OFF_W2 + o * MLP_H + i] = g2[ib][r];
            g[OFF_W3 + o * MLP_H + i] = g3[ib][r];
        }
        if (lk == 0 && r < MLP_OUT) g[OFF_W4 + r * MLP_H + c] = g4[r];
    }
    auto over_lk = [](float v) {
        v += __shfl_xor(v, 16);
        return v + __shfl_xor(v, 32);
    };
    gb1 = over_lk(gb1);
    gb2 = over_lk(gb2);
    gb3 = over_lk(gb3);
    gb4 = over_lk(gb4);
    lsum = over_lk(lsum);
    for (int o = 1; o < 16; o <<= 1) lsum += __shfl_xor(lsum, o);
    if (lk == 0) {
        g[OFF_B1 + c] = gb1;
        g[OFF_B2 + c] = gb2;
        g[OFF_B3 + c] = gb3;
        if (w == 0 && li < MLP_OUT) g[OFF_B4 + li] = gb4;
    }
    if (threadIdx.x == 0) loss[blockIdx.x] = lsum;
}

// Sum of the partial gradients, then (optionally) Adam: GS slices of rows side
// by side, each in order, the slices added in order (one lane per parameter
// over 32 rows: 9 us).  The last workgroup sums the loss, also to loss_host
// (pinned) when given.
constexpr int GS = 8;

__global__ __launch_bounds__(64 * GS) void mlp_grad_kernel(float *params, const float *part,
                                                           int rows, float *grad, float *mom,
                                                           float *var, int adam, float lr,
                                                           float b1, float b2, float bc1,
                                                           float bc2, float epsa,
                                                           const float *loss, float *lsum,
                                                           float *loss_host)
{
    __shared__ float sh[GS][64];
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (blockIdx.x == gridDim.x - 1) {
        float s = 0.f;
        for (int c = threadIdx.x; c < rows; c += 64 * GS) s += loss[c];
        for (int o = 1; o < 64; o <<= 1) s += __shfl_xor(s, o);
        if (l == 0) sh[w][0] = s;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int q = 1; q < GS; ++q) s += sh[q][0];
            *lsum = s;
            if (loss_host) *loss_host = s;
        }
        return;
    }
    const int k = blockIdx.x * 64 + l, kc = min(k, MLP_NP - 1);
    const int len = (rows + GS - 1) / GS, c1 = min(rows, (w + 1) * len);
    float g = 0.f;
    int c = w * len;
    for (; c + 8 <= c1; c += 8) {
        float v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = part[(size_t)(c + q) * MLP_NP + kc];
#pragma unroll
        for (int q = 0; q < 8; ++q) g += v[q];
    }
    for (; c < c1; ++c) g += part[(size_t)c * MLP_NP + kc];
    sh[w][l] = g;
    __syncthreads();
    if (w > 0 || k >= MLP_NP) return;
    for (int q = 1; q < GS; ++q) g += sh[q][l];
    grad[k] = g;
    if (adam) {
        const float mk = b1 * mom[k] + (1.f - b1) * g;
        const float vk = b2 * var[k] + (1.f - b2) * g * g;
        mom[k] = mk;
        var[k] = vk;
        params[k] -= lr * (mk / bc1) / (sqrtf(vk / bc2) + epsa);
    }
}

}  // namespace

struct Mlp {
    DBuf<float> params, mom, var, grad, part;
    DBuf<float> loss, lsum;
    DBuf<float> xin, yout;
    int64_t steps = 0;
    bool ready = false;
    bool have_loss = false;
};

static Mlp *get_mlp(vlm_ctx *ctx);

int mlp_forward_dev(vlm_ctx *ctx, int64_t m, const float *X, float *Y)
{
    Mlp *M = get_mlp(ctx);
    if (!M) return fail(ctx, VLM_ERR_ALLOC, "mlp allocation failed");
    if (m <= 0) return VLM_OK;
    const int64_t ntiles = (m + TS - 1) / TS;
    const unsigned grid = (unsigned)(ntiles < 1024 ? ntiles : 1024);
    hipLaunchKernelGGL(mlp_forward_kernel, dim3(grid), dim3(256), 0, ctx->stream, M->params.p,
                       m, X, Y);
    VLM_HIP(hipGetLastError());
    return VLM_OK;
}

// Gradient (and optionally one Adam step) on a device batch.
int mlp_train_dev(vlm_ctx *ctx, int64_t m, const float *X, const float *T, int adam, float lr,
                  float *loss_pin, int keep_loss)
{
    Mlp *M = get_mlp(ctx);
    if (!M) return fail(ctx, VLM_ERR_ALLOC, "mlp allocation failed");
    if (m <= 0) return VLM_OK;
    const int64_t ntiles = (m + TS - 1) / TS;
    const int rows = (int)(ntiles < MLP_ROWS ? ntiles : MLP_ROWS);
    VLM_HIP(M->part.reserve((size_t)rows * MLP_NP));
    VLM_HIP(M->loss.reserve((size_t)rows));
    hipLaunchKernelGGL(mlp_train_tile_kernel, dim3((unsigned)rows), dim3(256), 0, ctx->stream,
                       M->params.p, m, X, T, M->part.p, M->loss.p);
    VLM_HIP(hipGetLastError());
    float bc1 = 1.f, bc2 = 1.f;
    const float b1 = 0.9f, b2 = 0.999f;
    if (adam) {
        M->steps += 1;
        bc1 = 1.f - std::pow(b1, (float)M->steps);
        bc2 = 1.f - std::pow(b2, (float)M->steps);
    }
    const bool want_loss = loss_pin || keep_loss;
    float *lsum = want_loss ? M->lsum.p : M->lsum.p + 1;
    hipLaunchKernelGGL(mlp_grad_kernel, dim3((MLP_NP + 63) / 64 + 1), dim3(64 * GS), 0,
                       ctx->stream, M->params.p, M->part.p, rows, M->grad.p, M->mom.p, M->var.p,
                       adam, lr, b1, b2, bc1, bc2, 1e-8f, M->loss.p, lsum,
                       loss_pin);
    VLM_HIP(hipGetLastError());
    if (want_loss) M->have_loss = true;
    return loss_pin ? sync_stream(ctx) : VLM_OK;
}

// Loss of the last training call that kept it on the device (0 if none).
int mlp_read_loss(vlm_ctx *ctx, float *loss)
{
    *loss = 0.f;
    Mlp *M = ctx->mlp;
    if (!M || !M->have_loss) return VLM_OK;
    return d2h(ctx, loss, M->lsum.p, sizeof(float));
}

// Deterministic small-scale initialisation (uniform +-sqrt(6/(in+out)),
// zero biases) from a fixed-seed linear congruential stream.
static void mlp_init_host(std::vector<float> &p, unsigned long long seed)
{
    p.assign(MLP_NP, 0.f);
    unsigned long long s = seed * 6364136223846793005ULL + 1442695040888963407ULL;
    auto uni = [&]() {
        s = s * 6364136223846793005ULL + 1442695040888963407ULL;
        return (float)((s >> 11) * (1.0 / 9007199254740992.0)) * 2.f - 1.f;
    };
    auto fill = [&](int off, int nout, int nin) {
        const float a = std::sqrt(6.f / (float)(nin + nout));
        for (int k = 0; k < nout * nin; ++k) p[off + k] = a * uni();
    };
    fill(OFF_W1, MLP_H, MLP_IN);
    fill(OFF_W2, MLP_H, MLP_H);
    fill(OFF_W3, MLP_H, MLP_H);
    fill(OFF_W4, MLP_OUT, MLP_H);
    for (int k = 0; k < MLP_OUT * MLP_H; ++k) p[OFF_W4 + k] *= 0.1f;
}

static Mlp *get_mlp(vlm_ctx *ctx)
{
    if (ctx->mlp) return ctx->mlp;
    Mlp *M = new Mlp();
    if (M->params.reserve(MLP_NP) != hipSuccess || M->mom.reserve(MLP_NP) != hipSuccess ||
        M->var.reserve(MLP_NP) != hipSuccess || M->grad.reserve(MLP_NP) != hipSuccess ||
        M->lsum.reserve(2) != hipSuccess) {   // kept, not kept
        delete M;
        return nullptr;
    }
    std::vector<float> p;
    mlp_init_host(p, 20261202ULL);
    std::vector<float> z(MLP_NP, 0.f);
    if (hipMemcpy(M->params.p, p.data(), MLP_NP * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(M->mom.p, z.data(), MLP_NP * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(M->var.p, z.data(), MLP_NP * sizeof(float), hipMemcpyHostToDevice) != hipSuccess) {
        delete M;
        return nullptr;
    }
    ctx->mlp = M;
    return M;
}

void mlp_release(vlm_ctx *ctx)
{
    delete ctx->mlp;
    ctx->mlp = nullptr;
}

}  // namespace vlm

using namespace vlm;

extern "C" {

int vlm_mlp_num_params(void) { return MLP_NP; }

int vlm_mlp_set_params(vlm_ctx *ctx, const float *params)
{
    if (!ctx || !params) return VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    Mlp *M = get_mlp(ctx);
    if (!M) return fail(ctx, VLM_ERR_ALLOC, "mlp allocation failed");
    VLM_HIP(hipMemcpy(M->params.p, params, MLP_NP * sizeof(float), hipMemcpyHostToDevice));
    std::vector<float> z(MLP_NP, 0.f);
    VLM_HIP(hipMemcpy(M->mom.p, z.data(), MLP_NP * sizeof(float), hipMemcpyHostToDevice));
    VLM_HIP(hipMemcpy(M->var.p, z.data(), MLP_NP * sizeof(float), hipMemcpyHostToDevice));
    M->steps = 0;
    return VLM_OK;
}

int vlm_mlp_get_params(vlm_ctx *ctx, float *params)
{
    if (!ctx || !params) return VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    Mlp *M = get_mlp(ctx);
    if (!M) return fail(ctx, VLM_ERR_ALLOC, "mlp allocation failed");
    return d2h(ctx, params, M->params.p, MLP_NP * sizeof(float));
}

int vlm_mlp_forward(vlm_ctx *ctx, int64_t m, const float *x, float *y)
{
    if (!ctx || m < 0 || (m > 0 && (!x || !y))) return VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    Mlp *M = get_mlp(ctx);
    if (!M) return fail(ctx, VLM_ERR_ALLOC, "mlp allocation failed");
    if (m == 0) return VLM_OK;
    const size_t nx = sizeof(float) * (size_t)m * MLP_IN, ny = sizeof(float) * (size_t)m * MLP_OUT;
    if (nx + ny <= MLP_DIRECT) {
        char *hp = nullptr;
        VLM_TRY(pin_take(ctx, nx + ny, &hp));
        std::memcpy(hp, x, nx);
        VLM_TRY(mlp_forward_dev(ctx, m, reinterpret_cast<const float *>(hp),
                                reinterpret_cast<float *>(hp + nx)));
        VLM_TRY(sync_stream(ctx));
        std::memcpy(y, hp + nx, ny);
        return VLM_OK;
    }
    VLM_HIP(M->xin.reserve((size_t)m * MLP_IN));
    VLM_HIP(M->yout.reserve((size_t)m * MLP_OUT));
    VLM_TRY(h2d(ctx, M->xin.p, x, nx));
    VLM_TRY(mlp_forward_dev(ctx, m, M->xin.p, M->yout.p));
    return d2h(ctx, y, M->yout.p, ny);
}

// A host batch where the training kernel reads it (each value once): in the
// pinned arena up to MLP_DIRECT bytes, else in a device copy.  *loss receives
// a pinned slot, taken with the batch (a later request may recycle the arena).
static int batch_in(vlm_ctx *ctx, Mlp *M, int64_t m, const float *x, const float *t,
                    const float **X, const float **T, float **loss)
{
    const size_t nx = sizeof(float) * (size_t)m * MLP_IN, nt = sizeof(float) * (size_t)m * MLP_OUT;
    const bool direct = nx + nt <= MLP_DIRECT;
    if (!direct) {
        VLM_HIP(M->xin.reserve((size_t)m * (MLP_IN + MLP_OUT)));
        VLM_TRY(h2d(ctx, M->xin.p, x, nx));
        VLM_TRY(h2d(ctx, M->xin.p + m * MLP_IN, t, nt));
    }
    char *hp = nullptr;
    VLM_TRY(pin_take(ctx, sizeof(float) + (direct ? nx + nt : 0), &hp));
    if (direct) {
        std::memcpy(hp, x, nx);
        std::memcpy(hp + nx, t, nt);
    }
    *X = direct ? reinterpret_cast<const float *>(hp) : M->xin.p;
    *T = *X + m * MLP_IN;
    *loss = reinterpret_cast<float *>(hp + (direct ? nx + nt : 0));
    return VLM_OK;
}

int vlm_mlp_loss_grad(vlm_ctx *ctx, int64_t m, const float *x, const float *t, float *grad,
                      float *loss)
{
    if (!ctx || m <= 0 || !x || !t) return VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    Mlp *M = get_mlp(ctx);
    if (!M) return fail(ctx, VLM_ERR_ALLOC, "mlp allocation failed");
    const float *X, *T;
    float *l = nullptr;
    VLM_TRY(batch_in(ctx, M, m, x, t, &X, &T, &l));
    VLM_TRY(mlp_train_dev(ctx, m, X, T, 0, 0.f, l));
    if (loss) *loss = *l;
    if (grad) return d2h(ctx, grad, M->grad.p, MLP_NP * sizeof(float));
    return VLM_OK;
}

int vlm_mlp_train_step(vlm_ctx *ctx, int64_t m, const float *x, const float *t, float lr,
                       float *loss)
{
    if (!ctx || m <= 0 || !x || !t) return VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    Mlp *M = get_mlp(ctx);
    if (!M) return fail(ctx, VLM_ERR_ALLOC, "mlp allocation failed");
    const float *X, *T;
    float *l = nullptr;
    VLM_TRY(batch_in(ctx, M, m, x, t, &X, &T, &l));
    VLM_TRY(mlp_train_dev(ctx, m, X, T, 1, lr, l));
    if (loss) *loss = *l;
    return VLM_OK;
}

}  // extern "C"
