// AIC assembly and the circulation solve.
//
// rotor_calcAIC (classdef.f90:4151-4179) builds AIC(row,col) = vr_vind of
// wing ring col at collocation point row, projected on nCap(row), and
// inverts it once (inv2 -> DGETRF + DGETRI, libMath.f90:48-83); every step
// then forms gamVec = AIC_inv . RHS (matmulAX, libMath.f90:105-122).
// Here the matrix is factorised once (LU with partial pivoting, kept on the
// device) and every step solves by two triangular sweeps plus iterative
// refinement on an FP64 residual RHS - AIC . gam.
//
// Factorisation: lu_factor_device (lu_mfma.hip).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "vlm_internal.h"

namespace vlm {

int lu_factor_device(vlm_ctx *ctx, int n, double *A, int *ipiv, int *info_dev);

namespace {

constexpr double EPS2 = kEps * kEps;

__device__ __forceinline__ void fil64(const double *P, const double *A, const double *B,
                                      double rc, double *v)
{
    // vf_vind in the reference's own operation order (classdef.f90:476-503)
    const double r1x = P[0] - A[0], r1y = P[1] - A[1], r1z = P[2] - A[2];
    const double r2x = P[0] - B[0], r2y = P[1] - B[1], r2z = P[2] - B[2];
    const double r0x = r1x - r2x, r0y = r1y - r2y, r0z = r1z - r2z;
    const double cx = r1y * r2z - r1z * r2y;
    const double cy = r1z * r2x - r1x * r2z;
    const double cz = r1x * r2y - r1y * r2x;
    const double c2 = cx * cx + cy * cy + cz * cz;
    if (c2 > EPS2) {
        const double n1 = sqrt(r1x * r1x + r1y * r1y + r1z * r1z);
        const double n2 = sqrt(r2x * r2x + r2y * r2y + r2z * r2z);
        double u1x = 0, u1y = 0, u1z = 0, u2x = 0, u2y = 0, u2z = 0;
        if (n1 > kEps) {
            u1x = r1x / n1;
            u1y = r1y / n1;
            u1z = r1z / n1;
        }
        if (n2 > kEps) {
            u2x = r2x / n2;
            u2y = r2y / n2;
            u2z = r2z / n2;
        }
        const double dot = r0x * (u1x - u2x) + r0y * (u1y - u2y) + r0z * (u1z - u2z);
        const double q = rc * sqrt(r0x * r0x + r0y * r0y + r0z * r0z);
        const double den = sqrt(q * q * q * q + c2 * c2);
        const double s = kInv4Pi * dot / den;
        v[0] += cx * s;
        v[1] += cy * s;
        v[2] += cz * s;
    }
}

// One lane per (row, col): unit-strength ring col at CP row, dotted with
// nCap(row).  Column-major A.
__global__ void aic_kernel(int n, const double *wc, const double *wrc, const double *cp,
                           const double *ncap, double *A)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (int64_t)n * n) return;
    const int row = (int)(e % n), col = (int)(e / n);
    const double *c = wc + 12 * (size_t)col;
    const double *rc = wrc + 4 * (size_t)col;
    double v[3] = {0.0, 0.0, 0.0};
    for (int f = 0; f < 4; ++f) fil64(cp + 3 * row, c + 3 * f, c + 3 * ((f + 1) & 3), rc[f], v);
    A[e] = v[0] * ncap[3 * row] + v[1] * ncap[3 * row + 1] + v[2] * ncap[3 * row + 2];
}

// ---------------------------------------------------------------------
// Systems larger than one wave's (n > 96): substitutions over blocks of
// TB rows, one workgroup per block and sweep.  A block needs the solved
// blocks before it (forward: those above; backward: those below), and the
// workgroups run side by side: each takes a ticket, tickets 0..nb-1 are the
// forward blocks top down, nb..2nb-1 the backward blocks bottom up, and a
// block waits only for blocks of lower tickets, whose workgroups have
// started already, so every wait ends whatever the dispatch order.  A wave
// polls the solved values themselves: the buffers are filled with a NaN of
// a payload no value is published with (SENT), and a value arrives as one
// 64-bit store.  The matrix tile of the next block column is loaded while
// the values of this one are awaited.
//
// Bound by the chain of blocks: one store-to-load trip between compute
// units and one 64-step substitution in a wave per block.  The sweep this
// replaces (one workgroup, one column per barrier, pivots applied by one
// lane) took 99 us per solve at n = 160 and 4.37 ms at n = 2176; the lane
// per row of the residual 22 and 634 us.
constexpr int TB = 64;
constexpr unsigned long long SENT = 0x7FFC0DEADBEEF001ull;

__device__ __forceinline__ unsigned long long load_agent(const unsigned long long *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void publish(unsigned long long *p, double v)
{
    unsigned long long u = (unsigned long long)__double_as_longlong(v);
    if (u == SENT) u = 0x7FF8000000000000ull;
    __hip_atomic_store(p, u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ double readlane_d(double v, int lane)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Device state of one solve: ticket, convergence and the number of
// corrections, the maximum norms as bit patterns (unsigned order is the
// order of non-negative doubles), and the two sweeps' block results.
struct SolveWork {
    int *ticket, *st;                        // st: converged, corrections applied
    unsigned long long *rmax, *bmax;         // rmax[2]: residual it writes rmax[it & 1]
    unsigned long long *y, *z;               // nb * TB each
};

__global__ __launch_bounds__(256) void solve_init_kernel(int n, const double *b, SolveWork w)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int np = (n + TB - 1) / TB * TB;
    if (i < np) {
        w.y[i] = SENT;
        w.z[i] = SENT;
    }
    if (blockIdx.x == 0) {
        __shared__ double sm[4];
        if (threadIdx.x == 0) {
            *w.ticket = 0;
            w.st[0] = 0;
            w.st[1] = 0;
            w.rmax[0] = 0;
        }
        double m = 0.0;
        for (int k = threadIdx.x; k < n; k += 256) m = fmax(m, fabs(b[k]));
        for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
        if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = m;
        __syncthreads();
        if (threadIdx.x == 0)
            *w.bmax = (unsigned long long)__double_as_longlong(
                fmax(fmax(sm[0], sm[1]), fmax(sm[2], sm[3])));
    }
}

// x = (LU)^-1 P rhs, or, for a correction (acc), x += it unless the last
// residual met tol.  perm[i] is the row of the right-hand side that the
// pivoting moves to row i.
__global__ __launch_bounds__(256) void lu_sweeps_kernel(int n, const double *LU, const int *perm,
                                                        const double *rhs, double *x, int acc,
                                                        int it, double tol, SolveWork w)
{
    __shared__ double D[TB * TB];   // diagonal block, column-major
    __shared__ double part[4][TB];
    __shared__ int tk;
    const int tid = threadIdx.x, lane = tid & 63, q = tid >> 6;
    const bool conv = acc && (w.st[0] || __longlong_as_double((long long)w.rmax[it & 1]) <=
                                             tol * __longlong_as_double((long long)*w.bmax));
    if (tid == 0) tk = atomicAdd(w.ticket, 1);
    __syncthreads();
    if (conv) {
        // the flag only for the launches that follow: this launch decides by
        // the norms, which nothing in it changes
        if (tk == 0 && tid == 0) w.st[0] = 1;
        return;
    }
    if (tk == 0 && tid == 0 && acc) w.st[1] += 1;
    const int nb = (n + TB - 1) / TB;
    const bool back = tk >= nb;
    const int blk = back ? 2 * nb - 1 - tk : tk;
    const int r0 = blk * TB, row = r0 + lane;
    const size_t ld = (size_t)n;
    for (int e = tid; e < TB * TB; e += 256) {
        const int i = r0 + (e & 63), j = r0 + (e >> 6);
        D[e] = (i < n && j < n) ? LU[i + ld * j] : (i == j ? 1.0 : 0.0);
    }
    // the blocks this one needs, in the order they are solved: this wave
    // takes 16 columns of each
    const int nk = back ? nb - 1 - blk : blk;
    const unsigned long long *src = back ? w.z : w.y;
    auto col0 = [&](int k) { return (back ? nb - 1 - k : k) * TB + 16 * q; };
    double t[16], s = 0.0;
    const int rc = row < n ? row : n - 1;
    auto load = [&](int k) {
#pragma unroll
        for (int c = 0; c < 16; ++c) {
            const int j = col0(k) + c;
            const double v = LU[rc + ld * (j < n ? j : n - 1)];
            t[c] = (row < n && j < n) ? v : 0.0;
        }
    };
    if (nk > 0) load(0);
    for (int k = 0; k < nk; ++k) {
        double a[16];
#pragma unroll
        for (int c = 0; c < 16; ++c) a[c] = t[c];
        if (k + 1 < nk) load(k + 1);
        const unsigned long long *p = src + col0(k) + (lane & 15);
        unsigned long long u = load_agent(p);
        while (__any(u == SENT)) {
            __builtin_amdgcn_s_sleep(1);
            u = load_agent(p);
        }
        const double v = __longlong_as_double((long long)u);
#pragma unroll
        for (int c = 0; c < 16; ++c) s += a[c] * readlane_d(v, c);
    }
    part[q][lane] = s;
    __syncthreads();
    if (q > 0) return;
    double v;
    if (back) {   // own forward block
        unsigned long long u = load_agent(w.y + row);
        while (__any(u == SENT)) {
            __builtin_amdgcn_s_sleep(1);
            u = load_agent(w.y + row);
        }
        v = __longlong_as_double((long long)u);
    } else {
        v = row < n ? rhs[perm[row]] : 0.0;
    }
    v -= (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
    if (row >= n) v = 0.0;
    // A solved value is kept in y; the rows behind it go on being updated
    // with what no one reads (a zero factor would turn them into NaN where a
    // value is infinite).
    constexpr int SU = 8;   // columns whose LDS reads issue ahead of the chain
    double y = 0.0;
    if (!back) {
        for (int j = 0; j < TB; j += SU) {
            double l[SU];
#pragma unroll
            for (int u = 0; u < SU; ++u) l[u] = D[lane + TB * (j + u)];
#pragma unroll
            for (int u = 0; u < SU; ++u) {
                const double xj = readlane_d(v, j + u);
                y = lane == j + u ? xj : y;
                v -= l[u] * xj;
            }
        }
        publish(w.y + row, y);
        return;
    }
    // v / d by the reciprocal and one correction of the remainder, or by
    // division where a reciprocal leaves the normal range or a value is not
    // finite (seen at the end, as the correction makes it NaN)
    const double d = D[lane + TB * lane], rd = 1.0 / d, v0 = v;
    bool plain = __any(!(fabs(rd) < 1e300 && fabs(rd) > 1e-300)) != 0;
    for (;;) {
        v = v0;
        for (int j = TB - SU; j >= 0; j -= SU) {
            double l[SU];
#pragma unroll
            for (int u = 0; u < SU; ++u) l[u] = D[lane + TB * (j + u)];
#pragma unroll
            for (int u = SU - 1; u >= 0; --u) {
                const double g = v * rd;
                double e = __builtin_fma(__builtin_fma(-g, d, v), rd, g);
                if (plain) e = v / d;
                const double xj = readlane_d(e, j + u);
                y = lane == j + u ? xj : y;
                v -= l[u] * xj;
            }
        }
        if (plain || !__any(!(fabs(y) < __builtin_inf()))) break;
        plain = true;
    }
    publish(w.z + row, y);
    if (row < n) x[row] = acc ? x[row] + y : y;
}

// r = b - A x and its maximum norm: RROWS rows per workgroup, the columns
// in RSL slices (A is read once, in runs of 256 bytes).  Clears the sweep
// buffers and the ticket for the correction that follows.
constexpr int RROWS = 32, RSL = 32;

__global__ __launch_bounds__(RROWS * RSL) void residual_kernel(int n, const double *A,
                                                               const double *x, const double *b,
                                                               double *r, int it, SolveWork w)
{
    __shared__ double part[RSL][RROWS + 1];
    const int l = threadIdx.x % RROWS, q = threadIdx.x / RROWS;
    const int i = blockIdx.x * RROWS + l;
    if (w.st[0]) return;
    double s = 0.0;
    if (i < n)
        for (int j = q; j < n; j += RSL) s += A[i + (size_t)n * j] * x[j];
    part[q][l] = s;
    const int np = (n + TB - 1) / TB * TB;
    const int e = blockIdx.x * RROWS * RSL + threadIdx.x;
    for (int k = e; k < np; k += gridDim.x * RROWS * RSL) {
        w.y[k] = SENT;
        w.z[k] = SENT;
    }
    if (e == 0) {
        *w.ticket = 0;
        w.rmax[(it + 1) & 1] = 0;   // read last by the previous correction
    }
    __syncthreads();
    if (q > 0) return;
    double t = 0.0;
    for (int k = 0; k < RSL; ++k) t += part[k][l];
    t = i < n ? b[i] - t : 0.0;
    if (i < n) r[i] = t;
    // NaNs do not count
    unsigned long long m = t == t ? (unsigned long long)__double_as_longlong(fabs(t)) : 0ull;
    for (int o = 16; o > 0; o >>= 1) {
        const unsigned long long v = __shfl_xor(m, o, 32);
        m = v > m ? v : m;
    }
    if (l == 0) atomicMax(w.rmax + (it & 1), m);
}

// rotor_map_gam (classdef.f90:4181-4196): blades ib <= nbConvect take
// their part of gamVec; with axisymmetry (nbConvect = 1) every blade takes
// blade 1's.
__global__ void map_gam_kernel(const double *x, double *wg, int per_blade, int nb, int nbc)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= per_blade * nb) return;
    const int b = e / per_blade, k = e - b * per_blade;
    if (b < nbc) wg[e] = x[e];
    else if (nbc == 1) wg[e] = x[k];
}

// The whole solve with refinement in one wave for n <= 64 R: lane l holds
// rows l + 64 r (r < R) of x, b and r in the pivoted order; LU and the
// pivoted A are staged in LDS (both fit the 160 KB of a gfx950 CU up to n =
// 96).  The workgroup has SOLVE_STAGE threads so that the staging copy keeps
// many loads in flight; after it every wave but the first leaves.
// Bound by the instructions of that wave, one every four cycles: a column of
// a substitution is two readlanes (x_j), a select (x_j kept, so that rows
// already solved may be overwritten and need no mask) and R FMAs, and U is
// scaled by its diagonal off that chain.  Order 90 with three
// corrections takes 38 us; with masks, a division per column and the row
// swaps in the wave it took 56.
constexpr int SOLVE_STAGE = 512;
constexpr int SOLVE_WAVE_N = 64;   // one row per lane
constexpr int SOLVE_WAVE_N2 = 96;  // two rows per lane

__device__ __forceinline__ double wave_max(double v)
{
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off));
    return v;
}

// One column of a substitution: x_j of v[r], the rows of v[Q0..Q1].
template <int R, int Q0, int Q1>
__device__ __forceinline__ void wave_column(double xj, const double (&c)[R], double (&v)[R])
{
#pragma unroll
    for (int q = Q0; q <= Q1; ++q) v[q] -= c[q] * xj;
}

constexpr int WSU = 8;   // columns whose LDS reads issue ahead of the chain

// Columns [64 r, min(n, 64 r + 64)) forward with the unit lower triangle.
template <int R, int r>
__device__ __forceinline__ void wave_forward(int n, const double *sLU, double (&v)[R],
                                             double (&x)[R])
{
    const int l = threadIdx.x, j1 = min(n, 64 * r + 64);
    for (int j = 64 * r; j < j1; j += WSU) {
        double c[WSU][R];
#pragma unroll
        for (int u = 0; u < WSU; ++u)
#pragma unroll
            for (int q = r; q < R; ++q)
                c[u][q] = sLU[min(l + 64 * q, n - 1) + n * min(j + u, n - 1)];
#pragma unroll
        for (int u = 0; u < WSU; ++u) {
            if (j + u >= j1) break;
            const double xj = readlane_d(v[r], (j + u) & 63);
            x[r] = l == ((j + u) & 63) ? xj : x[r];
            wave_column<R, r, R - 1>(xj, c[u], v);
        }
    }
}

// The same columns backward with the upper triangle, its rows scaled by rd
// (v already divided by the diagonal), or, plain, with a division by d_j.
template <int R, int r>
__device__ __forceinline__ void wave_backward(int n, const double *sLU, const double (&d)[R],
                                              const double (&rd)[R], bool plain, double (&v)[R],
                                              double (&x)[R])
{
    const int l = threadIdx.x;
    for (int j = min(n, 64 * r + 64) - 1; j >= 64 * r; j -= WSU) {
        double c[WSU][R];
#pragma unroll
        for (int u = 0; u < WSU; ++u)
#pragma unroll
            for (int q = 0; q <= r; ++q) {
                const double t = sLU[min(l + 64 * q, n - 1) + n * max(j - u, 0)];
                c[u][q] = plain ? t : t * rd[q];
            }
#pragma unroll
        for (int u = 0; u < WSU; ++u) {
            if (j - u < 64 * r) break;
            double xj = readlane_d(v[r], (j - u) & 63);
            if (plain) xj /= readlane_d(d[r], (j - u) & 63);
            x[r] = l == ((j - u) & 63) ? xj : x[r];
            wave_column<R, 0, r>(xj, c[u], v);
        }
    }
}

// v <- (LU)^-1 v.  plain: a reciprocal of the diagonal leaves the normal
// range.
template <int R>
__device__ void wave_lu_solve(int n, const double *sLU, const double (&d)[R],
                              const double (&rd)[R], bool plain, double (&v)[R])
{
    double x[R];
#pragma unroll
    for (int q = 0; q < R; ++q) x[q] = 0.0;
    wave_forward<R, 0>(n, sLU, v, x);
    if constexpr (R > 1) wave_forward<R, R - 1>(n, sLU, v, x);
#pragma unroll
    for (int q = 0; q < R; ++q) v[q] = plain ? x[q] : x[q] / d[q];
    if constexpr (R > 1) wave_backward<R, R - 1>(n, sLU, d, rd, plain, v, x);
    wave_backward<R, 0>(n, sLU, d, rd, plain, v, x);
#pragma unroll
    for (int q = 0; q < R; ++q) v[q] = x[q];
}

// Where the one-wave solve leaves its results: x and (converged, corrections)
// in pinned host memory, and with wg the wing circulation of a rotor of nb
// blades (nbc of them convected) of per panels each.
struct SolveOut {
    double *x, *wg;
    int *st, per, nb, nbc;
};

template <int R, int NMAX>
__global__ __launch_bounds__(SOLVE_STAGE) void solve_wave_kernel(int n, const double *A,
                                                                 const double *LU,
                                                                 const int *perm, const double *b,
                                                                 int max_iter, double tol,
                                                                 SolveOut o)
{
    static_assert(R <= 2, "two blocks of columns");
    __shared__ double sLU[NMAX * NMAX], sA[NMAX * NMAX];
    __shared__ int sperm[NMAX];
    const int l = threadIdx.x;
    for (int k = l; k < n; k += SOLVE_STAGE) sperm[k] = perm[k];
    __syncthreads();
    // eight loads of each matrix in flight per lane
    for (int k0 = 0; k0 < n * n; k0 += 8 * SOLVE_STAGE) {
        double u[8], a[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int k = min(k0 + i * SOLVE_STAGE + l, n * n - 1), j = k / n;
            u[i] = LU[k];
            a[i] = A[sperm[k - n * j] + n * j];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int k = k0 + i * SOLVE_STAGE + l;
            if (k < n * n) {
                sLU[k] = u[i];
                sA[k] = a[i];
            }
        }
    }
    __syncthreads();
    if (l >= 64) return;
    double bl[R], xv[R], rl[R], d[R], rd[R];
    double bm = 0.0;
    bool odd = false;
#pragma unroll
    for (int q = 0; q < R; ++q) {
        const int row = l + 64 * q;
        bl[q] = row < n ? b[sperm[row]] : 0.0;
        bm = fmax(bm, fabs(bl[q]));
        xv[q] = bl[q];
        d[q] = row < n ? sLU[row + n * row] : 1.0;
        rd[q] = 1.0 / d[q];
        odd = odd || !(fabs(rd[q]) < 1e300 && fabs(rd[q]) > 1e-300);
    }
    const bool plain = __any(odd) != 0;
    const double bmax = wave_max(bm);
    wave_lu_solve<R>(n, sLU, d, rd, plain, xv);
    int conv = 0, corr = 0;
    for (int it = 0; it < max_iter; ++it) {
#pragma unroll
        for (int q = 0; q < R; ++q) rl[q] = l + 64 * q < n ? bl[q] : 0.0;
        for (int j = 0; j < n; j += 8) {
            double a[8][R];
#pragma unroll
            for (int u = 0; u < 8; ++u)
#pragma unroll
                for (int q = 0; q < R; ++q)
                    a[u][q] = sA[min(l + 64 * q, n - 1) + n * min(j + u, n - 1)];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                if (j + u >= n) break;
                const double xj = readlane_d(R == 1 || j < 64 ? xv[0] : xv[R - 1], (j + u) & 63);
                wave_column<R, 0, R - 1>(xj, a[u], rl);
            }
        }
#pragma unroll
        for (int q = 0; q < R; ++q) rl[q] = l + 64 * q < n ? rl[q] : 0.0;
        double rm = 0.0;
#pragma unroll
        for (int q = 0; q < R; ++q) rm = fmax(rm, fabs(rl[q]));
        if (wave_max(rm) <= tol * bmax) {
            conv = 1;
            break;
        }
        ++corr;
        wave_lu_solve<R>(n, sLU, d, rd, plain, rl);
#pragma unroll
        for (int q = 0; q < R; ++q) xv[q] += rl[q];
    }
#pragma unroll
    for (int q = 0; q < R; ++q)
        if (l + 64 * q < n) o.x[l + 64 * q] = xv[q];
    if (l == 0) {
        o.st[0] = conv;
        o.st[1] = corr;
    }
    if (!o.wg) return;
    // rotor_map_gam: blade 1 for every blade of an axisymmetric rotor
    for (int e = 0; e < o.per * o.nb; e += 64) {
        const int k = e + l, blade = k / o.per;
        const int src = blade < o.nbc ? k : o.nbc == 1 ? k - blade * o.per : n;
        double g = 0.0;
#pragma unroll
        for (int q = 0; q < R; ++q) {
            const double t = __shfl(xv[q], src & 63);
            if (src >> 6 == q) g = t;
        }
        if (k < o.per * o.nb && src < n) o.wg[k] = g;
    }
}

// x = A^-1 rhs by the LU factors plus up to max_iter refinement steps on
// the FP64 residual.  Everything is enqueued: the convergence test runs on
// the device (later corrections are skipped once it passes), so the only
// synchronisation is the final download.  perm: the row permutation that
// the pivots compose to.  With a rotor given,
// the solution also becomes its device wing circulation (rotor_map_gam).
int solve_refine(vlm_ctx *ctx, int n, const double *A, const double *LU, const int *perm,
                 const double *rhs_h, double *x_h, int max_iter, double tol, int *iters,
                 Rotor *rotor = nullptr, bool deferred = false)
{
    const size_t np = (size_t)(n + TB - 1) / TB * TB;
    VLM_HIP(ctx->solve_tmp.reserve((size_t)3 * n + 2 * np + 5));
    double *x = ctx->solve_tmp.p + n, *r = x + n;
    const double *b = ctx->solve_tmp.p;
    if (rhs_h) VLM_TRY(h2d(ctx, ctx->solve_tmp.p, rhs_h, sizeof(double) * n));
    else b = rotor->rhs.p;   // left on the device by vlm_rotor_rhs
    const int per = rotor ? rotor->d.nc * rotor->d.ns : 0;
    // x and (converged, corrections) on the host
    char *hp = nullptr;
    VLM_TRY(pin_take(ctx, sizeof(double) * n + 2 * sizeof(int), &hp));
    int *hst = reinterpret_cast<int *>(hp + sizeof(double) * n);
    if (n <= SOLVE_WAVE_N2) {
        SolveOut o;
        o.x = reinterpret_cast<double *>(hp);
        o.st = hst;
        o.wg = rotor ? rotor->wg.p : nullptr;
        o.per = per;
        o.nb = rotor ? rotor->d.nb : 0;
        o.nbc = rotor ? rotor->d.nbConvect : 0;
        if (n <= SOLVE_WAVE_N)
            hipLaunchKernelGGL((solve_wave_kernel<1, SOLVE_WAVE_N>), dim3(1), dim3(SOLVE_STAGE),
                               0, ctx->stream, n, A, LU, perm, b, max_iter, tol, o);
        else
            hipLaunchKernelGGL((solve_wave_kernel<2, SOLVE_WAVE_N2>), dim3(1), dim3(SOLVE_STAGE),
                               0, ctx->stream, n, A, LU, perm, b, max_iter, tol, o);
        VLM_HIP(hipGetLastError());
    } else {
        SolveWork w;
        w.y = reinterpret_cast<unsigned long long *>(r + n);
        w.z = w.y + np;
        w.rmax = w.z + np;
        w.bmax = w.rmax + 2;
        w.st = reinterpret_cast<int *>(w.bmax + 1);
        w.ticket = w.st + 2;
        const dim3 gs(2 * (unsigned)(np / TB)), gr((n + RROWS - 1) / RROWS);
        hipLaunchKernelGGL(solve_init_kernel, dim3((unsigned)((np + 255) / 256)), dim3(256), 0,
                           ctx->stream, n, b, w);
        hipLaunchKernelGGL(lu_sweeps_kernel, gs, dim3(256), 0, ctx->stream, n, LU, perm, b, x, 0,
                           0, tol, w);
        for (int it = 0; it < max_iter; ++it) {
            hipLaunchKernelGGL(residual_kernel, gr, dim3(RROWS * RSL), 0, ctx->stream, n, A, x, b,
                               r, it, w);
            hipLaunchKernelGGL(lu_sweeps_kernel, gs, dim3(256), 0, ctx->stream, n, LU, perm, r, x,
                               1, it, tol, w);
        }
        if (rotor)
            hipLaunchKernelGGL(map_gam_kernel, dim3((per * rotor->d.nb + 255) / 256), dim3(256),
                               0, ctx->stream, x, rotor->wg.p, per, rotor->d.nb,
                               rotor->d.nbConvect);
        VLM_HIP(hipGetLastError());
        VLM_HIP(hipMemcpyAsync(hp, x, sizeof(double) * n, hipMemcpyDeviceToHost, ctx->stream));
        VLM_HIP(hipMemcpyAsync(hst, w.st, 2 * sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
    }
    if (deferred) {
        if (!iters) return defer(ctx, {{x_h, hp, sizeof(double) * n}});
        return defer(ctx, {{x_h, hp, sizeof(double) * n},
                           {iters, reinterpret_cast<const char *>(hst + 1), sizeof(int)}});
    }
    VLM_TRY(sync_stream(ctx));
    std::memcpy(x_h, hp, sizeof(double) * n);
    if (iters) *iters = hst[1];
    return VLM_OK;
}

// Row permutation of a pivot sequence: row i of P b is row perm[i] of b.
// Pivots outside the matrix (a matrix of NaNs has none) move nothing.
void compose_pivots(int n, const int *piv, int *perm)
{
    for (int i = 0; i < n; ++i) perm[i] = i;
    for (int k = 0; k < n; ++k)
        if (piv[k] >= 0 && piv[k] < n) std::swap(perm[k], perm[piv[k]]);
}

// The row permutation that solve_refine reads, after the pivots and info.
const int *solve_pivots(vlm_ctx *ctx, int ir)
{
    return ctx->piv[ir] + ctx->aic_n[ir] + 1;
}

}  // namespace
}  // namespace vlm

using namespace vlm;

extern "C" {

int vlm_rotor_calc_aic(vlm_ctx *ctx, int ir, const double *cp, const double *ncap, double *Aout)
{
    if (!ctx || ir < 0 || ir >= (int)ctx->rotors.size()) return VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    if (!cp || !ncap) return fail(ctx, VLM_ERR_ARG, "null buffer");
    Rotor &r = *ctx->rotors[ir];
    const int n = r.nring;
    if (ctx->aic_n[ir] != n) {
        if (ctx->aic[ir]) (void)hipFree(ctx->aic[ir]);
        if (ctx->lu[ir]) (void)hipFree(ctx->lu[ir]);
        if (ctx->piv[ir]) (void)hipFree(ctx->piv[ir]);
        ctx->aic[ir] = ctx->lu[ir] = nullptr;
        ctx->piv[ir] = nullptr;
        VLM_HIP(hipMalloc(reinterpret_cast<void **>(&ctx->aic[ir]), sizeof(double) * n * n));
        VLM_HIP(hipMalloc(reinterpret_cast<void **>(&ctx->lu[ir]), sizeof(double) * n * n));
        VLM_HIP(hipMalloc(reinterpret_cast<void **>(&ctx->piv[ir]), sizeof(int) * (2 * n + 1)));
        ctx->aic_n[ir] = n;
    }
    VLM_HIP(ctx->hostio.reserve((size_t)6 * n));
    double *geo = ctx->hostio.p;
    VLM_TRY(h2d(ctx, geo, cp, sizeof(double) * 3 * n));
    VLM_TRY(h2d(ctx, geo + 3 * n, ncap, sizeof(double) * 3 * n));
    const int64_t nn = (int64_t)n * n;
    hipLaunchKernelGGL(aic_kernel, dim3((unsigned)((nn + 255) / 256)), dim3(256), 0, ctx->stream,
                       n, r.wc.p, r.wrc.p, geo, geo + 3 * n, ctx->aic[ir]);
    VLM_HIP(hipGetLastError());
    VLM_HIP(hipMemcpyAsync(ctx->lu[ir], ctx->aic[ir], sizeof(double) * nn,
                           hipMemcpyDeviceToDevice, ctx->stream));
    VLM_TRY(lu_factor_device(ctx, n, ctx->lu[ir], ctx->piv[ir], ctx->piv[ir] + n));
    std::vector<int> piv((size_t)2 * n + 1);   // pivots, info, row permutation
    char *hp = nullptr;
    VLM_TRY(pin_take(ctx, sizeof(int) * (n + 1), &hp));
    VLM_HIP(hipMemcpyAsync(hp, ctx->piv[ir], sizeof(int) * (n + 1), hipMemcpyDeviceToHost,
                           ctx->stream));
    VLM_TRY(sync_stream(ctx));
    std::memcpy(piv.data(), hp, sizeof(int) * (n + 1));
    if (Aout) VLM_TRY(d2h(ctx, Aout, ctx->aic[ir], sizeof(double) * nn));
    const int info = piv[n];
    compose_pivots(n, piv.data(), piv.data() + n + 1);
    VLM_TRY(h2d(ctx, ctx->piv[ir] + n + 1, piv.data() + n + 1, sizeof(int) * n));
    if (info != 0) return fail(ctx, VLM_ERR_SINGULAR, "AIC is singular (zero pivot)");
    return VLM_OK;
}

int vlm_rotor_solve(vlm_ctx *ctx, int ir, const double *rhs, double *gam, int max_iter,
                    double tol, int *iters)
{
    if (!ctx || ir < 0 || ir >= (int)ctx->rotors.size()) return VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    if (!rhs || !gam) return fail(ctx, VLM_ERR_ARG, "null buffer");
    if (!ctx->lu[ir]) return fail(ctx, VLM_ERR_STATE, "vlm_rotor_calc_aic not called");
    const int n = ctx->aic_n[ir];
    return solve_refine(ctx, n, ctx->aic[ir], ctx->lu[ir], solve_pivots(ctx, ir), rhs, gam, max_iter,
                        tol, iters, ctx->rotors[ir]);
}

int vlm_rotor_solve_deferred(vlm_ctx *ctx, int ir, const double *rhs, double *gam, int max_iter,
                             double tol, int *iters)
{
    if (!ctx || ir < 0 || ir >= (int)ctx->rotors.size()) return VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    if (!gam) return fail(ctx, VLM_ERR_ARG, "null buffer");
    if (!ctx->lu[ir]) return fail(ctx, VLM_ERR_STATE, "vlm_rotor_calc_aic not called");
    if (!rhs && !ctx->rotors[ir]->panels_set)
        return fail(ctx, VLM_ERR_STATE, "no right-hand side on the device (vlm_rotor_rhs)");
    const int n = ctx->aic_n[ir];
    return solve_refine(ctx, n, ctx->aic[ir], ctx->lu[ir], solve_pivots(ctx, ir), rhs, gam, max_iter,
                        tol, iters, ctx->rotors[ir], true);
}

int vlm_lu_factor(vlm_ctx *ctx, int n, double *A, int *ipiv)
{
    if (!ctx || n <= 0 || !A || !ipiv) return VLM_ERR_ARG;
    VLM_DEVICE(ctx);
    const Trim trim{ctx};
    const size_t nn = (size_t)n * n;
    VLM_HIP(ctx->hostio.reserve(nn));
    VLM_HIP(ctx->hostio_i.reserve((size_t)n + 1));
    double *dA = ctx->hostio.p;
    int *dp = ctx->hostio_i.p;
    VLM_TRY(h2d(ctx, dA, A, sizeof(double) * nn));
    VLM_TRY(lu_factor_device(ctx, n, dA, dp, dp + n));
    std::vector<int> piv((size_t)n + 1);   // pivots, info
    VLM_TRY(d2h(ctx, A, dA, sizeof(double) * nn));
    VLM_TRY(d2h(ctx, piv.data(), dp, sizeof(int) * (n + 1)));
    std::memcpy(ipiv, piv.data(), sizeof(int) * n);
    const int info = piv[n];
    if (info != 0) return fail(ctx, VLM_ERR_SINGULAR, "matrix is singular (zero pivot)");
    return VLM_OK;
}

int vlm_lu_solve_refine(vlm_ctx *ctx, int n, const double *A, const double *LU, const int *ipiv,
                        const double *rhs, double *x, int max_iter, double tol, int *iters)
{
    if (!ctx || n <= 0 || !A || !LU || !ipiv || !rhs || !x) return VLM_ERR_ARG;
    for (int k = 0; k < n; ++k)
        if (ipiv[k] < 0 || ipiv[k] >= n) return fail(ctx, VLM_ERR_ARG, "pivot out of range");
    std::vector<int> perm((size_t)n);
    compose_pivots(n, ipiv, perm.data());
    VLM_DEVICE(ctx);
    const Trim trim{ctx};
    const size_t nn = (size_t)n * n;
    VLM_HIP(ctx->hostio.reserve(2 * nn));
    VLM_HIP(ctx->hostio_i.reserve((size_t)n + 1));
    double *dA = ctx->hostio.p, *dLU = dA + nn;
    int *dp = ctx->hostio_i.p;
    VLM_TRY(h2d(ctx, dA, A, sizeof(double) * nn));
    VLM_TRY(h2d(ctx, dLU, LU, sizeof(double) * nn));
    VLM_TRY(h2d(ctx, dp, perm.data(), sizeof(int) * n));
    return solve_refine(ctx, n, dA, dLU, dp, rhs, x, max_iter, tol, iters);
}

}  // extern "C"
