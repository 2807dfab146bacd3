// qrot_sweep.hip -- the QROT dual objective, its gradient and the primal value
// of the rounded plan, as sweeps over the cost matrix with
// D_ij = (alpha_i + beta_j - M_ij)_+ (src/qrot_problem.cpp:37-96, :10-26).
//
//   objective   sum of D^2; with the gradient also the row and column sums of D;
//   rounding    (approx_proj, src/approx_proj.h:6-26, of T = D / reg)
//     x = min(a / T1, 1)                the objective sweep's row sums give it
//     c = T'x, y = min(b / c, 1)        second sweep: column sums
//     err_b = b - y c
//     err_a = a - diag(x) T y           third sweep: row sums, and with them
//     <P, M> and ||P||^2 of P = diag(x) T diag(y) + err_a err_b' / |err_a|_1:
//       <P, M>  = sum xTyM + sum_i err_a_i (M err_b)_i / l1
//       ||P||^2 = sum (xTy)^2 + 2 sum_i err_a_i (xTy err_b)_i / l1
//                 + ||err_a||^2 ||err_b||^2 / l1^2.
//   T is never divided element by element: 1 / reg is applied to the sums.
//
// A workgroup (4 waves) takes a strip of 256 C columns (lane l: the quads at
// 256 c + 4 l) over `rows` rows, each wave R rows at a time.  A row's sum
// crosses the lanes once per 256 C columns (one 256-column strip per wave
// spent more on the cross-lane steps than on the elements).  Bound by the read
// of M (268 MB at 8192^2 FP32: 42 us at the 6.4 TB/s of a bare read) and, in
// the first and third sweep, by the FP64 work and the row sums beside it.
// Measured there, per history entry with its primal value: 73 us (objective) +
// 79 + 2 x 94 + 102 us (rounding) in five sweeps before; 60 (objective) + 44 +
// 69 us now.  Every reduction has a fixed order.
#include <algorithm>
#include <cmath>
#include <memory>

#include "dense_device.hpp"
#include "problem.hpp"
#include "qrot.hpp"

namespace regot {
namespace {

using namespace dev;

enum { SW_GRAD = 0, SW_OBJ = 1, SW_COLS = 2, SW_LAST = 3 };

// Four adjacent entries of a row: one 16-byte load (FP32) or two (FP64).
template <typename TM>
struct Quad;
template <>
struct Quad<float> {
    float4 a;
    __device__ __forceinline__ void load(const float* p, int o0, int, bool nt)
    {
        a = ld_m(p + o0, nt);
    }
    __device__ __forceinline__ float raw(int q) const { return vget<float4, float>(a, q); }
};
template <>
struct Quad<double> {
    double2 a, b;
    __device__ __forceinline__ void load(const double* p, int o0, int o1, bool nt)
    {
        a = ld_m(p + o0, nt);
        b = ld_m(p + o1, nt);
    }
    __device__ __forceinline__ double raw(int q) const
    {
        return q < 2 ? vget<double2, double>(a, q) : vget<double2, double>(b, q - 2);
    }
};

template <typename TM, int MODE, int C, int R, bool NT>
__global__ __launch_bounds__(256) void k_qrot_sweep(
    const TM* __restrict__ M, long ldm, int n, int m, const double* __restrict__ alpha,
    const double* __restrict__ beta, const double* __restrict__ x, const double* __restrict__ y,
    const double* __restrict__ eb, int rows, double* __restrict__ rowpart,
    double* __restrict__ colpart, double* __restrict__ scal)
{
    constexpr bool COLS = MODE == SW_GRAD || MODE == SW_COLS;
    constexpr int NR = MODE == SW_GRAD ? 1 : MODE == SW_LAST ? 3 : 0;   // sums per row
    constexpr int NS = MODE == SW_LAST ? 2 : MODE == SW_COLS ? 0 : 1;   // scalars
    __shared__ double red[COLS ? 4 : 1][COLS ? 256 * C : 1];
    __shared__ double ss[4][2];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int strip = blockIdx.x, blk = blockIdx.y;
    const int r0 = blk * rows;
    const int r1 = min(n, r0 + rows);

    // Columns past m have potential -inf: D = 0.  A vector with no column reads
    // the row's first instead, so that every load is unconditional.
    int o0[C], o1[C];
    double b[C][4], yq[C][4], eq[C][4], cs[C][4];
    bool in[C][4];
#pragma unroll
    for (int c = 0; c < C; c++) {
        const int j0 = (strip * C + c) * 256 + 4 * lane;
        o0[c] = j0 < m ? j0 : 0;
        o1[c] = j0 + 2 < m ? j0 + 2 : 0;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int j = j0 + q;
            in[c][q] = j < m;
            const int jc = j < m ? j : m - 1;
            b[c][q] = in[c][q] ? beta[jc] : -INFINITY;
            if (MODE == SW_LAST) {
                yq[c][q] = in[c][q] ? y[jc] : 0.0;
                eq[c][q] = in[c][q] ? eb[jc] : 0.0;
            }
            if (COLS) cs[c][q] = 0.0;
        }
    }
    double s1 = 0.0, s2 = 0.0;
    for (int r = r0 + wave * R; r < r1; r += 4 * R) {
        Quad<TM> mv[R][C];
        double ai[R], xi[R];
#pragma unroll
        for (int k = 0; k < R; k++) {
            const int i = r + k < r1 ? r + k : r1 - 1;
            const TM* Mi = M + static_cast<long>(i) * ldm;
#pragma unroll
            for (int c = 0; c < C; c++) mv[k][c].load(Mi, o0[c], o1[c], NT);
            // rows past the block: D = 0
            ai[k] = r + k < r1 ? alpha[i] : -INFINITY;
            if (MODE == SW_COLS || MODE == SW_LAST) xi[k] = x[i];
        }
        double rs[R * (NR > 0 ? NR : 1)];
#pragma unroll
        for (int k = 0; k < R; k++) {
            double A = 0.0, B = 0.0, E = 0.0, u1 = 0.0, u2 = 0.0;
#pragma unroll
            for (int c = 0; c < C; c++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    TM raw = mv[k][c].raw(q);
                    // outside the matrix: what lies there must not meet err_b = 0
                    if (MODE == SW_LAST) raw = in[c][q] ? raw : TM(0);
                    const double v = static_cast<double>(raw);
                    const double d = fmax((ai[k] + b[c][q]) - v, 0.0);
                    if (MODE == SW_GRAD) {
                        A += d;
                        cs[c][q] += d;
                    }
                    if (MODE == SW_GRAD || MODE == SW_OBJ) s1 = fma(d, d, s1);
                    if (MODE == SW_COLS) cs[c][q] = fma(d, xi[k], cs[c][q]);
                    if (MODE == SW_LAST) {
                        const double t = d * yq[c][q];
                        A += t;
                        B = fma(eq[c][q], v, B);
                        E = fma(t, eq[c][q], E);
                        // an infinite M has D = 0, whose product must be 0
                        u1 = fma(t, fmin(v, 0x1.fffffffffffffp1023), u1);
                        u2 = fma(t, t, u2);
                    }
                }
            if (NR >= 1) rs[k * NR] = A;
            if (NR == 3) {
                rs[k * NR + 1] = B;
                rs[k * NR + 2] = E;
                s1 = fma(xi[k], u1, s1);
                s2 = fma(xi[k] * xi[k], u2, s2);
            }
        }
        if (NR > 0) {
            wave_sums<R * (NR > 0 ? NR : 1)>(rs);
            if (lane == 0)
#pragma unroll
                for (int k = 0; k < R; k++)
                    if (r + k < r1)
#pragma unroll
                        for (int q = 0; q < NR; q++)
                            rowpart[(static_cast<long>(q) * gridDim.x + strip) * n + r + k] =
                                rs[k * NR + q];
        }
    }
    if (COLS) {
#pragma unroll
        for (int c = 0; c < C; c++)
#pragma unroll
            for (int q = 0; q < 4; q++) red[wave][256 * c + 4 * lane + q] = cs[c][q];
    }
    if (NS > 0) {
        s1 = wave_sum0(s1);
        if (NS > 1) s2 = wave_sum0(s2);
        if (lane == 0) {
            ss[wave][0] = s1;
            ss[wave][1] = s2;
        }
    }
    __syncthreads();
    if (COLS)
        for (int t = threadIdx.x; t < 256 * C; t += 256) {
            const int j = strip * 256 * C + t;
            if (j < m)
                colpart[static_cast<long>(blk) * m + j] =
                    ((red[0][t] + red[1][t]) + red[2][t]) + red[3][t];
        }
    if (threadIdx.x < NS) {
        const int q = threadIdx.x;
        scal[NS * (static_cast<long>(blk) * gridDim.x + strip) + q] =
            ((ss[0][q] + ss[1][q]) + ss[2][q]) + ss[3][q];
    }
}

// Sum over np partials (stride apart) of entry t, by the 4 waves of a workgroup
// for its 64 entries: wave w takes partials w, w + 4, ... with eight loads in
// flight; the result is on wave 0's lanes.
__device__ __forceinline__ double fold64(const double* __restrict__ p, int np, long stride,
                                         bool valid, int wave, int lane, double (*sm)[64])
{
    double v = 0.0;
    if (valid) {
        int s = wave;
        for (; s + 28 < np; s += 32) {
            double u[8];
#pragma unroll
            for (int k = 0; k < 8; k++) u[k] = p[(s + 4 * k) * stride];
#pragma unroll
            for (int k = 0; k < 8; k++) v += u[k];
        }
        for (; s < np; s += 4) v += p[s * stride];
    }
    __syncthreads();   // sm may still be read from the fold before
    sm[wave][lane] = v;
    __syncthreads();
    return wave == 0 ? ((sm[0][lane] + sm[1][lane]) + sm[2][lane]) + sm[3][lane] : 0.0;
}

// Entries 0..n-1: rows, n..n+m-1: columns.  Row and column sums of D (with
// rsum), the rounding's row scales x, the gradient (tau = 0) and per workgroup
// {sum g^2, alpha'a + beta'b, 1'alpha, 1'beta}.
__global__ __launch_bounds__(256) void k_qrot_obj_fold(
    const double* __restrict__ rowpart, int nstrip, const double* __restrict__ colpart, int nblk,
    const double* __restrict__ alpha, const double* __restrict__ beta,
    const double* __restrict__ a, const double* __restrict__ bm, int n, int m, double reg,
    double* __restrict__ rsum, double* __restrict__ csum, double* __restrict__ x,
    double* __restrict__ grad, double* __restrict__ part)
{
    __shared__ double sm[4][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long blk = static_cast<long>(blockIdx.y) * gridDim.x + blockIdx.x;   // wide_grid
    const long e = blk * 64 + lane;
    const bool row = e < n;
    const bool valid = e < static_cast<long>(n) + m;
    if (blk * 64 >= static_cast<long>(n) + m) return;
    double v = 0.0;
    if (rsum)
        v = fold64(row ? rowpart + e : colpart + (e - n), row ? nstrip : nblk, row ? n : m, valid,
                   wave, lane, sm);
    if (wave != 0) return;
    double w[4] = {0.0, 0.0, 0.0, 0.0};
    if (valid) {
        const double target = row ? a[e] : bm[e - n];
        const double pot = row ? alpha[e] : beta[e - n];
        if (rsum) {
            if (row) {
                rsum[e] = v;
                x[e] = fmin(target / (v / reg), 1.0);
            } else {
                csum[e - n] = v;
            }
            const double g = v - reg * target;
            if (grad) grad[e] = g;
            w[0] = g * g;
        }
        w[1] = pot * target;
        w[2] = row ? pot : 0.0;
        w[3] = row ? 0.0 : pot;
    }
    wave_sums<4>(w);
    if (lane == 0) {
#pragma unroll
        for (int q = 0; q < 4; q++) part[4 * blk + q] = w[q];
    }
}

// Sums of `count` groups of NV doubles by one workgroup of 256, on every thread.
template <int NV>
__device__ __forceinline__ void total256(const double* __restrict__ p, int count, double (&v)[NV])
{
#pragma unroll
    for (int q = 0; q < NV; q++) v[q] = 0.0;
    for (int i = threadIdx.x; i < count; i += 256)
#pragma unroll
        for (int q = 0; q < NV; q++) v[q] += p[static_cast<long>(i) * NV + q];
    block_sums_256<NV>(v);
}

// out = {f, ||g||^2, sum D^2}, f = 0.5 sum D^2 - reg (alpha'a + beta'b)
//       + tau/2 (1'alpha - 1'beta)^2.
__global__ __launch_bounds__(256) void k_qrot_obj_total(const double* __restrict__ part, int np,
                                                        const double* __restrict__ sq, int nsq,
                                                        double reg, double tau,
                                                        double* __restrict__ out)
{
    double v[4], s[1];
    total256<4>(part, np, v);
    total256<1>(sq, nsq, s);
    if (threadIdx.x == 0) {
        const double d = v[2] - v[3];
        double f = 0.5 * s[0] - reg * v[1];
        if (tau > 0.0) f += 0.5 * tau * d * d;
        out[0] = f;
        out[1] = v[0];
        out[2] = s[0];
    }
}

// y = min(b / c, 1), err_b = b - y c, c = column sums / reg; ||err_b||^2 per
// workgroup.
__global__ __launch_bounds__(256) void k_qrot_cols_fold(const double* __restrict__ colpart,
                                                        int nblk, const double* __restrict__ b,
                                                        int m, double reg, double* __restrict__ y,
                                                        double* __restrict__ eb,
                                                        double* __restrict__ part)
{
    __shared__ double sm[4][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long blk = static_cast<long>(blockIdx.y) * gridDim.x + blockIdx.x;   // wide_grid
    const long j = blk * 64 + lane;
    if (blk * 64 >= m) return;
    const double v = fold64(colpart + j, nblk, m, j < m, wave, lane, sm);
    if (wave != 0) return;
    double w = 0.0;
    if (j < m) {
        const double c = v / reg;
        const double yj = fmin(b[j] / c, 1.0);
        const double e = b[j] - yj * c;
        y[j] = yj;
        eb[j] = e;
        w = e * e;
    }
    w = wave_sum0(w);
    if (lane == 0) part[blk] = w;
}

// err_a = a - x A / reg; per workgroup {|err_a|_1, ||err_a||^2,
// sum err_a (M err_b), sum err_a (xTy err_b)}.
__global__ __launch_bounds__(256) void k_qrot_rows_fold(const double* __restrict__ rowpart,
                                                        int nstrip, const double* __restrict__ a,
                                                        const double* __restrict__ x, int n,
                                                        double reg, double* __restrict__ part)
{
    __shared__ double sm[4][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long blk = static_cast<long>(blockIdx.y) * gridDim.x + blockIdx.x;   // wide_grid
    const long i = blk * 64 + lane;
    if (blk * 64 >= n) return;
    const long plane = static_cast<long>(nstrip) * n;
    const double A = fold64(rowpart + i, nstrip, n, i < n, wave, lane, sm);
    const double B = fold64(rowpart + plane + i, nstrip, n, i < n, wave, lane, sm);
    const double E = fold64(rowpart + 2 * plane + i, nstrip, n, i < n, wave, lane, sm);
    if (wave != 0) return;
    double w[4] = {0.0, 0.0, 0.0, 0.0};
    if (i < n) {
        const double ea = a[i] - x[i] * A / reg;
        w[0] = fabs(ea);
        w[1] = ea * ea;
        w[2] = ea * B;
        w[3] = ea * (x[i] * E / reg);
    }
    wave_sums<4>(w);
    if (lane == 0) {
#pragma unroll
        for (int q = 0; q < 4; q++) part[4 * blk + q] = w[q];
    }
}

// out = {<P, M>, ||P||^2}.
__global__ __launch_bounds__(256) void k_qrot_round_total(
    const double* __restrict__ scal, int nscal, const double* __restrict__ rpart, int nr,
    const double* __restrict__ cpart, int nc, double reg, double* __restrict__ out)
{
    double s[2], v[4], e[1];
    total256<2>(scal, nscal, s);
    total256<4>(rpart, nr, v);
    total256<1>(cpart, nc, e);
    if (threadIdx.x == 0) {
        const double l1 = v[0];
        out[0] = s[0] / reg + v[2] / l1;
        out[1] = s[1] / (reg * reg) + 2.0 * v[3] / l1 + (v[1] / l1) * (e[0] / l1);
    }
}

// Quads per lane.  Measured at 8192^2 FP32 with 2 / 4: gradient 62 / 67 us (4
// leaves 3 waves per SIMD), third sweep 69 / 84, column sweep 53 / 44 (no row
// sums, and half the column partials).  Four rows at a time instead of two:
// gradient 60.
int sweep_c(int m, int mode)
{
    if (mode == SW_COLS && m >= 1536) return 4;
    return m >= 320 ? 2 : 1;
}

// About 1024 workgroups, 16 rows (4 per wave) at least.
int sweep_rows(int n, int m, int mode)
{
    const int strips = ceil_div(m, 256 * sweep_c(m, mode));
    int rows = 16;
    while (rows < 512 && static_cast<long>(strips) * ceil_div(n, rows * 2) >= 1024) rows *= 2;
    return rows;
}

struct SweepGrid {
    int strips, blocks;
};
SweepGrid sweep_grid(int n, int m, int mode)
{
    return {ceil_div(m, 256 * sweep_c(m, mode)), ceil_div(n, sweep_rows(n, m, mode))};
}

template <typename TM, int MODE>
void sweep(regot_problem* p, const double* alpha, const double* beta, const QrotScratch& w,
           double* rowpart, double* colpart, double* scal)
{
    const int n = p->n, m = p->m;
    const int rows = sweep_rows(n, m, MODE);
    const SweepGrid sg = sweep_grid(n, m, MODE);
    const bool nt = static_cast<long>(n) * p->ldm * static_cast<long>(sizeof(TM)) > (256L << 20);
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(sg.strips, sg.blocks), dim3(256), 0, p->stream,
                           static_cast<const TM*>(p->dM), p->ldm, n, m, alpha, beta, w.x.p, w.y.p,
                           w.eb.p, rows, rowpart, colpart, scal);
        KERNEL_CHECK();
    };
    constexpr int RW = MODE == SW_GRAD ? 4 : 2;
    const int C = sweep_c(m, MODE);
    if (C == 1)
        nt ? go(k_qrot_sweep<TM, MODE, 1, 4, true>) : go(k_qrot_sweep<TM, MODE, 1, 4, false>);
    else if (C == 2)
        nt ? go(k_qrot_sweep<TM, MODE, 2, RW, true>) : go(k_qrot_sweep<TM, MODE, 2, RW, false>);
    else if constexpr (MODE == SW_COLS)
        nt ? go(k_qrot_sweep<TM, MODE, 4, 2, true>) : go(k_qrot_sweep<TM, MODE, 4, 2, false>);
}

template <int MODE>
void sweep_any(regot_problem* p, const double* alpha, const double* beta, const QrotScratch& w,
               double* rowpart, double* colpart, double* scal)
{
    if (p->bulk == 0)
        sweep<float, MODE>(p, alpha, beta, w, rowpart, colpart, scal);
    else
        sweep<double, MODE>(p, alpha, beta, w, rowpart, colpart, scal);
}

}  // namespace

void qrot_sweep_sizes(int n, int m, size_t* rowpart, size_t* colpart, size_t* scal)
{
    *rowpart = *colpart = *scal = 0;
    for (int mode : {SW_GRAD, SW_OBJ, SW_COLS, SW_LAST}) {
        const SweepGrid g = sweep_grid(n, m, mode);
        const size_t sums = mode == SW_LAST ? 3 : 1;
        *rowpart = std::max(*rowpart, sums * g.strips * n);
        *colpart = std::max(*colpart, static_cast<size_t>(g.blocks) * m);
        *scal = std::max(*scal, 2 * static_cast<size_t>(g.strips) * g.blocks);
    }
}

double qrot_obj_grad(regot_problem* p, const double* gamma, double* grad, double tau,
                     double* gnorm2)
{
    const int n = p->n, m = p->m;
    hipStream_t s = p->stream;
    if (!p->qrot) p->qrot = std::make_unique<QrotScratch>(n, m);
    QrotScratch& w = *p->qrot;
    const SweepGrid g = sweep_grid(n, m, grad ? SW_GRAD : SW_OBJ);
    const double* alpha = gamma;
    const double* beta = gamma + n;
    const int ne = ceil_div(static_cast<long>(n) + m, 64);
    if (grad)
        sweep_any<SW_GRAD>(p, alpha, beta, w, w.rowpart, w.colpart, w.sqpart);
    else
        sweep_any<SW_OBJ>(p, alpha, beta, w, nullptr, nullptr, w.sqpart);
    hipLaunchKernelGGL(k_qrot_obj_fold, wide_grid(ne), dim3(256), 0, s, w.rowpart.p, g.strips,
                       w.colpart.p, g.blocks, alpha, beta, p->a.p, p->b.p, n, m, p->reg,
                       grad ? w.rsum.p : nullptr, w.csum.p, w.x.p,
                       grad && !(tau > 0.0) ? grad : nullptr, w.epart.p);
    hipLaunchKernelGGL(k_qrot_obj_total, dim3(1), dim3(256), 0, s, w.epart.p, ne, w.sqpart.p,
                       g.strips * g.blocks, p->reg, tau,
                       grad && tau > 0.0 ? w.out.p : p->mscal.d);
    KERNEL_CHECK();
    if (grad && tau > 0.0)   // the gradient's tau term needs 1'alpha - 1'beta first
        launch_qrot_finish(alpha, beta, p->a, p->b, n, m, p->reg, tau, w.out.p + 2, w.rsum,
                           w.csum, grad, w.fpart, w.gpart, p->mscal.d, s);
    HIP_CHECK(hipStreamSynchronize(s));
    if (gnorm2) *gnorm2 = p->mscal.h[1];
    return p->mscal.h[0];
}

double qrot_primal(regot_problem* p, const double* alpha, const double* beta, bool fresh)
{
    const int n = p->n, m = p->m;
    hipStream_t s = p->stream;
    if (!p->qrot) p->qrot = std::make_unique<QrotScratch>(n, m);
    QrotScratch& w = *p->qrot;
    if (!fresh) {
        const SweepGrid g = sweep_grid(n, m, SW_GRAD);
        sweep_any<SW_GRAD>(p, alpha, beta, w, w.rowpart, w.colpart, w.sqpart);
        const int ne = ceil_div(static_cast<long>(n) + m, 64);
        hipLaunchKernelGGL(k_qrot_obj_fold, wide_grid(ne), dim3(256), 0, s, w.rowpart.p, g.strips,
                           w.colpart.p, g.blocks, alpha, beta, p->a.p, p->b.p, n, m, p->reg, w.rsum.p,
                           w.csum.p, w.x.p, static_cast<double*>(nullptr), w.epart.p);
        KERNEL_CHECK();
    }
    const int nc = ceil_div(m, 64), nr = ceil_div(n, 64);
    sweep_any<SW_COLS>(p, alpha, beta, w, nullptr, w.colpart, nullptr);
    hipLaunchKernelGGL(k_qrot_cols_fold, wide_grid(nc), dim3(256), 0, s, w.colpart.p,
                       sweep_grid(n, m, SW_COLS).blocks, p->b.p, m, p->reg, w.y.p, w.eb.p, w.cpart.p);
    KERNEL_CHECK();
    const SweepGrid g = sweep_grid(n, m, SW_LAST);
    sweep_any<SW_LAST>(p, alpha, beta, w, w.rowpart, nullptr, w.scal);
    hipLaunchKernelGGL(k_qrot_rows_fold, wide_grid(nr), dim3(256), 0, s, w.rowpart.p, g.strips, p->a.p,
                       w.x.p, n, p->reg, w.epart.p);
    hipLaunchKernelGGL(k_qrot_round_total, dim3(1), dim3(256), 0, s, w.scal.p, g.strips * g.blocks,
                       w.epart.p, nr, w.cpart.p, nc, p->reg, p->mscal.d);
    KERNEL_CHECK();
    HIP_CHECK(hipStreamSynchronize(s));
    return p->mscal.h[0] + 0.5 * p->reg * p->mscal.h[1];
}

}  // namespace regot
