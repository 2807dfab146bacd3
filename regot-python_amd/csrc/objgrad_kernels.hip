// objgrad_kernels.hip -- objective and gradient of the dual in one pass over M.
//
// f(gamma) = reg sum_ij T_ij - alpha'a - betat'bt and
// g = [T 1 - a ; (T' 1 - b)_{0..m-2}],  T_ij = 2^((alpha_i + beta_j - M_ij) k),
// k = log2(e) / reg, in FP64 throughout (src/sinkhorn_problem_obj.cpp:139-297,
// 324-393 form the same T with FP64 exp and sum it in FP64; no shift is
// applied there either, so overflow and underflow behave alike).  2^x is the
// table-driven FP64 exp2 of dexp2.hpp (about 0.5 ulp), several times cheaper
// than the library routine, which bounded this pass by FP64 issue rate.
//
// The row and column sums come out of the same read of M, so each T_ij is
// formed once (the FP64 exponential is the expensive part of this pass).
// Tiling: a workgroup owns a 256-column strip of a block of rows; each lane
// owns 4 adjacent columns and the 4 waves take the block's rows round robin
// (coalesced row segments).  Row sums are reduced
// across the wave eight rows at a time and written per strip, column sums
// accumulate per lane down the block and are merged through LDS per block; two small
// kernels fold strips, blocks and the scalars in a fixed order.
#include <algorithm>

#include "dense_device.hpp"
#include "dexp2.hpp"
#include "problem.hpp"

namespace regot {
namespace {

// Wave sum by DPP and shuffle steps (the same bits on every lane).
__device__ __forceinline__ double wsum(double v) { return dev::group_sum<64>(v); }

// Columns per lane.  8 would spread each row's wave sum over twice the
// elements but needs 88 VGPRs, 5 waves per SIMD: measured slower (objective
// call at 16384^2 316 against 297 us, at 4096^2 61.5 against 51.0 us, with the
// wave sum per row).
constexpr int kCPL = 4;
constexpr int kStrip = 64 * kCPL;     // columns per workgroup strip

// Rows of a wave whose sums are formed together, and the pitch in doubles of
// their lane sums in LDS: 528 bytes put the 64 reads of 16 bytes of a
// reduction step on all banks evenly.
constexpr int kRowsTog = 8;
constexpr int kLanePitch = 66;

template <bool NT, typename V>
__device__ __forceinline__ V ldv(const V* p)
{
    return NT ? __builtin_nontemporal_load(p) : *p;
}

// Four columns of a row from c0 on; FULL: all of them are inside the matrix.
template <bool FULL, bool NT>
__device__ __forceinline__ void ldm4(const float* p, int c0, int m, float (&v)[4])
{
    if (FULL || c0 + 3 < m) {
        typedef float f4 __attribute__((ext_vector_type(4)));
        const f4 u = ldv<NT>(reinterpret_cast<const f4*>(p + c0));
        v[0] = u.x;
        v[1] = u.y;
        v[2] = u.z;
        v[3] = u.w;
    } else {
#pragma unroll
        for (int q = 0; q < 4; q++) v[q] = (c0 + q < m) ? p[c0 + q] : 0.f;
    }
}

template <bool FULL, bool NT>
__device__ __forceinline__ void ldm4(const double* p, int c0, int m, double (&v)[4])
{
    if (FULL || c0 + 3 < m) {
        typedef double d2 __attribute__((ext_vector_type(2)));
        const d2 u0 = ldv<NT>(reinterpret_cast<const d2*>(p + c0));
        const d2 u1 = ldv<NT>(reinterpret_cast<const d2*>(p + c0 + 2));
        v[0] = u0.x;
        v[1] = u0.y;
        v[2] = u1.x;
        v[3] = u1.y;
    } else {
#pragma unroll
        for (int q = 0; q < 4; q++) v[q] = (c0 + q < m) ? p[c0 + q] : 0.0;
    }
}

// alpha k64 + bk: one rounding on full strips, two on a ragged last one.  (The
// two forms agree to an ulp; which one is used is fixed here because an L-BFGS
// path follows the last bit.)
template <bool FULL>
__device__ __forceinline__ double row_col(double alpha, double k64, double bk)
{
#pragma clang fp contract(off)
    if (FULL) return fma(alpha, k64, bk);
    const double ak = alpha * k64;
    return ak + bk;
}

// The rows r, r + 4, ... < r1 of one tile (r the same on the whole wave):
// FULL = every column of the strip is inside the matrix (no per-element
// bounds), WT = weights x, y present.  Eight rows at a time: each lane leaves
// its four-column sum of every row in the wave's own LDS (lw), then lane 8 q + s
// adds row q's sums of lanes 8 s .. 8 s + 7 and three DPP steps finish the
// eight rows together: 16 VALU instructions for what took 18 per row, with
// the same pairing of lanes (1, 2, 4 apart, then 8, 16, 32) and so the same
// bits.
template <typename TM, bool FULL, bool WT, bool NT>
__device__ __forceinline__ void sums_rows_loop(const TM* __restrict__ M, long ldm, int n, int m,
                                               const double* __restrict__ alpha, double k64,
                                               const double* __restrict__ xw, int c0, int r, int r1,
                                               int strip, const double (&bk)[kCPL],
                                               const double (&yq)[kCPL], const double* tab,
                                               double* lw, double (&cs)[kCPL],
                                               double* __restrict__ rowpart)
{
    // Two rows per trip take turns in the two buffers.  That costs 10 more VGPRs
    // (70, 7 waves per SIMD): 210 against 235 us at 16384^2 FP32, where the issue
    // rate bounds, but 136 against 126 us at 8192^2 FP64, where the read does.
    constexpr int PAIR = (sizeof(TM) == 4 && !WT) ? 2 : 1;
    const int lane = threadIdx.x & 63;
    TM mv[2][kCPL];   // this row and the wave's next
    if (r < r1) ldm4<FULL, NT>(M + r * ldm, c0, m, mv[0]);
    for (; r < r1; r += 4 * kRowsTog) {
        const int cnt = min(kRowsTog, (r1 - r + 3) >> 2);
        // alpha of the eight rows on lanes 0 .. 7
        const double al = alpha[r + 4 * min(lane & 7, cnt - 1)];
#pragma unroll 1
        for (int h0 = 0; h0 < cnt; h0 += PAIR)
#pragma unroll
        for (int u = 0; u < PAIR; u++) {
            const int h = h0 + u;
            if (h >= cnt) break;   // wave-uniform
            // (the last row reads itself again)
            const int i = r + 4 * h;
            ldm4<FULL, NT>(M + static_cast<long>(i + 4 < r1 ? i + 4 : i) * ldm, c0, m, mv[1 - u]);
            const double ai = __hiloint2double(
                __builtin_amdgcn_readlane(__double2hiint(al), h),
                __builtin_amdgcn_readlane(__double2loint(al), h));
            double y[kCPL];
            bool far = false;
#pragma unroll
            for (int q = 0; q < kCPL; q++) {
                // 64 (alpha_i + beta_j - M_ij) / reg in log2 units
                y[q] = fma(-k64, static_cast<double>(mv[u][q]), row_col<FULL>(ai, k64, bk[q]));
                far = far || fabs(y[q]) >= dev::kExp2Fast;
            }
            if (__any(far)) {   // wave-uniform; NaN stays
#pragma unroll
                for (int q = 0; q < kCPL; q++) {
                    const double c = fmin(fmax(y[q], -70400.0), 70400.0);
                    y[q] = (y[q] != y[q]) ? y[q] : c;
                }
            }
            double rs = 0.0;
#pragma unroll
            for (int q = 0; q < kCPL; q++) {
                if (FULL || c0 + q < m) {
                    double t = dev::dexp2_64_fast(y[q], tab);
                    if (WT) t *= (xw ? xw[i] : 1.0) * yq[q];
                    rs = (q == 0 && !WT) ? t : rs + t;
                    cs[q] += t;
                }
            }
            lw[h * kLanePitch + lane] = rs;
            if (PAIR == 1)
#pragma unroll
                for (int q = 0; q < kCPL; q++) mv[0][q] = mv[1][q];
        }
        // the wave's LDS stores and loads stay in program order
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const int row = lane >> 3, seg = lane & 7;
        const double2* src = reinterpret_cast<const double2*>(lw + row * kLanePitch + 8 * seg);
        const double2 x0 = src[0], x1 = src[1], x2 = src[2], x3 = src[3];
        double s = ((x0.x + x0.y) + (x1.x + x1.y)) + ((x2.x + x2.y) + (x3.x + x3.y));
        s = dev::group_sum<8>(s);
        if (seg == 0 && row < cnt) rowpart[static_cast<long>(strip) * n + r + 4 * row] = s;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// grid (strips = ceil(m / kStrip), row blocks = ceil(n / rows)), 256 threads.
// beta has m entries (beta_{m-1} = 0).  Sums of w_ij = x_i T_ij y_j (WT:
// weights given, else 1): rowpart[strip * n + i] = sum of row i over the
// strip; colpart[block * m + j] (when non-null) = sum of column j over the
// block.  Each lane owns kCPL adjacent columns.
//
// Bound by the FP64 issue rate: at 16384^2 FP32 254 us at 30 VALU instructions
// per element, now 210 at 22.5 (84% of the cycles issue VALU, at the 2.0 GHz the
// card holds under FP64 load; the read of M alone takes 165 us).  What went: the
// wave sum per row (4 of the 30; see sums_rows_loop), the clamps and the NaN
// select of every exponential (3; now one test per row and the clamp on a branch),
// register moves.  At 4096^2 FP64 (134 MB) an evaluation call takes 53 us, before
// 72 with 15 us of that host round trips.
template <typename TM, bool WT, bool NT>
__global__ __launch_bounds__(256, WT ? 5 : 7) void k_sums_tile(const TM* __restrict__ M, long ldm, int n, int m,
                                                   const double* __restrict__ alpha,
                                                   const double* __restrict__ beta, double k,
                                                   int rows, const double* __restrict__ xw,
                                                   const double* __restrict__ yw,
                                                   double* __restrict__ rowpart,
                                                   double* __restrict__ colpart)
{
    // the waves' lane sums (kRowsTog kLanePitch each), then their column sums
    static_assert(kRowsTog * kLanePitch >= kStrip, "column sums take the same room");
    __shared__ __align__(16) double sm[4][kRowsTog * kLanePitch];
    __shared__ __align__(16) double tab[128];
    dev::exp2_tab_load(tab);
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int strip = blockIdx.x, blk = blockIdx.y;
    const int c0 = strip * kStrip + lane * kCPL;
    const int r0 = blk * rows;
    const int r1 = min(n, r0 + rows);
    // exponents in units of 1/64 (dexp2_64): exactly 64 times the log2 ones
    const double k64 = 64.0 * k;
    double bk[kCPL], yq[kCPL], cs[kCPL];
#pragma unroll
    for (int q = 0; q < kCPL; q++) {
        // (clamped, not skipped: the loads go out together)
        const int j = min(c0 + q, m - 1);
        const double bj = beta[j];
        bk[q] = (c0 + q < m) ? bj * k64 : 0.0;
        yq[q] = (WT && yw) ? yw[j] : 1.0;
        cs[q] = 0.0;
    }
    if ((strip + 1) * kStrip <= m)   // workgroup-uniform
        sums_rows_loop<TM, true, WT, NT>(M, ldm, n, m, alpha, k64, xw, c0, r0 + wave, r1, strip,
                                         bk, yq, tab, sm[wave], cs, rowpart);
    else
        sums_rows_loop<TM, false, WT, NT>(M, ldm, n, m, alpha, k64, xw, c0, r0 + wave, r1, strip,
                                          bk, yq, tab, sm[wave], cs, rowpart);
    if (!colpart) return;   // grid-uniform
#pragma unroll
    for (int q = 0; q < kCPL; q++) sm[wave][lane * kCPL + q] = cs[q];
    __syncthreads();
    for (int c = threadIdx.x; c < kStrip; c += 256) {
        const int j = strip * kStrip + c;
        if (j < m)
            colpart[static_cast<long>(blk) * m + j] =
                ((sm[0][c] + sm[1][c]) + sm[2][c]) + sm[3][c];
    }
}

// Four workgroup sums at once, each in bsum's order (wave sums, then the
// four wave totals left to right): one barrier instead of eight.
__device__ __forceinline__ void bsum4(double (&v)[4], double (*sm)[4])
{
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = wsum(v[q]);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int q = 0; q < 4; q++) sm[q][threadIdx.x >> 6] = v[q];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = ((sm[q][0] + sm[q][1]) + sm[q][2]) + sm[q][3];
}

// x[0] + x[pitch] + ... (cnt of them), 32 and then 8 loads in flight, added in
// order.  (Eight at a time k_sums_fold took 8.2 us at 16384^2, now 7.3.)
__device__ __forceinline__ double sum_strided(const double* __restrict__ x, long pitch, int cnt)
{
    double r = 0.0;
    int s = 0;
    for (; s + 32 <= cnt; s += 32) {
        double v[32];
#pragma unroll
        for (int u = 0; u < 32; u++) v[u] = x[(s + u) * pitch];
#pragma unroll
        for (int u = 0; u < 32; u++) r += v[u];
    }
    for (; s < cnt; s += 8) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = x[min(s + u, cnt - 1) * pitch];
#pragma unroll
        for (int u = 0; u < 8; u++) r += (s + u < cnt) ? v[u] : 0.0;
    }
    return r;
}

// Thread t < n: r_t = sum over strips, grad_t = r_t - a_t; thread t < m - 1:
// c_t = sum over blocks (when colpart is set), grad_{n+t} = c_t - b_t.
// part[4 wg + {0..3}] = this workgroup's sum r, sum alpha a, sum betat bt,
// sum g^2.
__global__ __launch_bounds__(256) void k_sums_fold(const double* __restrict__ rowpart, int nstrip,
                                                   const double* __restrict__ colpart, int nblk,
                                                   const double* __restrict__ alpha,
                                                   const double* __restrict__ beta,
                                                   const double* __restrict__ a,
                                                   const double* __restrict__ b, int n, int m,
                                                   double* __restrict__ grad,
                                                   double* __restrict__ part)
{
    __shared__ double sm44[4][4];
    const int t = blockIdx.x * 256 + threadIdx.x;
    double sr = 0.0, sa = 0.0, sb = 0.0, g2 = 0.0;
    if (t < n) {
        const double r = sum_strided(rowpart + t, n, nstrip);
        const double g = r - a[t];
        if (grad) grad[t] = g;
        sr = r;
        sa = alpha[t] * a[t];
        g2 = g * g;
    }
    if (t < m - 1) {
        sb = beta[t] * b[t];
        if (colpart) {
            const double c = sum_strided(colpart + t, m, nblk);
            const double g = c - b[t];
            if (grad) grad[n + t] = g;
            g2 += g * g;
        }
    }
    double v[4] = {sr, sa, sb, g2};
    bsum4(v, sm44);
    if (threadIdx.x == 0) {
        part[4 * blockIdx.x] = v[0];
        part[4 * blockIdx.x + 1] = v[1];
        part[4 * blockIdx.x + 2] = v[2];
        part[4 * blockIdx.x + 3] = v[3];
    }
}

// out[0] = reg sum r - alpha'a - betat'bt, out[1] = ||g||^2.
__global__ __launch_bounds__(256) void k_sums_final(const double* __restrict__ part, int npart,
                                                    double reg, double* __restrict__ out)
{
    __shared__ double sm44[4][4];
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    for (int i = threadIdx.x; i < npart; i += 256) {
        v[0] += part[4 * i];
        v[1] += part[4 * i + 1];
        v[2] += part[4 * i + 2];
        v[3] += part[4 * i + 3];
    }
    bsum4(v, sm44);
    if (threadIdx.x == 0) {
        out[0] = reg * v[0] - v[1] - v[2];
        out[1] = v[3];
    }
}

__global__ __launch_bounds__(256) void k_exp2_check(const double* __restrict__ x,
                                                    double* __restrict__ y, long count)
{
    __shared__ __align__(16) double tab[128];
    dev::exp2_tab_load(tab);
    __syncthreads();
    for (long i = static_cast<long>(blockIdx.x) * 256 + threadIdx.x; i < count;
         i += static_cast<long>(gridDim.x) * 256)
        y[i] = dev::dexp2(x[i], tab);
}

}  // namespace

void launch_exp2_check(const double* x, double* y, long count, hipStream_t s)
{
    if (count <= 0) return;
    hipLaunchKernelGGL(k_exp2_check, dim3(std::min(4096L, (count + 255) / 256)), dim3(256), 0, s,
                       x, y, count);
    KERNEL_CHECK();
}

// Rows per workgroup of the one-pass kernels: >= 1024 workgroups where the
// problem allows, 32 to 256 rows (the column partials stay <= n/32 rows;
// at 16384^2, 128- and 256-row blocks measured 7% faster than 64).
int sums_rows(int n, int m)
{
    const long nstrip = ceil_div(m, kStrip);
    long r = static_cast<long>(n) * nstrip / 1024;
    r = std::max(32L, std::min(256L, r));
    return static_cast<int>((r + 3) / 4 * 4);
}

void sums_scratch_sizes(int n, int m, long* rowpart, long* colpart, long* part)
{
    const long nstrip = ceil_div(m, kStrip), nblk = ceil_div(n, sums_rows(n, m));
    *rowpart = nstrip * n;
    *colpart = nblk * m;
    *part = 4L * ceil_div(std::max(n, m), 256);
}

// NT: a matrix that does not fit the 256 MB last-level cache is streamed.
template <typename TM, bool WT>
static void launch_sums_tile_t(const void* M, long ldm, int n, int m, const double* alpha,
                               const double* beta, double k, int rows, const double* x,
                               const double* y, double* rowpart, double* colpart, hipStream_t s)
{
    const dim3 grid(ceil_div(m, kStrip), ceil_div(n, rows));
    const bool nt = static_cast<double>(n) * ldm * sizeof(TM) > 256e6;
    hipLaunchKernelGGL((nt ? k_sums_tile<TM, WT, true> : k_sums_tile<TM, WT, false>), grid, dim3(256),
                       0, s, static_cast<const TM*>(M), ldm, n, m, alpha, beta, k, rows, x, y,
                       rowpart, colpart);
}

template <bool WT>
static void launch_sums_tile(int bulk, const void* M, long ldm, int n, int m, const double* alpha,
                             const double* beta, double k, int rows, const double* x,
                             const double* y, double* rowpart, double* colpart, hipStream_t s)
{
    if (bulk == 0)
        launch_sums_tile_t<float, WT>(M, ldm, n, m, alpha, beta, k, rows, x, y, rowpart, colpart,
                                      s);
    else
        launch_sums_tile_t<double, WT>(M, ldm, n, m, alpha, beta, k, rows, x, y, rowpart, colpart,
                                       s);
}

void launch_objgrad_fused(int bulk, const void* M, long ldm, int n, int m, const double* alpha,
                          const double* beta, const double* a, const double* b, double reg,
                          bool with_grad, double* grad, double* rowpart, double* colpart,
                          double* part, double* out, hipStream_t s)
{
    if (n <= 0 || m <= 0) fail(E_INVALID, "objective pass on an empty problem");
    const int nstrip = ceil_div(m, kStrip);
    const int rows = sums_rows(n, m);
    const int nblk = ceil_div(n, rows);
    const double k = 1.4426950408889634074 / reg;
    double* cp = with_grad ? colpart : nullptr;
    launch_sums_tile<false>(bulk, M, ldm, n, m, alpha, beta, k, rows, nullptr, nullptr, rowpart, cp,
                            s);
    KERNEL_CHECK();
    const int nf = ceil_div(std::max(n, m), 256);
    hipLaunchKernelGGL(k_sums_fold, dim3(nf), dim3(256), 0, s, rowpart, nstrip, cp, nblk, alpha,
                       beta, a, b, n, m, with_grad ? grad : nullptr, part);
    KERNEL_CHECK();
    hipLaunchKernelGGL(k_sums_final, dim3(1), dim3(256), 0, s, part, nf, reg, out);
    KERNEL_CHECK();
}

void launch_wsums(int bulk, const void* M, long ldm, int n, int m, const double* alpha,
                  const double* beta, double reg, const double* x, const double* y,
                  double* rowpart, double* colpart, hipStream_t s)
{
    if (n <= 0 || m <= 0) fail(E_INVALID, "weighted sums on an empty problem");
    const int rows = sums_rows(n, m);
    const double k = 1.4426950408889634074 / reg;
    if (x || y)
        launch_sums_tile<true>(bulk, M, ldm, n, m, alpha, beta, k, rows, x, y, rowpart, colpart, s);
    else
        launch_sums_tile<false>(bulk, M, ldm, n, m, alpha, beta, k, rows, nullptr, nullptr, rowpart,
                                colpart, s);
    KERNEL_CHECK();
}

int sums_strip_width() { return kStrip; }

}  // namespace regot
