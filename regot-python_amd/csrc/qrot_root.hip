// qrot_root.hip -- optimal_alpha / optimal_beta of the QROT dual in one read of
// the cost matrix (src/qrot_problem.cpp:365-418).
//
// Per row i (or column, over the transpose): the root x of
//   sum_j (x - y_j)_+ = c,   y_j = M_ij - pot_j,  c = reg w_i.
// The root lies in (y_min, y_min + c]: at y_min + c the smallest term alone
// gives c.  So only entries below y_min + c can be active, a handful of a row
// unless reg w is large against the spread of M.  One workgroup holds a row in
// registers (16 entries per thread, T threads, m <= 16 T <= 16384), finds
// y_min, appends the candidates to LDS in a fixed order, and one of its waves
// (they take turns) runs Newton's method from the right on them,
//   x <- (c + sum of y < x) / (their count),
// until the count no longer shrinks: the reference's formula on the same
// active set.  A wave with more than 64 candidates sends its row to the same
// iteration over all of the registers.
//
// Newton over the whole matrix took a read of M per step, about 16 steps per
// root solve from an all-active start.  Measured at 8192^2 FP32: rows 16 x 69
// us and columns 16 x 97 us before (pass and update), 47 us now for either
// (268 MB: 5.7 TB/s, bound by the read; the transpose, 2 x 268 MB once per
// call, serves the columns).
#include <cmath>

#include "dense_device.hpp"
#include "qrot.hpp"

namespace regot {
namespace {

using namespace dev;

constexpr int kRootE = 16;      // entries of a row per thread
constexpr int kRootCap = 64;    // candidates a wave hands over
constexpr int kRootMax = 1024 * kRootE;

template <typename TM, int T, bool NT>
__global__ __launch_bounds__(T) void k_qrot_row_root(const TM* __restrict__ M, long ldm, int n,
                                                     int m, const double* __restrict__ pot,
                                                     const double* __restrict__ w, double reg,
                                                     double* __restrict__ out)
{
    using VT = typename VecOf<TM>::type;
    constexpr int V = VecOf<TM>::N;
    constexpr int NC = kRootE / V;
    constexpr int NW = T / 64;
    __shared__ double mn[NW];
    __shared__ int cnt[NW];
    __shared__ double seg[NW][kRootCap];
    __shared__ double rs[NW];
    __shared__ int rk[NW];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // columns past m: potential -inf, so y = +inf, never active (a vector with
    // no column reads the row's first instead)
    int off[NC];
    double pt[NC][V];
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const int j0 = V * (threadIdx.x + c * T);
        off[c] = j0 < m ? j0 : 0;
#pragma unroll
        for (int v = 0; v < V; v++) pt[c][v] = j0 + v < m ? pot[j0 + v] : -INFINITY;
    }
    auto load = [&](int row, VT (&b)[NC]) {
        const TM* Mi = M + static_cast<long>(row) * ldm;
#pragma unroll
        for (int c = 0; c < NC; c++) b[c] = ld_m(Mi + off[c], NT);
    };
    VT cur[NC], nxt[NC];
    int turn = 0;
    load(blockIdx.x, cur);
    for (int row = blockIdx.x; row < n; row += gridDim.x) {
        const int next = row + static_cast<int>(gridDim.x);
        load(next < n ? next : row, nxt);
        const double c0 = reg * w[row];
        auto y = [&](int c, int v) {
            return static_cast<double>(vget<VT, TM>(cur[c], v)) - pt[c][v];
        };
        double lo = INFINITY;
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int v = 0; v < V; v++) lo = fmin(lo, y(c, v));
        const double wlo = -wave_max(-lo);
        if (lane == 0) mn[wave] = wlo;
        __syncthreads();
        double ymin = mn[0];
#pragma unroll
        for (int q = 1; q < NW; q++) ymin = fmin(ymin, mn[q]);
        const double x0 = ymin + c0;
        int found = 0;
        if (wlo < x0) {   // the same on every lane of the wave
#pragma unroll
            for (int c = 0; c < NC; c++)
#pragma unroll
                for (int v = 0; v < V; v++) {
                    const double yv = y(c, v);
                    const unsigned long long hit = __ballot(yv < x0);
                    if (hit != 0) {
                        const int at = found + __builtin_amdgcn_mbcnt_hi(
                                                   static_cast<unsigned>(hit >> 32),
                                                   __builtin_amdgcn_mbcnt_lo(
                                                       static_cast<unsigned>(hit), 0));
                        if (yv < x0 && at < kRootCap) seg[wave][at] = yv;
                        found += __popcll(hit);
                    }
                }
        }
        if (lane == 0) cnt[wave] = found;
        __syncthreads();
        int most = 0;
#pragma unroll
        for (int q = 0; q < NW; q++) most = max(most, cnt[q]);
        if (most <= kRootCap) {
            if (wave == turn) {
                double x = x0;
                int kprev = -1;
                for (;;) {
                    double S = 0.0;
                    int K = 0;
#pragma unroll
                    for (int q = 0; q < NW; q++) {
                        const int have = cnt[q];
                        if (have == 0) continue;
                        const double yv = lane < have ? seg[q][lane] : INFINITY;
                        S += yv < x ? yv : 0.0;
                        K += __popcll(__ballot(yv < x));
                    }
                    if (K == 0 || (kprev >= 0 && K >= kprev)) break;
                    x = (c0 + wave_sum0(S)) / K;
                    kprev = K;
                }
                if (lane == 0) out[row] = x;
            }
        } else {
            double x = x0;
            int kprev = -1;
            for (;;) {
                double S = 0.0;
                int K = 0;
#pragma unroll
                for (int c = 0; c < NC; c++)
#pragma unroll
                    for (int v = 0; v < V; v++) {
                        const double yv = y(c, v);
                        S += yv < x ? yv : 0.0;
                        K += __popcll(__ballot(yv < x));
                    }
                S = wave_sum0(S);
                if (lane == 0) {
                    rs[wave] = S;
                    rk[wave] = K;
                }
                __syncthreads();
                S = 0.0;
                K = 0;
#pragma unroll
                for (int q = 0; q < NW; q++) {
                    S += rs[q];
                    K += rk[q];
                }
                __syncthreads();
                // the same values on every wave: all leave together
                if (K == 0 || (kprev >= 0 && K >= kprev)) break;
                x = (c0 + S) / K;
                kprev = K;
            }
            if (threadIdx.x == 0) out[row] = x;
        }
        turn = turn + 1 == NW ? 0 : turn + 1;
#pragma unroll
        for (int c = 0; c < NC; c++) cur[c] = nxt[c];
    }
}

template <typename TM>
void row_root(const TM* M, long ldm, int n, int m, const double* pot, const double* w, double reg,
              double* out, int ncu, hipStream_t s)
{
    const bool nt = static_cast<long>(n) * ldm * static_cast<long>(sizeof(TM)) > (256L << 20);
    auto go = [&](auto kern, int T) {
        // about 16 waves per CU, each workgroup a few rows (the potentials
        // stay in its registers)
        long g = static_cast<long>(ncu > 0 ? ncu : 256) * 1024 / T;
        if (g > n) g = n;
        hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(g)), dim3(T), 0, s, M, ldm, n, m, pot,
                           w, reg, out);
        KERNEL_CHECK();
    };
    if (m <= 64 * kRootE) return nt ? go(k_qrot_row_root<TM, 64, true>, 64)
                                    : go(k_qrot_row_root<TM, 64, false>, 64);
    if (m <= 128 * kRootE) return nt ? go(k_qrot_row_root<TM, 128, true>, 128)
                                     : go(k_qrot_row_root<TM, 128, false>, 128);
    if (m <= 256 * kRootE) return nt ? go(k_qrot_row_root<TM, 256, true>, 256)
                                     : go(k_qrot_row_root<TM, 256, false>, 256);
    if (m <= 512 * kRootE) return nt ? go(k_qrot_row_root<TM, 512, true>, 512)
                                     : go(k_qrot_row_root<TM, 512, false>, 512);
    return nt ? go(k_qrot_row_root<TM, 1024, true>, 1024)
              : go(k_qrot_row_root<TM, 1024, false>, 1024);
}

}  // namespace

bool qrot_row_root_ok(int m) { return m <= kRootMax; }

void launch_qrot_row_root(int bulk, const void* M, long ldm, int n, int m, const double* pot,
                          const double* w, double reg, double* out, int ncu, hipStream_t s)
{
    if (n < 1 || m < 1 || !qrot_row_root_ok(m) || ldm < m)
        fail(E_INTERNAL, "QROT row roots: shape %d x %d", n, m);
    if (bulk == 0)
        row_root(static_cast<const float*>(M), ldm, n, m, pot, w, reg, out, ncu, s);
    else
        row_root(static_cast<const double*>(M), ldm, n, m, pot, w, reg, out, ncu, s);
}

}  // namespace regot
