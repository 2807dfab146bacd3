// bcd_rows.hip -- one BCD iteration in one read of the cost matrix, several
// rows per barrier (FP32 or FP64 storage and arithmetic).
//
// The iteration is that of bcd_fused.hip: a workgroup holds whole rows, and
// per row i
//
//   e_ij  = 2^((beta_j - M_ij) k - sh_i),  sh_i = log2 a_i - k alpha_{k,i}
//   tot_i = sum_j e_ij                     (= r_i / a_i, ~1 near the solution)
//   alpha_{k+1,i} = reg (log a_i - ln2 (sh_i + log2 tot_i))
//   u_ij  = e_ij (a_i / tot_i) = exp((alpha_{k+1,i} + beta_j - M_ij) / reg),
//
// whose column sums over the workgroup's rows go out as one FP64 value per
// column.  Thread t owns the V-column vectors at V t + V T c (V = 16 bytes of
// M, c < NC).  A step takes R rows: their vectors were loaded during the step
// before, the R row totals are reduced together (DPP within a wave, then one
// LDS exchange and one barrier, R NW <= 64 wave totals on the lanes of every
// wave), and each wave derives the R weights itself, the same bits everywhere.
// Against one row per barrier (bcd_fused.hip, which keeps m > 8192, where a
// row alone is 32 KB of loads) the chain of a row -- 6 cross-lane steps, LDS,
// barrier, 8 LDS reads, a division -- is paid once per R rows, the loads have
// no branch between them (so a wait covers only the rows it needs), and the
// row epilogue reads LDS records and needs no exponential: r_i = a_i tot_i.
//
// Measured, device time per iteration with the combine, before -> now (before:
// one row per barrier in FP32 with m > 1024, else row pass + column pass):
// 4096^2 FP32 34.0 -> 21.2 us, 8192^2 FP32 62.4 -> 50.9, 5003 x 3011 FP32
// 42.0 -> 22.6, 4096^2 FP64 78.2 -> 32.2, 1000 x 800 FP64 28.4 -> 10.3.  What
// bounds it: the two launches (about 2.5 us each), and the read of M from the
// Infinity Cache while it fits (4096^2 FP32: a bare read takes 10-12 us with
// its launch) or HBM (8192^2: 268 MB, 5.9 TB/s in the pass).
//
// Range: e and tot as in bcd_fused.hip; tot_i outside [lo, hi] (FP32
// arithmetic 2^-+20, FP64 2^-+400) or not a number redoes the row with its
// largest term as the shift.  A term flushed below the smallest normal drops
// < 2^-106 (FP32) or < 2^-600 (FP64) of a_i from a column sum.  A row of
// infinite costs has tot 0: alpha = +inf, and no part in the column sums.
#include "dense.hpp"
#include "dense_device.hpp"
#include "dexp2.hpp"

#include <cmath>

namespace regot {
namespace {

using namespace dev;

// Rows per workgroup are bounded by the per-row (shift, total) record kept
// for the epilogue.
constexpr int kRMaxRows = 1024;
constexpr int kRMaxCols = 8192;

// 2^(y / SC) in the arithmetic type.  FP64 takes the table of dexp2.hpp (tab in
// LDS), whose argument is 64 x: the factor goes into k and the shifts, exactly.
template <typename TA>
constexpr double kSc = sizeof(TA) == 8 ? 64.0 : 1.0;
__device__ __forceinline__ float ex2t(float x, const double*) { return ex2(x); }
__device__ __forceinline__ double ex2t(double y, const double* tab) { return dexp2_64(y, tab); }

__device__ __forceinline__ double readlane_f64(double v, int lane)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// log2 a_i - k alpha_i, the same bits wherever it is formed.
__device__ __forceinline__ double row_shift(double loga, double alpha, double k)
{
    return fma(-alpha, k, loga * kLog2e);
}

// R rows of the thread's vectors from row i0 on.  Rows past r1 - 1 read that row
// again, and a thread whose last vector (c = NC - 1) has no column reads its
// row's first (off[c]): in bounds, not used, and no branch between the loads.
template <typename TM, int NC, int R, bool NT>
__device__ __forceinline__ void load_rows(const TM* __restrict__ M, long ldm, long i0, long r1,
                                          const int (&off)[NC],
                                          typename VecOf<TM>::type (&out)[R][NC])
{
#pragma unroll
    for (int r = 0; r < R; r++) {
        const long i = (i0 + r < r1) ? i0 + r : r1 - 1;
        const TM* Mi = M + i * ldm;
#pragma unroll
        for (int c = 0; c < NC; c++) out[r][c] = ld_m(Mi + off[c], NT);
    }
}

// ONE: every workgroup has at most R rows, one step.  NT: nontemporal loads.
template <typename TM, typename TA, int T, int NC, int R, bool ONE, bool NT>
__global__ __launch_bounds__(T) void k_bcd_rows(
    const TM* __restrict__ M, long ldm, int n, int m, const double* __restrict__ beta, double k,
    double reg, const double* __restrict__ loga, const double* __restrict__ a,
    const double* __restrict__ alpha, double* __restrict__ alpha_out, int rpw,
    double* __restrict__ part, long pitch, double* __restrict__ rpart,
    const int* __restrict__ ctl)
{
    using VT = typename VecOf<TM>::type;
    constexpr int V = VecOf<TM>::N;
    constexpr int NW = T / 64;
    constexpr int SPAN = V * T;
    constexpr bool F64 = sizeof(TA) == 8;
    constexpr double LO = F64 ? 0x1p-400 : 0x1p-20, HI = F64 ? 0x1p400 : 0x1p20;
    static_assert(NW * R <= 64, "one lane per wave total");
    static_assert(R <= 4, "FP32 terms of a column between FP64 additions");
    __shared__ double red[2][NW * R];
    __shared__ double redx[NW];
    __shared__ double rsum[NW][3];
    // per row, for the epilogue: shift, total, log a, alpha, a
    __shared__ double rec[kRMaxRows][5];
    __shared__ __align__(16) double tab[F64 ? 128 : 2];

    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const long r0 = static_cast<long>(blockIdx.x) * rpw;
    const long r1 = (r0 + rpw < n) ? r0 + rpw : n;
    const int col0 = V * t;
    int vlast = m - (col0 + (NC - 1) * SPAN);
    vlast = vlast < 0 ? 0 : (vlast > V ? V : vlast);
    auto ok = [vlast](int c, int v) { return c < NC - 1 || v < vlast; };
    const double ks = k * kSc<TA>;

    int off[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) off[c] = (c < NC - 1 || vlast > 0) ? col0 + c * SPAN : 0;

    // the first rows and beta are on their way before the stop flag is looked at
    VT b0[R][NC], b1[R][NC];
    load_rows<TM, NC, R, NT>(M, ldm, r0, r1, off, b0);
    double bk[NC][V];
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int v = 0; v < V; v++) {
            const int j = col0 + c * SPAN + v;
            bk[c][v] = beta[(c < NC - 1 || j < m) ? j : m - 1] * ks;
        }
    // lane (r, w) of every wave: row r of the step
    const int lr = lane / NW;
    double la, al, av;
    {
        const long i = (r0 + lr < r1) ? r0 + lr : r1 - 1;
        la = loga[i];
        al = alpha[i];
        av = a[i];
    }
    if (F64) exp2_tab_load(tab);
    if (ctl[0] != 0) return;
    if (F64) __syncthreads();

    double acc[NC][V];
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int v = 0; v < V; v++) acc[c][v] = 0.0;

    // A shift of 1e30 makes every term 0.  The repeats of the last row have weight
    // 0 and must not have an infinite term; an infinite potential (a row without a
    // finite cost) or one that is not a number (a warm start's) says nothing of the
    // row's size, and the range test finds a shift if there is a finite term.
    auto shift_at = [&](long i) {
        const double s = row_shift(la, al, k);
        return (i + lr < r1 && __builtin_isfinite(s)) ? s : 1e30;
    };
    double next_shl = shift_at(r0);

    auto step = [&](VT (&cur)[R][NC], VT (&nxt)[R][NC], long i0, int slot) {
        const double la0 = la, al0 = al, av0 = av;
        double shl = next_shl;
        const bool row_in = lane < NW * R && i0 + lr < r1;
        if (!ONE) {
            // the next step's row data, then its rows
            long i = i0 + R + lr;
            i = (i < r1) ? i : r1 - 1;
            la = loga[i];
            al = alpha[i];
            av = a[i];
            load_rows<TM, NC, R, NT>(M, ldm, i0 + R, r1, off, nxt);
        }
        TA e[R][NC][V];
        double tot;
        for (int trial = 0;; trial++) {
            double S[R];
#pragma unroll
            for (int r = 0; r < R; r++) {
                const double sh = readlane_f64(shl, r * NW) * kSc<TA>;
                TA s = TA(0);
#pragma unroll
                for (int c = 0; c < NC; c++) {
#pragma unroll
                    for (int v = 0; v < V; v++) {
                        const double mv = static_cast<double>(vget<VT, TM>(cur[r][c], v));
                        TA x = static_cast<TA>(fma(-ks, mv, bk[c][v] - sh));
                        // the argument is masked, not the value: no branch
                        x = ok(c, v) ? x : TA(-1e30);
                        e[r][c][v] = ex2t(x, tab);
                        s += e[r][c][v];
                    }
                    // four FP64 exponentials (a row's arguments in FP32) are
                    // interleaved, not all of them: registers
                    if (F64 && (c * V) % 4 == 4 - V) __builtin_amdgcn_sched_barrier(0);
                }
                S[r] = static_cast<double>(s);
                __builtin_amdgcn_sched_barrier(0);
            }
            wave_sums<R>(S);
            if (lane == 0) {
#pragma unroll
                for (int r = 0; r < R; r++) red[slot][r * NW + wave] = S[r];
            }
            __syncthreads();
            tot = group_sum<NW>(red[slot][lane < NW * R ? lane : 0]);
            // tot has the same bits on every wave: the workgroup branches alike
            unsigned long long bad = __ballot(row_in && !(tot >= LO && tot <= HI));
            if (bad == 0 || trial != 0) break;
            // Rare (first iterations from a poor start): such rows take their
            // largest term as the shift and the step is formed again.
            while (bad != 0) {
                const int r = (__ffsll(bad) - 1) / NW;
                bad &= ~(((1ull << (NW - 1) << 1) - 1) << (r * NW));
                const TM* Mi = M + (i0 + r) * ldm;
                double tm = -INFINITY;
#pragma unroll
                for (int c = 0; c < NC; c++)
#pragma unroll
                    for (int v = 0; v < V; v++)
                        if (ok(c, v))
                            tm = fmax(tm, fma(-ks, static_cast<double>(Mi[off[c] + v]),
                                              bk[c][v]));
                tm = wave_max(tm);
                if (lane == 0) redx[wave] = tm;
                __syncthreads();
                double dm = redx[0];
#pragma unroll
                for (int q = 1; q < NW; q++) dm = fmax(dm, redx[q]);
                if (lr == r && dm > -INFINITY && dm < INFINITY) shl = dm * (1.0 / kSc<TA>);
                __syncthreads();   // redx and red[slot] are free again
            }
            load_rows<TM, NC, R, false>(M, ldm, i0, r1, off, cur);
            // vmcnt(0) here, so that the loop head does not have to wait for
            // every load in flight (the next step's) on the usual path
            __builtin_amdgcn_s_waitcnt(0x0F70);
        }
        const double w = (row_in && tot > 0.0) ? av0 / tot : 0.0;
        if (wave == 0 && row_in && (lane & (NW - 1)) == 0) {
            double* q = rec[i0 - r0 + lr];
            q[0] = shl;
            q[1] = tot;
            q[2] = la0;
            q[3] = al0;
            q[4] = av0;
        }
        TA wr[R];
#pragma unroll
        for (int r = 0; r < R; r++) wr[r] = static_cast<TA>(readlane_f64(w, r * NW));
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int v = 0; v < V; v++) {
                if (F64) {
#pragma unroll
                    for (int r = 0; r < R; r++)
                        acc[c][v] = fma(static_cast<double>(e[r][c][v]),
                                        static_cast<double>(wr[r]), acc[c][v]);
                } else {
                    // R <= 4 FP32 terms between FP64 additions
                    TA x = e[0][c][v] * wr[0];
#pragma unroll
                    for (int r = 1; r < R; r++) x = fma(e[r][c][v], wr[r], x);
                    acc[c][v] += static_cast<double>(x);
                }
            }
        // off the next step's path (the row data came before its rows)
        if (!ONE) next_shl = shift_at(i0 + R);
    };

    if (ONE) {
        step(b0, b1, r0, 0);
    } else {
#pragma unroll 1
        for (long i0 = r0; i0 < r1; i0 += 2 * R) {
            step(b0, b1, i0, 0);
            if (i0 + R >= r1) break;
            step(b1, b0, i0 + R, 1);
        }
    }

    // The records of up to 64 rows pass between lanes of wave 0 without a barrier;
    // the wave's LDS stores and loads stay in program order.
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();

    // pitch is a multiple of 16: whole vectors, also past m
    double* pw = part + static_cast<long>(blockIdx.x) * pitch + col0;
#pragma unroll
    for (int c = 0; c < NC; c++)
        if (c < NC - 1 || vlast > 0) {
#pragma unroll
            for (int v = 0; v < V; v += 2)
                *reinterpret_cast<double2*>(pw + c * SPAN + v) =
                    make_double2(acc[c][v], acc[c][v + 1]);
        }

    // Row epilogue, rows strided over the threads: alpha_{k+1} and the
    // stop-test sums at iterate k.  With the usual shift r_i = a_i tot_i.
    const int rows = static_cast<int>(r1 - r0);
    if (rows > 64) __syncthreads();   // else wave 0 alone, which wrote the records
    if (rows <= 64 && wave != 0) return;
    double x[3] = {0.0, 0.0, 0.0};
    for (int rr = t; rr < rows; rr += T) {
        const double sh = rec[rr][0], tot = rec[rr][1];
        const double lai = rec[rr][2], ali = rec[rr][3], ai = rec[rr][4];
        const double L = tot > 0.0 ? sh + log2(tot) : -INFINITY;
        alpha_out[r0 + rr] = reg * (lai - kLn2 * L);
        const bool usual = sh == row_shift(lai, ali, k);
        const double ri = usual ? ai * tot : exp2(ali * k + L);
        const double g = usual ? ai * (tot - 1.0) : ri - ai;
        x[0] += g * g;
        x[1] += ri;
        x[2] += ali * ai;
    }
    wave_sums<3>(x);
    if (rows <= 64) {
        if (lane == 0) {
#pragma unroll
            for (int q = 0; q < 3; q++) rpart[3 * blockIdx.x + q] = x[q];
        }
        return;
    }
    if (lane == 0) {
#pragma unroll
        for (int q = 0; q < 3; q++) rsum[wave][q] = x[q];
    }
    __syncthreads();
    if (t < 3) {
        double y = rsum[0][t];
        for (int v = 1; v < NW; v++) y += rsum[v][t];
        rpart[3 * blockIdx.x + t] = y;
    }
}

template <typename TM, typename TA, int T, int NC, int R>
void launch_one(const BcdRowsArgs& g, hipStream_t s)
{
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(g.nblk), dim3(T), 0, s, static_cast<const TM*>(g.M), g.ldm,
                           g.n, g.m, g.beta, g.k, g.reg, g.loga, g.a, g.alpha, g.alpha_out, g.rpw,
                           g.part, g.pitch, g.rpart, g.ctl);
        KERNEL_CHECK();
    };
    if (g.nt)
        go(k_bcd_rows<TM, TA, T, NC, R, false, true>);
    else if (g.rpw <= R)
        go(k_bcd_rows<TM, TA, T, NC, R, true, false>);
    else
        go(k_bcd_rows<TM, TA, T, NC, R, false, false>);
}

}  // namespace

bool bcd_rows_shape_ok(int n, int m, int ncu)
{
    return n >= 1 && m >= 1 && m <= kRMaxCols && ceil_div(n, bcd_fused_blocks(n, ncu)) <= kRMaxRows;
}

// The pass costs a workgroup 0.3 us per row (FP32 storage with FP64 arithmetic:
// 0.45) however few columns the row has, since its threads past them idle; the
// two-pass form costs a time per strip of columns (64 lanes x 16 bytes), and with
// one or two strips that is the smaller.  us per iteration, single read
// / two passes, at 128, 192, 256 and 512 rows per CU: FP32 x 256 columns 44 / 55,
// 63 / 65, 81 / 74, 154 / 112; x 512 45 / 59, 63 / 74, 82 / 90, 157 / 151; x 576
// 45 / 69, 63 / 92, 82 / 112, 157 / 209.  FP64 x 128 50 / 53, 71 / 64, 92 / 74,
// 175 / 114; x 256 50 / 65, 71 / 79, 93 / 95, 179 / 154; x 320 51 / 67, 72 / 88,
// 93 / 108, 178 / 198.  FP32 storage with FP64 arithmetic x 256 65 / 65, 92 / 78,
// 121 / 92; x 512 64 / 77, 92 / 100, 121 / 120, 235 / 209.
bool bcd_rows_pays(int bulk, bool precise, int n, int m, int ncu)
{
    const int strip = bulk == 0 ? 256 : 128;
    const int limit = bulk == 0 && !precise ? 192 : 128;
    const int rows = ceil_div(n, bcd_fused_blocks(n, ncu));
    return m > 2 * strip || rows <= limit * ceil_div(m, strip);
}

long bcd_part_pitch(int m) { return (static_cast<long>(m) + 15) / 16 * 16; }

void launch_bcd_rows(int bulk, bool precise, BcdRowsArgs g, hipStream_t s)
{
    g.rpw = ceil_div(g.n, g.nblk);
    if (g.n < 1 || g.m < 1 || g.m > kRMaxCols || g.rpw > kRMaxRows || g.pitch < g.m || g.pitch % 16)
        fail(E_INTERNAL, "BCD row pass: shape %d x %d over %d workgroups", g.n, g.m, g.nblk);
    if (static_cast<long>(g.rpw) * (g.nblk - 1) >= g.n)
        fail(E_INTERNAL, "BCD row pass: %d workgroups for %d rows", g.nblk, g.n);
    g.nt = static_cast<long>(g.n) * g.ldm * (bulk == 0 ? 4 : 8) > (256L << 20) ? 1 : 0;
    // Rows per step: about 32 KB of M per workgroup and step measured best (us
    // per iteration at R = 1 / 2 / 4: 4096^2 FP32 24.3 / 21.2 / 24.0, 5003 x
    // 3011 FP32 26.9 / 22.6 / 22.9, 2048^2 FP32 14.5 / 12.8 / 12.5, 6001 x 3000
    // FP64 38.7 / 35.4 / -, 8192^2 FP32 51.6 / 50.9 / -): fewer expose the
    // reduction, more overrun the memory pipe (a bare read of 64 MB by 256
    // workgroups takes 12.0 us with 64 KB in flight each, 15.3 with 128).
    // 1024 threads with half the columns each were slower everywhere.
    if (bulk == 0 && !precise) {
        if (g.m <= 1024) return launch_one<float, float, 256, 1, 4>(g, s);
        switch (ceil_div(g.m, 2048)) {
        case 1: return launch_one<float, float, 512, 1, 4>(g, s);
        case 2: return launch_one<float, float, 512, 2, 2>(g, s);
        case 3: return launch_one<float, float, 512, 3, 2>(g, s);
        default: return launch_one<float, float, 512, 4, 2>(g, s);
        }
    }
    if (bulk == 0) {
        if (g.m <= 1024) return launch_one<float, double, 256, 1, 4>(g, s);
        switch (ceil_div(g.m, 2048)) {
        case 1: return launch_one<float, double, 512, 1, 4>(g, s);
        case 2: return launch_one<float, double, 512, 2, 2>(g, s);
        case 3: return launch_one<float, double, 512, 3, 1>(g, s);
        default: return launch_one<float, double, 512, 4, 1>(g, s);
        }
    }
    if (g.m <= 512) return launch_one<double, double, 256, 1, 4>(g, s);
    switch (ceil_div(g.m, 1024)) {
    case 1: return launch_one<double, double, 512, 1, 4>(g, s);
    case 2: return launch_one<double, double, 512, 2, 2>(g, s);
    case 3: return launch_one<double, double, 512, 3, 2>(g, s);
    case 4: return launch_one<double, double, 512, 4, 2>(g, s);
    case 5: return launch_one<double, double, 512, 5, 1>(g, s);
    case 6: return launch_one<double, double, 512, 6, 1>(g, s);
    case 7: return launch_one<double, double, 512, 7, 1>(g, s);
    default: return launch_one<double, double, 512, 8, 1>(g, s);
    }
}

}  // namespace regot
