// cg_lds.hip -- the two sparse products of a CG iteration for large sets of
// stored entries, with the gathered vector in LDS.
//
// y = (sigma u) / (h1 + shift) and w = (h2 + shift) u - sigma' y with sigma as
// CSR and CSC (see hessian.hip for the iteration).  A product reads every entry
// once and, for each, one element of a vector of at most 18432 doubles.  From
// global memory that gather goes at about one cache line a clock and CU, which
// alone takes 22 us for the 13.4 M entries of 5% of 16384^2; the vector fits
// the CU's 160 KB of LDS, where 64 lanes' reads take some 16 clocks.  So one
// workgroup of 16 waves per CU copies the vector (128 KB from L2, 2 us) and
// takes a run of rows, its waves one row at a time by a counter in LDS; the
// next 512 entries are loaded while the current ones are added.  FP32 bulk: the
// entries are read as T in FP32 and 16-bit indices, 6 bytes instead of 12, and
// T / reg is formed as the builder forms it, so the value is the same; both
// copies then fit the 256 MB last-level cache together.  Every lane adds the
// same entries in the same order as one lane of k_cg_rows / k_cg_cols with 64
// lanes per row does, and the sums over lanes and columns pair alike: the
// results are the same bits.
//
// 13.4 M entries of 16384^2 in FP32 bulk: rows 39.7 -> 14.7 us, columns 41 ->
// 16.1 us (80 MB of entries each, 5.2 TB/s with the copy of the vector); what is
// left is that read and the copy.
#include <algorithm>

#include "cg.hpp"
#include "dense_device.hpp"

namespace regot {
namespace {

constexpr int kT = 1024;
constexpr int kWaves = kT / 64;
constexpr int kU = 8;           // entries per lane and step
constexpr int kWgRows = 96;     // rows (columns) per workgroup

// The entries' value, T / reg.
__device__ __forceinline__ double entry(float t, double scale)
{
    return static_cast<double>(t) * scale;
}
__device__ __forceinline__ double entry(double v, double) { return v; }

template <typename VT, typename IT>
struct Entries {
    VT v[kU];
    IT c[kU];
};

// The entries k + lane + 64 u of a row that ends at e; past the end the row's
// last one again (entry 0 when it has none), not used.
template <typename VT, typename IT>
__device__ __forceinline__ void fetch(const VT* __restrict__ val, const IT* __restrict__ ind, int k,
                                      int e, int lane, Entries<VT, IT>& b)
{
    const int last = e > 0 ? e - 1 : 0;
#pragma unroll
    for (int u = 0; u < kU; u++) {
        const int q = k + lane + 64 * u;
        const int i = q < e ? q : last;
        b.v[u] = val[i];
        b.c[u] = ind[i];
    }
}

// Workgroup b: rows (COLS: columns) b per .. b per + per - 1 of a CSR (CSC) with
// cnt of them, over a vector of nvec entries.  per is a multiple of 4.
template <typename VT, typename IT, bool COLS>
__global__ __launch_bounds__(kT) void k_cg_lds(CgArgs a0, CgArgs a1, const VT* __restrict__ val,
                                               const IT* __restrict__ ind, double scale, int cnt,
                                               int per, int nvec, int it)
{
    __shared__ __align__(16) double xs[kCgLdsVec];
    __shared__ double su[kWgRows], sh[kWgRows], sr[kWgRows], sg[kWgRows], sd[kWgRows];
    __shared__ int rp[kWgRows + 1];
    __shared__ int next;
    // (selected one by one: a selected struct goes to scratch)
    const bool second = blockIdx.y != 0;
    const double* const au = second ? a1.u : a0.u;
    const double* const ar = second ? a1.r : a0.r;
    double* const ay = second ? a1.y : a0.y;
    double* const aw = second ? a1.w : a0.w;
    double* const apart = second ? a1.part : a0.part;
    double* const ascal = second ? a1.scal : a0.scal;
    int* const actl = second ? a1.ctl : a0.ctl;
    double* const arep = second ? a1.rep : a0.rep;
    const double shift = a0.shift;
    const double* const ah = COLS ? a0.h2 : a0.h1;
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int r0 = blockIdx.x * per;
    const int nr = min(per, cnt - r0);
    const int* ptr = COLS ? a0.colptr : a0.rowptr;
    const double* vec = COLS ? ay : au;

    // everything that does not depend on the stop flag goes out with it
    double v = 0.0;
    if (COLS)
        for (int b = lane; b < a0.nbu; b += 64) v += apart[2 * a0.nbc + b];
    if (t <= nr) rp[t] = ptr[r0 + t];
    if (t < kWgRows) {
        const bool in = t < nr;
        const int j = r0 + (in ? t : 0);
        sh[t] = ah[j];
        if (COLS) {
            su[t] = au[j];
            sr[t] = ar[j];
            sg[t] = 0.0;
            sd[t] = 0.0;
        }
    }
    if (t == 0) next = kWaves;
    // the wave's first row and its first entries
    int row = wave, k = 0, e = 0;
    double acc = 0.0;
    Entries<VT, IT> b0, b1;
    if (row < nr) {
        k = ptr[r0 + row];
        e = ptr[r0 + row + 1];
        fetch(val, ind, k, e, lane, b0);
    }
    constexpr int kFill = kCgLdsVec / (2 * kT);
    const int last2 = (nvec & ~1) - 2;   // pairs past the end read the last one again
    double2 f[kFill];
#pragma unroll
    for (int q = 0; q < kFill; q++)
        f[q] = *reinterpret_cast<const double2*>(vec + min(2 * (t + kT * q), last2));
    const double tail = vec[nvec - 1];
    if (actl[0]) return;   // uniform
#pragma unroll
    for (int q = 0; q < kFill; q++)
        *reinterpret_cast<double2*>(xs + min(2 * (t + kT * q), last2)) = f[q];
    if (t == 0) xs[nvec - 1] = tail;
    if (COLS) {
        // every wave sums the update's r.r partials itself, in the same order
        const double rr = dev::group_sum<64>(v);
        if (rr < ascal[5]) {
            if (blockIdx.x == 0 && t == 0) {
                ascal[4] = rr;
                actl[1] = it;   // the converged update is not counted (Eigen's convention)
                actl[0] = 1;
                arep[0] = 1.0;
            }
            return;   // every workgroup alike
        }
        if (blockIdx.x == 0 && t == 0) ascal[4] = rr;
    }
    __syncthreads();

    if (row < nr) {
        // One step: start the loads of the next one, add the current entries,
        // finish the row with its last ones.  False: no rows are left.
        auto step = [&](const Entries<VT, IT>& cur,
                        Entries<VT, IT>& nxt) __attribute__((always_inline)) {
            int row2 = row, k2 = k + 64 * kU, e2 = e;
            if (k2 >= e) {   // uniform
                int g = 0;
                if (lane == 0) g = atomicAdd(&next, 1);
                row2 = __builtin_amdgcn_readfirstlane(g);
                if (row2 < nr) {
                    k2 = __builtin_amdgcn_readfirstlane(rp[row2]);
                    e2 = __builtin_amdgcn_readfirstlane(rp[row2 + 1]);
                }
            }
            if (row2 < nr) fetch(val, ind, k2, e2, lane, nxt);
#pragma unroll
            for (int u = 0; u < kU; u++) {
                const double s = fma(entry(cur.v[u], scale), xs[cur.c[u]], acc);
                acc = (k + lane + 64 * u < e) ? s : acc;
            }
            if (row2 != row) {
                const double sum = dev::group_sum<64>(acc);
                if (lane == 0) {
                    if (COLS) {
                        const double uj = su[row];
                        const double wj = sh[row] * uj + shift * uj - sum;
                        aw[r0 + row] = wj;
                        sg[row] = sr[row] * uj;
                        sd[row] = wj * uj;
                    } else {
                        ay[r0 + row] = sum / (sh[row] + shift);
                    }
                }
                acc = 0.0;
            }
            row = row2;
            k = k2;
            e = e2;
            return row < nr;
        };
        while (step(b0, b1) && step(b1, b0)) {
        }
    }
    if (!COLS) return;
    __syncthreads();
    // r.u and w.u of four columns each, in order
    if (4 * t < nr) {
        double g = 0.0, d = 0.0;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            g += sg[4 * t + q];
            d += sd[4 * t + q];
        }
        const int b = r0 / 4 + t;
        apart[2 * b] = g;
        apart[2 * b + 1] = d;
    }
}

__global__ __launch_bounds__(256) void k_cg_compact(const double* __restrict__ val,
                                                    const int* __restrict__ ind, long long nnz,
                                                    double reg, float* __restrict__ val32,
                                                    unsigned short* __restrict__ ind16)
{
    for (long long k = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x; k < nnz;
         k += static_cast<long long>(gridDim.x) * 256) {
        // (T / reg) reg differs from T by 3 roundings of FP64, far less than
        // half an ulp of the FP32 number T is
        val32[k] = static_cast<float>(val[k] * reg);
        ind16[k] = static_cast<unsigned short>(ind[k]);
    }
}

int rows_per_wg(int cnt, int ncu) { return (ceil_div(cnt, ncu) + 3) / 4 * 4; }

template <bool COLS>
void launch(const CgArgs& a0, const CgArgs& a1, const CgEntries& e, int ny, int it, int ncu,
            hipStream_t s)
{
    const int cnt = COLS ? a0.m1 : a0.n, nvec = COLS ? a0.n : a0.m1;
    if (!cg_lds_ok(a0.n, a0.m1, ncu)) fail(E_INTERNAL, "CG product of %d x %d", a0.n, a0.m1);
    const int per = rows_per_wg(cnt, ncu);
    const dim3 grid(ceil_div(cnt, per), ny);
    const float* v32 = COLS ? e.cval32 : e.rval32;
    if (v32)
        hipLaunchKernelGGL((k_cg_lds<float, unsigned short, COLS>), grid, dim3(kT), 0, s, a0, a1,
                           v32, COLS ? e.rowind16 : e.colind16, e.scale, cnt, per, nvec, it);
    else
        hipLaunchKernelGGL((k_cg_lds<double, int, COLS>), grid, dim3(kT), 0, s, a0, a1,
                           COLS ? a0.cval : a0.rval, COLS ? a0.rowind : a0.colind, 1.0, cnt, per,
                           nvec, it);
    KERNEL_CHECK();
}

}  // namespace

bool cg_lds_ok(int n, int m1, int ncu)
{
    return n > 1 && m1 > 1 && ncu > 0 && n <= kCgLdsVec && m1 <= kCgLdsVec &&
           rows_per_wg(n, ncu) <= kWgRows && rows_per_wg(m1, ncu) <= kWgRows;
}

void launch_cg_compact(const double* val, const int* ind, long long nnz, double reg, float* val32,
                       unsigned short* ind16, hipStream_t s)
{
    if (nnz <= 0) return;
    const int grid = static_cast<int>(std::min(16384LL, (nnz + 255) / 256));
    hipLaunchKernelGGL(k_cg_compact, dim3(grid), dim3(256), 0, s, val, ind, nnz, reg, val32, ind16);
    KERNEL_CHECK();
}

void launch_cg_rows_lds(const CgArgs& a0, const CgArgs& a1, const CgEntries& e, int ny, int ncu,
                        hipStream_t s)
{
    launch<false>(a0, a1, e, ny, 0, ncu, s);
}

void launch_cg_cols_lds(const CgArgs& a0, const CgArgs& a1, const CgEntries& e, int ny, int it,
                        int ncu, hipStream_t s)
{
    launch<true>(a0, a1, e, ny, it, ncu, s);
}

}  // namespace regot
