// cg.hpp -- state of the device-controlled CG on Delta (hessian.hip) and the
// products with the gathered vector in LDS (cg_lds.hip).
#pragma once

#include "common.hpp"

namespace regot {

// ctl: [0] done, [1] iterations when done, [2] how the set-up ended it (k_cg_begin).
// scal: [0..1] alpha by parity, [2..3] gamma by parity, [4] r.r of the last update,
// [5] stop threshold, [6] rhs.rhs, [7] w.u of the set-up.
struct CgArgs {
    const int* rowptr;
    const int* colind;
    const double* rval;
    const int* colptr;
    const int* rowind;
    const double* cval;
    const double* h1;
    const double* h2;
    double shift;
    int n, m1;
    double* x;
    double* r;
    double* p;
    double* s;
    double* w;
    double* u;
    double* y;      // n
    double* part;   // [2 nbc] r.u, w.u per column workgroup; [nbu] r.r per update workgroup
    double* scal;
    int* ctl;
    int nbc;        // column workgroups
    int nbu;        // update workgroups (256 entries each)
    const double* dinv;   // Jacobi preconditioner, or null
    double* rep;          // host-visible: rep[0] = 1 on stop
};

// The entries the products of cg_lds.hip read.  FP32 bulk: T itself (val32) and
// 16-bit indices, the value being T scale with scale = 1 / reg, as it is
// stored in FP64; FP64 bulk: the stored values and indices.
struct CgEntries {
    const float* rval32 = nullptr;
    const float* cval32 = nullptr;
    const unsigned short* colind16 = nullptr;
    const unsigned short* rowind16 = nullptr;
    double scale = 1.0;
};

// Longest gathered vector (n or m - 1).
constexpr int kCgLdsVec = 18432;

// Whether the products may run with their vector in LDS, on ncu workgroups.
bool cg_lds_ok(int n, int m1, int ncu);
// val32 = T of the stored values (T / reg), ind16 = the indices.
void launch_cg_compact(const double* val, const int* ind, long long nnz, double reg, float* val32,
                       unsigned short* ind16, hipStream_t s);
// The row and the column product of one iteration (k_cg_rows, k_cg_cols with 64
// lanes per row), ny right-hand sides.
void launch_cg_rows_lds(const CgArgs& a0, const CgArgs& a1, const CgEntries& e, int ny, int ncu,
                        hipStream_t s);
void launch_cg_cols_lds(const CgArgs& a0, const CgArgs& a1, const CgEntries& e, int ny, int it,
                        int ncu, hipStream_t s);

}  // namespace regot
