// qrot.hpp -- quadratically regularised OT (QROT) on the device: the dual
// passes (qrot_kernels.hip), the roots (qrot_root.hip), the objective and the
// rounded primal value (qrot_sweep.hip) and the host drivers (qrot.cpp).  The QROT dual variable is
// gamma = [alpha (n); beta (m)]: no elimination of beta_m.
#pragma once

#include <memory>

#include "problem.hpp"

namespace regot {

int qrot_rows(int n, int m);
// scratch of the sweeps (qrot_sweep.hip), in doubles
void qrot_sweep_sizes(int n, int m, size_t* rowpart, size_t* colpart, size_t* scal);
bool qrot_row_root_ok(int m);

// The generalised Hessian H = [diag(h1) sigma; sigma' diag(h2)] at one gamma
// (src/qrot_hess.h:11-36): sigma as a bitmask (launch_qrot_mask), h1 = sigma 1,
// h2 = sigma' 1, plus the vectors of its block solve.
struct QrotHess {
    DBuf<unsigned long long> mask;
    DBuf<double> h1, h2, hinv, tn, tn2, tm, tm2, ones, v, r, pv, q, dsc, rowpart4;
    HBuf<double> hs;
    double hinv_shift = -1.0;
    QrotHess(int n, int m)
    {
        mask.alloc(static_cast<size_t>(n) * ceil_div(m, 256) * 4);
        rowpart4.alloc(static_cast<size_t>(n) * ceil_div(m, 256) * 4);
        const int c = n > m ? n : m;
        h1.alloc(n);
        h2.alloc(m);
        hinv.alloc(n);
        tn.alloc(n);
        tn2.alloc(n);
        v.alloc(n);
        tm.alloc(m);
        tm2.alloc(m);
        r.alloc(m);
        pv.alloc(m);
        q.alloc(m);
        ones.alloc(c);
        dsc.alloc(8);
        hs.ensure(8);
    }
};

// Device scratch of the QROT passes and root iterations, sized for a shape;
// owned by the problem handle.
struct QrotScratch {
    DBuf<double> rowpart, colpart, sqpart, rsum, csum, out, spart, fpart, gpart;
    // rounding (qrot_primal): row / column scales, column errors, totals
    DBuf<double> x, y, eb, scal;
    DBuf<double> epart, cpart;   // per-workgroup sums of the folds
    DBuf<int> kpart, kprev, done, open;
    HBuf<int> hopen;
    std::unique_ptr<QrotHess> hess;
    // M transposed (m x n, pitch ldt) for the column roots: a workspace of the
    // call that is running (mt_state 0: not formed, 1: formed, -1: no room),
    // formed again by each call since the caller may own M (QrotCall)
    DBuf<unsigned char> mt;
    long ldt = 0;
    int mt_state = 0;
    QrotScratch(int n, int m)
    {
        const int rows = qrot_rows(n, m);
        const long nstrip = ceil_div(m, 256), nblk = ceil_div(n, rows);
        // shared by the 256-column tiles and the sweeps
        size_t srow, scol, sscal;
        qrot_sweep_sizes(n, m, &srow, &scol, &sscal);
        const size_t trow = static_cast<size_t>(nstrip) * n, tcol = static_cast<size_t>(nblk) * m;
        rowpart.alloc(trow > srow ? trow : srow);
        colpart.alloc(tcol > scol ? tcol : scol);
        sqpart.alloc(sscal);
        rsum.alloc(n);
        csum.alloc(m);
        out.alloc(3);
        const int nw = ceil_div(n > m ? n : m, 256);
        fpart.alloc(4 * static_cast<size_t>(nw));
        gpart.alloc(nw);
        const int c = n > m ? n : m;
        kprev.alloc(c);
        done.alloc(c);
        open.alloc(1);
        hopen.ensure(1);
        x.alloc(n);
        y.alloc(m);
        eb.alloc(m);
        scal.alloc(sscal);
        epart.alloc(4 * static_cast<size_t>(ceil_div(static_cast<long>(n) + m, 64)));
        cpart.alloc(ceil_div(m, 64));
    }
};
// Roots of every row in one read of M (m <= 16384, qrot_root.hip):
// out_i = the x with sum_j (x - (M_ij - pot_j))_+ = reg w_i.
void launch_qrot_row_root(int bulk, const void* M, long ldm, int n, int m, const double* pot,
                          const double* w, double reg, double* out, int ncu, hipStream_t s);
// The same roots by Newton passes over M (wider matrices, or no room for the
// transpose):
void launch_qrot_pl_init(double* xc, int* kprev, int* done, int count, int* open, hipStream_t s);
// One Newton step of the per-column (cols) or per-row roots; *open counts the
// entries still moving.
void launch_qrot_pl_step(int bulk, const void* M, long ldm, int n, int m, bool cols,
                         const double* pot, const double* w, double reg, double* xc,
                         int* kprev, int* done, double* spart, int* kpart, int* open,
                         hipStream_t s);
void launch_qrot_plan(int bulk, const void* M, long ldm, int n, int m, const double* alpha,
                      const double* beta, double reg, double* plan, long r0, int nr,
                      hipStream_t s);
// f into out[0] and (with grad) grad and ||grad||^2 into out[1]; part holds
// 4 ceil(max(n, m) / 256) doubles, gpart ceil(max(n, m) / 256).
void launch_qrot_finish(const double* alpha, const double* beta, const double* a,
                        const double* b, int n, int m, double reg, double tau, const double* sq,
                        const double* rsum, const double* csum, double* grad, double* part,
                        double* gpart, double* out, hipStream_t s);

void launch_qrot_fold(const double* part, int nparts, long stride, int count, double* out,
                      hipStream_t s);
// APDAGD's / PDAAM's plan pass P = cold P + tau plan(alpha, beta) (init: P = plan),
// then out[0] = <M, P>, out[1] = ||P||^2, out[2] = ||P1 - a||^2 + ||P'1 - b||^2
// (device); scratch as documented at the definition.
void launch_qrot_apd_plan(int bulk, const void* M, long ldm, int n, int m, const double* alpha,
                          const double* beta, double reg, double cold, double tau, bool init,
                          double* P,
                          long ldp, const double* a, const double* b, double* rowpart,
                          double* colpart, double* rsum, double* csum, double* wpart,
                          double* out, hipStream_t s);
void launch_qrot_sum1(const double* part, int count, double* out, hipStream_t s);

// sigma (bitmask, see QrotHess) at alpha, beta
void launch_qrot_mask(int bulk, const void* M, long ldm, int n, int m, const double* alpha,
                      const double* beta, unsigned long long* mask, hipStream_t s);
// Row sums of sigma_ij y_j (rows_out) into rowpart[(strip * 4 + k) * n + i]
// (4 partials per 256-column strip: fold 4 ceil(m / 256) of them) and column
// sums of sigma_ij x_i (cols_out) per block of qrot_rows rows into
// colpart[blk * m + j]; null x or y count ones.
void launch_qrot_sig(const unsigned long long* mask, int n, int m, bool rows_out, bool cols_out,
                     const double* x, const double* y, double* rowpart, double* colpart,
                     hipStream_t s);
void launch_qrot_ainv(const double* x, const double* h, double shift, double c, double* out,
                      int count, hipStream_t s);
void launch_qrot_delta_fin(const double* x, const double* h, double shift, const double* t,
                           double c, double* out, int count, hipStream_t s);
void launch_qrot_recip(const double* h, double shift, double* out, int count, hipStream_t s);
// out_i = (t_i + h_i x_i) + c
void launch_qrot_hfin(const double* x, const double* h, const double* t, double c, double* out,
                      int count, hipStream_t s);

// The generalised Hessian at device gamma (n + m) into the problem's QrotHess.
QrotHess& qrot_hess_build(regot_problem* p, const double* gamma);
// out (device, n + m) = (H + shift I + tau vv')^-1 rhs, v = [1; -1], by block
// elimination with CG on the Schur complement (Eigen's rules: from x0
// (device, m; may alias out + n) or zero, ||r||^2 < tol^2 ||rhs_beta||^2);
// returns the CG steps.
int qrot_hess_solve(regot_problem* p, QrotHess& H, const double* rhs, double shift, double tau,
                    double tol, int max_iter, double* out, const double* x0 = nullptr);
// out (device, n + m) = (H + tau vv') x (src/qrot_hess.cpp:193-214, shift 0).
void apply_qrot_hess(regot_problem* p, QrotHess& H, const double* x, double tau, double* out);

// f (and grad, ||grad||^2 when grad is non-null) of the QROT dual at device
// gamma (n + m), src/qrot_problem.cpp:226-258.
double qrot_obj_grad(regot_problem* p, const double* gamma, double* grad, double tau,
                     double* gnorm2);
// One call of the C-ABI that may form the transpose.  Its contents are forgotten
// at the end (M may change before the next call) and its memory stays with the
// handle up to kQrotKeep bytes: allocating and freeing 256 MiB takes 0.3 ms, a
// fifth of a three-iteration solve of such a matrix, 4 GiB 0.6 ms, which is less
// than one iteration on it.
constexpr size_t kQrotKeep = static_cast<size_t>(512) << 20;
struct QrotCall {
    regot_problem* p;
    explicit QrotCall(regot_problem* q) : p(q) {}
    QrotCall(const QrotCall&) = delete;
    QrotCall& operator=(const QrotCall&) = delete;
    ~QrotCall();
};
// Row pitch of M' in elements.
long qrot_transpose_pitch(int bulk, int n);
// optimal_beta (cols = true: out = beta (m) given alpha = pot) or
// optimal_alpha (cols = false: out = alpha (n) given beta = pot), device.
void qrot_optimal(regot_problem* p, bool cols, const double* pot, double* out);

// <P, M> + reg/2 ||P||^2 of P = approx_proj((alpha (+) beta - M)_+ / reg)
// for device alpha (n), beta (m).  fresh: the last sweep on this handle was
// qrot_obj_grad with a gradient at this very point, whose row scales are taken.
double qrot_primal(regot_problem* p, const double* alpha, const double* beta, bool fresh);
// The QROT plan (alpha (+) beta - M)+ / reg of a host dual (n + m) into host memory.
void qrot_plan_host(regot_problem* p, const double* dual, double* plan);

}  // namespace regot
