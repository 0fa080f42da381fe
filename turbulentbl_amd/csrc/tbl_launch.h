// tbl_launch.h -- host-side launchers of the device kernels (internal).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include "tbl_dev.h"

namespace tbl {

enum { PC_SSOR_RB = 1, PC_NONE = 2, PC_JACOBI = 3, PC_FAST = 4, PC_SSOR_BLOCK = 5 };
struct FastPC;

// stencil kernels (tbl_stencil.hip)
unsigned resid_blocks(const Geo &g);
unsigned rhs_blocks(const Geo &g, bool single);
// hpart (optional): the momentum kernel also forms the Helmholtz solve's first
// residual pass (block partials in k_helm_resid's layout, rhs_blocks of them)
template <class T> void launch_momentum_rhs(const Geo &g, const T *Ut, const T *P, T *Q, hipStream_t s,
                                            const unsigned char *brin = nullptr, unsigned char *brout = nullptr,
                                            double *hpart = nullptr);
template <class T> void launch_helm_resid(const Geo &g, const T *Q, const T *Ut, const void *ctrl, double *part, int first, hipStream_t s);
void launch_helm_fin(const Geo &g, void *ctrl, const double *part, int it, double errorstop, double floor_coef, hipStream_t s,
                     int nb = 0, const Pub &pub = Pub());
void launch_gs_init(void *ctrl, hipStream_t s);          // all components active, sums zero
template <class T> void launch_helm_sweep(const Geo &g, const T *Q, T *Ut, const void *ctrl, int colour, hipStream_t s);
template <class T> void launch_helm_zline(const Geo &g, const T *Q, T *Ut, const T *zf, const void *ctrl, int colour, hipStream_t s);
// one pass of the z-line zebra sweep: x neighbours from cur, span rows from
// ysrc, results to dst (see k_helm_zebra)
template <class T> void launch_helm_zebra(const Geo &g, const T *Q, const T *cur, const T *ysrc, T *dst, const T *zf,
                                          const void *ctrl, int colour, hipStream_t s);
// boundary / ghost values of the three velocity components, src -> dst
// (and the Gauss-Seidel control block of a new solve, as launch_gs_init)
template <class T> void launch_copy_faces3(const Geo &g, const T *src, T *dst, void *ctrl, hipStream_t s);
// per-slab lexicographic Gauss-Seidel sweep; threads a slab kernel needs, 0 if
// the slabs are too thick for one workgroup; values of scr that the sweep
// (lex) or the block SSOR needs
template <class T> void launch_helm_lex(const Geo &g, const T *Q, T *Ut, T *scr, const void *ctrl, hipStream_t s);
size_t slab_scratch(const Geo &g, bool lex);
bool slab_copy_pays(const Geo &g);
size_t slab_scratch_inplace(const Geo &g, bool lex);     // ... without the skewed copy (g.skew 0)
int slab_threads(const Geo &g, int nkmax);
size_t gs_ctrl_bytes();
void gs_ctrl_read(const void *host, int *active, int *sweeps, double *res);
// gate (optional): the Gauss-Seidel control block; the launch does nothing
// while any of its components is active
template <class T> void launch_ppe_rhs(const Geo &g, const T *Ut, double *pRhs, hipStream_t s, const void *gate = nullptr);
unsigned poisson_blocks(const Geo &g, bool single);   // partials written by launch_poisson with part
// out = A x (scaled); with part: also the block partials of <out, v0> (returns the block count)
template <class T>
unsigned launch_poisson(const Geo &g, const T *x, T *out, const int *active, const double *scale, hipStream_t s,
                        const T *v0 = nullptr, double *part = nullptr);
// bpart (optional): block partials of ||pRhs||^2, as many as part
template <class Tr> void launch_resid(const Geo &g, const double *pRhs, const double *PC, Tr *r, double *part, hipStream_t s,
                                      double *bpart = nullptr);
// mode: RU_CYCLE the correction of a finished one-step cycle; RU_GATED the
// same, doing nothing while gc's cycle is active (queued ahead of a host
// poll); RU_UNIT the tentative unit step PC + z0, doing nothing unless it is
enum { RU_CYCLE = 0, RU_GATED = 1, RU_UNIT = 2 };
template <class Tr>
void launch_resid_upd(const Geo &g, const double *pRhs, const double *PC, const Tr *Z, const GmCtrl *gc, double *PCn,
                      Tr *r, double *part, hipStream_t s, int mode = RU_CYCLE);
// part (FPC_*) applies to the fast preconditioner only
template <class T> void launch_precond(const Geo &g, int pc, const FastPC *fast, const T *r, T *scratch, T *out, const int *active, hipStream_t s,
                                       int part = 0);
template <class T> void launch_zero_faces(const Geo &g, T *x, hipStream_t s);
template <class T> void launch_save_inflow(const Geo &g, const T *Ut, T *Utold, hipStream_t s);
template <class T> void launch_project(const Geo &g, double *PC, T *Press, T *Ut, hipStream_t s);
template <class T> void launch_bcs(const Geo &g, T *Ut, const T *Utold, T *Press, const double *wall_w, hipStream_t s);
template <class T> void launch_recycle(const Geo &g, T *Ut, int i_rec0, double eps, const double *lamda_dev,
                                       const double *avg, const double *Wt, const int *newk, const double *Ume,
                                       const double *uf, hipStream_t s);

// fast separable Poisson preconditioner (tbl_fastpc.hip)
struct FastPC;
int fastpc_create(const Geo &g, const double *Ab, const double *At, const double *Ap, hipStream_t s, bool single,
                  FastPC **out, char *err, int errlen);
void fastpc_destroy(FastPC *f);
// parts of one application: all of it, its first transform, or the rest
enum { FPC_ALL = 0, FPC_HEAD = 1, FPC_TAIL = 2 };
template <class T> int run_fastpc(const FastPC *f, const Geo &g, const T *r, T *out, const int *active, hipStream_t s,
                                  int part = FPC_ALL);
// one fast solve of ncomp components (N values apart): operand and result in
// FP64 or in the storage type (FP64 contexts: FP64 both); add: out += result;
// mask: the operand's face rows are read as zero
struct FastIO {
    const void *in = nullptr;
    void *out = nullptr;
    int in64 = 0, out64 = 0, add = 0, mask = 0, ncomp = 1;
};
// out = (alpha I + beta A)^{-1} in, or its transpose
int run_fast_solve(const FastPC *f, const Geo &g, const FastIO &io, const int *active, double alpha, double beta,
                   bool transpose, hipStream_t s, int part = FPC_ALL);
// work fields for solves of ncomp components (synchronises when they grow; 1,
// and what there was, if there is no memory); solve_batched: whether three
// components may go through one solve
size_t fastpc_bytes(const FastPC *f);    // device memory held
// about what |M^-1 r| / |M^-1 b| is after one FP64 solve of A x = b (the same for any b)
double fastpc_reach(const FastPC *f);
int fastpc_reserve(FastPC *f, const Geo &g, int ncomp, hipStream_t s);
bool solve_batched(const Geo &g, bool single);

// Krylov kernels (tbl_krylov.hip)
unsigned vec_blocks(long N, bool single);
// x[0..n) = v (a kernel, not a memset: safe inside captured graphs)
void launch_fill(double *x, double v, long n, hipStream_t s);
template <class T> void launch_norm2(const T *x, long N, double *part, const int *active, hipStream_t s);
// part_b (optional): nb_r block partials of ||pRhs||^2 (start of a true-residual solve)
void launch_fin_start(GmCtrl *c, const double *part_r, int nb_r, const double *part_z, int nb_z, int first, hipStream_t s,
                      const double *part_b = nullptr);
// judges the tentative unit step: residual partials part_r, and the block
// partials of its preconditioned residual (part_z, reference's stopping rule)
void launch_fin_unit(GmCtrl *c, const double *part_r, int nb_r, const double *part_z, int nb_z, const Pub &pub, hipStream_t s);
// start of a pressure solve: the control block, and zero faces of PC (and of PC2)
void launch_gm_init(const Geo &g, GmCtrl *c, double errtol, double inner_tol, int kmax, int mmax, int mode, double *PC,
                    double *PC2, hipStream_t s);
// words 8-byte words at src to the host
void launch_publish(const void *src, int words, const Pub &pub, hipStream_t s);
template <class T> void launch_dots(const T *V, long ldv, int j, long N, const GmCtrl *c, double *part, hipStream_t s);
void launch_fin_dots(GmCtrl *c, const double *part, int nb, int j, hipStream_t s);
// store false: the norm of the new vector only, the vector is left as it was
template <class T> void launch_update(const T *V, long ldv, int j, long N, GmCtrl *c, double *part, hipStream_t s,
                                      bool store = true);
void launch_fin_update(GmCtrl *c, const double *part, int nb, int j, hipStream_t s);
// gated: does nothing while the cycle is active (queued ahead of a host poll)
void launch_fin_cycle(GmCtrl *c, hipStream_t s, int gated = 0);
template <class T> void launch_xupd(const T *V, long ldv, long N, const GmCtrl *c, double *PC, hipStream_t s);

// diagnostics (tbl_diag.hip)
struct RecDev {            // device-resident scalars of the recycling state
    double lamda, lamda03;
    int ksep;
};
template <class T> void launch_div_check(const Geo &g, const T *Ut, double *part, hipStream_t s);
void launch_fin_sum(const double *part, int nb, double *out, hipStream_t s);
// out2[0] = |sum of part| / nint, out2[1] = the sum
void launch_fin_div(const double *part, int nb, double nint, double *out2, hipStream_t s);
#define MF_BLK 64   // mass-flux partial blocks per plane
// device diagnostics record; the mass-flux partials (5 * MF_BLK) follow it
enum { DD_DIV = 0, DD_MASS = 1, DD_KE = 6, DD_BNORM = 7, DD_GUARD = 8, DD_NCOUNT = 9,
       DD_J = DD_NCOUNT + 5 * MF_BLK };   // behind the mass-flux partials: the objective of an adjoint window
template <class T> void launch_mass_flux(const Geo &g, const T *Ut, const int *planes, double *part, hipStream_t s);
// rec[DD_DIV] = sum of the nb divergence partials (nb > 0), rec[DD_MASS..] = mass
// flux (mpart given); publishes the record
void launch_fin_diag(const double *part, int nb, const double *mpart, double denom, double *rec, const Pub &pub, hipStream_t s);
template <class T> void launch_stats(const Geo &g, const T *Ut, double *sums, hipStream_t s);
template <class T> void launch_rescale(const Geo &g, int i_rec0, int nsamples, const T *Ut, double *sums,
                                       double *avg, RecDev *rec, double *Wt, int *newk, double *bltkns,
                                       double *deltastar, double *theta, double *uf, double *scan_scratch,
                                       hipStream_t s);
template <class T> void launch_ke(const Geo &g, int i_rec0, const T *Ut, const double *avg, double *part,
                                  int *guard, double *uf, hipStream_t s);
// acc (optional): the running window sum, acc(i) += tau(i)
template <class T> void launch_wall_shear(const Geo &g, const T *Ut, double *tau, hipStream_t s, double *acc = nullptr);
void launch_tau_window(const Geo &g, int window, double *acc, double *mean, double *cf, hipStream_t s);

// direct Helmholtz solve and the discrete adjoint (tbl_adjoint.hip)
template <class T> void launch_helm_rfield(const Geo &g, const T *Q, const T *u, T *r, int ncomp, hipStream_t s);
template <class To>
void launch_opT_res(const Geo &g, const double *b, const double *x, double alpha, double beta, To *r, int ncomp, hipStream_t s);
void launch_adj_tau(const Geo &g, double *lamU, int i0, int i1, double cJ, hipStream_t s);
// boundary values of a step's end velocity that the reversed conditions read (E, adj_end_len doubles)
long adj_end_len(const Geo &g);
template <class T> void launch_adj_save_end(const Geo &g, const T *U, double *E, hipStream_t s);
void launch_adj_bcs(const Geo &g, const double *E, double *lamU, double *lamP, double *grad, hipStream_t s);
void launch_adj_proj(const Geo &g, const double *lamU, const double *lamP, double *lamPhi, hipStream_t s);
void launch_adj_div(const Geo &g, const double *lamB, double *lamU, hipStream_t s);
template <class T>
void launch_adj_mom(const Geo &g, const T *U, const double *lamQ, double *lamU, double *lamP, hipStream_t s);
void launch_pc_extrap(double *pc, double *prev, long N, hipStream_t s);
void launch_tau_acc(const Geo &g, const double *tau, int i0, int i1, double cJ, double *J, hipStream_t s);

}  // namespace tbl
