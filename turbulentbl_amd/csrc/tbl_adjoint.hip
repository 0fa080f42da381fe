// tbl_adjoint.hip -- discrete adjoint of the TBL time step (FP64), and the
// direct Helmholtz solve that the forward steps of an adjoint window use.
//
// Inside a window that crosses no statistics rescale (dnssetbl.f90:986-1220)
// the recycling inflow is a constant overwrite of the i = 1 plane, and one
// step maps (Ut, Press) to (Ut, Press) through
//   Q = U - dt (conv(U) + Gp(P))                 (dnssetbl.f90:306-369)
//   U* = H^{-1} (Q + h B(U faces)), H = I - hA   (:371-433, solved exactly)
//   phi = A^{-1} D(U*)/dt                        (:437-671, solved exactly)
//   phi extended to the faces, P += phi, U = U* - dt G(phi)   (:673-726)
//   velocity and pressure boundary conditions    (:728-797)
// The kernels below apply the transposes of these blocks in reverse order.
// Every kernel gathers: one thread owns one output value and sums the
// contributions of the forward outputs that read it, so no two threads write
// the same address and the result is deterministic.  Indices are 0-based;
// the interior is i in [1,nX-2], j in [1,nY-2], k in [1,nZ-2].
#include <algorithm>

#include "tbl_dev.h"
#include "tbl_launch.h"

namespace tbl {


__device__ __forceinline__ bool inner(const Geo &g, int i, int j, int k)
{
    return i >= 1 && i <= g.nX - 2 && j >= 1 && j <= g.nY - 2 && k >= 1 && k <= g.nZ - 2;
}
__device__ __forceinline__ long lin(const Geo &g, int i, int j, int k)
{
    return (long)i + (long)g.nX * ((long)j + (long)g.nY * k);
}
__device__ __forceinline__ double sgn(double x) { return (double)((x > 0.0) - (x < 0.0)); }

// all-points 3-D launch: 64 x 4 (i,j) tiles, one k plane per block row
static inline dim3 all3(const Geo &g) { return dim3((g.nX + 63) / 64, (g.nY + 3) / 4, g.nZ); }
#define ALL3_IDX                                                   \
    const int i = blockIdx.x * 64 + (threadIdx.x & 63);            \
    const int j = blockIdx.y * 4 + (threadIdx.x >> 6);             \
    const int k = blockIdx.z;                                      \
    if (i >= g.nX || j >= g.nY) return;
// the same over ncomp components (N values apart, nZ plane rows each)
#define COMP3_IDX                                                  \
    const int i = blockIdx.x * 64 + (threadIdx.x & 63);            \
    const int j = blockIdx.y * 4 + (threadIdx.x >> 6);             \
    const int k = blockIdx.z % g.nZ;                               \
    const long comp = (long)(blockIdx.z / g.nZ) * g.N;             \
    if (i >= g.nX || j >= g.nY) return;
static inline dim3 comp3(const Geo &g, int ncomp) { return dim3((g.nX + 63) / 64, (g.nY + 3) / 4, g.nZ * ncomp); }

// ============================================================================
// direct Helmholtz solve (forward): residual field and interior update
// ============================================================================
// r = Q - H u on the interior, in the reference's residual form
// (dnssetbl.f90:378-386) evaluated in double; faces of r are left untouched
template <class T>
__global__ __launch_bounds__(256) void k_helm_rfield(Geo g, const T *__restrict__ Q, const T *__restrict__ u,
                                                    T *__restrict__ r)
{
    COMP3_IDX
    Q += comp; u += comp; r += comp;
    if (!inner(g, i, j, k)) return;
    const long c = lin(g, i, j, k), sk = g.sZ;
    const long cp = lin(g, i, jp1_of(j, g.nY), k), cm = lin(g, i, jm1_of(j, g.nY), k);
    const double rt1 = g.Ae * (double)u[c + 1] + g.Aw * (double)u[c - 1] + g.An * (double)u[cp] + g.As * (double)u[cm];
    const double rt2 = g.At[k] * (double)u[c + sk] + g.Ab[k] * (double)u[c - sk];
    r[c] = (T)((double)Q[c] - (1.0 - g.dt / g.Re * g.Ap[k]) * (double)u[c] + g.dt * (rt1 + rt2) / g.Re);
}

// ============================================================================
// transposed operators for the adjoint solves
// ============================================================================
// r = b - (alpha x + beta A^T x) on the interior, formed in FP64 and stored
// in To (FP32 for the refinement passes of a mixed context); x is zero off
// the interior.
// A^T x (c) = Ap(k) x(c) + Aw x(c+1) + Ae x(c-1) + As x(jp1) + An x(jm1)
//           + Ab(k+1) x(c+sk) + At(k-1) x(c-sk)
template <class To>
__global__ __launch_bounds__(256) void k_opT_res(Geo g, const double *__restrict__ b, const double *__restrict__ x,
                                                 double alpha, double beta, To *__restrict__ r)
{
    COMP3_IDX
    b += comp; x += comp; r += comp;
    if (!inner(g, i, j, k)) return;
    const long c = lin(g, i, j, k), sk = g.sZ;
    const long cp = lin(g, i, jp1_of(j, g.nY), k), cm = lin(g, i, jm1_of(j, g.nY), k);
    const double ax = g.Ap[k] * x[c] + g.Aw * x[c + 1] + g.Ae * x[c - 1] + g.As * x[cp] + g.An * x[cm] +
                      g.Ab[k + 1] * x[c + sk] + g.At[k - 1] * x[c - sk];
    r[c] = (To)(b[c] - (alpha * x[c] + beta * ax));
}

// ============================================================================
// objective: J = cJ * sum_{i in [i0,i1]} tau(i), tau of dnstbl/dnstbl.f90:1620-1668
// ============================================================================
// lamU += dJ/dU.  Thread per wall point (i, j), i in [0,nX-1], j in [1,nY-2].
__global__ void k_adj_tau(Geo g, double *__restrict__ lamU, int i0, int i1, double cJ)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y + 1;
    if (i >= g.nX) return;
    const long N = g.N, sk = g.sZ, c = lin(g, i, j, 0);
    const double s = cJ / g.Re, df1 = g.df1, df2 = g.df2;
    double *U = lamU, *W = lamU + 2 * N;
    if (i >= i0 && i <= i1) {
        // fder = ((U(k=2) - U(k=0)) df1^2 + (U(k=0) - U(k=1)) df2^2) / (df2 df1^2 - df2^2 df1)
        const double den = (df2 * (df1 * df1)) - ((df2 * df2) * df1);
        U[c] += s * ((df2 * df2) - (df1 * df1)) / den;
        U[c + sk] += s * (-(df2 * df2)) / den;
        U[c + 2 * sk] += s * (df1 * df1) / den;
    }
    // dw/dx at the wall of the stations within 3 of i
    double a = 0.0;
    for (int o = -3; o <= 3; o++) {
        const int st = i - o;                       // station st reads W(st + o) = W(i)
        if (o == 0 || st < i0 || st > i1) continue;
        if (st <= 2 || st >= g.nX - 3) {
            if (o == 1) a += 1.0 / (2.0 * g.dx);
            else if (o == -1) a -= 1.0 / (2.0 * g.dx);
        } else {
            const double w6 = (o == -3) ? -1.0 : (o == -2) ? 9.0 : (o == -1) ? -45.0 : (o == 1) ? 45.0 : (o == 2) ? -9.0 : 1.0;
            a += w6 / (60.0 * g.dx);
        }
    }
    W[c] += s * a;
}

// ============================================================================
// pressure boundary conditions, reversed (dnssetbl.f90:738-797)
// ============================================================================
// span copies P(i,0,k) = P(i,nY-2,k), P(i,nY-1,k) = P(i,1,k); thread per (i,k),
// component blockIdx.z
__global__ void k_adj_span(Geo g, double *__restrict__ lam)
{
    lam += blockIdx.z * g.N;
    const int i = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y;
    if (i >= g.nX) return;
    const long g0 = lin(g, i, 0, k), g1 = lin(g, i, g.nY - 1, k);
    lam[lin(g, i, g.nY - 2, k)] += lam[g0];
    lam[lin(g, i, 1, k)] += lam[g1];
    lam[g0] = 0.0;
    lam[g1] = 0.0;
}
// What the reversed boundary conditions read of the velocity at the end of a
// step: u(0,j,k) at E[j + nY k], then w(i,j,0) and w(i,j,1), nX nY values each
// (adj_end_len values; keeping the whole field took two copies of it a step).
long adj_end_len(const Geo &g) { return (long)g.nY * g.nZ + 2 * g.sZ; }
template <class T>
__global__ void k_adj_save_end(Geo g, const T *__restrict__ U, double *__restrict__ E)
{
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x, nu = (long)g.nY * g.nZ;
    if (e < nu) E[e] = (double)U[e * g.nX];
    else if (e < nu + 2 * g.sZ) E[e] = (double)U[2 * g.N + e - nu];
}
template <class T> void launch_adj_save_end(const Geo &g, const T *U, double *E, hipStream_t s)
{
    hipLaunchKernelGGL(k_adj_save_end<T>, dim3((unsigned)((adj_end_len(g) + 255) / 256)), dim3(256), 0, s, g, U, E);
}
template void launch_adj_save_end<double>(const Geo &, const double *, double *, hipStream_t);
template void launch_adj_save_end<float>(const Geo &, const float *, double *, hipStream_t);

// inflow pressure P(0,j,k) (:773-794); with the inflow plane fixed it depends
// on U(1), U(2), P(1), P(2) only.  Thread per interior (j, k).
__device__ __forceinline__ void adj_pin(const Geo &g, const double *E, double *lamU, double *lamP, int j, int k)
{
    const long c = lin(g, 0, j, k);
    const double L = lamP[c];
    lamP[c] = 0.0;
    const double dx = g.dx, Re = g.Re, u1 = E[j + (long)g.nY * k];
    const double f = 2.0 * dx / 3.0 * L;
    lamU[c + 1] += f * (u1 / dx + 2.0 / (dx * dx * Re));
    lamU[c + 2] += f * (-1.0 / (dx * dx * Re));
    lamP[c + 1] += 4.0 * L / 3.0;
    lamP[c + 2] += -L / 3.0;
}
// outflow pressure P(nX-1,j,k) = (3U(nX-1) - 4U(nX-2) + U(nX-3)) / (2 dx Re) (:767-771)
__device__ __forceinline__ void adj_pout(const Geo &g, double *lamU, double *lamP, int j, int k)
{
    const long c = lin(g, g.nX - 1, j, k);
    const double f = lamP[c] / (2.0 * g.dx * g.Re);
    lamP[c] = 0.0;
    lamU[c] += 3.0 * f;
    lamU[c - 1] += -4.0 * f;
    lamU[c - 2] += f;
}
// top pressure P(i,j,nZ-1) = (11W(nZ-1) - 18W(nZ-2) + 9W(nZ-3) - 2W(nZ-4)) JacInv(nZ-1) / (6 dXi Re) (:757-765)
__device__ __forceinline__ void adj_ptop(const Geo &g, double *lamW, double *lamP, int i, int j)
{
    const int kt = g.nZ - 1;
    const long c = lin(g, i, j, kt), sk = g.sZ;
    const double f = lamP[c] * g.JacInv[kt] / (6.0 * g.dXi * g.Re);
    lamP[c] = 0.0;
    lamW[c] += 11.0 * f;
    lamW[c - sk] += -18.0 * f;
    lamW[c - 2 * sk] += 9.0 * f;
    lamW[c - 3 * sk] += -2.0 * f;
}
// bottom pressure (:738-755): P(i,j,0) = P(i,j,1) - rt12 df1,
//   rt12 = -w1 (w2 - w1)/df1 + (rt1 + rt2 + rt3)/Re,
//   rt1 = (W(i-1,j,0) - 2 w1 + W(i+1,j,0))/dx^2, rt2 likewise in raw j +- 1,
//   rt3 = (2 df1 w3 - 2 df2 w2 + 2 (df2 - df1) w1)/(df1 df2^2 - df2 df1^2).
// (1) gather into lamW(.,.,0) over every wall point incl. span ghosts; reads
// the targets' lamP(.,.,0) without changing it
__device__ __forceinline__ void adj_pbot_w0(const Geo &g, const double *E, const double *lamP, double *lamW, int i, int j)
{
    const double df1 = g.df1, df2 = g.df2, Re = g.Re, dx = g.dx, dy = g.dy;
    auto tgt = [&](int ti, int tj) { return ti >= 1 && ti <= g.nX - 2 && tj >= 1 && tj <= g.nY - 2; };
    double acc = 0.0;
    if (tgt(i - 1, j)) acc += lamP[lin(g, i - 1, j, 0)] / (dx * dx * Re);
    if (tgt(i + 1, j)) acc += lamP[lin(g, i + 1, j, 0)] / (dx * dx * Re);
    if (tgt(i, j - 1)) acc += lamP[lin(g, i, j - 1, 0)] / (dy * dy * Re);
    if (tgt(i, j + 1)) acc += lamP[lin(g, i, j + 1, 0)] / (dy * dy * Re);
    acc = -df1 * acc;
    if (tgt(i, j)) {
        const long c = lin(g, i, j, 0);
        const double *w = E + (long)g.nY * g.nZ + c;
        const double w1 = w[0], w2 = w[g.sZ];
        const double den = (df1 * (df2 * df2) - (df2 * (df1 * df1)));
        const double d = -(w2 - 2.0 * w1) / df1 + (-2.0 / (dx * dx) - 2.0 / (dy * dy) + 2.0 * (df2 - df1) / den) / Re;
        acc += -df1 * lamP[c] * d;
    }
    lamW[lin(g, i, j, 0)] += acc;
}
// The four above in one launch: the inflow and outflow columns (j, k), the top
// plane (i, j), the bottom plane (i, j).  They read and write different values: the
// columns 0..2 and nX-3..nX-1 of planes 1..nZ-2, the planes nZ-4..nZ-1 of W and nZ-1
// of P, the plane 0 (nX, nZ >= 8).  With the three components of the velocity
// conditions a launch too, an adjoint step has 6 boundary launches instead of 15:
// gradients at 101x34x45 6.1 -> 5.85 ms, at 256x64x96 32.85 -> 32.45.
__global__ __launch_bounds__(256) void k_adj_pfaces(Geo g, const double *E, double *lamU, double *lamP)
{
    const long nx = (long)(g.nY - 2) * (g.nZ - 2), nt = (long)(g.nX - 2) * (g.nY - 2);
    long t = (long)blockIdx.x * 256 + threadIdx.x;
    if (t < nx) {
        const int j = (int)(t % (g.nY - 2)) + 1, k = (int)(t / (g.nY - 2)) + 1;
        adj_pin(g, E, lamU, lamP, j, k);
        adj_pout(g, lamU, lamP, j, k);
        return;
    }
    double *lamW = lamU + 2 * g.N;
    if ((t -= nx) < nt) {
        adj_ptop(g, lamW, lamP, (int)(t % (g.nX - 2)) + 1, (int)(t / (g.nX - 2)) + 1);
        return;
    }
    if ((t -= nt) < g.sZ) adj_pbot_w0(g, E, lamP, lamW, (int)(t % g.nX), (int)(t / g.nX));
}
// (2) per target: P(i,j,1) and W(i,j,1..2) terms, then the target is consumed
__global__ void k_adj_pbot_loc(Geo g, const double *__restrict__ E, double *__restrict__ lamP,
                               double *__restrict__ lamW)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x + 1, j = blockIdx.y + 1;
    if (i > g.nX - 2) return;
    const double df1 = g.df1, df2 = g.df2, Re = g.Re;
    const long c = lin(g, i, j, 0), sk = g.sZ;
    const double L = lamP[c];
    lamP[c] = 0.0;
    lamP[c + sk] += L;
    const double w1 = E[(long)g.nY * g.nZ + c];
    const double den = (df1 * (df2 * df2) - (df2 * (df1 * df1)));
    lamW[c + sk] += -df1 * L * (-w1 / df1 + (-2.0 * df2 / den) / Re);
    lamW[c + 2 * sk] += -df1 * L * ((2.0 * df1 / den) / Re);
}

// ============================================================================
// velocity boundary conditions, reversed (dnssetbl.f90:729-736), component blockIdx.z
// ============================================================================
// outflow u(nX-1,j,k) = (4u(nX-2) - u(nX-3))/3, k in [0,nZ-1]; thread per (j,k)
__global__ void k_adj_vout(Geo g, double *__restrict__ lam)
{
    lam += blockIdx.z * g.N;
    const int j = blockIdx.x * blockDim.x + threadIdx.x + 1, k = blockIdx.y;
    if (j > g.nY - 2) return;
    const long c = lin(g, g.nX - 1, j, k);
    const double L = lam[c];
    lam[c] = 0.0;
    lam[c - 1] += 4.0 * L / 3.0;
    lam[c - 2] += -L / 3.0;
}
// top u(i,j,nZ-1) = (4u(nZ-2) - u(nZ-3))/3, then the wall value u(i,j,0)
// (w = wall_w, the control: its adjoint is the gradient); thread per (i,j)
__global__ void k_adj_vtop_wall(Geo g, double *__restrict__ lam, double *__restrict__ grad)
{
    lam += blockIdx.z * g.N;
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y + 1;
    if (i >= g.nX) return;
    const long sk = g.sZ, ct = lin(g, i, j, g.nZ - 1), cw = lin(g, i, j, 0);
    const double L = lam[ct];
    lam[ct] = 0.0;
    lam[ct - sk] += 4.0 * L / 3.0;
    lam[ct - 2 * sk] += -L / 3.0;
    if (blockIdx.z == 2) grad[(long)i + (long)g.nX * j] += lam[cw];
    lam[cw] = 0.0;
}

// ============================================================================
// projection + pressure update, reversed (dnssetbl.f90:697-726)
// ============================================================================
// lamPhi(s) = [s interior] lamP(s) - dt (G^T lamU)(s), every point s
__global__ __launch_bounds__(256) void k_adj_proj(Geo g, const double *__restrict__ lamU, const double *__restrict__ lamP,
                                                 double *__restrict__ lamPhi)
{
    ALL3_IDX
    const long c = lin(g, i, j, k), N = g.N, sk = g.sZ;
    const double *lu = lamU, *lv = lamU + N, *lw = lamU + 2 * N;
    double gt = 0.0;
    if (j >= 1 && j <= g.nY - 2 && k >= 1 && k <= g.nZ - 2) {
        if (i - 1 >= 1 && i - 1 <= g.nX - 2) gt += 0.5 * g.invdx * lu[c - 1];
        if (i + 1 >= 1 && i + 1 <= g.nX - 2) gt -= 0.5 * g.invdx * lu[c + 1];
    }
    if (i >= 1 && i <= g.nX - 2 && k >= 1 && k <= g.nZ - 2 && j >= 1 && j <= g.nY - 2) {
        gt += 0.5 * g.invdy * (lv[lin(g, i, jm1_of(j, g.nY), k)] - lv[lin(g, i, jp1_of(j, g.nY), k)]);
    }
    if (i >= 1 && i <= g.nX - 2 && j >= 1 && j <= g.nY - 2) {
        if (k - 1 >= 1 && k - 1 <= g.nZ - 2) gt += 0.5 * g.invdXi * g.JacInv[k - 1] * lw[c - sk];
        if (k + 1 >= 1 && k + 1 <= g.nZ - 2) gt -= 0.5 * g.invdXi * g.JacInv[k + 1] * lw[c + sk];
    }
    lamPhi[c] = (inner(g, i, j, k) ? lamP[c] : 0.0) - g.dt * gt;
}
// face extrapolations of PCorr, reversed: x faces (k in [0,nZ-1]) then z faces
__global__ void k_adj_phi_x(Geo g, double *__restrict__ lp)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x + 1, k = blockIdx.y;
    if (j > g.nY - 2) return;
    const long c0 = lin(g, 0, j, k), cn = lin(g, g.nX - 1, j, k);
    const double L0 = lp[c0];
    lp[c0] = 0.0;
    lp[c0 + 1] += 4.0 * L0 / 3.0;
    lp[c0 + 2] += -L0 / 3.0;
    const double Ln = lp[cn];
    lp[cn] = 0.0;
    lp[cn - 1] += 5.0 * Ln / 2.0;
    lp[cn - 2] += -2.0 * Ln;
    lp[cn - 3] += Ln / 2.0;
}
__global__ void k_adj_phi_z(Geo g, double *__restrict__ lp)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y + 1;
    if (i >= g.nX) return;
    const long sk = g.sZ, c0 = lin(g, i, j, 0), cn = lin(g, i, j, g.nZ - 1);
    const double L0 = lp[c0];
    lp[c0] = 0.0;
    lp[c0 + sk] += 4.0 * L0 / 3.0;
    lp[c0 + 2 * sk] += -L0 / 3.0;
    const double Ln = lp[cn];
    lp[cn] = 0.0;
    lp[cn - sk] += 5.0 * Ln / 2.0;
    lp[cn - 2 * sk] += -2.0 * Ln;
    lp[cn - 3 * sk] += Ln / 2.0;
}

// ============================================================================
// PPE right-hand side, reversed (dnssetbl.f90:437-447): lamU += D^T lamB / dt
// ============================================================================
__global__ __launch_bounds__(256) void k_adj_div(Geo g, const double *__restrict__ lamB, double *__restrict__ lamU)
{
    ALL3_IDX
    const long c = lin(g, i, j, k), N = g.N, sk = g.sZ;
    const double rdt = 1.0 / g.dt;
    if (j >= 1 && j <= g.nY - 2 && k >= 1 && k <= g.nZ - 2) {
        double a = 0.0;
        if (i - 1 >= 1 && i - 1 <= g.nX - 2) a += lamB[c - 1];
        if (i + 1 >= 1 && i + 1 <= g.nX - 2) a -= lamB[c + 1];
        lamU[c] += 0.5 * g.invdx * rdt * a;
    }
    if (inner(g, i, j, k)) {
        const double a = lamB[lin(g, i, jm1_of(j, g.nY), k)] - lamB[lin(g, i, jp1_of(j, g.nY), k)];
        lamU[N + c] += 0.5 * g.invdy * rdt * a;
    }
    if (i >= 1 && i <= g.nX - 2 && j >= 1 && j <= g.nY - 2) {
        double a = 0.0;
        if (k - 1 >= 1 && k - 1 <= g.nZ - 2) a += lamB[c - sk] / (g.x3[k] - g.x3[k - 2]);
        if (k + 1 >= 1 && k + 1 <= g.nZ - 2) a -= lamB[c + sk] / (g.x3[k + 2] - g.x3[k]);
        lamU[2 * N + c] += rdt * a;
    }
}

// ============================================================================
// momentum RHS + Helmholtz boundary data + inflow, reversed
// (dnssetbl.f90:257-369,371-433)
// ============================================================================
// One direction of the transposed convection at a point s, from the values at
// offsets -2..2 (index q = offset + 2): f(p, q) the components, l(p, q) their
// adjoints (zero off the interior), component P the advecting velocity.
//  * A target at index q reads s at offset 2 - q, with the coefficient its own
//    advecting velocity, branch and second-order flag (bit q of `edge`) give:
//    acc[p] += coefficient l(p, q).
//  * The derivative of s's own term with respect to its advecting velocity,
//    summed over the components with their adjoints, is returned.
// d(q): the spacing of the target's Peclet number; jz(q) scales its coefficient
// (wall-normal: JacInv of its plane).  The values are read where they are
// used, a few at a time (the scheduling barriers keep it so): read up front
// they take 230 registers instead of 156.
template <int P, class Ff, class Fl, class Fd, class Fj>
__device__ __forceinline__ double conv_adj(Ff f, Fl l, Fd d, Fj jz, unsigned edge, double Re, double inv, double c12,
                                           double (&acc)[3])
{
    const double ci = c12 * inv, qi = 0.25 * inv, hi = 0.5 * inv;
    constexpr double wc[5] = {-1.0, 8.0, 0.0, -8.0, 1.0}, w4[5] = {1.0, -4.0, 6.0, -4.0, 1.0};   // at offset 2 - q
#pragma unroll
    for (int q = 0; q < 5; q++) {
        const double a = f(P, q);
        const double B = fabs(Re * a * d(q)) > 2.0 ? fabs(a) * qi : 0.0;
        const double full = __builtin_fma(w4[q], B, wc[q] * (a * ci));
        const double half = q == 1 ? a * hi : q == 3 ? -(a * hi) : 0.0;
        const double cf = ((edge >> q) & 1 ? half : full) * jz(q);
#pragma unroll
        for (int p = 0; p < 3; p++) acc[p] = __builtin_fma(cf, l(p, q), acc[p]);
        __builtin_amdgcn_sched_barrier(0);
    }
    double E = 0.0, M = 0.0, D = 0.0;
#pragma unroll
    for (int p = 0; p < 3; p++) {
        const double lc = l(p, 2), f0 = f(p, 0), f1 = f(p, 1), f3 = f(p, 3), f4 = f(p, 4);
        E = __builtin_fma(lc, f3 - f1, E);
        M = __builtin_fma(lc, f0 - f4, M);
        D = __builtin_fma(lc, __builtin_fma(-4.0, f3 + f1, __builtin_fma(6.0, f(p, 2), f4 + f0)), D);
        __builtin_amdgcn_sched_barrier(0);
    }
    const double a = f(P, 2);
    const double sk = fabs(Re * a * d(2)) > 2.0 ? sgn(a) * qi : 0.0;
    return ((edge >> 2) & 1 ? hi * E : __builtin_fma(sk, D, ci * __builtin_fma(8.0, E, M))) * jz(2);
}

// U is the step's linearisation point (after the inflow overwrite), lamQ the
// adjoint of Q (interior, zero elsewhere), lamU the adjoint of the Helmholtz
// output on entry.  On exit lamU holds the adjoint of the step's input
// velocity; lamP receives -dt Gp^T lamQ.  The span ghost rows pass through and
// are not visited.
//
// A block of 64 x AM_TJ columns marches a chunk of k planes.  The planes
// k-2..k+2 of U and lamQ live in register queues; plane k of the six fields,
// with its two-point halo (periodic span rows, streamwise columns clamped to
// the faces, where lamQ is zero), is staged in LDS (two buffers by plane
// parity, one LDS-only barrier a plane), so a thread loads each plane's six
// centre values and at most one halo element per field, a plane before they
// are used.  A thread per point that read its 100 stencil values through L1
// and L2 spent its time waiting for them, and so did a k march that took only
// the wall-normal ones from registers.  At 1024x192x160 (FP32 states) these
// took 2.22 and 1.87 ms, this one 1.04 ms (256x64x96 FP64: 91, 121 and 54 us);
// 0.50 ms is the field traffic at a copy's rate.
// T: storage type of U (mixed contexts keep FP32 states; the arithmetic and
// the adjoint are FP64).
#define AM_TJ 8
#define AM_W 68
#define AM_SINK (AM_W * (AM_TJ + 4))       // tile slot of threads and elements outside the field
#define AM_F (AM_SINK + 2)
#define AM_KMAX 32
template <class T>
__global__ __launch_bounds__(64 * AM_TJ) __attribute__((amdgpu_waves_per_eu(3)))
void k_adj_mom(Geo g, const T *__restrict__ U, const double *__restrict__ lamQ, double *__restrict__ lamU,
               double *__restrict__ lamP, int kchunk, unsigned nbx, unsigned nby, unsigned nbz)
{
    __shared__ T tu[2][3][AM_F];
    __shared__ double tq[2][3][AM_F];
    __shared__ double sz[2][AM_KMAX + 4];                         // dz3, JacInv of the planes k0-2 .. (0: no target)
    const unsigned L = xcd_remap(blockIdx.x, nbx * nby * nbz);
    const unsigned bx = L % nbx, by = (L / nbx) % nby, bz = L / (nbx * nby);
    const int nX = g.nX, nY = g.nY, nZ = g.nZ;
    const int t = threadIdx.x, lx = t & 63, ly = t >> 6;
    const int i0 = bx * 64, j0 = by * AM_TJ + 1;
    const int ti = min(64, nX - i0), tj = min(AM_TJ, nY - 1 - j0);    // tile columns and rows inside the field
    const bool live = lx < ti && ly < tj;
    const int i = i0 + min(lx, ti - 1), j = j0 + min(ly, tj - 1);
    const int k0 = (int)bz * kchunk, k1 = min(k0 + kchunk, nZ);
    const int sk = (int)g.sZ, c0 = i + nX * j;                   // 3N < 2^31 (checked at create)
    const long N = g.N;
    const double dt = g.dt, Re = g.Re, c12 = g.c12, h = g.dt / g.Re;
    const bool in_i = i >= 1 && i <= nX - 2;
    if (t < kchunk + 4) {
        const int kk = k0 - 2 + t;
        const bool ok = kk >= 1 && kk <= nZ - 2;
        sz[0][t] = ok ? g.x3[kk + 1] - g.x3[kk] : 0.0;
        sz[1][t] = ok ? g.JacInv[kk] : 0.0;
    }
    // second-order rows: bit q for the target at offset q - 2
    unsigned ex = 0, ey = 0;
#pragma unroll
    for (int q = 0; q < 5; q++) {
        const int tx = i + q - 2, ty = j + q - 2;
        if (tx <= 1 || tx >= nX - 2) ex |= 1u << q;
        if (ty == 1 || ty == nY - 2 || ty == nY - 1 || ty == 0) ey |= 1u << q;   // rows 0 and nY-1 stand for nY-2 and 1
    }
    // the thread's tile slot and its halo element (at most one per field)
    const int cslot = live ? (2 + ly) * AM_W + 2 + lx : AM_SINK;
    int hslot = AM_SINK, hoff = c0;
    {
        const int n = nY - 2;
        if (t < 256) {
            const int hr = t >> 6, hc = t & 63;
            const int v = hr < 2 ? j0 - 2 + hr : j0 + tj + hr - 2;
            if (hc < ti) {
                hslot = (hr < 2 ? hr : tj + hr) * AM_W + 2 + hc;
                hoff = ((((v - 1) % n + n) % n) + 1) * nX + i0 + hc;
            }
        } else if (t < 256 + 4 * AM_TJ) {
            const int hr = (t - 256) >> 2, hc = (t - 256) & 3;
            const int ii = hc < 2 ? i0 - 2 + hc : i0 + ti + hc - 2;
            if (hr < tj) {
                hslot = (2 + hr) * AM_W + (hc < 2 ? hc : ti + hc);
                hoff = (j0 + hr) * nX + min(max(ii, 0), nX - 1);
            }
        }
    }
    auto kp = [&](int kk) { return sk * max(0, min(kk, nZ - 1)); };
    // queues before step k's shift: planes k-3..k+1; then the loads in flight:
    // centre values of plane k+2, halo values of plane k
    double zU[3][5], zL[3][5], pl[3], hl[3];
    T pu[3], hu[3];
#pragma unroll
    for (int q = 1; q < 5; q++) {
        const int o = c0 + kp(k0 - 3 + q);
#pragma unroll
        for (int p = 0; p < 3; p++) {
            zU[p][q] = (double)U[p * N + o];
            zL[p][q] = lamQ[p * N + o];
        }
    }
#pragma unroll
    for (int p = 0; p < 3; p++) {
        pu[p] = U[p * N + c0 + kp(k0 + 2)];
        pl[p] = lamQ[p * N + c0 + kp(k0 + 2)];
        hu[p] = U[p * N + hoff + kp(k0)];
        hl[p] = lamQ[p * N + hoff + kp(k0)];
    }
    const int a0 = (2 + min(ly, tj - 1)) * AM_W + 2 + min(lx, ti - 1);
    for (int k = k0; k < k1; k++) {
        const int b = k & 1, c = c0 + sk * k;
#pragma unroll
        for (int p = 0; p < 3; p++) {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                zU[p][q] = zU[p][q + 1];
                zL[p][q] = zL[p][q + 1];
            }
            zU[p][4] = (double)pu[p];
            zL[p][4] = pl[p];
            tu[b][p][cslot] = (T)zU[p][2];
            tq[b][p][cslot] = zL[p][2];
            tu[b][p][hslot] = hu[p];
            tq[b][p][hslot] = hl[p];
        }
#pragma unroll
        for (int p = 0; p < 3; p++) {
            pu[p] = U[p * N + c0 + kp(k + 3)];
            pl[p] = lamQ[p * N + c0 + kp(k + 3)];
            hu[p] = U[p * N + hoff + kp(k + 1)];
            hl[p] = lamQ[p * N + hoff + kp(k + 1)];
        }
        const double lp = lamP[c];
        lds_barrier();
        const bool in_k = k >= 1 && k <= nZ - 2, si = in_i && in_k;
        double acc[3] = {0.0, 0.0, 0.0}, gp = 0.0, adv[3] = {0.0, 0.0, 0.0};
        auto one = [](int) { return 1.0; };
        __builtin_amdgcn_sched_barrier(0);
        if (in_k) {                                              // uniform over the block
            auto fx = [&](int p, int q) { return q == 2 ? zU[p][2] : (double)tu[b][p][a0 + q - 2]; };
            auto lqx = [&](int p, int q) { return q == 2 ? zL[p][2] : tq[b][p][a0 + q - 2]; };
            adv[0] = conv_adj<0>(fx, lqx, [&](int) { return g.dx; }, one, ex, Re, g.invdx, c12, acc);
            gp = 0.5 * g.invdx * (lqx(0, 1) - lqx(0, 3));
            auto fy = [&](int p, int q) { return q == 2 ? zU[p][2] : (double)tu[b][p][a0 + (q - 2) * AM_W]; };
            auto lqy = [&](int p, int q) { return q == 2 ? zL[p][2] : tq[b][p][a0 + (q - 2) * AM_W]; };
            adv[1] = conv_adj<1>(fy, lqy, [&](int) { return g.dy; }, one, ey, Re, g.invdy, c12, acc);   // l = 0 in the face columns
            gp += 0.5 * g.invdy * (lqy(1, 1) - lqy(1, 3));
        }
        // wall-normal (targets off the interior have lamQ = 0 and JacInv = 0 here)
        {
            unsigned ez = 0;
#pragma unroll
            for (int q = 0; q < 5; q++)
                if (k + q - 2 <= 1 || k + q - 2 >= nZ - 2) ez |= 1u << q;
            auto jz = [&](int q) { return sz[1][k - k0 + q]; };
            adv[2] = conv_adj<2>([&](int p, int q) { return zU[p][q]; }, [&](int p, int q) { return zL[p][q]; },
                                 [&](int q) { return sz[0][k - k0 + q]; }, jz, ez, Re, g.invdXi, c12, acc);
            gp += 0.5 * g.invdXi * (jz(1) * zL[2][1] - jz(3) * zL[2][3]);
        }
        double out[3];
        // base: the Helmholtz solve overwrote the interior (its input adjoint is
        // lamQ through Q's U term); faces pass through and feed the Helmholtz
        // right-hand side h B u(face)
        if (si) {
#pragma unroll
            for (int p = 0; p < 3; p++) out[p] = __builtin_fma(-dt, acc[p] + adv[p], zL[p][2]);
        } else {
#pragma unroll
            for (int p = 0; p < 3; p++) {
                double o = lamU[p * N + c];
                if (in_k) {
                    if (i == 0) o += h * g.Aw * tq[b][p][a0 + 1];
                    if (i == nX - 1) o += h * g.Ae * tq[b][p][a0 - 1];
                }
                if (in_i) {
                    if (k == 0) o += h * g.Ab[1] * zL[p][3];
                    if (k == nZ - 1) o += h * g.At[nZ - 2] * zL[p][1];
                }
                out[p] = __builtin_fma(-dt, acc[p], o);
                // the inflow plane is overwritten by the (frozen) recycling inflow
                if (i == 0 && in_k) out[p] = 0.0;
            }
        }
        if (live) {
#pragma unroll
            for (int p = 0; p < 3; p++) lamU[p * N + c] = out[p];
            lamP[c] = lp - dt * gp;
        }
    }
}

// J += cJ * sum_{i in [i0,i1]} tau(i), one thread, fixed order
__global__ void k_tau_acc(const double *__restrict__ tau, int i0, int i1, double cJ, double *__restrict__ J)
{
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    double a = 0.0;
    for (int i = i0; i <= i1; i++) a += tau[i];
    J[0] = J[0] + cJ * a;
}

// ============================================================================
// host launchers
// ============================================================================
void launch_tau_acc(const Geo &g, const double *tau, int i0, int i1, double cJ, double *J, hipStream_t s)
{
    hipLaunchKernelGGL(k_tau_acc, dim3(1), dim3(64), 0, s, tau, i0, i1, cJ, J);
}
template <class T>
void launch_helm_rfield(const Geo &g, const T *Q, const T *u, T *r, int ncomp, hipStream_t s)
{
    hipLaunchKernelGGL(k_helm_rfield<T>, comp3(g, ncomp), dim3(256), 0, s, g, Q, u, r);
}
template void launch_helm_rfield<double>(const Geo &, const double *, const double *, double *, int, hipStream_t);
template void launch_helm_rfield<float>(const Geo &, const float *, const float *, float *, int, hipStream_t);
template <class To>
void launch_opT_res(const Geo &g, const double *b, const double *x, double alpha, double beta, To *r, int ncomp, hipStream_t s)
{
    hipLaunchKernelGGL(k_opT_res<To>, comp3(g, ncomp), dim3(256), 0, s, g, b, x, alpha, beta, r);
}
template void launch_opT_res<double>(const Geo &, const double *, const double *, double, double, double *, int, hipStream_t);
template void launch_opT_res<float>(const Geo &, const double *, const double *, double, double, float *, int, hipStream_t);
void launch_adj_tau(const Geo &g, double *lamU, int i0, int i1, double cJ, hipStream_t s)
{
    hipLaunchKernelGGL(k_adj_tau, dim3((g.nX + 255) / 256, g.nY - 2), dim3(256), 0, s, g, lamU, i0, i1, cJ);
}
// pressure then velocity boundary conditions, reversed; grad += adjoint of wall_w
void launch_adj_bcs(const Geo &g, const double *E, double *lamU, double *lamP, double *grad, hipStream_t s)
{
    const long N = g.N;
    double *lamW = lamU + 2 * N;
    const dim3 b256(256);
    hipLaunchKernelGGL(k_adj_span, dim3((g.nX + 255) / 256, g.nZ), b256, 0, s, g, lamP);
    const long nf = (long)(g.nY - 2) * (g.nZ - 2) + (long)(g.nX - 2) * (g.nY - 2) + g.sZ;
    hipLaunchKernelGGL(k_adj_pfaces, dim3((unsigned)((nf + 255) / 256)), b256, 0, s, g, E, lamU, lamP);
    hipLaunchKernelGGL(k_adj_pbot_loc, dim3((g.nX - 2 + 255) / 256, g.nY - 2), b256, 0, s, g, E, lamP, lamW);
    hipLaunchKernelGGL(k_adj_span, dim3((g.nX + 255) / 256, g.nZ, 3), b256, 0, s, g, lamU);
    hipLaunchKernelGGL(k_adj_vout, dim3((g.nY - 2 + 255) / 256, g.nZ, 3), b256, 0, s, g, lamU);
    hipLaunchKernelGGL(k_adj_vtop_wall, dim3((g.nX + 255) / 256, g.nY - 2, 3), b256, 0, s, g, lamU, grad);
}
void launch_adj_proj(const Geo &g, const double *lamU, const double *lamP, double *lamPhi, hipStream_t s)
{
    hipLaunchKernelGGL(k_adj_proj, all3(g), dim3(256), 0, s, g, lamU, lamP, lamPhi);
    hipLaunchKernelGGL(k_adj_phi_x, dim3((g.nY - 2 + 255) / 256, g.nZ), dim3(256), 0, s, g, lamPhi);
    hipLaunchKernelGGL(k_adj_phi_z, dim3((g.nX + 255) / 256, g.nY - 2), dim3(256), 0, s, g, lamPhi);
}
void launch_adj_div(const Geo &g, const double *lamB, double *lamU, hipStream_t s)
{
    hipLaunchKernelGGL(k_adj_div, all3(g), dim3(256), 0, s, g, lamB, lamU);
}
// planes per block of k_adj_mom: the chunk with the least (rounds of blocks
// over the 256 CUs, one block of 8 waves each at 156 registers; 6 rows a block
// and two blocks were 1-2 % slower, 128 registers spill) x (planes + 4 queue
// planes), at most AM_KMAX
template <class T>
void launch_adj_mom(const Geo &g, const T *U, const double *lamQ, double *lamU, double *lamP, hipStream_t s)
{
    const unsigned nbx = (g.nX + 63) / 64, nby = (g.nY - 2 + AM_TJ - 1) / AM_TJ;
    int kc = 1;
    long best = -1;
    for (int q = AM_KMAX; q >= 1; q--) {
        const long cost = ((long)nbx * nby * ((g.nZ + q - 1) / q) + 255) / 256 * (q + 4);
        if (best < 0 || cost < best) { best = cost; kc = q; }
    }
    const unsigned nbz = (g.nZ + kc - 1) / kc;
    hipLaunchKernelGGL(k_adj_mom<T>, dim3(nbx * nby * nbz), dim3(64 * AM_TJ), 0, s, g, U, lamQ, lamU, lamP, kc, nbx, nby, nbz);
}
template void launch_adj_mom<double>(const Geo &, const double *, const double *, double *, double *, hipStream_t);
template void launch_adj_mom<float>(const Geo &, const float *, const double *, double *, double *, hipStream_t);

}  // namespace tbl
