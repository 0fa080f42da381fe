// tbl_krylov.hip -- restarted left-preconditioned GMRES kernels for the
// pressure Poisson equation (reference: dnssetbl/dnssetbl.f90:462-671).
//
// The reference runs modified Gram-Schmidt with one MPI_Allreduce per dot
// product and keeps h, c, s, g, y on every rank.  Here:
//  * Krylov vectors V_i are stored unnormalised with a scale sigma_i (the
//    true basis vector is sigma_i V_i), so no normalisation pass is needed;
//  * the j+1 dot products of one Arnoldi step are computed in one pass that
//    streams the new vector once per group of 8 basis vectors (classical
//    Gram-Schmidt; equal to the reference's modified Gram-Schmidt in exact
//    arithmetic), with wavefront-shuffle block reductions into fixed-order
//    partials (deterministic);
//  * the update z -= sum coef_i V_i and ||z||^2 are fused in one pass;
//  * Hessenberg, Givens rotations, the residual estimate, the stopping test
//    and the back substitution run on the device (single-block kernels), so
//    the host only polls a status word.
// Vectors are full-grid arrays whose boundary entries are zero, so every
// vector kernel runs over the contiguous range [0, N).
#include "tbl_dev.h"
#include "tbl_launch.h"

namespace tbl {

static constexpr int VB = 256;     // threads per block of the vector kernels
static constexpr int DG = 8;       // dot products per streaming pass

// blocks of the vector kernels: 1024 values each in FP64 (four a thread), so
// that a small grid still gives every CU its share, at most 4096 (90x80x50, up
// to 50 Krylov vectors, 352 blocks instead of 88: k_dots 76 -> 33 us with the
// grouped block sums, k_update 23 -> 16 us).  FP32 keeps 4096 values: the order of a norm's
// partials follows the blocks, and mixed solves keep their bits.
unsigned vec_blocks(long N, bool single)
{
    const long per = single ? 4096 : 1024;
    long nb = (N + per - 1) / per;
    if (nb > 4096) nb = 4096;
    if (nb < 1) nb = 1;
    return (unsigned)nb;
}

__device__ __forceinline__ void chunk_of(long N, long &b0, long &b1)
{
    const long nb = gridDim.x;
    const long per = ((N + nb - 1) / nb + 63) & ~63L;
    b0 = per * blockIdx.x;
    b1 = min(N, b0 + per);
}

template <class T>
__global__ __launch_bounds__(VB) void k_norm2(const T *__restrict__ x, long N, double *__restrict__ part,
                                             const int *__restrict__ active)
{
    __shared__ double sh[VB / 64];
    if (active && !*active) return;
    long b0, b1;
    chunk_of(N, b0, b1);
    double a = 0.0;
    // four elements per pass (four loads in flight per thread), summed in
    // ascending e as with one element per pass
    long e = b0 + threadIdx.x;
    for (; e + 3 * VB < b1; e += 4 * VB) {
        T v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = x[e + u * VB];
#pragma unroll
        for (int u = 0; u < 4; u++) { const double d = v[u]; a += d * d; }
    }
    for (; e < b1; e += VB) { double v = x[e]; a += v * v; }
    double s = block_sum<VB>(a, sh, threadIdx.x);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ __launch_bounds__(VB) void k_fill(double *__restrict__ x, double v, long n)
{
    for (long e = (long)blockIdx.x * VB + threadIdx.x; e < n; e += (long)gridDim.x * VB) x[e] = v;
}
void launch_fill(double *x, double v, long n, hipStream_t s)
{
    hipLaunchKernelGGL(k_fill, dim3(vec_blocks(n, false)), dim3(VB), 0, s, x, v, n);
}

// deterministic sum of nb partials by one block of NT threads
template <int NT = VB>
__device__ __forceinline__ double fin_sum(const double *part, int nb, double *sh)
{
    double a = 0.0;
#pragma unroll 8
    for (int q = threadIdx.x; q < nb; q += NT) a += part[q];
    return block_sum<NT>(a, sh, threadIdx.x);
}
// finishing blocks of the grid-wide reductions (up to ~16k partials)
static constexpr int FB = 1024;

// Start of a solve: the control block (the last workgroup), zeroed and given the
// solve's parameters, and the zero faces of the PCorr buffers, dnssetbl.f90:451-460
// (the others).  A kernel rather than a copy: the block is 33 KB, and a copy
// from pageable host memory holds the host until it has been staged.
__global__ __launch_bounds__(VB) void k_gm_init(Geo g, GmCtrl *c, double errtol, double inner_tol, int kmax, int mmax,
                                               int mode, double *PC, double *PC2)
{
    if (blockIdx.x + 1 < gridDim.x) {
        const long nX = g.nX, nY = g.nY, nZ = g.nZ, fz = nX * nY, fy = nX * nZ, fx = nY * nZ;
        long t = (long)blockIdx.x * VB + threadIdx.x, x;
        if (t < 2 * fz) {
            x = t % fz + (t < fz ? 0 : fz * (nZ - 1));
        } else if ((t -= 2 * fz) < 2 * fy) {
            const long q = t % fy;
            x = q % nX + nX * ((t < fy ? 0 : nY - 1) + nY * (q / nX));
        } else {
            if ((t -= 2 * fy) >= 2 * fx) return;
            x = (t < fx ? 0 : nX - 1) + nX * (t % fx);
        }
        PC[x] = 0.0;
        if (PC2) PC2[x] = 0.0;
        return;
    }
    static_assert(sizeof(GmCtrl) % sizeof(double) == 0, "GmCtrl is cleared in doubles");
    double *w = reinterpret_cast<double *>(c);
    for (unsigned q = threadIdx.x; q < sizeof(GmCtrl) / sizeof(double); q += VB) w[q] = 0.0;
    __syncthreads();
    if (threadIdx.x == 0) {
        c->errtol = errtol;
        c->inner_tol = inner_tol;
        c->kmax = kmax;
        c->mmax = mmax;
        c->mode = mode;
        c->st.sumnor = 1.0;
    }
}

__global__ __launch_bounds__(64) void k_publish(const unsigned long long *__restrict__ src, int words, Pub P)
{
    unsigned long long *d = static_cast<unsigned long long *>(P.dst);
    for (int q = threadIdx.x; q < words; q += 64) d[q] = src[q];
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(P.seq, P.val, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
void launch_publish(const void *src, int words, const Pub &pub, hipStream_t s)
{
    hipLaunchKernelGGL(k_publish, dim3(1), dim3(64), 0, s, (const unsigned long long *)src, words, pub);
}

// Start of a cycle in true-residual mode from the residual norm res (one thread)
__device__ __forceinline__ void start_true(GmCtrl *c, double res)
{
    GmStatus &st = c->st;
    c->inner_ref = res;
    // stop the cycle at inner_tol, or earlier once the estimated reduction
    // already brings the true residual below the target (with margin)
    const double need = res > 0.0 ? 0.3 * c->errtol * c->bnorm / res : 1.0;
    c->cycle_tol = need > c->inner_tol ? need : c->inner_tol;
    // pRhs = 0: the exact solution is PCorr = 0, which the host sets (the
    // relative test could only be met by an exact zero residual)
    if (c->bnorm == 0.0) st.zero_rhs = 1;
    const bool done = res <= c->errtol * c->bnorm || res == 0.0 || c->bnorm == 0.0;
    st.sumav = c->bnorm > 0.0 ? res / c->bnorm : 0.0;
    st.active = done ? 0 : 1;
    if (done) { st.outer_done = 1; st.conv = 1; }
}
// V_0 with norm rho opens a cycle (all threads; before one thread's stores)
__device__ __forceinline__ void open_cycle(GmCtrl *c, double rho)
{
    for (int q = threadIdx.x; q <= TBL_KMAX_LIMIT + 1; q += FB) c->g[q] = q ? 0.0 : rho;
    if (threadIdx.x == 0) c->sigma[0] = rho > 0.0 ? 1.0 / rho : 0.0;
}

// Cycle start: r was formed in double (true residual partials part_r), and
// V_0 = M^{-1} r (partials part_z of ||V_0||^2; part_r itself in true-residual
// mode).  dnssetbl.f90:536-546.
__global__ __launch_bounds__(FB) void k_fin_start(GmCtrl *c, const double *part_r, int nb_r,
                                                 const double *part_z, int nb_z, int first,
                                                 const double *part_b)
{
    __shared__ double sh[FB / 64];
    __shared__ double rho_s;
    const double r2 = fin_sum<FB>(part_r, nb_r, sh);
    const double z2 = part_z == part_r ? r2 : fin_sum<FB>(part_z, nb_z, sh);
    const double b2 = part_b ? fin_sum<FB>(part_b, nb_r, sh) : 0.0;
    if (threadIdx.x == 0) rho_s = sqrt(z2);
    __syncthreads();
    const double rho = rho_s;
    open_cycle(c, rho);
    if (threadIdx.x != 0) return;
    GmStatus &st = c->st;
    if (part_b) c->bnorm = sqrt(b2);
    st.true_res = sqrt(r2);
    st.cycle += 1;
    st.kit = 0;
    st.rho = rho;
    if (!(rho == rho) || !(st.true_res == st.true_res)) {
        st.nan = 1; st.active = 0; st.outer_done = 1;
    } else if (c->mode == GM_MODE_REF) {
        if (first) st.sumnor = rho;
        st.sumav = rho / st.sumnor;
        const bool go = (st.sumav > c->errtol) && rho > 0.0;
        st.active = go ? 1 : 0;
        if (!go) { st.outer_done = 1; st.conv = 1; }
    } else {
        start_true(c, rho);
    }
}

// A cycle whose preconditioner inverts A nearly exactly needs no Arnoldi step:
// PCorr + z_0 (z_0 = M^{-1} r, the Krylov step with coefficient 1) is formed
// together with its own residual (k_resid_upd, RU_UNIT), and that residual
// decides.  Accepted when it meets what the cycle asked for, it counts as the
// cycle's one step:
//  * true-residual mode: the residual reached the target, or fell by the
//    cycle's tolerance; the next cycle is open (its V_0 is that residual);
//  * the reference's rule: ||M^{-1} r|| (part_z) fell by errtol; the solve
//    has ended.
// Otherwise the cycle stays open and the host runs its Arnoldi steps from
// z_0 as if nothing had been tried.
__global__ __launch_bounds__(FB) void k_fin_unit(GmCtrl *c, const double *part_r, int nb_r, const double *part_z,
                                                int nb_z, Pub pub)
{
    __shared__ double sh[FB / 64];
    __shared__ double res_s;
    __shared__ int ok_s;
    GmStatus &st = c->st;
    if (!st.active) {
        if (threadIdx.x == 0) {
            st.unit_ok = 0;
            publish(pub, &st);
        }
        return;
    }
    const bool ref = c->mode == GM_MODE_REF;
    const double r2 = fin_sum<FB>(part_r, nb_r, sh);
    const double z2 = ref ? fin_sum<FB>(part_z, nb_z, sh) : 0.0;
    if (threadIdx.x == 0) {
        const double res = sqrt(r2), rho = sqrt(z2);
        bool ok;
        if (!(res == res) || !(rho == rho)) {
            st.nan = 1; st.active = 0; st.outer_done = 1;
            ok = false;
        } else if (ref) {
            ok = rho / st.sumnor <= c->errtol;
            if (ok) { st.sumav = rho / st.sumnor; st.active = 0; st.outer_done = 1; st.conv = 1; }
        } else {
            ok = res <= c->errtol * c->bnorm || res <= c->cycle_tol * c->inner_ref;
            if (ok) { st.cycle += 1; start_true(c, res); }
        }
        if (ok) { st.total += 1; st.kit = ref ? 1 : 0; st.rho = ref ? rho : res; st.true_res = res; }
        st.unit_ok = ok ? 1 : 0;
        publish(pub, &st);
        ok_s = ok && !ref;
        res_s = res;
    }
    __syncthreads();
    if (ok_s) open_cycle(c, res_s);
}

// d_i = <V_i, z> for i = 0..j, streamed in groups of DG basis vectors.
template <class T>
__global__ __launch_bounds__(VB) void k_dots(const T *__restrict__ V, long ldv, int j, long N,
                                            const GmCtrl *__restrict__ c, double *__restrict__ part)
{
    __shared__ double sh[2][DG][VB / 64];
    if (!c->st.active) return;
    const T *__restrict__ z = V + (long)(j + 1) * ldv;
    long b0, b1;
    chunk_of(N, b0, b1);
    const int nb = gridDim.x;
    for (int i0 = 0; i0 <= j; i0 += DG) {
        double acc[DG];
#pragma unroll
        for (int q = 0; q < DG; q++) acc[q] = 0.0;
        const int ng = min(DG, j + 1 - i0);
        // four elements per pass (four loads of each vector in flight per
        // thread); every sum runs in ascending e as with one element per pass
        long e = b0 + threadIdx.x;
        for (; e + 3 * VB < b1; e += 4 * VB) {
            double zv[4];
#pragma unroll
            for (int u = 0; u < 4; u++) zv[u] = z[e + u * VB];
#pragma unroll
            for (int q = 0; q < DG; q++) {
                if (q < ng) {
                    const T *Vq = V + (long)(i0 + q) * ldv + e;
                    T vq[4];
#pragma unroll
                    for (int u = 0; u < 4; u++) vq[u] = Vq[u * VB];
#pragma unroll
                    for (int u = 0; u < 4; u++) acc[q] += (double)vq[u] * zv[u];
                }
            }
        }
        for (; e < b1; e += VB) {
            const double zv = z[e];
#pragma unroll
            for (int q = 0; q < DG; q++)
                if (q < ng) acc[q] += (double)V[(long)(i0 + q) * ldv + e] * zv;
        }
        // the group's block sums together, each in block_sum's order
        const int par = (i0 / DG) & 1;
#pragma unroll
        for (int q = 0; q < DG; q++) {
            const double s = wave_sum(acc[q]);
            if ((threadIdx.x & 63) == 0) sh[par][q][threadIdx.x >> 6] = s;
        }
        __syncthreads();
        if (threadIdx.x < ng) {
            double s = 0.0;
#pragma unroll
            for (int w = 0; w < VB / 64; w++) s += sh[par][threadIdx.x][w];
            part[(long)(i0 + threadIdx.x) * nb + blockIdx.x] = s;
        }
    }
}

// z = M^{-1} A v_j with v_j normalised (the Poisson apply scales by sigma_j), so
// h(i,j) = <v_i, z> = sigma_i d_i and z - sum h(i,j) v_i = z - sum sigma_i^2 d_i V_i
// Block i forms the i-th product (one block in turn for all: 27 -> 4.8 us an
// Arnoldi step at up to 50 vectors).
__global__ __launch_bounds__(VB) void k_fin_dots(GmCtrl *c, const double *part, int nb, int j)
{
    __shared__ double sh[VB / 64];
    if (!c->st.active) return;
    const int i = blockIdx.x;
    const double d = fin_sum(part + (long)i * nb, nb, sh);
    if (threadIdx.x == 0) {
        GM_H(c, i, j) = c->sigma[i] * d;
        c->coef[i] = c->sigma[i] * c->sigma[i] * d;
    }
}

// z -= sum_i coef_i V_i (double arithmetic), partials of ||z||^2; STORE false
// leaves z as it was (the same norm: of the values rounded as stored)
template <class T, bool STORE>
__global__ __launch_bounds__(VB) void k_update(const T *__restrict__ V, long ldv, int j, long N,
                                              GmCtrl *__restrict__ c, double *__restrict__ part)
{
    __shared__ double sh[VB / 64];
    __shared__ double co[TBL_KMAX_LIMIT + 1];
    if (!c->st.active) return;
    for (int q = threadIdx.x; q <= j; q += VB) co[q] = c->coef[q];
    __syncthreads();
    T *z = const_cast<T *>(V) + (long)(j + 1) * ldv;
    long b0, b1;
    chunk_of(N, b0, b1);
    double a = 0.0;
    // four elements per pass, so that each thread has four loads of every
    // vector in flight; each element's operations and the order of the
    // squares' accumulation (ascending e) are those of one element per pass
    long e = b0 + threadIdx.x;
    for (; e + 3 * VB < b1; e += 4 * VB) {
        double s[4];
#pragma unroll
        for (int u = 0; u < 4; u++) s[u] = z[e + u * VB];
        for (int i = 0; i <= j; i++) {
            const double ci = co[i];
            const T *Vi = V + (long)i * ldv + e;
            T vi[4];
#pragma unroll
            for (int u = 0; u < 4; u++) vi[u] = Vi[u * VB];
#pragma unroll
            for (int u = 0; u < 4; u++) s[u] -= ci * (double)vi[u];
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const T st = (T)s[u];
            if (STORE) z[e + u * VB] = st;
            const double sd = st;
            a += sd * sd;
        }
    }
    for (; e < b1; e += VB) {
        double s = z[e];
        for (int i = 0; i <= j; i++) s -= co[i] * (double)V[(long)i * ldv + e];
        const T st = (T)s;
        if (STORE) z[e] = st;
        const double sd = st;
        a += sd * sd;
    }
    double s = block_sum<VB>(a, sh, threadIdx.x);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// new column of the Hessenberg, Givens rotations, residual estimate and the
// inner stopping test (dnssetbl.f90:619-655)
__global__ __launch_bounds__(VB) void k_fin_update(GmCtrl *c, const double *part, int nb, int j)
{
    __shared__ double sh[VB / 64];
    if (!c->st.active) return;
    double z2 = fin_sum(part, nb, sh);
    if (threadIdx.x != 0) return;
    GmStatus &st = c->st;
    const double nrm = sqrt(z2);
    GM_H(c, j + 1, j) = nrm;
    c->sigma[j + 1] = nrm > 0.0 ? 1.0 / nrm : 0.0;
    for (int i = 0; i < j; i++) {
        const double hik = c->cs[i] * GM_H(c, i, j) - c->sn[i] * GM_H(c, i + 1, j);
        const double hipk = c->sn[i] * GM_H(c, i, j) + c->cs[i] * GM_H(c, i + 1, j);
        GM_H(c, i, j) = hik;
        GM_H(c, i + 1, j) = hipk;
    }
    const double hjj = GM_H(c, j, j), hj1 = GM_H(c, j + 1, j);
    const double nu = sqrt(hjj * hjj + hj1 * hj1);
    if (nu > 0.0) {
        c->cs[j] = hjj / nu;
        c->sn[j] = -hj1 / nu;
        GM_H(c, j, j) = c->cs[j] * hjj - c->sn[j] * hj1;
        GM_H(c, j + 1, j) = 0.0;
        const double gk = c->cs[j] * c->g[j] - c->sn[j] * c->g[j + 1];
        const double gkp = c->sn[j] * c->g[j] + c->cs[j] * c->g[j + 1];
        c->g[j] = gk;
        c->g[j + 1] = gkp;
    }
    const double rho = fabs(c->g[j + 1]);
    st.rho = rho;
    st.kit = j + 1;
    st.total += 1;
    if (!(rho == rho)) { st.nan = 1; st.active = 0; st.outer_done = 1; return; }
    if (c->mode == GM_MODE_REF) {
        st.sumav = rho / st.sumnor;
        st.active = (st.sumav > c->errtol && st.kit < c->kmax) ? 1 : 0;
    } else {
        const double red = rho / c->inner_ref;
        st.active = (red > c->cycle_tol && st.kit < c->kmax) ? 1 : 0;
    }
}

// back substitution y = R^{-1} g (dnssetbl.f90:657-665); coef_i = y_i sigma_i
__global__ void k_fin_cycle(GmCtrl *c, int gated)
{
    if (threadIdx.x != 0) return;
    GmStatus &st = c->st;
    if (gated && st.active) return;
    const int kit = st.kit;
    st.active = 0;
    if (kit > 0) {
        c->y[kit - 1] = c->g[kit - 1] / GM_H(c, kit - 1, kit - 1);
        for (int i = kit - 2; i >= 0; i--) {
            double yi = c->g[i];
            for (int k = i + 1; k < kit; k++) yi = yi - GM_H(c, i, k) * c->y[k];
            c->y[i] = yi / GM_H(c, i, i);
        }
        for (int i = 0; i < kit; i++) c->coef[i] = c->y[i] * c->sigma[i];
    }
    if (c->mode == GM_MODE_REF) {
        if (!(st.sumav > c->errtol)) { st.outer_done = 1; st.conv = 1; }
    }
    if (st.cycle >= c->mmax) st.outer_done = 1;
}

// PCorr += sum_i coef_i V_i (double accumulation), dnssetbl.f90:667-669
template <class T>
__global__ __launch_bounds__(VB) void k_xupd(const T *__restrict__ V, long ldv, long N,
                                            const GmCtrl *__restrict__ c, double *__restrict__ PC)
{
    __shared__ double co[TBL_KMAX_LIMIT + 1];
    const int kit = c->st.kit;
    if (kit <= 0) return;
    for (int q = threadIdx.x; q < kit; q += VB) co[q] = c->coef[q];
    __syncthreads();
    long b0, b1;
    chunk_of(N, b0, b1);
    // four elements per pass (four loads of each vector in flight per
    // thread); each element's sum runs in ascending i as before
    long e = b0 + threadIdx.x;
    for (; e + 3 * VB < b1; e += 4 * VB) {
        double p[4];
#pragma unroll
        for (int u = 0; u < 4; u++) p[u] = PC[e + u * VB];
        for (int i = 0; i < kit; i++) {
            const T *Vi = V + (long)i * ldv + e;
            T vi[4];
#pragma unroll
            for (int u = 0; u < 4; u++) vi[u] = Vi[u * VB];
#pragma unroll
            for (int u = 0; u < 4; u++) p[u] = p[u] + (double)vi[u] * co[i];
        }
#pragma unroll
        for (int u = 0; u < 4; u++) PC[e + u * VB] = p[u];
    }
    for (; e < b1; e += VB) {
        double p = PC[e];
        for (int i = 0; i < kit; i++) p = p + (double)V[(long)i * ldv + e] * co[i];
        PC[e] = p;
    }
}

// ---------------------------------------------------------------- launchers
template <class T>
void launch_norm2(const T *x, long N, double *part, const int *active, hipStream_t s)
{
    hipLaunchKernelGGL(k_norm2<T>, dim3(vec_blocks(N, sizeof(T) == 4)), dim3(VB), 0, s, x, N, part, active);
}
void launch_fin_start(GmCtrl *c, const double *part_r, int nb_r, const double *part_z, int nb_z, int first, hipStream_t s,
                      const double *part_b)
{
    hipLaunchKernelGGL(k_fin_start, dim3(1), dim3(FB), 0, s, c, part_r, nb_r, part_z, nb_z, first, part_b);
}
void launch_fin_unit(GmCtrl *c, const double *part_r, int nb_r, const double *part_z, int nb_z, const Pub &pub, hipStream_t s)
{
    hipLaunchKernelGGL(k_fin_unit, dim3(1), dim3(FB), 0, s, c, part_r, nb_r, part_z, nb_z, pub);
}
void launch_gm_init(const Geo &g, GmCtrl *c, double errtol, double inner_tol, int kmax, int mmax, int mode, double *PC,
                    double *PC2, hipStream_t s)
{
    const long faces = 2 * ((long)g.nX * g.nY + (long)g.nX * g.nZ + (long)g.nY * g.nZ);
    hipLaunchKernelGGL(k_gm_init, dim3((unsigned)((faces + VB - 1) / VB + 1)), dim3(VB), 0, s, g, c, errtol, inner_tol, kmax,
                       mmax, mode, PC, PC2);
}
template <class T>
void launch_dots(const T *V, long ldv, int j, long N, const GmCtrl *c, double *part, hipStream_t s)
{
    hipLaunchKernelGGL(k_dots<T>, dim3(vec_blocks(N, sizeof(T) == 4)), dim3(VB), 0, s, V, ldv, j, N, c, part);
}
void launch_fin_dots(GmCtrl *c, const double *part, int nb, int j, hipStream_t s)
{
    hipLaunchKernelGGL(k_fin_dots, dim3(j + 1), dim3(VB), 0, s, c, part, nb, j);
}
template <class T>
void launch_update(const T *V, long ldv, int j, long N, GmCtrl *c, double *part, hipStream_t s, bool store)
{
    if (!store) {
        hipLaunchKernelGGL((k_update<T, false>), dim3(vec_blocks(N, sizeof(T) == 4)), dim3(VB), 0, s, V, ldv, j, N, c, part);
        return;
    }
    hipLaunchKernelGGL((k_update<T, true>), dim3(vec_blocks(N, sizeof(T) == 4)), dim3(VB), 0, s, V, ldv, j, N, c, part);
}
void launch_fin_update(GmCtrl *c, const double *part, int nb, int j, hipStream_t s)
{
    hipLaunchKernelGGL(k_fin_update, dim3(1), dim3(VB), 0, s, c, part, nb, j);
}
void launch_fin_cycle(GmCtrl *c, hipStream_t s, int gated)
{
    hipLaunchKernelGGL(k_fin_cycle, dim3(1), dim3(64), 0, s, c, gated);
}
template <class T>
void launch_xupd(const T *V, long ldv, long N, const GmCtrl *c, double *PC, hipStream_t s)
{
    hipLaunchKernelGGL(k_xupd<T>, dim3(vec_blocks(N, sizeof(T) == 4)), dim3(VB), 0, s, V, ldv, N, c, PC);
}
#define TBL_INST(T)                                                                                 \
    template void launch_norm2<T>(const T *, long, double *, const int *, hipStream_t);             \
    template void launch_dots<T>(const T *, long, int, long, const GmCtrl *, double *, hipStream_t); \
    template void launch_update<T>(const T *, long, int, long, GmCtrl *, double *, hipStream_t, bool); \
    template void launch_xupd<T>(const T *, long, long, const GmCtrl *, double *, hipStream_t);
TBL_INST(double)
TBL_INST(float)
#undef TBL_INST

// pc <- 2 pc - prev, prev <- old pc (linear extrapolation of the pressure
// correction in time, the initial guess of the next solve)
__global__ __launch_bounds__(256) void k_pc_extrap(double *__restrict__ pc, double *__restrict__ prev, long N)
{
    for (long e = (long)blockIdx.x * 256 + threadIdx.x; e < N; e += (long)gridDim.x * 256) {
        const double t = pc[e];
        pc[e] = 2.0 * t - prev[e];
        prev[e] = t;
    }
}
void launch_pc_extrap(double *pc, double *prev, long N, hipStream_t s)
{
    long nb = (N + 255) / 256;
    if (nb > 8192) nb = 8192;
    hipLaunchKernelGGL(k_pc_extrap, dim3((unsigned)nb), dim3(256), 0, s, pc, prev, N);
}

}  // namespace tbl
