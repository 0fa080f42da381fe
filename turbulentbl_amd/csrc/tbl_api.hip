// tbl_api.hip -- the extern "C" entry points of libtbl_hip.so (see include/tbl.h).
//
// One context = one device, one HIP stream, all fields resident in HBM in the
// reference's layout (Fortran order, i fastest).  FP64 mode stores every
// field in double; mixed mode stores velocity, pressure, Q and the Krylov
// basis in float and keeps PCorr, pRhs, the outer residual, the Gram-Schmidt
// coefficients, Hessenberg/Givens, divergence, statistics and the recycling
// rescale in double.
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdio.h>
#include <string.h>

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <exception>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <thread>
#include <utility>
#include <vector>

#include "../../include/tbl.h"
#include "tbl_dev.h"
#include "tbl_launch.h"

using namespace tbl;

struct TimerRec { hipEvent_t a, b; int cls; double bytes; int n; };   // n launches between a and b

struct tbl_ctx {
    tbl_params p;
    Geo g;
    hipStream_t s = nullptr;
    int dev = 0;
    bool mixed = false;
    size_t es = 8;                       // bytes per stored field element
    // host mesh (a1)
    std::vector<double> x1, x2, x3, Xi, Jac, Jac2, JacInv, Ab, At, Ap, rAp;
    double mass_denom = 1.0;
    // device buffers
    double *mesh = nullptr;
    void *Ut = nullptr, *Utold = nullptr, *Q = nullptr, *Press = nullptr;
    void *Ualt = nullptr;                // second velocity buffer of the zebra sweep (Ut and Ualt swap)
    int *slab = nullptr;                 // per-slab orderings: 0-based first/last interior plane per slab
    double *PCorr = nullptr, *pRhs = nullptr;
    double *PCprev = nullptr;            // PCorr of the step before (extrapolated initial guess)
    double *PCalt = nullptr;             // second PCorr buffer: the fused update + residual writes it
    int pc_hist = 0;                     // previous solutions available for the extrapolation
    void *V = nullptr, *W = nullptr, *scr = nullptr, *r = nullptr;
    void *r3 = nullptr;                  // three-component residual of the direct and transposed solves (zero faces)
    void *Z = nullptr;                   // flexible-GMRES preconditioned vectors (true-residual mode)
    long ldv = 0;
    double *part = nullptr;
    size_t npart = 0;
    size_t bytes = 0;                    // device memory held, without the fast solver's own
    GmCtrl *gm = nullptr;
    // pinned host block that kernels publish their results to (see Pub), and
    // its parts: GMRES status, Gauss-Seidel control, diagnostics record
    struct HostPub *hp = nullptr;
    unsigned pseq = 0;                   // sequence number of the last result asked for
    GmStatus *gm_h = nullptr;
    void *gs = nullptr, *gs_h = nullptr; // Gauss-Seidel control (device / published)
    double *sums = nullptr, *avg = nullptr, *Wt = nullptr, *Ume = nullptr, *uf = nullptr;
    double *bltkns = nullptr, *dstar = nullptr, *theta = nullptr, *wall_w = nullptr, *tau = nullptr;
    double *tausum = nullptr, *taumean = nullptr, *cf = nullptr;   // wall-shear window (a17)
    int nwin = 0;                        // wall-shear windows completed
    double *scan = nullptr;
    FastPC *fast = nullptr;
    void *zf = nullptr;                  // z-line Gauss-Seidel elimination factors (storage type)
    int *newk = nullptr;
    RecDev *rec = nullptr;
    int *guard = nullptr;                // in the diagnostics record
    double *dd = nullptr;                // device diagnostics record
    double *noalloc = nullptr;           // this device's copy of `scratch` (tbl_div_check_noalloc)
    double *dh = nullptr;                // published copy
    struct XferRing *ring = nullptr;     // pinned chunks of the host transfers
    bool have_wall_w = false;
    // Peclet-switch patterns of an adjoint window (record / replay): one byte
    // per cell and step, window of br_steps steps starting after step br_nstep0
    unsigned char *br = nullptr;
    int br_steps = 0, br_nstep0 = -1;
    const unsigned char *br_in = nullptr;   // momentum RHS: replay this pattern
    unsigned char *br_out = nullptr;        // momentum RHS: record into this
    // clock
    double time = 0.0;
    int nstep = 0, cnt = 0;
    bool uploaded = false;
    // timers
    unsigned tmask = 0;
    std::vector<TimerRec> pend;
    std::vector<hipEvent_t> pool;
    int tcount[TBL_K_NCLASS] = {0};
    double tms[TBL_K_NCLASS] = {0};
    double tbytes[TBL_K_NCLASS] = {0};
    std::string err;
};

struct HostPub {
    unsigned seq, pad;
    GmStatus gm;
    double gs[16], dd[DD_NCOUNT];
};

// (a failed call's error is cleared: it would be taken for that of the next launch)
#define HIPCHK(ctx, call)                                                                    \
    do {                                                                                     \
        hipError_t e_ = (call);                                                              \
        if (e_ != hipSuccess) {                                                              \
            (ctx)->err = std::string(#call) + ": " + hipGetErrorString(e_);                  \
            (void)hipGetLastError();                                                         \
            return (int)e_;                                                                  \
        }                                                                                    \
    } while (0)
#define CHK(expr)                \
    do {                         \
        int rc_ = (expr);        \
        if (rc_ != 0) return rc_;\
    } while (0)

static int fail(tbl_ctx *c, int code, const char *msg)
{
    if (c) c->err = msg;
    return code;
}

// ------------------------------------------------------------------ timers
static void timer_flush(tbl_ctx *c)
{
    if (c->pend.empty()) return;
    hipStreamSynchronize(c->s);
    for (auto &t : c->pend) {
        float ms = 0.f;
        hipEventElapsedTime(&ms, t.a, t.b);
        c->tcount[t.cls] += t.n;
        c->tms[t.cls] += ms;
        c->tbytes[t.cls] += t.bytes;
        c->pool.push_back(t.a);
        c->pool.push_back(t.b);
    }
    c->pend.clear();
}
static hipEvent_t ev_get(tbl_ctx *c)
{
    if (c->pool.empty()) {
        hipEvent_t e;
        hipEventCreate(&e);
        return e;
    }
    hipEvent_t e = c->pool.back();
    c->pool.pop_back();
    return e;
}
// Times the launches in its scope when the class is enabled; `bytes` is the
// algorithmic (compulsory) HBM traffic of those launches: each distinct array
// element read once and written once at its storage precision.
struct Tscope {
    tbl_ctx *c;
    int cls;
    double bytes;
    int n;                                 // launches in the scope (back to back, one pair of events)
    hipEvent_t a = nullptr;
    Tscope(tbl_ctx *c_, int cls_, double bytes_ = 0.0, int n_ = 1) : c(c_), cls(cls_), bytes(bytes_), n(n_)
    {
        if (c->tmask & (1u << cls)) {
            a = ev_get(c);
            hipEventRecord(a, c->s);
        }
    }
    ~Tscope()
    {
        if (a) {
            hipEvent_t b = ev_get(c);
            hipEventRecord(b, c->s);
            c->pend.push_back({a, b, cls, bytes, n});
            if (c->pend.size() > 4096) timer_flush(c);
        }
    }
};

// ------------------------------------------------------------------ a1: mesh
// dnssetbl.f90:183-247, same arithmetic as the reference (REAL(4) literals kept)
static void build_mesh(tbl_ctx *c)
{
    const tbl_params &p = c->p;
    const int nX = p.nX, nY = p.nY, nZ = p.nZ;
    c->x1.assign(nX, 0.0); c->x2.assign(nY, 0.0); c->x3.assign(nZ, 0.0); c->Xi.assign(nZ, 0.0);
    c->Jac.assign(nZ, 0.0); c->Jac2.assign(nZ, 0.0); c->JacInv.assign(nZ, 0.0);
    c->Ab.assign(nZ, 0.0); c->At.assign(nZ, 0.0); c->Ap.assign(nZ, 0.0); c->rAp.assign(nZ, 0.0);
    const double dx = p.Lx / (double)(nX - 1), dy = p.Ly / (double)(nY - 1), dXi = p.Lz / (double)(nZ - 1);
    for (int i = 0; i < nX - 1; i++) c->x1[i + 1] = c->x1[i] + dx;
    for (int i = 0; i < nY - 1; i++) c->x2[i + 1] = c->x2[i] + dy;
    for (int k = 0; k < nZ - 1; k++) c->Xi[k + 1] = c->Xi[k] + dXi;
    const double delta = p.delta, Lzd = p.Lz, Lhd = p.Lz * 0.5;
    const double Lzf = (double)(float)p.Lz, Lhf = (double)(float)(p.Lz * 0.5);
    for (int k = 0; k < nZ; k++) {
        const double a = delta * 0.5 * (c->Xi[k] - Lzf);
        const double ch = cosh(0.5 * delta * (c->Xi[k] - Lzf));
        c->x3[k] = Lzd + Lzd * tanh(a) / (tanh(Lhd * delta));
        c->Jac[k] = Lhd * delta / (tanh(Lhf * delta) * (ch * ch));
        c->Jac2[k] = -(Lhd * (delta * delta) * tanh(0.5 * delta * (c->Xi[k] - Lzf)) / (tanh(Lhf * delta) * (ch * ch)));
    }
    for (int k = 0; k < nZ; k++) {
        const double J = c->Jac[k];
        c->Ab[k] = 1.0 / (dXi * dXi * J * J) + c->Jac2[k] / (2.0 * dXi * J * J * J);
        c->At[k] = 1.0 / (dXi * dXi * J * J) - c->Jac2[k] / (2.0 * dXi * J * J * J);
        c->Ap[k] = -2.0 * ((1.0 / (dx * dx)) + (1.0 / (dy * dy)) + (1.0 / (dXi * dXi * J * J)));
        c->rAp[k] = 1.0 / c->Ap[k];
        c->JacInv[k] = 1.0 / J;
    }
    Geo &g = c->g;
    g.nX = nX; g.nY = nY; g.nZ = nZ;
    g.sZ = (long)nX * nY;
    g.N = (long)nX * nY * nZ;
    g.dx = dx; g.dy = dy; g.dXi = dXi;
    g.invdx = 1.0 / dx; g.invdy = 1.0 / dy; g.invdXi = 1.0 / dXi;
    g.c12 = 1.0 / 12.0;
    g.Aw = 1.0 / (dx * dx); g.Ae = 1.0 / (dx * dx); g.An = 1.0 / (dy * dy); g.As = 1.0 / (dy * dy);
    g.df1 = c->x3[1] - c->x3[0];
    g.df2 = c->x3[2] - c->x3[0];
    g.dt = p.dt; g.Re = p.Re; g.Ue = p.Ue; g.omega = p.omega;
    g.scheme = p.scheme;
    for (int q = 0; q < 3; q++) g.forc[q] = p.forc[q];
    c->mass_denom = (c->x3[nZ - 2] - c->x3[1]) * (c->x2[nY - 2] - c->x2[1]);
}

extern "C" void tbl_default_params(tbl_params *p)
{
    memset(p, 0, sizeof(*p));
    p->nX = 90; p->nY = 80; p->nZ = 50;
    p->Lx = 12.0; p->Ly = 4.0; p->Lz = 3.4; p->delta = 1.95;
    p->dt = 1.0e-4; p->Re = 150.92; p->Ue = 19.798;
    p->omega = (double)1.835f;
    p->i_rec = 68; p->freq_tim_avg = 500;
    const int pl[5] = {5, 20, 40, 60, 85};
    for (int q = 0; q < 5; q++) p->planes[q] = pl[q];
    p->precision = TBL_FP64;
    p->errorstop = 1.0e-6; p->gs_mmax = 1000;
    p->tol_mode = TBL_TOL_REF; p->errtol = 1.0e-5; p->kmax = 50; p->mmax = 1000;
    p->precond = TBL_PC_FAST; p->inner_tol = 1.0e-3;
    p->helm_mode = TBL_HELM_ZEBRA;
    p->fail_on_noconv = 0; p->wall_shear_window = 0; p->pc_extrap = 0;
    p->scheme = TBL_SCHEME_SETBL;
    p->forc[0] = p->forc[1] = p->forc[2] = 0.0;
    p->slabs = 1;
}

static int h2d(tbl_ctx *c, void *d, const void *h, size_t b);

// device memory of the context, cleared; its sum is what tbl_device_bytes reports
template <class X> static hipError_t alloc_clear(tbl_ctx *c, X **ptr, size_t bytes)
{
    if (bytes == 0) bytes = 8;
    hipError_t e = hipMalloc((void **)ptr, bytes);
    if (e != hipSuccess) { *ptr = nullptr; return e; }
    c->bytes += bytes;
    return hipMemsetAsync(*ptr, 0, bytes, c->s);
}
template <class X> static int dalloc(tbl_ctx *c, X **ptr, size_t bytes)
{
    HIPCHK(c, alloc_clear(c, ptr, bytes));
    return 0;
}
// for memory that a slower route does without: 1 (and *ptr null) if there is none
template <class X> static int try_alloc(tbl_ctx *c, X **ptr, size_t bytes)
{
    if (alloc_clear(c, ptr, bytes) == hipSuccess) return 0;
    (void)hipGetLastError();                   // the next launch is not what failed
    return 1;
}

// ------------------------------------------------------------------ static scratch
// Scratch of tbl_div_check_noalloc: the block partials of the divergence sum,
// in a file-scope device array so that the call allocates nothing.  Every
// device holds its own copy until the process ends; host code uses the
// device address hipGetSymbolAddress returns for it (never the array's name,
// which on the host is a stand-in and not a device address).
#define TBL_NOALLOC_PARTS 32768
#define TBL_MAX_DEVICES 64
static __device__ __align__(256) double scratch[TBL_NOALLOC_PARTS];
static std::mutex scratch_mu;
static double *scratch_dev[TBL_MAX_DEVICES];

// once per device, with that device current (called from tbl_create)
static int scratch_setup(tbl_ctx *c)
{
    if (c->dev < 0 || c->dev >= TBL_MAX_DEVICES) return fail(c, TBL_EARG, "device index above 63");
    std::lock_guard<std::mutex> lk(scratch_mu);
    if (!scratch_dev[c->dev]) {
        void *ptr = nullptr;
        HIPCHK(c, hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        scratch_dev[c->dev] = (double *)ptr;
    }
    c->noalloc = scratch_dev[c->dev];
    return 0;
}

static int create_impl(tbl_ctx *c)
{
    const tbl_params &p = c->p;
    const long N = (long)p.nX * p.nY * p.nZ;
    HIPCHK(c, hipGetDevice(&c->dev));
    HIPCHK(c, hipStreamCreateWithFlags(&c->s, hipStreamNonBlocking));
    CHK(scratch_setup(c));
    build_mesh(c);
    const int nZ = p.nZ;
    CHK(dalloc(c, &c->mesh, sizeof(double) * 7 * nZ));
    std::vector<double> m;
    for (auto *v : {&c->x3, &c->Jac2, &c->JacInv, &c->Ab, &c->At, &c->Ap, &c->rAp}) m.insert(m.end(), v->begin(), v->end());
    HIPCHK(c, hipMemcpyAsync(c->mesh, m.data(), sizeof(double) * m.size(), hipMemcpyHostToDevice, c->s));
    c->g.x3 = c->mesh; c->g.Jac2 = c->mesh + nZ; c->g.JacInv = c->mesh + 2 * nZ; c->g.Ab = c->mesh + 3 * nZ;
    c->g.At = c->mesh + 4 * nZ; c->g.Ap = c->mesh + 5 * nZ; c->g.rAp = c->mesh + 6 * nZ;

    c->es = c->mixed ? sizeof(float) : sizeof(double);
    CHK(dalloc(c, &c->Ut, 3 * N * c->es));
    CHK(dalloc(c, &c->Utold, 3 * N * c->es));
    CHK(dalloc(c, &c->Q, 3 * N * c->es));
    CHK(dalloc(c, &c->Press, N * c->es));
    CHK(dalloc(c, &c->PCorr, N * sizeof(double)));
    CHK(dalloc(c, &c->pRhs, N * sizeof(double)));
    c->ldv = (N + 63) & ~63L;
    CHK(dalloc(c, &c->V, (size_t)(p.kmax + 1) * c->ldv * c->es));
    CHK(dalloc(c, &c->W, N * c->es));
    CHK(dalloc(c, &c->r, N * c->es));
    if (p.tol_mode == TBL_TOL_TRUE) CHK(dalloc(c, &c->Z, (size_t)p.kmax * c->ldv * c->es));
    if (p.helm_mode == TBL_HELM_ZEBRA) CHK(dalloc(c, &c->Ualt, 3 * N * c->es));
    c->g.nslab = 0; c->g.nkmax = 0; c->g.skew = 0; c->g.slab = nullptr;
    c->g.rblk = c->mixed ? 8192 : 2048;
    c->g.rpl = c->mixed ? p.nZ : 12;
    size_t nscr = N, ncopy = 0;                // of scr; with the slab sweeps' copy in it
    if (p.helm_mode == TBL_HELM_LEX_SLAB || p.precond == TBL_PC_SSOR_BLOCK) {
        // the reference's slab bounds (dnssetbl.f90:76-92): nZ/P planes per
        // rank, the remainder to the high ranks; the first and last rank
        // exclude the wall and top boundary planes
        const int P = p.slabs, nZ = p.nZ;
        std::vector<int> b(P + 1), e(P), sl(2 * P);
        int it1 = nZ / P;
        const int it2 = P - nZ % P;
        b[0] = 1;
        for (int r = 0; r < P; r++) {
            if (r == it2) it1 = it1 + 1;
            e[r] = b[r] + it1 - 1;
            b[r + 1] = e[r] + 1;
        }
        int nkmax = 0;
        for (int r = 0; r < P; r++) {
            const int bn = (r == 0) ? b[r] + 1 : b[r], en = (r == P - 1) ? e[r] - 1 : e[r];
            if (en < bn) return fail(c, TBL_EARG, "slabs: every slab needs at least one interior plane");
            sl[2 * r] = bn - 1;
            sl[2 * r + 1] = en - 1;
            nkmax = std::max(nkmax, en - bn + 1);
        }
        c->g.nslab = P;
        c->g.nkmax = nkmax;
        if (!slab_threads(c->g, nkmax))
            return fail(c, TBL_EARG, "slabs: a slab needs more than 512 threads (ceil((nY-2)/64)*64 * "
                                     "ceil(planes/32)); use more slabs");
        CHK(dalloc(c, &c->slab, sizeof(int) * 2 * P));
        HIPCHK(c, hipMemcpyAsync(c->slab, sl.data(), sizeof(int) * 2 * P, hipMemcpyHostToDevice, c->s));
        c->g.slab = c->slab;
        const bool lex = p.helm_mode == TBL_HELM_LEX_SLAB;
        if (slab_copy_pays(c->g)) ncopy = std::max(nscr, slab_scratch(c->g, lex));
        nscr = std::max(nscr, slab_scratch_inplace(c->g, lex));
    }
    if (p.helm_mode == TBL_HELM_ZLINE_RB || p.helm_mode == TBL_HELM_ZEBRA) {
        // elimination factors of the partitioned wall-normal line solve (the
        // line matrix a = -h Ab, b = 1 - h Ap, c = -h At is the same for every
        // column): interior planes k = 1..nZ-2 in C balanced chunks of at most
        // LC planes; per k the forward multiplier a and reciprocal pivot R,
        // the forward c', and the back-substituted a'', c''; per chunk the
        // F-row rhs coupling c0; per first/last unknown the reduced-system
        // Thomas factors.  Computed in double, stored in the storage type.
        const int nZ = p.nZ, nz = nZ - 2;
        if (nz < 2 || nz > 512) return fail(c, TBL_EARG, "z-line Gauss-Seidel needs 4 <= nZ <= 514");
        const int LC = nz <= 256 ? 16 : 32, C = (nz + LC - 1) / LC;
        const double h = p.dt / p.Re;
        std::vector<double> zd(5 * (size_t)nZ + 7 * (size_t)C, 0.0);
        double *za = zd.data(), *zR = za + nZ, *zC = za + 2 * nZ, *zA2 = za + 3 * nZ, *zC2 = za + 4 * nZ;
        double *zc0 = za + 5 * nZ, *rA = zc0 + C, *rg = rA + 2 * C, *re = rg + 2 * C;
        std::vector<double> ap(nZ, 0.0), cp(nZ, 0.0), B(2 * C), Cc(2 * C);
        for (int ch = 0; ch < C; ch++) {
            const int kb = 1 + (int)(((long)ch * nz) / C), ke = 1 + (int)(((long)(ch + 1) * nz) / C) - 1;
            const int M = ke - kb + 1;
            const double a0 = (kb == 1) ? 0.0 : -(h * c->Ab[kb]);
            const double b0 = 1.0 - h * c->Ap[kb];
            const double c0 = (kb == nZ - 2) ? 0.0 : -(h * c->At[kb]);
            for (int k = kb + 1; k <= ke; k++) {
                const double a = -(h * c->Ab[k]), b = 1.0 - h * c->Ap[k];
                const double cc = (k == nZ - 2) ? 0.0 : -(h * c->At[k]);
                if (k == kb + 1) {
                    const double R = 1.0 / b;
                    ap[k] = a * R; cp[k] = cc * R;
                    za[k] = 0.0; zR[k] = R;
                } else {
                    const double R = 1.0 / (b - a * cp[k - 1]);
                    ap[k] = -(a * ap[k - 1]) * R; cp[k] = cc * R;
                    za[k] = a; zR[k] = R;
                }
                zC[k] = cp[k];
            }
            if (M >= 3) {
                zA2[ke - 1] = ap[ke - 1];
                zC2[ke - 1] = cp[ke - 1];
                for (int k = ke - 2; k >= kb + 1; k--) {
                    zA2[k] = ap[k] - cp[k] * zA2[k + 1];
                    zC2[k] = -(cp[k] * zC2[k + 1]);
                }
            }
            rA[2 * ch] = a0;
            if (M >= 3) {
                B[2 * ch] = b0 - c0 * zA2[kb + 1];
                Cc[2 * ch] = -(c0 * zC2[kb + 1]);
                zc0[ch] = c0;
            } else {
                B[2 * ch] = b0;
                Cc[2 * ch] = c0;
                zc0[ch] = 0.0;
            }
            rA[2 * ch + 1] = ap[ke];
            B[2 * ch + 1] = 1.0;
            Cc[2 * ch + 1] = cp[ke];
        }
        rg[0] = 1.0 / B[0];
        re[0] = Cc[0] * rg[0];
        for (int s2 = 1; s2 < 2 * C; s2++) {
            rg[s2] = 1.0 / (B[s2] - rA[s2] * re[s2 - 1]);
            re[s2] = Cc[s2] * rg[s2];
        }
        CHK(dalloc(c, &c->zf, zd.size() * c->es));
        if (c->mixed) {
            std::vector<float> zs(zd.begin(), zd.end());
            CHK(h2d(c, c->zf, zs.data(), zs.size() * sizeof(float)));
        } else {
            CHK(h2d(c, c->zf, zd.data(), zd.size() * sizeof(double)));
        }
        HIPCHK(c, hipStreamSynchronize(c->s));
    }
    if (p.precond == TBL_PC_FAST || p.helm_mode == TBL_HELM_DIRECT) {
        char msg[256];
        HIPCHK(c, hipStreamSynchronize(c->s));
        if (fastpc_create(c->g, c->Ab.data(), c->At.data(), c->Ap.data(), c->s, c->mixed, &c->fast, msg, sizeof(msg)))
            return fail(c, TBL_EARG, msg);
    }
    // partials: [0, 6*nbr+8) for tile reductions (Gauss-Seidel uses 6 per tile);
    // GMRES puts the residual partials at 0 and the vector partials at nbr+8,
    // (kmax+1) groups of vec_blocks(N) each
    const size_t nbr = resid_blocks(c->g), nbv = vec_blocks(N, c->mixed);
    c->npart = 6 * nbr + 8 + (size_t)(p.kmax + 2) * (nbv + 8);
    c->npart = std::max(c->npart, nbr + 8 + (size_t)poisson_blocks(c->g, c->mixed));   // fused first dot fits
    c->npart = std::max(c->npart, 6 * (size_t)rhs_blocks(c->g, c->mixed));             // fused first residual pass fits
    CHK(dalloc(c, &c->part, c->npart * sizeof(double)));
    CHK(dalloc(c, &c->gm, sizeof(GmCtrl)));
    // fine-grained (coherent), so that a running kernel's stores reach the host
    HIPCHK(c, hipHostMalloc((void **)&c->hp, sizeof(HostPub), hipHostMallocCoherent));
    memset(c->hp, 0, sizeof(HostPub));
    if (gs_ctrl_bytes() > sizeof(c->hp->gs)) return fail(c, TBL_EARG, "Gauss-Seidel control block above its host copy");
    c->gm_h = &c->hp->gm;
    c->gs_h = c->hp->gs;
    c->dh = c->hp->dd;
    CHK(dalloc(c, &c->gs, gs_ctrl_bytes()));
    const long M = (long)p.nX * p.nZ;
    CHK(dalloc(c, &c->sums, 9 * M * sizeof(double)));
    CHK(dalloc(c, &c->avg, 9 * M * sizeof(double)));
    CHK(dalloc(c, &c->Wt, M * sizeof(double)));
    CHK(dalloc(c, &c->Ume, p.nZ * sizeof(double)));
    CHK(dalloc(c, &c->uf, 3L * p.nY * p.nZ * sizeof(double)));
    CHK(dalloc(c, &c->bltkns, p.nX * sizeof(double)));
    CHK(dalloc(c, &c->dstar, p.nX * sizeof(double)));
    CHK(dalloc(c, &c->theta, p.nX * sizeof(double)));
    CHK(dalloc(c, &c->tau, p.nX * sizeof(double)));
    CHK(dalloc(c, &c->tausum, p.nX * sizeof(double)));
    CHK(dalloc(c, &c->taumean, p.nX * sizeof(double)));
    CHK(dalloc(c, &c->cf, p.nX * sizeof(double)));
    CHK(dalloc(c, &c->wall_w, (size_t)p.nX * p.nY * sizeof(double)));
    CHK(dalloc(c, &c->scan, 2 * (p.nZ + 2) * sizeof(double)));
    CHK(dalloc(c, &c->newk, p.nZ * sizeof(int)));
    CHK(dalloc(c, &c->rec, sizeof(RecDev)));
    CHK(dalloc(c, &c->dd, (DD_J + 1) * sizeof(double)));
    c->guard = (int *)(c->dd + DD_GUARD);
    RecDev r0 = {1.0, 1.0, 0};
    HIPCHK(c, hipMemcpyAsync(c->rec, &r0, sizeof(r0), hipMemcpyHostToDevice, c->s));
    std::vector<int> nk(p.nZ);
    for (int k = 0; k < p.nZ; k++) nk[k] = (k < p.nZ - 1) ? k + 1 : p.nZ - 1;
    HIPCHK(c, hipMemcpyAsync(c->newk, nk.data(), sizeof(int) * p.nZ, hipMemcpyHostToDevice, c->s));
    // last, so that the copy takes nothing that the context cannot do without
    c->g.skew = ncopy && !try_alloc(c, &c->scr, ncopy * c->es);
    if (!c->scr) CHK(dalloc(c, &c->scr, nscr * c->es));
    HIPCHK(c, hipStreamSynchronize(c->s));
    return 0;
}

// message of the last tbl_create that failed on this thread: no context
// exists then, so tbl_last_error(NULL, ...) returns it
static thread_local std::string create_err;

// the parameter checks of tbl_create; nullptr if p is valid
static const char *params_error(const tbl_params *p)
{
    if (p->nX < 8 || p->nY < 8 || p->nZ < 8) return "nX, nY and nZ must each be at least 8";
    if (p->nY & 1) return "nY must be even (the periodic span's nY-2 rows are coloured red-black)";
    if ((double)p->nX * p->nY * p->nZ * 3.0 > 2.0e9) return "nX*nY*nZ*3 must not exceed 2e9 (32-bit in-field offsets)";
    if (!(p->dt > 0.0) || !(p->Re > 0.0)) return "dt and Re must be positive";
    if (p->kmax < 1 || p->kmax > TBL_KMAX_LIMIT) return "kmax must be in 1..64";
    if (p->i_rec < 2 || p->i_rec > p->nX - 1) return "i_rec must be in 2..nX-1";
    if (p->freq_tim_avg < 1) return "freq_tim_avg must be at least 1";
    if (p->wall_shear_window < 0) return "wall_shear_window must be 0 (off) or positive";
    for (int q = 0; q < 5; q++)
        if (p->planes[q] < 1 || p->planes[q] > p->nX) return "mass-flux planes must be in 1..nX";
    if (p->precision != TBL_FP64 && p->precision != TBL_MIXED) return "unknown precision";
    if (p->precond != TBL_PC_SSOR_RB && p->precond != TBL_PC_NONE && p->precond != TBL_PC_JACOBI &&
        p->precond != TBL_PC_FAST && p->precond != TBL_PC_SSOR_BLOCK)
        return "unknown preconditioner";
    if (p->helm_mode != TBL_HELM_POINT_RB && p->helm_mode != TBL_HELM_ZLINE_RB && p->helm_mode != TBL_HELM_DIRECT &&
        p->helm_mode != TBL_HELM_ZEBRA && p->helm_mode != TBL_HELM_LEX_SLAB)
        return "unknown helm_mode";
    if (p->slabs < 1 || p->slabs > 256) return "slabs must be in 1..256";
    if (p->tol_mode != TBL_TOL_REF && p->tol_mode != TBL_TOL_TRUE) return "unknown tol_mode";
    if (p->scheme != TBL_SCHEME_SETBL && p->scheme != TBL_SCHEME_DNSTBL) return "unknown convection scheme";
    return nullptr;
}

extern "C" int tbl_create(const tbl_params *p, tbl_ctx **out)
{
    if (!p || !out) {
        create_err = "tbl_create: NULL params or output pointer";
        return TBL_EARG;
    }
    *out = nullptr;
    if (const char *e = params_error(p)) {
        create_err = std::string("tbl_create: ") + e;
        return TBL_EARG;
    }
    tbl_ctx *c = new tbl_ctx();
    c->p = *p;
    c->mixed = (p->precision == TBL_MIXED);
    int rc = create_impl(c);
    if (rc) {
        create_err = "tbl_create: " + c->err;
        tbl_destroy(c);
        return rc;
    }
    create_err.clear();
    *out = c;
    return 0;
}

static void ring_free(tbl_ctx *c);
extern "C" int tbl_destroy(tbl_ctx *c)
{
    if (!c) return 0;
    if (c->s) hipStreamSynchronize(c->s);
    timer_flush(c);
    for (auto e : c->pool) hipEventDestroy(e);
    void *dev[] = {c->mesh, c->Ut, c->Ualt, c->Utold, c->Q, c->Press, c->PCorr, c->pRhs, c->V, c->W, c->scr, c->r, c->Z,
                   c->part, c->gm, c->gs, c->sums, c->avg, c->Wt, c->Ume, c->uf, c->bltkns, c->dstar,
                   c->theta, c->tau, c->tausum, c->taumean, c->cf, c->wall_w, c->scan, c->newk, c->rec, c->dd, c->zf, c->br, c->PCprev,
                   c->PCalt, c->slab, c->r3};
    for (void *d : dev)
        if (d) hipFree(d);
    if (c->fast) fastpc_destroy(c->fast);
    if (c->hp) hipHostFree(c->hp);
    ring_free(c);
    if (c->s) hipStreamDestroy(c->s);
    delete c;
    return 0;
}

extern "C" int tbl_last_error(const tbl_ctx *c, char *buf, int len)
{
    if (!buf || len <= 0) return TBL_EARG;
    snprintf(buf, len, "%s", c ? c->err.c_str() : create_err.c_str());
    return 0;
}

extern "C" int tbl_sync(tbl_ctx *c)
{
    if (!c) return TBL_EARG;
    HIPCHK(c, hipStreamSynchronize(c->s));
    return 0;
}

extern "C" double tbl_device_bytes(const tbl_ctx *c)
{
    if (!c) return 0.0;
    return (double)(c->bytes + (c->fast ? fastpc_bytes(c->fast) : 0));
}

// ------------------------------------------------------------------ fields
static size_t field_len(const tbl_ctx *c, int f)
{
    const size_t N = (size_t)c->g.N;
    return (f == TBL_F_UT || f == TBL_F_UTOLD || f == TBL_F_Q) ? 3 * N : N;
}
static void *field_ptr(tbl_ctx *c, int f, bool *is_double)
{
    *is_double = !c->mixed;
    switch (f) {
    case TBL_F_UT: return c->Ut;
    case TBL_F_UTOLD: return c->Utold;
    case TBL_F_Q: return c->Q;
    case TBL_F_PRESS: return c->Press;
    case TBL_F_WORK: return c->r;        // work vector whose boundary entries are never read
    case TBL_F_PCORR: *is_double = true; return c->PCorr;
    case TBL_F_PRHS: *is_double = true; return c->pRhs;
    }
    return nullptr;
}

// Host transfers of fields.  Host arrays are FP64 and mostly pageable; mixed
// contexts hold FP32.  A pageable copy runs at 18 GB/s from the device (31 to
// it), and converting and filling an array of untouched pages on one thread
// cost more than that: reading the velocity and pressure of 1024x256x192
// mixed took 300 ms, 60 steps' worth.  The field goes through a ring of pinned
// chunks instead: the copy engine fills (drains) them at 57 GB/s while a few
// threads convert and copy between the chunks and the host array.  The ring
// belongs to the context (XF_SLOTS chunks, allocated by the first transfer that
// takes it).  Up / down, before -> after: 1024x256x192 mixed velocity 167 / 213 ->
// 19 / 23 ms, 512x128x128 FP64 6.9 / 19.4 -> 5.1 / 5.9 ms; 4 to 16 threads differ
// by 10 %, 2 take half as long again from the device, chunks of 64 k values twice
// as long.  Four threads, which sleep while they wait for each other: eight that
// yielded ran a process whose other threads were busy into its CPU quota (16
// cores), and an upload of 18 M values that takes 4 ms took 38.  The waits for the
// copy engine spin (a download of 25 M values takes 5.1 ms and 20 ms of CPU):
// asking and sleeping in turn halves the CPU time and changes nothing on an idle
// host, but beside 16 busy threads that download takes 14 instead of 10 ms.
//
// A plain copy (move_plain) is the sooner one, and is taken,
//  * from and to page-locked memory in FP64, which the copy engine reads and
//    writes itself: 512x128x128 velocity 3.5 ms, through the ring 5.1;
//  * below the sizes XF_*: FP64 to the device 3 M values (128x80x80 velocity 0.56
//    against 0.66 ms), from it half a million; FP32, converted by the caller's
//    thread, 1.3 M (1.1 M values 0.23 against 0.25 ms, 1.5 M 0.34 against 0.30) and
//    0.4 M (0.29 M values 0.12 against 0.15, 0.5 M 0.18 against 0.15);
//  * where there is no pinned memory for the ring.
#define XF_SLOTS 8
#define XF_CHUNK ((size_t)1 << 18)       // elements per chunk: 2 MB of doubles
#define XF_D_UP (12 * XF_CHUNK)          // least elements through the ring
#define XF_D_DOWN (2 * XF_CHUNK)
#define XF_F_UP (5 * XF_CHUNK)
#define XF_F_DOWN (3 * XF_CHUNK / 2)
#define XF_THREADS 4
#define XF_NAP std::this_thread::sleep_for(std::chrono::microseconds(10))
struct XferRing {
    char *mem = nullptr, *buf[XF_SLOTS] = {nullptr};     // buf: into mem
    hipEvent_t ev[XF_SLOTS] = {nullptr};
};
static void ring_free(tbl_ctx *c)
{
    if (!c->ring) return;
    if (c->ring->mem) hipHostFree(c->ring->mem);
    for (int q = 0; q < XF_SLOTS; q++)
        if (c->ring->ev[q]) hipEventDestroy(c->ring->ev[q]);
    delete c->ring;
    c->ring = nullptr;
}
// 1 if there is no memory for it
static int ring_get(tbl_ctx *c)
{
    if (c->ring) return 0;
    c->ring = new (std::nothrow) XferRing();
    if (!c->ring) return 1;
    const size_t slot = XF_CHUNK * sizeof(double);
    hipError_t e = hipHostMalloc((void **)&c->ring->mem, XF_SLOTS * slot, hipHostMallocDefault);
    for (int q = 0; q < XF_SLOTS && e == hipSuccess; q++) {
        c->ring->buf[q] = c->ring->mem + q * slot;
        e = hipEventCreateWithFlags(&c->ring->ev[q], hipEventDisableTiming);
    }
    if (e == hipSuccess) return 0;
    (void)hipGetLastError();
    ring_free(c);
    return 1;
}
// chunk q of the host array to or from its slot
static void chunk_convert(char *slot, bool dbl, double *host, size_t m, bool to_dev)
{
    float *f = (float *)slot;
    if (dbl && to_dev) memcpy(slot, host, m * sizeof(double));
    else if (dbl) memcpy(host, slot, m * sizeof(double));
    else if (to_dev) for (size_t e = 0; e < m; e++) f[e] = (float)host[e];
    else for (size_t e = 0; e < m; e++) host[e] = f[e];
}
// the same without the ring
static int move_plain(tbl_ctx *c, void *dev, bool dbl, double *host, size_t n, bool to_dev)
{
    std::unique_ptr<float[]> tmp(dbl ? nullptr : new (std::nothrow) float[n]);
    if (!dbl && !tmp) return fail(c, TBL_EARG, "no host memory for a field's conversion");
    if (!dbl && to_dev)
        for (size_t e = 0; e < n; e++) tmp[e] = (float)host[e];
    void *h = dbl ? (void *)host : (void *)tmp.get();
    const size_t b = n * (dbl ? sizeof(double) : sizeof(float));
    HIPCHK(c, to_dev ? hipMemcpyAsync(dev, h, b, hipMemcpyHostToDevice, c->s)
                     : hipMemcpyAsync(h, dev, b, hipMemcpyDeviceToHost, c->s));
    HIPCHK(c, hipStreamSynchronize(c->s));
    if (!dbl && !to_dev)
        for (size_t e = 0; e < n; e++) host[e] = tmp[e];
    return 0;
}
// page-locked host memory, which the copy engine reads and writes itself
static bool is_pinned(const void *p)
{
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeHost;
    (void)hipGetLastError();                   // memory that the runtime does not know
    return false;
}
// n elements between dev (double or float) and host, in stream order; returns
// when they have arrived
static int move_field(tbl_ctx *c, void *dev, bool dbl, double *host, size_t n, bool to_dev)
{
    const size_t least = dbl ? (to_dev ? XF_D_UP : XF_D_DOWN) : (to_dev ? XF_F_UP : XF_F_DOWN);
    const long nch = (long)((n + XF_CHUNK - 1) / XF_CHUNK);
    std::unique_ptr<std::atomic<char>[]> done;                  // chunk q is converted
    if (n >= least && !(dbl && is_pinned(host)) && !ring_get(c)) done.reset(new (std::nothrow) std::atomic<char>[nch]);
    if (!done) return move_plain(c, dev, dbl, host, n, to_dev);
    for (long q = 0; q < nch; q++) done[q].store(0, std::memory_order_relaxed);
    XferRing &R = *c->ring;
    const size_t es = dbl ? sizeof(double) : sizeof(float);
    auto len = [&](long q) { return std::min(XF_CHUNK, n - (size_t)q * XF_CHUNK); };
    auto copy = [&](long q) -> hipError_t {                     // chunk q between its slot and the device
        char *d = (char *)dev + (size_t)q * XF_CHUNK * es, *h = R.buf[q % XF_SLOTS];
        hipError_t e = to_dev ? hipMemcpyAsync(d, h, len(q) * es, hipMemcpyHostToDevice, c->s)
                              : hipMemcpyAsync(h, d, len(q) * es, hipMemcpyDeviceToHost, c->s);
        return e == hipSuccess ? hipEventRecord(R.ev[q % XF_SLOTS], c->s) : e;
    };
    // the calling thread issues the copies in order; chunk q may be converted
    // from q < ready (to_dev: its slot is free; else: its copy was issued), and
    // done[q] follows
    std::atomic<long> next{0}, ready{to_dev ? std::min(nch, (long)XF_SLOTS) : 0};
    std::atomic<int> err{0};
    auto convert = [&](long q) {
        if (!to_dev) {
            const hipError_t e = hipEventSynchronize(R.ev[q % XF_SLOTS]);
            if (e != hipSuccess) { err.store((int)e); return; }
        }
        chunk_convert(R.buf[q % XF_SLOTS], dbl, host + (size_t)q * XF_CHUNK, len(q), to_dev);
        done[q].store(1, std::memory_order_release);
    };
    auto worker = [&]() {
        const hipError_t ed = hipSetDevice(c->dev);
        if (ed != hipSuccess) { err.store((int)ed); return; }
        for (long q; (q = next.fetch_add(1)) < nch;) {
            while (ready.load(std::memory_order_acquire) <= q) {
                if (err.load()) return;
                XF_NAP;
            }
            if (err.load()) return;
            convert(q);
        }
    };
    std::vector<std::thread> pool;
    const int nt = (int)std::min((long)XF_THREADS, nch);
    try {
        for (int t = 0; nt > 1 && t < nt; t++) pool.emplace_back(worker);
    } catch (const std::exception &) {                          // fewer threads, or none: the loops below still finish
    }
    // without workers the calling thread converts each chunk itself
    auto wait_done = [&](long q) {
        if (pool.empty()) { if (!done[q].load()) convert(q); return; }
        while (!done[q].load(std::memory_order_acquire) && !err.load()) XF_NAP;
    };
    long freed = 0;
    for (long q = 0; q < nch && !err.load(); q++) {
        if (to_dev) {
            wait_done(q);
            if (err.load()) break;
            const hipError_t e = copy(q);
            if (e != hipSuccess) { err.store((int)e); break; }
            if (q >= XF_SLOTS / 2) {                            // the slot of an earlier copy is free again
                const hipError_t e2 = hipEventSynchronize(R.ev[freed % XF_SLOTS]);
                if (e2 != hipSuccess) { err.store((int)e2); break; }
                freed++;
                ready.store(std::min(nch, freed + XF_SLOTS), std::memory_order_release);
            }
        } else {
            if (q >= XF_SLOTS) wait_done(q - XF_SLOTS);
            if (err.load()) break;
            const hipError_t e = copy(q);
            if (e != hipSuccess) { err.store((int)e); break; }
            ready.store(q + 1, std::memory_order_release);
        }
    }
    if (!to_dev)
        for (long q = std::max(0L, nch - XF_SLOTS); q < nch && !err.load(); q++) wait_done(q);
    for (auto &t : pool) t.join();
    const hipError_t es2 = hipStreamSynchronize(c->s);
    if (err.load()) HIPCHK(c, (hipError_t)err.load());
    HIPCHK(c, es2);
    return 0;
}
static int put_field(tbl_ctx *c, void *dst, bool dbl, const double *host, size_t n)
{
    return move_field(c, dst, dbl, const_cast<double *>(host), n, true);
}
static int get_field(tbl_ctx *c, const void *src, bool dbl, double *host, size_t n)
{
    return move_field(c, const_cast<void *>(src), dbl, host, n, false);
}

extern "C" int tbl_field_set(tbl_ctx *c, int f, const double *host)
{
    if (c && f == TBL_F_PCORR) c->pc_hist = 0;
    if (!c || !host || f < 0 || f > TBL_F_WORK) return TBL_EARG;
    bool dbl;
    void *d = field_ptr(c, f, &dbl);
    CHK(put_field(c, d, dbl, host, field_len(c, f)));
    if (f == TBL_F_UT) c->uploaded = true;
    if (f == TBL_F_WORK) {   // keep the work vector's faces zero (see op_impl)
        if (c->mixed) launch_zero_faces<float>(c->g, (float *)d, c->s);
        else launch_zero_faces<double>(c->g, (double *)d, c->s);
        HIPCHK(c, hipStreamSynchronize(c->s));
    }
    return 0;
}
extern "C" int tbl_field_get(tbl_ctx *c, int f, double *host)
{
    if (!c || !host || f < 0 || f > TBL_F_WORK) return TBL_EARG;
    bool dbl;
    void *d = field_ptr(c, f, &dbl);
    return get_field(c, d, dbl, host, field_len(c, f));
}
extern "C" int tbl_upload(tbl_ctx *c, const double *Ut, const double *Press, const double *PCorr)
{
    if (!c) return TBL_EARG;
    if (Ut) CHK(tbl_field_set(c, TBL_F_UT, Ut));
    if (Press) CHK(tbl_field_set(c, TBL_F_PRESS, Press));
    if (PCorr) CHK(tbl_field_set(c, TBL_F_PCORR, PCorr));
    if (PCorr) c->pc_hist = 0;
    return 0;
}
extern "C" int tbl_download(tbl_ctx *c, double *Ut, double *Press, double *PCorr)
{
    if (!c) return TBL_EARG;
    if (Ut) CHK(tbl_field_get(c, TBL_F_UT, Ut));
    if (Press) CHK(tbl_field_get(c, TBL_F_PRESS, Press));
    if (PCorr) CHK(tbl_field_get(c, TBL_F_PCORR, PCorr));
    return 0;
}

static int h2d(tbl_ctx *c, void *d, const void *h, size_t b)
{
    HIPCHK(c, hipMemcpyAsync(d, h, b, hipMemcpyHostToDevice, c->s));
    return 0;
}
static int d2h(tbl_ctx *c, void *h, const void *d, size_t b)
{
    HIPCHK(c, hipMemcpyAsync(h, d, b, hipMemcpyDeviceToHost, c->s));
    return 0;
}

// Results the host waits for (stopping tests, diagnostics): a kernel publishes
// them (Pub) and pub_wait spins on the sequence number, since the next launch
// waits on the host's wake-up.  Work gated on the device's own stopping flags
// can be queued in between: the GPU then runs it while the host waits.  The
// first POLL_SPIN_US microseconds spin tightly; after that every turn asks the
// stream for errors and yields the core (sched_yield), so a long wait does not
// keep a host core from the caller's other threads, and a stream that has
// failed or drained without publishing ends the wait.
#define POLL_SPIN_US 20
static Pub pub_of(tbl_ctx *c, void *dst)
{
    Pub p;
    p.seq = &c->hp->seq;
    p.dst = dst;
    p.val = ++c->pseq;
    return p;
}
static int pub_wait(tbl_ctx *c)
{
    auto there = [&] { return (int)(__atomic_load_n(&c->hp->seq, __ATOMIC_ACQUIRE) - c->pseq) >= 0; };
    const auto t0 = std::chrono::steady_clock::now();
    bool spin = true;
    while (!there()) {
        if (spin) {
            spin = std::chrono::steady_clock::now() - t0 < std::chrono::microseconds(POLL_SPIN_US);
            continue;
        }
        const hipError_t e = hipStreamQuery(c->s);
        if (e == hipSuccess && !there()) return fail(c, TBL_ESTATE, "a kernel ended without publishing its result");
        if (e != hipSuccess && e != hipErrorNotReady) HIPCHK(c, e);
        sched_yield();
    }
    return 0;
}
// the diagnostics record, after the kernels queued so far
static int read_diag(tbl_ctx *c)
{
    launch_publish(c->dd, DD_NCOUNT, pub_of(c, c->dh), c->s);
    HIPCHK(c, hipGetLastError());
    return pub_wait(c);
}
// the GMRES status, likewise
static void ask_status(tbl_ctx *c) { launch_publish(&c->gm->st, sizeof(GmStatus) / 8, pub_of(c, c->gm_h), c->s); }

extern "C" int tbl_set_state(tbl_ctx *c, const tbl_state *st)
{
    if (!c || !st) return TBL_EARG;
    const tbl_params &p = c->p;
    const size_t M = (size_t)p.nX * p.nZ;
    if (st->sums) CHK(h2d(c, c->sums, st->sums, 9 * M * 8));
    if (st->avg) CHK(h2d(c, c->avg, st->avg, 9 * M * 8));
    if (st->Wt) CHK(h2d(c, c->Wt, st->Wt, M * 8));
    if (st->newk) {
        for (int k = 0; k < p.nZ; k++)
            if (st->newk[k] < 1 || st->newk[k] > p.nZ) return fail(c, TBL_EARG, "newk out of range");
        CHK(h2d(c, c->newk, st->newk, p.nZ * sizeof(int)));
    }
    if (st->Ume) CHK(h2d(c, c->Ume, st->Ume, p.nZ * 8));
    if (st->Ufluc_rec) CHK(h2d(c, c->uf, st->Ufluc_rec, 3L * p.nY * p.nZ * 8));
    if (st->bltkns) CHK(h2d(c, c->bltkns, st->bltkns, p.nX * 8));
    if (st->deltastar) CHK(h2d(c, c->dstar, st->deltastar, p.nX * 8));
    if (st->theta) CHK(h2d(c, c->theta, st->theta, p.nX * 8));
    if (st->wall_w) {
        CHK(h2d(c, c->wall_w, st->wall_w, (size_t)p.nX * p.nY * 8));
        c->have_wall_w = true;
    }
    RecDev r = {st->lamda, st->lamda03, 0};
    CHK(h2d(c, c->rec, &r, sizeof(r)));
    c->time = st->time;
    c->nstep = st->nstep;
    c->cnt = st->cnt;
    HIPCHK(c, hipStreamSynchronize(c->s));
    return 0;
}

extern "C" int tbl_get_state(tbl_ctx *c, tbl_state *st)
{
    if (!c || !st) return TBL_EARG;
    const tbl_params &p = c->p;
    const size_t M = (size_t)p.nX * p.nZ;
    if (st->sums) CHK(d2h(c, st->sums, c->sums, 9 * M * 8));
    if (st->avg) CHK(d2h(c, st->avg, c->avg, 9 * M * 8));
    if (st->Wt) CHK(d2h(c, st->Wt, c->Wt, M * 8));
    if (st->newk) CHK(d2h(c, st->newk, c->newk, p.nZ * sizeof(int)));
    if (st->Ume) CHK(d2h(c, st->Ume, c->Ume, p.nZ * 8));
    if (st->Ufluc_rec) CHK(d2h(c, st->Ufluc_rec, c->uf, 3L * p.nY * p.nZ * 8));
    if (st->bltkns) CHK(d2h(c, st->bltkns, c->bltkns, p.nX * 8));
    if (st->deltastar) CHK(d2h(c, st->deltastar, c->dstar, p.nX * 8));
    if (st->theta) CHK(d2h(c, st->theta, c->theta, p.nX * 8));
    if (st->wall_w) CHK(d2h(c, st->wall_w, c->wall_w, (size_t)p.nX * p.nY * 8));
    RecDev r;
    CHK(d2h(c, &r, c->rec, sizeof(r)));
    HIPCHK(c, hipStreamSynchronize(c->s));
    st->lamda = r.lamda;
    st->lamda03 = r.lamda03;
    st->time = c->time;
    st->nstep = c->nstep;
    st->cnt = c->cnt;
    return 0;
}

extern "C" int tbl_get_mesh(const tbl_ctx *c, double *x1, double *x2, double *x3, double *Jac, double *Jac2,
                            double *Ab, double *At, double *Ap)
{
    if (!c) return TBL_EARG;
    auto cp = [](double *dst, const std::vector<double> &v) { if (dst) memcpy(dst, v.data(), v.size() * sizeof(double)); };
    cp(x1, c->x1); cp(x2, c->x2); cp(x3, c->x3); cp(Jac, c->Jac); cp(Jac2, c->Jac2);
    cp(Ab, c->Ab); cp(At, c->At); cp(Ap, c->Ap);
    return 0;
}

// ------------------------------------------------------------------ checkpoint
// Binary checkpoint of everything a step reads from earlier steps: the
// fields in their storage precision (bit for bit), the pressure-correction
// warm start (and the previous one of the extrapolated guess), the
// statistics and recycling state, the wall-shear window and the clock.
// Layout: 8-byte magic, the int32 header below, the double time, then one
// record per buffer (uint64 byte count, then the bytes), in a fixed order.
static const char CKPT_MAGIC[8] = {'T', 'B', 'L', 'C', 'K', 'P', 'T', '1'};
enum { CKPT_VERSION = 1 };
struct CkptHead {
    int version, nX, nY, nZ, precision, pc_hist, have_wall_w, nstep, cnt, nwin;
};
struct CkptRec {
    void *dev;
    size_t bytes;
};
static std::vector<CkptRec> ckpt_records(tbl_ctx *c)
{
    const tbl_params &p = c->p;
    const size_t N = (size_t)c->g.N, M = (size_t)p.nX * p.nZ;
    return {{c->Ut, 3 * N * c->es}, {c->Press, N * c->es}, {c->PCorr, N * 8},
            {c->PCprev, c->PCprev ? N * 8 : 0}, {c->sums, 9 * M * 8}, {c->avg, 9 * M * 8}, {c->Wt, M * 8},
            {c->Ume, (size_t)p.nZ * 8}, {c->uf, 3 * (size_t)p.nY * p.nZ * 8}, {c->bltkns, (size_t)p.nX * 8},
            {c->dstar, (size_t)p.nX * 8}, {c->theta, (size_t)p.nX * 8}, {c->wall_w, (size_t)p.nX * p.nY * 8},
            {c->newk, (size_t)p.nZ * sizeof(int)}, {c->rec, sizeof(RecDev)}, {c->tausum, (size_t)p.nX * 8},
            {c->taumean, (size_t)p.nX * 8}, {c->cf, (size_t)p.nX * 8}};
}
#define CKPT_CHUNK ((size_t)1 << 28)

extern "C" int tbl_checkpoint_save(tbl_ctx *c, const char *path)
{
    if (!c || !path) return TBL_EARG;
    if (!c->uploaded) return fail(c, TBL_ESTATE, "tbl_checkpoint_save before tbl_upload");
    HIPCHK(c, hipStreamSynchronize(c->s));
    FILE *f = fopen(path, "wb");
    if (!f) return fail(c, TBL_EARG, "tbl_checkpoint_save: cannot open the file for writing");
    CkptHead h = {CKPT_VERSION, c->p.nX, c->p.nY, c->p.nZ, c->p.precision, c->pc_hist, c->have_wall_w ? 1 : 0,
                  c->nstep, c->cnt, c->nwin};
    bool ok = fwrite(CKPT_MAGIC, 8, 1, f) == 1 && fwrite(&h, sizeof(h), 1, f) == 1 &&
              fwrite(&c->time, sizeof(double), 1, f) == 1;
    std::vector<char> buf;
    for (const CkptRec &r : ckpt_records(c)) {
        const uint64_t nb = r.bytes;
        ok = ok && fwrite(&nb, sizeof(nb), 1, f) == 1;
        for (size_t o = 0; ok && o < r.bytes; o += CKPT_CHUNK) {
            const size_t n = std::min(CKPT_CHUNK, r.bytes - o);
            buf.resize(n);
            hipError_t e = hipMemcpy(buf.data(), (char *)r.dev + o, n, hipMemcpyDeviceToHost);
            if (e != hipSuccess) {
                fclose(f);
                c->err = std::string("tbl_checkpoint_save: ") + hipGetErrorString(e);
                return (int)e;
            }
            ok = fwrite(buf.data(), 1, n, f) == n;
        }
    }
    ok = (fclose(f) == 0) && ok;
    return ok ? 0 : fail(c, TBL_EARG, "tbl_checkpoint_save: write failed");
}

extern "C" int tbl_checkpoint_load(tbl_ctx *c, const char *path)
{
    if (!c || !path) return TBL_EARG;
    FILE *f = fopen(path, "rb");
    if (!f) return fail(c, TBL_EARG, "tbl_checkpoint_load: cannot open the file");
    char magic[8];
    CkptHead h;
    double t = 0.0;
    if (fread(magic, 8, 1, f) != 1 || memcmp(magic, CKPT_MAGIC, 8) != 0 || fread(&h, sizeof(h), 1, f) != 1 ||
        fread(&t, sizeof(t), 1, f) != 1 || h.version != CKPT_VERSION) {
        fclose(f);
        return fail(c, TBL_EARG, "tbl_checkpoint_load: not a checkpoint of this version");
    }
    if (h.nX != c->p.nX || h.nY != c->p.nY || h.nZ != c->p.nZ || h.precision != c->p.precision) {
        fclose(f);
        return fail(c, TBL_EARG, "tbl_checkpoint_load: grid or precision differs from the context's");
    }
    HIPCHK(c, hipStreamSynchronize(c->s));
    std::vector<char> buf;
    const size_t N = (size_t)c->g.N;
    for (int q = 0; q < (int)ckpt_records(c).size(); q++) {
        uint64_t nb = 0;
        if (fread(&nb, sizeof(nb), 1, f) != 1) { fclose(f); return fail(c, TBL_EARG, "tbl_checkpoint_load: truncated file"); }
        if (q == 3 && nb > 0 && !c->PCprev) {          // the extrapolation history
            int rc = dalloc(c, &c->PCprev, N * sizeof(double));
            if (rc) { fclose(f); return rc; }
            HIPCHK(c, hipStreamSynchronize(c->s));
        }
        const CkptRec r = ckpt_records(c)[q];
        if (nb != r.bytes) { fclose(f); return fail(c, TBL_EARG, "tbl_checkpoint_load: record size mismatch"); }
        for (size_t o = 0; o < r.bytes; o += CKPT_CHUNK) {
            const size_t n = std::min(CKPT_CHUNK, r.bytes - o);
            buf.resize(n);
            if (fread(buf.data(), 1, n, f) != n) { fclose(f); return fail(c, TBL_EARG, "tbl_checkpoint_load: truncated file"); }
            hipError_t e = hipMemcpy((char *)r.dev + o, buf.data(), n, hipMemcpyHostToDevice);
            if (e != hipSuccess) {
                fclose(f);
                c->err = std::string("tbl_checkpoint_load: ") + hipGetErrorString(e);
                return (int)e;
            }
        }
    }
    fclose(f);
    c->pc_hist = h.pc_hist;
    c->have_wall_w = h.have_wall_w != 0;
    c->nstep = h.nstep;
    c->cnt = h.cnt;
    c->nwin = h.nwin;
    c->time = t;
    c->uploaded = true;
    return 0;
}

// ------------------------------------------------------------------ blocks
template <class T> static T *F(void *p) { return (T *)p; }

extern "C" int tbl_begin_step(tbl_ctx *c)
{
    if (!c) return TBL_EARG;
    if (!c->uploaded) return fail(c, TBL_ESTATE, "tbl_begin_step before tbl_upload");
    c->time = c->time + c->p.dt;
    c->nstep += 1;
    c->cnt += 1;
    // Utold = Ut (:257); the step reads Utold only at the inflow plane of u
    // (the (u - u_old)/dt term of the inflow pressure, :791), so only that
    // plane is saved
    if (c->mixed) launch_save_inflow<float>(c->g, F<float>(c->Ut), F<float>(c->Utold), c->s);
    else launch_save_inflow<double>(c->g, F<double>(c->Ut), F<double>(c->Utold), c->s);
    HIPCHK(c, hipGetLastError());
    return 0;
}

template <class T> static int recycle_impl(tbl_ctx *c)
{
    double eps = c->nstep * (5.0e-5);
    if (eps > 1.0) eps = 1.0;
    if (!(c->nstep > c->p.freq_tim_avg)) return 0;
    Tscope ts(c, TBL_K_RECYCLE, 6.0 * c->p.nY * c->p.nZ * 8);
    launch_recycle<T>(c->g, F<T>(c->Ut), c->p.i_rec - 1, eps, &c->rec->lamda, c->avg, c->Wt, c->newk, c->Ume,
                      c->uf, c->s);
    HIPCHK(c, hipGetLastError());
    return 0;
}
extern "C" int tbl_recycle_inflow(tbl_ctx *c)
{
    if (!c) return TBL_EARG;
    return c->mixed ? recycle_impl<float>(c) : recycle_impl<double>(c);
}

template <class T> static int rhs_impl(tbl_ctx *c, double *hpart = nullptr)
{
    Tscope ts(c, TBL_K_RHS, 7.0 * (double)c->g.N * sizeof(T));
    launch_momentum_rhs<T>(c->g, F<T>(c->Ut), F<T>(c->Press), F<T>(c->Q), c->s, c->br_in, c->br_out, hpart);
    HIPCHK(c, hipGetLastError());
    return 0;
}
extern "C" int tbl_momentum_rhs(tbl_ctx *c)
{
    if (!c) return TBL_EARG;
    return c->mixed ? rhs_impl<float>(c) : rhs_impl<double>(c);
}

// Components per launch of the direct and transposed solves.  Three (see
// solve_batched) need a residual field and work fields of three components,
// allocated by the first such solve; without the memory, and on larger grids,
// the solves go one by one, with the work vector r (its faces are zero) for the
// residual.
static int direct_batch(tbl_ctx *c)
{
    if (!solve_batched(c->g, c->mixed)) return 1;
    if (!c->r3 && try_alloc(c, &c->r3, 3 * (size_t)c->g.N * c->es)) return 1;
    return fastpc_reserve(c->fast, c->g, 3, c->s) ? 1 : 3;
}
// exact Helmholtz solve of the three components: u += (I - hA)^{-1} (Q - H u), by fast
// diagonalisation; in FP64 twice (one refinement step on the residual).  In
// FP32 storage once: I - hA is well conditioned (the stretched grid's
// largest h lambda is about 2), so one FP32 fast solve is already at the
// FP32 rounding of the stored field, which a refinement cannot improve
template <class T> static int helm_direct(tbl_ctx *c, int *sweeps, double *res)
{
    if (!c->fast) return fail(c, TBL_ESTATE, "direct Helmholtz solve without the fast solver");
    const Geo &g = c->g;
    const long N = g.N;
    const int nc = direct_batch(c);            // components per solve
    T *r = F<T>(nc == 3 ? c->r3 : c->r);
    const double h = c->p.dt / c->p.Re;
    const int passes = sizeof(T) == sizeof(double) ? 2 : 1;
    for (int p = 0; p < 3; p += nc) {
        FastIO io;
        io.in = r;
        io.out = F<T>(c->Ut) + p * N;
        io.in64 = io.out64 = sizeof(T) == sizeof(double);
        io.add = 1;
        io.ncomp = nc;
        for (int it = 0; it < passes; it++) {
            Tscope ts(c, TBL_K_HELM, 4.0 * nc * (double)N * sizeof(T));
            launch_helm_rfield<T>(g, F<T>(c->Q) + p * N, F<T>(c->Ut) + p * N, r, nc, c->s);
            if (run_fast_solve(c->fast, g, io, nullptr, 1.0, -h, false, c->s))
                return fail(c, TBL_EARG, "fast solver failure in the direct Helmholtz solve");
        }
    }
    HIPCHK(c, hipGetLastError());
    if (sweeps) for (int p = 0; p < 3; p++) sweeps[p] = passes;
    if (res) for (int p = 0; p < 3; p++) res[p] = 0.0;
    return 0;
}

// pre_nb > 0: the first residual pass was formed by the momentum kernel
// (pre_nb block partials in c->part)
// ppe_done (whole step only): the PPE right-hand side of the solution is
// queued behind each stopping-test read-back, gated on the device's active
// flags, and *ppe_done says whether the gated launch that ran was the final
// one (off while the PPE right-hand side's timer class is timed)
template <class T> static int helm_impl(tbl_ctx *c, double errorstop, int mmax, int *sweeps, double *res, int pre_nb = 0,
                                        bool *ppe_done = nullptr)
{
    if (ppe_done) *ppe_done = false;
    if (c->p.helm_mode == TBL_HELM_DIRECT) return helm_direct<T>(c, sweeps, res);
    const bool ppe_ahead = ppe_done && !(c->tmask & (1u << TBL_K_DIV));
    // the z-line sweep converges in a few iterations: poll the stopping test
    // of every residual pass (odd it >= 3) before launching the sweeps, so
    // that no sweep is launched for components that have all stopped; point
    // sweeps poll every 8 iterations on small grids
    const bool zebra = c->p.helm_mode == TBL_HELM_ZEBRA;
    const bool every = (c->g.N > 2000000 || c->p.helm_mode == TBL_HELM_ZLINE_RB || zebra ||
                        c->p.helm_mode == TBL_HELM_LEX_SLAB);
    // zebra: sweeps read cur and write alt, which then swap; the boundary and
    // ghost values (not changed by the solve) are copied into alt first
    T *cur = F<T>(c->Ut), *alt = zebra ? F<T>(c->Ualt) : nullptr;
    if (zebra) launch_copy_faces3<T>(c->g, cur, alt, c->gs, c->s);
    else launch_gs_init(c->gs, c->s);
    int act[3] = {1, 1, 1}, sw[3] = {0, 0, 0};
    double rs[3] = {0, 0, 0};
    bool fresh = false;                        // gs_h holds the final control block
    int it;
    for (it = 1; it <= mmax; it++) {
        if (it % 2 == 1) {
            const bool pre = (it == 1 && pre_nb > 0);
            if (!pre) {
                Tscope ts(c, TBL_K_HELM_RES, 2.0 * (act[0] + act[1] + act[2]) * (double)c->g.N * sizeof(T));
                launch_helm_resid<T>(c->g, F<T>(c->Q), zebra ? cur : F<T>(c->Ut), c->gs, c->part, it == 1 ? 1 : 0,
                                     c->s);
            }
            const bool poll = it >= 3 && (every || it % 8 == 1);
            launch_helm_fin(c->g, c->gs, c->part, it, errorstop, c->mixed ? 32.0 * 1.1920928955078125e-7 : 0.0, c->s,
                            pre ? pre_nb : 0, poll ? pub_of(c, c->gs_h) : Pub());
            if (poll) {
                if (ppe_ahead) launch_ppe_rhs<T>(c->g, zebra ? cur : F<T>(c->Ut), c->pRhs, c->s, c->gs);
                CHK(pub_wait(c));
                gs_ctrl_read(c->gs_h, act, sw, rs);
                if (!act[0] && !act[1] && !act[2]) {
                    fresh = true;
                    if (ppe_ahead) *ppe_done = true;
                    break;
                }
            }
        }
        // one timed launch per colour; algorithmic bytes of a colour pass: read
        // Q and the other colour's u, write this colour's u, i.e. 1.5 N values
        // per active component (the host's view of the active set is exact
        // when it polls every residual pass, an upper bound otherwise)
        if (zebra) {
            // algorithmic bytes of a zebra pass: Q, the pass's rows (x
            // neighbours), the other rows (span neighbours) and the new rows,
            // each half the grid: 2 N values per active component; an ended
            // component is copied through (N values)
            const int na = act[0] + act[1] + act[2];
            {
                // one timed scope for the sweep's two passes (launched back to
                // back): each event record leaves a gap of a few microseconds
                Tscope ts(c, TBL_K_HELM, 2.0 * (2.0 * na + 1.0 * (3 - na)) * (double)c->g.N * sizeof(T), 2);
                for (int colour = 0; colour < 2; colour++)
                    launch_helm_zebra<T>(c->g, F<T>(c->Q), cur, colour == 0 ? cur : alt, alt, F<T>(c->zf), c->gs,
                                         colour, c->s);
            }
            std::swap(cur, alt);
            HIPCHK(c, hipGetLastError());
            continue;
        }
        if (c->p.helm_mode == TBL_HELM_LEX_SLAB) {
            // one lexicographic sweep per slab: read Q, read and write u (the
            // neighbours come from registers, LDS and cache): 3 N values per
            // active component
            Tscope ts(c, TBL_K_HELM, 3.0 * (act[0] + act[1] + act[2]) * (double)c->g.N * sizeof(T));
            launch_helm_lex<T>(c->g, F<T>(c->Q), F<T>(c->Ut), F<T>(c->scr), c->gs, c->s);
            HIPCHK(c, hipGetLastError());
            continue;
        }
        for (int colour = 0; colour < 2; colour++) {
            Tscope ts(c, TBL_K_HELM, 1.5 * (act[0] + act[1] + act[2]) * (double)c->g.N * sizeof(T));
            if (c->p.helm_mode == TBL_HELM_ZLINE_RB)
                launch_helm_zline<T>(c->g, F<T>(c->Q), F<T>(c->Ut), F<T>(c->zf), c->gs, colour, c->s);
            else
                launch_helm_sweep<T>(c->g, F<T>(c->Q), F<T>(c->Ut), c->gs, colour, c->s);
        }
        HIPCHK(c, hipGetLastError());
    }
    if (!fresh) {
        launch_publish(c->gs, (int)(gs_ctrl_bytes() / 8), pub_of(c, c->gs_h), c->s);
        HIPCHK(c, hipGetLastError());
        CHK(pub_wait(c));
        gs_ctrl_read(c->gs_h, act, sw, rs);
    }
    if (zebra && cur != F<T>(c->Ut)) std::swap(c->Ut, c->Ualt);   // the solution is in cur
    bool capped = false;
    for (int p = 0; p < 3; p++)
        if (act[p]) { sw[p] = mmax; capped = true; }
    if (sweeps) for (int p = 0; p < 3; p++) sweeps[p] = sw[p];
    if (res) for (int p = 0; p < 3; p++) res[p] = rs[p];
    if (capped && c->p.fail_on_noconv) return fail(c, TBL_ENOCONV, "Gauss-Seidel reached gs_mmax");
    return 0;
}
extern "C" int tbl_diffusion_solve(tbl_ctx *c, double errorstop, int mmax, int *sweeps3, double *res3)
{
    if (!c || mmax < 1) return TBL_EARG;
    return c->mixed ? helm_impl<float>(c, errorstop, mmax, sweeps3, res3)
                    : helm_impl<double>(c, errorstop, mmax, sweeps3, res3);
}

template <class T> static int prhs_impl(tbl_ctx *c)
{
    Tscope ts(c, TBL_K_DIV, (double)c->g.N * (3.0 * sizeof(T) + 8.0));
    launch_ppe_rhs<T>(c->g, F<T>(c->Ut), c->pRhs, c->s);
    HIPCHK(c, hipGetLastError());
    return 0;
}
extern "C" int tbl_ppe_rhs(tbl_ctx *c)
{
    if (!c) return TBL_EARG;
    return c->mixed ? prhs_impl<float>(c) : prhs_impl<double>(c);
}

// algorithmic HBM bytes of one preconditioner application in storage type T:
// fast diagonalisation = four transforms and the line solve, each reading and
// writing the field once (10 N); block SSOR = forward (read r, write) and
// backward (read, write) sweeps (4 N); red-black SSOR = forward (read r, write
// the half sweep) and backward (read r and the half sweep, write) (5 N);
// Jacobi / none = read and write (2 N)
static double precond_bytes(const tbl_ctx *c, size_t es)
{
    const double N = (double)c->g.N;
    switch (c->p.precond) {
    case TBL_PC_FAST: return 10.0 * N * es;
    case TBL_PC_SSOR_BLOCK: return 4.0 * N * es;
    case TBL_PC_SSOR_RB: return 5.0 * N * es;
    default: return 2.0 * N * es;
    }
}

// restarted GMRES; each cycle forms the true residual in double (outer
// refinement) and runs at most kmax Arnoldi steps in the storage type T.
template <class T>
static int gmres_impl(tbl_ctx *c, double errtol, int kmax, int mmax, int *cycles, int *iters, double *true_res)
{
    const Geo &g = c->g;
    const long N = g.N;
    const unsigned nbv = vec_blocks(N, sizeof(T) == sizeof(float)), nbr = resid_blocks(g);
    T *V = F<T>(c->V), *W = F<T>(c->W), *scr = F<T>(c->scr), *r = F<T>(c->r);
    const long ldv = c->ldv;
    if (kmax > c->p.kmax) return fail(c, TBL_EARG, "kmax above the allocated restart length");
    const int mode = (c->p.tol_mode == TBL_TOL_TRUE) ? GM_MODE_TRUE : GM_MODE_REF;
    const int poll = (N > 2000000 || c->p.precond == TBL_PC_FAST) ? 1 : 4;
    // the second PCorr buffer of fused updates (TRUE) and of unit steps, which a
    // solve by the reference's rule does without where there is no memory for it
    const bool fused = mode == GM_MODE_TRUE && poll == 1;
    bool unit_steps = c->p.precond == TBL_PC_FAST && sizeof(T) == sizeof(double);
    // the reference's rule: a unit step that one solve's accuracy cannot meet is
    // not tried (a refused one costs a residual pass, a preconditioner application
    // and a norm: errtol 1e-14 at 256x64x96 389 -> 432 us a solve).  One that is
    // accepted saves 30 to 45 %, so the line lies low: on 26 grids of 1 k to 50 M
    // cells a solve reaches 0.3 to 10 times fastpc_reach, or rounding, 1e-15 to 2e-14.
    if (mode == GM_MODE_REF && unit_steps && errtol < fastpc_reach(c->fast)) unit_steps = false;
    if (fused && !c->PCalt) CHK(dalloc(c, &c->PCalt, (size_t)N * sizeof(double)));
    if (unit_steps && !c->PCalt && try_alloc(c, &c->PCalt, (size_t)N * sizeof(double))) unit_steps = false;
    const bool two = fused || unit_steps;
    launch_gm_init(g, c->gm, errtol, c->p.inner_tol, kmax, mmax, mode, c->PCorr, two ? c->PCalt : nullptr, c->s);
    double *part_r = c->part;                  // residual partials
    double *part_z = c->part + nbr + 8;        // norm partials (and dot partials)
    const bool fuse_dot = poisson_blocks(g, c->mixed) <= c->npart - nbr - 8;
    if (c->p.pc_extrap) {
        // initial guess 2 PCorr(n-1) - PCorr(n-2), both with zero faces
        if (!c->PCprev) CHK(dalloc(c, &c->PCprev, (size_t)N * sizeof(double)));
        if (c->pc_hist >= 2) launch_pc_extrap(c->PCorr, c->PCprev, N, c->s);
        else HIPCHK(c, hipMemcpyAsync(c->PCprev, c->PCorr, (size_t)N * sizeof(double), hipMemcpyDeviceToDevice, c->s));
        c->pc_hist = c->pc_hist < 2 ? c->pc_hist + 1 : 2;
    }
    const int *act = &c->gm->st.active;
    bool final_res = false;                    // st.true_res is the residual of the final PCorr
    if (mode == GM_MODE_TRUE) {
        // Flexible (right-preconditioned) GMRES: the Givens estimate is the true
        // residual, one preconditioner application per Arnoldi step, and the
        // correction x += sum y_i z_i uses the stored z_i = M^{-1} v_i.  Each
        // cycle starts from the double-precision residual (iterative refinement).
        T *Z = F<T>(c->Z);
        // A cycle that ends after one Arnoldi step (known exactly when the
        // host polls every step) leaves its correction PCorr += y z0 pending:
        // the next cycle's residual kernel forms it on the fly and writes the
        // updated PCorr to the second buffer, which then becomes PCorr.
        const bool fuse_upd = (poll == 1);
        // queue-ahead of the first transform (off while the preconditioner
        // class is timed, so that its timer brackets whole applications)
        const bool ahead = c->p.precond == TBL_PC_FAST && !(c->tmask & (1u << TBL_K_PRECOND));
        // a cycle that stops after its first Arnoldi step goes on with
        // fin_cycle and the next cycle's fused residual pass: both are queued
        // behind that step's status read-back, gated on the cycle having ended
        // (off while the residual class is timed)
        const bool ahead_res = fuse_upd && !(c->tmask & (1u << TBL_K_RESID));
        // With the fast preconditioner the first Arnoldi step is the last of its
        // cycle if the cycle asks for no more than one solve gives: its vector is
        // then only measured, and formed when the status asks for a second step
        // after all (1024x256x192 mixed 98 -> 77 us).  One FP32 solve gives 1e-4 to
        // 1e-5 on the larger grids (with an inner_tol of 1e-5 and the vector formed
        // after its norm, a solve of 1024x256x192 took 5.83 instead of 5.70 ms); in
        // FP64 a unit step was refused if the Arnoldi steps run before the last cycle.
        auto norm_only = [&](bool unit) {
            return c->p.precond == TBL_PC_FAST && kmax > 1 && (unit_steps ? unit : c->p.inner_tol >= 3e-5);
        };
        bool pend = false;
        bool queued = false;                   // the cycle's residual pass ran behind the last read-back
        // unit steps (k_fin_unit) while they are accepted, in FP64: the fast
        // preconditioner inverts A to its storage type's rounding, so a cycle
        // is z_0 = M^{-1} r, the residual of PCorr + z_0 and one read-back; the
        // operator apply, the dot product and the orthogonalisation pass of
        // the Arnoldi step are not run, nor the read-back at the solve's start.
        // The step's residual goes to the other of two vectors (v0, v1), so
        // that a refused step leaves v_0 for the Arnoldi steps; the other is W,
        // which these solves do not use otherwise (r is the caller's TBL_F_WORK).
        // Mixed contexts run the Arnoldi step: its coefficient differs from 1
        // in the seventh digit there, and a PCorr that differs at all moves
        // some value of the FP32 fields by a rounding, which grows to what
        // FP32 leaves open (the pressure of 333x94x131 after 40 steps: 4e-6,
        // and 1e-3 at a point where a switch of the convection tripped).
        bool unit = unit_steps;
        bool opened = false;                   // the last unit step opened this cycle
        bool head = false;                     // its first transform ran behind the last read-back
        T *v0 = V, *v1 = W;
        for (int m = 0; m < mmax; m++) {
            const bool try_unit = unit && m + 1 < mmax;   // the last cycle allowed is not followed by a start
            if (opened) {
            } else if (queued) {
                queued = false;
            } else if (pend) {
                Tscope ts(c, TBL_K_RESID, (double)N * (24.0 + 2.0 * sizeof(T)));
                launch_resid_upd<T>(g, c->pRhs, c->PCorr, Z, c->gm, c->PCalt, V, part_r, c->s);
                std::swap(c->PCorr, c->PCalt);
                pend = false;
            } else {
                // the first residual also gives ||pRhs|| (partials after part_r)
                Tscope ts(c, TBL_K_RESID, (double)N * (16.0 + sizeof(T)));
                launch_resid<T>(g, c->pRhs, c->PCorr, V, part_r, c->s, m == 0 ? part_z : nullptr);
            }
            if (!opened)
                launch_fin_start(c->gm, part_r, (int)nbr, part_r, (int)nbr, m == 0 ? 1 : 0, c->s,
                                 m == 0 ? part_z : nullptr);
            bool have_z0 = false;
            if (try_unit) {
                {
                    Tscope ts(c, TBL_K_PRECOND, precond_bytes(c, sizeof(T)));
                    launch_precond<T>(g, c->p.precond, c->fast, v0, scr, Z, act, c->s, head ? FPC_TAIL : FPC_ALL);
                }
                {
                    Tscope ts(c, TBL_K_RESID, (double)N * (24.0 + 2.0 * sizeof(T)));
                    launch_resid_upd<T>(g, c->pRhs, c->PCorr, Z, c->gm, c->PCalt, v1, part_r, c->s, RU_UNIT);
                }
                launch_fin_unit(c->gm, part_r, (int)nbr, nullptr, 0, pub_of(c, c->gm_h), c->s);
                HIPCHK(c, hipGetLastError());
                if (ahead) launch_precond<T>(g, c->p.precond, c->fast, v1, scr, Z, act, c->s, FPC_HEAD);
                CHK(pub_wait(c));
                opened = head = false;
                if (c->gm_h->unit_ok) {
                    std::swap(c->PCorr, c->PCalt);
                    std::swap(v0, v1);
                    opened = true;
                    head = ahead;
                }
                if (c->gm_h->outer_done) { final_res = true; break; }
                if (opened) continue;
                unit = false;
                have_z0 = true;
                if (v0 != V) HIPCHK(c, hipMemcpyAsync(V, v0, (size_t)N * sizeof(T), hipMemcpyDeviceToDevice, c->s));
                v0 = V;
            } else {
                // after an accepted unit step the status is known and v_0 may
                // lie in the other vector
                if (opened && v0 != V) {
                    HIPCHK(c, hipMemcpyAsync(V, v0, (size_t)N * sizeof(T), hipMemcpyDeviceToDevice, c->s));
                    v0 = V;
                }
                if (!opened) {
                    ask_status(c);
                    // the first Arnoldi step's first transform is queued behind the
                    // status, gated on st.active (0 exactly when the solve has
                    // ended), so the GPU works while the host waits for the status
                    if (ahead) launch_precond<T>(g, c->p.precond, c->fast, V, scr, Z, act, c->s, FPC_HEAD);
                    HIPCHK(c, hipGetLastError());
                    CHK(pub_wait(c));
                    if (c->gm_h->outer_done) { final_res = true; break; }
                    head = ahead;
                }
                opened = false;
            }
            bool one_step = false;             // the cycle stopped after its first Arnoldi step
            const bool measure = norm_only(unit);
            for (int j = 0; j < kmax; j++) {
                T *vj = V + (long)j * ldv, *vj1 = V + (long)(j + 1) * ldv, *zj = Z + (long)j * ldv;
                if (!(j == 0 && have_z0)) {
                    Tscope ts(c, TBL_K_PRECOND, precond_bytes(c, sizeof(T)));
                    launch_precond<T>(g, c->p.precond, c->fast, vj, scr, zj, act, c->s,
                                      (head && j == 0) ? FPC_TAIL : FPC_ALL);
                }
                if (j == 0) head = false;
                if (j == 0 && fuse_dot) {
                    // first Arnoldi step: the Poisson apply also forms <A z_0, v_0>
                    unsigned nbp;
                    {
                        Tscope ts(c, TBL_K_POISSON, 3.0 * (double)N * sizeof(T));
                        nbp = launch_poisson<T>(g, zj, vj1, act, &c->gm->sigma[j], c->s, V, part_z);
                    }
                    launch_fin_dots(c->gm, part_z, (int)nbp, j, c->s);
                } else {
                    {
                        Tscope ts(c, TBL_K_POISSON, 2.0 * (double)N * sizeof(T));
                        launch_poisson<T>(g, zj, vj1, act, &c->gm->sigma[j], c->s);
                    }
                    {
                        Tscope ts(c, TBL_K_DOTS, (j + 2.0) * (double)N * sizeof(T));
                        launch_dots<T>(V, ldv, j, N, c->gm, part_z, c->s);
                    }
                    launch_fin_dots(c->gm, part_z, (int)nbv, j, c->s);
                }
                {
                    Tscope ts(c, TBL_K_UPDATE, (j + (measure && j == 0 ? 2.0 : 3.0)) * (double)N * sizeof(T));
                    launch_update<T>(V, ldv, j, N, c->gm, part_z, c->s, !(measure && j == 0));
                }
                launch_fin_update(c->gm, part_z, (int)nbv, j, c->s);
                HIPCHK(c, hipGetLastError());
                if ((j + 1) % poll == 0 && j + 1 < kmax) {
                    ask_status(c);
                    const bool qa = ahead_res && j == 0 && m + 1 < mmax;
                    if (qa) {
                        launch_fin_cycle(c->gm, c->s, 1);
                        launch_resid_upd<T>(g, c->pRhs, c->PCorr, Z, c->gm, c->PCalt, V, part_r, c->s, RU_GATED);
                    }
                    HIPCHK(c, hipGetLastError());
                    CHK(pub_wait(c));
                    if (!c->gm_h->active) {
                        one_step = (j == 0);
                        if (qa) {
                            std::swap(c->PCorr, c->PCalt);
                            queued = true;
                        }
                        break;
                    }
                    if (measure && j == 0) {
                        Tscope ts(c, TBL_K_UPDATE, 3.0 * (double)N * sizeof(T));
                        launch_update<T>(V, ldv, j, N, c->gm, part_z, c->s);
                    }
                }
            }
            if (!queued) {                     // (queued: fin_cycle and PCorr += y z0 have run)
                launch_fin_cycle(c->gm, c->s);
                if (fuse_upd && one_step) {
                    pend = true;
                } else {
                    Tscope ts(c, TBL_K_XUPD);
                    launch_xupd<T>(Z, ldv, N, c->gm, c->PCorr, c->s);
                }
            }
            HIPCHK(c, hipGetLastError());
            // no read-back here: the next cycle's residual decides (its
            // synchronised status read covers this cycle), and the cycle cap
            // is the loop bound
        }
        if (pend) {                            // the cycle cap ended the loop
            Tscope ts(c, TBL_K_XUPD);
            launch_xupd<T>(Z, ldv, N, c->gm, c->PCorr, c->s);
        }
        if (!final_res) {
            ask_status(c);
            HIPCHK(c, hipGetLastError());
            CHK(pub_wait(c));
        }
    }
    for (int m = 0; m < mmax && mode == GM_MODE_REF; m++) {
        {
            Tscope ts(c, TBL_K_RESID, (double)N * (16.0 + sizeof(T)));
            launch_resid<T>(g, c->pRhs, c->PCorr, r, part_r, c->s);
        }
        {
            Tscope ts(c, TBL_K_PRECOND, precond_bytes(c, sizeof(T)));
            launch_precond<T>(g, c->p.precond, c->fast, r, scr, V, nullptr, c->s);
        }
        launch_norm2<T>(V, N, part_z, nullptr, c->s);
        launch_fin_start(c->gm, part_r, (int)nbr, part_z, (int)nbv, m == 0 ? 1 : 0, c->s);
        HIPCHK(c, hipGetLastError());
        if (m == 0 && unit_steps) {
            // unit step (k_fin_unit): the preconditioned residual of PCorr + V_0
            // (into W; r holds the residual) ends the solve, or is dropped
            {
                Tscope ts(c, TBL_K_RESID, (double)N * (24.0 + 2.0 * sizeof(T)));
                launch_resid_upd<T>(g, c->pRhs, c->PCorr, V, c->gm, c->PCalt, r, part_r, c->s, RU_UNIT);
            }
            {
                Tscope ts(c, TBL_K_PRECOND, precond_bytes(c, sizeof(T)));
                launch_precond<T>(g, c->p.precond, c->fast, r, scr, W, act, c->s);
            }
            launch_norm2<T>(W, N, part_z, act, c->s);
            launch_fin_unit(c->gm, part_r, (int)nbr, part_z, (int)nbv, pub_of(c, c->gm_h), c->s);
            HIPCHK(c, hipGetLastError());
            CHK(pub_wait(c));
            if (c->gm_h->unit_ok) std::swap(c->PCorr, c->PCalt);
            if (c->gm_h->outer_done) { final_res = true; break; }
        }
        for (int j = 0; j < kmax; j++) {
            T *vj = V + (long)j * ldv, *vj1 = V + (long)(j + 1) * ldv;
            {
                Tscope ts(c, TBL_K_POISSON, 2.0 * (double)N * sizeof(T));
                launch_poisson<T>(g, vj, W, act, &c->gm->sigma[j], c->s);
            }
            {
                Tscope ts(c, TBL_K_PRECOND, precond_bytes(c, sizeof(T)));
                launch_precond<T>(g, c->p.precond, c->fast, W, scr, vj1, act, c->s);
            }
            {
                Tscope ts(c, TBL_K_DOTS, (j + 2.0) * (double)N * sizeof(T));
                launch_dots<T>(V, ldv, j, N, c->gm, part_z, c->s);
            }
            launch_fin_dots(c->gm, part_z, (int)nbv, j, c->s);
            {
                Tscope ts(c, TBL_K_UPDATE, (j + 3.0) * (double)N * sizeof(T));
                launch_update<T>(V, ldv, j, N, c->gm, part_z, c->s);
            }
            launch_fin_update(c->gm, part_z, (int)nbv, j, c->s);
            HIPCHK(c, hipGetLastError());
            if ((j + 1) % poll == 0 && j + 1 < kmax) {
                ask_status(c);
                HIPCHK(c, hipGetLastError());
                CHK(pub_wait(c));
                if (!c->gm_h->active) break;
            }
        }
        launch_fin_cycle(c->gm, c->s);
        {
            Tscope ts(c, TBL_K_XUPD);
            launch_xupd<T>(V, ldv, N, c->gm, c->PCorr, c->s);
        }
        ask_status(c);
        HIPCHK(c, hipGetLastError());
        CHK(pub_wait(c));
        if (c->gm_h->outer_done) break;
    }
    GmStatus st = *c->gm_h;
    if (st.nan) return fail(c, TBL_ENAN, "non-finite residual in the pressure solve");
    if (st.zero_rhs) {
        // ||pRhs|| = 0 (true-residual mode): A is nonsingular, so PCorr = 0
        launch_fill(c->PCorr, 0.0, N, c->s);
        HIPCHK(c, hipGetLastError());
        final_res = false;
    }
    // true residual after the solve (the reference reports none; logged here).
    // A flexible solve that stopped at a cycle start has just formed it from
    // the same kernel and partials.
    double tr = st.true_res;
    if (!final_res) {
        launch_resid<double>(g, c->pRhs, c->PCorr, nullptr, part_r, c->s);
        launch_fin_sum(part_r, (int)nbr, c->dd + DD_BNORM, c->s);
        CHK(read_diag(c));
        tr = sqrt(c->dh[DD_BNORM]);
    }
    if (cycles) *cycles = st.cycle;
    if (iters) *iters = st.total;
    if (true_res) *true_res = tr;
    c->gm_h->true_res = tr;
    if (!st.conv && c->p.fail_on_noconv) return fail(c, TBL_ENOCONV, "GMRES reached mmax");
    return 0;
}
extern "C" int tbl_ppe_solve(tbl_ctx *c, double errtol, int kmax, int mmax, int *cycles, int *iters, double *true_res)
{
    if (!c || kmax < 1 || mmax < 1) return TBL_EARG;
    return c->mixed ? gmres_impl<float>(c, errtol, kmax, mmax, cycles, iters, true_res)
                    : gmres_impl<double>(c, errtol, kmax, mmax, cycles, iters, true_res);
}

template <class T> static int project_impl(tbl_ctx *c)
{
    Tscope ts(c, TBL_K_PROJECT, (double)c->g.N * (8.0 + 8.0 * sizeof(T)));
    launch_project<T>(c->g, c->PCorr, F<T>(c->Press), F<T>(c->Ut), c->s);
    HIPCHK(c, hipGetLastError());
    return 0;
}
extern "C" int tbl_project(tbl_ctx *c)
{
    if (!c) return TBL_EARG;
    return c->mixed ? project_impl<float>(c) : project_impl<double>(c);
}

template <class T> static int bcs_impl(tbl_ctx *c)
{
    // the boundary faces of the three velocity components and the pressure,
    // read and written
    const double faces = 2.0 * ((double)c->g.nX * c->g.nY + (double)c->g.nY * c->g.nZ + (double)c->g.nX * c->g.nZ);
    Tscope ts(c, TBL_K_BCS, 8.0 * faces * sizeof(T));
    launch_bcs<T>(c->g, F<T>(c->Ut), F<T>(c->Utold), F<T>(c->Press), c->have_wall_w ? c->wall_w : nullptr, c->s);
    HIPCHK(c, hipGetLastError());
    return 0;
}
extern "C" int tbl_apply_bcs(tbl_ctx *c)
{
    if (!c) return TBL_EARG;
    return c->mixed ? bcs_impl<float>(c) : bcs_impl<double>(c);
}

// block partials of the divergence sum and of the mass fluxes; launch_fin_diag
// (fin_diag) finishes them into the diagnostics record
template <class T> static int div_impl(tbl_ctx *c)
{
    Tscope ts(c, TBL_K_DIAG, 3.0 * (double)c->g.N * sizeof(T));      // the three velocity components
    launch_div_check<T>(c->g, F<T>(c->Ut), c->part, c->s);
    HIPCHK(c, hipGetLastError());
    return 0;
}
static int fin_diag(tbl_ctx *c, bool div, bool mass, bool pub)
{
    launch_fin_diag(c->part, div ? (int)resid_blocks(c->g) : 0, mass ? c->dd + DD_NCOUNT : nullptr, c->mass_denom, c->dd,
                    pub ? pub_of(c, c->dh) : Pub(), c->s);
    HIPCHK(c, hipGetLastError());
    return 0;
}
static double div_metric(const tbl_ctx *c, double s)
{
    const tbl_params &p = c->p;
    return fabs(s) / ((p.nY - 2) * (p.nX - 2) * (p.nZ - 2));
}
extern "C" int tbl_div_check(tbl_ctx *c, double *div, double *signed_sum)
{
    if (!c) return TBL_EARG;
    CHK(c->mixed ? div_impl<float>(c) : div_impl<double>(c));
    CHK(fin_diag(c, true, false, true));
    CHK(pub_wait(c));
    const double s = c->dh[DD_DIV];
    if (signed_sum) *signed_sum = s;
    if (div) *div = div_metric(c, s);
    return 0;
}

// tbl_div_check on caller-owned device memory with the block partials in the
// static scratch: no allocation, no host synchronisation
extern "C" int tbl_div_check_noalloc(tbl_ctx *c, const void *Ut_dev, double *out_dev)
{
    if (!c) return TBL_EARG;
    if (!Ut_dev || !out_dev) return fail(c, TBL_EARG, "tbl_div_check_noalloc: NULL device pointer");
    if (!c->noalloc) return fail(c, TBL_ESTATE, "tbl_div_check_noalloc: static scratch not set up");
    const unsigned nb = resid_blocks(c->g);
    if (nb > TBL_NOALLOC_PARTS) {
        char m[160];
        snprintf(m, sizeof(m), "tbl_div_check_noalloc: this grid needs %u partials, the static scratch holds %d",
                 nb, TBL_NOALLOC_PARTS);
        return fail(c, TBL_EARG, m);
    }
    const tbl_params &p = c->p;
    const double nint = (double)((p.nY - 2) * (p.nX - 2) * (p.nZ - 2));
    if (c->mixed) launch_div_check<float>(c->g, (const float *)Ut_dev, c->noalloc, c->s);
    else launch_div_check<double>(c->g, (const double *)Ut_dev, c->noalloc, c->s);
    launch_fin_div(c->noalloc, (int)nb, nint, out_dev, c->s);
    HIPCHK(c, hipGetLastError());
    return 0;
}

template <class T> static int mass_impl(tbl_ctx *c)
{
    Tscope ts(c, TBL_K_DIAG, 5.0 * (double)c->g.nY * c->g.nZ * sizeof(T));   // u on the five planes
    launch_mass_flux<T>(c->g, F<T>(c->Ut), c->p.planes, c->dd + DD_NCOUNT, c->s);
    HIPCHK(c, hipGetLastError());
    return 0;
}
extern "C" int tbl_mass_flux(tbl_ctx *c, double *mass5)
{
    if (!c) return TBL_EARG;
    CHK(c->mixed ? mass_impl<float>(c) : mass_impl<double>(c));
    CHK(fin_diag(c, false, true, mass5 != nullptr));
    if (mass5) {
        CHK(pub_wait(c));
        memcpy(mass5, c->dh + DD_MASS, 5 * sizeof(double));
    }
    return 0;
}

template <class T> static int stats_impl(tbl_ctx *c)
{
    // the velocity, and the nine (nX, nZ) sums read and written
    Tscope ts(c, TBL_K_DIAG, 3.0 * (double)c->g.N * sizeof(T) + 18.0 * (double)c->g.nX * c->g.nZ * 8.0);
    launch_stats<T>(c->g, F<T>(c->Ut), c->sums, c->s);
    HIPCHK(c, hipGetLastError());
    return 0;
}
extern "C" int tbl_stats_accumulate(tbl_ctx *c)
{
    if (!c) return TBL_EARG;
    return c->mixed ? stats_impl<float>(c) : stats_impl<double>(c);
}

template <class T> static int rescale_impl(tbl_ctx *c)
{
    Tscope ts(c, TBL_K_RESCALE);
    launch_rescale<T>(c->g, c->p.i_rec - 1, c->p.freq_tim_avg, F<T>(c->Ut), c->sums, c->avg, c->rec, c->Wt,
                      c->newk, c->bltkns, c->dstar, c->theta, c->uf, c->scan, c->s);
    HIPCHK(c, hipGetLastError());
    return 0;
}
extern "C" int tbl_rescale(tbl_ctx *c)
{
    if (!c) return TBL_EARG;
    return c->mixed ? rescale_impl<float>(c) : rescale_impl<double>(c);
}

template <class T> static int ke_impl(tbl_ctx *c)
{
    Tscope ts(c, TBL_K_DIAG, 3.0 * (double)c->g.N * sizeof(T));      // the velocity against the means
    launch_ke<T>(c->g, c->p.i_rec - 1, F<T>(c->Ut), c->avg, c->part, c->guard, c->uf, c->s);
    launch_fin_sum(c->part, (int)resid_blocks(c->g), c->dd + DD_KE, c->s);
    HIPCHK(c, hipGetLastError());
    return 0;
}
extern "C" int tbl_ke_guard(tbl_ctx *c, double *ke, int *guard)
{
    if (!c) return TBL_EARG;
    HIPCHK(c, hipMemsetAsync(c->guard, 0, sizeof(int), c->s));
    CHK(c->mixed ? ke_impl<float>(c) : ke_impl<double>(c));
    CHK(read_diag(c));
    const tbl_params &p = c->p;
    if (ke) *ke = c->dh[DD_KE] / (double)(p.nX * (p.nY - 2) * (p.nZ - 2));
    if (guard) memcpy(guard, c->dh + DD_GUARD, sizeof(int));
    return 0;
}

template <class T> static int tau_impl(tbl_ctx *c, double *acc = nullptr)
{
    Tscope ts(c, TBL_K_DIAG, 3.0 * (double)c->g.sZ * sizeof(T));     // u on the three wall planes
    launch_wall_shear<T>(c->g, F<T>(c->Ut), c->tau, c->s, acc);
    HIPCHK(c, hipGetLastError());
    return 0;
}
extern "C" int tbl_wall_shear(tbl_ctx *c, double *tau)
{
    if (!c) return TBL_EARG;
    CHK(c->mixed ? tau_impl<float>(c) : tau_impl<double>(c));
    if (tau) {
        CHK(d2h(c, tau, c->tau, c->p.nX * sizeof(double)));
        HIPCHK(c, hipStreamSynchronize(c->s));
    }
    return 0;
}

extern "C" int tbl_wall_shear_mean(tbl_ctx *c, double *tau_mean, double *cf, int *nwindows)
{
    if (!c) return TBL_EARG;
    if (c->p.wall_shear_window <= 0) return fail(c, TBL_ESTATE, "tbl_wall_shear_mean: wall_shear_window is 0 (off)");
    if (tau_mean) CHK(d2h(c, tau_mean, c->taumean, c->p.nX * sizeof(double)));
    if (cf) CHK(d2h(c, cf, c->cf, c->p.nX * sizeof(double)));
    HIPCHK(c, hipStreamSynchronize(c->s));
    if (nwindows) *nwindows = c->nwin;
    return 0;
}

// ------------------------------------------------------------------ whole step
extern "C" int tbl_step(tbl_ctx *c, int nsteps, tbl_diag *diag)
{
    if (!c || nsteps < 0) return TBL_EARG;
    const tbl_params &p = c->p;
    for (int n = 0; n < nsteps; n++) {
        tbl_diag d;
        memset(&d, 0, sizeof(d));
        bool ppe_done = false;                 // the diffusion solve queued the PPE right-hand side
        CHK(tbl_begin_step(c));
        CHK(tbl_recycle_inflow(c));
        if (p.helm_mode != TBL_HELM_DIRECT) {
            // the momentum kernel also forms the Gauss-Seidel solve's first
            // residual pass (same values, one read of the fields)
            const int nb = (int)rhs_blocks(c->g, c->mixed);
            CHK(c->mixed ? rhs_impl<float>(c, c->part) : rhs_impl<double>(c, c->part));
            HIPCHK(c, hipGetLastError());
            CHK(c->mixed ? helm_impl<float>(c, p.errorstop, p.gs_mmax, d.gs_sweeps, nullptr, nb, &ppe_done)
                         : helm_impl<double>(c, p.errorstop, p.gs_mmax, d.gs_sweeps, nullptr, nb, &ppe_done));
        } else {
            CHK(tbl_momentum_rhs(c));
            CHK(tbl_diffusion_solve(c, p.errorstop, p.gs_mmax, d.gs_sweeps, nullptr));
        }
        if (!ppe_done) CHK(tbl_ppe_rhs(c));
        CHK(tbl_ppe_solve(c, p.errtol, p.kmax, p.mmax, &d.gm_cycles, &d.gm_iters, &d.gm_true_res));
        d.gm_sumav = c->gm_h->sumav;
        CHK(tbl_project(c));
        CHK(tbl_apply_bcs(c));
        CHK(c->mixed ? div_impl<float>(c) : div_impl<double>(c));
        CHK(c->mixed ? mass_impl<float>(c) : mass_impl<double>(c));
        if (p.wall_shear_window > 0) {
            // a17 window: tau of every step into the running sum; mean and C_f
            // at the window's last step (dnstbl/dnstbl.f90:1666-1682)
            CHK(c->mixed ? tau_impl<float>(c, c->tausum) : tau_impl<double>(c, c->tausum));
            if (c->nstep % p.wall_shear_window == 0) {
                Tscope ts(c, TBL_K_DIAG);
                launch_tau_window(c->g, p.wall_shear_window, c->tausum, c->taumean, c->cf, c->s);
                HIPCHK(c, hipGetLastError());
                c->nwin += 1;
                d.cf_ready = 1;
            }
        }
        CHK(tbl_stats_accumulate(c));
        if (c->nstep % p.freq_tim_avg == 0) {
            CHK(tbl_rescale(c));
            d.rescaled = 1;
        }
        // the kinetic energy reuses the divergence's partials, so they are
        // finished before it; otherwise the finishing kernel is the step's last
        const bool ke_on = c->cnt > p.freq_tim_avg;
        CHK(fin_diag(c, true, true, !ke_on));
        int gd = 0;
        if (ke_on) {
            HIPCHK(c, hipMemsetAsync(c->guard, 0, sizeof(int), c->s));
            CHK(c->mixed ? ke_impl<float>(c) : ke_impl<double>(c));
            CHK(read_diag(c));
            memcpy(&gd, c->dh + DD_GUARD, sizeof(int));
        } else {
            CHK(pub_wait(c));
        }
        d.div_signed = c->dh[DD_DIV];
        d.div = div_metric(c, d.div_signed);
        for (int q = 0; q < 5; q++) d.mass[q] = c->dh[DD_MASS + q];
        d.ke = ke_on ? c->dh[DD_KE] / (double)(p.nX * (p.nY - 2) * (p.nZ - 2)) : 0.0;
        d.guard = gd;
        d.nstep = c->nstep;
        if (diag) diag[n] = d;
        // the guard is a bit set (1: fluctuation > 25, 2: non-finite), both
        // bits may be set by different nodes
        if ((gd & 2) || !(d.div_signed == d.div_signed)) return fail(c, TBL_ENAN, "non-finite field");
        if (gd & 1) return fail(c, TBL_EBLOWUP, "very large fluctuations (> 25)");
    }
    return 0;
}

// ------------------------------------------------------------------ discrete adjoint
// Work buffers of one adjoint window, one allocation a call: the adjoint fields,
// cleared, then the snapshots, which are stored before they are read.  A forward
// evaluation needs none.  An allocation and a clear for each of ten buffers, the
// snapshots' included, and the start state stored for a forward evaluation too,
// took 0.1 of the 1.25 ms of a forward call at 64x32x48, 1.3 of the 35.4 ms of a
// gradient at 256x64x96 and 2.1 of the 69.0 ms at 1024x192x160 mixed; two
// allocations, 0.3 of the 6.7 ms at 303x62x105 mixed.  Where there is no memory
// for both, the snapshots are taken alone and the fields after the forward sweep,
// so that J is there if the call fails for them.
struct AdjWin {
    char *mem = nullptr, *own = nullptr; // own: the snapshots, if they are an allocation of their own
    double *lamU = nullptr, *lamP = nullptr, *lamQ = nullptr, *lamPhi = nullptr, *lamB = nullptr;
    double *grad = nullptr;
    double *E = nullptr, *Enew = nullptr;   // end-of-step boundary values (launch_adj_save_end): of this step, of the one before
    double *Jd = nullptr;
    char *snapbuf = nullptr;             // nslots states: Ut, Press in the storage type, PCorr in double
    size_t slot_bytes = 0;
    int nslots = 0;
    std::vector<int> sn, sc;
    std::vector<double> st;
    int i0 = 0, i1 = 0;
    double cJ = 0.0;
    int nfwd = 0, nadj = 0;
    int nstep0 = 0;
    int brmode = 0;          // 1 record the Peclet switches, 2 replay them (first sweep only)
};
// bytes of the adjoint fields, each from a multiple of 256; with mem, set up there
static size_t adj_fields(tbl_ctx *c, AdjWin &A, char *mem)
{
    const size_t N = (size_t)c->g.N, ne = (size_t)adj_end_len(c->g), nw = (size_t)c->p.nX * c->p.nY;
    struct { double **p; size_t n; } sub[] = {{&A.lamU, 3 * N}, {&A.lamP, N}, {&A.lamQ, 3 * N}, {&A.lamPhi, N},
                                              {&A.lamB, N}, {&A.E, ne}, {&A.Enew, ne}, {&A.grad, nw}};
    size_t at = 0;
    for (auto &f : sub) {
        if (mem) *f.p = (double *)(mem + at);
        at += (f.n * 8 + 255) & ~(size_t)255;
    }
    return at;
}
// the snapshots, and the adjoint fields if both find room
static int adj_alloc(tbl_ctx *c, AdjWin &A)
{
    const size_t snaps = (size_t)A.nslots * A.slot_bytes, fields = adj_fields(c, A, nullptr);
    if (hipMalloc((void **)&A.mem, fields + snaps) == hipSuccess) {
        adj_fields(c, A, A.mem);
        A.snapbuf = A.mem + fields;
        HIPCHK(c, hipMemsetAsync(A.mem, 0, fields, c->s));
        return 0;
    }
    (void)hipGetLastError();
    A.mem = nullptr;
    HIPCHK(c, hipMalloc((void **)&A.own, snaps));
    A.snapbuf = A.own;
    return 0;
}
// the adjoint fields, if they are not there yet
static int adj_alloc_fields(tbl_ctx *c, AdjWin &A)
{
    if (A.mem) return 0;
    const size_t fields = adj_fields(c, A, nullptr);
    HIPCHK(c, hipMalloc((void **)&A.mem, fields));
    adj_fields(c, A, A.mem);
    HIPCHK(c, hipMemsetAsync(A.mem, 0, fields, c->s));
    return 0;
}
// snapshot = Ut (3N), Press (N) in the storage type, PCorr (N, double) and
// the step counters
static int snap_store(tbl_ctx *c, AdjWin &A, int slot)
{
    const size_t N = (size_t)c->g.N, es = c->es;
    char *b = A.snapbuf + (size_t)slot * A.slot_bytes;
    HIPCHK(c, hipMemcpyAsync(b, c->Ut, 3 * N * es, hipMemcpyDeviceToDevice, c->s));
    HIPCHK(c, hipMemcpyAsync(b + 3 * N * es, c->Press, N * es, hipMemcpyDeviceToDevice, c->s));
    HIPCHK(c, hipMemcpyAsync(b + 4 * N * es, c->PCorr, N * 8, hipMemcpyDeviceToDevice, c->s));
    A.sn[slot] = c->nstep;
    A.sc[slot] = c->cnt;
    A.st[slot] = c->time;
    return 0;
}
static int snap_restore(tbl_ctx *c, AdjWin &A, int slot)
{
    const size_t N = (size_t)c->g.N, es = c->es;
    const char *b = A.snapbuf + (size_t)slot * A.slot_bytes;
    HIPCHK(c, hipMemcpyAsync(c->Ut, b, 3 * N * es, hipMemcpyDeviceToDevice, c->s));
    HIPCHK(c, hipMemcpyAsync(c->Press, b + 3 * N * es, N * es, hipMemcpyDeviceToDevice, c->s));
    HIPCHK(c, hipMemcpyAsync(c->PCorr, b + 4 * N * es, N * 8, hipMemcpyDeviceToDevice, c->s));
    c->nstep = A.sn[slot];
    c->cnt = A.sc[slot];
    c->time = A.st[slot];
    c->pc_hist = 0;
    return 0;
}
// exact pressure solve: PCorr += A^{-1} (pRhs - A PCorr), twice; in a mixed
// context with the residual formed in double and the inverse applied by the
// FP32 fast solver (iterative refinement: each pass gains about the FP32
// solver's accuracy, 1e-6, so two passes leave ~1e-12)
template <class T> static int ppe_direct(tbl_ctx *c)
{
    const Geo &g = c->g;
    T *r = F<T>(c->r);                         // its faces stay zero
    FastIO io;
    io.in = r;
    io.out = c->PCorr;
    io.in64 = sizeof(T) == sizeof(double);
    io.out64 = io.add = 1;
    launch_zero_faces<double>(g, c->PCorr, c->s);
    const int passes = 2;
    for (int it = 0; it < passes; it++) {
        launch_resid<T>(g, c->pRhs, c->PCorr, r, c->part, c->s);
        if (run_fast_solve(c->fast, g, io, nullptr, 0.0, 1.0, false, c->s))
            return fail(c, TBL_EARG, "fast solver failure in the direct pressure solve");
    }
    HIPCHK(c, hipGetLastError());
    return 0;
}
// one step of the window: the reference's step with exact solves, no statistics
static int win_step(tbl_ctx *c, AdjWin &A, bool accJ)
{
    CHK(tbl_begin_step(c));
    CHK(tbl_recycle_inflow(c));
    if (accJ && A.brmode) {
        unsigned char *b = c->br + (size_t)(c->nstep - A.nstep0 - 1) * (size_t)c->g.N;
        if (A.brmode == 1) c->br_out = b;
        else c->br_in = b;
    }
    const int rc = tbl_momentum_rhs(c);
    c->br_in = nullptr;
    c->br_out = nullptr;
    CHK(rc);
    CHK(c->mixed ? helm_direct<float>(c, nullptr, nullptr) : helm_direct<double>(c, nullptr, nullptr));
    CHK(tbl_ppe_rhs(c));
    CHK(c->mixed ? ppe_direct<float>(c) : ppe_direct<double>(c));
    CHK(tbl_project(c));
    CHK(tbl_apply_bcs(c));
    if (accJ) {
        if (c->mixed) launch_wall_shear<float>(c->g, (const float *)c->Ut, c->tau, c->s);
        else launch_wall_shear<double>(c->g, (const double *)c->Ut, c->tau, c->s);
        launch_tau_acc(c->g, c->tau, A.i0, A.i1, A.cJ, A.Jd, c->s);
    }
    HIPCHK(c, hipGetLastError());
    A.nfwd++;
    return 0;
}
// x = (alpha I + beta A)^{-T} b on the interior planes, by iterative
// refinement in FP64: x = M^{-T} b, then x += M^{-T} (b - (alpha I + beta A)^T x),
// M^{-T} the transposed fast solve.  FP64 contexts: the FP64 fast solver,
// two passes.  Mixed contexts: the FP32 fast solver on the FP64 residual
// rounded to FP32, also two passes (each gains about the FP32 solver's
// accuracy, 1e-6), x and the residual accumulated in FP64.  Values of b off
// the interior are not read; x is written on planes 1..nZ-2 (zero on their
// face rows).  The transforms read b and write and correct x in FP64
// themselves: copies of b without its faces and in FP32, and the passes that
// widened and added the result, moved 60 bytes a cell more.
static int solve_T(tbl_ctx *c, const double *b, double *x, double alpha, double beta, int ncomp)
{
    const Geo &g = c->g;
    const int nc = ncomp == 3 ? direct_batch(c) : 1;
    void *r = nc == 3 ? c->r3 : c->r;
    for (int p = 0; p < ncomp; p += nc) {
        const double *bp = b + (long)p * g.N;
        double *xp = x + (long)p * g.N;
        FastIO io;
        io.in = bp;
        io.out = xp;
        io.in64 = io.out64 = io.mask = 1;
        io.ncomp = nc;
        if (run_fast_solve(c->fast, g, io, nullptr, alpha, beta, true, c->s)) return fail(c, TBL_EARG, "fast solver failure");
        if (c->mixed) launch_opT_res<float>(g, bp, xp, alpha, beta, F<float>(r), nc, c->s);
        else launch_opT_res<double>(g, bp, xp, alpha, beta, F<double>(r), nc, c->s);
        io.in = r;
        io.in64 = !c->mixed;
        io.mask = 0;
        io.add = 1;
        if (run_fast_solve(c->fast, g, io, nullptr, alpha, beta, true, c->s)) return fail(c, TBL_EARG, "fast solver failure");
    }
    return 0;
}
// adjoint of step n: on entry the fields hold the state after step n-1,
// A.E the boundary values of the velocity after step n, A.lamU / A.lamP the
// adjoint of the state after step n; on exit they hold the adjoint of the
// state after step n-1 (including dJ_{n-1}/dU) and A.E the boundary values of
// the velocity after step n-1.
// In a mixed context the states are FP32; the adjoint kernels convert what
// they read to double, so the adjoint is accumulated in FP64 about the
// mixed-precision trajectory.
static int adj_step(tbl_ctx *c, AdjWin &A, int n)
{
    const Geo &g = c->g;
    const size_t N = (size_t)g.N;
    const double h = c->p.dt / c->p.Re;
    if (c->mixed) launch_adj_save_end<float>(g, F<float>(c->Ut), A.Enew, c->s);
    else launch_adj_save_end<double>(g, F<double>(c->Ut), A.Enew, c->s);
    CHK(tbl_begin_step(c));
    CHK(tbl_recycle_inflow(c));               // linearisation point of the convection
    launch_adj_bcs(g, A.E, A.lamU, A.lamP, A.grad, c->s);
    launch_adj_proj(g, A.lamU, A.lamP, A.lamPhi, c->s);
    CHK(solve_T(c, A.lamPhi, A.lamB, 0.0, 1.0, 1));
    launch_adj_div(g, A.lamB, A.lamU, c->s);
    CHK(solve_T(c, A.lamU, A.lamQ, 1.0, -h, 3));
    if (c->mixed) launch_adj_mom<float>(g, F<float>(c->Ut), A.lamQ, A.lamU, A.lamP, c->s);
    else launch_adj_mom<double>(g, F<double>(c->Ut), A.lamQ, A.lamU, A.lamP, c->s);
    std::swap(A.E, A.Enew);
    if (n - 1 >= 1) launch_adj_tau(g, A.lamU, A.i0, A.i1, A.cJ, c->s);
    HIPCHK(c, hipGetLastError());
    A.nadj++;
    return 0;
}
static long long binom_capped(int n, int k)
{
    long long r = 1;
    for (int q = 1; q <= k; q++) {
        r = r * (n - k + q) / q;
        if (r > (1LL << 40)) return 1LL << 40;
    }
    return r;
}
// reverse steps a+1..b; the state after step a is in snapshot slot_a and
// `free` further slots (slot_a+1 ...) may be used.  Checkpoint placement of
// the binomial schedule: with r the least repetition number such that
// C(free + r, free) >= b - a, the segment after the new checkpoint m is
// reversible with free-1 snapshots at repetition r.
static int revolve_split(int a, int b, int free)
{
    const int L = b - a;
    int r = 0;
    while (binom_capped(free + r, free) < L) r++;
    const long long bl = binom_capped(free - 1 + r, free - 1);
    int m = b - (int)(bl < (long long)(L - 1) ? bl : (long long)(L - 1));
    return m <= a ? a + 1 : m;
}
static int revolve(tbl_ctx *c, AdjWin &A, int a, int b, int slot_a, int free)
{
    if (b - a == 1) {
        CHK(snap_restore(c, A, slot_a));
        return adj_step(c, A, b);
    }
    if (free == 0) {
        for (int n = b; n > a; n--) {
            CHK(snap_restore(c, A, slot_a));
            for (int m = a + 1; m <= n - 1; m++) CHK(win_step(c, A, false));
            CHK(adj_step(c, A, n));
        }
        return 0;
    }
    const int m = revolve_split(a, b, free);
    CHK(snap_restore(c, A, slot_a));
    for (int k = a + 1; k <= m; k++) CHK(win_step(c, A, false));
    CHK(snap_store(c, A, slot_a + 1));
    CHK(revolve(c, A, m, b, slot_a + 1, free - 1));
    return revolve(c, A, a, m, slot_a, free);
}
// The schedule's first descent (restore a, step to m, store, recurse on
// (m, b)) runs the same steps as the window's J sweep: the sweep stores those
// checkpoints as it passes them (first_descent), and the reverse sweep starts
// here, skipping the forward steps of that descent.
static void first_descent(int n, int nsnap, std::vector<int> &at)
{
    at.assign(n + 1, -1);                      // at[state index] = slot, or -1
    int a = 0, slot = 0, free = nsnap;
    while (n - a > 1 && free > 0) {
        const int m = revolve_split(a, n, free);
        at[m] = slot + 1;
        a = m;
        slot++;
        free--;
    }
}
static int revolve_top(tbl_ctx *c, AdjWin &A, int a, int b, int slot_a, int free)
{
    if (b - a == 1 || free == 0) return revolve(c, A, a, b, slot_a, free);
    const int m = revolve_split(a, b, free);   // stored in slot_a + 1 by the J sweep
    CHK(revolve_top(c, A, m, b, slot_a + 1, free - 1));
    return revolve(c, A, a, m, slot_a, free);
}

extern "C" int tbl_adjoint_window(tbl_ctx *c, const tbl_adjoint_opts *o, const double *wall_w, double *J, double *dJdw,
                                  int *nfwd, int *nadj)
{
    if (!c || !o) return TBL_EARG;
    const tbl_params &p = c->p;
    if (p.scheme != TBL_SCHEME_SETBL || p.forc[0] != 0.0 || p.forc[1] != 0.0 || p.forc[2] != 0.0)
        return fail(c, TBL_EARG, "the adjoint window differentiates the dnssetbl convection scheme without forcing");
    if (!c->uploaded) return fail(c, TBL_ESTATE, "tbl_adjoint_window before tbl_upload");
    if (o->nsteps < 1 || o->nsnap < 1 || o->i0 < 2 || o->i1 < o->i0 || o->i1 > p.nX - 1)
        return fail(c, TBL_EARG, "invalid adjoint window options");
    for (int n = c->nstep + 1; n <= c->nstep + o->nsteps; n++)
        if (n % p.freq_tim_avg == 0) return fail(c, TBL_EARG, "the adjoint window crosses a statistics rescale");
    if (!c->fast) {
        char msg[256];
        HIPCHK(c, hipStreamSynchronize(c->s));
        if (fastpc_create(c->g, c->Ab.data(), c->At.data(), c->Ap.data(), c->s, c->mixed, &c->fast, msg, sizeof(msg)))
            return fail(c, TBL_EARG, msg);
    }
    if (wall_w) {
        CHK(h2d(c, c->wall_w, wall_w, (size_t)p.nX * p.nY * 8));
        c->have_wall_w = true;
    }
    const size_t N = (size_t)c->g.N;
    AdjWin A;
    A.nstep0 = c->nstep;
    A.brmode = o->branch_mode;
    if (o->branch_mode == 1) {
        if (c->br_steps < o->nsteps) {
            if (c->br) hipFree(c->br);
            c->br = nullptr;
            c->bytes -= (size_t)c->br_steps * N;
            c->br_steps = 0;
            CHK(dalloc(c, &c->br, (size_t)o->nsteps * N));
            c->br_steps = o->nsteps;
        }
        c->br_nstep0 = c->nstep;
    } else if (o->branch_mode == 2) {
        if (!c->br || c->br_nstep0 != c->nstep || c->br_steps < o->nsteps)
            return fail(c, TBL_ESTATE, "no recorded Peclet-switch pattern for this window");
        if (!o->forward_only) return fail(c, TBL_EARG, "a replayed switch pattern is for forward evaluations only");
    } else if (o->branch_mode != 0) {
        return fail(c, TBL_EARG, "invalid branch_mode");
    }
    A.i0 = o->i0 - 1;
    A.i1 = o->i1 - 1;
    A.cJ = 1.0 / ((double)o->nsteps * (double)(o->i1 - o->i0 + 1) * (double)(p.nY - 2));
    A.nslots = o->forward_only ? 0 : o->nsnap + 2;       // start, checkpoints, final state
    A.sn.assign(A.nslots, 0);
    A.sc.assign(A.nslots, 0);
    A.st.assign(A.nslots, 0.0);
    int rc = 0;
    auto run = [&]() -> int {
        A.Jd = c->dd + DD_J;
        HIPCHK(c, hipMemsetAsync(A.Jd, 0, 8, c->s));
        A.slot_bytes = (4 * N * c->es + N * 8 + 255) & ~(size_t)255;
        if (!o->forward_only) {
            CHK(adj_alloc(c, A));
            CHK(snap_store(c, A, 0));
        }
        std::vector<int> at;
        if (!o->forward_only) first_descent(o->nsteps, o->nsnap, at);
        for (int n = 1; n <= o->nsteps; n++) {
            CHK(win_step(c, A, true));
            if (!o->forward_only && at[n] >= 0) CHK(snap_store(c, A, at[n]));
        }
        double Jh = 0.0;
        CHK(d2h(c, &Jh, A.Jd, 8));
        HIPCHK(c, hipStreamSynchronize(c->s));
        if (J) *J = Jh;
        if (o->forward_only) return 0;
        const int fin = A.nslots - 1;
        CHK(snap_store(c, A, fin));
        CHK(adj_alloc_fields(c, A));
        if (c->mixed) launch_adj_save_end<float>(c->g, F<float>(c->Ut), A.E, c->s);
        else launch_adj_save_end<double>(c->g, F<double>(c->Ut), A.E, c->s);
        launch_adj_tau(c->g, A.lamU, A.i0, A.i1, A.cJ, c->s);
        CHK(revolve_top(c, A, 0, o->nsteps, 0, o->nsnap));
        CHK(snap_restore(c, A, fin));
        if (dJdw) CHK(d2h(c, dJdw, A.grad, (size_t)p.nX * p.nY * 8));
        HIPCHK(c, hipStreamSynchronize(c->s));
        return 0;
    };
    rc = run();
    if (nfwd) *nfwd = A.nfwd;
    if (nadj) *nadj = A.nadj;
    hipStreamSynchronize(c->s);
    if (A.mem) hipFree(A.mem);
    if (A.own) hipFree(A.own);
    return rc;
}

// ------------------------------------------------------------------ operator hooks
template <class T> static int op_impl(tbl_ctx *c, int op, const double *in, double *out)
{
    const size_t N = (size_t)c->g.N;
    T *x = F<T>(c->r), *y = F<T>(c->V);   // V slot 0 doubles as the output
    CHK(put_field(c, x, !c->mixed, in, N));
    // the Krylov work buffers keep zero faces (the separable preconditioner's
    // wall-normal transform carries face rows through): drop the input's faces;
    // the Poisson apply reads them as its Dirichlet values, so apply it first
    if (op == 0) {
        HIPCHK(c, hipMemsetAsync(y, 0, N * c->es, c->s));
        launch_poisson<T>(c->g, x, y, nullptr, nullptr, c->s);
        launch_zero_faces<T>(c->g, x, c->s);
        HIPCHK(c, hipGetLastError());
        CHK(get_field(c, y, !c->mixed, out, N));
        return 0;
    }
    launch_zero_faces<T>(c->g, x, c->s);
    HIPCHK(c, hipMemsetAsync(y, 0, N * c->es, c->s));
    launch_precond<T>(c->g, c->p.precond, c->fast, x, F<T>(c->scr), y, nullptr, c->s);
    HIPCHK(c, hipGetLastError());
    CHK(get_field(c, y, !c->mixed, out, N));
    return 0;
}
extern "C" int tbl_apply_operator(tbl_ctx *c, int op, const double *in, double *out)
{
    if (!c || !in || !out || op < 0 || op > 1) return TBL_EARG;
    return c->mixed ? op_impl<float>(c, op, in, out) : op_impl<double>(c, op, in, out);
}

// ------------------------------------------------------------------ timers
extern "C" int tbl_timer_enable(tbl_ctx *c, unsigned mask)
{
    if (!c) return TBL_EARG;
    timer_flush(c);
    c->tmask = mask;
    return 0;
}
extern "C" int tbl_timer_read(tbl_ctx *c, int *count, double *ms, double *bytes)
{
    if (!c) return TBL_EARG;
    timer_flush(c);
    for (int q = 0; q < TBL_K_NCLASS; q++) {
        if (count) count[q] = c->tcount[q];
        if (ms) ms[q] = c->tms[q];
        if (bytes) bytes[q] = c->tbytes[q];
        c->tcount[q] = 0;
        c->tms[q] = 0.0;
        c->tbytes[q] = 0.0;
    }
    return 0;
}
