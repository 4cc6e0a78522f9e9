// Multigrid-preconditioned CG for the served unit-square families (Poisson
// P1 / P2, elasticity P1 with a per-cell coefficient, homogeneous Dirichlet
// data on the whole boundary, penalized fixed rows as in the reference's
// solve_direct!, src/solvers.jl:647-652).
//
// The reference solves these systems with a sparse factorization or an
// unpreconditioned Krylov method (src/solvers.jl:38-59, 622-660); the
// solution it defines is the FP64 solution of the penalized system, which this
// solver reaches to the requested relative residual.  The preconditioner is
// this library's own: one V-cycle of a geometric hierarchy
//   level 0      the request's own matrix (P1, P2 or P1 x 2 on N x N),
//   [level 1     P1 on the same mesh, when level 0 is P2],
//   then         P1 on ceil(N_l / 2) x ceil(N_l / 2), down to N_l <= 4,
// each coarse matrix assembled by the same row-owner kernels from a
// coefficient coarsened by the geometric mean of the fine cells whose
// centroid lies in the coarse cell.  Transfers are linear interpolation on the
// coarse triangulation (nested or not) and its exact transpose, both written
// as gathers so that every sum has a fixed order; fixed dofs receive no
// correction and carry no residual.  Smoothing is Chebyshev of degree 2 on
// D^-1 A with lmax the Gershgorin bound of D^-1 A: of the first kind over
// [lmax/8, lmax], or of the fourth kind on hierarchies of one P1 component
// under CG (MgCheb).  The coarsest level is solved exactly with its dense
// inverse.  Pre- and post-smoothing are the same polynomial, so the V-cycle is
// symmetric and CG applies.  All scalars live on the device; the host only polls a status
// copy.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include <hip/hip_ext.h>

#include "grmp_internal.h"
#include "grmp_rowset.h"
#include "grmp_sparse.h"
#include "grmp_square.h"

static inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

// Start / stop events of a profiled launch come from a pool that collecting
// refills, so hipEventCreate runs only while the pool grows; every creation
// is checked, and a launch whose pair cannot be created runs unprofiled.
static bool ev_take(std::vector<hipEvent_t> &pool, hipEvent_t &e0, hipEvent_t &e1)
{
    e0 = e1 = nullptr;
    while (pool.size() < 2) {
        hipEvent_t e = nullptr;
        if (hipEventCreate(&e) != hipSuccess || e == nullptr) return false;
        pool.push_back(e);
    }
    e1 = pool.back();
    pool.pop_back();
    e0 = pool.back();
    pool.pop_back();
    return true;
}

#define MG_MAX_LEVELS 16
#define MG_DENSE_MAX 64  // dofs of the coarsest level (P1 x 2 on 4 x 4: 50)

// The smoother is a degree-2 Chebyshev polynomial of D^-1 A,
//   x1 = x0 + d0,  d0 = it / lmax D^-1 r0
//   x2 = x1 + c1 d0 + c2 / lmax D^-1 (b - A x1),
// pre- and post-smoothing alike, so the cycle stays symmetric.  Two choices
// of its coefficients, by the operator of the level:
//   first kind on [lmax/8, lmax]:  theta = 9/16 lmax, delta = 7/16 lmax,
//     rho0 = 7/9, rho1 = 63/113;  it = 16/9, c1 = rho1 rho0, c2 = 288/113
//   fourth kind (Lottes, "Optimal polynomial smoothers for multigrid
//     V-cycles", 2023):  it = 4/3, c1 = 1/5, c2 = 12/5.  No lower end of the
//     interval: it weighs the middle of the spectrum by what the coarse
//     correction leaves of it.
// CG iterations to the same residual with the first and the fourth kind (1e-10; P1 200^2 21 and 18,
// P1 1000^2 28 and 22, a heat step on 1024^2 24 and 18; P2 500^2 22 and 22,
// P2 1023^2 24 and 24, elasticity 383^2 39 and 42; aggregation on tetrahedra 33
// and 34): hierarchies of one P1 component under CG take the fourth kind, the
// others the first.  So does the velocity block of MINRES, which gains less
// than the counts vary with the mesh (256^2: 234 and 224).
struct MgCheb {
    double lam;           // Gershgorin bound of D^-1 A
    double it, c1, c2;
};
#define CHEB_FIRST_KIND {0.0, 16.0 / 9.0, 49.0 / 113.0, 288.0 / 113.0}
#define CHEB_FOURTH_KIND {0.0, 4.0 / 3.0, 1.0 / 5.0, 12.0 / 5.0}
// What the fourth kind leaves is smoother: at the same residual the error is 1.6
// times the first kind's on average (Poisson 100^2 ... 1023^2; at most 3.0), 2.4
// times in heat steps (256^2 ... 2048^2, dt 1e-4; at most 4.3).  With it CG goes on
// to this part of rtol, about one iteration more, so that a solve to rtol is as
// accurate as with the first kind.
#define CHEB_FOURTH_MARGIN 0.4

// done: 0 iterating, 2 the updated residual met rtol (the true residual is
// checked next), 1 finished (status says how), 3 the check of a request in a
// batch asks for a restart from the true residual
struct MgScal {
    double rz, pq, rr, rr0, alpha, beta, relres, rtol;
    int it, done, status, maxit;
    double best;      // smallest true relative residual seen at a check
    double rstop;     // updated relative residual at which CG stops for the check (at most rtol)
    int restarts, pad;
};

enum MgRed { RED_INIT = 0, RED_ALPHA = 1, RED_CONV = 2, RED_BETA = 3, RED_VERIFY = 4, RED_RESTART = 5 };
// the scalar step of W on the reduced values a (and b for RED_INIT); one thread
template <int W>
__device__ __forceinline__ void mg_scalar(MgScal *sc, double a, double b)
{
    if (W == RED_INIT) {  // a = r.z, b = r.r of the start residual
        sc->rz = a;
        sc->rr0 = b;
        sc->rr = b;
        sc->beta = 0.0;
        sc->relres = b > 0.0 ? 1.0 : 0.0;
        if (!(b > 0.0)) sc->done = 1;  // zero right-hand side: x = 0
        else if (!(a > 0.0) || !isfinite(a)) { sc->status = GRMP_ERR_NONFINITE; sc->done = 1; }
    } else if (W == RED_ALPHA) {
        sc->pq = a;
        if (!(a > 0.0) || !isfinite(a)) { sc->status = GRMP_ERR_NONFINITE; sc->done = 1; return; }
        sc->alpha = sc->rz / a;
    } else if (W == RED_CONV) {
        sc->rr = a;
        sc->it += 1;
        sc->relres = sqrt(a / sc->rr0);
        if (!isfinite(a)) { sc->status = GRMP_ERR_NONFINITE; sc->done = 1; }
        else if (sc->relres <= sc->rstop || (sc->it >= sc->maxit && sc->relres <= sc->rtol)) sc->done = 2;
        else if (sc->it >= sc->maxit) { sc->status = GRMP_ERR_NOCONV; sc->done = 1; }
    } else if (W == RED_VERIFY) {  // a = |b - A x|^2
        const double tr = sqrt(a / sc->rr0);
        sc->rr = a;
        sc->relres = tr;
        if (!isfinite(a)) { sc->status = GRMP_ERR_NONFINITE; sc->done = 1; }
        else if (tr <= sc->rtol) sc->done = 1;
        else if (sc->restarts >= 3 || (sc->restarts > 0 && tr > 0.5 * sc->best)) {
            // the true residual stopped improving: the FP64 floor of b - A x
            // (1e-13 .. 1e-10 relative for these problems) is accepted within
            // 100 rtol, as the engine does
            if (!(tr <= 100.0 * sc->rtol)) sc->status = GRMP_ERR_NOCONV;
            sc->done = 1;
        } else {
            sc->restarts += 1;
            sc->best = sc->restarts == 1 || tr < sc->best ? tr : sc->best;
        }
    } else if (W == RED_RESTART) {  // a = r.z of the true residual: p = z
        if (!(a > 0.0) || !isfinite(a)) { sc->status = GRMP_ERR_NONFINITE; sc->done = 1; return; }
        sc->rz = a;
        sc->beta = 0.0;
    } else {
        if (!isfinite(a)) { sc->status = GRMP_ERR_NONFINITE; sc->done = 1; return; }
        sc->beta = a / sc->rz;
        sc->rz = a;
    }
}

// ------------------------------------------------------------ row kernels
// The V-cycle's row products (RESID, CHEB_*) read FP32 copies of the level
// values and accumulate in FP64: the preconditioner moves 8 instead of 12
// bytes per nonzero.  The CG product (PCG_Q) and the true residual of the
// convergence check (TRUE_RESID) read the FP64 values, so the accepted
// solutions meet rtol against the FP64 operator.
enum MgOp { OP_RESID = 0, OP_CHEB_PRE = 1, OP_CHEB_POST1 = 2, OP_CHEB_POST2 = 3, OP_PCG_Q = 4, OP_TRUE_RESID = 5,
            OP_AGG_POST1 = 6 };
template <int OP>
struct MgF64 {
    static constexpr bool value = OP == OP_PCG_Q || OP == OP_TRUE_RESID;
};

struct MgRows {
    const int32_t *rp, *ci;
    const double *val;
    const float *val32;  // FP32 copy (fixed rows 0) for the V-cycle's products
    const uint8_t *fixed;
    int64_t n;
    const double *v;     // the vector A multiplies
    const double *b, *dinv, *d;
    double *o1, *o2;
    const MgCheb *ch;
    const MgScal *sc;
    double *part;        // block partials (OP_PCG_Q: p.q; OP_CHEB_POST2 at level 0: r.z)
    const int32_t *agg;  // OP_AGG_POST1: coarse row of each row, the scale of the correction
    double scale;
};

// d0 = D^-1 b / theta, the first step of the pre-smoothing from x0 = 0.  The
// kernel that produces a level's right-hand side (the restriction, the CG
// update, the true residual, the preconditioner's input) writes d0 beside it,
// 16 bytes a row, so that the pre-smoothing product gathers one array per
// nonzero.  Forming d0 inside the product gathered b, D^-1 and the mask per
// nonzero: 59 us on 4.2M P1 rows against 45 us with d0 stored (the
// producers take 16 bytes a row more).
__device__ __forceinline__ double cheb_first(bool fx, double dinv, double b, const MgCheb &ch)
{
    return fx ? 0.0 : dinv * b * (ch.it / ch.lam);
}

// 256 rows per block through the LDS-staged row product, then the epilogue:
//   RESID   o1 = b - A v
//   TRUE_RESID  the same, and o2 = d0 of the residual      [+ partials of o1 . o1]
//   PRE     v = d0:  o1 = (1 + C1) d0 + C2 D^-1 (b - A d0)
//   POST1   v = x:   d = D^-1 (b - A x) / theta -> o1,  x + d -> o2
//   POST2   v = x1:  o1 = x1 + C1 d + C2 D^-1 (b - A x1)   [+ partials of b . o1]
//   PCG_Q   o1 = A v                                        [+ partials of v . o1]
//   AGG_POST1  POST1 with the aggregates' prolongation e = scale P v, v on the
//           coarse rows, folded in: the columns are the aggregates of A's, so
//           the product is A P v, and with b the residual of x = d
//           d = D^-1 (b - A e) / theta -> o1,  x + e + d -> o2
// Fixed rows get 0 (no residual, no correction).
template <int OP>
__device__ __forceinline__ double mg_epilogue(int64_t i, double s, bool fx, const double *__restrict__ v,
                                              const double *__restrict__ b, const double *__restrict__ dinv,
                                              const double *__restrict__ d, const MgCheb *__restrict__ ch,
                                              double *__restrict__ o1, double *__restrict__ o2)
{
    if (OP == OP_RESID) {
        o1[i] = fx ? 0.0 : b[i] - s;
    } else if (OP == OP_TRUE_RESID) {
        const double r = fx ? 0.0 : b[i] - s;
        o1[i] = r;
        o2[i] = cheb_first(fx, dinv[i], r, *ch);
        return r * r;
    } else if (OP == OP_CHEB_PRE) {
        o1[i] = fx ? 0.0 : (1.0 + ch->c1) * v[i] + ch->c2 / ch->lam * dinv[i] * (b[i] - s);
    } else if (OP == OP_CHEB_POST1) {
        const double dd = fx ? 0.0 : dinv[i] * (b[i] - s) * (ch->it / ch->lam);
        o1[i] = dd;
        o2[i] = v[i] + dd;
    } else if (OP == OP_CHEB_POST2) {
        const double z = fx ? 0.0 : v[i] + ch->c1 * d[i] + ch->c2 / ch->lam * dinv[i] * (b[i] - s);
        o1[i] = z;
        return b[i] * z;
    } else {
        const double q = fx ? 0.0 : s;
        o1[i] = q;
        return v[i] * q;
    }
    return 0.0;
}

template <int OP>
// Nonzeros staged per 256-row chunk: 2048 FP64 products (16 KB of LDS)
// lets twice as many workgroups share a CU as SPMV_CAP does; on the served
// stream that took the batched residual from 3.2 to 4.4 TB/s.  The sum order
// does not depend on it.
#define MG_ROWS_CAP (SPMV_CAP / 2)
__device__ __forceinline__ void mg_rows_body(const MgRows &a, int64_t r0, int pidx)
{
    __shared__ double lds[MG_ROWS_CAP];
    const int64_t r1 = r0 + KB < a.n ? r0 + KB : a.n;
    double s;
    if constexpr (MgF64<OP>::value) s = csr_rows_lds<double, double, double, MG_ROWS_CAP>(a.rp, a.ci, a.val, a.v, r0, r1, lds);
    else s = csr_rows_lds<double, float, double, MG_ROWS_CAP>(a.rp, a.ci, a.val32, a.v, r0, r1, lds);
    const int64_t i = r0 + threadIdx.x;
    double pa = 0.0, pb = 0.0;
    if constexpr (OP == OP_AGG_POST1) {
        if (i < r1) {
            const bool fx = a.fixed[i] != 0;
            const double dd = fx ? 0.0 : a.dinv[i] * (a.b[i] - a.scale * s) * (a.ch->it / a.ch->lam);
            const double x = fx ? a.d[i] : a.d[i] + a.scale * a.v[a.agg[i]];
            a.o1[i] = dd;
            a.o2[i] = x + dd;
        }
    } else if (i < r1) {
        pa = mg_epilogue<OP>(i, s, a.fixed[i] != 0, a.v, a.b, a.dinv, a.d, a.ch, a.o1, a.o2);
    }
    if ((OP == OP_CHEB_POST2 || OP == OP_PCG_Q || OP == OP_TRUE_RESID) && a.part) {
        block_sum2(pa, pb);
        if (threadIdx.x == 0) a.part[pidx] = pa;
    }
}

template <int OP>
__global__ __launch_bounds__(KB) void k_mg_rows(MgRows a)
{
    if (a.sc->done) return;
    mg_rows_body<OP>(a, (int64_t)blockIdx.x * KB, blockIdx.x);
}

// the residual on levels of at least MG_FINE_ROWS rows: the same rows as
// k_mg_rows<OP_RESID> under its own name, the kernel the profiled runs time
#define MG_FINE_ROWS (1 << 21)
__global__ __launch_bounds__(KB) void k_mg_resid_fine(MgRows a)
{
    if (a.sc->done) return;
    mg_rows_body<OP_RESID>(a, (int64_t)blockIdx.x * KB, blockIdx.x);
}

// What the smoothing of a level takes from its matrix: the FP32 copy of the
// values for the V-cycle's products (fixed rows 0: their 1e60 penalty has no
// FP32 value, and their products are not used) and the Gershgorin bound
// max_i sum_j |A_ij| / A_ii over the free rows (a max, so the result does not
// depend on the order of the atomics).  One launch for all levels of a
// hierarchy, each a range of blocks of 256 rows.
struct MgPrepLevel {
    const int32_t *rp;
    const double *val, *dinv;
    const uint8_t *fixed;
    float *val32;
    MgCheb *ch;
    int64_t n;
    int blk0, fourth;  // fourth: coefficients of the fourth kind
};
struct MgPrep {
    int nlev, blocks;
    MgPrepLevel lv[MG_MAX_LEVELS];
};

__global__ void k_mg_prep_cheb(MgPrep P)
{
    const int l = threadIdx.x;
    if (l < P.nlev) *P.lv[l].ch = P.lv[l].fourth ? MgCheb CHEB_FOURTH_KIND : MgCheb CHEB_FIRST_KIND;
}

// Bound by the values, 12 bytes a nonzero: they pass through LDS, read and
// written coalesced, and are read once for both results; a block whose bound
// does not exceed the present one leaves the atomic out.  Two kernels of a
// thread a row, an atomic a wave and two launches and a fill a level took
// 1.26 ms on the hierarchy of P2 1023^2 and 5.4 ms on 48 served requests'.
// The P2 solve went from 37.6 to 35.8 ms, the algebraic one of the 128^3 tets
// from 56.0 to 54.6 ms.
#define MG_PREP_CAP 2048
__device__ __forceinline__ void mg_prep_body(const MgPrepLevel &L, int blk)
{
    __shared__ double lds[MG_PREP_CAP];
    const int t = threadIdx.x;
    const int64_t r0 = (int64_t)(blk - L.blk0) * KB, r1 = r0 + KB < L.n ? r0 + KB : L.n, r = r0 + t;
    const int32_t base = L.rp[r0], end = L.rp[r1];
    int32_t my0 = 0, my1 = 0;
    bool fx = false;
    if (r < r1) {
        my0 = L.rp[r];
        my1 = L.rp[r + 1];
        fx = L.fixed[r] != 0;
    }
    const double *__restrict__ val = L.val;
    float *__restrict__ val32 = L.val32;
    double s = 0.0;
    for (int32_t c0 = base; c0 < end; c0 += MG_PREP_CAP) {
        const int32_t c1 = c0 + MG_PREP_CAP < end ? c0 + MG_PREP_CAP : end;
        __syncthreads();
        constexpr int U = MG_PREP_CAP / KB;
        double w[U];
#pragma unroll
        for (int u = 0; u < U; ++u) w[u] = c0 + t + u * KB < c1 ? val[c0 + t + u * KB] : 0.0;
#pragma unroll
        for (int u = 0; u < U; ++u) lds[t + u * KB] = w[u];
        __syncthreads();
        const int32_t a = my0 > c0 ? my0 : c0, b = my1 < c1 ? my1 : c1;
        for (int32_t k = a; k < b; ++k) {
            if (fx) lds[k - c0] = 0.0;
            else s += fabs(lds[k - c0]);
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (c0 + t + u * KB < c1) val32[c0 + t + u * KB] = (float)lds[t + u * KB];
    }
    s = r < r1 && !fx ? s * fabs(L.dinv[r]) : 0.0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s = fmax(s, __shfl_down(s, o, 64));
    unsigned long long *lam = (unsigned long long *)&L.ch->lam;
    if ((t & 63) == 0 && s > 0.0) {
        const unsigned long long v = (unsigned long long)__double_as_longlong(s);
        if (v > __hip_atomic_load(lam, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(lam, v);
    }
}

__global__ __launch_bounds__(KB) void k_mg_prep(MgPrep P)
{
    int l = 0;
    while (l + 1 < P.nlev && (int)blockIdx.x >= P.lv[l + 1].blk0) ++l;
    mg_prep_body(P.lv[l], blockIdx.x);
}

// the coefficients of n levels (and of their copies in the LDS image), the bounds kept
struct MgChebSet {
    int n, fourth;
    MgCheb *ch[2 * MG_MAX_LEVELS];
};
__global__ void k_mg_cheb_kind(MgChebSet P)
{
    const int l = threadIdx.x;
    if (l >= P.n) return;
    MgCheb c = P.fourth ? MgCheb CHEB_FOURTH_KIND : MgCheb CHEB_FIRST_KIND;
    c.lam = P.ch[l]->lam;
    *P.ch[l] = c;
}

static void mg_prep_add(MgPrep &P, const int32_t *rp, const double *val, const double *dinv, const uint8_t *fixed,
                        float *val32, MgCheb *ch, int64_t n, bool fourth)
{
    P.lv[P.nlev++] = MgPrepLevel{rp, val, dinv, fixed, val32, ch, n, P.blocks, fourth ? 1 : 0};
    P.blocks += (int)nblk(n, KB);
}

static void mg_prep_launch(const MgPrep &P, hipStream_t st)
{
    hipLaunchKernelGGL(k_mg_prep_cheb, dim3(1), dim3(64), 0, st, P);
    hipLaunchKernelGGL(k_mg_prep, dim3(P.blocks), dim3(KB), 0, st, P);
}

// ------------------------------------------------------------- transfers
// Fine node (i, j) of the Nf-square lies in coarse square (ic, jc) of the
// Nc-triangulation at offsets u = un / Nf, v = vn / Nf in [0, 1] (integers:
// i Nc = ic Nf + un), in its lower triangle when u >= v.  The interpolation
// weight of coarse node (ic + dx, jc + dy) there is w / Nf with
//   (0,0): Nf - max(un, vn)    (1,0): max(un - vn, 0)
//   (1,1): min(un, vn)         (0,1): max(vn - un, 0)
// (the barycentric coordinates of both triangles in one formula); prolongation
// and restriction both evaluate it, so P^T is exactly the transpose of P.
__device__ __forceinline__ void p1_coord(int Nf, int Nc, int i, int &ic, int &un)
{
    ic = i * Nc / Nf;
    if (ic > Nc - 1) ic = Nc - 1;
    un = i * Nc - ic * Nf;
}

__device__ __forceinline__ int p1_weight(int Nf, int dx, int dy, int un, int vn)
{
    if (dx == 0 && dy == 0) return Nf - (un > vn ? un : vn);
    if (dx == 1 && dy == 0) return un > vn ? un - vn : 0;
    if (dx == 1 && dy == 1) return un < vn ? un : vn;
    return vn > un ? vn - un : 0;  // (0,1)
}

// component and node of item t, components blocked by node count: at most
// three components, so subtracting beats a 64-bit division
__device__ __forceinline__ int p1_split(int64_t nn, int64_t &t)
{
    int k = 0;
    while (t >= nn) {
        t -= nn;
        ++k;
    }
    return k;
}

// xf += P xc on free fine dofs (components blocked by node count); t < nnf * ncomp
__device__ __forceinline__ void prolong_p1_one(int64_t Nf64, int64_t Nc64, int ncomp, const double *__restrict__ xc,
                                               const uint8_t *__restrict__ fixed_f, double *__restrict__ xf, int64_t t)
{
    const int Nf = (int)Nf64, Nc = (int)Nc64;
    const int64_t nnf = (int64_t)(Nf + 1) * (Nf + 1), nnc = (int64_t)(Nc + 1) * (Nc + 1);
    if (fixed_f[t]) return;
    int64_t node64 = t;
    const int k = p1_split(nnf, node64);
    const uint32_t node = (uint32_t)node64;
    const int row = (int)(node / (uint32_t)(Nf + 1));
    int ic, un, jc, vn;
    p1_coord(Nf, Nc, (int)node - row * (Nf + 1), ic, un);
    p1_coord(Nf, Nc, row, jc, vn);
    const double inv = 1.0 / (double)Nf;
    const double *x = xc + k * nnc + (int64_t)jc * (Nc + 1) + ic;
    double s = (double)p1_weight(Nf, 0, 0, un, vn) * inv * x[0];
    s += (double)p1_weight(Nf, 1, 0, un, vn) * inv * x[1];
    s += (double)p1_weight(Nf, 1, 1, un, vn) * inv * x[Nc + 2];
    s += (double)p1_weight(Nf, 0, 1, un, vn) * inv * x[Nc + 1];
    xf[t] += s;
}

// the value of P^T rf at coarse dof t < nnc * ncomp, 0 on fixed ones.  Fine
// node (i, j) has weight Nf - max(|a|, |b|) for a b >= 0 and
// max(Nf - |a| - |b|, 0) otherwise, a = i Nc - I Nf and b = j Nc - J Nf being
// its offsets from coarse node (I, J) in units of 1 / (Nf Nc): p1_weight's
// four cases in one formula.  Nc = ceil(Nf / 2), so the nodes with |a| < Nf
// are at most four in a row: a 4 x 4 window whose loads are all in flight at
// once.  Walking the index box node by node instead (a division and a
// dependent load per step) made this a serial chain of memory latencies:
// 10.2 us per launch whatever the size, against 3.4 us.
__device__ __forceinline__ double restrict_p1_one(int64_t Nf64, int64_t Nc64, const double *__restrict__ rf,
                                                  const uint8_t *__restrict__ fixed_c, int64_t t)
{
    const int Nf = (int)Nf64, Nc = (int)Nc64;
    const int64_t nnf = (int64_t)(Nf + 1) * (Nf + 1), nnc = (int64_t)(Nc + 1) * (Nc + 1);
    if (fixed_c[t]) return 0.0;
    int64_t node64 = t;
    const int k = p1_split(nnc, node64);
    const uint32_t node = (uint32_t)node64;
    const int J = (int)(node / (uint32_t)(Nc + 1)), I = (int)node - J * (Nc + 1);
    const int i0 = I >= 1 ? (I - 1) * Nf / Nc + 1 : 0, j0 = J >= 1 ? (J - 1) * Nf / Nc + 1 : 0;
    const double inv = 1.0 / (double)Nf;
    const double *r = rf + k * nnf;
    int w[4][4];
    double v[4][4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int j = j0 + q, b = j * Nc - J * Nf;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int i = i0 + p, a = i * Nc - I * Nf;
            const int aa = a < 0 ? -a : a, ab = b < 0 ? -b : b;
            int wt = (a < 0) == (b < 0) ? Nf - (aa > ab ? aa : ab) : Nf - aa - ab;
            if (wt < 0 || i > Nf || j > Nf) wt = 0;
            w[q][p] = wt;
            v[q][p] = 0.0;
            if (wt != 0) v[q][p] = r[(int64_t)j * (Nf + 1) + i];
        }
    }
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int p = 0; p < 4; ++p)
            if (w[q][p] != 0) s += (double)w[q][p] * inv * v[q][p];
    return s;
}

// P1 -> P2 on the same N-square, added into x2: node dofs copy (t < nn),
// face dofs take the mean of their end nodes (t < nc: each face is handled by
// the one cell whose CellFaceSign is +1 for it, its first appearance)
__device__ __forceinline__ void prolong_p2_one(int64_t N, const int32_t *__restrict__ cells,
                                               const int8_t *__restrict__ fsign, const double *__restrict__ x1,
                                               const uint8_t *__restrict__ fixed2, double *__restrict__ x2, int64_t t)
{
    const int64_t nn = (N + 1) * (N + 1), nc = 2 * N * N;
    if (t < nn && !fixed2[t]) x2[t] += x1[t];
    if (t >= nc) return;
    int64_t f[3];
    sq_cellfaces(N, t, f);
    for (int k = 0; k < 3; ++k) {
        if (fsign[k * nc + t] <= 0) continue;
        const int64_t dof = nn + f[k];
        if (fixed2[dof]) continue;
        const int32_t a = cells[k * nc + t], b = cells[((k + 1) % 3) * nc + t];
        x2[dof] += 0.5 * (x1[a] + x1[b]);
    }
}

// its transpose (v < nn): node v gathers r2[v] and half of each incident
// face's entry (left / right horizontal, lower / upper vertical, lower-left /
// upper-right diagonal)
__device__ __forceinline__ double restrict_p2_one(int64_t N, const double *__restrict__ r2,
                                                  const uint8_t *__restrict__ fixed1, int64_t v)
{
    const int64_t nn = (N + 1) * (N + 1);
    if (fixed1[v]) return 0.0;
    const int64_t i = v % (N + 1), j = v / (N + 1);
    const double *rf = r2 + nn;
    double s = 0.0;
    if (i > 0) s += rf[sq_H(N, i - 1, j)];
    if (i < N) s += rf[sq_H(N, i, j)];
    if (j > 0) s += rf[sq_V(N, i, j - 1)];
    if (j < N) s += rf[sq_V(N, i, j)];
    if (i > 0 && j > 0) s += rf[sq_D(N, i - 1, j - 1)];
    if (i < N && j < N) s += rf[sq_D(N, i, j)];
    return r2[v] + 0.5 * s;
}

__global__ void k_mg_prolong_p1(int64_t Nf, int64_t Nc, int ncomp, const double *__restrict__ xc,
                                const uint8_t *__restrict__ fixed_f, double *__restrict__ xf, const MgScal *sc)
{
    if (sc->done) return;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < (Nf + 1) * (Nf + 1) * ncomp) prolong_p1_one(Nf, Nc, ncomp, xc, fixed_f, xf, t);
}

// b_c = P^T r_f and, for the coarse level's smoothing, d_c = d0 of b_c
__global__ void k_mg_restrict_p1(int64_t Nf, int64_t Nc, int ncomp, const double *__restrict__ rf,
                                 const uint8_t *__restrict__ fixed_c, const double *__restrict__ dinv_c,
                                 const MgCheb *__restrict__ ch_c, double *__restrict__ bc, double *__restrict__ dc,
                                 const MgScal *sc)
{
    if (sc->done) return;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (Nc + 1) * (Nc + 1) * ncomp) return;
    const double b = restrict_p1_one(Nf, Nc, rf, fixed_c, t);
    bc[t] = b;
    dc[t] = cheb_first(fixed_c[t] != 0, dinv_c[t], b, *ch_c);
}

__global__ void k_mg_prolong_p2(int64_t N, const int32_t *__restrict__ cells, const int8_t *__restrict__ fsign,
                                const double *__restrict__ x1, const uint8_t *__restrict__ fixed2,
                                double *__restrict__ x2, const MgScal *sc)
{
    if (sc->done) return;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    prolong_p2_one(N, cells, fsign, x1, fixed2, x2, t);
}

__global__ void k_mg_restrict_p2(int64_t N, const double *__restrict__ r2, const uint8_t *__restrict__ fixed1,
                                 const double *__restrict__ dinv1, const MgCheb *__restrict__ ch1,
                                 double *__restrict__ b1, double *__restrict__ d1, const MgScal *sc)
{
    if (sc->done) return;
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= (N + 1) * (N + 1)) return;
    const double b = restrict_p2_one(N, r2, fixed1, v);
    b1[v] = b;
    d1[v] = cheb_first(fixed1[v] != 0, dinv1[v], b, *ch1);
}

// coarse coefficient: geometric mean of the fine cells whose centroid lies in
// the coarse cell (centroids in units of 1 / (3 Nf); same integer test as the
// fine-to-coarse location above).  A coarse cell without a fine centroid
// (not met for Nf <= 2048) takes the fine cell holding its own centroid.
__device__ __forceinline__ int64_t mg_cell_of(int64_t Nf, int64_t Nc, int64_t X, int64_t Y)
{
    // point (X, Y) / (3 Nf) in the Nc-triangulation
    int64_t ic = X * Nc / (3 * Nf), jc = Y * Nc / (3 * Nf);
    if (ic > Nc - 1) ic = Nc - 1;
    if (jc > Nc - 1) jc = Nc - 1;
    const int64_t un = X * Nc - ic * 3 * Nf, vn = Y * Nc - jc * 3 * Nf;
    return 2 * (jc * Nc + ic) + (un >= vn ? 0 : 1);
}

__device__ __forceinline__ void coarse_kappa_one(int64_t Nf, int64_t Nc, const double *__restrict__ kf,
                                                 double *__restrict__ kc, int64_t cc)
{
    if (cc >= 2 * Nc * Nc) return;
    const int64_t sq = cc >> 1, jc = sq / Nc, ic = sq % Nc;
    // fine squares overlapping the coarse square
    const int64_t ilo = ic * Nf / Nc, jlo = jc * Nf / Nc;
    int64_t ihi = ((ic + 1) * Nf + Nc - 1) / Nc, jhi = ((jc + 1) * Nf + Nc - 1) / Nc;
    if (ihi > Nf) ihi = Nf;
    if (jhi > Nf) jhi = Nf;
    double s = 0.0;
    int cnt = 0;
    for (int64_t j = jlo; j < jhi; ++j)
        for (int64_t i = ilo; i < ihi; ++i)
            for (int up = 0; up < 2; ++up) {
                const int64_t X = 3 * i + (up ? 1 : 2), Y = 3 * j + (up ? 2 : 1);
                if (mg_cell_of(Nf, Nc, X, Y) != cc) continue;
                s += log(kf[2 * (j * Nf + i) + up]);
                ++cnt;
            }
    if (cnt == 0) {
        // centroid of the coarse cell in units of 1 / (3 Nc), located among fine cells
        const int64_t Xc = 3 * ic + ((cc & 1) ? 1 : 2), Yc = 3 * jc + ((cc & 1) ? 2 : 1);
        kc[cc] = kf[mg_cell_of(Nc, Nf, Xc, Yc)];
        return;
    }
    kc[cc] = exp(s / cnt);
}

__global__ void k_mg_coarse_kappa(int64_t Nf, int64_t Nc, const double *__restrict__ kf, double *__restrict__ kc)
{
    coarse_kappa_one(Nf, Nc, kf, kc, (int64_t)blockIdx.x * blockDim.x + threadIdx.x);
}

// ------------------------------------------------------ coarsest level
// Dense inverse of the coarsest matrix (fixed rows and columns replaced by
// the identity), in-place Gauss-Jordan in LDS by one block.  The matrix is
// symmetric positive definite, so no pivoting is needed.
__device__ __forceinline__ void dense_inv_block(const int32_t *__restrict__ rp, const int32_t *__restrict__ ci,
                                                const double *__restrict__ val, const uint8_t *__restrict__ fixed,
                                                int n, double *__restrict__ inv)
{
    __shared__ double M[MG_DENSE_MAX * MG_DENSE_MAX];
    __shared__ double f[MG_DENSE_MAX];
    const int t = threadIdx.x;
    for (int e = t; e < n * n; e += blockDim.x) M[e] = 0.0;
    __syncthreads();
    if (t < n) {
        if (fixed[t]) {
            M[t * n + t] = 1.0;
        } else {
            for (int32_t k = rp[t]; k < rp[t + 1]; ++k)
                if (!fixed[ci[k]]) M[t * n + ci[k]] = val[k];
        }
    }
    __syncthreads();
    for (int k = 0; k < n; ++k) {
        const double p = M[k * n + k];
        __syncthreads();
        if (t < n) M[k * n + t] = (t == k ? 1.0 : M[k * n + t]) / p;
        __syncthreads();
        if (t < n) f[t] = t == k ? 0.0 : M[t * n + k];
        __syncthreads();
        for (int e = t; e < n * n; e += blockDim.x) {
            const int r = e / n, c = e - r * n;
            if (r == k) continue;
            M[e] = (c == k ? 0.0 : M[e]) - f[r] * M[k * n + c];
        }
        __syncthreads();
    }
    for (int e = t; e < n * n; e += blockDim.x) inv[e] = M[e];
}

__global__ __launch_bounds__(256) void k_mg_dense_inv(const int32_t *__restrict__ rp, const int32_t *__restrict__ ci,
                                                      const double *__restrict__ val, const uint8_t *__restrict__ fixed,
                                                      int n, double *__restrict__ inv)
{
    dense_inv_block(rp, ci, val, fixed, n, inv);
}

__global__ void k_mg_dense_apply(const double *__restrict__ inv, const double *__restrict__ b, int n,
                                 double *__restrict__ x, const MgScal *sc)
{
    if (sc->done) return;
    const int i = threadIdx.x;
    if (i >= n) return;
    double s = 0.0;
    for (int j = 0; j < n; ++j) s += inv[i * n + j] * b[j];
    x[i] = s;
}

// --------------------------------------------------------------- PCG
__global__ void k_mg_dot(const double *__restrict__ a, const double *__restrict__ b, int64_t n, double *part,
                         const MgScal *sc)
{
    if (sc->done) return;
    const int64_t i = (int64_t)blockIdx.x * KB + threadIdx.x;
    double pa = i < n ? a[i] * b[i] : 0.0, pb = 0.0;
    block_sum2(pa, pb);
    if (threadIdx.x == 0) part[blockIdx.x] = pa;
}

// x += alpha p, r -= alpha q; partials of r.r; d = d0 of the new r
__global__ void k_mg_axpy(double *__restrict__ x, double *__restrict__ r, const double *__restrict__ p,
                          const double *__restrict__ q, const uint8_t *__restrict__ fixed,
                          const double *__restrict__ dinv, const MgCheb *__restrict__ ch, double *__restrict__ d,
                          int64_t n, double *part, const MgScal *sc)
{
    if (sc->done) return;
    const double al = sc->alpha;
    const MgCheb c = *ch;
    const int64_t i = (int64_t)blockIdx.x * KB + threadIdx.x;
    double pa = 0.0, pb = 0.0;
    if (i < n) {
        x[i] += al * p[i];
        const double ri = r[i] - al * q[i];
        r[i] = ri;
        d[i] = cheb_first(fixed[i] != 0, dinv[i], ri, c);
        pa = ri * ri;
    }
    block_sum2(pa, pb);
    if (threadIdx.x == 0) part[blockIdx.x] = pa;
}

// r = rhs on the free rows, 0 on the fixed ones; d = d0 of it
__device__ __forceinline__ double mg_start_one(const double *__restrict__ rhs, const uint8_t *__restrict__ fixed,
                                               const double *__restrict__ dinv, const MgCheb *__restrict__ ch,
                                               double *__restrict__ r, double *__restrict__ d, int64_t i)
{
    const bool fx = fixed[i] != 0;
    const double ri = fx ? 0.0 : rhs[i];
    r[i] = ri;
    d[i] = cheb_first(fx, dinv[i], ri, *ch);
    return ri;
}

__global__ void k_mg_start(const double *__restrict__ rhs, const uint8_t *__restrict__ fixed,
                           const double *__restrict__ dinv, const MgCheb *__restrict__ ch, double *__restrict__ r,
                           double *__restrict__ d, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) mg_start_one(rhs, fixed, dinv, ch, r, d, i);
}

__global__ void k_mg_update_p(double *__restrict__ p, const double *__restrict__ z, int64_t n, const MgScal *sc)
{
    if (sc->done) return;
    const double be = sc->beta;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = z[i] + be * p[i];
}

// a check (2) or a restart (3) was requested: resume the kernels for it
__global__ void k_mg_verify_begin(MgScal *sc)
{
    if (threadIdx.x == 0 && sc->done >= 2) sc->done = 0;
}

// ------------------------------------------------- one-workgroup kernels
// Levels with at most block_rows rows run inside one workgroup of MG_BT
// threads, phases separated by workgroup barriers: the coarse end of every
// V-cycle in one launch, and for requests whose finest level is that small,
// whole CG iterations in one launch.  Rows are summed in column order by one
// thread each.
#define MG_BT 1024

struct MgBLevel {
    const int32_t *rp, *ci;
    const double *val, *dinv;
    const float *val32;
    const uint8_t *fixed;
    double *x, *b, *r, *d;
    const MgCheb *ch;
    int64_t n;
    int N, fe, ncomp, pad;
    const int32_t *cells;  // P2 level: its mesh, for the P1 -> P2 prolongation
    const int8_t *fsign;
};

// The levels of a one-workgroup coarse end packed into LDS: an image of their
// matrices (FP32 values, 16-bit columns and row pointers, D^-1, masks, lambda,
// aggregates) laid out once per hierarchy in device memory and copied in at
// the kernel's start, and behind it the level vectors, which never leave LDS.
// Offsets are in bytes from the start of LDS.
#define MG_PACK_LEVELS 12
#define MG_LDS_MAX (155 * 1024)  // of a CU's 160 KB; the reductions' static arrays need the rest
enum MgTransfer { TR_P1 = 0, TR_P2 = 1, TR_AGG = 2 };
struct MgPackLevel {
    int32_t n, N, fe, ncomp;
    int32_t tr;                   // transfer to the next level
    int32_t val, ci, rp, dinv, fix, ch;
    int32_t agg, mptr, midx;      // TR_AGG: row -> coarse row, and the coarse rows' members
    int32_t x, b, r, d;
};
struct MgPack {
    int32_t nlev;                 // 0: does not fit, the levels stay in device memory
    int32_t image, lds;           // bytes of the image (a multiple of 16) and in all
    int32_t ninv;
    const char *img;
    const double *inv;            // dense inverse of the last level
    const int32_t *cells;         // TR_P2: the fine level's mesh
    const int8_t *fsign;
    double scale;                 // TR_AGG: of the coarse correction
    MgPackLevel lv[MG_PACK_LEVELS];
};

struct MgBDesc {
    int first, nlev, nb0, pad;  // levels first .. nlev-1 run in the workgroup
    MgBLevel lv[MG_MAX_LEVELS];
    const double *inv;          // coarsest level's dense inverse
    double *x, *r, *z, *p, *q;  // level-0 CG vectors
    const double *rhs;
    double *part, *part2;       // level-0 block partials (nb0 entries)
    MgScal *sc;
    MgPack pack;                // the same levels in LDS, where they fit
};

// sum over the workgroup, returned to every thread
__device__ double blk_sum(double v)
{
    __shared__ double ws[MG_BT / 64];
    v = wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < MG_BT / 64; ++k) t += ws[k];
    return t;
}

// The fixed-order sum of nb partials by one workgroup of MG_BT threads, the
// same for a request alone and in a batch.  One workgroup, so bound by the
// latency of its loads: eight are in flight per thread, which takes the 16,401
// partials of 4.2M rows in three rounds, 5.0 us (256 threads with one load at a
// time: 17 us, and three of them an iteration).  Four loads: 5.3 us, sixteen 5.0.
#define MG_RED_U 8
__device__ double red_sum(const double *__restrict__ part, int nb)
{
    double a = 0.0;
    for (int k = threadIdx.x; k < nb; k += MG_RED_U * MG_BT) {
        double v[MG_RED_U];
#pragma unroll
        for (int u = 0; u < MG_RED_U; ++u) v[u] = k + u * MG_BT < nb ? part[k + u * MG_BT] : 0.0;
#pragma unroll
        for (int u = 0; u < MG_RED_U; ++u) a += v[u];
    }
    return blk_sum(a);
}

// one block: the sum of the partials, then the scalar step
template <int W>
__global__ __launch_bounds__(MG_BT) void k_mg_red(const double *__restrict__ part, int nb,
                                                  const double *__restrict__ part2, MgScal *sc)
{
    if (sc->done) return;
    const double a = red_sum(part, nb), b = W == RED_INIT ? red_sum(part2, nb) : 0.0;
    if (threadIdx.x == 0) mg_scalar<W>(sc, a, b);
}

// rows of level L through the epilogue OP; returns this thread's partial
template <int OP>
__device__ double blk_rows(const MgBLevel &L, const double *v, const double *b, const double *d, double *o1,
                           double *o2)
{
    double part = 0.0;
    for (int64_t i = threadIdx.x; i < L.n; i += MG_BT) {
        double s = 0.0;
        if constexpr (MgF64<OP>::value)
            for (int32_t k = L.rp[i]; k < L.rp[i + 1]; ++k) s += L.val[k] * v[L.ci[k]];
        else
            for (int32_t k = L.rp[i]; k < L.rp[i + 1]; ++k) s += (double)L.val32[k] * v[L.ci[k]];
        part += mg_epilogue<OP>(i, s, L.fixed[i] != 0, v, b, L.dinv, d, L.ch, o1, o2);
    }
    return part;
}

// V-cycle over levels D.first .. D.nlev-1 (x_first = V(b_first)); returns the
// workgroup total of b_0 . x_0 when D.first == 0
__device__ double blk_vcycle(const MgBDesc &D)
{
    const int L1 = D.nlev - 1;
    for (int l = D.first; l < L1; ++l) {
        const MgBLevel &L = D.lv[l], &C = D.lv[l + 1];
        for (int64_t i = threadIdx.x; i < L.n; i += MG_BT)
            L.d[i] = cheb_first(L.fixed[i] != 0, L.dinv[i], L.b[i], *L.ch);
        __syncthreads();
        blk_rows<OP_CHEB_PRE>(L, L.d, L.b, nullptr, L.x, nullptr);
        __syncthreads();
        blk_rows<OP_RESID>(L, L.x, L.b, nullptr, L.r, nullptr);
        __syncthreads();
        for (int64_t t = threadIdx.x; t < C.n; t += MG_BT) {
            C.b[t] = L.fe == GRMP_FE_H1P2 ? restrict_p2_one(L.N, L.r, C.fixed, t)
                                          : restrict_p1_one(L.N, C.N, L.r, C.fixed, t);
        }
        __syncthreads();
    }
    {
        const MgBLevel &C = D.lv[L1];
        const int n = (int)C.n;
        for (int i = threadIdx.x; i < n; i += MG_BT) {
            double s = 0.0;
            for (int j = 0; j < n; ++j) s += D.inv[i * n + j] * C.b[j];
            C.x[i] = s;
        }
        __syncthreads();
    }
    double rz = 0.0;
    for (int l = L1 - 1; l >= D.first; --l) {
        const MgBLevel &L = D.lv[l], &C = D.lv[l + 1];
        if (L.fe == GRMP_FE_H1P2) {
            const int64_t nn = (int64_t)(L.N + 1) * (L.N + 1), nc = 2ll * L.N * L.N;
            for (int64_t t = threadIdx.x; t < (nn > nc ? nn : nc); t += MG_BT)
                prolong_p2_one(L.N, L.cells, L.fsign, C.x, L.fixed, L.x, t);
        } else {
            for (int64_t t = threadIdx.x; t < L.n; t += MG_BT)
                prolong_p1_one(L.N, C.N, L.ncomp, C.x, L.fixed, L.x, t);
        }
        __syncthreads();
        blk_rows<OP_CHEB_POST1>(L, L.x, L.b, nullptr, L.d, L.r);
        __syncthreads();
        const double p = blk_rows<OP_CHEB_POST2>(L, L.r, L.b, L.d, L.x, nullptr);
        __syncthreads();
        if (l == 0) rz = blk_sum(p);
    }
    if (D.first == 0 && L1 == 0) {  // a single level: z is the exact solve
        double p = 0.0;
        for (int64_t i = threadIdx.x; i < D.lv[0].n; i += MG_BT) p += D.lv[0].b[i] * D.lv[0].x[i];
        rz = blk_sum(p);
    }
    return rz;
}

// ---- the same V-cycle with everything in LDS
// Latency-bound: about seven short phases a level with a workgroup barrier
// after each.  With matrices and vectors in device memory every phase waited
// for a chain of three or four L2 reads (row pointer, column and value, x,
// epilogue operands): 59-104 us per V-cycle of 25 ... 1,089 rows a level.  One
// coalesced copy of the image (about 100 KB) and LDS latencies after it take
// 30-35 us.
__device__ __forceinline__ void pk_stage(const MgPack &P, char *lds)
{
    const uint4 *src = reinterpret_cast<const uint4 *>(P.img);
    uint4 *dst = reinterpret_cast<uint4 *>(lds);
    for (int k = threadIdx.x; k < P.image / 16; k += MG_BT) dst[k] = src[k];
}

// this thread's share of the dense inverse: row t / 16, columns t % 16 + 16 m
__device__ __forceinline__ void pk_load_inv(const MgPack &P, double inv[4])
{
    const int i = threadIdx.x >> 4, n = P.ninv;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const int j = (threadIdx.x & 15) + 16 * m;
        inv[m] = i < n && j < n ? P.inv[i * n + j] : 0.0;
    }
}

// rows of level L through the epilogue OP (as blk_rows); returns this thread's partial
template <int OP>
__device__ __forceinline__ double pk_rows(const MgPackLevel &L, char *lds, int ov, int oo1, int oo2)
{
    const float *val = reinterpret_cast<const float *>(lds + L.val);
    const uint16_t *ci = reinterpret_cast<const uint16_t *>(lds + L.ci);
    const uint16_t *rp = reinterpret_cast<const uint16_t *>(lds + L.rp);
    const double *v = reinterpret_cast<const double *>(lds + ov);
    const double *b = reinterpret_cast<const double *>(lds + L.b), *d = reinterpret_cast<const double *>(lds + L.d);
    const double *dinv = reinterpret_cast<const double *>(lds + L.dinv);
    const MgCheb *ch = reinterpret_cast<const MgCheb *>(lds + L.ch);
    const uint8_t *fix = reinterpret_cast<const uint8_t *>(lds + L.fix);
    double *o1 = reinterpret_cast<double *>(lds + oo1), *o2 = reinterpret_cast<double *>(lds + oo2);
    double part = 0.0;
    for (int i = threadIdx.x; i < L.n; i += MG_BT) {
        const int k0 = rp[i], k1 = rp[i + 1];
        double s = 0.0;
        for (int k = k0; k < k1; k += 4) {  // four products in flight; past the row's end its last entry again, unused
            float w[4];
            int c[4];
            double xv[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int e = k + u < k1 ? k + u : k1 - 1;
                w[u] = val[e];
                c[u] = ci[e];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) xv[u] = v[c[u]];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (k + u < k1) s += (double)w[u] * xv[u];
        }
        // b and d are read before o1 / o2 of the same row are written
        part += mg_epilogue<OP>(i, s, fix[i] != 0, v, b, dinv, d, ch, o1, o2);
    }
    return part;
}

// x_0 = V(b_0) on the packed levels; b_0 is set, row by row by the thread that
// owns it.  Returns this thread's partial of b_0 . x_0; x_0 likewise is
// complete for a thread's own rows.
__device__ double pk_vcycle(const MgPack &P, char *lds, const double inv[4])
{
    const int L1 = P.nlev - 1;
    {
        const MgPackLevel &L = P.lv[0];
        const double *b = reinterpret_cast<const double *>(lds + L.b);
        const double *dinv = reinterpret_cast<const double *>(lds + L.dinv);
        const uint8_t *fix = reinterpret_cast<const uint8_t *>(lds + L.fix);
        double *d = reinterpret_cast<double *>(lds + L.d);
        const MgCheb ch = *reinterpret_cast<const MgCheb *>(lds + L.ch);
        for (int i = threadIdx.x; i < L.n; i += MG_BT) d[i] = cheb_first(fix[i] != 0, dinv[i], b[i], ch);
    }
    __syncthreads();
    for (int l = 0; l < L1; ++l) {
        const MgPackLevel &L = P.lv[l], &C = P.lv[l + 1];
        pk_rows<OP_CHEB_PRE>(L, lds, L.d, L.x, L.x);
        __syncthreads();
        pk_rows<OP_RESID>(L, lds, L.x, L.r, L.r);
        __syncthreads();
        const double *r = reinterpret_cast<const double *>(lds + L.r);
        const double *dinv = reinterpret_cast<const double *>(lds + C.dinv);
        const uint8_t *fix = reinterpret_cast<const uint8_t *>(lds + C.fix);
        double *bc = reinterpret_cast<double *>(lds + C.b), *dc = reinterpret_cast<double *>(lds + C.d);
        const MgCheb ch = *reinterpret_cast<const MgCheb *>(lds + C.ch);
        for (int t = threadIdx.x; t < C.n; t += MG_BT) {
            double s;
            if (L.tr == TR_P1) {
                s = restrict_p1_one(L.N, C.N, r, fix, t);
            } else if (L.tr == TR_P2) {
                s = restrict_p2_one(L.N, r, fix, t);
            } else {
                const uint16_t *mp = reinterpret_cast<const uint16_t *>(lds + L.mptr);
                const uint16_t *mi = reinterpret_cast<const uint16_t *>(lds + L.midx);
                s = 0.0;
                for (int k = mp[t]; k < mp[t + 1]; ++k) s += r[mi[k]];
            }
            bc[t] = s;
            dc[t] = cheb_first(fix[t] != 0, dinv[t], s, ch);
        }
        __syncthreads();
    }
    {  // dense solve: sixteen lanes a row
        const MgPackLevel &C = P.lv[L1];
        const double *b = reinterpret_cast<const double *>(lds + C.b);
        double s = 0.0;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const int j = (threadIdx.x & 15) + 16 * m;
            if (j < C.n) s += inv[m] * b[j];
        }
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) s += __shfl_xor(s, o, 16);
        const int i = threadIdx.x >> 4;
        if ((threadIdx.x & 15) == 0 && i < C.n) reinterpret_cast<double *>(lds + C.x)[i] = s;
        __syncthreads();
    }
    double part = 0.0;
    for (int l = L1 - 1; l >= 0; --l) {
        const MgPackLevel &L = P.lv[l], &C = P.lv[l + 1];
        const double *xc = reinterpret_cast<const double *>(lds + C.x);
        double *x = reinterpret_cast<double *>(lds + L.x);
        const uint8_t *fix = reinterpret_cast<const uint8_t *>(lds + L.fix);
        if (L.tr == TR_P1) {
            for (int t = threadIdx.x; t < L.n; t += MG_BT) prolong_p1_one(L.N, C.N, L.ncomp, xc, fix, x, t);
        } else if (L.tr == TR_P2) {
            const int nn = (L.N + 1) * (L.N + 1), nc = 2 * L.N * L.N;
            for (int t = threadIdx.x; t < (nn > nc ? nn : nc); t += MG_BT)
                prolong_p2_one(L.N, P.cells, P.fsign, xc, fix, x, t);
        } else {
            const uint16_t *agg = reinterpret_cast<const uint16_t *>(lds + L.agg);
            for (int t = threadIdx.x; t < L.n; t += MG_BT)
                if (agg[t] != 0xffff) x[t] += P.scale * xc[agg[t]];
        }
        __syncthreads();
        pk_rows<OP_CHEB_POST1>(L, lds, L.x, L.d, L.r);
        __syncthreads();
        part = pk_rows<OP_CHEB_POST2>(L, lds, L.r, L.x, L.x);
        __syncthreads();
    }
    if (L1 == 0) {  // a single level: x is the exact solve
        const double *b = reinterpret_cast<const double *>(lds + P.lv[0].b);
        const double *x = reinterpret_cast<const double *>(lds + P.lv[0].x);
        for (int i = threadIdx.x; i < P.lv[0].n; i += MG_BT) part += b[i] * x[i];
    }
    return part;
}

// packed V-cycle from b to x in device memory
__device__ __forceinline__ double pk_apply(const MgPack &P, char *lds, const double inv[4],
                                           const double *__restrict__ b, double *__restrict__ x)
{
    double *lb = reinterpret_cast<double *>(lds + P.lv[0].b);
    const double *lx = reinterpret_cast<const double *>(lds + P.lv[0].x);
    const int n = P.lv[0].n;
    for (int i = threadIdx.x; i < n; i += MG_BT) lb[i] = b[i];
    const double part = pk_vcycle(P, lds, inv);
    for (int i = threadIdx.x; i < n; i += MG_BT) x[i] = lx[i];
    return part;
}

// the levels D.first .. D.nlev-1 of a V-cycle in one workgroup; returns the
// workgroup total of b_0 . x_0 when D.first == 0
__device__ double blk_coarse(const MgBDesc &D, char *lds)
{
    if (D.pack.nlev == 0) return blk_vcycle(D);
    double inv[4];
    pk_load_inv(D.pack, inv);
    pk_stage(D.pack, lds);
    __syncthreads();
    const MgBLevel &L = D.lv[D.first];
    const double part = pk_apply(D.pack, lds, inv, L.b, L.x);
    return D.first == 0 ? blk_sum(part) : 0.0;
}

// one level's part of the image
struct MgPackSrc {
    const int32_t *rp, *ci;
    const float *val32;
    const double *dinv;
    const MgCheb *ch;
    const uint8_t *fixed;
    const int32_t *agg, *mptr, *midx;  // aggregates (TR_AGG), or nullptr
    int32_t nnz, nc;                   // nonzeros; rows of the next level
};
__device__ __forceinline__ void mg_pack_one(const MgPackLevel &L, const MgPackSrc &S, char *__restrict__ img, int t)
{
    if (t < S.nnz) {
        reinterpret_cast<float *>(img + L.val)[t] = S.val32[t];
        reinterpret_cast<uint16_t *>(img + L.ci)[t] = (uint16_t)S.ci[t];
    }
    if (t <= L.n) reinterpret_cast<uint16_t *>(img + L.rp)[t] = (uint16_t)S.rp[t];
    if (t < L.n) {
        reinterpret_cast<double *>(img + L.dinv)[t] = S.dinv[t];
        reinterpret_cast<uint8_t *>(img + L.fix)[t] = S.fixed[t];
        if (S.agg) {
            reinterpret_cast<uint16_t *>(img + L.agg)[t] = S.agg[t] < 0 ? (uint16_t)0xffff : (uint16_t)S.agg[t];
            reinterpret_cast<uint16_t *>(img + L.midx)[t] = (uint16_t)S.midx[t];
        }
    }
    if (S.agg && t <= S.nc) reinterpret_cast<uint16_t *>(img + L.mptr)[t] = (uint16_t)S.mptr[t];
    if (t == 0) *reinterpret_cast<MgCheb *>(img + L.ch) = *S.ch;
}

__global__ void k_mg_pack(MgPackLevel L, MgPackSrc S, char *__restrict__ img)
{
    mg_pack_one(L, S, img, blockIdx.x * blockDim.x + threadIdx.x);
}

// coarse end of a V-cycle (levels D.first ..); at D.first == 0 also the
// level-0 partials of r.z (total in part[0], zeros after it)
__global__ __launch_bounds__(MG_BT) void k_mg_vcycle_block(const MgBDesc *__restrict__ Dp, const MgScal *sc)
{
    extern __shared__ __align__(16) char pk_lds[];
    if (sc->done) return;
    const MgBDesc &D = *Dp;
    const double rz = blk_coarse(D, pk_lds);
    if (D.first == 0)
        for (int k = threadIdx.x; k < D.nb0; k += MG_BT) D.part[k] = k == 0 ? rz : 0.0;
}

// up to iters CG iterations of a request whose levels all fit the workgroup,
// with the true-residual check and restart of mg_job_verify done in place
__device__ void mg_pcg_block_body(const MgBDesc &D, MgScal *sc, int iters, char *lds)
{
    const MgBLevel &L0 = D.lv[0];
    const int64_t n = L0.n;
    const bool packed = D.pack.nlev > 0;
    double inv[4] = {0.0, 0.0, 0.0, 0.0};
    if (packed) {  // staged once for all the iterations
        if (sc->done == 1) return;
        pk_load_inv(D.pack, inv);
        pk_stage(D.pack, lds);
    }
    auto vcycle = [&]() -> double {
        return packed ? blk_sum(pk_apply(D.pack, lds, inv, D.r, D.z)) : blk_vcycle(D);
    };
    for (int k = 0; k < iters; ++k) {
        __syncthreads();
        const int st = sc->done;
        __syncthreads();
        if (st == 1) return;
        if (st == 2) {  // the updated residual met rtol: check b - A x
            blk_rows<OP_TRUE_RESID>(L0, D.x, D.rhs, nullptr, D.r, L0.d);
            __syncthreads();
            double p = 0.0;
            for (int64_t i = threadIdx.x; i < n; i += MG_BT) p += D.r[i] * D.r[i];
            const double rr = blk_sum(p);
            if (threadIdx.x == 0) {
                sc->done = 0;
                mg_scalar<RED_VERIFY>(sc, rr, 0.0);
            }
            __syncthreads();
            if (sc->done) continue;
            const double rz = vcycle();
            if (threadIdx.x == 0) mg_scalar<RED_RESTART>(sc, rz, 0.0);
            __syncthreads();
            if (sc->done) continue;
            for (int64_t i = threadIdx.x; i < n; i += MG_BT) D.p[i] = D.z[i];
            continue;
        }
        const double pq = blk_sum(blk_rows<OP_PCG_Q>(L0, D.p, nullptr, nullptr, D.q, nullptr));
        if (threadIdx.x == 0) mg_scalar<RED_ALPHA>(sc, pq, 0.0);
        __syncthreads();
        if (sc->done) continue;
        const double al = sc->alpha;
        double p = 0.0;
        for (int64_t i = threadIdx.x; i < n; i += MG_BT) {
            D.x[i] += al * D.p[i];
            const double ri = D.r[i] - al * D.q[i];
            D.r[i] = ri;
            p += ri * ri;
        }
        const double rr = blk_sum(p);
        if (threadIdx.x == 0) mg_scalar<RED_CONV>(sc, rr, 0.0);
        __syncthreads();
        if (sc->done) continue;
        const double rz = vcycle();
        if (threadIdx.x == 0) mg_scalar<RED_BETA>(sc, rz, 0.0);
        __syncthreads();
        if (sc->done) continue;
        const double be = sc->beta;
        for (int64_t i = threadIdx.x; i < n; i += MG_BT) D.p[i] = D.z[i] + be * D.p[i];
    }
}

__global__ __launch_bounds__(MG_BT) void k_mg_pcg_block(const MgBDesc *__restrict__ Dp, MgScal *sc, int iters)
{
    extern __shared__ __align__(16) char pk_lds[];
    mg_pcg_block_body(*Dp, sc, iters, pk_lds);
}

// ------------------------------------------------------ lockstep batches
// Requests in flight advance together: every phase of a CG iteration and of
// its V-cycle is one launch over a table of 256-row tiles of all requests
// taking part, each tile naming its request and level.  Requests whose
// levels all fit one workgroup run in one launch, a workgroup each.  The
// reductions stay per request (one block each, the same fixed order), so a
// request's iterates are the ones it has alone.
struct MgTile {
    int32_t req, level, row0, pad;
};

// a tile is MG_TILE_CHUNKS consecutive 256-row chunks of one level, handled
// by one workgroup chunk after chunk: the tile and descriptor lookups that
// start a workgroup are paid once per tile.  Partials stay per 256-row chunk.
// Two measured best for the batched residual on the served stream (217 us
// per launch against 223-228 us with four and 222-225 us with one).
#ifndef MG_TILE_CHUNKS
#define MG_TILE_CHUNKS 2
#endif

__device__ __forceinline__ MgRows mg_tile_rows(const MgBDesc &D, int level)
{
    const MgBLevel &L = D.lv[level];
    MgRows a;
    a.rp = L.rp;
    a.ci = L.ci;
    a.val = L.val;
    a.val32 = L.val32;
    a.fixed = L.fixed;
    a.n = L.n;
    a.v = nullptr;
    a.b = nullptr;
    a.dinv = L.dinv;
    a.d = nullptr;
    a.o1 = nullptr;
    a.o2 = nullptr;
    a.ch = L.ch;
    a.sc = D.sc;
    a.part = nullptr;
    return a;
}

template <int OP>
__global__ __launch_bounds__(KB) void k_mgb_rows(const MgTile *__restrict__ T, const MgBDesc *const *__restrict__ Dp)
{
    const MgTile t = T[blockIdx.x];
    const MgBDesc &D = *Dp[t.req];
    if (D.sc->done) return;
    const MgBLevel &L = D.lv[t.level];
    MgRows a = mg_tile_rows(D, t.level);
    if (OP == OP_RESID) {
        a.v = L.x;
        a.b = L.b;
        a.o1 = L.r;
    } else if (OP == OP_CHEB_PRE) {
        a.v = L.d;
        a.b = L.b;
        a.o1 = L.x;
    } else if (OP == OP_CHEB_POST1) {
        a.v = L.x;
        a.b = L.b;
        a.o1 = L.d;
        a.o2 = L.r;
    } else if (OP == OP_CHEB_POST2) {
        a.v = L.r;
        a.b = L.b;
        a.d = L.d;
        a.o1 = L.x;
        a.part = t.level == 0 ? D.part : nullptr;
    } else if (OP == OP_PCG_Q) {
        a.v = D.p;
        a.o1 = D.q;
        a.part = D.part;
    }
    for (int c = 0; c < MG_TILE_CHUNKS; ++c) {
        const int64_t r0 = t.row0 + (int64_t)c * KB;
        if (r0 >= L.n) break;
        mg_rows_body<OP>(a, r0, (int)(r0 / KB));
    }
}

// tiles over the rows of coarse level t.level (> 0)
__global__ __launch_bounds__(KB) void k_mgb_restrict(const MgTile *__restrict__ T,
                                                     const MgBDesc *const *__restrict__ Dp)
{
    const MgTile t = T[blockIdx.x];
    const MgBDesc &D = *Dp[t.req];
    if (D.sc->done) return;
    const MgBLevel &F = D.lv[t.level - 1], &C = D.lv[t.level];
    for (int c = 0; c < MG_TILE_CHUNKS; ++c) {
        const int64_t i = t.row0 + (int64_t)c * KB + threadIdx.x;
        if (i >= C.n) break;
        const double b = F.fe == GRMP_FE_H1P2 ? restrict_p2_one(F.N, F.r, C.fixed, i)
                                              : restrict_p1_one(F.N, C.N, F.r, C.fixed, i);
        C.b[i] = b;
        C.d[i] = cheb_first(C.fixed[i] != 0, C.dinv[i], b, *C.ch);
    }
}

// items of fine level t.level: its rows, or for P2 max(nodes, cells)
__global__ __launch_bounds__(KB) void k_mgb_prolong(const MgTile *__restrict__ T,
                                                    const MgBDesc *const *__restrict__ Dp)
{
    const MgTile t = T[blockIdx.x];
    const MgBDesc &D = *Dp[t.req];
    if (D.sc->done) return;
    const MgBLevel &F = D.lv[t.level], &C = D.lv[t.level + 1];
    for (int c = 0; c < MG_TILE_CHUNKS; ++c) {
        const int64_t i = t.row0 + (int64_t)c * KB + threadIdx.x;
        if (F.fe == GRMP_FE_H1P2) {
            const int64_t nn = (int64_t)(F.N + 1) * (F.N + 1), nc = 2ll * F.N * F.N;
            if (i < (nn > nc ? nn : nc)) prolong_p2_one(F.N, F.cells, F.fsign, C.x, F.fixed, F.x, i);
        } else if (i < F.n) {
            prolong_p1_one(F.N, C.N, F.ncomp, C.x, F.fixed, F.x, i);
        }
    }
}

// level-0 tiles: x += alpha p, r -= alpha q, partials of r.r, d0 of the new r
__global__ __launch_bounds__(KB) void k_mgb_axpy(const MgTile *__restrict__ T, const MgBDesc *const *__restrict__ Dp)
{
    const MgTile t = T[blockIdx.x];
    const MgBDesc &D = *Dp[t.req];
    if (D.sc->done) return;
    const MgBLevel &L = D.lv[0];
    const double al = D.sc->alpha;
    const MgCheb ch = *L.ch;
    const int64_t n = L.n;
    for (int c = 0; c < MG_TILE_CHUNKS; ++c) {
        const int64_t r0 = t.row0 + (int64_t)c * KB;
        if (r0 >= n) break;
        const int64_t i = r0 + threadIdx.x;
        double pa = 0.0, pb = 0.0;
        if (i < n) {
            D.x[i] += al * D.p[i];
            const double ri = D.r[i] - al * D.q[i];
            D.r[i] = ri;
            L.d[i] = cheb_first(L.fixed[i] != 0, L.dinv[i], ri, ch);
            pa = ri * ri;
        }
        block_sum2(pa, pb);
        if (threadIdx.x == 0) D.part[r0 / KB] = pa;
    }
}

__global__ __launch_bounds__(KB) void k_mgb_update_p(const MgTile *__restrict__ T,
                                                     const MgBDesc *const *__restrict__ Dp)
{
    const MgTile t = T[blockIdx.x];
    const MgBDesc &D = *Dp[t.req];
    if (D.sc->done) return;
    const double be = D.sc->beta;
    for (int c = 0; c < MG_TILE_CHUNKS; ++c) {
        const int64_t i = t.row0 + (int64_t)c * KB + threadIdx.x;
        if (i < D.lv[0].n) D.p[i] = D.z[i] + be * D.p[i];
    }
}

// one block per request: the fixed-order sum of its partials, then step W
template <int W>
__global__ __launch_bounds__(MG_BT) void k_mgb_red(const MgBDesc *const *__restrict__ Dp,
                                                   const int32_t *__restrict__ reqs)
{
    const MgBDesc &D = *Dp[reqs[blockIdx.x]];
    if (D.sc->done) return;
    const double a = red_sum(D.part, D.nb0);
    if (threadIdx.x == 0) mg_scalar<W>(D.sc, a, 0.0);
}

// The check of the requests whose updated residual met rtol (done 2; the
// others' tiles return at once): r = b - A x, d0 of it, partials of r.r
__global__ __launch_bounds__(KB) void k_mgb_true_resid(const MgTile *__restrict__ T,
                                                       const MgBDesc *const *__restrict__ Dp)
{
    const MgTile t = T[blockIdx.x];
    const MgBDesc &D = *Dp[t.req];
    if (D.sc->done != 2) return;
    MgRows a = mg_tile_rows(D, 0);
    a.v = D.x;
    a.b = D.rhs;
    a.o1 = D.r;
    a.o2 = D.lv[0].d;
    a.part = D.part;
    for (int c = 0; c < MG_TILE_CHUNKS; ++c) {
        const int64_t r0 = t.row0 + (int64_t)c * KB;
        if (r0 >= a.n) break;
        mg_rows_body<OP_TRUE_RESID>(a, r0, (int)(r0 / KB));
    }
}

__global__ __launch_bounds__(MG_BT) void k_mgb_red_verify(const MgBDesc *const *__restrict__ Dp,
                                                          const int32_t *__restrict__ reqs)
{
    const MgBDesc &D = *Dp[reqs[blockIdx.x]];
    if (D.sc->done != 2) return;
    const double a = red_sum(D.part, D.nb0);
    if (threadIdx.x != 0) return;
    D.sc->done = 0;
    mg_scalar<RED_VERIFY>(D.sc, a, 0.0);
    if (D.sc->done == 0) D.sc->done = 3;
}

__global__ __launch_bounds__(MG_BT) void k_mgb_vcycle_block(const MgBDesc *const *__restrict__ Dp,
                                                            const int32_t *__restrict__ reqs)
{
    extern __shared__ __align__(16) char pk_lds[];
    const MgBDesc &D = *Dp[reqs[blockIdx.x]];
    if (D.sc->done) return;
    const double rz = blk_coarse(D, pk_lds);
    if (D.first == 0)
        for (int k = threadIdx.x; k < D.nb0; k += MG_BT) D.part[k] = k == 0 ? rz : 0.0;
}

__global__ __launch_bounds__(MG_BT) void k_mgb_pcg_block(const MgBDesc *const *__restrict__ Dp,
                                                         const int32_t *__restrict__ reqs, int iters)
{
    extern __shared__ __align__(16) char pk_lds[];
    const MgBDesc &D = *Dp[reqs[blockIdx.x]];
    mg_pcg_block_body(D, D.sc, iters, pk_lds);
}

__global__ void k_mgb_status(const MgBDesc *const *__restrict__ Dp, int n, MgStatus *__restrict__ out)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const MgScal *sc = Dp[i]->sc;
    out[i].relres = sc->relres;
    out[i].it = sc->it;
    out[i].done = sc->done;
    out[i].status = sc->status;
    out[i].pad = 0;
}

// Setup of a group of requests: each step one launch over a table of the
// group's levels or requests, an entry a range of blocks from blk0.
struct MgKapEntry {
    const double *kf;
    double *kc;
    int Nf, Nc, blk0, pad;
};
struct MgPackEntry {
    MgPackLevel L;
    MgPackSrc S;
    char *img;
    int blk0, pad;
};
struct MgInvEntry {
    const int32_t *rp, *ci;
    const double *val;
    const uint8_t *fixed;
    double *inv;
    int64_t n;
};
struct MgInitEntry {
    MgBDesc D;
    MgScal s;
    MgBDesc *ddesc;
    MgScal *sc;
};

template <class E>
__device__ __forceinline__ int mg_entry_of(const E *__restrict__ e, int n, int blk)
{
    int lo = 0, hi = n;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (e[mid].blk0 <= blk) lo = mid;
        else hi = mid;
    }
    return lo;
}

__global__ __launch_bounds__(KB) void k_mgb_coarse_kappa(const MgKapEntry *__restrict__ E, int n)
{
    const MgKapEntry &k = E[mg_entry_of(E, n, blockIdx.x)];
    coarse_kappa_one(k.Nf, k.Nc, k.kf, k.kc, (int64_t)((int)blockIdx.x - k.blk0) * KB + threadIdx.x);
}

__global__ void k_mgb_prep_cheb(const MgPrepLevel *__restrict__ E, int n)
{
    const int l = blockIdx.x * blockDim.x + threadIdx.x;
    if (l < n) *E[l].ch = E[l].fourth ? MgCheb CHEB_FOURTH_KIND : MgCheb CHEB_FIRST_KIND;
}

__global__ __launch_bounds__(KB) void k_mgb_prep(const MgPrepLevel *__restrict__ E, int n)
{
    mg_prep_body(E[mg_entry_of(E, n, blockIdx.x)], blockIdx.x);
}

__global__ __launch_bounds__(256) void k_mgb_dense_inv(const MgInvEntry *__restrict__ E)
{
    const MgInvEntry &e = E[blockIdx.x];
    dense_inv_block(e.rp, e.ci, e.val, e.fixed, (int)e.n, e.inv);
}

__global__ __launch_bounds__(KB) void k_mgb_pack(const MgPackEntry *__restrict__ E, int n)
{
    const MgPackEntry &e = E[mg_entry_of(E, n, blockIdx.x)];
    mg_pack_one(e.L, e.S, e.img, ((int)blockIdx.x - e.blk0) * KB + (int)threadIdx.x);
}

// the requests' descriptors and scalars in their places
__global__ __launch_bounds__(KB) void k_mgb_init(const MgInitEntry *__restrict__ E)
{
    const MgInitEntry &e = E[blockIdx.x];
    static_assert(sizeof(MgBDesc) % 4 == 0 && sizeof(MgScal) % 4 == 0, "copied in 32-bit words");
    const uint32_t *d = reinterpret_cast<const uint32_t *>(&e.D), *s = reinterpret_cast<const uint32_t *>(&e.s);
    for (int k = threadIdx.x; k < (int)(sizeof(MgBDesc) / 4); k += KB) reinterpret_cast<uint32_t *>(e.ddesc)[k] = d[k];
    for (int k = threadIdx.x; k < (int)(sizeof(MgScal) / 4); k += KB) reinterpret_cast<uint32_t *>(e.sc)[k] = s[k];
}

// level-0 tiles: r = rhs on the free rows and d0 of it, x = p = 0, partials of r.r
__global__ __launch_bounds__(KB) void k_mgb_start(const MgTile *__restrict__ T, const MgBDesc *const *__restrict__ Dp)
{
    const MgTile t = T[blockIdx.x];
    const MgBDesc &D = *Dp[t.req];
    const MgBLevel &L = D.lv[0];
    for (int c = 0; c < MG_TILE_CHUNKS; ++c) {
        const int64_t r0 = t.row0 + (int64_t)c * KB;
        if (r0 >= L.n) break;
        const int64_t i = r0 + threadIdx.x;
        double pa = 0.0, pb = 0.0;
        if (i < L.n) {
            const double ri = mg_start_one(D.rhs, L.fixed, L.dinv, L.ch, D.r, L.d, i);
            D.x[i] = 0.0;
            D.p[i] = 0.0;
            pa = ri * ri;
        }
        block_sum2(pa, pb);
        if (threadIdx.x == 0) D.part2[r0 / KB] = pa;
    }
}

__global__ __launch_bounds__(MG_BT) void k_mgb_red_init(const MgBDesc *const *__restrict__ Dp)
{
    const MgBDesc &D = *Dp[blockIdx.x];
    if (D.sc->done) return;
    const double a = red_sum(D.part, D.nb0), b = red_sum(D.part2, D.nb0);
    if (threadIdx.x == 0) mg_scalar<RED_INIT>(D.sc, a, b);
}

// ------------------------------------------------------ packing (host)
static size_t mg_lds_limit()
{
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
        return 0;
    return std::min<size_t>((size_t)std::max(v - 1024, 0), MG_LDS_MAX);
}

struct MgPackShape {
    int64_t n, nnz;
    int N, fe, ncomp, tr;
};
// Offsets of the levels (the last one solved by its dense inverse); false, and
// P.nlev = 0, if they do not fit: 16-bit indices and the LDS of one workgroup.
static bool mg_pack_layout(MgPack &P, const MgPackShape *sh, int nlev)
{
    memset(&P, 0, sizeof(P));
    if (nlev < 1 || nlev > MG_PACK_LEVELS || sh[nlev - 1].n > MG_DENSE_MAX) return false;
    const size_t limit = mg_lds_limit();
    size_t off = 0;
    auto take = [&](size_t bytes, size_t align) {
        off = (off + align - 1) / align * align;
        const size_t o = off;
        off += bytes;
        return (int32_t)o;
    };
    for (int l = 0; l < nlev; ++l) {
        const MgPackShape &S = sh[l];
        if (S.n >= 0xffff || S.nnz >= 0xffff || off > limit) return false;
        MgPackLevel &L = P.lv[l];
        L.n = (int32_t)S.n;
        L.N = S.N;
        L.fe = S.fe;
        L.ncomp = S.ncomp;
        L.tr = S.tr;
        L.dinv = take(8 * S.n, 8);
        L.ch = take(sizeof(MgCheb), 8);
        L.val = take(4 * S.nnz, 4);
        L.ci = take(2 * S.nnz, 2);
        L.rp = take(2 * (S.n + 1), 2);
        if (S.tr == TR_AGG && l + 1 < nlev) {
            L.agg = take(2 * S.n, 2);
            L.midx = take(2 * S.n, 2);
            L.mptr = take(2 * (sh[l + 1].n + 1), 2);
        }
        L.fix = take(S.n, 1);
    }
    off = (off + 15) / 16 * 16;
    P.image = (int32_t)off;
    for (int l = 0; l < nlev; ++l) {
        MgPackLevel &L = P.lv[l];
        L.x = take(8 * sh[l].n, 8);
        L.b = take(8 * sh[l].n, 8);
        L.r = take(8 * sh[l].n, 8);
        L.d = take(8 * sh[l].n, 8);
    }
    if (off > limit) return false;
    P.lds = (int32_t)off;
    P.ninv = (int32_t)sh[nlev - 1].n;
    P.nlev = nlev;
    return true;
}

// the kernels with a packed coarse end take more than 64 KB of dynamic LDS
static int mg_allow_lds(grmp_ctx *ctx, const void *kernel)
{
    GRMP_HIP(ctx, hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, MG_LDS_MAX));
    return GRMP_OK;
}

// ------------------------------------------------------------- the job
struct MgLevel {
    MgLevelIn in;
    int64_t n = 0, nnz = 0, nc = 0;
    double *kappa = nullptr, *val = nullptr, *dinv = nullptr, *x = nullptr, *b = nullptr, *r = nullptr, *d = nullptr;
    float *dinv32 = nullptr;
    float *val32 = nullptr;  // FP32 copy of val for the V-cycle, fixed rows 0
    MgCheb *ch = nullptr;
    DevForm *dforms = nullptr;
    DevForm hforms[4];
};

struct MgJob {
    grmp_ctx *ctx = nullptr;
    hipStream_t st = nullptr;
    int nlev = 0;
    MgLevel lv[MG_MAX_LEVELS];
    char *buf = nullptr;
    size_t bytes = 0;
    double *x = nullptr, *rhs = nullptr, *r = nullptr, *z = nullptr, *p = nullptr, *q = nullptr;
    double *part = nullptr, *part2 = nullptr, *inv = nullptr;
    MgScal *sc = nullptr;
    int nb0 = 0;
    int first_small = 0;      // first level that runs inside one workgroup
    size_t img_bytes = 0;     // of its LDS image
    bool fourth = false;      // smoother coefficients of the fourth kind
    char *img = nullptr;      // LDS image of those levels
    MgBDesc hdesc;
    MgBDesc *ddesc = nullptr;
    hipEvent_t ev = nullptr;
    // grid-path chunk of CG iterations captured once and replayed
    bool use_graph = false;
    int graph_iters = 0;
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
    // profile: event pairs around every OP_RESID launch, with its algorithmic bytes
    bool profile = false;
    std::vector<hipEvent_t> pev, pool;  // profiled launches in flight; free events
    std::vector<double> pbytes;
    double prof_s = 0.0, prof_bytes = 0.0;
    int64_t prof_launches = 0;
};

static inline size_t al256(size_t x) { return (x + 255) & ~(size_t)255; }

static size_t mg_layout(MgJob *j, bool assign)
{
    size_t off = 0;
    auto take = [&](size_t bytes) { size_t o = off; off += al256(bytes); return o; };
    const int64_t n0 = j->lv[0].n;
    const int nb0 = (int)nblk(n0, KB);
    size_t o_x = take(n0 * 8), o_rhs = take(n0 * 8), o_r = take(n0 * 8), o_z = take(n0 * 8), o_p = take(n0 * 8),
           o_q = take(n0 * 8), o_part = take(nb0 * 8), o_part2 = take(nb0 * 8), o_sc = take(sizeof(MgScal)),
           o_desc = take(sizeof(MgBDesc));
    const MgLevel &c = j->lv[j->nlev - 1];
    size_t o_inv = take(c.n * c.n * 8), o_img = take(j->img_bytes);
    std::vector<size_t> o(MG_MAX_LEVELS * 10);
    for (int l = 0; l < j->nlev; ++l) {
        const MgLevel &L = j->lv[l];
        const bool own_kappa = l > 0 && L.in.N != j->lv[l - 1].in.N;
        o[10 * l + 0] = own_kappa || l == 0 ? take(L.nc * 8) : 0;
        o[10 * l + 1] = take(L.nnz * 8);
        o[10 * l + 2] = take(L.n * 8);
        o[10 * l + 3] = take(L.n * 4);
        o[10 * l + 4] = l == 0 ? 0 : take(L.n * 8);  // x (level 0: z)
        o[10 * l + 5] = l == 0 ? 0 : take(L.n * 8);  // b (level 0: r)
        o[10 * l + 6] = take(L.n * 8);
        o[10 * l + 7] = take(L.n * 8);
        o[10 * l + 8] = take(sizeof(MgCheb) + sizeof(DevForm) * 4);
        o[10 * l + 9] = take(L.nnz * 4);
    }
    if (!assign) return off;
    char *B = j->buf;
    j->x = (double *)(B + o_x);
    j->rhs = (double *)(B + o_rhs);
    j->r = (double *)(B + o_r);
    j->z = (double *)(B + o_z);
    j->p = (double *)(B + o_p);
    j->q = (double *)(B + o_q);
    j->part = (double *)(B + o_part);
    j->part2 = (double *)(B + o_part2);
    j->sc = (MgScal *)(B + o_sc);
    j->ddesc = (MgBDesc *)(B + o_desc);
    j->inv = (double *)(B + o_inv);
    j->img = B + o_img;
    j->nb0 = nb0;
    for (int l = 0; l < j->nlev; ++l) {
        MgLevel &L = j->lv[l];
        const bool own_kappa = l > 0 && L.in.N != j->lv[l - 1].in.N;
        L.kappa = (own_kappa || l == 0) ? (double *)(B + o[10 * l + 0]) : j->lv[l - 1].kappa;
        L.val = (double *)(B + o[10 * l + 1]);
        L.dinv = (double *)(B + o[10 * l + 2]);
        L.dinv32 = (float *)(B + o[10 * l + 3]);
        L.x = l == 0 ? j->z : (double *)(B + o[10 * l + 4]);
        L.b = l == 0 ? j->r : (double *)(B + o[10 * l + 5]);
        L.r = (double *)(B + o[10 * l + 6]);
        L.d = (double *)(B + o[10 * l + 7]);
        L.ch = (MgCheb *)(B + o[10 * l + 8]);
        L.dforms = (DevForm *)(B + o[10 * l + 8] + sizeof(MgCheb));
        L.val32 = (float *)(B + o[10 * l + 9]);
    }
    return off;
}

// the packed form of the levels from first_small on
static bool mg_job_pack_layout(const MgJob *j, MgPack &P)
{
    MgPackShape sh[MG_MAX_LEVELS];
    for (int l = j->first_small; l < j->nlev; ++l) {
        const MgLevel &L = j->lv[l];
        sh[l - j->first_small] = MgPackShape{L.n, L.nnz, L.in.N, L.in.fe, L.in.ncomp,
                                             L.in.fe == GRMP_FE_H1P2 ? TR_P2 : TR_P1};
    }
    return mg_pack_layout(P, sh, j->nlev - j->first_small);
}

// the first level that may run inside one workgroup: a request with at most
// block_rows rows runs whole in it, otherwise its levels with at most
// coarse_rows rows do
static int mg_first_small(const int64_t *n, int nlev, int block_rows, int coarse_rows)
{
    if (n[0] <= block_rows) return 0;
    int f = nlev - 1;
    while (f > 1 && n[f - 1] <= std::max(coarse_rows, MG_DENSE_MAX)) --f;
    return f;
}

// Bytes of a job's buffer at most, for levels of n rows and up to nnz
// nonzeros: which of them make up the LDS image depends on their nonzeros, so
// it is counted with all that may.
int64_t mg_job_bytes(int nlev, const int64_t *n, const int64_t *nnz, const int64_t *nc, const int *N, int block_rows,
                     int coarse_rows)
{
    MgJob j;
    j.nlev = nlev;
    for (int l = 0; l < nlev; ++l) {
        j.lv[l].n = n[l];
        j.lv[l].nnz = nnz[l];
        j.lv[l].nc = nc[l];
        j.lv[l].in.N = N[l];
    }
    for (int l = mg_first_small(n, nlev, block_rows, coarse_rows); l < nlev; ++l)
        j.img_bytes += 11 * n[l] + 6 * nnz[l] + sizeof(MgCheb) + 32;  // mg_pack_layout's arrays and their padding
    j.img_bytes = std::min<size_t>(j.img_bytes, MG_LDS_MAX);
    return (int64_t)mg_layout(&j, false);
}

static void fill_desc(MgJob *j)
{
    MgBDesc &D = j->hdesc;
    memset(&D, 0, sizeof(D));
    D.first = j->first_small;
    D.nlev = j->nlev;
    D.nb0 = j->nb0;
    for (int l = 0; l < j->nlev; ++l) {
        const MgLevel &L = j->lv[l];
        MgBLevel &B = D.lv[l];
        B.rp = L.in.A->rowptr;
        B.ci = L.in.A->cols;
        B.val = L.val;
        B.val32 = L.val32;
        B.dinv = L.dinv;
        B.fixed = L.in.A->fixed;
        B.x = L.x;
        B.b = L.b;
        B.r = L.r;
        B.d = L.d;
        B.ch = L.ch;
        B.n = L.n;
        B.N = L.in.N;
        B.fe = L.in.fe;
        B.ncomp = L.in.ncomp;
        B.cells = L.in.sp->mesh->cells;
        B.fsign = L.in.sp->mesh->fsign;
    }
    D.inv = j->inv;
    D.x = j->x;
    D.r = j->r;
    D.z = j->z;
    D.p = j->p;
    D.q = j->q;
    D.rhs = j->rhs;
    D.part = j->part;
    D.part2 = j->part2;
    D.sc = j->sc;
    if (mg_job_pack_layout(j, D.pack)) {
        D.pack.img = j->img;
        D.pack.inv = j->inv;
        D.pack.cells = D.lv[j->first_small].cells;
        D.pack.fsign = D.lv[j->first_small].fsign;
    }
}

// the LDS image, once the levels' values, bounds and inverse are enqueued
static MgPackSrc mg_pack_src(const MgJob *j, int k)
{
    const MgLevel &L = j->lv[j->first_small + k];
    return MgPackSrc{L.in.A->rowptr, L.in.A->cols, L.val32, L.dinv, L.ch, L.in.A->fixed,
                     nullptr,        nullptr,      nullptr, (int32_t)L.nnz, 0};
}

static void mg_job_pack(MgJob *j)
{
    const MgPack &P = j->hdesc.pack;
    for (int k = 0; k < P.nlev; ++k) {
        const MgLevel &L = j->lv[j->first_small + k];
        hipLaunchKernelGGL(k_mg_pack, dim3(nblk(std::max(L.nnz, L.n + 1), 256)), dim3(256), 0, j->st, P.lv[k],
                           mg_pack_src(j, k), j->img);
    }
}

int mg_job_create(grmp_ctx *ctx, hipStream_t st, const MgLevelIn *in, int nlev, bool profile, int block_rows,
                  int coarse_rows, bool graph, MgJob **out)
{
    GRMP_CHECK(ctx, nlev >= 1 && nlev <= MG_MAX_LEVELS, GRMP_ERR_ARG, "multigrid: %d levels", nlev);
    for (int l = 0; l < nlev; ++l) {
        const MgLevelIn &L = in[l];
        GRMP_CHECK(ctx, L.A && L.sp && L.A->have_pattern && L.sp->mesh->kind == MESH_UNITSQUARE && L.sp->mesh->N == L.N &&
                            L.A->n == L.sp->ndofs && L.A->n < (1ll << 31),
                   GRMP_ERR_ARG, "multigrid: level %d is not an assembled unit-square pattern", l);
        if (l > 0) {
            const MgLevelIn &F = in[l - 1];
            const bool p2 = F.fe == GRMP_FE_H1P2 && L.fe == GRMP_FE_H1P1 && L.N == F.N && L.ncomp == 1 && F.ncomp == 1;
            const bool p1 = F.fe == GRMP_FE_H1P1 && L.fe == GRMP_FE_H1P1 && L.N == (F.N + 1) / 2 && L.ncomp == F.ncomp;
            GRMP_CHECK(ctx, p2 || p1, GRMP_ERR_ARG, "multigrid: level %d does not coarsen level %d", l, l - 1);
        }
    }
    GRMP_CHECK(ctx, in[nlev - 1].A->n <= MG_DENSE_MAX, GRMP_ERR_ARG, "multigrid: coarsest level has %lld > %d dofs",
               (long long)in[nlev - 1].A->n, MG_DENSE_MAX);
    MgJob *j = new MgJob();
    j->ctx = ctx;
    j->st = st;
    j->nlev = nlev;
    j->profile = profile;
    j->use_graph = graph && !profile;  // events cannot be recorded inside a stream capture
    for (int l = 0; l < nlev; ++l) {
        j->lv[l].in = in[l];
        j->lv[l].n = in[l].A->n;
        j->lv[l].nnz = in[l].A->nnz;
        j->lv[l].nc = in[l].sp->mesh->ncells;
    }
    {
        int64_t rows[MG_MAX_LEVELS];
        for (int l = 0; l < nlev; ++l) rows[l] = j->lv[l].n;
        j->first_small = mg_first_small(rows, nlev, block_rows, coarse_rows);
    }
    // a coarse end that does not fit LDS gives its finest levels to grid
    // kernels: six launches of about 4.5 us against the 104 us that elasticity's
    // 1,250 ... 32 rows took in device memory
    MgPack P;
    bool fits = mg_job_pack_layout(j, P);
    while (!fits && j->first_small > 0 && j->first_small < nlev - 1) {
        ++j->first_small;
        fits = mg_job_pack_layout(j, P);
    }
    j->img_bytes = fits ? P.image : 0;
    j->bytes = mg_layout(j, false);
    hipError_t e = ctx_malloc(ctx, (void **)&j->buf, j->bytes, st);
    if (e != hipSuccess) {
        delete j;
        return grmp_fail(ctx, e == hipErrorOutOfMemory ? GRMP_ERR_OOM : GRMP_ERR_HIP, "multigrid: device buffer");
    }
    mg_layout(j, true);
    fill_desc(j);
    if (mg_allow_lds(ctx, (const void *)k_mg_vcycle_block) || mg_allow_lds(ctx, (const void *)k_mg_pcg_block) ||
        mg_allow_lds(ctx, (const void *)k_mgb_vcycle_block) || mg_allow_lds(ctx, (const void *)k_mgb_pcg_block)) {
        (void)hipFreeAsync(j->buf, st);
        delete j;
        return GRMP_ERR_HIP;
    }
    if (hipEventCreateWithFlags(&j->ev, hipEventDisableTiming) != hipSuccess) {
        (void)hipFreeAsync(j->buf, st);
        delete j;
        return grmp_fail(ctx, GRMP_ERR_HIP, "multigrid: event");
    }
    *out = j;
    return GRMP_OK;
}

double *mg_job_kappa0(MgJob *j) { return j->lv[0].kappa; }
double *mg_job_rhs(MgJob *j) { return j->rhs; }
const double *mg_job_solution(const MgJob *j) { return j->x; }

static void rows_args(MgRows &a, const MgLevel &L, const MgJob *j)
{
    memset(&a, 0, sizeof(a));
    a.rp = L.in.A->rowptr;
    a.ci = L.in.A->cols;
    a.val = L.val;
    a.val32 = L.val32;
    a.fixed = L.in.A->fixed;
    a.n = L.n;
    a.dinv = L.dinv;
    a.ch = L.ch;
    a.sc = j->sc;
}

// Residuals on levels of at least MG_FINE_ROWS rows run as k_mg_resid_fine;
// when profiled, each such launch carries a start / stop event pair bound to
// its own dispatch (hipExtLaunchKernelGGL), kept with its algorithmic bytes:
// values and columns, row pointers, x gathered once, b read, r written, mask.
template <int OP>
static void launch_rows(MgJob *j, const MgRows &a, int64_t nnz = 0)
{
    if (OP == OP_RESID && a.n >= MG_FINE_ROWS) {
        if (!j->profile) {
            hipLaunchKernelGGL(k_mg_resid_fine, dim3(nblk(a.n, KB)), dim3(KB), 0, j->st, a);
            return;
        }
        hipEvent_t e0, e1;
        if (!ev_take(j->pool, e0, e1)) {
            hipLaunchKernelGGL(k_mg_resid_fine, dim3(nblk(a.n, KB)), dim3(KB), 0, j->st, a);
            return;
        }
        hipExtLaunchKernelGGL(k_mg_resid_fine, dim3(nblk(a.n, KB)), dim3(KB), 0, j->st, e0, e1, 0, a);
        j->pev.push_back(e0);
        j->pev.push_back(e1);
        // FP32 values + int32 columns, row pointers, x gathered once, b, r, mask
        j->pbytes.push_back((double)nnz * 8.0 + 4.0 * (a.n + 1) + 24.0 * a.n + 1.0 * a.n);
        return;
    }
    hipLaunchKernelGGL(k_mg_rows<OP>, dim3(nblk(a.n, KB)), dim3(KB), 0, j->st, a);
}

// restriction of level l's residual r_l into b_{l+1}
static void mg_restrict(MgJob *j, int l)
{
    const MgLevel &F = j->lv[l], &C = j->lv[l + 1];
    if (F.in.fe == GRMP_FE_H1P2)
        hipLaunchKernelGGL(k_mg_restrict_p2, dim3(nblk(C.n, 256)), dim3(256), 0, j->st, (int64_t)F.in.N, F.r,
                           C.in.A->fixed, C.dinv, C.ch, C.b, C.d, j->sc);
    else
        hipLaunchKernelGGL(k_mg_restrict_p1, dim3(nblk(C.n, 256)), dim3(256), 0, j->st, (int64_t)F.in.N,
                           (int64_t)C.in.N, F.in.ncomp, F.r, C.in.A->fixed, C.dinv, C.ch, C.b, C.d, j->sc);
}

static void mg_prolong(MgJob *j, int l)
{
    const MgLevel &F = j->lv[l], &C = j->lv[l + 1];
    if (F.in.fe == GRMP_FE_H1P2) {
        const grmp_mesh *m = F.in.sp->mesh;
        const int64_t nn = m->nnodes, nc = m->ncells;
        hipLaunchKernelGGL(k_mg_prolong_p2, dim3(nblk(std::max(nn, nc), 256)), dim3(256), 0, j->st, (int64_t)F.in.N,
                           m->cells, m->fsign, C.x, F.in.A->fixed, F.x, j->sc);
    } else {
        hipLaunchKernelGGL(k_mg_prolong_p1, dim3(nblk(F.n, 256)), dim3(256), 0, j->st, (int64_t)F.in.N,
                           (int64_t)C.in.N, F.in.ncomp, C.x, F.in.A->fixed, F.x, j->sc);
    }
}

// x_0 (= z) = V(b_0 (= r)), d_0 holding d0 of r; the level-0 block partials of r.z land in part.
// Levels below first_small run as grid kernels, the rest in one workgroup.
static void mg_vcycle(MgJob *j)
{
    const int F = j->first_small;
    for (int l = 0; l < F; ++l) {
        MgLevel &L = j->lv[l];
        MgRows a;
        rows_args(a, L, j);
        a.v = L.d;
        a.b = L.b;
        a.o1 = L.x;
        launch_rows<OP_CHEB_PRE>(j, a);
        rows_args(a, L, j);
        a.v = L.x;
        a.b = L.b;
        a.o1 = L.r;
        launch_rows<OP_RESID>(j, a, L.nnz);
        mg_restrict(j, l);
    }
    hipLaunchKernelGGL(k_mg_vcycle_block, dim3(1), dim3(MG_BT), j->hdesc.pack.lds, j->st, j->ddesc, j->sc);
    for (int l = F - 1; l >= 0; --l) {
        MgLevel &L = j->lv[l];
        mg_prolong(j, l);
        MgRows a;
        rows_args(a, L, j);
        a.v = L.x;
        a.b = L.b;
        a.o1 = L.d;
        a.o2 = L.r;
        launch_rows<OP_CHEB_POST1>(j, a);
        rows_args(a, L, j);
        a.v = L.r;
        a.b = L.b;
        a.d = L.d;
        a.o1 = L.x;
        a.part = l == 0 ? j->part : nullptr;
        launch_rows<OP_CHEB_POST2>(j, a);
    }
}

static bool mg_job_p1(const MgJob *j) { return j->lv[0].in.fe == GRMP_FE_H1P1 && j->lv[0].in.ncomp == 1; }

double mg_job_margin(const MgJob *j) { return mg_job_p1(j) ? CHEB_FOURTH_MARGIN : 1.0; }

// FP32 values and Gershgorin bounds of all levels
static void mg_job_prep(MgJob *j)
{
    MgPrep P;
    P.nlev = P.blocks = 0;
    for (int l = 0; l < j->nlev; ++l) {
        MgLevel &L = j->lv[l];
        mg_prep_add(P, L.in.A->rowptr, L.val, L.dinv, L.in.A->fixed, L.val32, L.ch, L.n, mg_job_p1(j));
    }
    mg_prep_launch(P, j->st);
    j->fourth = mg_job_p1(j);
}

// the hierarchy's coefficients for CG (fourth) or as MINRES' preconditioner,
// if they are not those already
static int mg_job_kind(MgJob *j, bool fourth)
{
    if (!mg_job_p1(j) || fourth == j->fourth) return GRMP_OK;
    MgChebSet P;
    P.n = 0;
    P.fourth = fourth ? 1 : 0;
    for (int l = 0; l < j->nlev; ++l) P.ch[P.n++] = j->lv[l].ch;
    for (int k = 0; k < j->hdesc.pack.nlev; ++k)
        P.ch[P.n++] = reinterpret_cast<MgCheb *>(j->img + j->hdesc.pack.lv[k].ch);
    hipLaunchKernelGGL(k_mg_cheb_kind, dim3(1), dim3(64), 0, j->st, P);
    GRMP_HIP(j->ctx, hipGetLastError());
    j->fourth = fourth;
    return GRMP_OK;
}

// level values, smoother bounds and the coarsest inverse: once per operator
static int mg_job_assemble(MgJob *j)
{
    grmp_ctx *ctx = j->ctx;
    hipStream_t st = j->st;
    for (int l = 0; l < j->nlev; ++l) {
        MgLevel &L = j->lv[l];
        if (l > 0 && L.in.N != j->lv[l - 1].in.N)
            hipLaunchKernelGGL(k_mg_coarse_kappa, dim3(nblk(L.nc, 256)), dim3(256), 0, st, (int64_t)j->lv[l - 1].in.N,
                               (int64_t)L.in.N, j->lv[l - 1].kappa, L.kappa);
        GRMP_TRY(assemble_values(L.in.A, L.kappa, L.dforms, L.hforms, L.val, nullptr, L.dinv, L.dinv32, st));
    }
    mg_job_prep(j);
    const MgLevel &C = j->lv[j->nlev - 1];
    hipLaunchKernelGGL(k_mg_dense_inv, dim3(1), dim3(256), 0, st, C.in.A->rowptr, C.in.A->cols, C.val, C.in.A->fixed,
                       (int)C.n, j->inv);
    mg_job_pack(j);
    GRMP_HIP(ctx, hipMemcpyAsync(j->ddesc, &j->hdesc, sizeof(MgBDesc), hipMemcpyHostToDevice, st));
    return GRMP_OK;
}

// Krylov state for the right-hand side in mg_job_rhs: scalars reset,
// x = 0, r = rhs (0 on fixed rows), z = V(r), p = 0 then p = z
static int mg_job_start(MgJob *j, double rtol, int maxit)
{
    grmp_ctx *ctx = j->ctx;
    hipStream_t st = j->st;
    GRMP_TRY(mg_job_kind(j, true));
    MgScal s0;
    memset(&s0, 0, sizeof(s0));
    s0.rtol = rtol;
    s0.rstop = rtol * mg_job_margin(j);
    s0.maxit = maxit;
    GRMP_HIP(ctx, hipMemcpyAsync(j->sc, &s0, sizeof(s0), hipMemcpyHostToDevice, st));
    const int64_t n = j->lv[0].n;
    GRMP_HIP(ctx, hipMemsetAsync(j->x, 0, n * 8, st));
    GRMP_HIP(ctx, hipMemsetAsync(j->p, 0, n * 8, st));
    hipLaunchKernelGGL(k_mg_start, dim3(nblk(n, 256)), dim3(256), 0, st, j->rhs, j->lv[0].in.A->fixed, j->lv[0].dinv,
                       j->lv[0].ch, j->r, j->lv[0].d, n);
    mg_vcycle(j);
    hipLaunchKernelGGL(k_mg_dot, dim3(j->nb0), dim3(KB), 0, st, j->r, j->r, n, j->part2, j->sc);
    hipLaunchKernelGGL(k_mg_red<RED_INIT>, dim3(1), dim3(MG_BT), 0, st, j->part, j->nb0, j->part2, j->sc);
    hipLaunchKernelGGL(k_mg_update_p, dim3(nblk(n, 256)), dim3(256), 0, st, j->p, j->z, n, j->sc);
    GRMP_HIP(ctx, hipGetLastError());
    return GRMP_OK;
}

int mg_job_setup(MgJob *j, double rtol, int maxit)
{
    GRMP_TRY(mg_job_assemble(j));
    return mg_job_start(j, rtol, maxit);
}

static int mg_iterate_grid(MgJob *j, int iters);

int mg_job_iterate(MgJob *j, int iters)
{
    if (j->first_small == 0) {  // every level fits one workgroup: whole iterations in one launch
        hipLaunchKernelGGL(k_mg_pcg_block, dim3(1), dim3(MG_BT), j->hdesc.pack.lds, j->st, j->ddesc, j->sc, iters);
        GRMP_HIP(j->ctx, hipGetLastError());
        return GRMP_OK;
    }
    if (!j->use_graph) return mg_iterate_grid(j, iters);
    if (!j->gexec || j->graph_iters != iters) {
        if (j->gexec) (void)hipGraphExecDestroy(j->gexec);
        if (j->graph) (void)hipGraphDestroy(j->graph);
        j->gexec = nullptr;
        j->graph = nullptr;
        mg_job_collect(j);  // profiled launches made before the capture
        for (hipEvent_t e : j->pev) j->pool.push_back(e);
        j->pev.clear();
        j->pbytes.clear();
        GRMP_HIP(j->ctx, hipStreamBeginCapture(j->st, hipStreamCaptureModeThreadLocal));
        const int rc = mg_iterate_grid(j, iters);
        hipGraph_t g = nullptr;
        const hipError_t e = hipStreamEndCapture(j->st, &g);
        GRMP_TRY(rc);
        GRMP_HIP(j->ctx, e);
        j->graph = g;
        GRMP_HIP(j->ctx, hipGraphInstantiate(&j->gexec, j->graph, nullptr, nullptr, 0));
        j->graph_iters = iters;
    }
    GRMP_HIP(j->ctx, hipGraphLaunch(j->gexec, j->st));
    return GRMP_OK;
}

// the grid-path iterations as individual launches (no memset or host sync:
// the sequence can be captured)
static int mg_iterate_grid(MgJob *j, int iters)
{
    const MgLevel &L0 = j->lv[0];
    const int64_t n = L0.n;
    for (int k = 0; k < iters; ++k) {
        MgRows a;
        rows_args(a, L0, j);
        a.v = j->p;
        a.o1 = j->q;
        a.part = j->part;
        launch_rows<OP_PCG_Q>(j, a);
        hipLaunchKernelGGL(k_mg_red<RED_ALPHA>, dim3(1), dim3(MG_BT), 0, j->st, j->part, j->nb0, nullptr, j->sc);
        hipLaunchKernelGGL(k_mg_axpy, dim3(j->nb0), dim3(KB), 0, j->st, j->x, j->r, j->p, j->q, L0.in.A->fixed,
                           L0.dinv, L0.ch, L0.d, n, j->part, j->sc);
        hipLaunchKernelGGL(k_mg_red<RED_CONV>, dim3(1), dim3(MG_BT), 0, j->st, j->part, j->nb0, nullptr, j->sc);
        mg_vcycle(j);
        hipLaunchKernelGGL(k_mg_red<RED_BETA>, dim3(1), dim3(MG_BT), 0, j->st, j->part, j->nb0, nullptr, j->sc);
        hipLaunchKernelGGL(k_mg_update_p, dim3(nblk(n, 256)), dim3(256), 0, j->st, j->p, j->z, n, j->sc);
    }
    GRMP_HIP(j->ctx, hipGetLastError());
    return GRMP_OK;
}

// The updated residual met rtol: replace it by the true residual b - A x;
// accept if that meets rtol too, else restart CG from it (p = z), at most
// three times and only while each check halves the previous one.
bool mg_job_block(const MgJob *j) { return j->first_small == 0; }

// moves a set-up job to another stream (the caller has ordered it after the
// job's work on the old one); its later launches and its release go there
void mg_job_set_stream(MgJob *j, hipStream_t st) { j->st = st; }

// p = z = V r of the true residual r
static void mg_job_restart_from(MgJob *j)
{
    const int64_t n = j->lv[0].n;
    mg_vcycle(j);
    hipLaunchKernelGGL(k_mg_red<RED_RESTART>, dim3(1), dim3(MG_BT), 0, j->st, j->part, j->nb0, nullptr, j->sc);
    hipLaunchKernelGGL(k_mg_update_p, dim3(nblk(n, 256)), dim3(256), 0, j->st, j->p, j->z, n, j->sc);
}

int mg_job_verify(MgJob *j)
{
    if (j->first_small == 0) return GRMP_OK;  // k_mg_pcg_block checks in place
    // with a captured chunk, event pairs are kept for replays: the check's
    // launches stay out of the profiled set then
    struct Unprofiled {
        MgJob *j;
        bool was;
        ~Unprofiled() { j->profile = was; }
    } guard{j, j->profile};
    if (j->gexec) j->profile = false;
    const MgLevel &L0 = j->lv[0];
    hipLaunchKernelGGL(k_mg_verify_begin, dim3(1), dim3(1), 0, j->st, j->sc);
    MgRows a;
    rows_args(a, L0, j);
    a.v = j->x;
    a.b = j->rhs;
    a.o1 = j->r;
    a.o2 = L0.d;
    a.part = j->part;
    launch_rows<OP_TRUE_RESID>(j, a, L0.nnz);
    hipLaunchKernelGGL(k_mg_red<RED_VERIFY>, dim3(1), dim3(MG_BT), 0, j->st, j->part, j->nb0, nullptr, j->sc);
    mg_job_restart_from(j);
    GRMP_HIP(j->ctx, hipGetLastError());
    return GRMP_OK;
}

// the restart that a batch's check asked for (done 3)
int mg_job_restart(MgJob *j)
{
    hipLaunchKernelGGL(k_mg_verify_begin, dim3(1), dim3(1), 0, j->st, j->sc);
    mg_job_restart_from(j);
    GRMP_HIP(j->ctx, hipGetLastError());
    return GRMP_OK;
}

int mg_job_status_async(MgJob *j, MgStatus *host)
{
    static_assert(sizeof(MgStatus) == 24, "MgStatus layout");
    MgStatus *dst = host;
    // relres, then it / done / status as laid out in MgScal
    GRMP_HIP(j->ctx, hipMemcpyAsync(&dst->relres, &j->sc->relres, 8, hipMemcpyDeviceToHost, j->st));
    GRMP_HIP(j->ctx, hipMemcpyAsync(&dst->it, &j->sc->it, 12, hipMemcpyDeviceToHost, j->st));
    GRMP_HIP(j->ctx, hipEventRecord(j->ev, j->st));
    return GRMP_OK;
}

bool mg_job_status_ready(MgJob *j) { return hipEventQuery(j->ev) != hipErrorNotReady; }

int mg_job_wait(MgJob *j)
{
    GRMP_HIP(j->ctx, hipEventSynchronize(j->ev));
    return GRMP_OK;
}

// Adds the timings of the profiled launches whose work has completed (the
// caller saw the status event of the chunk): a replayed graph keeps its event
// pairs for the next replay, individually launched ones are released.
void mg_job_collect(MgJob *j)
{
    if (!j->profile) return;
    for (size_t k = 0; k + 1 < j->pev.size(); k += 2) {
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, j->pev[k], j->pev[k + 1]) != hipSuccess) continue;
        j->prof_s += ms * 1e-3;
        j->prof_bytes += j->pbytes[k / 2];
        j->prof_launches += 1;
    }
    if (j->gexec) return;
    for (hipEvent_t e : j->pev) j->pool.push_back(e);
    j->pev.clear();
    j->pbytes.clear();
}

void mg_job_profile(MgJob *j, double *seconds, double *bytes, int64_t *launches)
{
    *seconds = j->prof_s;
    *bytes = j->prof_bytes;
    *launches = j->prof_launches;
}

void mg_job_destroy(MgJob *j)
{
    if (!j) return;
    if (j->gexec) (void)hipGraphExecDestroy(j->gexec);
    if (j->graph) (void)hipGraphDestroy(j->graph);
    for (hipEvent_t e : j->pev) (void)hipEventDestroy(e);
    for (hipEvent_t e : j->pool) (void)hipEventDestroy(e);
    if (j->ev) (void)hipEventDestroy(j->ev);
    if (j->buf) (void)hipFreeAsync(j->buf, j->st);
    delete j;
}

// ---------------------------------------------------- lockstep batch (host)
struct MgSeg {
    int64_t off = 0, cnt = 0;
};

struct MgBatch {
    grmp_ctx *ctx = nullptr;
    hipStream_t st = nullptr;
    bool profile = false;
    // device tables and their pinned staging (rewritten each run, after the previous run's wait)
    MgTile *dtiles = nullptr, *htiles = nullptr;
    size_t tcap = 0;
    const MgBDesc **ddesc = nullptr, **hdesc = nullptr;
    int32_t *dreq = nullptr, *hreq = nullptr;
    MgStatus *dstat = nullptr, *hstat = nullptr;
    int rcap = 0;
    hipEvent_t ev = nullptr;
    // profile: event pairs around each batched residual launch, with its bytes
    std::vector<hipEvent_t> pev, pool;  // profiled launches in flight; free events
    std::vector<double> pbytes;
    double prof_s = 0.0, prof_bytes = 0.0;
    int64_t prof_launches = 0;
};

int mg_batch_create(grmp_ctx *ctx, hipStream_t st, bool profile, MgBatch **out)
{
    MgBatch *b = new MgBatch();
    b->ctx = ctx;
    b->st = st;
    b->profile = profile;
    if (hipEventCreateWithFlags(&b->ev, hipEventDisableTiming) != hipSuccess) {
        delete b;
        return grmp_fail(ctx, GRMP_ERR_HIP, "multigrid batch: event");
    }
    *out = b;
    return GRMP_OK;
}

static int batch_reserve(MgBatch *b, size_t tiles, int reqs)
{
    grmp_ctx *ctx = b->ctx;
    if (tiles > b->tcap) {
        const size_t cap = std::max(tiles, b->tcap * 2);
        if (b->dtiles) (void)hipFreeAsync(b->dtiles, b->st);
        if (b->htiles) {
            (void)hipStreamSynchronize(b->st);
            (void)hipHostFree(b->htiles);
        }
        b->dtiles = nullptr;
        b->htiles = nullptr;
        GRMP_HIP(ctx, ctx_malloc(ctx, (void **)&b->dtiles, cap * sizeof(MgTile), b->st));
        GRMP_HIP(ctx, hipHostMalloc((void **)&b->htiles, cap * sizeof(MgTile), hipHostMallocDefault));
        b->tcap = cap;
    }
    if (reqs > b->rcap) {
        const int cap = std::max(reqs, 2 * b->rcap);
        (void)hipStreamSynchronize(b->st);
        if (b->ddesc) (void)hipFree((void *)b->ddesc);
        if (b->dreq) (void)hipFree(b->dreq);
        if (b->dstat) (void)hipFree(b->dstat);
        if (b->hdesc) (void)hipHostFree((void *)b->hdesc);
        if (b->hreq) (void)hipHostFree(b->hreq);
        if (b->hstat) (void)hipHostFree(b->hstat);
        GRMP_HIP(ctx, ctx_malloc_fixed(ctx, (void **)&b->ddesc, cap * sizeof(MgBDesc *)));
        GRMP_HIP(ctx, ctx_malloc_fixed(ctx, (void **)&b->dreq, cap * sizeof(int32_t)));
        GRMP_HIP(ctx, ctx_malloc_fixed(ctx, (void **)&b->dstat, cap * sizeof(MgStatus)));
        GRMP_HIP(ctx, hipHostMalloc((void **)&b->hdesc, cap * sizeof(MgBDesc *), hipHostMallocDefault));
        GRMP_HIP(ctx, hipHostMalloc((void **)&b->hreq, cap * sizeof(int32_t), hipHostMallocDefault));
        GRMP_HIP(ctx, hipHostMalloc((void **)&b->hstat, cap * sizeof(MgStatus), hipHostMallocDefault));
        b->rcap = cap;
    }
    return GRMP_OK;
}

static inline unsigned ublk(int64_t n) { return (unsigned)n; }

// tile segments of the jobs grid: per grid level l its rows, the next level's
// rows (restriction), its prolongation items
struct MgBSegs {
    int Fmax = 0;
    std::vector<MgSeg> lev, res, pro;
};

static MgBSegs mgb_segs(MgJob *const *jobs, const std::vector<int> &grid, std::vector<MgTile> &T)
{
    MgBSegs S;
    for (int g : grid) S.Fmax = std::max(S.Fmax, jobs[g]->first_small);
    auto add = [&](MgSeg &sg, int lev, bool next, bool items) {
        sg.off = (int64_t)T.size();
        for (int g : grid) {
            const MgJob *j = jobs[g];
            if (j->first_small <= lev) continue;
            const int L = next ? lev + 1 : lev;
            int64_t cnt = j->lv[L].n;
            if (items && j->lv[lev].in.fe == GRMP_FE_H1P2) {
                const int64_t N = j->lv[lev].in.N;
                cnt = std::max((N + 1) * (N + 1), 2 * N * N);
            }
            for (int64_t r0 = 0; r0 < cnt; r0 += (int64_t)KB * MG_TILE_CHUNKS) T.push_back(MgTile{g, L, (int32_t)r0, 0});
        }
        sg.cnt = (int64_t)T.size() - sg.off;
    };
    S.lev.resize(S.Fmax);
    S.res.resize(S.Fmax);
    S.pro.resize(S.Fmax);
    for (int l = 0; l < S.Fmax; ++l) {
        add(S.lev[l], l, false, false);
        add(S.res[l], l, true, false);
        add(S.pro[l], l, false, true);
    }
    return S;
}

// one V-cycle of the requests: the grid levels of those in grid over the
// tiles dt, the coarse ends of the nr requests R; b: profile its residuals
static void mgb_vcycle(MgBatch *b, hipStream_t st, MgJob *const *jobs, const std::vector<int> &grid, const MgBSegs &S,
                       const MgTile *dt, const MgBDesc *const *D, const int32_t *R, int nr, int lds)
{
    const std::vector<MgSeg> &lev = S.lev, &res = S.res, &pro = S.pro;
    const int Fmax = S.Fmax;
    auto tiles = [&](const MgSeg &sg) { return dt + sg.off; };
    for (int l = 0; l < Fmax; ++l) {
        if (lev[l].cnt == 0) continue;
        hipLaunchKernelGGL(k_mgb_rows<OP_CHEB_PRE>, dim3(ublk(lev[l].cnt)), dim3(KB), 0, st, tiles(lev[l]), D);
        hipEvent_t e0, e1;
        if (b && b->profile && ev_take(b->pool, e0, e1)) {
            hipExtLaunchKernelGGL(k_mgb_rows<OP_RESID>, dim3(ublk(lev[l].cnt)), dim3(KB), 0, st, e0, e1, 0,
                                  tiles(lev[l]), D);
            b->pev.push_back(e0);
            b->pev.push_back(e1);
            double bytes = 0.0;
            for (int g : grid)
                if (jobs[g]->first_small > l) {
                    const MgLevel &Lv = jobs[g]->lv[l];
                    bytes += (double)Lv.nnz * 8.0 + 4.0 * (Lv.n + 1) + 25.0 * Lv.n;
                }
            b->pbytes.push_back(bytes);
        } else {
            hipLaunchKernelGGL(k_mgb_rows<OP_RESID>, dim3(ublk(lev[l].cnt)), dim3(KB), 0, st, tiles(lev[l]), D);
        }
        hipLaunchKernelGGL(k_mgb_restrict, dim3(ublk(res[l].cnt)), dim3(KB), 0, st, tiles(res[l]), D);
    }
    hipLaunchKernelGGL(k_mgb_vcycle_block, dim3(nr), dim3(MG_BT), lds, st, D, R);
    for (int l = Fmax - 1; l >= 0; --l) {
        if (lev[l].cnt == 0) continue;
        hipLaunchKernelGGL(k_mgb_prolong, dim3(ublk(pro[l].cnt)), dim3(KB), 0, st, tiles(pro[l]), D);
        hipLaunchKernelGGL(k_mgb_rows<OP_CHEB_POST1>, dim3(ublk(lev[l].cnt)), dim3(KB), 0, st, tiles(lev[l]), D);
        hipLaunchKernelGGL(k_mgb_rows<OP_CHEB_POST2>, dim3(ublk(lev[l].cnt)), dim3(KB), 0, st, tiles(lev[l]), D);
    }
}

// The setup of many jobs (on the stream st), each step one launch for all:
// coarse coefficients by depth, the assembly of every level (assemble_batch,
// the same values as mg_job_assemble's per-level launches), level values and
// bounds, coarsest inverses, LDS images, descriptors, and the start of CG with
// the first V-cycle (as mg_job_start).  A job at a time these were some 60
// small launches and copies each; 48 requests had a full batch 30 ms after they
// came, now 8, and take 92.5 ms where they took 94.4.
int mg_jobs_setup_batched(MgJob *const *jobs, int n, hipStream_t st, double *const rtol, int maxit)
{
    if (n <= 0) return GRMP_OK;
    grmp_ctx *ctx = jobs[0]->ctx;
    std::vector<AsmBatchItem> items;
    std::vector<std::vector<MgKapEntry>> kap;
    std::vector<int> kapblk;
    std::vector<MgPrepLevel> prep;
    std::vector<MgInvEntry> inv;
    std::vector<MgPackEntry> pack;
    std::vector<MgInitEntry> init(n);
    std::vector<const MgBDesc *> dp;
    std::vector<int32_t> reqs;
    std::vector<MgTile> T;
    std::vector<int> grid;
    int prepblk = 0, packblk = 0, lds = 0;
    for (int k = 0; k < n; ++k) {
        MgJob *j = jobs[k];
        GRMP_CHECK(ctx, j->st == st, GRMP_ERR_ARG, "batched multigrid setup: jobs on different streams");
        size_t depth = 0;
        for (int l = 0; l < j->nlev; ++l) {
            MgLevel &L = j->lv[l];
            if (l > 0 && L.in.N != j->lv[l - 1].in.N) {
                if (depth == kap.size()) {
                    kap.emplace_back();
                    kapblk.push_back(0);
                }
                kap[depth].push_back(MgKapEntry{j->lv[l - 1].kappa, L.kappa, j->lv[l - 1].in.N, L.in.N, kapblk[depth], 0});
                kapblk[depth] += (int)nblk(L.nc, KB);
                ++depth;
            }
            items.push_back(AsmBatchItem{L.in.A, L.kappa, L.val, L.dinv, L.dinv32});
            prep.push_back(MgPrepLevel{L.in.A->rowptr, L.val, L.dinv, L.in.A->fixed, L.val32, L.ch, L.n, prepblk,
                                       mg_job_p1(j) ? 1 : 0});
            prepblk += (int)nblk(L.n, KB);
        }
        j->fourth = mg_job_p1(j);
        const MgLevel &C = j->lv[j->nlev - 1];
        inv.push_back(MgInvEntry{C.in.A->rowptr, C.in.A->cols, C.val, C.in.A->fixed, j->inv, C.n});
        const MgPack &P = j->hdesc.pack;
        lds = std::max(lds, P.lds);
        for (int q = 0; q < P.nlev; ++q) {
            pack.push_back(MgPackEntry{P.lv[q], mg_pack_src(j, q), j->img, packblk, 0});
            const MgLevel &L = j->lv[j->first_small + q];
            packblk += (int)nblk(std::max(L.nnz, L.n + 1), KB);
        }
        MgInitEntry &e = init[k];
        e.D = j->hdesc;
        memset(&e.s, 0, sizeof(e.s));
        e.s.rtol = rtol[k];
        e.s.rstop = rtol[k] * mg_job_margin(j);
        e.s.maxit = maxit;
        e.ddesc = j->ddesc;
        e.sc = j->sc;
        dp.push_back(j->ddesc);
        reqs.push_back(k);
        if (j->first_small > 0) grid.push_back(k);
    }
    const MgBSegs sg = mgb_segs(jobs, grid, T);
    MgSeg all;  // level-0 tiles of every job
    all.off = (int64_t)T.size();
    for (int k = 0; k < n; ++k)
        for (int64_t r0 = 0; r0 < jobs[k]->lv[0].n; r0 += (int64_t)KB * MG_TILE_CHUNKS)
            T.push_back(MgTile{k, 0, (int32_t)r0, 0});
    all.cnt = (int64_t)T.size() - all.off;

    std::vector<char> h;
    auto put = [&](const void *p, size_t bytes) {
        const size_t o = h.size();
        h.resize(al256(o + bytes));
        memcpy(h.data() + o, p, bytes);
        return o;
    };
    std::vector<size_t> o_kap;
    for (auto &k : kap) o_kap.push_back(put(k.data(), k.size() * sizeof(MgKapEntry)));
    const size_t o_prep = put(prep.data(), prep.size() * sizeof(MgPrepLevel));
    const size_t o_inv = put(inv.data(), inv.size() * sizeof(MgInvEntry));
    const size_t o_pack = put(pack.data(), pack.size() * sizeof(MgPackEntry));
    const size_t o_init = put(init.data(), init.size() * sizeof(MgInitEntry));
    const size_t o_dp = put(dp.data(), dp.size() * sizeof(const MgBDesc *));
    const size_t o_reqs = put(reqs.data(), reqs.size() * sizeof(int32_t));
    const size_t o_T = put(T.data(), T.size() * sizeof(MgTile));
    char *d = nullptr;
    GRMP_HIP(ctx, ctx_malloc(ctx, (void **)&d, h.size(), st));
    auto run = [&]() -> int {
        GRMP_HIP(ctx, hipMemcpyAsync(d, h.data(), h.size(), hipMemcpyHostToDevice, st));
        for (size_t k = 0; k < kap.size(); ++k)
            hipLaunchKernelGGL(k_mgb_coarse_kappa, dim3(kapblk[k]), dim3(KB), 0, st, (const MgKapEntry *)(d + o_kap[k]),
                               (int)kap[k].size());
        GRMP_HIP(ctx, hipGetLastError());
        GRMP_TRY(assemble_batch(ctx, st, items.data(), (int)items.size()));
        const int np = (int)prep.size(), nk = (int)pack.size();
        hipLaunchKernelGGL(k_mgb_prep_cheb, dim3(nblk(np, 64)), dim3(64), 0, st, (const MgPrepLevel *)(d + o_prep), np);
        hipLaunchKernelGGL(k_mgb_prep, dim3(prepblk), dim3(KB), 0, st, (const MgPrepLevel *)(d + o_prep), np);
        hipLaunchKernelGGL(k_mgb_dense_inv, dim3(n), dim3(256), 0, st, (const MgInvEntry *)(d + o_inv));
        if (nk > 0)
            hipLaunchKernelGGL(k_mgb_pack, dim3(packblk), dim3(KB), 0, st, (const MgPackEntry *)(d + o_pack), nk);
        hipLaunchKernelGGL(k_mgb_init, dim3(n), dim3(KB), 0, st, (const MgInitEntry *)(d + o_init));
        const MgBDesc *const *D = (const MgBDesc *const *)(d + o_dp);
        const MgTile *dt = (const MgTile *)(d + o_T);
        hipLaunchKernelGGL(k_mgb_start, dim3(ublk(all.cnt)), dim3(KB), 0, st, dt + all.off, D);
        mgb_vcycle(nullptr, st, jobs, grid, sg, dt, D, (const int32_t *)(d + o_reqs), n, lds);
        hipLaunchKernelGGL(k_mgb_red_init, dim3(n), dim3(MG_BT), 0, st, D);
        hipLaunchKernelGGL(k_mgb_update_p, dim3(ublk(all.cnt)), dim3(KB), 0, st, dt + all.off, D);
        GRMP_HIP(ctx, hipGetLastError());
        return GRMP_OK;
    };
    const int rc = run();
    // the upload reads h: on success assemble_batch, behind it, has waited for the stream
    if (rc) (void)hipStreamSynchronize(st);
    (void)hipFreeAsync(d, st);
    return rc;
}

// Enqueues iters lockstep iterations of the n jobs (all set up on the
// batch's stream), then a status copy for each job into mg_batch_status().
int mg_batch_run(MgBatch *b, MgJob *const *jobs, int n, int iters)
{
    grmp_ctx *ctx = b->ctx;
    hipStream_t st = b->st;
    std::vector<int> grid, blk;
    int lds_grid = 0, lds_blk = 0;  // LDS of the one-workgroup kernels: the largest of their jobs
    for (int i = 0; i < n; ++i) {
        const int lds = jobs[i]->hdesc.pack.lds;
        if (jobs[i]->first_small == 0) {
            blk.push_back(i);
            lds_blk = std::max(lds_blk, lds);
        } else {
            grid.push_back(i);
            lds_grid = std::max(lds_grid, lds);
        }
    }
    std::vector<MgTile> T;
    const MgBSegs sg = mgb_segs(jobs, grid, T);
    GRMP_TRY(batch_reserve(b, std::max<size_t>(T.size(), 1), std::max(n, 1)));
    memcpy(b->htiles, T.data(), T.size() * sizeof(MgTile));
    for (int i = 0; i < n; ++i) b->hdesc[i] = jobs[i]->ddesc;
    for (size_t k = 0; k < grid.size(); ++k) b->hreq[k] = grid[k];
    for (size_t k = 0; k < blk.size(); ++k) b->hreq[grid.size() + k] = blk[k];
    if (!T.empty())
        GRMP_HIP(ctx, hipMemcpyAsync(b->dtiles, b->htiles, T.size() * sizeof(MgTile), hipMemcpyHostToDevice, st));
    GRMP_HIP(ctx, hipMemcpyAsync((void *)b->ddesc, (const void *)b->hdesc, n * sizeof(MgBDesc *), hipMemcpyHostToDevice,
                                 st));
    GRMP_HIP(ctx, hipMemcpyAsync(b->dreq, b->hreq, n * sizeof(int32_t), hipMemcpyHostToDevice, st));
    const MgBDesc *const *D = b->ddesc;
    const int32_t *G = b->dreq, *Bk = b->dreq + grid.size();
    const int ng = (int)grid.size(), nbk = (int)blk.size();
    for (int k = 0; k < iters && ng > 0; ++k) {
        const MgSeg &L0 = sg.lev[0];
        const MgTile *T0 = b->dtiles + L0.off;
        hipLaunchKernelGGL(k_mgb_rows<OP_PCG_Q>, dim3(ublk(L0.cnt)), dim3(KB), 0, st, T0, D);
        hipLaunchKernelGGL(k_mgb_red<RED_ALPHA>, dim3(ng), dim3(MG_BT), 0, st, D, G);
        hipLaunchKernelGGL(k_mgb_axpy, dim3(ublk(L0.cnt)), dim3(KB), 0, st, T0, D);
        hipLaunchKernelGGL(k_mgb_red<RED_CONV>, dim3(ng), dim3(MG_BT), 0, st, D, G);
        mgb_vcycle(b, st, jobs, grid, sg, b->dtiles, D, G, ng, lds_grid);
        hipLaunchKernelGGL(k_mgb_red<RED_BETA>, dim3(ng), dim3(MG_BT), 0, st, D, G);
        hipLaunchKernelGGL(k_mgb_update_p, dim3(ublk(L0.cnt)), dim3(KB), 0, st, T0, D);
    }
    // the requests that met rtol are checked here, in two launches for all: one
    // after the other, each behind a status copy and with the V-cycle of a
    // restart that hardly any needs, they kept the batch waiting up to 4 ms at a
    // time (48 requests 92.5 -> 87.3 ms)
    if (ng > 0) {
        hipLaunchKernelGGL(k_mgb_true_resid, dim3(ublk(sg.lev[0].cnt)), dim3(KB), 0, st, b->dtiles + sg.lev[0].off, D);
        hipLaunchKernelGGL(k_mgb_red_verify, dim3(ng), dim3(MG_BT), 0, st, D, G);
    }
    if (nbk > 0) hipLaunchKernelGGL(k_mgb_pcg_block, dim3(nbk), dim3(MG_BT), lds_blk, st, D, Bk, iters);
    hipLaunchKernelGGL(k_mgb_status, dim3(nblk(n, 256)), dim3(256), 0, st, D, n, b->dstat);
    GRMP_HIP(ctx, hipMemcpyAsync(b->hstat, b->dstat, n * sizeof(MgStatus), hipMemcpyDeviceToHost, st));
    GRMP_HIP(ctx, hipEventRecord(b->ev, st));
    GRMP_HIP(ctx, hipGetLastError());
    return GRMP_OK;
}

int mg_batch_wait(MgBatch *b)
{
    GRMP_HIP(b->ctx, hipEventSynchronize(b->ev));
    for (size_t k = 0; k + 1 < b->pev.size(); k += 2) {
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, b->pev[k], b->pev[k + 1]) == hipSuccess) {
            b->prof_s += ms * 1e-3;
            b->prof_bytes += b->pbytes[k / 2];
            b->prof_launches += 1;
        }
        b->pool.push_back(b->pev[k]);
        b->pool.push_back(b->pev[k + 1]);
    }
    b->pev.clear();
    b->pbytes.clear();
    return GRMP_OK;
}

const MgStatus *mg_batch_status(const MgBatch *b) { return b->hstat; }

void mg_batch_profile(const MgBatch *b, double *seconds, double *bytes, int64_t *launches)
{
    *seconds = b->prof_s;
    *bytes = b->prof_bytes;
    *launches = b->prof_launches;
}

void mg_batch_destroy(MgBatch *b)
{
    if (!b) return;
    (void)hipStreamSynchronize(b->st);
    if (b->dtiles) (void)hipFree(b->dtiles);
    if (b->htiles) (void)hipHostFree(b->htiles);
    if (b->ddesc) (void)hipFree((void *)b->ddesc);
    if (b->dreq) (void)hipFree(b->dreq);
    if (b->dstat) (void)hipFree(b->dstat);
    if (b->hdesc) (void)hipHostFree((void *)b->hdesc);
    if (b->hreq) (void)hipHostFree(b->hreq);
    if (b->hstat) (void)hipHostFree(b->hstat);
    for (hipEvent_t e : b->pev) (void)hipEventDestroy(e);
    for (hipEvent_t e : b->pool) (void)hipEventDestroy(e);
    if (b->ev) (void)hipEventDestroy(b->ev);
    delete b;
}

// ------------------------------------------------- one multigrid solve
// The served path's V-cycle CG for one caller-built hierarchy: level 0 is
// the caller's system (its forms are assembled by the job with the job's
// own cell coefficient), coarser levels are rediscretizations on the unit
// squares of ceil(N/2) down to N <= 4.  The solution is 0 on fixed rows
// (homogeneous Dirichlet data).  A handle keeps the assembled hierarchy for
// further right-hand sides, as the reference keeps its factorization while
// the matrix is unchanged.  Iterations are chunked as in the server: status
// after each chunk, the true-residual check when the scalars ask.
struct grmp_mg {
    grmp_ctx *ctx;
    MgJob *job;
    MgStatus *h;  // pinned
    const grmp_matrix *A0;
    int64_t n;
    // a second copy of the hierarchy's values and vectors on a stream of its
    // own, so that two components' V-cycles run at the same time
    // (mg_precond_apply_pair); built on first use
    std::vector<MgLevelIn> in;
    MgJob *job2 = nullptr;
    hipStream_t st2 = nullptr;
    hipEvent_t fork = nullptr, join = nullptr;
};

extern "C" int grmp_mg_destroy(grmp_mg *m)
{
    if (!m) return GRMP_OK;
    if (m->job) {
        (void)hipStreamSynchronize(m->ctx->stream);
        mg_job_destroy(m->job);
        (void)hipStreamSynchronize(m->ctx->stream);
    }
    if (m->st2) {
        (void)hipStreamSynchronize(m->st2);
        if (m->job2) mg_job_destroy(m->job2);
        (void)hipStreamSynchronize(m->st2);
        (void)hipStreamDestroy(m->st2);
    }
    if (m->fork) (void)hipEventDestroy(m->fork);
    if (m->join) (void)hipEventDestroy(m->join);
    if (m->h) (void)hipHostFree(m->h);
    delete m;
    return GRMP_OK;
}

extern "C" int grmp_mg_create(grmp_ctx *ctx, int nlev, const grmp_matrix *const *levels,
                              const grmp_space *const *spaces, const grmp_vector *kappa0, grmp_mg **out)
{
    if (!ctx || !levels || !spaces || !kappa0 || !out) return GRMP_ERR_ARG;
    *out = nullptr;
    GRMP_CHECK(ctx, nlev >= 1 && nlev <= MG_MAX_LEVELS, GRMP_ERR_ARG, "grmp_mg_create: %d levels", nlev);
    for (int l = 0; l < nlev; ++l)
        GRMP_CHECK(ctx, levels[l] && spaces[l] && levels[l]->ctx == ctx && levels[l]->nblocks == 1 &&
                            levels[l]->spaces[0] == spaces[l],
                   GRMP_ERR_ARG, "grmp_mg_create: level %d is not a one-block matrix over its space", l);
    const grmp_mesh *m0 = spaces[0]->mesh;
    GRMP_CHECK(ctx, kappa0->ctx == ctx && kappa0->n == m0->ncells, GRMP_ERR_ARG,
               "grmp_mg_create: kappa0 needs one value per level-0 cell (%lld)", (long long)m0->ncells);
    std::vector<MgLevelIn> in(nlev);
    for (int l = 0; l < nlev; ++l)
        in[l] = MgLevelIn{levels[l], spaces[l], spaces[l]->mesh->N, spaces[l]->fe, spaces[l]->ncomp};
    std::lock_guard<std::mutex> g(ctx->mu);
    hipStream_t st = ctx->stream;
    grmp_mg *m = new grmp_mg{ctx, nullptr, nullptr, levels[0], levels[0]->n};
    m->in = in;
    int rc = GRMP_OK;
    do {
        if ((rc = mg_job_create(ctx, st, in.data(), nlev, false, 2048, 2048, false, &m->job))) break;
        if (hipHostMalloc((void **)&m->h, sizeof(MgStatus), hipHostMallocDefault) != hipSuccess) {
            rc = grmp_fail(ctx, GRMP_ERR_HIP, "grmp_mg_create: status buffer");
            break;
        }
        if (hipMemcpyAsync(mg_job_kappa0(m->job), kappa0->d, sizeof(double) * m0->ncells, hipMemcpyDeviceToDevice,
                           st) != hipSuccess) {
            rc = grmp_fail(ctx, GRMP_ERR_HIP, "grmp_mg_create: coefficient");
            break;
        }
        if ((rc = mg_job_assemble(m->job))) break;
        if (hipStreamSynchronize(st) != hipSuccess) rc = grmp_fail(ctx, GRMP_ERR_HIP, "grmp_mg_create: assembly");
    } while (0);
    if (rc) {
        grmp_mg_destroy(m);
        return rc;
    }
    *out = m;
    return GRMP_OK;
}

extern "C" int grmp_mg_apply(grmp_mg *m, const grmp_vector *b, grmp_vector *x, double rtol, int64_t maxit,
                             grmp_solve_info *info)
{
    if (!m || !b || !x) return GRMP_ERR_ARG;
    grmp_ctx *ctx = m->ctx;
    GRMP_CHECK(ctx, b->ctx == ctx && x->ctx == ctx && b->n == m->n && x->n == m->n && b->d != x->d, GRMP_ERR_ARG,
               "grmp_mg_apply: b and x need the level-0 length %lld and distinct storage", (long long)m->n);
    GRMP_CHECK(ctx, rtol > 0.0 && rtol < 1.0 && maxit >= 1 && maxit <= (1 << 30), GRMP_ERR_ARG,
               "grmp_mg_apply: rtol in (0, 1) and maxit >= 1 needed");
    std::lock_guard<std::mutex> g(ctx->mu);
    hipStream_t st = ctx->stream;
    const double t0 = wall_seconds();
    MgJob *j = m->job;
    MgStatus *h = m->h;
    memset(h, 0, sizeof(MgStatus));
    int rc = GRMP_OK;
    do {
        if (hipMemcpyAsync(mg_job_rhs(j), b->d, sizeof(double) * m->n, hipMemcpyDeviceToDevice, st) != hipSuccess) {
            rc = grmp_fail(ctx, GRMP_ERR_HIP, "grmp_mg_apply: right-hand side");
            break;
        }
        if ((rc = zero_fixed_launch(m->A0, mg_job_rhs(j), st))) break;
        if ((rc = mg_job_start(j, rtol, (int)maxit))) break;
        if ((rc = mg_job_iterate(j, 4)) || (rc = mg_job_status_async(j, h)) || (rc = mg_job_wait(j))) break;
        while (h->done != 1) {
            if (h->done == 2) {
                rc = mg_job_verify(j);
                if (!rc && mg_job_block(j)) rc = mg_job_iterate(j, 1);
            } else {
                rc = mg_job_iterate(j, 4);
            }
            if (rc || (rc = mg_job_status_async(j, h)) || (rc = mg_job_wait(j))) break;
        }
        if (rc) break;
        if (hipMemcpyAsync(x->d, mg_job_solution(j), sizeof(double) * m->n, hipMemcpyDeviceToDevice, st) !=
                hipSuccess ||
            hipStreamSynchronize(st) != hipSuccess)
            rc = grmp_fail(ctx, GRMP_ERR_HIP, "grmp_mg_apply: solution");
    } while (0);
    grmp_solve_info inf;
    memset(&inf, 0, sizeof(inf));
    inf.status = h->status;
    inf.iterations = h->it;
    inf.relres = h->relres;
    inf.outer = 1;
    inf.seconds = wall_seconds() - t0;
    if (info) *info = inf;
    if (rc) {
        (void)hipStreamSynchronize(st);
        return rc;
    }
    if (inf.status == GRMP_ERR_NOCONV)
        return grmp_fail(ctx, GRMP_ERR_NOCONV, "grmp_mg_apply: no convergence, relres %.3e after %lld iterations",
                         inf.relres, (long long)inf.iterations);
    return inf.status;
}

// ------------------------------------------- one V-cycle as a preconditioner
// r_0 = v with the fixed rows zeroed and d0 of it; the device scalars are
// reset so the V-cycle kernels run (a finished CG leaves done set)
__global__ void k_mg_pc_in(const double *__restrict__ v, const uint8_t *__restrict__ fixed,
                           const double *__restrict__ dinv, const MgCheb *__restrict__ ch, double *__restrict__ r,
                           double *__restrict__ d, MgScal *__restrict__ sc, int64_t n, const int *__restrict__ skip)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int sk = skip ? *skip : 0;  // skip: the V-cycle's kernels see a finished solve
    if (i == 0) {
        sc->done = sk ? 1 : 0;
        sc->status = 0;
    }
    if (i >= n || sk) return;
    const bool fx = fixed[i] != 0;
    const double ri = fx ? 0.0 : v[i];
    r[i] = ri;
    d[i] = cheb_first(fx, dinv[i], ri, *ch);
}

int64_t mg_level0_rows(const grmp_mg *m) { return m->n; }

// z = V v: one V-cycle of the hierarchy from a zero start on stream st (the
// hierarchy's own stream): symmetric and positive definite, so it can
// precondition MINRES as it does CG.  z and v are n-vectors of the level-0
// numbering; fixed rows of z are 0.
// the second hierarchy of mg_precond_apply_pair: the same levels assembled
// from the same coefficient, so its V-cycle gives the first one's bits
int mg_pair_prepare(grmp_mg *m)
{
    if (m->job2) return GRMP_OK;
    grmp_ctx *ctx = m->ctx;
    if (!m->st2 && hipStreamCreateWithFlags(&m->st2, hipStreamNonBlocking) != hipSuccess) {
        m->st2 = nullptr;
        return grmp_fail(ctx, GRMP_ERR_HIP, "multigrid pair: stream");
    }
    if ((!m->fork && hipEventCreateWithFlags(&m->fork, hipEventDisableTiming) != hipSuccess) ||
        (!m->join && hipEventCreateWithFlags(&m->join, hipEventDisableTiming) != hipSuccess))
        return grmp_fail(ctx, GRMP_ERR_HIP, "multigrid pair: events");
    MgJob *j2 = nullptr;
    GRMP_TRY(mg_job_create(ctx, m->st2, m->in.data(), (int)m->in.size(), false, 2048, 2048, false, &j2));
    int rc = GRMP_OK;
    // the first hierarchy's coefficient is complete on the context stream
    if (hipStreamSynchronize(ctx->stream) != hipSuccess ||
        hipMemcpyAsync(mg_job_kappa0(j2), mg_job_kappa0(m->job), sizeof(double) * m->in[0].sp->mesh->ncells,
                       hipMemcpyDeviceToDevice, m->st2) != hipSuccess)
        rc = grmp_fail(ctx, GRMP_ERR_HIP, "multigrid pair: coefficient");
    if (!rc) rc = mg_job_assemble(j2);
    if (!rc && hipStreamSynchronize(m->st2) != hipSuccess) rc = grmp_fail(ctx, GRMP_ERR_HIP, "multigrid pair: assembly");
    if (rc) {
        (void)hipStreamSynchronize(m->st2);
        mg_job_destroy(j2);
        return rc;
    }
    m->job2 = j2;
    return GRMP_OK;
}

// z = V(r), d0 of r in place, into the caller's z: level 0 works there (the
// cycle writes every row of it) unless the whole cycle is one workgroup's
static int mg_vcycle_into(MgJob *j, double *z)
{
    if (j->first_small == 0) {
        mg_vcycle(j);
        GRMP_HIP(j->ctx, hipMemcpyAsync(z, j->z, sizeof(double) * j->lv[0].n, hipMemcpyDeviceToDevice, j->st));
        return GRMP_OK;
    }
    double *own = j->lv[0].x;
    j->lv[0].x = z;
    mg_vcycle(j);
    j->lv[0].x = own;
    return GRMP_OK;
}

// z0 = V v0 on the hierarchy's stream st and z1 = V v1 on the second
// hierarchy's stream, at the same time; st waits for both
int mg_precond_apply_pair(grmp_mg *m, const double *v0, double *z0, const double *v1, double *z1, hipStream_t st)
{
    MgJob *j = m->job, *j2 = m->job2;
    const int64_t n = m->n;
    GRMP_CHECK(m->ctx, st == j->st && j2, GRMP_ERR_ARG, "multigrid preconditioner pair: not prepared");
    GRMP_TRY(mg_job_kind(j, false));
    GRMP_TRY(mg_job_kind(j2, false));
    GRMP_HIP(m->ctx, hipEventRecord(m->fork, st));
    GRMP_HIP(m->ctx, hipStreamWaitEvent(m->st2, m->fork, 0));
    hipLaunchKernelGGL(k_mg_pc_in, dim3(nblk(n, 256)), dim3(256), 0, m->st2, v1, m->A0->fixed, j2->lv[0].dinv,
                       j2->lv[0].ch, j2->r, j2->lv[0].d, j2->sc, n, nullptr);
    GRMP_TRY(mg_vcycle_into(j2, z1));
    hipLaunchKernelGGL(k_mg_pc_in, dim3(nblk(n, 256)), dim3(256), 0, st, v0, m->A0->fixed, j->lv[0].dinv,
                       j->lv[0].ch, j->r, j->lv[0].d, j->sc, n, nullptr);
    GRMP_TRY(mg_vcycle_into(j, z0));
    GRMP_HIP(m->ctx, hipEventRecord(m->join, m->st2));
    GRMP_HIP(m->ctx, hipStreamWaitEvent(st, m->join, 0));
    GRMP_HIP(m->ctx, hipGetLastError());
    return GRMP_OK;
}

int mg_precond_apply(grmp_mg *m, const double *v, double *z, hipStream_t st)
{
    MgJob *j = m->job;
    const int64_t n = m->n;
    GRMP_CHECK(m->ctx, st == j->st, GRMP_ERR_ARG, "multigrid preconditioner: not the hierarchy's stream");
    GRMP_TRY(mg_job_kind(j, false));
    hipLaunchKernelGGL(k_mg_pc_in, dim3(nblk(n, 256)), dim3(256), 0, st, v, m->A0->fixed, j->lv[0].dinv, j->lv[0].ch,
                       j->r, j->lv[0].d, j->sc, n, nullptr);
    GRMP_TRY(mg_vcycle_into(j, z));
    GRMP_HIP(m->ctx, hipGetLastError());
    return GRMP_OK;
}

extern "C" int grmp_mg_solve(grmp_ctx *ctx, int nlev, const grmp_matrix *const *levels,
                             const grmp_space *const *spaces, const grmp_vector *kappa0, const grmp_vector *b,
                             grmp_vector *x, double rtol, int64_t maxit, grmp_solve_info *info)
{
    grmp_mg *m = nullptr;
    GRMP_TRY(grmp_mg_create(ctx, nlev, levels, spaces, kappa0, &m));
    const int rc = grmp_mg_apply(m, b, x, rtol, maxit, info);
    grmp_mg_destroy(m);
    return rc;
}

// ================================================================ AMG
// Algebraic multigrid for symmetric positive definite systems on any mesh
// (the geometric hierarchy above needs generated unit squares).
//   aggregation   two passes of pairwise matching per level: a free row pairs
//                 with its strongest free neighbour (the largest positive
//                 -a_ij / sqrt(a_ii a_jj), ties to the smaller index) when the
//                 choice is mutual, in three handshake rounds; a row left over
//                 joins the pair of its strongest matched neighbour, or stays
//                 single when it has none.
//                 No absolute threshold: on coarse 3D levels with 20-30
//                 neighbours per row every normalized coupling is small.
//   coarse level  the Galerkin product P^T A P of the piecewise-constant P, a
//                 thread a coarse row (rows of more than 255 columns: every
//                 entry keyed (agg i, agg j), stably sorted, runs summed).
//   cycle         V(1,1) with the Chebyshev smoothing of the geometric levels
//                 (FP32-stored values, FP64 vectors), the coarse correction
//                 scaled by AMG_SCALE (plain aggregation under-corrects smooth
//                 error; the scaled cycle stays symmetric and positive
//                 definite for a scale below 2), the dense inverse on the
//                 coarsest level (at most MG_DENSE_MAX rows).
//   Krylov        FP64 CG with the device scalars and the true-residual check
//                 of the geometric solver.
// Fixed (penalized) rows are eliminated: x_d = b_d / A_dd, and they belong to
// no aggregate.  Every step is deterministic: handshakes read the previous
// round's state only, the sorts are stable and the sums run in a fixed order.
#define AMG_MAX_LEVELS 24
#define AMG_THETA 0.0
// 1.8 measured best over 1.3-1.9: 48 / 66 / 35 iterations on the 2048^2 P1,
// 2048^2 P2 and 160^3 tet Poisson systems, against 70 / 101 / 36 with 1.5
#define AMG_SCALE 1.8

struct AmgLevel {
    int64_t n = 0, nnz = 0;
    const int32_t *rp = nullptr, *ci = nullptr;  // level 0: the matrix's pattern
    const double *val = nullptr;                 // level 0: the matrix's FP64 values
    const uint8_t *fixed = nullptr;              // coarse levels: all zero
    float *val32 = nullptr;
    double *dinv = nullptr;
    MgCheb *ch = nullptr;
    double *x = nullptr, *b = nullptr, *r = nullptr, *d = nullptr;  // level 0: x = z, b = r of the CG
    int32_t *agg = nullptr;                      // row -> row of the next level (-1: fixed)
    int32_t *cagg = nullptr;                     // aggregate of each nonzero's column (fixed: the next level's n)
    int32_t *mptr = nullptr, *midx = nullptr;    // rows of this level: their members on the previous one
};

struct grmp_amg {
    grmp_ctx *ctx = nullptr;
    const grmp_matrix *A = nullptr;
    int nlev = 0;
    AmgLevel lv[AMG_MAX_LEVELS];
    double *inv = nullptr;
    double *x = nullptr, *rhs = nullptr, *r = nullptr, *z = nullptr, *p = nullptr, *q = nullptr;
    double *part = nullptr, *part2 = nullptr;
    MgScal *sc = nullptr;
    int nb0 = 0;
    MgPack pack;            // levels first .. nlev-1 run in one workgroup (nlev > 1)
    int first = 0;
    char *img = nullptr;    // their LDS image
    MgStatus *h = nullptr;  // pinned
    hipEvent_t ev = nullptr;
    std::vector<void *> mem;  // device allocations of the hierarchy
    int64_t nnz_total = 0;    // summed nonzeros of every level
};

template <class T>
static int amg_alloc(grmp_amg *m, T **p, size_t count)
{
    GRMP_TRY(dalloc(m->ctx, p, count));
    m->mem.push_back((void *)*p);
    return GRMP_OK;
}

// Lanes of a row in the aggregation's row scans: each entry is a chain of
// dependent loads (the neighbour's state, and a search of its row where the
// matrix is not symmetric), so the row's entries go side by side.  On the
// 128^3 tetrahedra a choice on the symmetric fine level takes 184 us (one lane:
// 382), on a coarse one 50 (109), the diagonal 15 (24); the solve 53.8 -> 51.1
// ms.  Eight lanes measured the same.
#define AMG_LANES 4
// diagonal of each row (0 if it has none)
__global__ void k_amg_diag(const int32_t *__restrict__ rp, const int32_t *__restrict__ ci,
                           const double *__restrict__ val, int64_t n, double *__restrict__ diag)
{
    const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / AMG_LANES;
    const int q = threadIdx.x % AMG_LANES;
    if (i >= n) return;
    int32_t at = -1;
    for (int32_t k = rp[i] + q; k < rp[i + 1]; k += AMG_LANES)
        if (ci[k] == i) at = k;
#pragma unroll
    for (int o = 1; o < AMG_LANES; o <<= 1) at = max(at, __shfl_xor(at, o, AMG_LANES));
    if (q == 0) diag[i] = at < 0 ? 0.0 : val[at];
}

// -(a_ij + a_ji) / 2: the strength of the pair (i, j) seen from both rows, so
// that both rows of a pair rank it alike when A is nonsymmetric (a Newton
// matrix); equal to -a_ij bit for bit when a_ji == a_ij.  Columns are
// ascending within a row (pattern and Galerkin levels alike); a_ji missing
// from row j counts as a_ij.
__device__ __forceinline__ double amg_pair_coupling(const int32_t *__restrict__ rp, const int32_t *__restrict__ ci,
                                                    const double *__restrict__ val, int32_t i, int32_t j, double aij)
{
    int32_t lo = rp[j], hi = rp[j + 1];
    while (lo < hi) {
        const int32_t mid = (lo + hi) >> 1;
        if (ci[mid] < i) lo = mid + 1;
        else hi = mid;
    }
    const double aji = (lo < rp[j + 1] && ci[lo] == i) ? val[lo] : aij;
    return -0.5 * (aij + aji);
}

// A key of the pair {i, j}, the same from both rows: the SplitMix64 finalizer
// (Steele, Lea, Flood 2014) of the ordered pair.  Equal strengths, which a
// structured mesh gives everywhere, are ranked by it; ranking them by the
// neighbour's index lets choices chain instead of pairing, and the coarsening
// of such a level stalls (P2 on 256 x 256 squares: 65029 -> 62672 rows).
__device__ __forceinline__ uint64_t amg_pair_key(int32_t i, int32_t j)
{
    const uint64_t lo = (uint64_t)(uint32_t)(i < j ? i : j), hi = (uint64_t)(uint32_t)(i < j ? j : i);
    uint64_t z = (lo << 32 | hi) + 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// best[i]: the strongest free, unmatched neighbour of the free, unmatched row
// i, or -1 (fixed == nullptr: no fixed rows); ties go to the larger pair key,
// then to the smaller index, so that strongest pairs are chosen from both ends
// SYM: a_ji == a_ij bit for bit, so a row needs no look at its neighbours'
// rows (the binary searches were most of the 154 us per launch on tetrahedra)
template <bool SYM>
__global__ void k_amg_best(const int32_t *__restrict__ rp, const int32_t *__restrict__ ci,
                           const double *__restrict__ val, const double *__restrict__ diag,
                           const uint8_t *__restrict__ fixed, const int32_t *__restrict__ mate, int64_t n,
                           double theta, int32_t *__restrict__ best)
{
    const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / AMG_LANES;
    const int q = threadIdx.x % AMG_LANES;
    if (i >= n) return;
    int32_t bj = -1;
    const double di = diag[i];
    if (mate[i] < 0 && !(fixed && fixed[i]) && di > 0.0) {
        double bs = 0.0;
        uint64_t bk = 0;
        auto take = [&](double st, uint64_t key, int32_t j) {
            if (bj < 0 || st > bs || (st == bs && (key > bk || (key == bk && j < bj)))) {
                bs = st;
                bk = key;
                bj = j;
            }
        };
        for (int32_t k = rp[i] + q; k < rp[i + 1]; k += AMG_LANES) {
            const int32_t j = ci[k];
            if (j == i || mate[j] >= 0 || (fixed && fixed[j]) || !(diag[j] > 0.0)) continue;
            const double st = (SYM ? -val[k] : amg_pair_coupling(rp, ci, val, (int32_t)i, j, val[k])) /
                              sqrt(di * diag[j]);
            if (!(st > theta)) continue;
            take(st, amg_pair_key((int32_t)i, j), j);
        }
#pragma unroll
        for (int o = 1; o < AMG_LANES; o <<= 1) {  // the order is total, so the lanes' maxima give the row's
            const double os = __shfl_xor(bs, o, AMG_LANES);
            const uint64_t ok = __shfl_xor((unsigned long long)bk, o, AMG_LANES);
            const int32_t oj = __shfl_xor(bj, o, AMG_LANES);
            if (oj >= 0) take(os, ok, oj);
        }
    }
    if (q == 0) best[i] = bj;
}

// mutual choices pair up (each row writes only its own mate)
__global__ void k_amg_match(const int32_t *__restrict__ best, int32_t *__restrict__ mate, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int32_t j = best[i];
    if (mate[i] < 0 && j >= 0 && best[j] == (int32_t)i) mate[i] = j;
}

// a free row left unmatched joins the pair of its strongest matched
// neighbour (join[i] = that neighbour), else stays single (join[i] = -1)
template <bool SYM>
__global__ void k_amg_join(const int32_t *__restrict__ rp, const int32_t *__restrict__ ci,
                           const double *__restrict__ val, const double *__restrict__ diag,
                           const uint8_t *__restrict__ fixed, const int32_t *__restrict__ mate, int64_t n,
                           int32_t *__restrict__ join)
{
    const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / AMG_LANES;
    const int q = threadIdx.x % AMG_LANES;
    if (i >= n) return;
    int32_t bj = -1;
    const double di = diag[i];
    if (mate[i] < 0 && !(fixed && fixed[i]) && di > 0.0) {
        double bs = 0.0;
        auto take = [&](double st, int32_t j) {
            if (bj < 0 || st > bs || (st == bs && j < bj)) {
                bs = st;
                bj = j;
            }
        };
        for (int32_t k = rp[i] + q; k < rp[i + 1]; k += AMG_LANES) {
            const int32_t j = ci[k];
            if (j == i || mate[j] < 0 || (fixed && fixed[j]) || !(diag[j] > 0.0)) continue;
            const double st = (SYM ? -val[k] : amg_pair_coupling(rp, ci, val, (int32_t)i, j, val[k])) /
                              sqrt(di * diag[j]);
            if (st > 0.0) take(st, j);
        }
#pragma unroll
        for (int o = 1; o < AMG_LANES; o <<= 1) {
            const double os = __shfl_xor(bs, o, AMG_LANES);
            const int32_t oj = __shfl_xor(bj, o, AMG_LANES);
            if (oj >= 0) take(os, oj);
        }
    }
    if (q == 0) join[i] = bj;
}

// lead[i] = 1 for the first row of each pair and for rows left single
__global__ void k_amg_lead(const int32_t *__restrict__ mate, const int32_t *__restrict__ join,
                           const uint8_t *__restrict__ fixed, int64_t n, int32_t *__restrict__ lead)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (fixed && fixed[i]) {
        lead[i] = 0;
        return;
    }
    const int32_t m = mate[i];
    lead[i] = m >= 0 ? ((int32_t)i <= m ? 1 : 0) : (join[i] < 0 ? 1 : 0);
}

__global__ void k_amg_assign(const int32_t *__restrict__ mate, const int32_t *__restrict__ join,
                             const uint8_t *__restrict__ fixed, const int32_t *__restrict__ id, int64_t n,
                             int32_t *__restrict__ agg)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (fixed && fixed[i]) {
        agg[i] = -1;
        return;
    }
    int32_t m = mate[i], r = (int32_t)i;
    if (m < 0 && join[i] >= 0) {  // the pair of the neighbour it joined
        r = join[i];
        m = mate[r];
    }
    agg[i] = m < 0 ? id[r] : id[m < r ? m : r];
}

// agg[i] = a2[a1[i]] (composition of two pairwise passes)
__global__ void k_amg_compose(const int32_t *__restrict__ a1, const int32_t *__restrict__ a2, int64_t n,
                              int32_t *__restrict__ agg)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    agg[i] = a1[i] < 0 ? -1 : a2[a1[i]];
}

// Galerkin keys: entry (i, j) -> agg i * nc + agg j; entries of fixed rows or
// columns get the sentinel nc * nc (sorted last, dropped)
__global__ void k_amg_keys(const int32_t *__restrict__ rp, const int32_t *__restrict__ ci,
                           const double *__restrict__ val, const int32_t *__restrict__ agg, int64_t n, int64_t nc,
                           uint64_t *__restrict__ keys, double *__restrict__ vals)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int32_t ai = agg[i];
    for (int32_t k = rp[i]; k < rp[i + 1]; ++k) {
        const int32_t aj = agg[ci[k]];
        const bool in = ai >= 0 && aj >= 0;
        keys[k] = in ? (uint64_t)ai * (uint64_t)nc + (uint64_t)aj : (uint64_t)nc * (uint64_t)nc;
        vals[k] = in ? val[k] : 0.0;
    }
}

// the coarse CSR from the sorted unique keys (rows ascending, columns ascending within a row)
__global__ void k_amg_rowcount(const uint64_t *__restrict__ ukeys, int64_t m, int64_t nc, int32_t *__restrict__ cnt)
{
    const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= m) return;
    atomicAdd(&cnt[ukeys[u] / (uint64_t)nc], 1);
}

__global__ void k_amg_cols(const uint64_t *__restrict__ ukeys, int64_t m, int64_t nc, int32_t *__restrict__ cols)
{
    const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= m) return;
    cols[u] = (int32_t)(ukeys[u] % (uint64_t)nc);
}

// members of each aggregate: keys agg (fixed rows -> nc, sorted last), values the row
__global__ void k_amg_member_keys(const int32_t *__restrict__ agg, int64_t n, int32_t nc, int32_t *__restrict__ key,
                                  int32_t *__restrict__ idx)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    key[i] = agg[i] < 0 ? nc : agg[i];
    idx[i] = (int32_t)i;
}

__global__ void k_amg_member_count(const int32_t *__restrict__ agg, int64_t n, int32_t *__restrict__ cnt)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (agg[i] >= 0) atomicAdd(&cnt[agg[i]], 1);
}

__global__ void k_amg_dinv(const double *__restrict__ diag, const uint8_t *__restrict__ fixed, int64_t n,
                           double *__restrict__ dinv)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    dinv[i] = (fixed[i] || !(diag[i] > 0.0)) ? 0.0 : 1.0 / diag[i];
}

// restriction b_c[I] = sum of r over the members of I, in row order; d_c = d0 of b_c
__global__ void k_amg_restrict(const int32_t *__restrict__ mptr, const int32_t *__restrict__ midx,
                               const double *__restrict__ r, const uint8_t *__restrict__ fixed_c,
                               const double *__restrict__ dinv_c, const MgCheb *__restrict__ ch_c,
                               double *__restrict__ bc, double *__restrict__ dc, int64_t nc, const MgScal *sc)
{
    if (sc->done) return;
    const int64_t I = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (I >= nc) return;
    double s = 0.0;
    for (int32_t k = mptr[I]; k < mptr[I + 1]; ++k) s += r[midx[k]];
    bc[I] = s;
    dc[I] = cheb_first(fixed_c[I] != 0, dinv_c[I], s, *ch_c);
}

// The residual and its restriction in one launch: four lanes a coarse row,
// each a member's row (a level's free rows are all members; the fixed ones'
// residual is not read), the sums in row order as above.  The rows are read
// uncoalesced, out of L2 on the levels it is taken for, where two launches are
// bound by their latency.  A CG iteration with no level / levels up to 2^15 / up to
// 2^17 rows fused (best of eight solves, which differ by 0.5 %): P1 100^2 80.9 /
// 78.6 / 78.7 us, P1 512^2 160.0 / 157.0 / 155.1, P2 211^2 141.6 / 139.5 / 138.5,
// tets 50^3 209.4 / 206.2 / 207.1, 75^3 294.5 / 290.7 / 293.5.  On the 128^3 tets'
// solve limits of 2^15 / 2^17 / 2^19 rows and none took 53.8 / 54.3 / 55.3 / 59.4 ms.
#define AMG_RR_LANES 4
#define AMG_RR_ROWS (1 << 15)
__global__ __launch_bounds__(256) void k_amg_resid_restrict(MgRows a, const int32_t *__restrict__ mptr,
                                                            const int32_t *__restrict__ midx,
                                                            const uint8_t *__restrict__ fixed_c,
                                                            const double *__restrict__ dinv_c,
                                                            const MgCheb *__restrict__ ch_c, double *__restrict__ bc,
                                                            double *__restrict__ dc, int64_t nc)
{
    if (a.sc->done) return;
    const int64_t I = ((int64_t)blockIdx.x * 256 + threadIdx.x) / AMG_RR_LANES;
    const int q = threadIdx.x % AMG_RR_LANES;
    if (I >= nc) return;
    const int32_t *__restrict__ rp = a.rp, *__restrict__ ci = a.ci;
    const float *__restrict__ val = a.val32;
    const double *__restrict__ v = a.v;
    const int32_t m0 = mptr[I], m1 = mptr[I + 1];
    double s = 0.0;
    for (int32_t k0 = m0; k0 < m1; k0 += AMG_RR_LANES) {
        double ri = 0.0;
        if (k0 + q < m1) {
            const int32_t i = midx[k0 + q], e0 = rp[i], e1 = rp[i + 1];
            const double bi = a.b[i];
            double p = 0.0;
            for (int32_t e = e0; e < e1; e += 8) {  // past the row's end its last entry again, unused
                int32_t c[8];
                float w[8];
                double xv[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int32_t f = e + u < e1 ? e + u : e1 - 1;
                    c[u] = ci[f];
                    w[u] = val[f];
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) xv[u] = v[c[u]];
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (e + u < e1) p += (double)w[u] * xv[u];
            }
            ri = bi - p;
            a.o1[i] = ri;
        }
        const int left = m1 - k0;
#pragma unroll
        for (int u = 0; u < AMG_RR_LANES; ++u) {
            const double ru = __shfl(ri, u, AMG_RR_LANES);
            if (u < left) s += ru;
        }
    }
    if (q == 0) {
        bc[I] = s;
        dc[I] = cheb_first(fixed_c[I] != 0, dinv_c[I], s, *ch_c);
    }
}

// the aggregate of every nonzero's column, nc where the column is fixed (the
// coarse vectors hold a zero there)
__global__ void k_amg_cagg(const int32_t *__restrict__ ci, const int32_t *__restrict__ agg, int64_t nnz, int32_t nc,
                           int32_t *__restrict__ cagg)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nnz) return;
    const int32_t a = agg[ci[k]];
    cagg[k] = a < 0 ? nc : a;
}

// the coarse end of the cycle: x = V(b) on the packed levels.  Launched level
// by level these few hundred rows took six launches of 2.5-5 us a level.
__global__ __launch_bounds__(MG_BT) void k_amg_vcycle_block(MgPack P, const double *__restrict__ b,
                                                            double *__restrict__ x, const MgScal *sc)
{
    extern __shared__ __align__(16) char pk_lds[];
    if (sc->done) return;
    double inv[4];
    pk_load_inv(P, inv);
    pk_stage(P, pk_lds);
    __syncthreads();
    pk_apply(P, pk_lds, inv, b, x);
}

// One pairwise pass over a level (rp, ci, val, fixed): agg[n], *nc.
static int amg_pairwise(grmp_ctx *ctx, const int32_t *rp, const int32_t *ci, const double *val, const uint8_t *fixed,
                        int64_t n, bool sym, int32_t *agg, int64_t *nc)
{
    hipStream_t st = ctx->stream;
    double *diag = nullptr;
    int32_t *mate = nullptr, *best = nullptr, *lead = nullptr, *id = nullptr;
    int rc = GRMP_OK;
    do {
        if ((rc = dalloc(ctx, &diag, n)) || (rc = dalloc(ctx, &mate, n)) || (rc = dalloc(ctx, &best, n)) ||
            (rc = dalloc(ctx, &lead, n)) || (rc = dalloc(ctx, &id, n + 1)))
            break;
        hipLaunchKernelGGL(k_amg_diag, dim3(nblk(n * AMG_LANES, 256)), dim3(256), 0, st, rp, ci, val, n, diag);
        if (hipMemsetAsync(mate, 0xff, sizeof(int32_t) * n, st) != hipSuccess) {
            rc = grmp_fail(ctx, GRMP_ERR_HIP, "AMG aggregation: memset");
            break;
        }
        for (int round = 0; round < 3; ++round) {
            if (sym)
                hipLaunchKernelGGL(k_amg_best<true>, dim3(nblk(n * AMG_LANES, 256)), dim3(256), 0, st, rp, ci, val, diag, fixed,
                                   mate, n, AMG_THETA, best);
            else
                hipLaunchKernelGGL(k_amg_best<false>, dim3(nblk(n * AMG_LANES, 256)), dim3(256), 0, st, rp, ci, val, diag, fixed,
                                   mate, n, AMG_THETA, best);
            hipLaunchKernelGGL(k_amg_match, dim3(nblk(n, 256)), dim3(256), 0, st, best, mate, n);
        }
        if (sym)
            hipLaunchKernelGGL(k_amg_join<true>, dim3(nblk(n * AMG_LANES, 256)), dim3(256), 0, st, rp, ci, val, diag, fixed, mate, n,
                               best);
        else
            hipLaunchKernelGGL(k_amg_join<false>, dim3(nblk(n * AMG_LANES, 256)), dim3(256), 0, st, rp, ci, val, diag, fixed, mate,
                               n, best);
        hipLaunchKernelGGL(k_amg_lead, dim3(nblk(n, 256)), dim3(256), 0, st, mate, best, fixed, n, lead);
        if ((rc = exclusive_scan_i32(ctx, lead, id, n))) break;
        int32_t cnt = 0;
        if (hipMemcpyAsync(&cnt, id + n, sizeof(int32_t), hipMemcpyDeviceToHost, st) != hipSuccess ||
            hipStreamSynchronize(st) != hipSuccess) {
            rc = grmp_fail(ctx, GRMP_ERR_HIP, "AMG aggregation: count");
            break;
        }
        hipLaunchKernelGGL(k_amg_assign, dim3(nblk(n, 256)), dim3(256), 0, st, mate, best, fixed, id, n, agg);
        *nc = cnt;
        if (hipGetLastError() != hipSuccess) rc = grmp_fail(ctx, GRMP_ERR_HIP, "AMG aggregation: launch");
    } while (0);
    dfree(ctx, diag);
    dfree(ctx, mate);
    dfree(ctx, best);
    dfree(ctx, lead);
    dfree(ctx, id);
    return rc;
}

// Galerkin product of a level with the aggregation agg (nc aggregates): the
// coarse CSR in new device arrays (caller frees, or keeps via amg_alloc-owned
// copies).  This form sorts every entry by its coarse (row, column); it takes
// the coarse rows too wide for amg_galerkin's sets.
static int amg_galerkin_sorted(grmp_ctx *ctx, const int32_t *rp, const int32_t *ci, const double *val, int64_t n, int64_t nnz,
                        const int32_t *agg, int64_t nc, int32_t **crp, int32_t **cci, double **cval, int64_t *cnnz)
{
    hipStream_t st = ctx->stream;
    *crp = nullptr;
    *cci = nullptr;
    *cval = nullptr;
    uint64_t *k0 = nullptr, *k1 = nullptr, *uk = nullptr;
    double *v0 = nullptr, *v1 = nullptr, *us = nullptr;
    int32_t *cnt = nullptr;
    int rc = GRMP_OK;
    do {
        if ((rc = dalloc(ctx, &k0, nnz)) || (rc = dalloc(ctx, &k1, nnz)) || (rc = dalloc(ctx, &v0, nnz)) ||
            (rc = dalloc(ctx, &v1, nnz)) || (rc = dalloc(ctx, &uk, nnz)) || (rc = dalloc(ctx, &us, nnz)))
            break;
        hipLaunchKernelGGL(k_amg_keys, dim3(nblk(n, 256)), dim3(256), 0, st, rp, ci, val, agg, n, nc, k0, v0);
        int bits = 1;
        while (bits < 64 && ((uint64_t)1 << bits) <= (uint64_t)nc * (uint64_t)nc) ++bits;
        if ((rc = sort_pairs_u64_f64(ctx, k0, k1, v0, v1, nnz, bits))) break;
        int64_t m = 0;
        if ((rc = reduce_runs_u64_f64(ctx, k1, v1, nnz, uk, us, &m))) break;
        // the sentinel run (entries of fixed rows or columns) is the last one
        uint64_t last = 0;
        if (m > 0) {
            if (hipMemcpyAsync(&last, uk + (m - 1), sizeof(uint64_t), hipMemcpyDeviceToHost, st) != hipSuccess ||
                hipStreamSynchronize(st) != hipSuccess) {
                rc = grmp_fail(ctx, GRMP_ERR_HIP, "AMG Galerkin: readback");
                break;
            }
            if (last == (uint64_t)nc * (uint64_t)nc) --m;
        }
        if ((rc = dalloc(ctx, &cnt, nc)) || (rc = dalloc(ctx, crp, nc + 1)) || (rc = dalloc(ctx, cci, m)) ||
            (rc = dalloc(ctx, cval, m)))
            break;
        if (hipMemsetAsync(cnt, 0, sizeof(int32_t) * nc, st) != hipSuccess ||
            hipMemcpyAsync(*cval, us, sizeof(double) * m, hipMemcpyDeviceToDevice, st) != hipSuccess) {
            rc = grmp_fail(ctx, GRMP_ERR_HIP, "AMG Galerkin: copy");
            break;
        }
        hipLaunchKernelGGL(k_amg_rowcount, dim3(nblk(m, 256)), dim3(256), 0, st, uk, m, nc, cnt);
        hipLaunchKernelGGL(k_amg_cols, dim3(nblk(m, 256)), dim3(256), 0, st, uk, m, nc, *cci);
        if ((rc = exclusive_scan_i32(ctx, cnt, *crp, nc))) break;
        *cnnz = m;
        if (hipGetLastError() != hipSuccess) rc = grmp_fail(ctx, GRMP_ERR_HIP, "AMG Galerkin: launch");
    } while (0);
    dfree(ctx, k0);
    dfree(ctx, k1);
    dfree(ctx, v0);
    dfree(ctx, v1);
    dfree(ctx, uk);
    dfree(ctx, us);
    dfree(ctx, cnt);
    if (rc) {
        dfree(ctx, *crp);
        dfree(ctx, *cci);
        dfree(ctx, *cval);
    }
    return rc;
}

// members of each aggregate: midx lists the rows sorted by aggregate and row,
// mptr[I] .. mptr[I + 1] those of aggregate I (rows outside any come last)
static int amg_members(grmp_ctx *ctx, const int32_t *agg, int64_t n, int64_t nc, int32_t *mptr, int32_t *midx)
{
    hipStream_t st = ctx->stream;
    int32_t *key = nullptr, *idx = nullptr, *skey = nullptr, *cnt = nullptr;
    int rc = GRMP_OK;
    do {
        if ((rc = dalloc(ctx, &key, n)) || (rc = dalloc(ctx, &idx, n)) || (rc = dalloc(ctx, &skey, n)) ||
            (rc = dalloc(ctx, &cnt, nc)))
            break;
        hipLaunchKernelGGL(k_amg_member_keys, dim3(nblk(n, 256)), dim3(256), 0, st, agg, n, (int32_t)nc, key, idx);
        int bits = 1;
        while (bits < 31 && ((int64_t)1 << bits) <= nc) ++bits;
        if ((rc = sort_pairs_i32_i32(ctx, key, skey, idx, midx, n, bits))) break;
        if (hipMemsetAsync(cnt, 0, sizeof(int32_t) * nc, st) != hipSuccess) {
            rc = grmp_fail(ctx, GRMP_ERR_HIP, "AMG members: memset");
            break;
        }
        hipLaunchKernelGGL(k_amg_member_count, dim3(nblk(n, 256)), dim3(256), 0, st, agg, n, cnt);
        rc = exclusive_scan_i32(ctx, cnt, mptr, nc);
    } while (0);
    dfree(ctx, key);
    dfree(ctx, idx);
    dfree(ctx, skey);
    dfree(ctx, cnt);
    return rc;
}

// The Galerkin rows by ownership, as the element patterns are built: one
// thread per coarse row collects the aggregates of its members' columns in a
// sorted LDS set (FILL: and adds the values at their places, members and
// columns in ascending order).  Against sorting all entries by (row, column)
// it reads the matrix twice instead of moving 16 bytes an entry through six
// radix passes: with the product of the second pass in place of one from the
// fine level, the 128^3 tets' solve 93.5 -> 74.3 ms.
template <int B, int RMAX, bool FILL>
__global__ __launch_bounds__(B) void k_amg_galerkin(const int32_t *__restrict__ mptr, const int32_t *__restrict__ midx,
                                                    const int32_t *__restrict__ rp, const int32_t *__restrict__ ci,
                                                    const double *__restrict__ val, const int32_t *__restrict__ agg,
                                                    int64_t nc, int32_t *__restrict__ cnt, int *__restrict__ flag,
                                                    const int32_t *__restrict__ crp, int32_t *__restrict__ cci,
                                                    double *__restrict__ cval)
{
    __shared__ int32_t set[RMAX * B];
    const int64_t I = (int64_t)blockIdx.x * B + threadIdx.x;
    if (I >= nc) return;
    int n = 0;
    bool ok = true;
    const int32_t m0 = mptr[I], m1 = mptr[I + 1];
    for (int32_t m = m0; m < m1; ++m) {
        const int32_t i = midx[m], k1 = rp[i + 1];
        for (int32_t k = rp[i]; k < k1; k += 4) {  // four columns' aggregates in flight
            int32_t a[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) a[u] = k + u < k1 ? agg[ci[k + u]] : -1;
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (a[u] >= 0) ok &= set_insert<B>(set, n, RMAX, a[u]);
        }
    }
    if (!FILL) {
        if (!ok) atomicOr(flag, 1);
        cnt[I] = n;
        return;
    }
    const int32_t base = crp[I];
    for (int p = 0; p < n; ++p) {
        cci[base + p] = set[p * B + threadIdx.x];
        cval[base + p] = 0.0;
    }
    for (int32_t m = m0; m < m1; ++m) {
        const int32_t i = midx[m], k1 = rp[i + 1];
        for (int32_t k = rp[i]; k < k1; k += 4) {
            int32_t a[4];
            double v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                a[u] = k + u < k1 ? agg[ci[k + u]] : -1;
                v[u] = k + u < k1 ? val[k + u] : 0.0;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (a[u] >= 0) cval[base + set_find<B>(set, n, a[u])] += v[u];
        }
    }
}

// Galerkin product with the aggregates' members; coarse rows of up to 32, else
// 64, else 255 entries, wider ones by sorting
static int amg_galerkin(grmp_ctx *ctx, const int32_t *rp, const int32_t *ci, const double *val, int64_t n, int64_t nnz,
                        const int32_t *agg, const int32_t *mptr, const int32_t *midx, int64_t nc, int32_t **crp,
                        int32_t **cci, double **cval, int64_t *cnnz)
{
    hipStream_t st = ctx->stream;
    *crp = nullptr;
    *cci = nullptr;
    *cval = nullptr;
    int32_t *cnt = nullptr;
    int rc = GRMP_OK, width = 0;
    const dim3 grid(nblk(nc, 64)), blk(64);
    do {
        if ((rc = dalloc(ctx, &cnt, nc)) || (rc = dalloc(ctx, crp, nc + 1))) break;
        int flag = 1;
        for (; width < 3 && flag; ++width) {
            if (hipMemsetAsync(ctx->dflag, 0, sizeof(int), st) != hipSuccess) {
                rc = grmp_fail(ctx, GRMP_ERR_HIP, "AMG Galerkin: memset");
                break;
            }
            if (width == 0)
                hipLaunchKernelGGL((k_amg_galerkin<64, 32, false>), grid, blk, 0, st, mptr, midx, rp, ci, val, agg, nc,
                                   cnt, ctx->dflag, nullptr, nullptr, nullptr);
            else if (width == 1)
                hipLaunchKernelGGL((k_amg_galerkin<64, 64, false>), grid, blk, 0, st, mptr, midx, rp, ci, val, agg, nc,
                                   cnt, ctx->dflag, nullptr, nullptr, nullptr);
            else
                hipLaunchKernelGGL((k_amg_galerkin<64, 255, false>), grid, blk, 0, st, mptr, midx, rp, ci, val, agg, nc,
                                   cnt, ctx->dflag, nullptr, nullptr, nullptr);
            // the scan is enqueued before the flag is known: one synchronization for both
            int32_t m = 0;
            if ((rc = exclusive_scan_i32(ctx, cnt, *crp, nc))) break;
            if (hipMemcpyAsync(&flag, ctx->dflag, sizeof(int), hipMemcpyDeviceToHost, st) != hipSuccess ||
                hipMemcpyAsync(&m, *crp + nc, sizeof(int32_t), hipMemcpyDeviceToHost, st) != hipSuccess ||
                hipStreamSynchronize(st) != hipSuccess) {
                rc = grmp_fail(ctx, GRMP_ERR_HIP, "AMG Galerkin: count");
                break;
            }
            *cnnz = m;
        }
        if (rc) break;
        if (flag) {
            dfree(ctx, cnt);
            dfree(ctx, *crp);
            return amg_galerkin_sorted(ctx, rp, ci, val, n, nnz, agg, nc, crp, cci, cval, cnnz);
        }
        if ((rc = dalloc(ctx, cci, *cnnz)) || (rc = dalloc(ctx, cval, *cnnz))) break;
        if (width == 1)
            hipLaunchKernelGGL((k_amg_galerkin<64, 32, true>), grid, blk, 0, st, mptr, midx, rp, ci, val, agg, nc, cnt,
                               ctx->dflag, *crp, *cci, *cval);
        else if (width == 2)
            hipLaunchKernelGGL((k_amg_galerkin<64, 64, true>), grid, blk, 0, st, mptr, midx, rp, ci, val, agg, nc, cnt,
                               ctx->dflag, *crp, *cci, *cval);
        else
            hipLaunchKernelGGL((k_amg_galerkin<64, 255, true>), grid, blk, 0, st, mptr, midx, rp, ci, val, agg, nc, cnt,
                               ctx->dflag, *crp, *cci, *cval);
        if (hipGetLastError() != hipSuccess) rc = grmp_fail(ctx, GRMP_ERR_HIP, "AMG Galerkin: launch");
    } while (0);
    dfree(ctx, cnt);
    if (rc) {
        dfree(ctx, *crp);
        dfree(ctx, *cci);
        dfree(ctx, *cval);
    }
    return rc;
}

// smoother data of a level: FP32 values, inverse diagonal, Gershgorin bound
static int amg_level_smoother(grmp_amg *m, AmgLevel &L)
{
    grmp_ctx *ctx = m->ctx;
    hipStream_t st = ctx->stream;
    double *diag = nullptr;
    GRMP_TRY(amg_alloc(m, &L.val32, L.nnz));
    GRMP_TRY(amg_alloc(m, &L.dinv, L.n));
    GRMP_TRY(amg_alloc(m, &L.ch, 1));
    GRMP_TRY(dalloc(ctx, &diag, L.n));
    hipLaunchKernelGGL(k_amg_diag, dim3(nblk(L.n * AMG_LANES, 256)), dim3(256), 0, st, L.rp, L.ci, L.val, L.n, diag);
    hipLaunchKernelGGL(k_amg_dinv, dim3(nblk(L.n, 256)), dim3(256), 0, st, diag, L.fixed, L.n, L.dinv);
    MgPrep P;
    P.nlev = P.blocks = 0;
    mg_prep_add(P, L.rp, L.val, L.dinv, L.fixed, L.val32, L.ch, L.n, false);
    mg_prep_launch(P, st);
    dfree(ctx, diag);
    GRMP_HIP(ctx, hipGetLastError());
    return GRMP_OK;
}

static void amg_free(grmp_amg *m)
{
    if (!m) return;
    for (void *p : m->mem) dfree(m->ctx, p);
    m->mem.clear();
    if (m->h) (void)hipHostFree(m->h);
    if (m->ev) (void)hipEventDestroy(m->ev);
    delete m;
}

// Whether a_ij == a_ji bit for bit: the symmetric pattern type evaluates each
// local pair once, lower dof first, and both entries sum the same cells in the
// same order.  Not the Newton and Hooke forms, nor the coarse levels.
static bool amg_symmetric(const grmp_matrix *A)
{
    for (const FormRec &r : A->forms)
        if (r.kind != FK_LAPLACE_P1TRI && r.kind != FK_LAPLACE_P2TRI && r.kind != FK_LAPLACE_P1TET &&
            r.kind != FK_MASS_P1TRI && r.kind != FK_MASS_P2TRI)
            return false;
    return !A->forms.empty();
}

static int amg_build(grmp_amg *m)
{
    grmp_ctx *ctx = m->ctx;
    hipStream_t st = ctx->stream;
    const grmp_matrix *A = m->A;
    AmgLevel &L0 = m->lv[0];
    L0.n = A->n;
    L0.nnz = A->nnz;
    L0.rp = A->rowptr;
    L0.ci = A->cols;
    L0.val = A->val64;
    L0.fixed = A->fixed;
    m->nlev = 1;
    m->nnz_total = L0.nnz;
    GRMP_TRY(amg_level_smoother(m, L0));
    for (;;) {
        AmgLevel &F = m->lv[m->nlev - 1];
        // coarsest once few enough free rows remain (the dense inverse replaces fixed rows by the identity)
        if (F.n <= MG_DENSE_MAX) break;
        GRMP_CHECK(ctx, m->nlev < AMG_MAX_LEVELS, GRMP_ERR_UNSUPPORTED,
                   "AMG: %lld rows left after %d levels", (long long)F.n, m->nlev);
        // first pairwise pass on the level, second on the intermediate Galerkin
        // product; the coarse operator is the product of the second pass, half
        // the rows of the first: P2^T (P1^T A P1) P2
        int32_t *a1 = nullptr, *a2 = nullptr, *irp = nullptr, *ici = nullptr, *mp = nullptr, *mi = nullptr;
        double *ival = nullptr;
        int32_t *crp = nullptr, *cci = nullptr;
        double *cval = nullptr;
        int64_t n1 = 0, n2 = 0, innz = 0, cnnz = 0;
        const bool sym = m->nlev == 1 && amg_symmetric(A);
        int rc = GRMP_OK;
        do {
            if ((rc = dalloc(ctx, &a1, F.n))) break;
            if ((rc = amg_pairwise(ctx, F.rp, F.ci, F.val, F.fixed, F.n, sym, a1, &n1))) break;
            if (n1 == 0) {
                rc = grmp_fail(ctx, GRMP_ERR_ARG, "AMG: no free rows");
                break;
            }
            if ((rc = dalloc(ctx, &mp, n1 + 1)) || (rc = dalloc(ctx, &mi, F.n))) break;
            if ((rc = amg_members(ctx, a1, F.n, n1, mp, mi))) break;
            if ((rc = amg_galerkin(ctx, F.rp, F.ci, F.val, F.n, F.nnz, a1, mp, mi, n1, &irp, &ici, &ival, &innz))) break;
            if ((rc = dalloc(ctx, &a2, n1))) break;
            if ((rc = amg_pairwise(ctx, irp, ici, ival, nullptr, n1, false, a2, &n2))) break;
            if (n2 > F.n - F.n / 10) {  // coarsening stalled
                rc = grmp_fail(ctx, GRMP_ERR_UNSUPPORTED, "AMG: coarsening stalled at %lld rows", (long long)F.n);
                break;
            }
            if ((rc = amg_members(ctx, a2, n1, n2, mp, mi))) break;
            if ((rc = amg_galerkin(ctx, irp, ici, ival, n1, innz, a2, mp, mi, n2, &crp, &cci, &cval, &cnnz))) break;
            if ((rc = amg_alloc(m, &F.agg, F.n))) break;
            hipLaunchKernelGGL(k_amg_compose, dim3(nblk(F.n, 256)), dim3(256), 0, st, a1, a2, F.n, F.agg);
        } while (0);
        dfree(ctx, irp);
        dfree(ctx, ici);
        dfree(ctx, ival);
        dfree(ctx, mp);
        dfree(ctx, mi);
        dfree(ctx, a1);
        dfree(ctx, a2);
        if (crp) m->mem.push_back(crp);
        if (cci) m->mem.push_back(cci);
        if (cval) m->mem.push_back(cval);
        GRMP_TRY(rc);
        AmgLevel &C = m->lv[m->nlev];
        C.n = n2;
        C.nnz = cnnz;
        C.rp = crp;
        C.ci = cci;
        C.val = cval;
        uint8_t *cfix = nullptr;
        GRMP_TRY(amg_alloc(m, &cfix, C.n));
        GRMP_HIP(ctx, hipMemsetAsync(cfix, 0, C.n, st));
        C.fixed = cfix;
        // members of each coarse row, in fine-row order, for the restriction
        GRMP_TRY(amg_alloc(m, &C.midx, F.n));
        GRMP_TRY(amg_alloc(m, &C.mptr, C.n + 1));
        GRMP_TRY(amg_members(ctx, F.agg, F.n, C.n, C.mptr, C.midx));
        ++m->nlev;
        m->nnz_total += C.nnz;
        GRMP_TRY(amg_level_smoother(m, C));
    }
    // vectors: level 0 aliases the CG's z and r; coarse levels own theirs
    const int64_t n0 = L0.n;
    m->nb0 = (int)nblk(n0, KB);
    GRMP_TRY(amg_alloc(m, &m->x, n0));
    GRMP_TRY(amg_alloc(m, &m->rhs, n0));
    GRMP_TRY(amg_alloc(m, &m->r, n0));
    GRMP_TRY(amg_alloc(m, &m->z, n0));
    GRMP_TRY(amg_alloc(m, &m->p, n0));
    GRMP_TRY(amg_alloc(m, &m->q, n0));
    GRMP_TRY(amg_alloc(m, &m->part, m->nb0));
    GRMP_TRY(amg_alloc(m, &m->part2, m->nb0));
    GRMP_TRY(amg_alloc(m, &m->sc, 1));
    for (int l = 0; l < m->nlev; ++l) {
        AmgLevel &L = m->lv[l];
        if (l == 0) {
            L.x = m->z;
            L.b = m->r;
        } else {
            // one entry more, kept 0: what the fixed columns' cagg points to
            GRMP_TRY(amg_alloc(m, &L.x, L.n + 1));
            GRMP_HIP(ctx, hipMemsetAsync(L.x + L.n, 0, sizeof(double), st));
            GRMP_TRY(amg_alloc(m, &L.b, L.n));
        }
        GRMP_TRY(amg_alloc(m, &L.r, L.n));
        GRMP_TRY(amg_alloc(m, &L.d, L.n));
    }
    const AmgLevel &C = m->lv[m->nlev - 1];
    GRMP_TRY(amg_alloc(m, &m->inv, C.n * C.n));
    hipLaunchKernelGGL(k_mg_dense_inv, dim3(1), dim3(256), 0, st, C.rp, C.ci, C.val, C.fixed, (int)C.n, m->inv);
    memset(&m->pack, 0, sizeof(m->pack));
    if (m->nlev > 1) {
        // the most levels from the coarsest up that fit one workgroup's LDS (the coarsest always does)
        MgPackShape sh[AMG_MAX_LEVELS];
        for (int l = 0; l < m->nlev; ++l) sh[l] = MgPackShape{m->lv[l].n, m->lv[l].nnz, 0, 0, 1, TR_AGG};
        m->first = 0;
        for (int f = m->nlev - 1; f >= 1; --f) {
            MgPack P;
            if (!mg_pack_layout(P, sh + f, m->nlev - f)) break;
            m->pack = P;
            m->first = f;
        }
        GRMP_CHECK(ctx, m->first >= 1, GRMP_ERR_UNSUPPORTED, "AMG: the coarsest level does not fit LDS");
        GRMP_TRY(mg_allow_lds(ctx, (const void *)k_amg_vcycle_block));
        GRMP_TRY(amg_alloc(m, &m->img, m->pack.image));
        m->pack.img = m->img;
        m->pack.inv = m->inv;
        m->pack.scale = AMG_SCALE;
        for (int k = 0; k < m->pack.nlev; ++k) {
            const AmgLevel &L = m->lv[m->first + k];
            const AmgLevel *N = k + 1 < m->pack.nlev ? &m->lv[m->first + k + 1] : nullptr;
            const MgPackSrc S{L.rp, L.ci, L.val32, L.dinv, L.ch, L.fixed, N ? L.agg : nullptr,
                              N ? N->mptr : nullptr, N ? N->midx : nullptr, (int32_t)L.nnz,
                              N ? (int32_t)N->n : 0};
            const int64_t items = std::max(std::max(L.nnz, L.n + 1), N ? N->n + 1 : (int64_t)0);
            hipLaunchKernelGGL(k_mg_pack, dim3(nblk(items, 256)), dim3(256), 0, st, m->pack.lv[k], S, m->img);
        }
        for (int l = 0; l < m->first; ++l) {
            AmgLevel &L = m->lv[l];
            GRMP_TRY(amg_alloc(m, &L.cagg, L.nnz));
            hipLaunchKernelGGL(k_amg_cagg, dim3(nblk(L.nnz, 256)), dim3(256), 0, st, L.ci, L.agg, L.nnz,
                               (int32_t)m->lv[l + 1].n, L.cagg);
        }
    }
    GRMP_HIP(ctx, hipGetLastError());
    GRMP_HIP(ctx, hipStreamSynchronize(st));
    return GRMP_OK;
}

static void amg_rows(MgRows &a, const AmgLevel &L, const grmp_amg *m)
{
    memset(&a, 0, sizeof(a));
    a.rp = L.rp;
    a.ci = L.ci;
    a.val = L.val;
    a.val32 = L.val32;
    a.fixed = L.fixed;
    a.n = L.n;
    a.dinv = L.dinv;
    a.ch = L.ch;
    a.sc = m->sc;
}

// z (= x_0) = V(r (= b_0)), d_0 holding d0 of r; level-0 partials of r.z land in part
static void amg_vcycle(grmp_amg *m)
{
    hipStream_t st = m->ctx->stream;
    if (m->nlev == 1) {  // z = the dense solve, partials of r.z
        const AmgLevel &C = m->lv[0];
        hipLaunchKernelGGL(k_mg_dense_apply, dim3(1), dim3(MG_DENSE_MAX), 0, st, m->inv, C.b, (int)C.n, C.x, m->sc);
        hipLaunchKernelGGL(k_mg_dot, dim3(m->nb0), dim3(KB), 0, st, m->r, m->z, C.n, m->part, m->sc);
        return;
    }
    const int F = m->first;
    for (int l = 0; l < F; ++l) {
        const AmgLevel &L = m->lv[l], &C = m->lv[l + 1];
        MgRows a;
        amg_rows(a, L, m);
        a.v = L.d;
        a.b = L.b;
        a.o1 = L.x;
        hipLaunchKernelGGL(k_mg_rows<OP_CHEB_PRE>, dim3(nblk(L.n, KB)), dim3(KB), 0, st, a);
        amg_rows(a, L, m);
        a.v = L.x;
        a.b = L.b;
        a.o1 = L.r;
        if (L.n <= AMG_RR_ROWS) {
            hipLaunchKernelGGL(k_amg_resid_restrict, dim3(nblk(C.n * AMG_RR_LANES, 256)), dim3(256), 0, st, a, C.mptr,
                               C.midx, C.fixed, C.dinv, C.ch, C.b, C.d, C.n);
            continue;
        }
        hipLaunchKernelGGL(k_mg_rows<OP_RESID>, dim3(nblk(L.n, KB)), dim3(KB), 0, st, a);
        hipLaunchKernelGGL(k_amg_restrict, dim3(nblk(C.n, 256)), dim3(256), 0, st, C.mptr, C.midx, L.r, C.fixed,
                           C.dinv, C.ch, C.b, C.d, C.n, m->sc);
    }
    hipLaunchKernelGGL(k_amg_vcycle_block, dim3(1), dim3(MG_BT), m->pack.lds, st, m->pack, m->lv[F].b, m->lv[F].x,
                       m->sc);
    for (int l = F - 1; l >= 0; --l) {
        // the prolongation is part of the first smoothing step: A (x + e) = A x + (A P) v with the residual of x
        // still in r, so the pass over x goes and the gathers read the coarse vector
        const AmgLevel &L = m->lv[l], &C = m->lv[l + 1];
        MgRows a;
        amg_rows(a, L, m);
        a.ci = L.cagg;
        a.v = C.x;
        a.b = L.r;
        a.d = L.x;
        a.agg = L.agg;
        a.scale = AMG_SCALE;
        a.o1 = L.d;
        a.o2 = L.r;
        hipLaunchKernelGGL(k_mg_rows<OP_AGG_POST1>, dim3(nblk(L.n, KB)), dim3(KB), 0, st, a);
        amg_rows(a, L, m);
        a.v = L.r;
        a.b = L.b;
        a.d = L.d;
        a.o1 = L.x;
        a.part = l == 0 ? m->part : nullptr;
        hipLaunchKernelGGL(k_mg_rows<OP_CHEB_POST2>, dim3(nblk(L.n, KB)), dim3(KB), 0, st, a);
    }
}

static void amg_iterate(grmp_amg *m, int iters)
{
    hipStream_t st = m->ctx->stream;
    const AmgLevel &L0 = m->lv[0];
    const int64_t n = L0.n;
    for (int k = 0; k < iters; ++k) {
        MgRows a;
        amg_rows(a, L0, m);
        a.v = m->p;
        a.o1 = m->q;
        a.part = m->part;
        hipLaunchKernelGGL(k_mg_rows<OP_PCG_Q>, dim3(nblk(n, KB)), dim3(KB), 0, st, a);
        hipLaunchKernelGGL(k_mg_red<RED_ALPHA>, dim3(1), dim3(MG_BT), 0, st, m->part, m->nb0, nullptr, m->sc);
        hipLaunchKernelGGL(k_mg_axpy, dim3(m->nb0), dim3(KB), 0, st, m->x, m->r, m->p, m->q, L0.fixed, L0.dinv, L0.ch,
                           L0.d, n, m->part, m->sc);
        hipLaunchKernelGGL(k_mg_red<RED_CONV>, dim3(1), dim3(MG_BT), 0, st, m->part, m->nb0, nullptr, m->sc);
        amg_vcycle(m);
        hipLaunchKernelGGL(k_mg_red<RED_BETA>, dim3(1), dim3(MG_BT), 0, st, m->part, m->nb0, nullptr, m->sc);
        hipLaunchKernelGGL(k_mg_update_p, dim3(nblk(n, 256)), dim3(256), 0, st, m->p, m->z, n, m->sc);
    }
}

// the true residual b - A x (FP64 values): accept, or restart CG from it
static void amg_verify(grmp_amg *m)
{
    hipStream_t st = m->ctx->stream;
    const AmgLevel &L0 = m->lv[0];
    const int64_t n = L0.n;
    hipLaunchKernelGGL(k_mg_verify_begin, dim3(1), dim3(1), 0, st, m->sc);
    MgRows a;
    amg_rows(a, L0, m);
    a.v = m->x;
    a.b = m->rhs;
    a.o1 = m->r;
    a.o2 = L0.d;
    hipLaunchKernelGGL(k_mg_rows<OP_TRUE_RESID>, dim3(nblk(n, KB)), dim3(KB), 0, st, a);
    hipLaunchKernelGGL(k_mg_dot, dim3(m->nb0), dim3(KB), 0, st, m->r, m->r, n, m->part, m->sc);
    hipLaunchKernelGGL(k_mg_red<RED_VERIFY>, dim3(1), dim3(MG_BT), 0, st, m->part, m->nb0, nullptr, m->sc);
    amg_vcycle(m);
    hipLaunchKernelGGL(k_mg_red<RED_RESTART>, dim3(1), dim3(MG_BT), 0, st, m->part, m->nb0, nullptr, m->sc);
    hipLaunchKernelGGL(k_mg_update_p, dim3(nblk(n, 256)), dim3(256), 0, st, m->p, m->z, n, m->sc);
}

static int amg_status(grmp_amg *m)
{
    hipStream_t st = m->ctx->stream;
    GRMP_HIP(m->ctx, hipMemcpyAsync(&m->h->relres, &m->sc->relres, 8, hipMemcpyDeviceToHost, st));
    GRMP_HIP(m->ctx, hipMemcpyAsync(&m->h->it, &m->sc->it, 12, hipMemcpyDeviceToHost, st));
    GRMP_HIP(m->ctx, hipEventRecord(m->ev, st));
    GRMP_HIP(m->ctx, hipEventSynchronize(m->ev));
    return GRMP_OK;
}

extern "C" int grmp_amg_destroy(grmp_amg *m)
{
    if (!m) return GRMP_OK;
    grmp_ctx *ctx = m->ctx;
    std::lock_guard<std::mutex> g(ctx->mu);
    (void)hipStreamSynchronize(ctx->stream);
    amg_free(m);
    return GRMP_OK;
}

// z = V v: one V-cycle of the hierarchy from a zero start (fixed rows 0), as
// the right preconditioner of BiCGStab on a matrix of the hierarchy's rows,
// e.g. the Newton matrix it was built from
int amg_precond_apply(grmp_amg *m, const double *v, double *z, hipStream_t st, const int *skip)
{
    GRMP_CHECK(m->ctx, st == m->ctx->stream, GRMP_ERR_ARG,
               "algebraic multigrid preconditioner: not the hierarchy's stream");
    AmgLevel &L0 = m->lv[0];
    hipLaunchKernelGGL(k_mg_pc_in, dim3(nblk(L0.n, 256)), dim3(256), 0, st, v, L0.fixed, L0.dinv, L0.ch, m->r, L0.d, m->sc,
                       L0.n, skip);
    // level 0 works in the caller's z (the cycle writes every row of it), so nothing is copied out
    double *own = L0.x;
    L0.x = z;
    amg_vcycle(m);
    L0.x = own;
    GRMP_HIP(m->ctx, hipGetLastError());
    return GRMP_OK;
}

int64_t amg_level0_rows(const grmp_amg *m) { return m->lv[0].n; }
grmp_ctx *amg_context(const grmp_amg *m) { return m->ctx; }

extern "C" int grmp_amg_create(grmp_matrix *A, grmp_amg **out)
{
    if (!A || !out) return GRMP_ERR_ARG;
    *out = nullptr;
    grmp_ctx *ctx = A->ctx;
    GRMP_CHECK(ctx, A->have_pattern && A->val64 && A->fixed && A->n >= 1, GRMP_ERR_ARG,
               "grmp_amg_create: matrix not assembled in FP64");
    std::lock_guard<std::mutex> g(ctx->mu);
    grmp_amg *m = new grmp_amg();
    m->ctx = ctx;
    m->A = A;
    int rc = GRMP_OK;
    if (hipHostMalloc((void **)&m->h, sizeof(MgStatus), hipHostMallocDefault) != hipSuccess ||
        hipEventCreateWithFlags(&m->ev, hipEventDisableTiming) != hipSuccess) {
        m->h = nullptr;
        rc = grmp_fail(ctx, GRMP_ERR_HIP, "grmp_amg_create: status buffer");
    }
    if (!rc) rc = amg_build(m);
    if (rc) {
        (void)hipStreamSynchronize(ctx->stream);
        amg_free(m);
        return rc;
    }
    *out = m;
    return GRMP_OK;
}

extern "C" int grmp_amg_info(const grmp_amg *m, int *nlev, int64_t *coarse_rows, double *complexity)
{
    if (!m) return GRMP_ERR_ARG;
    if (nlev) *nlev = m->nlev;
    if (coarse_rows) *coarse_rows = m->lv[m->nlev - 1].n;
    if (complexity) *complexity = (double)m->nnz_total / (double)std::max<int64_t>(m->lv[0].nnz, 1);
    return GRMP_OK;
}

extern "C" int grmp_amg_apply(grmp_amg *m, const grmp_vector *b, grmp_vector *x, double rtol, int64_t maxit,
                              grmp_solve_info *info)
{
    if (!m || !b || !x) return GRMP_ERR_ARG;
    grmp_ctx *ctx = m->ctx;
    const int64_t n = m->lv[0].n;
    GRMP_CHECK(ctx, b->ctx == ctx && x->ctx == ctx && b->n == n && x->n == n, GRMP_ERR_ARG,
               "grmp_amg_apply: b and x need length %lld", (long long)n);
    GRMP_CHECK(ctx, rtol > 0.0 && rtol < 1.0 && maxit >= 1 && maxit <= (1 << 30), GRMP_ERR_ARG,
               "grmp_amg_apply: rtol in (0, 1) and maxit >= 1 needed");
    std::lock_guard<std::mutex> g(ctx->mu);
    hipStream_t st = ctx->stream;
    const double t0 = wall_seconds();
    MgStatus *h = m->h;
    memset(h, 0, sizeof(MgStatus));
    int rc = GRMP_OK;
    do {
        // x = b_d / A_dd on fixed rows, 0 elsewhere; r = b - A x on free rows; z = V(r); p = z
        MgScal s0;
        memset(&s0, 0, sizeof(s0));
        s0.rtol = s0.rstop = rtol;
        s0.maxit = (int)maxit;
        if (hipMemcpyAsync(m->sc, &s0, sizeof(s0), hipMemcpyHostToDevice, st) != hipSuccess ||
            hipMemcpyAsync(m->rhs, b->d, sizeof(double) * n, hipMemcpyDeviceToDevice, st) != hipSuccess ||
            hipMemsetAsync(m->p, 0, sizeof(double) * n, st) != hipSuccess) {
            rc = grmp_fail(ctx, GRMP_ERR_HIP, "grmp_amg_apply: start");
            break;
        }
        if ((rc = init_x_launch(m->A, m->A->val64, m->rhs, m->x, st))) break;
        MgRows a;
        amg_rows(a, m->lv[0], m);
        a.v = m->x;
        a.b = m->rhs;
        a.o1 = m->r;
        a.o2 = m->lv[0].d;
        hipLaunchKernelGGL(k_mg_rows<OP_TRUE_RESID>, dim3(nblk(n, KB)), dim3(KB), 0, st, a);
        amg_vcycle(m);
        hipLaunchKernelGGL(k_mg_dot, dim3(m->nb0), dim3(KB), 0, st, m->r, m->r, n, m->part2, m->sc);
        hipLaunchKernelGGL(k_mg_red<RED_INIT>, dim3(1), dim3(MG_BT), 0, st, m->part, m->nb0, m->part2, m->sc);
        hipLaunchKernelGGL(k_mg_update_p, dim3(nblk(n, 256)), dim3(256), 0, st, m->p, m->z, n, m->sc);
        amg_iterate(m, 4);
        if ((rc = amg_status(m))) break;
        while (h->done != 1) {
            if (h->done == 2) amg_verify(m);
            else amg_iterate(m, 4);
            if ((rc = amg_status(m))) break;
        }
        if (rc) break;
        if (hipMemcpyAsync(x->d, m->x, sizeof(double) * n, hipMemcpyDeviceToDevice, st) != hipSuccess ||
            hipStreamSynchronize(st) != hipSuccess)
            rc = grmp_fail(ctx, GRMP_ERR_HIP, "grmp_amg_apply: solution");
    } while (0);
    grmp_solve_info inf;
    memset(&inf, 0, sizeof(inf));
    inf.status = h->status;
    inf.iterations = h->it;
    inf.relres = h->relres;
    inf.outer = 1;
    inf.seconds = wall_seconds() - t0;
    if (info) *info = inf;
    if (rc) {
        (void)hipStreamSynchronize(st);
        return rc;
    }
    if (inf.status == GRMP_ERR_NOCONV)
        return grmp_fail(ctx, GRMP_ERR_NOCONV, "grmp_amg_apply: no convergence, relres %.3e after %lld iterations",
                         inf.relres, (long long)inf.iterations);
    return inf.status;
}
