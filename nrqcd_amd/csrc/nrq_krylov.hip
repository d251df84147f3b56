// nrq_krylov.hip -- batched solvers for the NRQCD Crank-Nicolson systems
// (replaces PETSc KSP, nrqcd.f90:786-804, 1103-1105, 1123, 1161).
//
// A CN step of R colour-vector fields psi_r solves
//   (1 + beta_r K) x_r = y_r,   y_r = (1 + alpha_r K) psi_r
// for all r at once; every stencil launch streams the links once per chunk of
// NC slots.  Solvers:
//  * KRYLOV_GMRES_FP64: GMRES(m), FP64, zero guess (PETSc's defaults).  K is
//    Hermitian, so classical Gram-Schmidt needs the last two basis vectors only
//    (k_gm_lanczos).
//  * KRYLOV_GMRES_MIXED: FP64 iterative refinement around FP32 GMRES(m)
//    corrections.
//  * KRYLOV_FGMRES_CNN: flexible GMRES(m) in FP64 whose right preconditioner
//    is z = v - f1 + f2 + N(v, f1, f2) with f1 = beta K v, f2 = beta K f1:
//    the second-order Neumann polynomial of A^-1 corrected by the learned
//    network of nrq_cnn.hip, which sees each direction with its two
//    covariant features (K is the covariant Laplacian, so the inputs
//    transform like v under gauge transformations, and the beta scaling
//    makes them mass-independent).
//  * KRYLOV_FGMRES_CNN_MIXED: FP64 iterative refinement around FP32 FGMRES(m)
//    corrections with the same network.
//  * KRYLOV_CHEB_FP64 / KRYLOV_CHEB_MIXED: Chebyshev iteration on the known
//    spectral segment of A_r, in FP64 or as FP32 corrections inside FP64
//    iterative refinement.  Step counts are planned from a priori bounds, so
//    the usual CN step needs one host synchronisation; the FP64 true residual
//    then confirms convergence (and more steps, or GMRES, follow if not).
// In every case ||y - A x|| <= tol ||y|| with the FP64 operator decides
// convergence: precision and solver change the work, never the answer.
#include "nrq_krylov.h"
#include "nrq_cnn.h"
#include "nrq_gmres.h"
#include "nrq_hop_tile.h"
#include "nrq_map.h"
#include <algorithm>
#include <cmath>
#include <complex>
#include <cstdio>
#include <cstdlib>
#include <cstring>

namespace nrq {

const void *gauge_links(const nrq_gauge *h);

constexpr int CHEB_MAX = 64;  // Chebyshev steps per coefficient table
constexpr int SBS = 256;      // threads per block in the stencil kernels (site-block maps)
constexpr int SBS_WAVE = 512; // at most, with one work item per wavefront (wave-item map)
#ifndef CN_WAVES
#define CN_WAVES 4 // wavefronts per SIMD the stencil kernels' registers must allow
#endif
constexpr double FP32_CORR_ERR = 1e-6; // relative error assumed for an FP32 correction

// ---------------------------------------------------------------------------
// device helpers
// ---------------------------------------------------------------------------

// Re(conj(a) b) in FP64
template <typename T> __device__ __forceinline__ double redot(cplx<T> a, cplx<T> b)
{
    return (double)a.re * b.re + (double)a.im * b.im;
}

template <typename T> __device__ __forceinline__ cplx<T> to(cplx<double> a) { return {(T)a.re, (T)a.im}; }

__device__ __forceinline__ double g_dsum(const geom &g)
{
    return 1.0 / (g.a[1] * g.a[1]) + 1.0 / (g.a[2] * g.a[2]) + 1.0 / (g.a[3] * g.a[3]);
}

// Per-slot fields of one chunk, read in the compute type T (NT: streaming
// loads, for values no other thread reads).  The slot pointers are the same
// for a whole block, so every load is a scalar base plus a 32-bit offset.
template <int NC, typename T, typename S, bool NT = false> struct ld_fields {
    const cplx<S> *f[NC];
    __device__ __forceinline__ cplx<T> operator()(int q, int c, int64_t vol, uint32_t site) const
    {
        const cplx<S> *p = at32(f[q] + (int64_t)c * vol, site);
        const cplx<S> v = NT ? load_nt(p) : *p;
        return {(T)v.re, (T)v.im};
    }
};

// hop_q = sum_i (U_i(x) f_q(x+i) + U_i(x-i)^+ f_q(x-i)) / a_i^2 at x = s for
// the slots q < NC of one chunk; with dsum = sum_i 1/a_i^2 the kinetic
// operator of nrqcd.f90:1210-1242 (without its coefficient) is
//   K f(s) = dsum f(s) - hop / 2
//          = sum_i [f(s) - (U_i(s) f(s+i) + U_i(s-i)^+ f(s-i))/2] / a_i^2.
// ld(q, c, V, site) returns colour c of slot q's field at site; it
// must be readable for every q (a chunk's unused slots read a used slot's
// field, and the caller drops their results).  The kernels are bound by
// memory latency, so each of the six hops issues its 9 link loads and all
// 3 NC field loads at once, with no branch between them: one round trip per
// hop.  Only rows 1 and 2 of each link are read and row 3 is rebuilt as
// conj(row1 x row2), exact for SU(3) up to the links' rounding, a third fewer
// link loads, which are half of these kernels' memory time: for FP64 links
// (rebuilt to FP64 rounding) and in FP32 arithmetic on FP32 links (the
// correction solves, whose results the FP64 residual checks).  FP64
// arithmetic on FP32-stored links reads whole links, so that the FP64
// residual is that of the stored operator and not of its SU(3) projection.
template <int NC, typename T, typename RL, typename LD>
__device__ __forceinline__ void hop_chunk(const cplx<RL> *__restrict__ u, const LD &ld, const lsite &p, const geom &g,
                                          cplx<T> (&hop)[NC][3])
{
#pragma unroll
    for (int q = 0; q < NC; ++q)
#pragma unroll
        for (int c = 0; c < 3; ++c) hop[q][c] = {T(0), T(0)};
    // a loop, not unrolled: unrolled, the compiler hoists the loads of all six
    // hops to the top and spills them
#pragma unroll 1
    for (int h = 0; h < 6; ++h) {
        const int i = h >> 1;
        const bool fwd = (h & 1) == 0;
        const T ia2 = T(1.0 / (g.a[i + 1] * g.a[i + 1]));
        // forward: U_i(s) and f(s+i); backward: U_i(s-i) and f(s-i)
        const int64_t sl = fwd ? p.s : site_dn(g, p, i).s;
        const int64_t sf = fwd ? site_up(g, p, i).s : sl;
        constexpr bool REC = sizeof(RL) == 8 || sizeof(T) == 4;
        constexpr int NE = REC ? 6 : 9;
        cplx<RL> lk[9];
        cplx<T> f[NC][3];
#pragma unroll
        for (int e = 0; e < NE; ++e) lk[e] = *at32(u + ((int64_t)i * 9 + e) * g.vol, (uint32_t)sl);
#pragma unroll
        for (int q = 0; q < NC; ++q)
#pragma unroll
            for (int c = 0; c < 3; ++c) f[q][c] = ld(q, c, g.vol, (uint32_t)sf);
        // hop += (U f) / a_i^2, the product in the compute type
        cplx<T> w[9];
#pragma unroll
        for (int e = 0; e < NE; ++e) w[e] = {(T)lk[e].re, (T)lk[e].im};
        if (REC)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const int c1 = (c + 1) % 3, c2 = (c + 2) % 3;
                cplx<T> v = {T(0), T(0)};
                mac_cc(v, w[c1], w[3 + c2]);
                const cplx<T> a = {-w[c2].re, -w[c2].im};
                mac_cc(v, a, w[3 + c1]);
                w[6 + c] = v;
            }
#pragma unroll
        for (int q = 0; q < NC; ++q)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                cplx<T> t = {T(0), T(0)};
                if (fwd) {
                    mac(t, w[3 * c], f[q][0]);
                    mac(t, w[3 * c + 1], f[q][1]);
                    mac(t, w[3 * c + 2], f[q][2]);
                } else {
                    mac_cn(t, w[c], f[q][0]);
                    mac_cn(t, w[3 + c], f[q][1]);
                    mac_cn(t, w[6 + c], f[q][2]);
                }
                hop[q][c].re = fmx(ia2, t.re, hop[q][c].re);
                hop[q][c].im = fmx(ia2, t.im, hop[q][c].im);
            }
    }
}

// The chunk's own values of slot fields: v[q][c] = ld(q, c, V, s), all
// issued before any store of the caller.
template <int NC, typename T, typename LD>
__device__ __forceinline__ void own_chunk(const LD &ld, int64_t s, int64_t vol, cplx<T> (&v)[NC][3])
{
#pragma unroll
    for (int q = 0; q < NC; ++q)
#pragma unroll
        for (int c = 0; c < 3; ++c) v[q][c] = ld(q, c, vol, (uint32_t)s);
}

// Per-slot sums of v[q] over the block (wave = false; every thread of the
// block must call this) or over the wavefront (wave = true: the wave-item
// map, one chunk per wavefront).  The sum of slot r0 + q < nf goes to
// partial[(r0 + q) * nsb + t].
template <int NC>
__device__ __forceinline__ void chunk_partials(double (&v)[NC], int r0, int nf, int64_t t, int64_t nsb,
                                               double *__restrict__ partial, bool wave)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (wave) {
#pragma unroll
        for (int q = 0; q < NC; ++q) {
            const double x = wsum(v[q]);
            if (lane == 0 && r0 + q < nf) partial[(int64_t)(r0 + q) * nsb + t] = x;
        }
        return;
    }
    __shared__ double sh[NC][SBS / 64];
#pragma unroll
    for (int q = 0; q < NC; ++q) {
        const double x = wsum(v[q]);
        if (lane == 0) sh[q][w] = x;
    }
    __syncthreads();
    if (threadIdx.x < NC && r0 + (int)threadIdx.x < nf) {
        const int q = threadIdx.x;
        double x = 0;
        for (int k = 0; k < SBS / 64; ++k) x += sh[q][k];
        partial[(int64_t)(r0 + q) * nsb + t] = x;
    }
}

// ---------------------------------------------------------------------------
// stencil kernels (grid: lf_map with one work item per chunk of NC slots)
// ---------------------------------------------------------------------------

// The slots of chunk r0 that a stencil kernel computes: on[q] for slot
// r0 + q, and every load pointer of an unused slot aimed at the first used
// one (same addresses, so its loads hit the cache).  False when no slot of
// the chunk is used.
template <int NC>
__device__ __forceinline__ bool chunk_slots(int r0, int nf, const int *__restrict__ active, bool (&on)[NC], int (&rs)[NC])
{
    int first = -1;
#pragma unroll
    for (int q = 0; q < NC; ++q) {
        on[q] = r0 + q < nf && (!active || active[r0 + q]);
        if (on[q] && first < 0) first = r0 + q;
    }
#pragma unroll
    for (int q = 0; q < NC; ++q) rs[q] = on[q] ? r0 + q : first;
    return first >= 0;
}

// out_r = in_r + beta_r K in_r for the active slots; with gco (not null)
// instead out_r = -beta_r gco_r K in_r.
template <int NC, typename RL, typename T>
__global__ __launch_bounds__(SBS_WAVE, CN_WAVES) void k_stencil(const cplx<RL> *__restrict__ u, slots<T> in, slots<T> out,
                                                 const cplx<double> *__restrict__ beta, const int *__restrict__ active,
                                                 int nf, geom g, lf_map mp, const cplx<double> *__restrict__ gco)
{
    lsite p;
    int chunk;
    if (!lf_site(mp, g, p, chunk)) return;
    const int64_t s = p.s;
    const int r0 = chunk * NC;
    bool on[NC];
    int rs[NC];
    if (!chunk_slots<NC>(r0, nf, active, on, rs)) return;
    ld_fields<NC, T, T> ld;
#pragma unroll
    for (int q = 0; q < NC; ++q) ld.f[q] = in.p[rs[q]];
    cplx<T> hop[NC][3];
    hop_chunk<NC, T>(u, ld, p, g, hop);
    cplx<T> v0[NC][3];
    own_chunk<NC, T>(ld, s, g.vol, v0);
    const T dsum = T(g_dsum(g));
#pragma unroll
    for (int q = 0; q < NC; ++q) {
        if (!on[q]) continue;
        cplx<T> *o = out.p[r0 + q];
        cplx<T> cf;
        if (gco) {
            const cplx<double> b = beta[r0 + q], gc = gco[r0 + q];
            cf = to<T>(cplx<double>{-(b.re * gc.re - b.im * gc.im), -(b.re * gc.im + b.im * gc.re)});
        } else {
            cf = to<T>(beta[r0 + q]);
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const cplx<T> kf = dsum * v0[q][c] - T(0.5) * hop[q][c];
            store_nt(at32(o + (int64_t)c * g.vol, (uint32_t)s), gco ? cf * kf : v0[q][c] + cf * kf);
        }
    }
}

// w_r = v_r + beta_r K v_r for the active slots, with the partial <v_r, K v_r>
// per site block (real: K is Hermitian), which costs no reading: both are at
// hand.  64^3, 12 columns, FP64: 83 us without the sum, and 102 us for the pass of dot
// products that it replaces.
template <int NC, typename RL, typename T>
__global__ __launch_bounds__(SBS_WAVE, CN_WAVES) void k_krylov_op(const cplx<RL> *__restrict__ u, slots<T> v, slots<T> w,
                                                   const cplx<double> *__restrict__ beta, const int *__restrict__ active,
                                                   int nf, geom g, lf_map mp, double *__restrict__ partial)
{
    lsite p = {0, 0, 0, 0};
    int64_t t = 0;
    int chunk;
    const bool valid = lf_site(mp, g, p, chunk, t);
    const int64_t s = p.s;
    const int r0 = chunk * NC;
    double kap[NC] = {};
    bool on[NC];
    int rs[NC];
    if (valid && chunk_slots<NC>(r0, nf, active, on, rs)) {
        ld_fields<NC, T, T> ld;
#pragma unroll
        for (int q = 0; q < NC; ++q) ld.f[q] = v.p[rs[q]];
        cplx<T> hop[NC][3];
        hop_chunk<NC, T>(u, ld, p, g, hop);
        cplx<T> v0[NC][3];
        own_chunk<NC, T>(ld, s, g.vol, v0);
        const T dsum = T(g_dsum(g));
#pragma unroll
        for (int q = 0; q < NC; ++q) {
            if (!on[q]) continue;
            const cplx<T> bt = to<T>(beta[r0 + q]);
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const cplx<T> kf = dsum * v0[q][c] - T(0.5) * hop[q][c];
                store_nt(at32(w.p[r0 + q] + (int64_t)c * g.vol, (uint32_t)s), v0[q][c] + bt * kf);
                kap[q] += redot(v0[q][c], kf);
            }
        }
    }
    chunk_partials<NC>(kap, r0, nf, t, mp.nsb, partial, mp.mode >= 3);
}

// Right-hand side and initial guess of a CN step for slot r:
//   y_r = psi_r + alpha_r K psi_r                     (S psi, nrqcd.f90:1112)
//   x_r = psi_r + g_r K psi_r  (guess != 0)  or  x_r = 0  (x.p[r] null: neither)
// with g_r = alpha_r - beta_r the first-order expansion of
// (1 + beta K)^-1 (1 + alpha K).  Partial ||y_r||^2 per site block.  With wk,
// K psi_r also goes to kout in FP32: the guess's residual is exactly
// y - (1 + beta K) x = -beta g K^2 psi.
template <int NC, typename RL>
__global__ __launch_bounds__(SBS_WAVE, CN_WAVES) void k_cn_rhs(const cplx<RL> *__restrict__ u, slots<double> psi, slots<double> y,
                                                slots<double> x, const cplx<double> *__restrict__ alpha,
                                                const cplx<double> *__restrict__ gco, int guess, int nf, geom g, lf_map mp,
                                                double *__restrict__ partial, slots<float> kout, int wk)
{
    lsite p = {0, 0, 0, 0};
    int64_t t = 0;
    int chunk;
    const bool valid = lf_site(mp, g, p, chunk, t);
    const int64_t s = p.s;
    const int r0 = chunk * NC;
    double nrm[NC] = {};
    bool on[NC];
    int rs[NC];
    if (valid && chunk_slots<NC>(r0, nf, nullptr, on, rs)) {
        ld_fields<NC, double, double> ld;
#pragma unroll
        for (int q = 0; q < NC; ++q) ld.f[q] = psi.p[rs[q]];
        cplx<double> hop[NC][3];
        hop_chunk<NC, double>(u, ld, p, g, hop);
        cplx<double> v0[NC][3];
        own_chunk<NC, double>(ld, s, g.vol, v0);
        const double dsum = g_dsum(g);
#pragma unroll
        for (int q = 0; q < NC; ++q) {
            if (!on[q]) continue;
            const int r = r0 + q;
            const cplx<double> a = alpha[r], gc = gco[r];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const int64_t cv = (int64_t)c * g.vol;
                const cplx<double> kf = dsum * v0[q][c] - 0.5 * hop[q][c];
                const cplx<double> yv = v0[q][c] + a * kf;
                store_nt(at32(y.p[r] + cv, (uint32_t)s), yv);
                if (x.p[r])
                    store_nt(at32(x.p[r] + cv, (uint32_t)s), guess ? v0[q][c] + gc * kf : cplx<double>{0.0, 0.0});
                if (wk) store_nt(at32(kout.p[r] + cv, (uint32_t)s), cplx<float>{(float)kf.re, (float)kf.im});
                nrm[q] += nrm2(yv);
            }
        }
    }
    chunk_partials<NC>(nrm, r0, nf, t, mp.nsb, partial, mp.mode >= 3);
}

// True residual r_r = y_r - (1 + beta_r K) x_r in the arithmetic type T for the
// active slots (all when active is null), stored to res as type TR when
// WRITE_RES; partial ||r_r||^2 per site block.
template <int NC, typename RL, typename T, typename TR, bool WRITE_RES>
__global__ __launch_bounds__(SBS_WAVE, CN_WAVES) void k_cn_resid(const cplx<RL> *__restrict__ u, slots<T> x, slots<T> y,
                                                  slots<TR> res, const cplx<double> *__restrict__ beta,
                                                  const int *__restrict__ active, int nf, geom g, lf_map mp,
                                                  double *__restrict__ partial)
{
    lsite p = {0, 0, 0, 0};
    int64_t t = 0;
    int chunk;
    const bool valid = lf_site(mp, g, p, chunk, t);
    const int64_t s = p.s;
    const int r0 = chunk * NC;
    double nrm[NC] = {};
    bool on[NC];
    int rs[NC];
    if (valid && chunk_slots<NC>(r0, nf, active, on, rs)) {
        ld_fields<NC, T, T> ld;
        ld_fields<NC, T, T, true> ly;
#pragma unroll
        for (int q = 0; q < NC; ++q) {
            ld.f[q] = x.p[rs[q]];
            ly.f[q] = y.p[rs[q]];
        }
        cplx<T> hop[NC][3];
        hop_chunk<NC, T>(u, ld, p, g, hop);
        cplx<T> v0[NC][3], yv[NC][3];
        own_chunk<NC, T>(ld, s, g.vol, v0);
        own_chunk<NC, T>(ly, s, g.vol, yv);
        const T dsum = T(g_dsum(g));
#pragma unroll
        for (int q = 0; q < NC; ++q) {
            if (!on[q]) continue;
            const int r = r0 + q;
            const cplx<T> bt = to<T>(beta[r]);
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const cplx<T> rr = yv[q][c] - (v0[q][c] + bt * (dsum * v0[q][c] - T(0.5) * hop[q][c]));
                if (WRITE_RES) store_nt(at32(res.p[r] + (int64_t)c * g.vol, (uint32_t)s), cplx<TR>{(TR)rr.re, (TR)rr.im});
                nrm[q] += nrm2(rr);
            }
        }
    }
    chunk_partials<NC>(nrm, r0, nf, t, mp.nsb, partial, mp.mode >= 3);
}

// One Chebyshev step on the segment [1, 1 + beta_r kmax] of the spectrum of
// A_r = 1 + beta_r K, fused with the operator application:
//   x_{k+1} = rho_r (x_k + (b_r - A_r x_k) / c_r) + (1 - rho_r) x_{k-1}
// c_r = 1 + beta_r kmax / 2 is the segment centre.  mode 0: as above, x_{k-1}
// read from xprev; 1: first step (rho = 1, no x_{k-1}); 2: from a zero start,
// x_k = b / c implicit (xk is b) and x_{k-1} = 0; 3: x_{k-1} = b / c implicit.
// x_{k+1} goes to xnext, or with fin to fout = fin + x_{k+1} in FP64 (the
// last step of a correction solve adds the correction to the FP64 iterate).
// xprev and xnext may be the same fields: each thread reads its own values of
// x_{k-1} before it writes them.
template <int NC, typename RL, typename T>
__global__ __launch_bounds__(SBS_WAVE, CN_WAVES) void k_cheb(const cplx<RL> *__restrict__ u, slots<T> xk, slots<T> xprev, slots<T> xnext,
                                              slots<T> b, const cplx<double> *__restrict__ beta,
                                              const cplx<double> *__restrict__ coef, const int *__restrict__ active, int nf,
                                              geom g, lf_map mp, int mode, int fin, slots<double> fin_in,
                                              slots<double> fin_out)
{
    lsite p;
    int chunk;
    if (!lf_site(mp, g, p, chunk)) return;
    const int64_t s = p.s;
    const int r0 = chunk * NC;
    bool on[NC];
    int rs[NC];
    if (!chunk_slots<NC>(r0, nf, active, on, rs)) return;
    ld_fields<NC, T, T> ld;
    ld_fields<NC, T, T, true> lb, lp;
    ld_fields<NC, double, double, true> lf;
#pragma unroll
    for (int q = 0; q < NC; ++q) {
        ld.f[q] = xk.p[rs[q]];
        lb.f[q] = b.p[rs[q]];
        lp.f[q] = xprev.p[rs[q]];
        lf.f[q] = fin_in.p[rs[q]];
    }
    cplx<T> hop[NC][3];
    hop_chunk<NC, T>(u, ld, p, g, hop);
    cplx<T> v0[NC][3], bs[NC][3];
    own_chunk<NC, T>(ld, s, g.vol, v0);
    if (mode != 2) own_chunk<NC, T>(lb, s, g.vol, bs);
    const T dsum = T(g_dsum(g));
#pragma unroll
    for (int q = 0; q < NC; ++q) {
        if (!on[q]) continue;
        const int r = r0 + q;
        const cplx<T> bt = to<T>(beta[r]);
        const cplx<T> ic = to<T>(coef[2 * r]); // 1 / c_r
        const cplx<T> rho = to<T>(coef[2 * r + 1]);
        const cplx<T> one_m_rho = {T(1) - rho.re, -rho.im};
        // x_{k-1} and the FP64 iterate per slot (xprev may be xnext)
        cplx<T> xp[3];
        cplx<double> xo[3];
        if (mode == 0)
#pragma unroll
            for (int c = 0; c < 3; ++c) xp[c] = lp(q, c, g.vol, (uint32_t)s);
        if (fin)
#pragma unroll
            for (int c = 0; c < 3; ++c) xo[c] = lf(q, c, g.vol, (uint32_t)s);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const int64_t cv = (int64_t)c * g.vol;
            const cplx<T> kf = dsum * v0[q][c] - T(0.5) * hop[q][c];
            const cplx<T> bq = mode == 2 ? v0[q][c] : bs[q][c];
            const cplx<T> x0 = mode == 2 ? ic * v0[q][c] : v0[q][c];
            const cplx<T> ax = mode == 2 ? ic * kf : kf;
            cplx<T> nx = rho * (x0 + ic * (bq - (x0 + bt * ax)));
            if (mode == 3) nx = nx + one_m_rho * (ic * bq);
            else if (mode == 0) nx = nx + one_m_rho * xp[c];
            if (fin)
                store_nt(at32(fin_out.p[r] + cv, (uint32_t)s),
                         cplx<double>{xo[c].re + (double)nx.re, xo[c].im + (double)nx.im});
            else
                store_nt(at32(xnext.p[r] + cv, (uint32_t)s), nx);
        }
    }
}

// ---------------------------------------------------------------------------
// the same kernels through LDS tiles (k_hop_tile of nrq_hop_tile.h): what
// each does at a site of slot r once it has the hop
// ---------------------------------------------------------------------------

// k_stencil
template <typename T> struct tile_stencil {
    static constexpr bool NORM = false;
    struct pre {};
    slots<T> src, out;
    const cplx<double> *beta, *gco;
    const int *active;
    __device__ __forceinline__ bool on(int r) const { return !active || active[r]; }
    __device__ __forceinline__ const cplx<T> *in(int r) const { return src.p[r]; }
    __device__ __forceinline__ void load(int, int64_t, uint32_t, pre &) const {}
    __device__ __forceinline__ void use(int r, int64_t vol, uint32_t s, const pre &, const cplx<T> (&f)[3],
                                        const cplx<T> (&hop)[3], T dsum, double &) const
    {
        cplx<double> b = beta[r];
        if (gco) {
            const cplx<double> gc = gco[r];
            b = {-(b.re * gc.re - b.im * gc.im), -(b.re * gc.im + b.im * gc.re)};
        }
        const cplx<T> cf = to<T>(b);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const cplx<T> kf = dsum * f[c] - T(0.5) * hop[c];
            store_nt(at32(out.p[r] + (int64_t)c * vol, s), gco ? cf * kf : f[c] + cf * kf);
        }
    }
    __device__ __forceinline__ void sum(int, unsigned, double) const {}
};

// k_krylov_op
template <typename T> struct tile_krylov_op {
    static constexpr bool NORM = true;
    struct pre {};
    slots<T> v, w;
    const cplx<double> *beta;
    const int *active;
    double *partial;
    int64_t nsb;
    __device__ __forceinline__ bool on(int r) const { return active[r]; }
    __device__ __forceinline__ const cplx<T> *in(int r) const { return v.p[r]; }
    __device__ __forceinline__ void load(int, int64_t, uint32_t, pre &) const {}
    __device__ __forceinline__ void use(int r, int64_t vol, uint32_t s, const pre &, const cplx<T> (&f)[3],
                                        const cplx<T> (&hop)[3], T dsum, double &kap) const
    {
        const cplx<T> bt = to<T>(beta[r]);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const cplx<T> kf = dsum * f[c] - T(0.5) * hop[c];
            store_nt(at32(w.p[r] + (int64_t)c * vol, s), f[c] + bt * kf);
            kap += redot(f[c], kf);
        }
    }
    __device__ __forceinline__ void sum(int r, unsigned i, double v) const { partial[(int64_t)r * nsb + i] = v; }
};

// k_cn_rhs
struct tile_rhs {
    static constexpr bool NORM = true;
    struct pre {};
    slots<double> psi, y, x;
    slots<float> kout;
    const cplx<double> *alpha, *gco;
    double *partial;
    int64_t nsb;
    int guess, wk;
    __device__ __forceinline__ bool on(int) const { return true; }
    __device__ __forceinline__ const cplx<double> *in(int r) const { return psi.p[r]; }
    __device__ __forceinline__ void load(int, int64_t, uint32_t, pre &) const {}
    __device__ __forceinline__ void use(int r, int64_t vol, uint32_t s, const pre &, const cplx<double> (&f)[3],
                                        const cplx<double> (&hop)[3], double dsum, double &nrm) const
    {
        const cplx<double> a = alpha[r], gc = gco[r];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const int64_t cv = (int64_t)c * vol;
            const cplx<double> kf = dsum * f[c] - 0.5 * hop[c];
            const cplx<double> yv = f[c] + a * kf;
            store_nt(at32(y.p[r] + cv, s), yv);
            if (x.p[r]) store_nt(at32(x.p[r] + cv, s), guess ? f[c] + gc * kf : cplx<double>{0.0, 0.0});
            if (wk) store_nt(at32(kout.p[r] + cv, s), cplx<float>{(float)kf.re, (float)kf.im});
            nrm += nrm2(yv);
        }
    }
    __device__ __forceinline__ void sum(int r, unsigned i, double v) const { partial[(int64_t)r * nsb + i] = v; }
};

// k_cn_resid
template <typename T, typename TR, bool WRITE_RES> struct tile_resid {
    static constexpr bool NORM = true;
    struct pre {
        cplx<T> y[3];
    };
    slots<T> x, y;
    slots<TR> res;
    const cplx<double> *beta;
    const int *active;
    double *partial;
    int64_t nsb;
    __device__ __forceinline__ bool on(int r) const { return !active || active[r]; }
    __device__ __forceinline__ const cplx<T> *in(int r) const { return x.p[r]; }
    __device__ __forceinline__ void load(int r, int64_t vol, uint32_t s, pre &v) const
    {
#pragma unroll
        for (int c = 0; c < 3; ++c) v.y[c] = load_nt(at32((const cplx<T> *)y.p[r] + (int64_t)c * vol, s));
    }
    __device__ __forceinline__ void use(int r, int64_t vol, uint32_t s, const pre &v, const cplx<T> (&f)[3],
                                        const cplx<T> (&hop)[3], T dsum, double &nrm) const
    {
        const cplx<T> bt = to<T>(beta[r]);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const cplx<T> rr = v.y[c] - (f[c] + bt * (dsum * f[c] - T(0.5) * hop[c]));
            if (WRITE_RES) store_nt(at32(res.p[r] + (int64_t)c * vol, s), cplx<TR>{(TR)rr.re, (TR)rr.im});
            nrm += nrm2(rr);
        }
    }
    __device__ __forceinline__ void sum(int r, unsigned i, double v) const { partial[(int64_t)r * nsb + i] = v; }
};

// k_cheb; FIN: with the FP64 iterate (fin, FP32 corrections only).  In FP64 it compiles to
// 168 VGPRs and 24 B of scratch per thread (k_cheb: 20 B at 128 VGPRs), which its times include.
template <typename T, bool FIN> struct tile_cheb {
    static constexpr bool NORM = false;
    struct pre {
        cplx<T> b[3], xp[3];
        cplx<double> xo[FIN ? 3 : 1];
    };
    slots<T> xk, xprev, xnext, b;
    slots<double> fin_in, fin_out;
    const cplx<double> *beta, *coef;
    const int *active;
    int mode;
    __device__ __forceinline__ bool on(int r) const { return !active || active[r]; }
    __device__ __forceinline__ const cplx<T> *in(int r) const { return xk.p[r]; }
    __device__ __forceinline__ void load(int r, int64_t vol, uint32_t s, pre &v) const
    {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const int64_t cv = (int64_t)c * vol;
            if (mode != 2) v.b[c] = load_nt(at32((const cplx<T> *)b.p[r] + cv, s));
            if (mode == 0) v.xp[c] = load_nt(at32((const cplx<T> *)xprev.p[r] + cv, s));
            if (FIN) v.xo[c] = load_nt(at32((const cplx<double> *)fin_in.p[r] + cv, s));
        }
    }
    __device__ __forceinline__ void use(int r, int64_t vol, uint32_t s, const pre &v, const cplx<T> (&f)[3],
                                        const cplx<T> (&hop)[3], T, double &) const
    {
        // c_r = 1 + beta_r dsum, so x_k's own value cancels in
        // x_k + (b - x_k - beta_r (dsum x_k - hop / 2)) / c_r = (b + beta_r hop / 2) / c_r
        const cplx<double> bd = beta[r], icd = coef[2 * r], rd = coef[2 * r + 1];
        const cplx<T> ra = to<T>(rd * icd); // rho / c_r
        const cplx<double> half = {0.5 * bd.re, 0.5 * bd.im}, om = {1.0 - rd.re, -rd.im};
        const cplx<T> hb = to<T>(mode == 2 ? half * icd : half), pb = to<T>(mode == 3 ? om * icd : om);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const int64_t cv = (int64_t)c * vol;
            const cplx<T> bq = mode == 2 ? f[c] : v.b[c];
            cplx<T> t = bq, nx = {T(0), T(0)};
            mac(t, hb, hop[c]);
            mac(nx, ra, t);
            if (mode == 3) mac(nx, pb, bq);
            else if (mode == 0) mac(nx, pb, v.xp[c]);
            if (FIN)
                store_nt(at32(fin_out.p[r] + cv, s), cplx<double>{v.xo[c].re + (double)nx.re, v.xo[c].im + (double)nx.im});
            else
                store_nt(at32(xnext.p[r] + cv, s), nx);
        }
    }
    __device__ __forceinline__ void sum(int, unsigned, double) const {}
};

// ---------------------------------------------------------------------------
// vector kernels (grid: VBLOCKS x slots)
// ---------------------------------------------------------------------------

// Coefficients of a CN step, passed by value (three small copies from pageable
// memory held the queue for longer than the launch of this kernel): cpar = alpha and
// alpha - beta, beta, and every slot of mask active.
struct step_params {
    cplx<double> alpha[NSLOTS], beta[NSLOTS];
    unsigned long long mask;
};
__global__ __launch_bounds__(64) void k_set_step(step_params p, cplx<double> *__restrict__ cpar, cplx<double> *__restrict__ beta,
                                                 int *__restrict__ active)
{
    const int r = threadIdx.x;
    if (r >= NSLOTS) return;
    cpar[r] = p.alpha[r];
    cpar[NSLOTS + r] = p.alpha[r] - p.beta[r];
    beta[r] = p.beta[r];
    active[r] = (int)(p.mask >> r & 1ull);
}

// The Chebyshev coefficients of nf slots and k steps (2 nf k <= CHEB_ARGS) into the
// table of stride 2 NSLOTS.
constexpr int CHEB_ARGS = 192;
struct cheb_args {
    cplx<double> v[CHEB_ARGS];
};
__global__ __launch_bounds__(CHEB_ARGS) void k_set_cheb(cheb_args a, int nf, int k, cplx<double> *__restrict__ tab)
{
    const int t = threadIdx.x;
    if (t < 2 * nf * k) tab[(int64_t)2 * NSLOTS * (t / (2 * nf)) + t % (2 * nf)] = a.v[t];
}

// active[r] = bit r of mask
__global__ __launch_bounds__(64) void k_set_mask(int *__restrict__ active, unsigned long long mask)
{
    if (threadIdx.x < NSLOTS) active[threadIdx.x] = (int)(mask >> threadIdx.x & 1ull);
}

template <typename T>
__global__ __launch_bounds__(VTHREADS) void k_norm2(const cplx<T> *__restrict__ x, int64_t n, const int *__restrict__ active,
                                                    double *__restrict__ partial)
{
    const int r = blockIdx.y;
    if (!active[r]) return;
    __shared__ double sh[8];
    double nrm = 0;
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x)
        nrm += nrm2(x[(int64_t)r * n + k]);
    nrm = block_sum(nrm, sh);
    if (threadIdx.x == 0) partial[(int64_t)r * gridDim.x + blockIdx.x] = nrm;
}

// dst32_r = src64_r / sqrt(nrm2[r])  (normalised FP32 right-hand side)
__global__ void k_demote(const cplx<double> *__restrict__ src, cplx<float> *__restrict__ dst, int64_t n,
                         const double *__restrict__ nrm2v, const int *__restrict__ active)
{
    const int r = blockIdx.y;
    if (!active[r]) return;
    const double inv = nrm2v[r] > 0 ? 1.0 / sqrt(nrm2v[r]) : 0.0;
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) {
        const cplx<double> a = src[(int64_t)r * n + k];
        dst[(int64_t)r * n + k] = {(float)(a.re * inv), (float)(a.im * inv)};
    }
}

// x64_r += sqrt(nrm2[r]) d32_r
__global__ void k_promote_add(cplx<double> *__restrict__ x, const cplx<float> *__restrict__ d, int64_t n,
                              const double *__restrict__ nrm2v, const int *__restrict__ active)
{
    const int r = blockIdx.y;
    if (!active[r]) return;
    const double sc = sqrt(nrm2v[r]);
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) {
        const cplx<float> a = d[(int64_t)r * n + k];
        x[(int64_t)r * n + k] = x[(int64_t)r * n + k] + sc * cplx<double>{(double)a.re, (double)a.im};
    }
}

// FP32 copy of rows 1 and 2 of every link ([dir][e][site], e < 6): the FP32
// stencils rebuild row 3, so rows 3 of the copy are neither written nor read.
__global__ void k_links_to_f32(const cplx<double> *__restrict__ u, cplx<float> *__restrict__ v, int64_t vol)
{
    const int64_t n6 = 6 * vol;
    for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < 3 * n6; j += (int64_t)gridDim.x * blockDim.x) {
        const int64_t k = j + (j / n6) * 3 * vol; // dir * 9V + e * V + site
        v[k] = {(float)u[k].re, (float)u[k].im};
    }
}

// dst_r = src_r (n complex numbers per slot)
__global__ void k_copy_slots(slots<double> src, slots<double> dst, int64_t n)
{
    const int r = blockIdx.y;
    const cplx<double> *a = src.p[r];
    cplx<double> *d = dst.p[r];
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) d[k] = a[k];
}

// ---------------------------------------------------------------------------
// workspace
// ---------------------------------------------------------------------------
struct workspace {
    int64_t vol = 0;
    int m = 0;
    int64_t nsb = 0;                   // site blocks of the stencil launches
    int ext[3] = {0, 0, 0};            // lattice extents the buffers were sized for
    int rcap = 0;                      // slots the field buffers hold
    void *basis = nullptr;             // (m+1) x rcap x 3V complex double (or float)
    cplx<double> *y = nullptr, *x = nullptr, *t = nullptr, *res = nullptr;
    cplx<float> *y32 = nullptr, *x32 = nullptr, *t32 = nullptr, *res32 = nullptr;
    cplx<float> *links32 = nullptr;    // FP32 copy of the links for the inner solves
    cplx<double> *beta = nullptr, *cpar = nullptr, *cpart = nullptr;
    gm_state gm = {};                  // GMRES scalars, in the buffers gmz, gmd, gmi
    cplx<double> *gmz = nullptr;
    double *gmd = nullptr;
    int *gmi = nullptr;
    cplx<double> *negone = nullptr;    // -1 per slot: k_stencil with it as gco gives beta K in
    cplx<double> *cheb = nullptr;      // Chebyshev coefficients [iteration][slot][2]
    double *rpart = nullptr, *spart = nullptr, *nrm = nullptr;
    int *active = nullptr;
    cplx<double> *fptr[NSLOTS] = {};   // heavy field of each slot in the current CN step
    cplx<double> *zbasis = nullptr;    // FGMRES: preconditioned directions, m x rcap x 3V
    int zm = 0;
    int *ibuf = nullptr;               // pinned host, NSLOTS each: cycle flags of even and odd steps, used, fallen
    double *nbuf = nullptr;            // pinned host (NRM doubles)
    hipEvent_t ev[2] = {nullptr, nullptr}; // end of even and odd GMRES steps

    // layout of nrm and nbuf, NSLOTS each: working norms, ||y||^2, saved refinement ||r||^2
    static constexpr int NRM_Y = NSLOTS, NRM_SAVED = 2 * NSLOTS, NRM = 3 * NSLOTS;
    static constexpr int I_USED = 2 * NSLOTS, I_FALLEN = 3 * NSLOTS, I_ALL = 4 * NSLOTS;

    void release()
    {
        void *dev[] = {basis, y, x, t, res, y32, x32, t32, res32, links32, beta, cpar, gmz, gmd, gmi, cpart,
                       rpart, spart, nrm, active, cheb, negone};
        for (void *q : dev)
            if (q) (void)hipFree(q);
        if (ibuf) (void)hipHostFree(ibuf);
        if (nbuf) (void)hipHostFree(nbuf);
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
        if (zbasis) (void)hipFree(zbasis);
        *this = workspace();
    }

    // Buffers for lattice volume v, GMRES restart mm and at least r slots
    // (r = 0: the per-slot scalars only; field buffers are kept).
    int reserve(int64_t v, int mm, int r)
    {
        r = std::max(r, rcap);
        const geom &lg = lat().g;
        // the partial-sum buffer depends on the extents, not only on V
        const bool same = lg.n0 == ext[0] && lg.n1 == ext[1] && lg.n2 == ext[2];
        if (v == vol && mm == m && r == rcap && same) return NRQ_OK;
        release();
        const int rc = std::max(r, 1);
        const size_t f64 = (size_t)3 * (size_t)v * sizeof(cplx<double>) * rc;
        const size_t f32 = f64 / 2;
        int64_t sb = 0;
        for (int md = 0; md <= 4; ++md) sb = std::max(sb, make_lf_map(lg, md >= 3 ? SBS_WAVE : SBS, 8, md, 1).nsb);
        const hop_tiles tl = hop_tiles_for(lg, 1); // fewer groups, more runs
        sb = std::max(sb, (int64_t)tl.ntx * tl.nty * tl.nzr);
        auto dm = [](void **p, size_t b) { return hipMalloc(p, b) == hipSuccess; };
        bool ok = dm(&basis, f64 * (size_t)(mm + 1)) && dm((void **)&y, f64) && dm((void **)&x, f64) &&
                  dm((void **)&t, f64) && dm((void **)&res, f64) && dm((void **)&y32, f32) &&
                  dm((void **)&x32, f32) && dm((void **)&t32, f32) && dm((void **)&res32, f32) &&
                  dm((void **)&links32, (size_t)27 * (size_t)v * sizeof(cplx<float>)) &&
                  dm((void **)&beta, sizeof(cplx<double>) * NSLOTS) && dm((void **)&cpar, sizeof(cplx<double>) * 2 * NSLOTS) &&
                  dm((void **)&negone, sizeof(cplx<double>) * NSLOTS) &&
                  dm((void **)&cheb, sizeof(cplx<double>) * 2 * NSLOTS * CHEB_MAX) &&
                  dm((void **)&gmz, sizeof(cplx<double>) * gm_zcount(mm)) &&
                  dm((void **)&gmd, sizeof(double) * gm_dcount(mm)) &&
                  dm((void **)&gmi, sizeof(int) * GM_ICOUNT) &&
                  dm((void **)&cpart, sizeof(cplx<double>) * NSLOTS * (mm + 1) * VBLOCKS) &&
                  dm((void **)&rpart, sizeof(double) * std::max(KRYLOV_REDUCE_DOUBLES, (size_t)NSLOTS * VBLOCKS * 8)) &&
                  dm((void **)&spart, sizeof(double) * NSLOTS * (size_t)sb) && dm((void **)&nrm, sizeof(double) * NRM) &&
                  dm((void **)&active, sizeof(int) * NSLOTS) &&
                  hipHostMalloc((void **)&ibuf, sizeof(int) * I_ALL, hipHostMallocDefault) == hipSuccess &&
                  hipHostMalloc((void **)&nbuf, sizeof(double) * NRM, hipHostMallocDefault) == hipSuccess &&
                  hipEventCreateWithFlags(&ev[0], hipEventDisableTiming) == hipSuccess &&
                  hipEventCreateWithFlags(&ev[1], hipEventDisableTiming) == hipSuccess;
        if (!ok) {
            (void)hipGetLastError();
            release();
            return fail(NRQ_ERR_ALLOC, "CN: workspace allocation failed (V=%lld, m=%d, %d slots)", (long long)v, mm, rc);
        }
        {
            std::vector<cplx<double>> m1(NSLOTS, cplx<double>{-1.0, 0.0});
            if (hipMemcpy(negone, m1.data(), sizeof(cplx<double>) * NSLOTS, hipMemcpyHostToDevice) != hipSuccess) {
                (void)hipGetLastError();
                release();
                return fail(NRQ_ERR_HIP, "CN: workspace initialisation failed");
            }
        }
        gm = gm_layout(mm, gmz, gmd, gmi);
        vol = v;
        m = mm;
        rcap = rc;
        nsb = sb;
        ext[0] = lg.n0;
        ext[1] = lg.n1;
        ext[2] = lg.n2;
        return NRQ_OK;
    }
};
static workspace g_ws;

int krylov_reserve(int64_t vol, int m, int slots) { return g_ws.reserve(vol, m, slots); }
const cplx<double> *krylov_last_rhs() { return g_ws.y; }

static int reserve_zbasis()
{
    if (g_ws.zbasis && g_ws.zm == g_ws.m) return NRQ_OK;
    if (g_ws.zbasis) (void)hipFree(g_ws.zbasis);
    g_ws.zbasis = nullptr;
    const size_t b = (size_t)g_ws.m * g_ws.rcap * 3 * (size_t)g_ws.vol * sizeof(cplx<double>);
    if (hipMalloc((void **)&g_ws.zbasis, b) != hipSuccess) {
        (void)hipGetLastError();
        return fail(NRQ_ERR_ALLOC, "CN: FGMRES basis allocation failed");
    }
    g_ws.zm = g_ws.m;
    return NRQ_OK;
}
void krylov_release() { g_ws.release(); }
double *krylov_reduce_scratch() { return g_ws.rpart; }
double *krylov_host_scratch() { return g_ws.nbuf; }

// The slots with act[r] != 0 as a bit mask.
static unsigned long long mask_of(const std::vector<int> &act)
{
    unsigned long long b = 0;
    for (size_t r = 0; r < act.size(); ++r) b |= (unsigned long long)(act[r] != 0) << r;
    return b;
}

// Slot mask of the next launches (a kernel argument: a copy from pageable host
// memory would hold the queue and the host for longer).
static int upload_active(const std::vector<int> &act)
{
    hipLaunchKernelGGL(k_set_mask, dim3(1), dim3(64), 0, stream(), g_ws.active, mask_of(act));
    NRQ_HIP(hipGetLastError());
    return NRQ_OK;
}

// Launch shape of the stencil kernels: slots per thread (NC, sharing each
// link load) for FP64 and for FP32 arithmetic, and the site-block mapping of
// make_lf_map.  NRQ_CN_SHAPE="nc64,nc32,mode,xcd" in the environment sets
// the initial value, nrq_cn_set_shape changes it.  The results of the shapes agree
// up to rounding: partial sums follow the site blocks (and the LDS tiles of the default
// shape), and the tiled Chebyshev step is an algebraically equal update (tile_cheb).
struct cn_shape {
    // measured fastest at 128^3 with 12 fields: one work item per wavefront,
    // y-band z-sweep order, each XCD walking whole bands
    int nc64 = 2, nc32 = 4, mode = 4, xcd = 8;
};
static bool cn_nc_ok(int v) { return v == 1 || v == 2 || v == 4; }
static cn_shape read_shape()
{
    cn_shape sh;
    if (const char *e = getenv("NRQ_CN_SHAPE")) {
        int a = 0, b = 0, c = 0, d = 0;
        if (sscanf(e, "%d,%d,%d,%d", &a, &b, &c, &d) == 4) {
            if (cn_nc_ok(a)) sh.nc64 = a;
            if (cn_nc_ok(b)) sh.nc32 = b;
            if (c >= 0 && c <= 4) sh.mode = c;
            if (d == 1 || d == 8) sh.xcd = d;
        }
    }
    return sh;
}
static cn_shape &shape_mut()
{
    static cn_shape sh = read_shape();
    return sh;
}
static const cn_shape &shape() { return shape_mut(); }
template <typename T> static int nc_of() { return sizeof(T) == 8 ? shape().nc64 : shape().nc32; }

// stencil launch map for nf slots, nc per thread
static lf_map cn_map(int nf, int nc)
{
    return make_lf_map(lat().g, shape().mode >= 3 ? SBS_WAVE : SBS, shape().xcd, shape().mode, (nf + nc - 1) / nc);
}

// Whether a launch of nf slots goes through the LDS tiles: where they pay
// (hop_tiles_pay) and no other shape than the default was chosen.
static bool use_tiles(int nf, hop_op op, hop_tiles *t)
{
    if (shape().mode != 4 || shape().xcd != 8) return false;
    *t = hop_tiles_for(lat().g, nf);
    return hop_tiles_pay(lat().g, *t, nf, op);
}
static_assert(NSLOT_GROUPS * HT_F == NSLOTS, "hop_tiles_pay has a column for every batch");
template <typename T> constexpr hop_op op_of() { return sizeof(T) == 8 ? HOP_FP64 : HOP_FP32; }
static dim3 tile_grid(const hop_tiles &t) { return dim3(hop_grid(t)); }

// Runs the statements after `nc` with the compile-time chunk width NCV equal
// to nc (1, 2 or 4).
#define NC_DISPATCH(nc, ...)                                                                                             \
    do {                                                                                                                 \
        if ((nc) == 1) {                                                                                                 \
            constexpr int NCV = 1;                                                                                       \
            __VA_ARGS__;                                                                                                 \
        } else if ((nc) == 2) {                                                                                          \
            constexpr int NCV = 2;                                                                                       \
            __VA_ARGS__;                                                                                                 \
        } else {                                                                                                         \
            constexpr int NCV = 4;                                                                                       \
            __VA_ARGS__;                                                                                                 \
        }                                                                                                                \
    } while (0)

static unsigned grid_of(const lf_map &mp) { return lf_blocks(mp); }

// slot r -> base + r * 3V (workspace fields)
template <typename T> static slots<T> ws_slots(cplx<T> *base, int R)
{
    slots<T> t = {};
    for (int r = 0; r < R; ++r) t.p[r] = base + (int64_t)r * 3 * g_ws.vol;
    return t;
}
template <typename T> static slots<T> ws_slots(const cplx<T> *base, int R) { return ws_slots((cplx<T> *)base, R); }

// slot r -> the heavy field of the current CN step
static slots<double> psi_slots(int R)
{
    slots<double> t = {};
    for (int r = 0; r < R; ++r) t.p[r] = g_ws.fptr[r];
    return t;
}

// out[r] = sum of the nblk partials of slot r (r < nf; active may be null),
// also to the pinned host (may be null)
static int fold_slots(const double *partial, int64_t nblk, int nf, const int *active, double *out, double *host)
{
    hipLaunchKernelGGL(k_fold_slots, dim3(nf), dim3(FOLD_THREADS), 0, stream(), partial, nblk, active, out, host);
    NRQ_HIP(hipGetLastError());
    return NRQ_OK;
}

// Waits for the stream: the sums folded so far are in g_ws.nbuf.
static int wait_sums()
{
    NRQ_HIP(hipStreamSynchronize(stream()));
    return NRQ_OK;
}

// out_r = in_r + beta_r K in_r for the active slots
template <typename RL, typename T>
static void launch_stencil(const cplx<RL> *u, const slots<T> &in, const slots<T> &out, int nf,
                           const int *active, const cplx<double> *gco = nullptr)
{
    hop_tiles tl;
    if (use_tiles(nf, op_of<T>(), &tl)) {
        const tile_stencil<T> op = {in, out, g_ws.beta, gco, active};
        hipLaunchKernelGGL((k_hop_tile<RL, T, tile_stencil<T>>), tile_grid(tl), dim3(HT_THREADS), 0, stream(), u, op, nf,
                           lat().g, tl);
        return;
    }
    const int nc = nc_of<T>();
    const lf_map mp = cn_map(nf, nc);
    NC_DISPATCH(nc, hipLaunchKernelGGL((k_stencil<NCV, RL, T>), dim3(grid_of(mp)), dim3(mp.bs), 0, stream(), u, in, out,
                                       g_ws.beta, active, nf, lat().g, mp, gco));
}

// w_r = A_r v_r and partial <v_r, K v_r> to g_ws.spart for the active slots.
// Returns the partials per slot.
template <typename RL, typename T>
static int64_t launch_krylov_op(const cplx<RL> *u, int R, const slots<T> &v, const slots<T> &w, const int *active)
{
    hop_tiles tl;
    if (use_tiles(R, op_of<T>(), &tl)) {
        const int64_t nsb = (int64_t)tl.ntx * tl.nty * tl.nzr;
        const tile_krylov_op<T> op = {v, w, g_ws.beta, active, g_ws.spart, nsb};
        hipLaunchKernelGGL((k_hop_tile<RL, T, tile_krylov_op<T>>), tile_grid(tl), dim3(HT_THREADS), 0, stream(), u, op, R,
                           lat().g, tl);
        return nsb;
    }
    const int nc = nc_of<T>();
    const lf_map mp = cn_map(R, nc);
    NC_DISPATCH(nc, hipLaunchKernelGGL((k_krylov_op<NCV, RL, T>), dim3(grid_of(mp)), dim3(mp.bs), 0, stream(), u, v, w,
                                       g_ws.beta, active, R, lat().g, mp, g_ws.spart));
    return mp.nsb;
}

// One Chebyshev step (k_cheb) for the active slots of R
template <typename RL, typename T>
static void launch_cheb(const cplx<RL> *links, const slots<T> &xk, const slots<T> &xnext, const slots<T> &b,
                        const cplx<double> *cf, int R, int mode, int fin, const slots<double> &fi, const slots<double> &fo)
{
    hop_tiles tl;
    if (use_tiles(R, sizeof(T) == 8 ? HOP_FP64_CHEB : HOP_FP32, &tl)) {
        if constexpr (sizeof(T) == 4) // the FP64 iterate is a correction's
            if (fin) {
                const tile_cheb<T, true> op = {xk, xnext, xnext, b, fi, fo, g_ws.beta, cf, g_ws.active, mode};
                hipLaunchKernelGGL((k_hop_tile<RL, T, tile_cheb<T, true>>), tile_grid(tl), dim3(HT_THREADS), 0, stream(),
                                   links, op, R, lat().g, tl);
                return;
            }
        const tile_cheb<T, false> op = {xk, xnext, xnext, b, fi, fo, g_ws.beta, cf, g_ws.active, mode};
        hipLaunchKernelGGL((k_hop_tile<RL, T, tile_cheb<T, false>>), tile_grid(tl), dim3(HT_THREADS), 0, stream(), links, op, R,
                           lat().g, tl);
        return;
    }
    const int nc = nc_of<T>();
    const lf_map mp = cn_map(R, nc);
    NC_DISPATCH(nc, hipLaunchKernelGGL((k_cheb<NCV, RL, T>), dim3(grid_of(mp)), dim3(mp.bs), 0, stream(), links, xk, xnext,
                                       xnext, b, g_ws.beta, cf, g_ws.active, R, lat().g, mp, mode, fin, fi, fo));
}

// True residual r = y - A x of the R slots x (the active ones; all when active
// is null) in the arithmetic type T (r stored as TR when WRITE); partial
// ||r||^2 to g_ws.spart.  Returns the partials per slot.
template <typename RL, typename T, typename TR, bool WRITE>
static int64_t launch_resid(const cplx<RL> *u, int R, const slots<T> &x, const slots<T> &y, const slots<TR> &res,
                            const int *active)
{
    hop_tiles tl;
    if (use_tiles(R, op_of<T>(), &tl)) {
        const int64_t nsb = (int64_t)tl.ntx * tl.nty * tl.nzr;
        const tile_resid<T, TR, WRITE> op = {x, y, res, g_ws.beta, active, g_ws.spart, nsb};
        hipLaunchKernelGGL((k_hop_tile<RL, T, tile_resid<T, TR, WRITE>>), tile_grid(tl), dim3(HT_THREADS), 0, stream(), u, op,
                           R, lat().g, tl);
        return nsb;
    }
    const int nc = nc_of<T>();
    const lf_map mp = cn_map(R, nc);
    NC_DISPATCH(nc, hipLaunchKernelGGL((k_cn_resid<NCV, RL, T, TR, WRITE>), dim3(grid_of(mp)), dim3(mp.bs), 0, stream(), u, x,
                                       y, res, g_ws.beta, active, R, lat().g, mp, g_ws.spart));
    return mp.nsb;
}

// Right-hand sides y and guesses x of a CN step (k_cn_rhs); partial ||y||^2
// to g_ws.spart.  Returns the partials per slot.
template <typename RL>
static int64_t launch_rhs(const cplx<RL> *u, int R, const slots<double> &psi, const slots<double> &y,
                          const slots<double> &x, int guess, const slots<float> &kout, int wk)
{
    hop_tiles tl;
    if (use_tiles(R, HOP_FP64, &tl)) {
        const int64_t nsb = (int64_t)tl.ntx * tl.nty * tl.nzr;
        const tile_rhs op = {psi, y, x, kout, g_ws.cpar, g_ws.cpar + NSLOTS, g_ws.spart, nsb, guess, wk};
        hipLaunchKernelGGL((k_hop_tile<RL, double, tile_rhs>), tile_grid(tl), dim3(HT_THREADS), 0, stream(), u, op, R,
                           lat().g, tl);
        return nsb;
    }
    const int nc = shape().nc64;
    const lf_map mp = cn_map(R, nc);
    NC_DISPATCH(nc, hipLaunchKernelGGL((k_cn_rhs<NCV, RL>), dim3(grid_of(mp)), dim3(mp.bs), 0, stream(), u, psi, y, x,
                                       g_ws.cpar, g_ws.cpar + NSLOTS, guess, R, lat().g, mp, g_ws.spart, kout, wk));
    return mp.nsb;
}

int krylov_norms2(const cplx<double> *x, int nf, double *out)
{
    std::vector<int> all(nf, 1);
    if (int e = upload_active(all)) return e;
    const int64_t n = 3 * g_ws.vol;
    const unsigned nb = vblocks(n);
    hipLaunchKernelGGL(k_norm2<double>, dim3(nb, nf), dim3(VTHREADS), 0, stream(), x, n, g_ws.active, g_ws.rpart);
    NRQ_HIP(hipGetLastError());
    if (int e = fold_slots(g_ws.rpart, nb, nf, g_ws.active, g_ws.nrm, g_ws.nbuf)) return e;
    if (int e = wait_sums()) return e;
    memcpy(out, g_ws.nbuf, sizeof(double) * nf);
    return NRQ_OK;
}

// f1_r = beta_r K in_r, f2_r = beta_r K f1_r for the active slots of R
template <typename RL, typename T>
static int bk_features(const cplx<RL> *u, const slots<T> &in, const slots<T> &f1, const slots<T> &f2, int R, const int *active)
{
    launch_stencil<RL, T>(u, in, f1, R, active, g_ws.negone);
    launch_stencil<RL, T>(u, f1, f2, R, active, g_ws.negone);
    NRQ_HIP(hipGetLastError());
    return NRQ_OK;
}

int krylov_rhs_features(const nrq_gauge *gf, int R, const cplx<double> **f1, const cplx<double> **f2)
{
    if (R <= 0 || R > g_ws.rcap) return fail(NRQ_ERR_ARG, "CN: %d features for a workspace of %d slots", R, g_ws.rcap);
    std::vector<int> all(R, 1);
    if (int e = upload_active(all)) return e;
    const slots<double> y = ws_slots(g_ws.y, R), a = ws_slots(g_ws.t, R), b = ws_slots(g_ws.res, R);
    const int e = gf->precision == 64 ? bk_features<double, double>((const cplx<double> *)gauge_links(gf), y, a, b, R, g_ws.active)
                                      : bk_features<float, double>((const cplx<float> *)gauge_links(gf), y, a, b, R, g_ws.active);
    if (e) return e;
    *f1 = g_ws.t;
    *f2 = g_ws.res;
    return NRQ_OK;
}

// ||r|| / ||y||; 0 for a zero right-hand side (x = 0 solves it), and not a number
// where one of the two is not finite, so that `rel <= tol` fails
static double rel_of(double rn, double bn) { return bn == 0.0 ? 0.0 : rn / bn; }
// a norm from its square, which rounding may have left below zero
static double norm_of(double v) { return v < 0 ? 0.0 : std::sqrt(v); }

// column solves handed from FGMRES to plain GMRES since the library loaded
static int64_t g_fallbacks = 0;
// CN coefficients beta of the slots of the current step, on the host (the
// learned preconditioner scales its inputs and output per slot)
static cplx<double> g_beta_host[NSLOTS];

// ---------------------------------------------------------------------------
// GMRES(m) core: solves (1 + beta_r K) x_r = b_r for the slots with act[r],
// from the current x (x = 0 when zero_guess: x is then only written, and
// becomes 0 for the slots that need no step), until the T-precision true
// residual satisfies ||b - A x|| <= tol ||b|| or its[r] reaches maxit.
// rel_out[r] receives the last true relative residual.  beta must already be
// on the device; res is scratch, and may hold b.
//
// Without a network the basis is a Lanczos basis: the operator leaves the only dot
// product that is not known beforehand, and the Gram-Schmidt update reads three
// vectors where the dot products and the update of step j read 2 j + 4.  64^3, 12 columns,
// 7 iterations: 1.91 ms a step where orthogonalising against the whole basis took 2.97.  The
// iterates are the same in exact arithmetic, and the counts were on steps
// up to 5,000 times the usual one (77 iterations a column, m = 30 and 8; FP32 corrections
// with m = 8 there need 976 in place of 982 iterations in all).
//
// A step is three launches (operator, Gram-Schmidt update, rotation; four on the
// largest lattices, five with a network) that need nothing from the host: the rotations and the
// decision whether a slot goes on are made on the device (k_gm_step), which
// every kernel of the next step looks at.  The host enqueues step j + 2 once it
// has seen step j end, so the queue does not run empty; the one step enqueued
// too many leaves at its first instruction.
// ---------------------------------------------------------------------------
// With net (FGMRES): z_j = M(W_j), A z_j in place of A W_j, x from the z_j (M
// is positively homogeneous, so z_j carries the scale factor of W_j).  A slot
// whose network output makes the Arnoldi step non-finite, whose cycle reduces
// its residual by less than FGMRES_STALL, or that has not converged after
// FGMRES_CYCLES cycles leaves the solve with x intact and fallen[r] = 1, for
// the caller to finish with plain GMRES.
constexpr double FGMRES_STALL = 0.1;
constexpr int FGMRES_CYCLES = 4;
template <typename T, typename RL>
static int gmres_core(const cplx<RL> *links, int R, const cplx<T> *b, const slots<T> &x, cplx<T> *basis, cplx<T> *t,
                      cplx<T> *res, bool zero_guess, const double *bnorm, std::vector<int> act, double tol, int m,
                      int64_t maxit, std::vector<int64_t> &its, double *rel_out, int64_t &cycles,
                      nrq_cnn *net = nullptr, cplx<T> *zbasis = nullptr, std::vector<int> *fallen = nullptr)
{
    const int64_t n = 3 * g_ws.vol;
    const unsigned nb = vblocks(n);
    const gm_state gm = g_ws.gm;
    const slots<T> bs = ws_slots(b, R), rs = ws_slots(res, R);
    std::vector<double> rn(R, 0.0);
    const cplx<T> *r0 = res; // residual the next cycle starts from
    // ||b - A x||^2 of the slots in `on` (device mask) to g_ws.nbuf; WRITE: and the residual to res
    auto residual = [&](bool write, const int *on) -> int {
        const int64_t nsb = write ? launch_resid<RL, T, T, true>(links, R, x, bs, rs, on)
                                  : launch_resid<RL, T, T, false>(links, R, x, bs, rs, on);
        NRQ_HIP(hipGetLastError());
        return fold_slots(g_ws.spart, nsb, R, on, g_ws.nrm, g_ws.nbuf);
    };
    if (zero_guess) {
        r0 = b;
        for (int r = 0; r < R; ++r) rn[r] = bnorm[r];
    } else {
        if (int e = upload_active(act)) return e;
        if (int e = residual(true, g_ws.active)) return e;
        if (int e = wait_sums()) return e;
        for (int r = 0; r < R; ++r) rn[r] = act[r] ? norm_of(g_ws.nbuf[r]) : 0.0;
    }
    for (int r = 0; r < R; ++r) {
        if (!act[r]) continue;
        rel_out[r] = rel_of(rn[r], bnorm[r]);
        if (rn[r] <= tol * bnorm[r]) act[r] = 0;
    }
    std::vector<int> ncycles(R, 0);
    std::vector<double> rn_start(R, 0.0);
    bool first = true;
    while (true) {
        bool any = false;
        for (int r = 0; r < R; ++r) any = any || act[r];
        if (!any) {
            if (first && zero_guess) {
                // no slot needs a step: x = 0
                for (int r = 0; r < R; ++r) NRQ_HIP(hipMemsetAsync(x.p[r], 0, sizeof(cplx<T>) * (size_t)n, stream()));
            }
            break;
        }
        ++cycles;
        rn_start = rn;
        gm_start in = {};
        for (int r = 0; r < R; ++r) {
            in.rn[r] = rn[r];
            in.stop[r] = tol * bnorm[r];
            in.left[r] = (int)std::min<int64_t>(m, std::max<int64_t>(1, maxit - its[r]));
        }
        in.act = mask_of(act);
        hipLaunchKernelGGL(k_gm_begin, dim3(1), dim3(64), 0, stream(), gm, in);
        if (net && r0 == res) {
            // res holds features below: the starting residual moves to the basis
            NRQ_HIP(hipMemcpyAsync(basis, res, sizeof(cplx<T>) * (size_t)n * R, hipMemcpyDeviceToDevice, stream()));
            r0 = basis;
        }
        const gm_basis<T> W = {r0, basis};
        std::vector<int> cycle = act;
        for (int j = 0; j < m; ++j) {
            // with a network the host needs the slots that are left
            const int seen = net ? j - 1 : j - 2;
            if (seen >= 0) {
                NRQ_HIP(hipEventSynchronize(g_ws.ev[seen & 1]));
                bool busy = false;
                for (int r = 0; r < R; ++r) {
                    cycle[r] = *(volatile int *)(g_ws.ibuf + (seen & 1) * NSLOTS + r);
                    busy = busy || cycle[r];
                }
                if (!busy) break;
            }
            cplx<T> *w = basis + (size_t)(j + 1) * R * n;
            const slots<T> vj = ws_slots(W.at(j, 0, R, n), R);
            const int nv = j + 1;
            if (net) {
                // z_j = M(W_j) from W_j and its features beta K W_j (in t) and
                // (beta K)^2 W_j (in res; the next cycle's residual is
                // recomputed after this loop)
                cplx<T> *zj = zbasis + (size_t)j * R * n;
                if (int e = bk_features<RL, T>(links, vj, ws_slots(t, R), rs, R, gm.cyc)) return e;
                const cplx<T> *vp[NSLOTS], *f1p[NSLOTS], *f2p[NSLOTS];
                cplx<T> *zp[NSLOTS];
                for (int r = 0; r < R; ++r) {
                    vp[r] = vj.p[r];
                    f1p[r] = t + (size_t)r * n;
                    f2p[r] = res + (size_t)r * n;
                    zp[r] = zj + (size_t)r * n;
                }
                if (int e = cnn_precondition<T>(net, vp, f1p, f2p, zp, R, cycle.data(), g_beta_host, gm.sc + j, gm.m + 1)) return e;
                launch_stencil<RL, T>(links, ws_slots(zj, R), ws_slots(w, R), R, gm.cyc);
                hipLaunchKernelGGL(k_mdot<T>, dim3(nb, R), dim3(VTHREADS), 0, stream(), W, nv, (const cplx<T> *)w, n, R,
                                   (const int *)gm.cyc, g_ws.cpart);
                hipLaunchKernelGGL(k_gm_dots, dim3((nv * R + 3) / 4), dim3(256), 0, stream(), g_ws.cpart, (int)nb, nv, R, gm);
                hipLaunchKernelGGL(k_cgs_update<T>, dim3(nb, R), dim3(VTHREADS), 0, stream(), W, nv, w, n, R, gm, g_ws.rpart);
            } else {
                const int64_t nsb = launch_krylov_op<RL, T>(links, R, vj, ws_slots(w, R), gm.cyc);
                if (nsb <= LANCZOS_FOLD) {
                    hipLaunchKernelGGL((k_lanczos_update<T, true>), dim3(nb, R), dim3(VTHREADS), 0, stream(), W, j, w, n, R, gm,
                                       g_ws.rpart, g_ws.spart, nsb, g_ws.beta);
                } else {
                    hipLaunchKernelGGL(k_gm_lanczos, dim3(R), dim3(VTHREADS), 0, stream(), g_ws.spart, nsb, j, g_ws.beta, gm);
                    hipLaunchKernelGGL((k_lanczos_update<T, false>), dim3(nb, R), dim3(VTHREADS), 0, stream(), W, j, w, n, R, gm,
                                       g_ws.rpart, g_ws.spart, nsb, g_ws.beta);
                }
            }
            hipLaunchKernelGGL(k_gm_step, dim3(R), dim3(VTHREADS), 0, stream(), g_ws.rpart, (int)nb, j, net ? 1 : 0, gm,
                               g_ws.ibuf + (j & 1) * NSLOTS);
            NRQ_HIP(hipGetLastError());
            NRQ_HIP(hipEventRecord(g_ws.ev[j & 1], stream()));
        }
        hipLaunchKernelGGL(k_gm_solve, dim3(R), dim3(64), 0, stream(), gm, net ? 1 : 0, g_ws.ibuf + workspace::I_USED,
                           g_ws.ibuf + workspace::I_FALLEN);
        const gm_basis<T> X = net ? gm_basis<T>{zbasis, zbasis} : W;
        hipLaunchKernelGGL(k_xupdate<T>, dim3(nb, R), dim3(VTHREADS), 0, stream(), x, X, R, n, gm, first && zero_guess ? 1 : 0);
        // true residual in precision T
        if (int e = residual(false, gm.act)) return e;
        if (int e = wait_sums()) return e;
        first = false;
        bool again = false;
        for (int r = 0; r < R; ++r) {
            if (!act[r]) continue;
            its[r] += g_ws.ibuf[workspace::I_USED + r];
            const bool fell = net && g_ws.ibuf[workspace::I_FALLEN + r];
            if (fell) (*fallen)[r] = 1;
            rn[r] = norm_of(g_ws.nbuf[r]);
            rel_out[r] = rel_of(rn[r], bnorm[r]);
            // a residual that is not finite stays so (with a network plain GMRES takes over)
            if (rn[r] <= tol * bnorm[r] || its[r] >= maxit || (!net && !std::isfinite(rn[r]))) {
                act[r] = 0;
                continue;
            }
            if (net && (fell || !(rn[r] <= FGMRES_STALL * rn_start[r]) || ++ncycles[r] >= FGMRES_CYCLES)) {
                act[r] = 0;
                (*fallen)[r] = 1;
            }
            again = again || act[r];
        }
        if (again) {
            // another cycle starts from the residual: one more pass stores it
            if (int e = upload_active(act)) return e;
            if (int e = residual(true, g_ws.active)) return e;
            r0 = res;
        }
    }
    return NRQ_OK;
}

// ---------------------------------------------------------------------------
// Chebyshev iteration.  A_r = 1 + beta_r K is normal and K has its spectrum in
// [0, kmax], kmax = sum_i 2/a_i^2 (K = sum_i (1 - (T_i + T_i^+)/2)/a_i^2 with
// unitary hops T_i), so the spectrum of A_r lies on the segment from 1 to
// 1 + beta_r kmax.  With centre c and half-width d of that segment and
// sigma = c/d, the residual after k steps is bounded by ||r0|| / |T_k(sigma)|.
// ---------------------------------------------------------------------------
typedef std::complex<double> zc;

static double cheb_kmax()
{
    const geom &g = lat().g;
    return 2.0 / (g.a[1] * g.a[1]) + 2.0 / (g.a[2] * g.a[2]) + 2.0 / (g.a[3] * g.a[3]);
}

// 1 / |T_k(sigma)|
static double cheb_bound(zc sg, int k)
{
    zc t0 = 1.0, t1 = sg;
    for (int j = 1; j < k; ++j) {
        const zc t2 = 2.0 * sg * t1 - t0;
        t0 = t1;
        t1 = t2;
    }
    return 1.0 / std::abs(t1);
}

// Smallest k < CHEB_MAX with 1/|T_k(sigma)| <= target (CHEB_MAX if none).
static int cheb_steps(zc sg, double target)
{
    for (int k = 1; k < CHEB_MAX; ++k)
        if (cheb_bound(sg, k) <= target) return k;
    return CHEB_MAX;
}

// Bound on ||y - A x0|| / ||y|| for the initial guess.  With the first-order
// guess x0 = psi + (alpha - beta) K psi the residual is
// -beta (alpha - beta) K^2 psi, and ||y|| >= min_{0<=l<=kmax} |1 + alpha l| ||psi||.
static double guess_bound(zc a, zc b, bool guess, double kmax)
{
    if (!guess) return 1.0;
    const double lam = a.real() < 0 ? std::min(kmax, -a.real() / std::norm(a)) : 0.0;
    const double mn = std::abs(1.0 + a * lam);
    if (!(mn > 0)) return 1.0;
    return std::min(1.0, 1.05 * std::abs(b) * std::abs(a - b) * kmax * kmax / mn);
}

// Coefficient table for k steps; tab[j] = {1/c_r, rho_r of step j}.
static int cheb_table(int R, const std::vector<zc> &beta, int k, double kmax)
{
    std::vector<cplx<double>> tab((size_t)2 * NSLOTS * k, cplx<double>{0.0, 0.0});
    for (int r = 0; r < R; ++r) {
        const zc c = 1.0 + beta[r] * (kmax / 2), d = beta[r] * (kmax / 2);
        const zc sg = c / d, ic = 1.0 / c;
        zc rho = 1.0;
        for (int j = 0; j < k; ++j) {
            if (j == 1) rho = 1.0 / (1.0 - 1.0 / (2.0 * sg * sg));
            else if (j > 1) rho = 1.0 / (1.0 - rho / (4.0 * sg * sg));
            tab[(size_t)2 * NSLOTS * j + 2 * r] = {ic.real(), ic.imag()};
            tab[(size_t)2 * NSLOTS * j + 2 * r + 1] = {rho.real(), rho.imag()};
        }
    }
    if (2 * R * k <= CHEB_ARGS) { // 12 slots and 8 steps, 48 and 2
        cheb_args a = {};
        for (int j = 0; j < k; ++j) std::copy_n(&tab[(size_t)2 * NSLOTS * j], 2 * R, &a.v[2 * R * j]);
        hipLaunchKernelGGL(k_set_cheb, dim3(1), dim3(CHEB_ARGS), 0, stream(), a, R, k, g_ws.cheb);
        NRQ_HIP(hipGetLastError());
        return NRQ_OK;
    }
    NRQ_HIP(hipMemcpyAsync(g_ws.cheb, tab.data(), sizeof(cplx<double>) * tab.size(), hipMemcpyHostToDevice, stream()));
    return NRQ_OK;
}

// k Chebyshev steps on A x = b for the active slots.  zero_start: x starts at
// 0 and steps 0 and 1 are folded into the first launch (k >= 2); otherwise
// from the iterate in `x`.  x and xalt alternate; *out receives the buffer
// holding x_k.  With fin_in/fin_out the last step instead stores
// fin_out = fin_in + x_k in FP64.
template <typename RL, typename T>
static int cheb_run(const cplx<RL> *links, int R, const cplx<T> *b, cplx<T> *x, cplx<T> *xalt, bool zero_start,
                    const std::vector<zc> &beta, int k, double kmax, cplx<T> **out, const slots<double> *fin_in = nullptr,
                    const slots<double> *fin_out = nullptr)
{
    if (zero_start && k < 2) k = 2;
    if (k > CHEB_MAX) k = CHEB_MAX;
    if (int e = cheb_table(R, beta, k, kmax)) return e;
    const slots<T> tb = ws_slots(b, R);
    const slots<double> none = {};
    cplx<T> *cur = x, *other = xalt;
    for (int j = zero_start ? 1 : 0; j < k; ++j) {
        const int mode = zero_start ? (j == 1 ? 2 : (j == 2 ? 3 : 0)) : (j == 0 ? 1 : 0);
        // mode 2 reads b and writes cur; the other modes read cur and write other
        const slots<T> txk = mode == 2 ? tb : ws_slots(cur, R);
        const slots<T> tnext = ws_slots(mode == 2 ? cur : other, R);
        const int fin = (fin_in && j == k - 1) ? 1 : 0;
        const slots<double> fi = fin ? *fin_in : none, fo = fin ? *fin_out : none;
        const cplx<double> *cf = g_ws.cheb + (size_t)2 * NSLOTS * j;
        launch_cheb<RL, T>(links, txk, tnext, tb, cf, R, mode, fin, fi, fo);
        if (mode != 2) std::swap(cur, other);
    }
    NRQ_HIP(hipGetLastError());
    *out = cur;
    return NRQ_OK;
}

// FP64 true residual of the slot fields x with its norms into g_ws.nrm[0, R);
// res32 (may be null) receives the residual in FP32.
template <typename RL>
static int cn_resid(const cplx<RL> *u, int R, const slots<double> &x, cplx<float> *res32)
{
    const slots<double> y = ws_slots(g_ws.y, R);
    int64_t nsb;
    if (res32)
        nsb = launch_resid<RL, double, float, true>(u, R, x, y, ws_slots(res32, R), nullptr);
    else
        nsb = launch_resid<RL, double, float, false>(u, R, x, y, slots<float>{}, nullptr);
    NRQ_HIP(hipGetLastError());
    return fold_slots(g_ws.spart, nsb, R, nullptr, g_ws.nrm, g_ws.nbuf);
}

// Per-slot convergence check of the residual norms in g_ws.nbuf; returns
// true if a slot is still active.  need[r] receives the residual reduction
// still needed.
static bool check_slots(int R, const std::vector<double> &bn, double tol, std::vector<int> &act, std::vector<double> &rel,
                        std::vector<double> &need)
{
    bool any = false;
    for (int r = 0; r < R; ++r) {
        if (!act[r]) continue;
        const double rr = norm_of(g_ws.nbuf[r]);
        rel[r] = rel_of(rr, bn[r]);
        if (rr <= tol * bn[r] || !std::isfinite(rr)) { // not finite: no step mends that
            act[r] = 0;
            continue;
        }
        any = true;
        need[r] = 0.3 * tol * bn[r] / rr;
    }
    return any;
}

// Chebyshev solve from the guess in g_ws.x.  On return *in_psi tells whether
// the iterate is already in the heavy field (else in *xfinal).  Slots still
// active on return go on with GMRES.
template <typename RL>
static int cheb_solve(const cplx<RL> *u, int R, const std::vector<zc> &alpha, const std::vector<zc> &beta,
                      std::vector<double> &bn, const krylov_params &p, std::vector<int> &act, std::vector<double> &rel,
                      std::vector<int64_t> &its, int64_t &cycles, cplx<double> **xfinal, bool *in_psi)
{
    const double kmax = cheb_kmax();
    std::vector<zc> sig(R);
    std::vector<double> b0(R);
    for (int r = 0; r < R; ++r) {
        const zc d = beta[r] * (kmax / 2);
        sig[r] = std::abs(d) > 0 ? (1.0 + d) / d : zc(1e30, 0.0);
        b0[r] = guess_bound(alpha[r], beta[r], p.extrapolate, kmax);
    }
    std::vector<double> need(R, 1.0);
    auto steps_for = [&](double floor_) {
        int k = 1;
        for (int r = 0; r < R; ++r)
            if (act[r]) k = std::max(k, cheb_steps(sig[r], std::max(need[r], floor_)));
        return k;
    };
    auto bn_from_host = [&]() {
        for (int r = 0; r < R; ++r) bn[r] = norm_of(g_ws.nbuf[workspace::NRM_Y + r]);
    };
    *in_psi = false;
    if (p.kind == KRYLOV_CHEB_FP64) {
        // the first round takes enough steps for the a priori guess bound
        for (int r = 0; r < R; ++r) need[r] = 0.3 * p.tol / b0[r];
        cplx<double> *x = g_ws.x;
        for (int round = 0; round < 8; ++round) {
            const int k = steps_for(0.0);
            ++cycles;
            cplx<double> *xk = nullptr;
            if (int e = cheb_run<RL, double>(u, R, g_ws.y, x, x == g_ws.x ? g_ws.t : g_ws.x, false, beta, k, kmax, &xk)) return e;
            x = xk;
            for (int r = 0; r < R; ++r) its[r] += act[r] ? k : 0;
            if (int e = cn_resid<RL>(u, R, ws_slots(x, R), nullptr)) return e;
            if (int e = wait_sums()) return e;
            if (round == 0) bn_from_host();
            if (!check_slots(R, bn, p.tol, act, rel, need)) break;
            if (int e = upload_active(act)) return e;
        }
        *xfinal = x;
        return NRQ_OK;
    }
    // mixed: FP64 residual -> FP32 Chebyshev correction d from zero whose
    // last step stores x + d into the heavy field (from the guess the first
    // time, in place afterwards)
    const cplx<float> *l32;
    if (sizeof(RL) == 8) {
        hipLaunchKernelGGL(k_links_to_f32, dim3(4096), dim3(256), 0, stream(), (const cplx<double> *)u, g_ws.links32, g_ws.vol);
        NRQ_HIP(hipGetLastError());
        l32 = g_ws.links32;
    } else {
        l32 = (const cplx<float> *)u;
    }
    const slots<double> tpsi = psi_slots(R), tx = ws_slots(g_ws.x, R);
    if (p.extrapolate) {
        // the guess's residual -beta g K^2 psi from K psi (FP32, left in t32
        // by the right-hand-side pass): one FP32 stencil pass instead of an
        // FP64 residual pass; the FP64 true residual after the correction
        // still decides
        launch_stencil<float, float>(l32, ws_slots((const cplx<float> *)g_ws.t32, R), ws_slots(g_ws.y32, R), R,
                                     g_ws.active, g_ws.cpar + NSLOTS);
        NRQ_HIP(hipGetLastError());
    } else if (int e = cn_resid<RL>(u, R, tx, g_ws.y32)) {
        return e;
    }
    auto correct = [&](int k) -> int {
        cplx<float> *d = nullptr;
        const slots<double> &from = *in_psi ? tpsi : tx;
        if (int e = cheb_run<float, float>(l32, R, g_ws.y32, g_ws.x32, g_ws.t32, true, beta, k, kmax, &d, &from, &tpsi))
            return e;
        *in_psi = true;
        return cn_resid<RL>(u, R, tpsi, g_ws.y32);
    };
    // corrections planned from the a priori bound, without synchronisation
    std::vector<double> bnd = b0;
    for (int plan = 0; plan < 3; ++plan) {
        bool more = false;
        for (int r = 0; r < R; ++r) {
            need[r] = bnd[r] > 0.3 * p.tol ? 0.3 * p.tol / bnd[r] : 1.0;
            more = more || bnd[r] > 0.3 * p.tol;
        }
        if (!more) break;
        const int k = std::max(2, steps_for(3e-7));
        ++cycles;
        if (int e = correct(k)) return e;
        for (int r = 0; r < R; ++r) {
            its[r] += k;
            bnd[r] *= cheb_bound(sig[r], k) + FP32_CORR_ERR;
        }
    }
    if (!*in_psi) {
        // the bound asks for no correction: the guess goes to the heavy field, and its
        // residual is measured like any other's
        hipLaunchKernelGGL(k_copy_slots, dim3(vblocks(3 * g_ws.vol), R), dim3(VTHREADS), 0, stream(), tx, tpsi, 3 * g_ws.vol);
        NRQ_HIP(hipGetLastError());
        *in_psi = true;
        if (int e = cn_resid<RL>(u, R, tpsi, g_ws.y32)) return e;
    }
    if (int e = wait_sums()) return e;
    bn_from_host();
    // measured corrections (in place) until converged
    for (int round = 0; round < 8; ++round) {
        if (!check_slots(R, bn, p.tol, act, rel, need)) break;
        if (int e = upload_active(act)) return e;
        const int k = std::max(2, steps_for(3e-7));
        ++cycles;
        if (int e = correct(k)) return e;
        for (int r = 0; r < R; ++r) its[r] += act[r] ? k : 0;
        if (int e = wait_sums()) return e;
    }
    return NRQ_OK;
}

// FP64 iterative refinement around FP32 GMRES corrections, from the guess in
// g_ws.x; with net, the corrections are FP32 FGMRES with the network (slots
// the network does not help finish their correction with plain FP32 GMRES).
template <typename RL>
static int gmres_mixed(const cplx<RL> *u, int R, std::vector<double> &bn, const krylov_params &p, std::vector<int> &act,
                       std::vector<double> &rel, std::vector<int64_t> &its, int64_t &cycles, nrq_cnn *net = nullptr)
{
    const int64_t n = 3 * g_ws.vol;
    const cplx<float> *l32;
    if (sizeof(RL) == 8) {
        hipLaunchKernelGGL(k_links_to_f32, dim3(4096), dim3(256), 0, stream(), (const cplx<double> *)u, g_ws.links32, g_ws.vol);
        NRQ_HIP(hipGetLastError());
        l32 = g_ws.links32;
    } else {
        l32 = (const cplx<float> *)u;
    }
    std::vector<double> one(R, 1.0);
    const slots<double> tx = ws_slots(g_ws.x, R), tres = ws_slots(g_ws.res, R);
    for (int outer = 0; outer < 40; ++outer) {
        // FP64 true residual r = y - A x
        const int64_t nsb = launch_resid<RL, double, double, true>(u, R, tx, ws_slots(g_ws.y, R), tres, nullptr);
        NRQ_HIP(hipGetLastError());
        if (int e = fold_slots(g_ws.spart, nsb, R, nullptr, g_ws.nrm, g_ws.nbuf)) return e;
        if (int e = wait_sums()) return e;
        bool any = false;
        for (int r = 0; r < R; ++r) {
            if (!act[r]) continue;
            const double rr = norm_of(g_ws.nbuf[r]);
            rel[r] = rel_of(rr, bn[r]);
            if (rr <= p.tol * bn[r] || its[r] >= p.maxit || !std::isfinite(rr)) act[r] = 0;
            any = any || act[r];
        }
        if (!any) break;
        ++cycles;
        // ||r||^2 of this refinement step at nrm[NRM_SAVED ..): the inner solve reuses nrm[0, R)
        double *rnorm2 = g_ws.nrm + workspace::NRM_SAVED;
        NRQ_HIP(hipMemcpyAsync(rnorm2, g_ws.nrm, sizeof(double) * R, hipMemcpyDeviceToDevice, stream()));
        // normalised FP32 correction problem A d = r / ||r||
        if (int e = upload_active(act)) return e;
        hipLaunchKernelGGL(k_demote, dim3(vblocks(n), R), dim3(VTHREADS), 0, stream(), (const cplx<double> *)g_ws.res, g_ws.y32, n,
                           (const double *)rnorm2, g_ws.active);
        std::vector<double> inner_rel(R, 0.0);
        int64_t inner_cycles = 0;
        const double itol = std::max(p.inner_tol, std::max(p.tol / 1e-3, 2e-7));
        std::vector<int> fallen(R, 0);
        if (int e = gmres_core<float, float>(l32, R, g_ws.y32, ws_slots(g_ws.x32, R), (cplx<float> *)g_ws.basis, g_ws.t32, g_ws.res32, true,
                                             one.data(), act, itol, p.restart, p.maxit, its, inner_rel.data(), inner_cycles,
                                             net, (cplx<float> *)g_ws.zbasis, net ? &fallen : nullptr))
            return e;
        int nfall = 0;
        for (int f : fallen) nfall += f;
        if (nfall) {
            g_fallbacks += nfall;
            if (int e = gmres_core<float, float>(l32, R, g_ws.y32, ws_slots(g_ws.x32, R), (cplx<float> *)g_ws.basis, g_ws.t32, g_ws.res32,
                                                 false, one.data(), fallen, itol, p.restart, p.maxit, its, inner_rel.data(),
                                                 inner_cycles))
                return e;
        }
        // gmres_core left the slot masks of the inner solve on the device;
        // the refinement updates every slot that is still active here
        if (int e = upload_active(act)) return e;
        hipLaunchKernelGGL(k_promote_add, dim3(vblocks(n), R), dim3(VTHREADS), 0, stream(), g_ws.x, (const cplx<float> *)g_ws.x32, n,
                           (const double *)rnorm2, g_ws.active);
        NRQ_HIP(hipGetLastError());
    }
    return NRQ_OK;
}

template <typename RL>
static int cn_step_t(const cplx<RL> *u, int R, const std::vector<zc> &alpha, const std::vector<zc> &beta,
                     const krylov_params &p, nrq_solve_stats *st)
{
    const int64_t n = 3 * g_ws.vol;
    std::vector<double> bn(R, 0.0), rel(R, 0.0);
    std::vector<int64_t> its(R, 0);
    int64_t cycles = 0;
    std::vector<int> act(R, 1);
    const bool guess = p.extrapolate && p.kind != KRYLOV_GMRES_FP64;
    // right-hand sides and guesses; ||y||^2 to nrm[NRM_Y ..)
    const slots<double> tpsi = psi_slots(R), ty = ws_slots(g_ws.y, R), tx = ws_slots(g_ws.x, R);
    // mixed Chebyshev from the guess takes K psi (FP32) for its first correction
    const int wk = guess && p.kind == KRYLOV_CHEB_MIXED ? 1 : 0;
    // GMRES from a zero guess writes x whole
    const bool no_x = !guess && (p.kind == KRYLOV_GMRES_FP64 || p.kind == KRYLOV_FGMRES_CNN);
    const int64_t nsb = launch_rhs<RL>(u, R, tpsi, ty, no_x ? slots<double>{} : tx, guess ? 1 : 0, ws_slots(g_ws.t32, R), wk);
    NRQ_HIP(hipGetLastError());
    if (int e = fold_slots(g_ws.spart, nsb, R, nullptr, g_ws.nrm + workspace::NRM_Y, g_ws.nbuf + workspace::NRM_Y)) return e;
    cplx<double> *xsol = g_ws.x;
    bool in_psi = false;
    int status = NRQ_OK;
    if (p.kind == KRYLOV_CHEB_FP64 || p.kind == KRYLOV_CHEB_MIXED) {
        if (int e = cheb_solve<RL>(u, R, alpha, beta, bn, p, act, rel, its, cycles, &xsol, &in_psi)) return e;
        bool left = false;
        for (int r = 0; r < R; ++r) left = left || act[r];
        if (left) {
            // spectrum bound violated (e.g. links far from unitary): GMRES from here
            if (in_psi) {
                hipLaunchKernelGGL(k_copy_slots, dim3(vblocks(n), R), dim3(VTHREADS), 0, stream(), tpsi, tx, n);
                NRQ_HIP(hipGetLastError());
                in_psi = false;
            } else if (xsol != g_ws.x) {
                NRQ_HIP(hipMemcpyAsync(g_ws.x, xsol, sizeof(cplx<double>) * (size_t)n * R, hipMemcpyDeviceToDevice, stream()));
            }
            xsol = g_ws.x;
            status = gmres_core<double, RL>(u, R, g_ws.y, tx, (cplx<double> *)g_ws.basis, g_ws.t, g_ws.res, false,
                                            bn.data(), act, p.tol, p.restart, p.maxit, its, rel.data(), cycles);
        }
    } else {
        if (int e = wait_sums()) return e;
        for (int r = 0; r < R; ++r) bn[r] = norm_of(g_ws.nbuf[workspace::NRM_Y + r]);
        if (p.kind == KRYLOV_GMRES_FP64) {
            // from a zero guess, straight into the heavy field
            status = gmres_core<double, RL>(u, R, g_ws.y, tpsi, (cplx<double> *)g_ws.basis, g_ws.t, g_ws.res, true,
                                            bn.data(), act, p.tol, p.restart, p.maxit, its, rel.data(), cycles);
            in_psi = true;
        } else if (p.kind == KRYLOV_FGMRES_CNN) {
            nrq_cnn *net = cn_preconditioner();
            if (!net) return fail(NRQ_ERR_STATE, "CN: FGMRES needs a network (nrq_cn_set_preconditioner)");
            if (int e = reserve_zbasis()) return e;
            std::vector<int> fallen(R, 0);
            status = gmres_core<double, RL>(u, R, g_ws.y, tx, (cplx<double> *)g_ws.basis, g_ws.t, g_ws.res,
                                            !p.extrapolate, bn.data(), act, p.tol, p.restart, p.maxit, its, rel.data(),
                                            cycles, net, g_ws.zbasis, &fallen);
            int nfall = 0;
            for (int f : fallen) nfall += f;
            if (!status && nfall) {
                // the network did not help these slots: plain GMRES (the
                // operator's diagonal is constant, so Jacobi scaling leaves
                // GMRES unchanged) from the iterate reached so far
                g_fallbacks += nfall;
                status = gmres_core<double, RL>(u, R, g_ws.y, tx, (cplx<double> *)g_ws.basis, g_ws.t, g_ws.res,
                                                false, bn.data(), fallen, p.tol, p.restart, p.maxit, its, rel.data(),
                                                cycles);
            }
        } else if (p.kind == KRYLOV_FGMRES_CNN_MIXED) {
            nrq_cnn *net = cn_preconditioner();
            if (!net) return fail(NRQ_ERR_STATE, "CN: FGMRES needs a network (nrq_cn_set_preconditioner)");
            if (int e = reserve_zbasis()) return e;
            status = gmres_mixed<RL>(u, R, bn, p, act, rel, its, cycles, net);
        } else
            status = gmres_mixed<RL>(u, R, bn, p, act, rel, its, cycles);
    }
    if (status) return status;
    if (!in_psi) {
        // psi_f = x for every slot
        hipLaunchKernelGGL(k_copy_slots, dim3(vblocks(n), R), dim3(VTHREADS), 0, stream(), ws_slots(xsol, R), tpsi, n);
        NRQ_HIP(hipGetLastError());
    }
    double worst = 0;
    int64_t total = 0;
    for (int r = 0; r < R; ++r) {
        worst = worse(worst, rel[r]);
        total += its[r];
    }
    if (st) {
        st->iterations += total;
        st->restarts += cycles;
        st->max_true_relres = worse(st->max_true_relres, worst);
    }
    if (!(worst <= p.tol))
        return fail(NRQ_ERR_NOCONV, "CN: Krylov solver stopped (maxit=%lld) with true relative residual %.3e > %.1e",
                    (long long)p.maxit, worst, p.tol);
    return NRQ_OK;
}

int krylov_cn_step(const nrq_gauge *gf, cplx<double> *const *fields, int R, const cplx<double> *alpha,
                   const cplx<double> *beta, const krylov_params &p, nrq_solve_stats *st)
{
    if (R <= 0) return NRQ_OK;
    if (R > NSLOTS) return fail(NRQ_ERR_ARG, "CN: %d fields exceed the batch of %d", R, NSLOTS);
    if (g_ws.vol != lat().g.vol || g_ws.rcap < R) return fail(NRQ_ERR_STATE, "CN: workspace not reserved for this solve");
    step_params par = {};
    std::vector<zc> a(R), b(R);
    for (int r = 0; r < R; ++r) {
        if (!fields[r]) return fail(NRQ_ERR_ARG, "CN: null field %d", r);
        g_ws.fptr[r] = fields[r];
        a[r] = zc(alpha[r].re, alpha[r].im);
        b[r] = zc(beta[r].re, beta[r].im);
        par.alpha[r] = alpha[r];
        par.beta[r] = g_beta_host[r] = beta[r];
        par.mask |= 1ull << r;
    }
    hipLaunchKernelGGL(k_set_step, dim3(1), dim3(64), 0, stream(), par, g_ws.cpar, g_ws.beta, g_ws.active);
    NRQ_HIP(hipGetLastError());
    if (gf->precision == 64) return cn_step_t<double>((const cplx<double> *)gauge_links(gf), R, a, b, p, st);
    return cn_step_t<float>((const cplx<float> *)gauge_links(gf), R, a, b, p, st);
}

} // namespace nrq

using namespace nrq;

extern "C" int nrq_cn_set_shape(int nc64, int nc32, int tiling, int xcd_remap)
{
    if (!cn_nc_ok(nc64) || !cn_nc_ok(nc32)) return fail(NRQ_ERR_ARG, "CN shape: slots per thread must be 1, 2 or 4");
    if (tiling < 0 || tiling > 4) return fail(NRQ_ERR_ARG, "CN shape: tiling %d out of range", tiling);
    if (xcd_remap != 1 && xcd_remap != 8) return fail(NRQ_ERR_ARG, "CN shape: XCD remap must be 1 or 8");
    cn_shape &sh = shape_mut();
    sh.nc64 = nc64;
    sh.nc32 = nc32;
    sh.mode = tiling;
    sh.xcd = xcd_remap;
    return NRQ_OK;
}

extern "C" int nrq_cn_get_shape(int *nc64, int *nc32, int *tiling, int *xcd_remap)
{
    if (!nc64 || !nc32 || !tiling || !xcd_remap) return fail(NRQ_ERR_ARG, "null argument");
    const cn_shape &sh = shape();
    *nc64 = sh.nc64;
    *nc32 = sh.nc32;
    *tiling = sh.mode;
    *xcd_remap = sh.xcd;
    return NRQ_OK;
}

extern "C" int nrq_cn_fallbacks(int64_t *count)
{
    if (!count) return fail(NRQ_ERR_ARG, "null argument");
    *count = g_fallbacks;
    return NRQ_OK;
}
