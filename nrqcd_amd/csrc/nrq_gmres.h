// nrq_gmres.h -- vector kernels and device-side scalars of batched GMRES(m),
// shared by the kinetic Crank-Nicolson solvers and the full Hamiltonian.
//
// After the operator, an Arnoldi step of all slots is k_mdot, k_gm_dots,
// k_cgs_update and k_gm_step; for a shifted Hermitian operator k_lanczos_update
// (after k_gm_lanczos on large lattices) and k_gm_step; a cycle is k_gm_begin, its steps, k_gm_solve and
// k_xupdate.  None of them needs the host, and every sum of a slot runs in an
// order that depends on the vector length alone.
#pragma once
#include "nrq_krylov.h"
#include <algorithm>
#include <cmath>

namespace nrq {

constexpr int VBLOCKS = 256;  // most blocks per slot in the vector kernels
constexpr int VTHREADS = 256;

// Base pointers of the slot fields of one launch (3V complex numbers each,
// colour-major); a slot's field may live in the workspace or in the heavy
// field's own storage.  Passed to the kernels by value.
template <typename T> struct slots {
    cplx<T> *p[NSLOTS];
};

__device__ __forceinline__ double wsum(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}

// Block-level sum across the block's waves; result valid in thread 0.
__device__ __forceinline__ double block_sum(double v, double *sh)
{
    v = wsum(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) sh[w] = v;
    __syncthreads();
    double t = 0;
    if (threadIdx.x == 0)
        for (int k = 0; k < (int)(blockDim.x >> 6); ++k) t += sh[k];
    return t;
}

template <typename T> __device__ __forceinline__ double nrm2(cplx<T> a) { return (double)a.re * a.re + (double)a.im * a.im; }

// Blocks per slot of the vector kernels: four elements per thread up to
// VBLOCKS blocks.  Fewer elements per thread cost more in partial sums than
// they gain (16^3, 12 columns: k_mdot with 256 blocks of 48 elements took
// 29 us, with 12 blocks of 1,024 7 us).
static inline unsigned vblocks(int64_t n)
{
    return (unsigned)std::min<int64_t>(VBLOCKS, std::max<int64_t>(1, (n + 4 * VTHREADS - 1) / (4 * VTHREADS)));
}

// Krylov basis of one GMRES cycle.  The vectors are kept as the orthogonal-
// isation left them, W_i, with their scale factors 1 / ||W_i|| beside them
// (gm_state::sc): the unit vectors are v_i = sc_i W_i, and no pass over memory
// normalises them (at 64^3 with 12 columns that pass took 45 us of the 455 us
// of an iteration).  W_0, the residual the cycle starts from, stays where it
// is.
template <typename T> struct gm_basis {
    const cplx<T> *w0; // W_0, slot-major
    cplx<T> *w;        // W_i, i >= 1, at w + i * nf * n
    __device__ __host__ __forceinline__ const cplx<T> *at(int i, int r, int nf, int64_t n) const
    {
        return i == 0 ? w0 + (int64_t)r * n : w + ((int64_t)i * nf + r) * n;
    }
};

// Per-slot GMRES scalars on the device (allocated for restart m): the
// Hessenberg columns and rotations live where the sums are made, so that a
// step's kernels follow each other without the host.
struct gm_state {
    cplx<double> *H;    // [slot][column j][row i], (m + 1) x m per slot, rotated in place
    cplx<double> *sn;   // [slot][m] rotations
    cplx<double> *g;    // [slot][m + 1] rotated right-hand side
    cplx<double> *coef; // [slot][m + 1] coefficients of the next combination of W_i
    double *cs;         // [slot][m]
    double *sc;         // [slot][m + 1] 1 / ||W_i||
    double *stop;       // [slot] |g_{j+1}| at or below this ends the slot's cycle
    int *left;          // [slot] steps the iteration cap still allows
    int *used;          // [slot] columns of the cycle
    int *fallen;        // [slot] the network's direction was not finite
    int *cyc;           // [slot] the slot's cycle goes on
    int *act;           // [slot] the slot is part of this cycle
    int m;
};

// What the host gives a cycle, passed by value.
struct gm_start {
    double rn[NSLOTS], stop[NSLOTS];
    int left[NSLOTS];
    unsigned long long act;
};

// Layout of a gm_state for restart m in three device buffers of gm_zcount(m)
// complex doubles, gm_dcount(m) doubles and GM_ICOUNT ints.
inline size_t gm_zcount(int m) { return (size_t)NSLOTS * ((size_t)(m + 1) * m + m + 2 * (m + 1)); }
inline size_t gm_dcount(int m) { return (size_t)NSLOTS * (m + (m + 1) + 1); }
constexpr size_t GM_ICOUNT = (size_t)NSLOTS * 5;
inline gm_state gm_layout(int m, cplx<double> *z, double *d, int *i)
{
    gm_state gm;
    gm.m = m;
    gm.H = z;
    gm.sn = z + (size_t)NSLOTS * (m + 1) * m;
    gm.g = gm.sn + (size_t)NSLOTS * m;
    gm.coef = gm.g + (size_t)NSLOTS * (m + 1);
    gm.cs = d;
    gm.sc = gm.cs + (size_t)NSLOTS * m;
    gm.stop = gm.sc + (size_t)NSLOTS * (m + 1);
    gm.left = i;
    gm.used = i + NSLOTS;
    gm.fallen = i + 2 * NSLOTS;
    gm.cyc = i + 3 * NSLOTS;
    gm.act = i + 4 * NSLOTS;
    return gm;
}

static __global__ __launch_bounds__(64) void k_gm_begin(gm_state st, gm_start in)
{
    const int r = threadIdx.x;
    if (r >= NSLOTS) return;
    const int on = (int)(in.act >> r & 1ull);
    st.cyc[r] = st.act[r] = on;
    st.used[r] = st.fallen[r] = 0;
    st.stop[r] = in.stop[r];
    st.left[r] = in.left[r];
    st.g[(int64_t)r * (st.m + 1)] = {in.rn[r], 0.0};
    st.sc[(int64_t)r * (st.m + 1)] = in.rn[r] > 0 ? 1.0 / in.rn[r] : 0.0;
}

// partial[r][i][blk] = this block's share of <W_i,r, w_r>, i < nv (FP64 sums).
// The basis vectors go in groups of MDOT_G, each group in one pass that reads
// w_r once (PETSc's VecMDot); per thread and per block the sums run in the
// same order for every grouping.
constexpr int MDOT_G = 8;
template <typename T>
__global__ __launch_bounds__(VTHREADS) void k_mdot(gm_basis<T> basis, int nv, const cplx<T> *__restrict__ w, int64_t n, int nf,
                                                   const int *__restrict__ active, cplx<double> *__restrict__ partial)
{
    const int r = blockIdx.y;
    if (!active[r]) return;
    __shared__ double sh[VTHREADS / 64][2 * MDOT_G];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const cplx<T> *wr = w + (int64_t)r * n;
    for (int i0 = 0; i0 < nv; i0 += MDOT_G) {
        const int gn = nv - i0 < MDOT_G ? nv - i0 : MDOT_G;
        double re[MDOT_G], im[MDOT_G];
        const cplx<T> *b[MDOT_G];
#pragma unroll
        for (int j = 0; j < MDOT_G; ++j) {
            re[j] = im[j] = 0;
            b[j] = basis.at(j < gn ? i0 + j : i0, r, nf, n);
        }
        for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) {
            const cplx<T> x = wr[k];
#pragma unroll
            for (int j = 0; j < MDOT_G; ++j) {
                if (j >= gn) break;
                const cplx<T> a = b[j][k];
                re[j] += (double)a.re * x.re + (double)a.im * x.im;
                im[j] += (double)a.re * x.im - (double)a.im * x.re;
            }
        }
        __syncthreads(); // sh is free (previous group read)
#pragma unroll
        for (int j = 0; j < MDOT_G; ++j) {
            const double x = wsum(re[j]), y = wsum(im[j]);
            if (lane == 0) {
                sh[wv][2 * j] = x;
                sh[wv][2 * j + 1] = y;
            }
        }
        __syncthreads();
        if ((int)threadIdx.x < 2 * gn) {
            double t = 0;
            for (int k = 0; k < VTHREADS / 64; ++k) t += sh[k][threadIdx.x];
            const int j = threadIdx.x >> 1;
            double *o = (double *)&partial[((int64_t)r * nv + i0 + j) * gridDim.x + blockIdx.x];
            o[threadIdx.x & 1] = t;
        }
    }
}

// h_i = <v_i, A v_j> of step j from the partials of <W_i, A W_j>, one wavefront
// per (slot, i) (lane l sums partials l, l + 64, ..., then the wavefront sum: a
// fixed order, and 64 loads in flight instead of one); and the coefficient
// sc_i h_i with which W_i enters the Gram-Schmidt update.
static __global__ __launch_bounds__(256) void k_gm_dots(const cplx<double> *__restrict__ partial, int nblk, int nv, int nf, gm_state st)
{
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (t >= nv * nf) return;
    const int r = t / nv, i = t - r * nv;
    if (!st.cyc[r]) return;
    double re = 0, im = 0;
    for (int b = lane; b < nblk; b += 64) {
        const cplx<double> v = partial[(int64_t)t * nblk + b];
        re += v.re;
        im += v.im;
    }
    re = wsum(re);
    im = wsum(im);
    if (lane == 0) {
        const double *sc = st.sc + (int64_t)r * (st.m + 1);
        const double f = sc[i] * sc[nv - 1];
        const cplx<double> h = {f * re, f * im};
        st.H[((int64_t)r * st.m + nv - 1) * (st.m + 1) + i] = h;
        st.coef[(int64_t)r * (st.m + 1) + i] = sc[i] * h;
    }
}

// Step j of slot r = blockIdx.x for A = 1 + beta K with K Hermitian: the Krylov
// space of A is that of K, so <v_i, A v_j> vanishes for i < j - 1 (Lanczos), and
//   <v_j, A v_j> = 1 + beta kappa,  kappa = <v_j, K v_j> from the operator's partials,
//   <v_{j-1}, A v_j> = beta conj(<v_j, A v_{j-1}> / beta) = (beta / conj(beta)) ||W_j||.
// The column of H (written by the block with `write`) and the two coefficients of the
// Gram-Schmidt update, which thread 0 returns in c.
__device__ __forceinline__ void lanczos_column(const double *__restrict__ partial, int64_t nblk, int r, int j,
                                               const cplx<double> *__restrict__ beta, const gm_state &st, double *sh, bool write,
                                               cplx<double> (&c)[2])
{
    double k = 0;
    for (int64_t b = threadIdx.x; b < nblk; b += VTHREADS) k += partial[(int64_t)r * nblk + b];
    k = block_sum(k, sh);
    if (threadIdx.x != 0) return;
    const double *sc = st.sc + (int64_t)r * (st.m + 1);
    cplx<double> *H = st.H + ((int64_t)r * st.m + j) * (st.m + 1);
    const cplx<double> b = beta[r];
    k *= sc[j] * sc[j];
    const cplx<double> hj = {1.0 + b.re * k, b.im * k};
    c[0] = sc[j] * hj;
    c[1] = {0.0, 0.0};
    if (write) H[j] = hj;
    if (j == 0) return;
    const double b2 = b.re * b.re + b.im * b.im, h = b2 > 0 && sc[j] > 0 ? 1.0 / (sc[j] * b2) : 0.0;
    const cplx<double> hp = h * (b * b);
    c[1] = sc[j - 1] * hp;
    if (!write) return;
    for (int i = 0; i < j - 1; ++i) H[i] = {0.0, 0.0};
    H[j - 1] = hp;
}

// coef[j], coef[j - 1] and the column of H, where k_lanczos_update is not to form them
static __global__ __launch_bounds__(VTHREADS) void k_gm_lanczos(const double *__restrict__ partial, int64_t nblk, int j,
                                                                const cplx<double> *__restrict__ beta, gm_state st)
{
    const int r = blockIdx.x;
    if (!st.cyc[r]) return;
    __shared__ double sh[VTHREADS / 64];
    cplx<double> c[2];
    lanczos_column(partial, nblk, r, j, beta, st, sh, true, c);
    if (threadIdx.x != 0) return;
    cplx<double> *coef = st.coef + (int64_t)r * (st.m + 1);
    coef[j] = c[0];
    if (j) coef[j - 1] = c[1];
}

// W_{j+1} = sc_j (A W_j) - coef_j W_j - coef_{j-1} W_{j-1} (A W_j in w, in place)
// and partial ||W_{j+1}||^2.  With FOLD every block sums the operator's partials itself
// and forms the coefficients, one launch of 3.6 us less per step; it does so where
// there are at most LANCZOS_FOLD of them (each block reads them all).  Without and
// with it: 10 meson steps at 9x14x15 3.83 and 3.60 ms, 45x22x13 with 24 fields (202
// partials) 606 and 589 us, 64^3 with 12 fields (tiles) 1.80 and 1.78 ms a step.
constexpr int64_t LANCZOS_FOLD = 1024;
template <typename T, bool FOLD>
__global__ __launch_bounds__(VTHREADS) void k_lanczos_update(gm_basis<T> basis, int j, cplx<T> *__restrict__ w, int64_t n, int nf,
                                                             gm_state st, double *__restrict__ partial,
                                                             const double *__restrict__ kpart, int64_t nblk,
                                                             const cplx<double> *__restrict__ beta)
{
    const int r = blockIdx.y;
    if (!st.cyc[r]) return;
    __shared__ double sh[8];
    __shared__ cplx<double> cs[2];
    cplx<double> c[2];
    if (FOLD) {
        lanczos_column(kpart, nblk, r, j, beta, st, sh, blockIdx.x == 0, c);
        if (threadIdx.x == 0) cs[0] = c[0], cs[1] = c[1];
        __syncthreads();
        c[0] = cs[0], c[1] = cs[1];
    } else {
        const cplx<double> *coef = st.coef + (int64_t)r * (st.m + 1);
        c[0] = coef[j];
        c[1] = j ? coef[j - 1] : cplx<double>{0.0, 0.0};
    }
    const double scj = st.sc[(int64_t)r * (st.m + 1) + j];
    cplx<T> *wr = w + (int64_t)r * n;
    const cplx<T> *vj = basis.at(j, r, nf, n), *vp = j ? basis.at(j - 1, r, nf, n) : nullptr;
    double nrm = 0;
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) {
        const cplx<T> w0 = wr[k], v = vj[k];
        cplx<double> a = {scj * (double)w0.re, scj * (double)w0.im};
        if (vp) {
            const cplx<T> q = vp[k];
            a = a - c[1] * cplx<double>{(double)q.re, (double)q.im};
        }
        a = a - c[0] * cplx<double>{(double)v.re, (double)v.im};
        const cplx<T> o = {(T)a.re, (T)a.im};
        wr[k] = o;
        nrm += nrm2(o);
    }
    nrm = block_sum(nrm, sh);
    if (threadIdx.x == 0) partial[(int64_t)r * gridDim.x + blockIdx.x] = nrm;
}

// out[r] = sum_b partial[r * nblk + b] for the slot r = blockIdx.x if
// active[r] (active may be null); fixed summation order.  FOLD_THREADS
// threads with four independent sums each keep enough loads in flight for
// the V / 64 partials of the wave-item map.  host (pinned, may be null)
// receives the sums as well.
constexpr int FOLD_THREADS = 1024;
static __global__ __launch_bounds__(FOLD_THREADS) void k_fold_slots(const double *__restrict__ partial, int64_t nblk,
                                                             const int *__restrict__ active, double *__restrict__ out,
                                                             double *__restrict__ host)
{
    const int r = blockIdx.x;
    if (active && !active[r]) return;
    __shared__ double sh[FOLD_THREADS / 64];
    const double *p = partial + (int64_t)r * nblk;
    double s0 = 0, s1 = 0, s2 = 0, s3 = 0;
    constexpr int64_t STEP = 4 * FOLD_THREADS;
    for (int64_t b = threadIdx.x; b < nblk; b += STEP) {
        s0 += p[b];
        if (b + FOLD_THREADS < nblk) s1 += p[b + FOLD_THREADS];
        if (b + 2 * FOLD_THREADS < nblk) s2 += p[b + 2 * FOLD_THREADS];
        if (b + 3 * FOLD_THREADS < nblk) s3 += p[b + 3 * FOLD_THREADS];
    }
    double s = block_sum((s0 + s1) + (s2 + s3), sh);
    if (threadIdx.x == 0) {
        out[r] = s;
        if (host) host[r] = s;
    }
}

// Gram-Schmidt update W_nv = sc_j (A W_j) - sum_{i < nv} coef_i W_i (j = nv - 1,
// A W_j in w, in place) and partial ||W_nv||^2
template <typename T>
__global__ __launch_bounds__(VTHREADS) void k_cgs_update(gm_basis<T> basis, int nv, cplx<T> *__restrict__ w, int64_t n, int nf,
                                                         gm_state st, double *__restrict__ partial)
{
    const int r = blockIdx.y;
    if (!st.cyc[r]) return;
    __shared__ double sh[8];
    cplx<T> *wr = w + (int64_t)r * n;
    const double scj = st.sc[(int64_t)r * (st.m + 1) + nv - 1];
    const cplx<double> *h = st.coef + (int64_t)r * (st.m + 1);
    double nrm = 0;
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) {
        const cplx<T> w0 = wr[k];
        cplx<double> a = {scj * (double)w0.re, scj * (double)w0.im};
        for (int i = 0; i < nv; ++i) {
            const cplx<T> v = basis.at(i, r, nf, n)[k];
            a = a - h[i] * cplx<double>{(double)v.re, (double)v.im};
        }
        const cplx<T> o = {(T)a.re, (T)a.im};
        wr[k] = o;
        nrm += nrm2(o);
    }
    nrm = block_sum(nrm, sh);
    if (threadIdx.x == 0) partial[(int64_t)r * gridDim.x + blockIdx.x] = nrm;
}

// End of Arnoldi step j of slot r = blockIdx.x: ||W_{j+1}|| from its partials,
// the Givens rotation of column j and the residual estimate; the slot's cycle
// ends at `stop`, at its iteration cap, or (net) when a coefficient is not
// finite, which leaves the columns before j (without net such a column ends the
// cycle too and stays in it: x, and the residual that the host then sees, are not
// finite either).  Whether it goes on is also written to *host_cyc (pinned).
static __global__ __launch_bounds__(VTHREADS) void k_gm_step(const double *__restrict__ partial, int nblk, int j, int net, gm_state st,
                                                      int *__restrict__ host_cyc)
{
    const int r = blockIdx.x;
    if (!st.cyc[r]) {
        if (threadIdx.x == 0) host_cyc[r] = 0;
        return;
    }
    __shared__ double sh[VTHREADS / 64];
    double v = 0;
    for (int b = threadIdx.x; b < nblk; b += blockDim.x) v += partial[(int64_t)r * nblk + b];
    v = block_sum(v, sh);
    if (threadIdx.x != 0) return;
    const int m = st.m;
    cplx<double> *H = st.H + ((int64_t)r * m + j) * (m + 1), *g = st.g + (int64_t)r * (m + 1), *sn = st.sn + (int64_t)r * m;
    double *cs = st.cs + (int64_t)r * m;
    if (net) {
        bool fin = isfinite(v);
        for (int i = 0; i <= j; ++i) fin = fin && isfinite(H[i].re) && isfinite(H[i].im);
        if (!fin) {
            st.cyc[r] = 0;
            st.fallen[r] = 1;
            host_cyc[r] = 0;
            return;
        }
    }
    const double hn = v < 0 ? 0.0 : sqrt(v); // what is not a number stays so
    st.sc[(int64_t)r * (m + 1) + j + 1] = hn > 0 ? 1.0 / hn : 0.0;
    cplx<double> a = H[0];
    for (int i = 0; i < j; ++i) {
        const cplx<double> c = H[i + 1];
        H[i] = cs[i] * a + sn[i] * c;
        a = cs[i] * c - cmul(sn[i], a); // -conj(sn) a + cs c
    }
    const double na = sqrt(a.re * a.re + a.im * a.im), den = sqrt(a.re * a.re + a.im * a.im + hn * hn);
    double c = 1;
    cplx<double> sj = {0.0, 0.0};
    if (den > 0) {
        c = na / den;
        sj = na > 0 ? (hn / den / na) * a : cplx<double>{1.0, 0.0};
    }
    cs[j] = c;
    sn[j] = sj;
    H[j] = c * a + hn * sj;
    const cplx<double> gj = g[j];
    const cplx<double> gn = cmul(sj, gj);
    g[j + 1] = {-gn.re, -gn.im};
    g[j] = c * gj;
    st.used[r] = j + 1;
    // not finite: the cycle ends here, and the true residual tells the host
    const bool end = sqrt(gn.re * gn.re + gn.im * gn.im) <= st.stop[r] || j + 1 >= st.left[r] || !isfinite(hn);
    if (end) st.cyc[r] = 0;
    host_cyc[r] = end ? 0 : 1;
}

// End of a cycle: back substitution H y = g of slot r = blockIdx.x, with the
// scale factors of the basis folded into coef; used and fallen go to the
// pinned host arrays.  A solution that is not finite (net) keeps x (used = 0
// in *st.used, with fallen set).
static __global__ __launch_bounds__(64) void k_gm_solve(gm_state st, int net, int *__restrict__ host_used, int *__restrict__ host_fallen)
{
    const int r = blockIdx.x;
    if (threadIdx.x != 0) return;
    const int m = st.m, n = st.act[r] ? st.used[r] : 0;
    cplx<double> *y = st.coef + (int64_t)r * (m + 1);
    const cplx<double> *g = st.g + (int64_t)r * (m + 1);
    const double *sc = st.sc + (int64_t)r * (m + 1);
    host_used[r] = n;
    bool fin = true;
    for (int i = n - 1; i >= 0; --i) {
        cplx<double> s = g[i];
        for (int k = i + 1; k < n; ++k) s = s - st.H[((int64_t)r * m + k) * (m + 1) + i] * y[k];
        const cplx<double> d = st.H[((int64_t)r * m + i) * (m + 1) + i];
        // s / d with d scaled by its larger part first
        const double big = fmax(fabs(d.re), fabs(d.im));
        const cplx<double> q = {d.re / big, d.im / big};
        const double q2 = (q.re * q.re + q.im * q.im) * big;
        const cplx<double> t = cmul(q, s);
        y[i] = {t.re / q2, t.im / q2};
        fin = fin && isfinite(y[i].re) && isfinite(y[i].im);
    }
    for (int i = 0; i < n; ++i) y[i] = sc[i] * y[i];
    if (net && !fin) st.fallen[r] = 1;
    st.used[r] = net && !fin ? 0 : n;
    host_fallen[r] = st.fallen[r];
}

// x_r = (zero ? 0 : x_r) + sum_{i < used_r} coef_i V_i,r with V the basis (or
// the preconditioned directions).  Slots without columns keep x, or get 0.
template <typename T>
__global__ __launch_bounds__(VTHREADS) void k_xupdate(slots<T> x, gm_basis<T> basis, int nf, int64_t n, gm_state st, int zero)
{
    const int r = blockIdx.y;
    const int nv = st.used[r];
    if (nv == 0 && !zero) return;
    cplx<T> *xr = x.p[r];
    const cplx<double> *y = st.coef + (int64_t)r * (st.m + 1);
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) {
        cplx<double> a = {0.0, 0.0};
        if (!zero) {
            const cplx<T> x0 = xr[k];
            a = {(double)x0.re, (double)x0.im};
        }
        for (int i = 0; i < nv; ++i) {
            const cplx<T> v = basis.at(i, r, nf, n)[k];
            a = a + y[i] * cplx<double>{(double)v.re, (double)v.im};
        }
        xr[k] = {(T)a.re, (T)a.im};
    }
}

} // namespace nrq
