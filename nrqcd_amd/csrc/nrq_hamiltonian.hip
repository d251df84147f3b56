// nrq_hamiltonian.hip -- the Crank-Nicolson step with the full NRQCD
// Hamiltonian of BuildSystemMatrix (nrqcd.f90:1175-1387): the kinetic c1 term
// plus the c2 (magnetic), c3 (E derivative) and c4 (spin-orbit) terms, taken
// when any of c2..c4 is non-zero.
//
// S = 1 + sum_t a_t T_t with (dt the step width, pre = -i dt a0 / 2)
//   T_1 psi = sum_i [psi(x) - (U_i(x) psi(x+i) + U_i(x-i)^+ psi(x-i))/2] / a_i^2,
//            a_1 = pre c1 / M;
//   T_2 = C2CS(Bsum(x)),  Bsum = sum_i (F_jk - F_kj)/2 (nrqcd.f90:1669-1693; no
//            Pauli matrix, a reference quirk), a_2 = pre (-c2) / (2M);
//   T_3 = C2CS(Dsum(x)),  Dsum = sum_i (U_i(x) e_i(x+i) U_i(x)^+
//            - U_i(x-i)^+ e_i(x-i) U_i(x-i)) / (2 a_i), e = -F_0i,
//            a_3 = pre (-c3) / (8 M^2);
//   T_4 hops to x +- i with Kron(G, sigma_k) for the cyclic (eps = +1) and
//            anticyclic (eps = -1) (i, j, k):
//            to x + i: G = eps (e_j(x) U_i(x) + U_i(x) e_j(x+i)) / (2 a_i),
//            to x - i: G = -eps (e_j(x) W + W e_j(x-i)) / (2 a_i), W = U_i(x-i)^+,
//            a_4 = pre (-c4) i / (8 M^2).
// The field strength F_ij = Re[ArgLogU(P_ij)] / (a_i a_j) is the element-wise
// real part (gaugeconfiguration_su3.f90:1563-1581) with the spatial plaquette
// or, for F_0j, the temporal plaquette exp(i E_j^a T^a) (:1656-1679).  The
// antiquark uses (-M, conj c) (nrqcd.f90:1130-1161).
//
// Per step: rhs = S psi, then S^+ psi' = rhs (S^+ = 1 + sum_t conj(a_t) T_t^+)
// for every column of both propagators.  c4 mixes the spin rows, so a column
// is the pair of colour-vector fields (2j, 2j+1), 6V complex doubles,
// contiguous in the field storage.  The solver is FP64 GMRES(m) with
// classical Gram-Schmidt and zero initial guess (PETSc's defaults,
// nrqcd.f90:803-804) that stops on the FP64 true relative residual.
//
// The field strengths (kernel k_ham_fields: 3 temporal and 6 spatial
// logarithms per site) and the colour matrices Dsum and G (k_ham_blocks) are
// built once per step; k_ham_apply applies S or S^+ to several columns at
// once.
#include "nrq_gmres.h"
#include "nrq_grouplog.h"
#include "nrq_map.h"
#include <algorithm>
#include <array>
#include <cmath>
#include <cstdlib>
#include <complex>
#include <vector>

namespace nrq {

const void *gauge_links(const nrq_gauge *h);

constexpr int HAM_THREADS = 256;
constexpr int HAM_FLD = 36;   // doubles per site: F0_j (3 x 9), Bsum (9)
constexpr int HAM_BLK = 13;   // colour matrices per site: Dsum, G[i][sign][p]
constexpr int HAM_MAXCOL = 12; // columns per apply launch (6 per propagator)
constexpr int HAM_NC = 2;      // columns per thread of the operator (k_ham_apply has the figures)
constexpr int HAM_FIELD_THREADS = 3 * 64; // k_ham_fields: three wavefronts, 64 sites
constexpr int HAM_SITES = 64;  // threads per block of the operator: one wavefront
constexpr size_t HAM_BATCH_BYTES = (size_t)16 << 30; // Krylov storage of the columns solved together

template <typename R> __device__ __forceinline__ mat3<double> ham_link(const cplx<R> *u, int64_t vol, int dir, int64_t s)
{
    mat3<double> m;
    const cplx<R> *p = u + (int64_t)dir * 9 * vol;
#pragma unroll
    for (int e = 0; e < 9; ++e) {
        const cplx<R> a = p[(int64_t)e * vol + s];
        m.m[e] = {(double)a.re, (double)a.im};
    }
    return m;
}

__device__ __forceinline__ mat3<double> madd(const mat3<double> &a, const mat3<double> &b, double sb)
{
    mat3<double> r;
#pragma unroll
    for (int e = 0; e < 9; ++e) r.m[e] = {a.m[e].re + sb * b.m[e].re, a.m[e].im + sb * b.m[e].im};
    return r;
}

// F0_j(x) and Bsum(x) into fld[(q * 9 + e) V + s], q = 0..2 for F0_j, 3 for Bsum.
// Bound by the 9 matrix logarithms of a site, long dependent chains of FP64
// arithmetic, so they are spread over wavefronts: for 64 sites the three of a block
// with blockIdx.y = 0 take the two plaquette orders of one plane each (the terms of
// Bsum meet in LDS, summed in a fixed order), the three of the other block F0_j.
// 33x30x27: 107 us with one thread per site, 76 us so.
template <typename R>
__global__ __launch_bounds__(HAM_FIELD_THREADS) void k_ham_fields(const cplx<R> *__restrict__ u, const R *__restrict__ ef, geom g,
                                                       double *__restrict__ fld)
{
    __shared__ double part[3][9][64];
    const int lane = threadIdx.x & 63, i = threadIdx.x >> 6;
    const int64_t V = g.vol, s0 = (int64_t)blockIdx.x * 64 + lane;
    const bool in = s0 < V;
    const int64_t s = in ? s0 : V - 1;
    if (blockIdx.y == 1) {
        double al[8];
        for (int a = 0; a < 8; ++a) al[a] = (double)ef[((int64_t)i * 8 + a) * V + s];
        const mat3<double> H = group_log_matrix(exp_i_hermitian(algebra_matrix(al)));
        const double sc = 1.0 / (g.a[0] * g.a[i + 1]);
        if (in)
            for (int e = 0; e < 9; ++e) fld[((int64_t)i * 9 + e) * V + s] = H.m[e].re * sc;
        return;
    }
    const int j = (i + 1) % 3, k = (i + 2) % 3;
    const lsite p = make_site(g, s);
    double b[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    for (int o = 0; o < 2; ++o) {
        // P_mn(x) = U_m(x) U_n(x+m) U_m(x+n)^+ U_n(x)^+ for (m, n) = (j, k), then (k, j)
        const int m = o == 0 ? j : k, n = o == 0 ? k : j;
        const mat3<double> P = mul_nd(mul_nd(mul(ham_link(u, V, m, s), ham_link(u, V, n, site_up(g, p, m).s)),
                                             ham_link(u, V, m, site_up(g, p, n).s)),
                                      ham_link(u, V, n, s));
        const mat3<double> H = group_log_matrix(P);
        const double sc = (o == 0 ? 0.5 : -0.5) / (g.a[m + 1] * g.a[n + 1]);
        for (int e = 0; e < 9; ++e) b[e] += H.m[e].re * sc;
    }
    for (int e = 0; e < 9; ++e) part[i][e][lane] = b[e];
    __syncthreads();
    if (!in) return;
    for (int e = i; e < 9; e += 3)
        fld[((int64_t)27 + e) * V + s] = part[0][e][lane] + part[1][e][lane] + part[2][e][lane];
}

__device__ __forceinline__ mat3<double> ham_e(const double *__restrict__ fld, int64_t V, int j, int64_t s)
{
    mat3<double> m;
#pragma unroll
    for (int e = 0; e < 9; ++e) m.m[e] = {-fld[((int64_t)j * 9 + e) * V + s], 0.0};
    return m;
}

// Dsum (matrix 0) and G[i][sign][p] (matrix 1 + (2 i + sign) 2 + p) into
// blk[(mat * 9 + e) V + s].
template <typename R>
__global__ __launch_bounds__(HAM_THREADS) void k_ham_blocks(const cplx<R> *__restrict__ u, const double *__restrict__ fld,
                                                           geom g, cplx<double> *__restrict__ blk)
{
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.vol) return;
    const int64_t V = g.vol;
    const lsite p = make_site(g, s);
    mat3<double> dsum;
    set_zero(dsum);
    for (int i = 0; i < 3; ++i) {
        const int64_t sp = site_up(g, p, i).s, sm = site_dn(g, p, i).s;
        const double inv2a = 1.0 / (2.0 * g.a[i + 1]);
        const mat3<double> Ui = ham_link(u, V, i, s), Um = ham_link(u, V, i, sm);
        // c3: U e_i(x+i) U^+ - Um^+ e_i(x-i) Um
        const mat3<double> t1 = mul_nd(mul(Ui, ham_e(fld, V, i, sp)), Ui);
        const mat3<double> t2 = mul(mul_dn(Um, ham_e(fld, V, i, sm)), Um);
        dsum = madd(dsum, madd(t1, t2, -1.0), inv2a);
        // c4
        mat3<double> W;
        for (int e = 0; e < 9; ++e) W.m[e] = {Um.m[3 * (e % 3) + e / 3].re, -Um.m[3 * (e % 3) + e / 3].im};
        for (int q = 0; q < 2; ++q) {
            const int j = q == 0 ? (i + 1) % 3 : (i + 2) % 3;
            const double eps = q == 0 ? 1.0 : -1.0;
            const mat3<double> ex = ham_e(fld, V, j, s);
            const mat3<double> gp = madd(mul(ex, Ui), mul(Ui, ham_e(fld, V, j, sp)), 1.0);
            const mat3<double> gm = madd(mul(ex, W), mul(W, ham_e(fld, V, j, sm)), 1.0);
            const int mp = 1 + (2 * i + 0) * 2 + q, mm = 1 + (2 * i + 1) * 2 + q;
            for (int e = 0; e < 9; ++e) {
                blk[((int64_t)mp * 9 + e) * V + s] = {eps * inv2a * gp.m[e].re, eps * inv2a * gp.m[e].im};
                blk[((int64_t)mm * 9 + e) * V + s] = {-eps * inv2a * gm.m[e].re, -eps * inv2a * gm.m[e].im};
            }
        }
    }
    for (int e = 0; e < 9; ++e) blk[(int64_t)e * V + s] = dsum.m[e];
}

struct ham_cols {
    const cplx<double> *in[HAM_MAXCOL];
    cplx<double> *out[HAM_MAXCOL];
    cplx<double> a[HAM_MAXCOL][4];
    const cplx<double> *b; // HAM_RESIDUAL: right-hand sides, column after column
    const int *active;     // columns to work on (may be null: all)
    double *partial;       // HAM_RHS, HAM_RESIDUAL: [column][site block] sums of |out|^2
    int n; // columns
};

// w = sigma_k (a v) with the Pauli matrices of the reference's table
// (su2.f90:68-88): [[0,1],[1,0]], [[0,i],[-i,0]], diag(1,-1).
__device__ __forceinline__ void ham_pauli(int k, cplx<double> a, const cplx<double> (&v)[2][3], cplx<double> (&w)[2][3])
{
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const cplx<double> t0 = a * v[0][c], t1 = a * v[1][c];
        if (k == 0) w[0][c] = t1, w[1][c] = t0;
        else if (k == 1) w[0][c] = {-t1.im, t1.re}, w[1][c] = {t0.im, -t0.re};
        else w[0][c] = t0, w[1][c] = {-t1.re, -t1.im};
    }
}

__device__ __forceinline__ void ham_load(const cplx<double> *__restrict__ x, int64_t V, int64_t s, cplx<double> (&v)[2][3])
{
#pragma unroll
    for (int sp = 0; sp < 2; ++sp)
#pragma unroll
        for (int c = 0; c < 3; ++c) v[sp][c] = x[((int64_t)sp * 3 + c) * V + s];
}

__device__ __forceinline__ mat3<double> ham_blk(const cplx<double> *__restrict__ blk, int64_t V, int m, int64_t s)
{
    mat3<double> r;
#pragma unroll
    for (int e = 0; e < 9; ++e) r.m[e] = blk[((int64_t)m * 9 + e) * V + s];
    return r;
}

// acc[sp] += M v[sp] (ADJ: M^+ v[sp])
template <bool ADJ>
__device__ __forceinline__ void ham_colour(const mat3<double> &M, const cplx<double> (&v)[2][3], cplx<double> (&acc)[2][3])
{
#pragma unroll
    for (int sp = 0; sp < 2; ++sp)
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                if (ADJ) mac_cn(acc[sp][r], M.m[3 * c + r], v[sp][c]);
                else mac(acc[sp][r], M.m[3 * r + c], v[sp][c]);
            }
}

// Ends a stage of the operator: the accumulators are complete before any operand of
// the next stage is loaded.  Without it the compiler gathers the loads of all stages
// ahead of the arithmetic (228 to 489 spilled registers).
template <int NC> __device__ __forceinline__ void ham_stage_end(cplx<double> (&acc)[NC][2][3])
{
#pragma unroll
    for (int q = 0; q < NC; ++q)
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int c = 0; c < 3; ++c) asm volatile("" : "+v"(acc[q][r][c].re), "+v"(acc[q][r][c].im));
    __builtin_amdgcn_sched_barrier(0);
}

enum ham_mode {
    HAM_ADJOINT = 0,  // y = S^+ x
    HAM_RHS = 1,      // y = S x, with the partial sums of |y|^2
    HAM_RESIDUAL = 2, // y = b - S^+ x, with the partial sums of |y|^2
};

// The operator for the columns of `cols`.  Bound by the reads through L2: per
// site 20 colour matrices (links, field strengths and the colour blocks of the
// derivative and spin-orbit terms, 2.8 KB) against 42 numbers of each column, so a
// thread applies the matrices it has loaded to HAM_NC columns; and each term's
// coefficient goes into the vector before the matrix, which leaves one accumulator
// per column where the terms held four.  The grid is site blocks x column groups with the
// group fastest, and each XCD walks one contiguous range of it, so the groups of a
// site block share its matrices through that XCD's L2.  33x30x27,
// 12 columns, FP64: 76 us with one column per thread, 46 us with two; three and four
// (one wavefront per SIMD for their registers) make a whole step 5 and 17 % slower.  The
// residual form, one launch per cycle, spills 20 (FP32 links 28) bytes per thread at 256 VGPRs.
template <typename R, int MODE>
__global__ __launch_bounds__(HAM_SITES, 2) void k_ham_apply(const cplx<R> *__restrict__ u, const double *__restrict__ fld,
                                                         const cplx<double> *__restrict__ blk, geom g, ham_cols cols)
{
    constexpr bool ADJ = MODE != HAM_RHS;
    const unsigned lb = xcd_block(gridDim.x, 8), ng = (unsigned)((cols.n + HAM_NC - 1) / HAM_NC);
    const unsigned sb = lb / ng, c0 = lb % ng * HAM_NC;
    int col[HAM_NC];
    bool on[HAM_NC], any = false;
#pragma unroll
    for (int q = 0; q < HAM_NC; ++q) {
        // the last group repeats the last column
        const bool real = (int)c0 + q < cols.n;
        col[q] = real ? (int)c0 + q : cols.n - 1;
        on[q] = real && (!cols.active || cols.active[col[q]]);
        any = any || on[q];
    }
    if (!any) return;
    const int64_t V = g.vol, t = (int64_t)sb * HAM_SITES + threadIdx.x;
    const bool inside = t < V;
    const int64_t s = inside ? t : V - 1;
    const lsite p = make_site(g, s);
    const double w2[3] = {1.0 / (g.a[1] * g.a[1]), 1.0 / (g.a[2] * g.a[2]), 1.0 / (g.a[3] * g.a[3])};
    auto coef = [&](int q, int k) {
        const cplx<double> a = cols.a[col[q]][k];
        return ADJ ? cplx<double>{a.re, -a.im} : a;
    };
    cplx<double> acc[HAM_NC][2][3], v[HAM_NC][2][3], w[2][3];
    {
        double B[9];
#pragma unroll
        for (int e = 0; e < 9; ++e) B[e] = fld[((int64_t)27 + e) * V + s];
        const mat3<double> D = ham_blk(blk, V, 0, s);
#pragma unroll
        for (int q = 0; q < HAM_NC; ++q) ham_load(cols.in[col[q]], V, s, v[q]);
#pragma unroll
        for (int q = 0; q < HAM_NC; ++q) {
            // 1 + the site-diagonal part of the kinetic term, c2 and c3
            const cplx<double> a0 = coef(q, 0), a1 = coef(q, 1), a2 = coef(q, 2);
            const double ws = w2[0] + w2[1] + w2[2];
            const cplx<double> d = {ws * a0.re, ws * a0.im};
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    acc[q][r][c] = v[q][r][c];
                    mac(acc[q][r][c], d, v[q][r][c]);
                    w[r][c] = a1 * v[q][r][c];
                }
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int c = 0; c < 3; ++c)
#pragma unroll
                    for (int e = 0; e < 3; ++e) {
                        const double b = B[ADJ ? 3 * e + c : 3 * c + e];
                        acc[q][r][c].re += b * w[r][e].re;
                        acc[q][r][c].im += b * w[r][e].im;
                    }
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int c = 0; c < 3; ++c) w[r][c] = a2 * v[q][r][c];
            ham_colour<ADJ>(D, w, acc[q]);
        }
        ham_stage_end(acc);
    }
    // hops to x + i and x - i, one at a time: the operands of all six would not fit
#pragma unroll 1
    for (int h = 0; h < 6; ++h) {
        const int i = h >> 1, dn = h & 1;
        const int64_t sn = dn ? site_dn(g, p, i).s : site_up(g, p, i).s;
        const double w2i = i == 0 ? w2[0] : i == 1 ? w2[1] : w2[2];
#pragma unroll
        for (int q = 0; q < HAM_NC; ++q) ham_load(cols.in[col[q]], V, sn, v[q]);
        const mat3<double> U = ham_link(u, V, i, dn ? sn : s);
        // kinetic: -(U_i(x) v(x+i) or U_i(x-i)^+ v(x-i)) / 2
#pragma unroll
        for (int q = 0; q < HAM_NC; ++q) {
            const cplx<double> a0 = coef(q, 0), f = {-0.5 * w2i * a0.re, -0.5 * w2i * a0.im};
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int c = 0; c < 3; ++c) w[r][c] = f * v[q][r][c];
            if (dn) ham_colour<true>(U, w, acc[q]);
            else ham_colour<false>(U, w, acc[q]);
        }
        ham_stage_end(acc);
        // spin-orbit: G of this site and hop, or the adjoint of the neighbour's G of
        // the opposite hop
        const int gm = 1 + (2 * i + (ADJ ? 1 - dn : dn)) * 2;
#pragma unroll 1
        for (int o = 0; o < 2; ++o) {
            const mat3<double> G = ham_blk(blk, V, gm + o, ADJ ? sn : s);
            const int k = o == 0 ? (i + 2) % 3 : (i + 1) % 3;
#pragma unroll
            for (int q = 0; q < HAM_NC; ++q) {
                ham_pauli(k, coef(q, 3), v[q], w);
                ham_colour<ADJ>(G, w, acc[q]);
            }
            ham_stage_end(acc);
        }
    }
#pragma unroll
    for (int q = 0; q < HAM_NC; ++q) {
        if (!on[q]) continue;
        cplx<double> *y = cols.out[col[q]];
        double nrm = 0;
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const int64_t at = ((int64_t)r * 3 + c) * V + s;
                cplx<double> z = acc[q][r][c];
                if (MODE == HAM_RESIDUAL) z = cols.b[6 * V * col[q] + at] - z;
                if (inside) y[at] = z;
                nrm += nrm2(z);
            }
        if (MODE != HAM_ADJOINT) {
            nrm = wsum(inside ? nrm : 0.0);
            if (threadIdx.x == 0) cols.partial[(int64_t)col[q] * (gridDim.x / ng) + sb] = nrm;
        }
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

struct ham_workspace {
    scratch_buf fld, blk, basis, vec, cpart, rpart, spart, gmz, gmd, gmi, nrm;
    // pinned, kept until the process ends: NSLOTS sums, then NSLOTS each of cycle
    // flags of even and odd steps, columns used, and (unused here) network falls
    double *sums = nullptr;
    int *flags = nullptr;
    hipEvent_t ev[2] = {nullptr, nullptr}; // end of even and odd Arnoldi steps
};
static ham_workspace g_ham;

struct ham_operator {
    const void *u;
    int precision;
    geom g;
    const double *fld;
    const cplx<double> *blk;
    unsigned nsb; // site blocks
};

template <int MODE> static void ham_apply(const ham_operator &op, const ham_cols &cols)
{
    const dim3 grd(op.nsb * (unsigned)((cols.n + HAM_NC - 1) / HAM_NC));
    if (op.precision == 64)
        hipLaunchKernelGGL((k_ham_apply<double, MODE>), grd, dim3(HAM_SITES), 0, stream(), (const cplx<double> *)op.u, op.fld, op.blk, op.g, cols);
    else
        hipLaunchKernelGGL((k_ham_apply<float, MODE>), grd, dim3(HAM_SITES), 0, stream(), (const cplx<float> *)op.u, op.fld, op.blk, op.g, cols);
}

// The squared norms of nc columns from the operator's partials, to g_ham.sums
// (columns without active[c] keep what is there), once the stream is done.
static int ham_norms(const ham_operator &op, int nc, const int *active)
{
    hipLaunchKernelGGL(k_fold_slots, dim3(nc), dim3(FOLD_THREADS), 0, stream(), (const double *)g_ham.spart.ptr,
                       (int64_t)op.nsb, active, (double *)g_ham.nrm.ptr, g_ham.sums);
    NRQ_HIP(hipGetLastError());
    NRQ_HIP(hipStreamSynchronize(stream()));
    return NRQ_OK;
}

// Right-hand sides b = S x, then GMRES(m) for S^+ x_c = b_c on nc columns
// (n = 6V complex each), zero initial guess, into x, stopping on
// ||b_c - S^+ x_c|| <= tol ||b_c||.  The columns run in lockstep, each through exactly
// the operations (and summation order) it would take alone.  The scalars of the
// iteration stay on the device (nrq_gmres.h); the host looks at the cycle flags of one
// step while the next is queued.  33x30x27, 12 columns: 1.07 ms a step where one
// synchronisation per iteration, separate norm and scaling passes and launches per
// column took 1.59 ms with the operator then used.  A column that reaches maxit leaves NRQ_ERR_NOCONV as the
// result; the others finish.
static int ham_solve(const ham_operator &op, int nc, const cplx<double> (*a)[4], cplx<double> *b, cplx<double> *res,
                     cplx<double> *const *x, int64_t n, int m, int64_t maxit, double tol, nrq_solve_stats *st)
{
    const gm_state gm = gm_layout(m, (cplx<double> *)g_ham.gmz.ptr, (double *)g_ham.gmd.ptr, (int *)g_ham.gmi.ptr);
    cplx<double> *basis = (cplx<double> *)g_ham.basis.ptr, *cpart = (cplx<double> *)g_ham.cpart.ptr;
    double *rpart = (double *)g_ham.rpart.ptr;
    const unsigned nb = vblocks(n);
    int *const used = g_ham.flags + 2 * NSLOTS, *const fallen = g_ham.flags + 3 * NSLOTS;
    ham_cols cols = {};
    cols.n = nc;
    cols.b = b;
    cols.partial = (double *)g_ham.spart.ptr;
    slots<double> xs = {};
    for (int c = 0; c < nc; ++c) {
        xs.p[c] = x[c];
        cols.in[c] = x[c];
        cols.out[c] = b + (int64_t)c * n;
        for (int t = 0; t < 4; ++t) cols.a[c][t] = a[c][t];
    }
    ham_apply<HAM_RHS>(op, cols);
    if (int e = ham_norms(op, nc, nullptr)) return e;
    double bnorm[HAM_MAXCOL], rnorm[HAM_MAXCOL];
    int64_t its[HAM_MAXCOL] = {};
    unsigned long long act = 0; // not yet converged (x = 0, as KSPSolve returns for b = 0)
    for (int c = 0; c < nc; ++c) {
        bnorm[c] = rnorm[c] = std::sqrt(g_ham.sums[c]);
        if (g_ham.sums[c] == 0.0) continue;
        ++st->solves;
        act |= 1ull << c;
    }
    if (!act) {
        for (int c = 0; c < nc; ++c) NRQ_HIP(hipMemsetAsync(x[c], 0, sizeof(cplx<double>) * (size_t)n, stream()));
        return NRQ_OK;
    }
    const cplx<double> *r0 = b; // residual the cycle starts from
    int failed = -1;
    for (bool first = true; act; first = false) {
        gm_start in = {};
        for (int c = 0; c < nc; ++c) {
            in.rn[c] = rnorm[c];
            in.stop[c] = 0.5 * tol * bnorm[c];
            in.left[c] = (int)std::min<int64_t>(m, std::max<int64_t>(1, maxit - its[c]));
            st->restarts += (int64_t)(act >> c & 1ull);
        }
        in.act = act;
        hipLaunchKernelGGL(k_gm_begin, dim3(1), dim3(64), 0, stream(), gm, in);
        const gm_basis<double> W = {r0, basis};
        for (int k = 0; k < m; ++k) {
            if (k >= 2) {
                NRQ_HIP(hipEventSynchronize(g_ham.ev[k & 1]));
                bool busy = false;
                for (int c = 0; c < nc; ++c) busy = busy || *(volatile int *)(g_ham.flags + (k & 1) * NSLOTS + c);
                if (!busy) break;
            }
            cplx<double> *w = basis + (int64_t)(k + 1) * nc * n;
            for (int c = 0; c < nc; ++c) {
                cols.in[c] = W.at(k, c, nc, n);
                cols.out[c] = w + (int64_t)c * n;
            }
            cols.active = gm.cyc;
            ham_apply<HAM_ADJOINT>(op, cols);
            const int nv = k + 1;
            hipLaunchKernelGGL(k_mdot<double>, dim3(nb, nc), dim3(VTHREADS), 0, stream(), W, nv, (const cplx<double> *)w, n, nc,
                               (const int *)gm.cyc, cpart);
            hipLaunchKernelGGL(k_gm_dots, dim3((nv * nc + 3) / 4), dim3(256), 0, stream(), cpart, (int)nb, nv, nc, gm);
            hipLaunchKernelGGL(k_cgs_update<double>, dim3(nb, nc), dim3(VTHREADS), 0, stream(), W, nv, w, n, nc, gm, rpart);
            hipLaunchKernelGGL(k_gm_step, dim3(nc), dim3(VTHREADS), 0, stream(), rpart, (int)nb, k, 0, gm,
                               g_ham.flags + (k & 1) * NSLOTS);
            NRQ_HIP(hipGetLastError());
            NRQ_HIP(hipEventRecord(g_ham.ev[k & 1], stream()));
        }
        hipLaunchKernelGGL(k_gm_solve, dim3(nc), dim3(64), 0, stream(), gm, 0, used, fallen);
        hipLaunchKernelGGL(k_xupdate<double>, dim3(nb, nc), dim3(VTHREADS), 0, stream(), xs, W, nc, n, gm, first ? 1 : 0);
        // the true residual r = b - S^+ x of every column that ran; the others' rows of
        // res are not read again
        for (int c = 0; c < nc; ++c) {
            cols.in[c] = x[c];
            cols.out[c] = res + (int64_t)c * n;
        }
        cols.active = gm.act;
        ham_apply<HAM_RESIDUAL>(op, cols);
        r0 = res;
        if (int e = ham_norms(op, nc, gm.act)) return e;
        for (int c = 0; c < nc; ++c) {
            if (!(act >> c & 1ull)) continue;
            rnorm[c] = std::sqrt(g_ham.sums[c]);
            its[c] += used[c];
            st->iterations += used[c];
            const bool conv = rnorm[c] <= tol * bnorm[c];
            // a residual that is not finite stays so
            if (!conv && its[c] < maxit && std::isfinite(rnorm[c])) continue;
            act &= ~(1ull << c);
            st->max_true_relres = worse(st->max_true_relres, rnorm[c] / bnorm[c]);
            if (!conv && failed < 0) failed = c;
        }
    }
    if (failed >= 0)
        return fail(NRQ_ERR_NOCONV, "CN (full Hamiltonian): no convergence after %lld iterations (relres %.3e)",
                    (long long)its[failed], rnorm[failed] / bnorm[failed]);
    return NRQ_OK;
}

int ham_cn_update(nrq_heavy *const *hs, const double *mass, int n, const nrq_gauge *gf, const double c[8],
                  double stepwidth, int restart, int64_t maxit, double tol, nrq_solve_stats *stats)
{
    const geom g = lat().g;
    const int64_t V = g.vol;
    const int64_t nvec = 6 * V;
    const int m = std::max(1, restart);
    // columns solved together: as many as fit HAM_BATCH_BYTES (NRQ_HAM_BATCH_BYTES
    // in the environment overrides it) of Krylov basis, residual and right-hand
    // side (m + 3 vectors each), at most HAM_MAXCOL
    size_t budget = HAM_BATCH_BYTES;
    if (const char *e = getenv("NRQ_HAM_BATCH_BYTES")) {
        const long long v = atoll(e);
        if (v > 0) budget = (size_t)v;
    }
    const size_t per_col = sizeof(cplx<double>) * (size_t)(m + 3) * (size_t)nvec;
    const int ncb = (int)std::max<size_t>(1, std::min<size_t>(HAM_MAXCOL, budget / per_col));
    if (int r = g_ham.fld.reserve(sizeof(double) * HAM_FLD * (size_t)V)) return r;
    if (int r = g_ham.blk.reserve(sizeof(cplx<double>) * 9 * HAM_BLK * (size_t)V)) return r;
    if (int r = g_ham.basis.reserve(sizeof(cplx<double>) * (size_t)(m + 1) * (size_t)nvec * ncb)) return r;
    if (int r = g_ham.vec.reserve(sizeof(cplx<double>) * 2 * (size_t)nvec * ncb)) return r;
    const int64_t nsb = (V + HAM_SITES - 1) / HAM_SITES;
    if (int r = g_ham.cpart.reserve(sizeof(cplx<double>) * (size_t)ncb * (size_t)m * VBLOCKS)) return r;
    if (int r = g_ham.rpart.reserve(sizeof(double) * (size_t)ncb * VBLOCKS)) return r;
    if (int r = g_ham.spart.reserve(sizeof(double) * (size_t)ncb * (size_t)nsb)) return r;
    if (int r = g_ham.gmz.reserve(sizeof(cplx<double>) * gm_zcount(m))) return r;
    if (int r = g_ham.gmd.reserve(sizeof(double) * gm_dcount(m))) return r;
    if (int r = g_ham.gmi.reserve(sizeof(int) * GM_ICOUNT)) return r;
    if (int r = g_ham.nrm.reserve(sizeof(double) * NSLOTS)) return r;
    if (!g_ham.sums && hipHostMalloc((void **)&g_ham.sums, sizeof(double) * NSLOTS, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        g_ham.sums = nullptr;
        return fail(NRQ_ERR_ALLOC, "CN (full Hamiltonian): pinned buffer allocation failed");
    }
    if (!g_ham.flags && hipHostMalloc((void **)&g_ham.flags, sizeof(int) * 4 * NSLOTS, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        g_ham.flags = nullptr;
        return fail(NRQ_ERR_ALLOC, "CN (full Hamiltonian): pinned buffer allocation failed");
    }
    for (hipEvent_t &e : g_ham.ev)
        if (!e) NRQ_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    ham_operator op;
    op.u = gauge_links(gf);
    op.precision = gf->precision;
    op.g = g;
    op.fld = (const double *)g_ham.fld.ptr;
    op.blk = (const cplx<double> *)g_ham.blk.ptr;
    op.nsb = (unsigned)nsb;
    const unsigned nbs = (unsigned)((V + HAM_THREADS - 1) / HAM_THREADS);
    if (gf->precision == 64) {
        hipLaunchKernelGGL(k_ham_fields<double>, dim3(op.nsb, 2), dim3(HAM_FIELD_THREADS), 0, stream(), (const cplx<double> *)op.u,
                           (const double *)gf->e, g, (double *)g_ham.fld.ptr);
        hipLaunchKernelGGL(k_ham_blocks<double>, dim3(nbs), dim3(HAM_THREADS), 0, stream(), (const cplx<double> *)op.u,
                           (const double *)g_ham.fld.ptr, g, (cplx<double> *)g_ham.blk.ptr);
    } else {
        hipLaunchKernelGGL(k_ham_fields<float>, dim3(op.nsb, 2), dim3(HAM_FIELD_THREADS), 0, stream(), (const cplx<float> *)op.u,
                           (const float *)gf->e, g, (double *)g_ham.fld.ptr);
        hipLaunchKernelGGL(k_ham_blocks<float>, dim3(nbs), dim3(HAM_THREADS), 0, stream(), (const cplx<float> *)op.u,
                           (const double *)g_ham.fld.ptr, g, (cplx<double> *)g_ham.blk.ptr);
    }
    NRQ_HIP(hipGetLastError());
    const double a0 = g.a[0];
    const std::complex<double> pre(0.0, -stepwidth / 2.0 * a0), I(0.0, 1.0);
    // right-hand sides after the ncb residual vectors
    cplx<double> *res = (cplx<double> *)g_ham.vec.ptr, *rhs = res + (int64_t)ncb * nvec;
    nrq_solve_stats st = {0, 0, 0, 0.0};
    int status = NRQ_OK;
    for (int hk = 0; hk < n; ++hk) {
        nrq_heavy *h = hs[hk];
        // the live columns of both propagators, solved ncb at a time
        std::vector<int> f0s;
        std::vector<std::array<cplx<double>, 4>> coefs;
        for (int prop = 0; prop < 2; ++prop) {
            const double M = prop == 0 ? mass[hk] : -mass[hk];
            std::complex<double> cc[4];
            for (int t = 0; t < 4; ++t) {
                cc[t] = std::complex<double>(c[2 * t], c[2 * t + 1]);
                if (prop == 1) cc[t] = std::conj(cc[t]);
            }
            const std::complex<double> at[4] = {pre * cc[0] / M, pre * (-cc[1]) / (2.0 * M),
                                                pre * (-cc[2]) / (8.0 * M * M), pre * (-cc[3]) * I / (8.0 * M * M)};
            std::array<cplx<double>, 4> a;
            for (int t = 0; t < 4; ++t) a[t] = {at[t].real(), at[t].imag()};
            for (int j = 0; j < 6; ++j) {
                const int f0 = 12 * prop + 2 * j;
                if (!((h->live >> f0) & 3u)) continue;
                f0s.push_back(f0);
                coefs.push_back(a);
            }
        }
        for (size_t c0 = 0; c0 < f0s.size(); c0 += (size_t)ncb) {
            const int nc = (int)std::min<size_t>((size_t)ncb, f0s.size() - c0);
            cplx<double> *xcol[HAM_MAXCOL];
            cplx<double> cof[HAM_MAXCOL][4];
            for (int c = 0; c < nc; ++c) {
                xcol[c] = (cplx<double> *)h->psi + (int64_t)f0s[c0 + c] * 3 * V;
                for (int t = 0; t < 4; ++t) cof[c][t] = coefs[c0 + c][t];
            }
            const int r = ham_solve(op, nc, cof, rhs, res, xcol, nvec, m, maxit, tol, &st);
            for (int c = 0; c < nc; ++c) h->live |= 3u << f0s[c0 + c]; // the spin-orbit term fills both spin rows
            if (r == NRQ_ERR_NOCONV) {
                status = r;
                continue;
            }
            if (r != NRQ_OK) return r;
        }
    }
    if (stats) *stats = st;
    return status;
}

} // namespace nrq
