// nrq_gaugefix.hip -- Coulomb gauge fixing and the transverse AA/EE
// correlators behind the gluon occupation f(p) = sqrt(AA EE)
// (gaugeconfiguration_su3.f90:1825-1972, 2269-2521; main.f90:3093-3189).
//
// Gauge fixing is Davies' Fourier-accelerated steepest descent.  Per
// iteration:
//   Delta(x) = sum_i skew(U_i(x - i) - U_i(x)),  skew(d) = (d - d^+)/2
// (not made traceless, as in the reference); stop when
// max_x ||Delta(x)||_F / 9 <= tol.  Otherwise Delta goes to momentum space,
// every mode with |p| > 1e-12 is multiplied by (p_max/|p|)^2, Delta comes back,
// is multiplied by alpha, and g(x) = exp(Delta(x)) transforms the links,
// U_i(x) <- g(x) U_i(x) g(x + i)^+.  E is not transformed (the reference's
// PerformGaugeTransformation touches only the links).  Delta is skew-Hermitian,
// nine real numbers per site, and the momentum-space multiplier is real and
// even in p, so it acts on each of them alone: the Hermitian -i Delta travels
// as GF_PLANES = 5 complex planes ((d0, d1), (d2, 0), q01, q02, q12) through
// one batched in-place hipFFT Z2Z pair instead of nine complex components (a
// measurement of 100 iterations with both correlators at 64^3: 21.5 -> 18.2 ms).
// The reference's x2p/p2x scales (a1 a2 a3 forward, 1 / physical volume
// backward, xpfft.f90:134-136), the acceleration and alpha are one multiply in
// momentum space.
//
// The correlators take the 24 fields A^a_i(x) = GetGroupLog(U_i(x))^a / a_i
// (or E^a_i(x) / (a_i a0)) to momentum space in one batched transform, two real
// fields of one direction per complex plane (12 planes; with 24 planes the
// electric correlator at 128^3 took 1.2 ms longer), and contract them per
// momentum with the transverse projector
// P_ij = Re[(delta_ij - conj(p_i) p_j / |p|^2) / 2] of the backward-derivative
// momentum (the reference's projector is a real function, lattice.f90:
// 1178-1195, so only the real part of the complex expression survives),
// divided by the physical volume and averaged over the generators.
//
// Group log: H = -i log U on the principal branch (eigenphases atan2(Im, Re)
// in (-pi, pi], su3.f90:318-334 via matrixoperations.f90:474-495), from the
// eigen-decomposition in nrq_grouplog.h.
#include "nrq_internal.h"
#include "nrq_grouplog.h"
#include "nrq_map.h"
#include "nrq_maxrow.h"
#include <hipfft/hipfft.h>
#include <algorithm>
#include <cmath>
#include <vector>

namespace nrq {

const void *gauge_links(const nrq_gauge *h);
void *gauge_links_mut(nrq_gauge *h);

constexpr double GF_ZERO_TOL = 1e-12; // tolerances.f90
constexpr int GF_THREADS = 256;
constexpr double GF_AHEAD = 1.5; // the next iteration is enqueued ahead above this many tolerances
constexpr int GF_PLANES = 5;    // complex planes of -i Delta
constexpr int CORR_PLANES = 12; // complex planes of 24 real fields: pair q of direction i in plane q + 4 i

template <typename R> __device__ __forceinline__ mat3<double> load_link_d(const cplx<R> *u, int64_t vol, int dir, int64_t s)
{
    mat3<double> m;
    const cplx<R> *p = u + (int64_t)dir * 9 * vol;
#pragma unroll
    for (int e = 0; e < 9; ++e) {
        const cplx<R> a = *at32(p + (int64_t)e * vol, (uint32_t)s);
        m.m[e] = {(double)a.re, (double)a.im};
    }
    return m;
}

// Backward-derivative lattice momentum of momentum index s (lattice.f90:963-979)
// and its squared norm.
__device__ __forceinline__ double lattice_momentum(const geom &g, int64_t s, cplx<double> (&p)[3])
{
    const lsite q = make_site(g, s);
    const int n[3] = {q.x, q.y, q.z};
    const int ext[3] = {g.n0, g.n1, g.n2};
    double pn2 = 0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const double arg = M_PI * (double)n[d] / (double)ext[d];
        double sn, cs;
        sincos(arg, &sn, &cs);
        const double mag = 2.0 * sn / g.a[d + 1];
        p[d] = {mag * cs, -mag * sn};
        pn2 += p[d].re * p[d].re + p[d].im * p[d].im;
    }
    return pn2;
}

// ---------------------------------------------------------------------------
// gauge fixing
// ---------------------------------------------------------------------------

// -i Delta(x) into GF_PLANES complex planes; the maximum of ||Delta||_F / 9
// raises `row`.  Bound by its link reads; each XCD walks one contiguous eighth
// of the lattice, so that U_i(x - i) is found in its L2 (with k_gf_apply in the
// same order, 100 iterations at 64^3: 17.3 -> 15.8 ms).
template <typename R>
__global__ __launch_bounds__(GF_THREADS) void k_gf_divergence(const cplx<R> *__restrict__ u, geom g,
                                                             cplx<double> *__restrict__ div, double *__restrict__ row)
{
    __shared__ double sh[GF_THREADS / 64];
    const int64_t s = (int64_t)xcd_block(gridDim.x, 8) * blockDim.x + threadIdx.x;
    double dev = 0;
    if (s < g.vol) {
        const lsite p = make_site(g, s);
        mat3<double> d;
        set_zero(d);
        for (int i = 0; i < 3; ++i) {
            const mat3<double> a = load_link_d(u, g.vol, i, site_dn(g, p, i).s);
            const mat3<double> b = load_link_d(u, g.vol, i, s);
            // skew(a - b) = ((a - b) - (a - b)^+) / 2, added entry by entry
#pragma unroll
            for (int r = 0; r < 3; ++r)
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const cplx<double> x = a.m[3 * r + c] - b.m[3 * r + c];
                    const cplx<double> y = a.m[3 * c + r] - b.m[3 * c + r];
                    d.m[3 * r + c] = d.m[3 * r + c] + cplx<double>{0.5 * (x.re - y.re), 0.5 * (x.im + y.im)};
                }
        }
        // -i d for the diagonal (its real part is exactly zero) and the upper triangle
        const cplx<double> q[GF_PLANES] = {{d.m[0].im, d.m[4].im},
                                           {d.m[8].im, 0.0},
                                           {d.m[1].im, -d.m[1].re},
                                           {d.m[2].im, -d.m[2].re},
                                           {d.m[5].im, -d.m[5].re}};
#pragma unroll
        for (int e = 0; e < GF_PLANES; ++e) div[(int64_t)e * g.vol + s] = q[e];
        double f = 0;
#pragma unroll
        for (int e = 0; e < 9; ++e) f += d.m[e].re * d.m[e].re + d.m[e].im * d.m[e].im;
        dev = sqrt(f) / 9.0;
    }
    dev = lane_max(dev);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = dev;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = 0;
        for (int k = 0; k < GF_THREADS / 64; ++k) m = fmax(m, sh[k]);
        row_raise(row, m);
    }
}

// The maximum of `row` to *out (pinned host memory); `next` starts at zero.
__global__ __launch_bounds__(MAXROW) void k_gf_fold_max(const double *__restrict__ row, double *__restrict__ next,
                                                       double *__restrict__ out)
{
    const double m = row_max(row);
    next[threadIdx.x] = 0.0;
    if (threadIdx.x == 0) *out = m;
}

// Whether the transformation of the iteration whose divergence maximum is in
// `row` is made: not once it is at or below the tolerance (or infinite, which
// the host reports).
__device__ __forceinline__ bool gf_goes_on(const double *__restrict__ row, double tol)
{
    const double m = row_max(row);
    return m > tol && m < INFINITY;
}

// Momentum-space step: scale = fwd * bwd * alpha, times (p_max/|p|)^2 where |p| > tol.
__global__ void k_gf_accelerate(cplx<double> *__restrict__ div, geom g, double pmax, double scale)
{
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.vol) return;
    cplx<double> p[3];
    const double pn = sqrt(lattice_momentum(g, s, p));
    double f = scale;
    if (pn > GF_ZERO_TOL) {
        const double r = pmax / pn;
        f *= r * r;
    }
#pragma unroll
    for (int e = 0; e < GF_PLANES; ++e) div[(int64_t)e * g.vol + s] = f * div[(int64_t)e * g.vol + s];
}

// g = exp(Delta) at site s: exp(iQ) with Q = -i Delta, its trace split off as
// a phase (the traceless part goes through the Cayley-Hamilton exponential).
__device__ __forceinline__ mat3<double> gf_group(const cplx<double> *__restrict__ div, int64_t vol, int64_t s)
{
    cplx<double> w[GF_PLANES];
#pragma unroll
    for (int e = 0; e < GF_PLANES; ++e) w[e] = div[(int64_t)e * vol + s];
    mat3<double> q;
    q.m[0] = {w[0].re, 0.0};
    q.m[4] = {w[0].im, 0.0};
    q.m[8] = {w[1].re, 0.0};
    q.m[1] = w[2];
    q.m[2] = w[3];
    q.m[5] = w[4];
    q.m[3] = conjg(w[2]);
    q.m[6] = conjg(w[3]);
    q.m[7] = conjg(w[4]);
    const double t = (q.m[0].re + q.m[4].re + q.m[8].re) / 3.0;
    q.m[0].re -= t;
    q.m[4].re -= t;
    q.m[8].re -= t;
    mat3<double> x = exp_i_hermitian(q);
    double sn, cs;
    sincos(t, &sn, &cs);
    const cplx<double> ph = {cs, sn};
#pragma unroll
    for (int e = 0; e < 9; ++e) x.m[e] = ph * x.m[e];
    return x;
}

// U_i(x) <- g(x) U_i(x) g(x + i)^+ for the three directions at x, with
// g = exp(Delta) formed here from Delta (gf_group) for x and its three
// forward neighbours, so no separate pass writes g: the exponentials are
// FP64 arithmetic inside a memory-bound kernel (46 us at 64^3 for 226 MB of
// links).  Blocks in the order of k_gf_divergence.
template <typename R>
__global__ __launch_bounds__(GF_THREADS) void k_gf_apply(cplx<R> *__restrict__ u, const cplx<double> *__restrict__ delta,
                                                         geom g, const double *__restrict__ row, double tol)
{
    if (!gf_goes_on(row, tol)) return;
    const int64_t s = (int64_t)xcd_block(gridDim.x, 8) * blockDim.x + threadIdx.x;
    if (s >= g.vol) return;
    const lsite p = make_site(g, s);
    const mat3<double> gx = gf_group(delta, g.vol, s);
    for (int i = 0; i < 3; ++i) {
        const int64_t sp = site_up(g, p, i).s;
        const mat3<double> gy = gf_group(delta, g.vol, sp);
        const mat3<double> v = mul_nd(mul(gx, load_link_d(u, g.vol, i, s)), gy);
        cplx<R> *b = u + (int64_t)i * 9 * g.vol;
#pragma unroll
        for (int e = 0; e < 9; ++e) *at32(b + (int64_t)e * g.vol, (uint32_t)s) = {(R)v.m[e].re, (R)v.m[e].im};
    }
}

// ---------------------------------------------------------------------------
// group log and correlators
// ---------------------------------------------------------------------------

// The 24 real fields, two per complex plane (components 2q, 2q + 1 of
// direction i = blockIdx.y in plane q + 4 i): A^a_i = GetGroupLog(U_i)^a / a_i,
// one thread per (site, direction).
template <typename R>
__global__ __launch_bounds__(GF_THREADS) void k_aa_fields(const cplx<R> *__restrict__ u, geom g, cplx<double> *__restrict__ fld)
{
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int i = blockIdx.y;
    if (s >= g.vol) return;
    double c[8];
    group_log_coords(load_link_d(u, g.vol, i, s), c);
#pragma unroll
    for (int q = 0; q < 4; ++q) fld[(int64_t)(q + 4 * i) * g.vol + s] = {c[2 * q] / g.a[i + 1], c[2 * q + 1] / g.a[i + 1]};
}

// The same of E^a_i / (a_i a0): a copy, one thread per site and plane
// (blockIdx.y).  One thread for all 24 values of a site, with the logarithm's
// registers, ran at a quarter of the bandwidth (128^3 FP32 479 us).
template <typename R>
__global__ __launch_bounds__(GF_THREADS) void k_ee_fields(const R *__restrict__ ef, geom g, cplx<double> *__restrict__ fld)
{
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int pl = blockIdx.y, i = pl >> 2, q = pl & 3; // plane q + 4 i
    if (s >= g.vol) return;
    const R *e = ef + ((int64_t)i * 8 + 2 * q) * g.vol;
    const double c0 = (double)*at32(e, (uint32_t)s), c1 = (double)*at32(e + g.vol, (uint32_t)s);
    fld[(int64_t)pl * g.vol + s] = {c0 / g.a[i + 1] / g.a[0], c1 / g.a[i + 1] / g.a[0]};
}

// out[s] = Re sum_a sum_ij F^a_i P_ij conj(F^a_j) * scale, scale = fwd^2 / (8 V_phys),
// P_ij = (delta_ij - Re(conj(p_i) p_j) / |p|^2) / 2
__global__ void k_corr_project(const cplx<double> *__restrict__ fld, geom g, double scale, double *__restrict__ out)
{
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.vol) return;
    cplx<double> p[3];
    const double pn2 = lattice_momentum(g, s, p);
    if (!(sqrt(pn2) >= GF_ZERO_TOL)) {
        out[s] = 0.0;
        return;
    }
    double rp[3][3];
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) rp[i][j] = (p[i].re * p[j].re + p[i].im * p[j].im) / pn2; // Re(conj(p_i) p_j) / |p|^2
    double acc = 0;
    for (int a = 0; a < 8; ++a) {
        cplx<double> f[3];
        for (int i = 0; i < 3; ++i) f[i] = fld[(int64_t)(a + 8 * i) * g.vol + s];
        double t = 0;
        for (int i = 0; i < 3; ++i)
            for (int j = 0; j < 3; ++j) {
                const double gij = f[i].re * f[j].re + f[i].im * f[j].im; // Re(f_i conj(f_j))
                t += ((i == j ? 1.0 : 0.0) - rp[i][j]) * gij;
            }
        acc += 0.5 * t;
    }
    out[s] = acc * scale;
}

// The same for the packed transforms of real fields.  With Z = F^a + i F^b
// per direction, F^a = (Z(p) + conj Z(-p)) / 2 and F^b likewise, so
//   sum_{a,b} Re[F_i conj(F_j)](p) = (Re[Z_i conj Z_j](p) + Re[Z_i conj Z_j](-p)) / 2
// without separating the two fields; P is even in p.  One thread per pair
// {p, -p} (the smaller in (z, y, x) order works, whole blocks of the rest
// leave at once) reads both momenta and writes both outputs, so every plane is
// read once: half the bytes of 24 unpacked planes.
__global__ __launch_bounds__(GF_THREADS) void k_corr_project_packed(const cplx<double> *__restrict__ fld, geom g,
                                                                   double scale, double *__restrict__ out)
{
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.vol) return;
    const lsite q = make_site(g, s);
    const int64_t sn = (q.x ? g.n0 - q.x : 0) + (int64_t)g.n0 * ((q.y ? g.n1 - q.y : 0) + (int64_t)g.n1 * (q.z ? g.n2 - q.z : 0));
    if (sn < s) return; // x fastest: the order of site indices is that of (z, y, x)
    cplx<double> p[3];
    const double pn2 = lattice_momentum(g, s, p);
    if (!(sqrt(pn2) >= GF_ZERO_TOL)) {
        out[s] = out[sn] = 0.0;
        return;
    }
    double gij[6] = {0, 0, 0, 0, 0, 0}; // (0,0) (1,1) (2,2) (0,1) (0,2) (1,2)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int64_t at = e == 0 ? s : sn;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            cplx<double> z[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) z[i] = fld[(int64_t)(k + 4 * i) * g.vol + at];
#pragma unroll
            for (int i = 0; i < 3; ++i) gij[i] += z[i].re * z[i].re + z[i].im * z[i].im;
            gij[3] += z[0].re * z[1].re + z[0].im * z[1].im;
            gij[4] += z[0].re * z[2].re + z[0].im * z[2].im;
            gij[5] += z[1].re * z[2].re + z[1].im * z[2].im;
        }
    }
    double acc = 0;
#pragma unroll
    for (int i = 0; i < 3; ++i) acc += (1.0 - (p[i].re * p[i].re + p[i].im * p[i].im) / pn2) * gij[i];
    acc -= 2.0 * ((p[0].re * p[1].re + p[0].im * p[1].im) * gij[3] + (p[0].re * p[2].re + p[0].im * p[2].im) * gij[4] +
                  (p[1].re * p[2].re + p[1].im * p[2].im) * gij[5]) / pn2;
    const double v = 0.25 * acc * scale;
    out[s] = v;
    out[sn] = v;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

static int gf_fft_fail(hipfftResult r, const char *what)
{
    return fail(NRQ_ERR_HIP, "hipFFT %s failed (%d)", what, (int)r);
}

// Largest |p| of the backward-derivative momenta: |p|^2 is a sum of one term
// per direction, so its maximum is the sum of the per-direction maxima.
static double max_momentum(const geom &g)
{
    const int ext[3] = {g.n0, g.n1, g.n2};
    double sum = 0;
    for (int d = 0; d < 3; ++d) {
        double m = 0;
        for (int n = 0; n < ext[d]; ++n) {
            const double arg = M_PI * (double)n / (double)ext[d];
            const double mag = 2.0 * std::sin(arg) / g.a[d + 1];
            const double re = mag * std::cos(arg), im = -mag * std::sin(arg);
            m = std::max(m, re * re + im * im);
        }
        sum += m;
    }
    return std::sqrt(sum);
}

// Events of one call, released on every exit path.
struct gf_events {
    hipEvent_t ev[2] = {nullptr, nullptr};
    ~gf_events()
    {
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
    }
};

// Batched in-place Z2Z plans, kept per (extents, batch) for the life of the
// process: plan creation costs milliseconds, a measurement repeated along a
// run should not pay it every time.
struct gf_plan_entry {
    int n0, n1, n2, batch;
    hipfftHandle plan;
};
static std::vector<gf_plan_entry> g_gf_plans;

static int gf_plan(const geom &g, int batch, hipfftHandle *out)
{
    for (const gf_plan_entry &e : g_gf_plans)
        if (e.n0 == g.n0 && e.n1 == g.n1 && e.n2 == g.n2 && e.batch == batch) {
            *out = e.plan;
            return hipfftSetStream(e.plan, stream()) == HIPFFT_SUCCESS ? NRQ_OK : fail(NRQ_ERR_HIP, "hipFFT set stream failed");
        }
    int dims[3] = {g.n2, g.n1, g.n0}; // row-major, x fastest
    hipfftHandle plan = 0;
    hipfftResult fr = hipfftPlanMany(&plan, 3, dims, nullptr, 1, (int)g.vol, nullptr, 1, (int)g.vol, HIPFFT_Z2Z, batch);
    if (fr != HIPFFT_SUCCESS) return gf_fft_fail(fr, "plan");
    fr = hipfftSetStream(plan, stream());
    if (fr != HIPFFT_SUCCESS) {
        hipfftDestroy(plan);
        return gf_fft_fail(fr, "set stream");
    }
    g_gf_plans.push_back({g.n0, g.n1, g.n2, batch, plan});
    *out = plan;
    return NRQ_OK;
}

template <typename R>
static int gaugefix_t(nrq_gauge *h, double tol, double alpha, int64_t maxit, int64_t *iterations, double *final_dev)
{
    const geom g = lat().g;
    const int64_t v = g.vol;
    const unsigned nblk = (unsigned)((v + GF_THREADS - 1) / GF_THREADS);
    // -i Delta (80 B per site) in the link buffer that the next leapfrog pass
    // overwrites, the maxima in the handle's reduction buffers: no allocation
    cplx<double> *fld = (cplx<double> *)h->u[h->cur ^ 1];
    double *rows = (double *)h->partials, *hmax = h->result;
    gf_events b;
    for (hipEvent_t &e : b.ev) NRQ_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    hipfftHandle plan = 0;
    if (int e = gf_plan(g, GF_PLANES, &plan)) return e;
    cplx<R> *u = (cplx<R> *)gauge_links_mut(h);
    const double fwd = g.a[1] * g.a[2] * g.a[3];
    const double bwd = 1.0 / ((double)g.n0 * g.a[1] * (double)g.n1 * g.a[2] * (double)g.n2 * g.a[3]);
    const double pmax = max_momentum(g);
    // row n % 3 holds the divergence maximum before transformation n; the fold
    // of row n clears that of n + 1, last read by transformation n - 2
    auto row = [&](int64_t n) { return rows + (n % 3) * MAXROW; };
    NRQ_HIP(hipMemsetAsync(rows, 0, sizeof(double) * 3 * MAXROW, stream()));
    auto measure = [&](int64_t n) -> int {
        hipLaunchKernelGGL(k_gf_divergence<R>, dim3(nblk), dim3(GF_THREADS), 0, stream(), u, g, fld, row(n));
        hipLaunchKernelGGL(k_gf_fold_max, dim3(1), dim3(MAXROW), 0, stream(), row(n), row(n + 1), hmax + (n & 1));
        NRQ_HIP(hipGetLastError());
        NRQ_HIP(hipEventRecord(b.ev[n & 1], stream()));
        return NRQ_OK;
    };
    // transformation n, made by k_gf_apply if the maximum before it asks for it, and
    // the maximum after it
    auto transform = [&](int64_t n) -> int {
        hipfftResult fr = hipfftExecZ2Z(plan, (hipfftDoubleComplex *)fld, (hipfftDoubleComplex *)fld, HIPFFT_FORWARD);
        if (fr != HIPFFT_SUCCESS) return gf_fft_fail(fr, "exec (forward)");
        hipLaunchKernelGGL(k_gf_accelerate, dim3(nblk), dim3(GF_THREADS), 0, stream(), fld, g, pmax, fwd * bwd * alpha);
        fr = hipfftExecZ2Z(plan, (hipfftDoubleComplex *)fld, (hipfftDoubleComplex *)fld, HIPFFT_BACKWARD);
        if (fr != HIPFFT_SUCCESS) return gf_fft_fail(fr, "exec (backward)");
        hipLaunchKernelGGL(k_gf_apply<R>, dim3(nblk), dim3(GF_THREADS), 0, stream(), u, fld, g, row(n), tol);
        // n + 1 uses the event and host slot of n - 1, which the host has read
        return measure(n + 1);
    };
    if (int e = measure(0)) return e;
    int64_t enqueued = 0, done = 0;
    double dev = 0;
    for (;; ++done) {
        // Where the last maximum was far above the tolerance the next transformation is
        // enqueued before the host looks at this one's, so the GPU does not wait for the host.
        // Near the tolerance, and before the first look, the host looks first (10 us): a
        // transformation that is then not made costs more (64^3 130 us, 96^3 440 us).
        if (enqueued == done && done < maxit && dev > GF_AHEAD * tol) {
            if (int e = transform(enqueued++)) return e;
        }
        NRQ_HIP(hipEventSynchronize(b.ev[done & 1]));
        dev = *(volatile double *)(hmax + (done & 1));
        if (!std::isfinite(dev) || dev <= tol || done >= maxit) break;
        if (enqueued == done)
            if (int e = transform(enqueued++)) return e;
    }
    // host values go back with an idle stream: a transformation that was enqueued too many ends here
    NRQ_HIP(hipStreamSynchronize(stream()));
    if (!std::isfinite(dev)) return fail(NRQ_ERR_NOCONV, "gauge fixing: non-finite divergence");
    if (iterations) *iterations = done;
    if (final_dev) *final_dev = dev;
    return NRQ_OK;
}

int transverse_project(const cplx<double> *fld, double scale, double *out)
{
    const geom g = lat().g;
    const int64_t v = g.vol;
    double *dout = nullptr;
    if (hipMalloc((void **)&dout, sizeof(double) * (size_t)v) != hipSuccess) {
        (void)hipGetLastError();
        return fail(NRQ_ERR_ALLOC, "correlators: device allocation failed (V=%lld)", (long long)v);
    }
    const unsigned nblk = (unsigned)((v + GF_THREADS - 1) / GF_THREADS);
    hipLaunchKernelGGL(k_corr_project, dim3(nblk), dim3(GF_THREADS), 0, stream(), fld, g, scale, dout);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(out, dout, sizeof(double) * (size_t)v, hipMemcpyDeviceToHost, stream());
    if (e == hipSuccess) e = hipStreamSynchronize(stream());
    (void)hipFree(dout);
    return e == hipSuccess ? NRQ_OK : check_hip(e, "transverse projection");
}

template <typename R> static int correlators_t(const nrq_gauge *h, double *aa, double *ee)
{
    const geom g = lat().g;
    const int64_t v = g.vol;
    const unsigned nblk = (unsigned)((v + GF_THREADS - 1) / GF_THREADS);
    // the planes and the result (200 B per site) in the link buffer that the
    // next leapfrog pass overwrites (216 B per site in FP32): no allocation
    static_assert(CORR_PLANES * sizeof(cplx<double>) + sizeof(double) <= 27 * sizeof(cplx<R>) || sizeof(R) == 8, "scratch");
    cplx<double> *fld = (cplx<double> *)h->u[h->cur ^ 1];
    double *dout = (double *)(fld + (int64_t)CORR_PLANES * v);
    hipfftHandle plan = 0;
    if (int e = gf_plan(g, CORR_PLANES, &plan)) return e;
    const double fwd = g.a[1] * g.a[2] * g.a[3];
    const double vphys = (double)g.n0 * g.a[1] * (double)g.n1 * g.a[2] * (double)g.n2 * g.a[3];
    const double scale = fwd * fwd / vphys / 8.0;
    const cplx<R> *u = (const cplx<R> *)gauge_links(h);
    const R *ef = (const R *)h->e;
    for (int which = 0; which < 2; ++which) {
        double *host = which == 0 ? aa : ee;
        if (!host) continue;
        if (which == 0)
            hipLaunchKernelGGL(k_aa_fields<R>, dim3(nblk, 3), dim3(GF_THREADS), 0, stream(), u, g, fld);
        else
            hipLaunchKernelGGL(k_ee_fields<R>, dim3(nblk, CORR_PLANES), dim3(GF_THREADS), 0, stream(), ef, g, fld);
        NRQ_HIP(hipGetLastError());
        hipfftResult fr = hipfftExecZ2Z(plan, (hipfftDoubleComplex *)fld, (hipfftDoubleComplex *)fld, HIPFFT_FORWARD);
        if (fr != HIPFFT_SUCCESS) return gf_fft_fail(fr, "exec (forward)");
        hipLaunchKernelGGL(k_corr_project_packed, dim3(nblk), dim3(GF_THREADS), 0, stream(), fld, g, scale, dout);
        NRQ_HIP(hipGetLastError());
        NRQ_HIP(hipMemcpyAsync(host, dout, sizeof(double) * (size_t)v, hipMemcpyDeviceToHost, stream()));
        NRQ_HIP(hipStreamSynchronize(stream()));
    }
    return NRQ_OK;
}

} // namespace nrq

using namespace nrq;

extern "C" int nrq_gauge_coulomb_gaugefix(nrq_gauge *h, double tol, double alpha, int64_t max_iterations,
                                          int64_t *iterations, double *final_deviation)
{
    if (!lat().initialised) return fail(NRQ_ERR_STATE, "lattice: not initialised");
    if (!h) return fail(NRQ_ERR_ARG, "null gauge configuration");
    if (h->vol != lat().g.vol) return fail(NRQ_ERR_STATE, "gauge configuration does not match the lattice");
    if (!(tol >= 0) || !std::isfinite(alpha) || max_iterations < 0)
        return fail(NRQ_ERR_ARG, "gauge fixing: tolerance %g, alpha %g, max iterations %lld", tol, alpha,
                    (long long)max_iterations);
    if (int r = ensure_device()) return r;
    return h->precision == 64 ? gaugefix_t<double>(h, tol, alpha, max_iterations, iterations, final_deviation)
                              : gaugefix_t<float>(h, tol, alpha, max_iterations, iterations, final_deviation);
}

extern "C" int nrq_gauge_transverse_correlators(const nrq_gauge *h, double *aa, double *ee)
{
    if (!lat().initialised) return fail(NRQ_ERR_STATE, "lattice: not initialised");
    if (!h) return fail(NRQ_ERR_ARG, "null gauge configuration");
    if (h->vol != lat().g.vol) return fail(NRQ_ERR_STATE, "gauge configuration does not match the lattice");
    if (int r = ensure_device()) return r;
    return h->precision == 64 ? correlators_t<double>(h, aa, ee) : correlators_t<float>(h, aa, ee);
}

extern "C" int nrq_lattice_max_norm2_momentum(double *out)
{
    if (!lat().initialised) return fail(NRQ_ERR_STATE, "lattice: not initialised");
    if (!out) return fail(NRQ_ERR_ARG, "null argument");
    *out = max_momentum(lat().g);
    return NRQ_OK;
}
