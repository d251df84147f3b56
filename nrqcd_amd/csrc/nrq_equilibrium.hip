// nrq_equilibrium.hip -- EquilibriumInit (gaugeconfiguration_su3.f90:380-814)
// on the GPU: thermal electric fields projected onto the Gauss law, then
// leapfrog equilibration, repeated nefieldinit times from cold links.
//
// Per outer iteration:
//   E^a_k(x) = Re(sigma r^a) a0, sigma = sqrt(4/beta), r: 8 complex normals
//     per site and direction from 16 uniforms of the host ranlxd stream in
//     lattice order (:455-466);
//   G(x) = [sum_i (E_i(x) - U_i(x-i)^+ E_i(x-i) U_i(x-i)) / a_i
//           - sum_a T^a Tr(T^a diag(rho(x)) / (a1 a2 a3))] / a0   (GetG, :781-813),
//   deviation = max_{x,a} 2 |Tr(T^a G(x))|                  (GetGdeviation, :724-779);
//   while deviation > tol, from the previous configuration (Jacobi sweep):
//     E_k(x) <- coordinates of kappa a0 (U_k(x) G(x) U_k(x)^+ G(x+k) - G(x)) + E_k(x),
//     kappa = 0.01 (:480-507; the product of G(x) and G(x+k) is the
//     reference's, taken literally);
//   nequilibrium leapfrog steps of step width 1 (:696-698).
// The default tolerance is the reference's single-precision literal 1E-3.
//
// One launch is one sweep (k_eq_sweep): it forms the new E from the old G and
// E, the new G from the new E, and the maximum of the deviation.  G(x) needs
// E_i(x - i) as well, which the thread of that site and direction also forms
// from G(x - i), G(x), U_i(x - i) and the old E_i(x - i), so nothing of the
// sweep has to pass through memory first; E and G alternate between two
// buffers.  A sweep is a serial chain of a few microseconds on a small lattice
// and one pass over U, E and G on a large one (960 B per site in FP64, against
// 1,872 B with separate project, Gauss and fold kernels).  Measured per sweep,
// FP64 storage: 6.5 us at 16^3 (three kernels of 6.9, 6.7 and 2.7 us with their
// gaps before), 69 us at 64^3 (54, 40 and 5 us); FP32 at 64^3 50 us (74 us).
//
// Sweeps run in batches without host synchronisation.  The maximum of the
// state before sweep j lies in row j of a table (nrq_maxrow.h); a sweep that finds its row at or below the tolerance writes nothing, and so
// leaves the next row at zero, which is below the tolerance too: exactly the
// reference's number of sweeps changes E.
#include "nrq_internal.h"
#include "nrq_maxrow.h"
#include <algorithm>
#include <cmath>
#include <vector>

namespace nrq {

const void *gauge_links(const nrq_gauge *h);

constexpr double EQ_KAPPA = 0.01;
constexpr int64_t EQ_MAX_PROJECTIONS = 1000000; // guard: the reference loops without bound

template <typename R> __device__ __forceinline__ mat3<double> eq_link(const cplx<R> *u, int64_t vol, int dir, int64_t s)
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

template <typename R> __device__ __forceinline__ mat3<double> eq_efield(const R *ef, int64_t vol, int dir, int64_t s)
{
    double al[8];
#pragma unroll
    for (int a = 0; a < 8; ++a) al[a] = (double)*at32(ef + ((int64_t)dir * 8 + a) * vol, (uint32_t)s);
    return algebra_matrix(al);
}

// G is Hermitian: its diagonal (planes 0, 1, 2) and upper triangle (re, im of
// 01, 02, 12 in planes 3..8), nine doubles per site.
__device__ __forceinline__ mat3<double> eq_herm(const double (&h)[9])
{
    mat3<double> m;
    m.m[0] = {h[0], 0.0};
    m.m[4] = {h[1], 0.0};
    m.m[8] = {h[2], 0.0};
    m.m[1] = {h[3], h[4]};
    m.m[2] = {h[5], h[6]};
    m.m[5] = {h[7], h[8]};
    m.m[3] = conjg(m.m[1]);
    m.m[6] = conjg(m.m[2]);
    m.m[7] = conjg(m.m[5]);
    return m;
}

__device__ __forceinline__ mat3<double> eq_load_g(const double *__restrict__ gm, int64_t vol, int64_t s)
{
    double h[9];
#pragma unroll
    for (int e = 0; e < 9; ++e) h[e] = *at32(gm + (int64_t)e * vol, (uint32_t)s);
    return eq_herm(h);
}

// The Hermitian product A B^+ (A = U H or U^+ H, B = U or U^+): diagonal real
// parts and upper triangle only.
__device__ __forceinline__ mat3<double> eq_herm_nd(const mat3<double> &a, const mat3<double> &b)
{
    double h[9];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        double d = 0.0;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            d = fmx(a.m[3 * r + k].re, b.m[3 * r + k].re, d);
            d = fmx(a.m[3 * r + k].im, b.m[3 * r + k].im, d);
        }
        h[r] = d;
    }
    const int pr[3] = {0, 0, 1}, pc[3] = {1, 2, 2};
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        cplx<double> t = {0.0, 0.0};
#pragma unroll
        for (int k = 0; k < 3; ++k) mac_nc(t, a.m[3 * pr[q] + k], b.m[3 * pc[q] + k]);
        h[3 + 2 * q] = t.re;
        h[4 + 2 * q] = t.im;
    }
    return eq_herm(h);
}

__device__ __forceinline__ mat3<double> eq_dagger(const mat3<double> &a)
{
    mat3<double> d;
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) d.m[3 * r + c] = conjg(a.m[3 * c + r]);
    return d;
}

// Coordinates of kdt (U G U^+ Gn - G) + E as stored (rounded to R): the
// projected E of one (site, direction).
template <typename R>
__device__ __forceinline__ void eq_projected(const mat3<double> &u, const mat3<double> &g, const mat3<double> &gn,
                                             const mat3<double> &e, double kdt, double (&out)[8])
{
    const mat3<double> a = mul(eq_herm_nd(mul(u, g), u), gn);
    mat3<double> t;
#pragma unroll
    for (int k = 0; k < 9; ++k)
        t.m[k] = {fmx(kdt, a.m[k].re - g.m[k].re, e.m[k].re), fmx(kdt, a.m[k].im - g.m[k].im, e.m[k].im)};
    two_re_trace_gen(t, out);
#pragma unroll
    for (int k = 0; k < 8; ++k) out[k] = (double)(R)out[k];
}

constexpr int EQ_SITES = 64; // sites per block, one per lane

// One projection sweep (PROJ), or G and the deviation of the E field as it is
// (PROJ = false: ef is read, ef_new and the old G are not used).  A block is
// EQ_SITES sites times six wavefronts: wave i (0..2) forms E_i(x) and its part
// E_i(x) / a_i of G(x); wave 3 + i forms E_i(x - i) and the part
// -U_i(x-i)^+ E_i(x-i) U_i(x-i) / a_i.  The parts meet in LDS and the first
// wave adds them.  Six short chains per site instead of one long one: at 16^3
// the whole sweep is one wavefront's latency.
template <typename R, bool PROJ>
__global__ __launch_bounds__(6 * EQ_SITES) void k_eq_sweep(const cplx<R> *__restrict__ u, const R *__restrict__ ef,
                                                         const double *__restrict__ gm, const double *__restrict__ rho,
                                                         geom g, double kdt, R *__restrict__ ef_new,
                                                         double *__restrict__ gm_new, double tol,
                                                         const double *__restrict__ row, double *__restrict__ row_new)
{
    __shared__ double part[6][9][EQ_SITES];
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int i = w < 3 ? w : w - 3;
    const int64_t V = g.vol;
    const int64_t s = (int64_t)blockIdx.x * EQ_SITES + lane;
    const bool in = s < V;
    if (PROJ) {
        // the deviation before this sweep, the same for every wave of the
        // grid: the sweeps past the last leave here (2.2 us each at 16^3, 9 us
        // at 64^3; a look just before the stores, to hide its latency, saved
        // nothing measurable on a full sweep and cost these 5 and 69 us)
        if (row_max(row) <= tol) return;
    }
    double e[8];
    lsite p = {0, 0, 0, 0};
    mat3<double> h;
    if (in) {
        p = make_site(g, s);
        const int64_t m = w < 3 ? s : site_dn(g, p, i).s; // the site whose E this thread forms
        const mat3<double> U = eq_link(u, V, i, m);
        const mat3<double> E = eq_efield(ef, V, i, m);
        if (PROJ) {
            const int64_t n = w < 3 ? site_up(g, p, i).s : s; // m + i
            eq_projected<R>(U, eq_load_g(gm, V, m), eq_load_g(gm, V, n), E, kdt, e);
            h = algebra_matrix(e);
        } else {
            h = E;
        }
        double sc = 1.0 / g.a[i + 1];
        if (w >= 3) {
            const mat3<double> ud = eq_dagger(U);
            h = eq_herm_nd(mul(ud, h), ud);
            sc = -sc;
        }
        const double v[9] = {h.m[0].re, h.m[4].re, h.m[8].re, h.m[1].re, h.m[1].im, h.m[2].re, h.m[2].im, h.m[5].re, h.m[5].im};
#pragma unroll
        for (int k = 0; k < 9; ++k) part[w][k][lane] = sc * v[k];
    }
    if (PROJ && in && w < 3) {
#pragma unroll
        for (int a = 0; a < 8; ++a) *at32(ef_new + ((int64_t)i * 8 + a) * V, (uint32_t)s) = (R)e[a];
    }
    __syncthreads();
    if (w != 0) return;
    double dev = 0.0;
    if (in) {
        double q[9];
#pragma unroll
        for (int k = 0; k < 9; ++k)
            q[k] = ((part[0][k][lane] + part[3][k][lane]) + (part[1][k][lane] + part[4][k][lane])) +
                   (part[2][k][lane] + part[5][k][lane]);
        if (rho) {
            // sum_a T^a Tr(T^a C), C = diag(rho) / (a1 a2 a3): Tr(T^a C) is
            // non-zero for the two diagonal generators only
            const double vcell = g.a[1] * g.a[2] * g.a[3];
            double c[8] = {0, 0, 0, 0, 0, 0, 0, 0};
            const double r0 = rho[3 * s] / vcell, r1 = rho[3 * s + 1] / vcell, r2 = rho[3 * s + 2] / vcell;
            c[2] = 0.5 * (r0 - r1);
            c[7] = 0.28867513459481288225457439025098 * (r0 + r1 - 2.0 * r2);
            const mat3<double> t = algebra_matrix(c);
            q[0] -= t.m[0].re;
            q[1] -= t.m[4].re;
            q[2] -= t.m[8].re;
        }
        const double ia0 = 1.0 / g.a[0];
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            q[k] *= ia0;
            *at32(gm_new + (int64_t)k * V, (uint32_t)s) = q[k];
        }
        double tr[8];
        two_re_trace_gen(eq_herm(q), tr);
        // What is not a number must not pass for a small deviation (a maximum drops it):
        // infinite where the E field as it is is looked at, at both ends of a projection.
        // The sweeps do without (it is part of their latency, 1 % of a thermal start at 16^3).
#pragma unroll
        for (int a = 0; a < 8; ++a) {
            const double t = fabs(tr[a]);
            dev = PROJ || t < INFINITY ? fmax(dev, t) : INFINITY;
        }
    }
    dev = lane_max(dev);
    if (lane == 0) row_raise(row_new, dev);
}

// Zeroes rows [first, first + n) of the deviation table (n blocks).
__global__ __launch_bounds__(MAXROW) void k_eq_clear(double *__restrict__ table, int first, int rows)
{
    table[(int64_t)((first + (int)blockIdx.x) % rows) * MAXROW + threadIdx.x] = 0.0;
}

// out[b] = maximum of row first + b
__global__ __launch_bounds__(MAXROW) void k_eq_rows(const double *__restrict__ table, int first, int rows,
                                                     double *__restrict__ out)
{
    const double v = row_max(table + (int64_t)((first + (int)blockIdx.x) % rows) * MAXROW);
    if (threadIdx.x == 0) out[blockIdx.x] = v;
}

// Sweeps launched per batch.  After the first batch the host looks at a batch
// while the next one runs, so it never waits with an empty queue.
constexpr int EQ_BATCH = 64;
constexpr int EQ_ROWS = 4 * EQ_BATCH; // ring of deviation rows: two batches in flight

template <typename R>
static int equilibrium_t(nrq_gauge *h, double beta, int64_t nefieldinit, int64_t nequilibrium, double tol,
                         const double *rho_host, double *energies, double *deviations, int64_t *projections)
{
    const geom g = lat().g;
    const int64_t V = g.vol;
    const unsigned nb = (unsigned)((V + EQ_SITES - 1) / EQ_SITES);
    struct bufs {
        double *gm[2] = {nullptr, nullptr};
        double *table = nullptr, *dev = nullptr, *rho = nullptr, *hdev = nullptr;
        void *ealt = nullptr;
        hipEvent_t ev[2] = {nullptr, nullptr};
        ~bufs()
        {
            for (int k = 0; k < 2; ++k) {
                if (gm[k]) (void)hipFree(gm[k]);
                if (ev[k]) (void)hipEventDestroy(ev[k]);
            }
            if (table) (void)hipFree(table);
            if (dev) (void)hipFree(dev);
            if (rho) (void)hipFree(rho);
            if (ealt) (void)hipFree(ealt);
            if (hdev) (void)hipHostFree(hdev);
        }
    } b;
    const size_t ebytes = sizeof(R) * 24 * (size_t)V;
    if (hipMalloc((void **)&b.gm[0], sizeof(double) * 9 * (size_t)V) != hipSuccess ||
        hipMalloc((void **)&b.gm[1], sizeof(double) * 9 * (size_t)V) != hipSuccess ||
        hipMalloc((void **)&b.table, sizeof(double) * EQ_ROWS * MAXROW) != hipSuccess ||
        hipMalloc((void **)&b.dev, sizeof(double) * 2 * EQ_BATCH) != hipSuccess || hipMalloc(&b.ealt, ebytes) != hipSuccess ||
        (rho_host && hipMalloc((void **)&b.rho, sizeof(double) * 3 * (size_t)V) != hipSuccess) ||
        hipHostMalloc((void **)&b.hdev, sizeof(double) * 2 * EQ_BATCH, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        return fail(NRQ_ERR_ALLOC, "EquilibriumInit: device allocation failed (V=%lld)", (long long)V);
    }
    for (int k = 0; k < 2; ++k) NRQ_HIP(hipEventCreateWithFlags(&b.ev[k], hipEventDisableTiming));
    if (rho_host) NRQ_HIP(hipMemcpyAsync(b.rho, rho_host, sizeof(double) * 3 * (size_t)V, hipMemcpyHostToDevice, stream()));
    if (int r = nrq_gauge_cold(h)) return r;
    R *ebuf[2] = {(R *)h->e, (R *)b.ealt};
    auto row = [&](int64_t j) { return b.table + (j % EQ_ROWS) * MAXROW; };
    // G (buffer 0) and deviation of the configuration in h->e (row 0); the
    // links are looked up at every use, since the leapfrog swaps their buffers
    auto start = [&](double *dev) -> int {
        hipLaunchKernelGGL(k_eq_clear, dim3(1), dim3(MAXROW), 0, stream(), b.table, 0, EQ_ROWS);
        hipLaunchKernelGGL((k_eq_sweep<R, false>), dim3(nb), dim3(6 * EQ_SITES), 0, stream(), (const cplx<R> *)gauge_links(h),
                           (const R *)h->e, (const double *)nullptr, b.rho, g, 0.0, (R *)nullptr, b.gm[0], tol,
                           (const double *)nullptr, row(0));
        hipLaunchKernelGGL(k_eq_rows, dim3(1), dim3(MAXROW), 0, stream(), b.table, 0, EQ_ROWS, b.dev);
        NRQ_HIP(hipGetLastError());
        NRQ_HIP(hipMemcpyAsync(b.hdev, b.dev, sizeof(double), hipMemcpyDeviceToHost, stream()));
        NRQ_HIP(hipStreamSynchronize(stream()));
        *dev = b.hdev[0];
        return NRQ_OK;
    };
    const double sigma = std::sqrt(4.0 / beta);
    const double a0 = g.a[0];
    const double twopi = 2.0 * M_PI;
    std::vector<R> ehost((size_t)24 * (size_t)V);
    for (int64_t it = 0; it < nefieldinit; ++it) {
        // thermal E: per site (lattice order) and direction, 8 complex
        // normals from 16 uniforms, real parts (random.f90:238-253)
        double uu[16];
        for (int64_t s = 0; s < V; ++s)
            for (int k = 0; k < 3; ++k) {
                rng_uniform(uu, 16);
                for (int a = 0; a < 8; ++a) {
                    const double re = std::sqrt(-2.0 * std::log(uu[2 * a])) * std::cos(twopi * uu[2 * a + 1]);
                    ehost[((size_t)k * 8 + a) * (size_t)V + (size_t)s] = (R)((sigma * re) * a0);
                }
            }
        NRQ_HIP(hipMemcpyAsync(h->e, ehost.data(), ebytes, hipMemcpyHostToDevice, stream()));
        double dev = 0;
        if (int r = start(&dev)) return r;
        auto not_finite = [&]() { return fail(NRQ_ERR_NOCONV, "EquilibriumInit: the Gauss-law deviation is not finite"); };
        if (!std::isfinite(dev)) return not_finite();
        const cplx<R> *u = (const cplx<R> *)gauge_links(h); // fixed during the projection
        // batch k: sweeps k EQ_BATCH .. and the deviations after them (rows
        // + 1 ..) to the pinned half k & 1; sweep j reads E and G buffer j & 1
        int64_t launched = 0;
        auto issue = [&]() -> int {
            const int64_t first = launched;
            const int half = (int)(first / EQ_BATCH & 1);
            hipLaunchKernelGGL(k_eq_clear, dim3(EQ_BATCH), dim3(MAXROW), 0, stream(), b.table,
                               (int)((first + 1) % EQ_ROWS), EQ_ROWS);
            for (; launched < first + EQ_BATCH; ++launched) {
                const int64_t j = launched;
                hipLaunchKernelGGL((k_eq_sweep<R, true>), dim3(nb), dim3(6 * EQ_SITES), 0, stream(), u,
                                   (const R *)ebuf[j & 1], (const double *)b.gm[j & 1], b.rho, g, EQ_KAPPA * a0,
                                   ebuf[(j + 1) & 1], b.gm[(j + 1) & 1], tol, (const double *)row(j), row(j + 1));
            }
            hipLaunchKernelGGL(k_eq_rows, dim3(EQ_BATCH), dim3(MAXROW), 0, stream(), b.table,
                               (int)((first + 1) % EQ_ROWS), EQ_ROWS, b.dev + half * EQ_BATCH);
            NRQ_HIP(hipGetLastError());
            NRQ_HIP(hipMemcpyAsync(b.hdev + half * EQ_BATCH, b.dev + half * EQ_BATCH, sizeof(double) * EQ_BATCH,
                                   hipMemcpyDeviceToHost, stream()));
            NRQ_HIP(hipEventRecord(b.ev[half], stream()));
            return NRQ_OK;
        };
        int64_t nproj = 0; // sweeps that changed E
        bool done = dev <= tol;
        if (!done)
            if (int r = issue()) return r;
        for (int64_t k = 0; !done; ++k) {
            const bool last = launched >= EQ_MAX_PROJECTIONS;
            if (!last && k > 0)
                if (int r = issue()) return r;
            NRQ_HIP(hipEventSynchronize(b.ev[k & 1]));
            const double *d = b.hdev + (k & 1) * EQ_BATCH;
            for (int q = 0; q < EQ_BATCH && !done; ++q) {
                ++nproj;
                dev = d[q];
                done = dev <= tol;
                if (!std::isfinite(dev)) return not_finite();
            }
            if (!done && !last && k == 0)
                if (int r = issue()) return r;
            if (!done && last && nproj >= launched)
                return fail(NRQ_ERR_NOCONV, "EquilibriumInit: Gauss-law projection above %g after %lld sweeps (deviation %g)",
                            tol, (long long)EQ_MAX_PROJECTIONS, dev);
        }
        if (nproj & 1) // the final E is in the second buffer
            NRQ_HIP(hipMemcpyAsync(h->e, b.ealt, ebytes, hipMemcpyDeviceToDevice, stream()));
        if (nequilibrium > 0)
            if (int r = nrq_gauge_leapfrog(h, 1.0, nequilibrium)) return r;
        if (energies)
            if (int r = nrq_gauge_energy(h, &energies[it])) return r;
        // the look at the state that the caller gets (which also ends with an idle stream)
        if (int r = start(&dev)) return r;
        if (!std::isfinite(dev)) return not_finite();
        if (deviations) deviations[it] = dev;
        if (projections) projections[it] = nproj;
    }
    return NRQ_OK;
}

} // namespace nrq

using namespace nrq;

extern "C" int nrq_gauge_equilibrium_init(nrq_gauge *h, double beta, int64_t nefieldinit, int64_t nequilibrium,
                                          double tolerance, const double *charge_density, double *energies,
                                          double *deviations, int64_t *projections)
{
    if (!lat().initialised) return fail(NRQ_ERR_STATE, "lattice: not initialised");
    if (!h || !h->u[0]) return fail(NRQ_ERR_ARG, "gauge: null or unallocated handle");
    if (h->vol != lat().g.vol) return fail(NRQ_ERR_STATE, "gauge: lattice changed since allocation");
    if (!(beta > 0) || !std::isfinite(beta)) return fail(NRQ_ERR_ARG, "EquilibriumInit: beta must be positive");
    if (nefieldinit < 0 || nequilibrium < 0) return fail(NRQ_ERR_ARG, "EquilibriumInit: negative iteration count");
    if (!rng_ready()) return fail(NRQ_ERR_STATE, "EquilibriumInit: random module not initialised");
    if (!(tolerance > 0)) tolerance = (double)1e-3f; // the reference's default, a single-precision literal
    if (int r = ensure_device()) return r;
    return h->precision == 64
               ? equilibrium_t<double>(h, beta, nefieldinit, nequilibrium, tolerance, charge_density, energies,
                                       deviations, projections)
               : equilibrium_t<float>(h, beta, nefieldinit, nequilibrium, tolerance, charge_density, energies,
                                      deviations, projections);
}
