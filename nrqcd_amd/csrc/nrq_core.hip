// nrq_core.hip -- error handling, the library stream, the lattice module and
// the host ranlxd generator.
#include "nrq_internal.h"
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>

namespace nrq {

static int g_last_code = 0;
static char g_last_msg[512] = "";

int fail(int code, const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_last_msg, sizeof(g_last_msg), fmt, ap);
    va_end(ap);
    g_last_code = code;
    return code;
}

int check_hip(hipError_t e, const char *what)
{
    return fail(NRQ_ERR_HIP, "HIP error %d (%s) in %s", (int)e, hipGetErrorString(e), what);
}

lattice_state &lat()
{
    static lattice_state s;
    return s;
}

static hipStream_t g_stream = nullptr;
static bool g_device_ok = false;

int ensure_device()
{
    if (g_device_ok) return NRQ_OK;
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n < 1)
        return fail(NRQ_ERR_HIP, "no HIP device available (hipGetDeviceCount: %s, count %d)",
                    hipGetErrorString(e), n);
    NRQ_HIP(hipStreamCreateWithFlags(&g_stream, hipStreamNonBlocking));
    g_device_ok = true;
    return NRQ_OK;
}

hipStream_t stream() { return g_stream; }

int scratch_buf::reserve(size_t n)
{
    if (n <= bytes) return NRQ_OK;
    if (ptr) (void)hipFree(ptr);
    ptr = nullptr;
    bytes = 0;
    hipError_t e = hipMalloc(&ptr, n);
    if (e != hipSuccess) {
        ptr = nullptr;
        return fail(NRQ_ERR_ALLOC, "hipMalloc(%zu) failed: %s", n, hipGetErrorString(e));
    }
    bytes = n;
    return NRQ_OK;
}

scratch_buf::~scratch_buf()
{
    // Process teardown: the runtime may already be gone; leak rather than
    // call into it.
}

// ---------------------------------------------------------------------------
// ranlxd (Luscher's RANLUX, double precision, 48-bit base; the algorithm of
// ranlxd_generator.f90:77-349).  Each refresh applies pr steps of the
// subtract-with-borrow recurrence x_n = x_{n-5} - x_{n-12} - carry in base
// b = 2^48 and hands out the last 12 numbers.  The numbers are held as their
// integer numerators; every step of the double-precision recurrence is exact.
//
// The pr steps are taken at once.  With x_0 ... x_11 the state in order of age,
// S = sum_n x_n b^n over the state and all that follows it is, b-adically, the
// fraction S = -Y / m (multiply the recurrence by b^n and sum):
//   m = b^12 - b^5 + 1,  Y = b^5 sum_{n<7} x_n b^n - sum_{n<12} x_n b^n + b^12 carry.
// Dropping the oldest digit, one step of the recurrence, multiplies Y by 1/b
// mod m: the equivalence of subtract-with-borrow with a linear congruential
// generator (S. Tezuka, P. L'Ecuyer, R. Couture, ACM TOMACS 3 (1993) 315;
// A. Sibidanov, Comput. Phys. Commun. 221 (2017) 299, uses it to skip).  So pr
// steps are one product with b^-pr mod m, the new digits are S mod b^12 =
// -Y / m = -Y (1 + b^5 + b^10) mod b^12, and the carry follows from Y.  A fresh
// seed's Y may be negative (its carry is not that of a running sequence); each
// step divides that excess by b, so it is gone within 12 < pr steps, and Y lies
// in (0, m), as the reduced product does.
// One 576-bit product per 12 numbers takes 15 ns a number on a Xeon core where the
// 397 dependent steps took 77, with the same bits; the thermal initial condition
// at 16^3 went from 35.5 to 31.4 ms.
// ---------------------------------------------------------------------------
namespace {
struct Ranlux48 {
    static constexpr int W = 9; // 576 bits = b^12 in 64-bit words, least significant first
    struct big {
        uint64_t w[W];
    };
    int64_t x[12];   // numerators of the state, x / 2^48 in [0, 1)
    int64_t carry = 0; // 0 or 1 (units of 2^-48)
    int ir = 0, ir_old = 0;
    int pr = 0;      // steps per refresh
    big skip;        // b^-pr mod m
    bool ready = false;

    // a + c and a - c mod 2^576; the carry / borrow is returned
    static int64_t add(big &a, const big &c)
    {
        unsigned __int128 t = 0;
        for (int k = 0; k < W; ++k) {
            t += (unsigned __int128)a.w[k] + c.w[k];
            a.w[k] = (uint64_t)t;
            t >>= 64;
        }
        return (int64_t)t;
    }
    static int64_t sub(big &a, const big &c)
    {
        uint64_t borrow = 0;
        for (int k = 0; k < W; ++k) {
            const unsigned __int128 t = (unsigned __int128)a.w[k] - c.w[k] - borrow;
            a.w[k] = (uint64_t)t;
            borrow = (uint64_t)(t >> 64) & 1;
        }
        return (int64_t)borrow;
    }
    // the n-word number v times b^5 = 2^240, mod 2^576
    static big times_b5(const uint64_t *v, int n)
    {
        big r;
        for (int k = 0; k < W; ++k) {
            const uint64_t hi = k >= 3 && k - 3 < n ? v[k - 3] : 0;
            const uint64_t lo = k >= 4 && k - 4 < n ? v[k - 4] : 0;
            r.w[k] = hi << 48 | lo >> 16;
        }
        return r;
    }
    static big b5m1() // b^5 - 1 = b^12 - m
    {
        constexpr uint64_t ones = ~uint64_t(0);
        return {{ones, ones, ones, ones >> 16}};
    }
    // a + top b^12 mod m, in [0, b^12)
    static void fold(big &a, int64_t top)
    {
        const big c = b5m1();
        for (; top > 0;) top += add(a, c) - 1;
        for (; top < 0;) top += 1 - sub(a, c);
    }
    // a c mod m, in [0, b^12)
    static big mul(const big &a, const big &c)
    {
        uint64_t p[2 * W] = {};
        for (int i = 0; i < W; ++i) {
            uint64_t over = 0;
            for (int j = 0; j < W; ++j) {
                const unsigned __int128 t = (unsigned __int128)a.w[i] * c.w[j] + p[i + j] + over;
                p[i + j] = (uint64_t)t;
                over = (uint64_t)(t >> 64);
            }
            p[i + W] = over;
        }
        // low half + h b^12 with h b^12 = h b^5 - h; what h b^5 has above b^12
        // is g = floor(h / b^7), and g b^12 = g b^5 - g
        big r, h, g = {};
        for (int k = 0; k < W; ++k) r.w[k] = p[k], h.w[k] = p[W + k];
        for (int k = 0; k < 4; ++k) g.w[k] = h.w[k + 5] >> 16 | (k < 3 ? h.w[k + 6] << 48 : 0);
        int64_t top = add(r, times_b5(h.w, W));
        top += add(r, times_b5(g.w, 4));
        top -= sub(r, h);
        top -= sub(r, g);
        fold(r, top);
        return r;
    }

    static void put_digit(big &a, int k, uint64_t v) // into zero bits
    {
        const int at = 48 * k / 64, sh = 48 * k % 64;
        a.w[at] |= v << sh;
        if (sh > 16) a.w[at + 1] |= v >> (64 - sh);
    }
    static uint64_t get_digit(const big &a, int k)
    {
        const int at = 48 * k / 64, sh = 48 * k % 64;
        uint64_t v = a.w[at] >> sh;
        if (sh > 16) v |= a.w[at + 1] << (64 - sh);
        return v & ((uint64_t(1) << 48) - 1);
    }

    int seed(int level, int64_t s)
    {
        if (level != 1 && level != 2) return -1;
        if (s <= 0 || s > 2147483647LL) return -2;
        pr = level == 1 ? 202 : 397;
        int bit[31];
        for (int k = 0; k < 31; ++k) bit[k] = (int)((s >> k) & 1);
        int a = 0, b = 18;
        for (int k = 0; k < 12; ++k) {
            int64_t acc = 0;
            for (int l = 0; l < 48; ++l) {
                acc = 2 * acc + (1 - bit[a]);
                bit[a] ^= bit[b];
                a = a == 30 ? 0 : a + 1;
                b = b == 30 ? 0 : b + 1;
            }
            x[k] = acc;
        }
        carry = 0;
        ir = 11;
        ir_old = 0;
        // 1/b = b^4 - b^11 mod m, to the power pr by squaring
        big q = {}, b11 = {};
        put_digit(q, 4, 1);
        put_digit(b11, 11, 1);
        fold(q, -sub(q, b11));
        skip = {{1}};
        for (int e = pr; e; e >>= 1) {
            if (e & 1) skip = mul(skip, q);
            q = mul(q, q);
        }
        ready = true;
        return 0;
    }

    void refresh()
    {
        big d = {}; // position ir holds the oldest number
        for (int k = 0; k < 12; ++k) put_digit(d, k, (uint64_t)x[ir + k < 12 ? ir + k : ir + k - 12]);
        big y = times_b5(d.w, W);
        fold(y, carry - sub(y, d));
        y = mul(y, skip);
        // into [0, m): a >= m = b^12 - (b^5 - 1) overflows b^12 with b^5 - 1 added
        big t = y;
        if (add(t, b5m1())) y = t;
        // d = -y (1 + b^5 + b^10) mod b^12
        t = times_b5(y.w, W);
        d = y;
        add(d, t);
        add(d, times_b5(t.w, W));
        big neg = {};
        sub(neg, d);
        // carry = (d - b^5 d + y) / b^12, d b^5 without what is above b^12
        t = neg;
        carry = -sub(t, times_b5(neg.w, W));
        carry += add(t, y);
        ir = (ir + pr) % 12;
        for (int k = 0; k < 12; ++k) x[ir + k < 12 ? ir + k : ir + k - 12] = (int64_t)get_digit(neg, k);
        ir_old = ir;
    }

    double next()
    {
        constexpr double UNIT = 1.0 / 281474976710656.0; // 2^-48, exact scaling
        ir = ir == 11 ? 0 : ir + 1;
        if (ir == ir_old) refresh();
        return (double)x[ir] * UNIT;
    }
};
Ranlux48 g_rng;
} // namespace

int rng_init(int level, int64_t s)
{
    int r = g_rng.seed(level, s);
    if (r == -1) return fail(NRQ_ERR_ARG, "ranlxd: luxury level must be 1 or 2");
    if (r == -2) return fail(NRQ_ERR_ARG, "ranlxd: seed must be in [1, 2^31-1]");
    return NRQ_OK;
}

void rng_uniform(double *r, int64_t n)
{
    if (!g_rng.ready) g_rng.seed(1, 1); // ranlxd_generator.f90:328-330
    for (int64_t k = 0; k < n; ++k) r[k] = g_rng.next();
}

bool rng_ready() { return g_rng.ready; }

} // namespace nrq

using namespace nrq;

extern "C" int nrq_last_error(char *buf, size_t n)
{
    if (buf && n) {
        strncpy(buf, g_last_msg, n - 1);
        buf[n - 1] = 0;
    }
    return g_last_code;
}

extern "C" const char *nrq_version(void) { return "nrqcd_amd 0.1 (gfx950)"; }

extern "C" int nrq_lattice_init(const int64_t ext[3], const double spacing[4])
{
    if (lat().initialised) return fail(NRQ_ERR_STATE, "lattice: already initialised");
    if (!ext || !spacing) return fail(NRQ_ERR_ARG, "lattice: null argument");
    for (int i = 0; i < 3; ++i)
        if (ext[i] < 1 || ext[i] > (1 << 20)) return fail(NRQ_ERR_ARG, "lattice: extent %d = %lld out of range", i + 1, (long long)ext[i]);
    for (int i = 0; i < 4; ++i)
        if (!(spacing[i] > 0) || !std::isfinite(spacing[i]))
            return fail(NRQ_ERR_ARG, "lattice: spacing a%d = %g must be positive", i, spacing[i]);
    // kernels index sites and grids with 32-bit arithmetic
    if (ext[0] * ext[1] * ext[2] > (int64_t)INT32_MAX / 32)
        return fail(NRQ_ERR_ARG, "lattice: volume %lld exceeds %d sites", (long long)(ext[0] * ext[1] * ext[2]),
                    INT32_MAX / 32);
    geom &g = lat().g;
    g.n0 = (int32_t)ext[0];
    g.n1 = (int32_t)ext[1];
    g.n2 = (int32_t)ext[2];
    g.vol = ext[0] * ext[1] * ext[2];
    for (int i = 0; i < 4; ++i) g.a[i] = spacing[i];
    lat().initialised = true;
    return NRQ_OK;
}

extern "C" int nrq_lattice_finalize(void)
{
    if (!lat().initialised) return fail(NRQ_ERR_STATE, "lattice: not initialised");
    gauge_forget_lattice();
    lat().initialised = false;
    return NRQ_OK;
}

#define NEED_LATTICE()                                                              \
    do {                                                                            \
        if (!lat().initialised) return fail(NRQ_ERR_STATE, "lattice: not initialised"); \
    } while (0)

static int check_idx(int64_t idx)
{
    if (idx < 1 || idx > lat().g.vol) return fail(NRQ_ERR_ARG, "lattice index %lld out of range", (long long)idx);
    return NRQ_OK;
}

extern "C" int nrq_lattice_size(int64_t *vol)
{
    NEED_LATTICE();
    if (!vol) return fail(NRQ_ERR_ARG, "null argument");
    *vol = lat().g.vol;
    return NRQ_OK;
}

extern "C" int nrq_lattice_index(const int64_t pos[3], int64_t *idx)
{
    NEED_LATTICE();
    const geom &g = lat().g;
    if (!pos || !idx) return fail(NRQ_ERR_ARG, "null argument");
    int64_t n[3] = {g.n0, g.n1, g.n2};
    for (int d = 0; d < 3; ++d)
        if (pos[d] < 1 || pos[d] > n[d]) return fail(NRQ_ERR_ARG, "position component %d out of range", d + 1);
    *idx = 1 + (pos[0] - 1) + n[0] * ((pos[1] - 1) + n[1] * (pos[2] - 1));
    return NRQ_OK;
}

static void position0(int64_t s, int64_t p[3])
{
    const geom &g = lat().g;
    p[0] = s % g.n0;
    p[1] = (s / g.n0) % g.n1;
    p[2] = s / ((int64_t)g.n0 * g.n1);
}

extern "C" int nrq_lattice_position(int64_t idx, int64_t pos[3])
{
    NEED_LATTICE();
    if (!pos) return fail(NRQ_ERR_ARG, "null argument");
    if (int r = check_idx(idx)) return r;
    int64_t p[3];
    position0(idx - 1, p);
    for (int d = 0; d < 3; ++d) pos[d] = p[d] + 1;
    return NRQ_OK;
}

extern "C" int nrq_lattice_neib(int dir, int64_t idx, int64_t *out)
{
    NEED_LATTICE();
    if (!out) return fail(NRQ_ERR_ARG, "null argument");
    if (dir < -3 || dir > 3) return fail(NRQ_ERR_ARG, "direction %d out of range", dir);
    if (int r = check_idx(idx)) return r;
    if (dir == 0) {
        *out = idx;
        return NRQ_OK;
    }
    const geom &g = lat().g;
    int64_t n[3] = {g.n0, g.n1, g.n2};
    int64_t p[3];
    position0(idx - 1, p);
    int d = (dir > 0 ? dir : -dir) - 1;
    p[d] = (p[d] + (dir > 0 ? 1 : n[d] - 1)) % n[d];
    *out = 1 + p[0] + n[0] * (p[1] + n[1] * p[2]);
    return NRQ_OK;
}

extern "C" int nrq_lattice_negative_index(int64_t idx, int64_t *out)
{
    NEED_LATTICE();
    if (!out) return fail(NRQ_ERR_ARG, "null argument");
    if (int r = check_idx(idx)) return r;
    const geom &g = lat().g;
    int64_t n[3] = {g.n0, g.n1, g.n2};
    int64_t p[3];
    position0(idx - 1, p);
    for (int d = 0; d < 3; ++d) p[d] = (n[d] - p[d]) % n[d];
    *out = 1 + p[0] + n[0] * (p[1] + n[1] * p[2]);
    return NRQ_OK;
}

extern "C" int nrq_lattice_momentum(int64_t idx, double pm[6])
{
    NEED_LATTICE();
    if (!pm) return fail(NRQ_ERR_ARG, "null argument");
    if (int r = check_idx(idx)) return r;
    const geom &g = lat().g;
    int64_t n[3] = {g.n0, g.n1, g.n2};
    int64_t p[3];
    position0(idx - 1, p);
    for (int d = 0; d < 3; ++d) {
        double arg = M_PI * (double)p[d] / (double)n[d];
        double mag = 2.0 * std::sin(arg) / g.a[d + 1];
        pm[2 * d] = mag * std::cos(arg);
        pm[2 * d + 1] = -mag * std::sin(arg);
    }
    return NRQ_OK;
}

extern "C" int nrq_lattice_norm2_momentum(int64_t idx, double *out)
{
    double pm[6];
    if (int r = nrq_lattice_momentum(idx, pm)) return r;
    double s = 0;
    for (int k = 0; k < 6; ++k) s += pm[k] * pm[k];
    *out = std::sqrt(s);
    return NRQ_OK;
}

extern "C" int nrq_random_init(int64_t seed) { return rng_init(2, seed); }

extern "C" int nrq_random_uniform(double *r, int64_t n)
{
    if (!r || n < 0) return fail(NRQ_ERR_ARG, "null argument or negative count");
    rng_uniform(r, n);
    return NRQ_OK;
}

// ---------------------------------------------------------------------------
// HIP events on the library stream, for timing from the host layer.
// ---------------------------------------------------------------------------
static hipEvent_t g_events[16];
static bool g_event_made[16];

extern "C" int nrq_event_record(int slot)
{
    if (slot < 0 || slot >= 16) return fail(NRQ_ERR_ARG, "event slot %d out of range", slot);
    if (int r = ensure_device()) return r;
    if (!g_event_made[slot]) {
        NRQ_HIP(hipEventCreate(&g_events[slot]));
        g_event_made[slot] = true;
    }
    NRQ_HIP(hipEventRecord(g_events[slot], stream()));
    return NRQ_OK;
}

extern "C" int nrq_event_elapsed(int start, int stop, double *ms)
{
    if (start < 0 || start >= 16 || stop < 0 || stop >= 16 || !ms) return fail(NRQ_ERR_ARG, "bad event slots");
    if (!g_event_made[start] || !g_event_made[stop]) return fail(NRQ_ERR_STATE, "event slot never recorded");
    NRQ_HIP(hipEventSynchronize(g_events[stop]));
    float t = 0;
    NRQ_HIP(hipEventElapsedTime(&t, g_events[start], g_events[stop]));
    *ms = t;
    return NRQ_OK;
}

extern "C" int nrq_synchronize(void)
{
    if (int r = ensure_device()) return r;
    NRQ_HIP(hipStreamSynchronize(stream()));
    return NRQ_OK;
}

// ---------------------------------------------------------------------------
// Streaming copy probe: the achievable HBM bandwidth of a plain read+write
// kernel on this device, and a known-size reference for hardware counters.
// ---------------------------------------------------------------------------
typedef double v2d __attribute__((ext_vector_type(2)));

__global__ __launch_bounds__(256) void k_stream_copy(const v2d *__restrict__ src, v2d *__restrict__ dst, int64_t n)
{
    // each thread keeps four 16-byte loads in flight
    const int64_t base = (int64_t)blockIdx.x * 1024 + threadIdx.x;
    v2d v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (base + 256 * k < n) v[k] = __builtin_nontemporal_load(src + base + 256 * k);
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (base + 256 * k < n) __builtin_nontemporal_store(v[k], dst + base + 256 * k);
}

extern "C" int nrq_bandwidth_probe(int64_t bytes, int reps, double *gbs)
{
    if (bytes < 4096 || reps < 1 || !gbs) return fail(NRQ_ERR_ARG, "bandwidth probe: bad arguments");
    if (int r = ensure_device()) return r;
    const int64_t n = bytes / (int64_t)sizeof(double2);
    double2 *a = nullptr, *b = nullptr;
    if (hipMalloc(&a, n * sizeof(double2)) != hipSuccess || hipMalloc(&b, n * sizeof(double2)) != hipSuccess) {
        if (a) (void)hipFree(a);
        return fail(NRQ_ERR_ALLOC, "bandwidth probe: allocation of %lld bytes failed", (long long)bytes);
    }
    NRQ_HIP(hipMemsetAsync(a, 0, n * sizeof(double2), stream()));
    hipEvent_t e0, e1;
    NRQ_HIP(hipEventCreate(&e0));
    NRQ_HIP(hipEventCreate(&e1));
    const unsigned blocks = (unsigned)((n + 1023) / 1024);
    hipLaunchKernelGGL(k_stream_copy, dim3(blocks), dim3(256), 0, stream(), (const v2d *)a, (v2d *)b, n); // warm-up
    NRQ_HIP(hipEventRecord(e0, stream()));
    for (int r = 0; r < reps; ++r)
        hipLaunchKernelGGL(k_stream_copy, dim3(blocks), dim3(256), 0, stream(), (const v2d *)a, (v2d *)b, n);
    NRQ_HIP(hipEventRecord(e1, stream()));
    NRQ_HIP(hipEventSynchronize(e1));
    float ms = 0;
    NRQ_HIP(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipFree(a);
    (void)hipFree(b);
    *gbs = 2.0 * (double)(n * sizeof(double2)) * reps / (ms * 1e-3) / 1e9;
    return NRQ_OK;
}
