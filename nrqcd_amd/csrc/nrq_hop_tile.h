// nrq_hop_tile.h -- the covariant hop of the CN stencils for whole lattices, the
// fields staged in LDS.
//
// hop(s) = sum_i (U_i(s) f(s+i) + U_i(s-i)^+ f(s-i)) / a_i^2 reads every field
// value seven times and every link once per field.  Read through the caches,
// what sets the time is the number of cache lines a CU asks for (about 190 a
// microsecond on MI355X, whether L2 or HBM serves them; the copy kernel's rate),
// not the bytes from HBM.  Here a block owns a 16 x 4 tile of (x, y) and a run of
// z planes, and each of its 12 wavefronts one colour field: a lane is a site.
// Per plane a wavefront loads the tile's own values of the next plane (3 loads)
// and its one-site halo (2 loads) and keeps the plane in its own part of LDS;
// the z neighbours are the lane's registers (the next plane's values, and
// U_z(s-z)^+ f(s-z) carried over from the plane before).  The links of a plane
// are loaded once per block, two planes in LDS by turns, so that one barrier per
// plane suffices, and are shared by the 12 fields.
//
// Measured at 128^3 with 12 fields (before: wave items of nrq_map.h): FP64
// residual 860 us (1237), right-hand side 1155 us (1538), FP32 Chebyshev step
// 598 to 860 us (889), FP32 operator 530 us (645); the traffic is within 15% of
// the algorithmic bytes.  A third of the lines are the x halo's (one line per
// row and side).  Tried without gain: six fields per block, or two blocks of
// 12 FP32 fields per CU (slower: link lines, spills), values of the plane after
// next in flight, a third fewer instructions (FP32 row 3 rebuilt once per link
// instead of once per field; kept, 2-4% on 48 fields).
//
// Sites beyond an extent that is not a multiple of the tile are filled with
// their periodic images, so the neighbours of the last row and column are found
// like any others; such lanes store nothing.  Any extents work; hop_tiles_pay
// says where it is faster.
#pragma once
#include "nrq_map.h"
#include <cmath>

namespace nrq {

constexpr int HT_X = 16, HT_Y = 4;       // tile, one site per lane
constexpr int HT_HX = HT_X + 2;          // with halo
constexpr int HT_CELLS = HT_HX * (HT_Y + 2);
constexpr int HT_HALO = 2 * HT_Y + 2 * HT_X; // halo cells of a plane (no corners)
constexpr int HT_F = 12;                    // fields (wavefronts) per block
constexpr int HT_THREADS = 64 * HT_F;
constexpr int NSLOT_GROUPS = 4; // groups of HT_F slots in a batch
constexpr int HT_CUS = 256; // one block per CU: LDS and the registers of its 12 wavefronts
// links of a plane that the tile needs: U_x from x - 1, U_y from y - 1, U_z
constexpr int HT_LX = (HT_X + 1) * HT_Y, HT_LY = HT_X * (HT_Y + 1), HT_LZ = HT_X * HT_Y;
constexpr int HT_L = HT_LX + HT_LY + HT_LZ;

struct hop_tiles {
    int ntx, nty; // tiles
    int zc, nzr;  // planes per run, runs
    int groups;   // groups of HT_F slots
};

// Block-uniform position of a block and its partial-sum index.
struct hop_block {
    int bx, by, z0, nz, group;
    unsigned index; // tile and run: 0 .. ntx nty nzr - 1
};

__device__ __forceinline__ hop_block hop_block_of(const hop_tiles &t, const geom &g)
{
    // groups fastest (they share the links), then tiles, then runs; each XCD
    // walks one contiguous range, so that halos are found in its L2
    const unsigned lb = xcd_block(gridDim.x, 8);
    hop_block b;
    b.index = lb / (unsigned)t.groups;
    b.group = (int)(lb - b.index * (unsigned)t.groups);
    const unsigned tiles = (unsigned)(t.ntx * t.nty);
    const unsigned zr = b.index / tiles, tile = b.index - zr * tiles;
    b.by = (int)(tile / (unsigned)t.ntx);
    b.bx = (int)(tile - (unsigned)b.by * (unsigned)t.ntx);
    b.z0 = (int)zr * t.zc;
    b.nz = g.n2 - b.z0 < t.zc ? g.n2 - b.z0 : t.zc;
    return b;
}

// One element as one vector load or store (a copy of the struct goes through
// memory where its address is only known to be a multiple of 8).
template <typename R> __device__ __forceinline__ cplx<R> get(const cplx<R> *p)
{
    const typename vec2_of<R>::type v = *(const typename vec2_of<R>::type *)p;
    return {v.x, v.y};
}
template <typename R> __device__ __forceinline__ void put(cplx<R> *p, cplx<R> a)
{
    typename vec2_of<R>::type v;
    v.x = a.re;
    v.y = a.im;
    *(typename vec2_of<R>::type *)p = v;
}

// The value is formed here, not sunk to its use further down: without it the
// compiler reads all links and neighbours of a plane first and spills them.
template <typename T> __device__ __forceinline__ void pin(cplx<T> (&v)[3])
{
#pragma unroll
    for (int c = 0; c < 3; ++c) asm volatile("" : "+v"(v[c].re), "+v"(v[c].im));
}

// Whole link from its NE stored elements (6: row 3 rebuilt) in the type T.
template <int NE, typename RL, typename T> __device__ __forceinline__ mat3<T> hop_link(const cplx<RL> (&l)[NE])
{
    mat3<T> w;
#pragma unroll
    for (int e = 0; e < NE; ++e) w.m[e] = {(T)l[e].re, (T)l[e].im};
    if (NE == 6) su3_row3(w);
    return w;
}

template <typename T> __device__ __forceinline__ void clear(cplx<T> (&t)[3])
{
#pragma unroll
    for (int c = 0; c < 3; ++c) t[c] = {T(0), T(0)};
}

// t += U f and t += U^+ f
template <typename T> __device__ __forceinline__ void hop_fwd(const mat3<T> &w, const cplx<T> (&f)[3], cplx<T> (&t)[3])
{
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        mac(t[c], w.m[3 * c], f[0]);
        mac(t[c], w.m[3 * c + 1], f[1]);
        mac(t[c], w.m[3 * c + 2], f[2]);
    }
}
template <typename T> __device__ __forceinline__ void hop_bwd(const mat3<T> &w, const cplx<T> (&f)[3], cplx<T> (&t)[3])
{
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        mac_cn(t[c], w.m[c], f[0]);
        mac_cn(t[c], w.m[3 + c], f[1]);
        mac_cn(t[c], w.m[6 + c], f[2]);
    }
}

// OP: what a kernel does with the hop.
//   bool on(r)               slot r is computed
//   const cplx<T> *in(r)     its field
//   typename OP::pre         values read at the site itself
//   load(r, vol, s, p)       reads them (early, beside the next plane's loads)
//   use(r, vol, s, p, f, hop, dsum, nrm)  stores the result, adds to nrm
//   sums(r, index, nrm)      the block's sum of slot r (every lane's nrm added)
template <typename RL, typename T, class OP>
__global__ __launch_bounds__(HT_THREADS) void k_hop_tile(const cplx<RL> *__restrict__ u, OP op, int nf, geom g, hop_tiles tm)
{
    constexpr bool REC = sizeof(RL) == 8 || sizeof(T) == 4;
    constexpr int NE = REC ? 6 : 9; // link elements read from memory
    // FP32: one thread per link loads its two rows, rebuilds the third and puts
    // all nine elements into LDS, so that the twelve fields do not each spend
    // 24 multiply-adds per link on it.
    // FP64: the two rows go to LDS element by element, the wavefronts rebuild.
    constexpr bool WHOLE = sizeof(T) == 4;
    constexpr int NS = WHOLE ? 9 : NE; // elements in LDS
    constexpr int NLK = NS * HT_L;
    constexpr int PL = WHOLE ? 6 : (NLK + HT_THREADS - 1) / HT_THREADS; // elements loaded per thread
    __shared__ __align__(16) cplx<RL> lnk[2][WHOLE ? NLK : PL * HT_THREADS]; // values past NLK are not used
    __shared__ __align__(16) cplx<T> fld[HT_F][3 * HT_CELLS + 1]; // one cell that takes what the last halo lanes load
    const hop_block b = hop_block_of(tm, g);
    const int t = threadIdx.x, lane = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int tx = lane & (HT_X - 1), ty = lane / HT_X;
    const int x0 = b.bx * HT_X, y0 = b.by * HT_Y;
    const bool valid = x0 + tx < g.n0 && y0 + ty < g.n1;
    const int r = b.group * HT_F + w;
    const bool on = r < nf && op.on(r);
    const int64_t vol = g.vol;
    const uint32_t plane = (uint32_t)g.n0 * (uint32_t)g.n1;
    auto cell = [&](int x, int y) { // site of periodic (x, y) >= -1 within its plane
        return (uint32_t)((x + g.n0) % g.n0) + (uint32_t)g.n0 * (uint32_t)((y + g.n1) % g.n1);
    };
    const uint32_t own = cell(x0 + tx, y0 + ty);

    // links of the plane: this thread's elements, in memory and in LDS order
    // (element e of the x links, then of the y links, then of the z links)
    int64_t lsrc[WHOLE ? 1 : PL];
    int ldst = 0, lstep = 0;
    auto link_at = [&](int region, int i) { // memory offset of element 0 and the site of link i of a region
        const int x = region == 0 ? x0 + i % (HT_X + 1) - 1 : x0 + i % HT_X;
        const int y = region == 0 ? y0 + i / (HT_X + 1) : (region == 1 ? y0 + i / HT_X - 1 : y0 + i / HT_X);
        return (int64_t)(9 * region) * vol + cell(x, y);
    };
    if constexpr (WHOLE) {
        const int region = t < HT_LX ? 0 : (t < HT_LX + HT_LY ? 1 : 2);
        const int i = region == 0 ? t : (region == 1 ? t - HT_LX : (t - HT_LX - HT_LY) % HT_LZ);
        lsrc[0] = link_at(region, i);
        lstep = region == 0 ? HT_LX : (region == 1 ? HT_LY : HT_LZ);
        ldst = (region == 0 ? 0 : (region == 1 ? NS * HT_LX : NS * (HT_LX + HT_LY))) + i;
    } else {
#pragma unroll
        for (int k = 0; k < PL; ++k) {
            int q = t + k * HT_THREADS;
            lsrc[k] = own;
            if (q < NS * HT_LX) {
                lsrc[k] = link_at(0, q % HT_LX) + (int64_t)(q / HT_LX) * vol;
            } else if (q < NS * (HT_LX + HT_LY)) {
                q -= NS * HT_LX;
                lsrc[k] = link_at(1, q % HT_LY) + (int64_t)(q / HT_LY) * vol;
            } else if (q < NLK) {
                q -= NS * (HT_LX + HT_LY);
                lsrc[k] = link_at(2, q % HT_LZ) + (int64_t)(q / HT_LZ) * vol;
            }
        }
    }
    // halo of the plane: two (colour, cell) values per lane
    uint32_t hsrc[2];
    int hdst[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int e = lane + 64 * k, c = e / HT_HALO;
        int h = e - c * HT_HALO, hx, hy;
        if (h < 2 * HT_Y) {
            hx = h & 1 ? HT_HX - 1 : 0;
            hy = 1 + (h >> 1);
        } else {
            h -= 2 * HT_Y;
            hx = 1 + (h & (HT_X - 1));
            hy = h >= HT_X ? HT_Y + 1 : 0;
        }
        hdst[k] = e < 3 * HT_HALO ? c * HT_CELLS + hy * HT_HX + hx : 3 * HT_CELLS;
        hsrc[k] = e < 3 * HT_HALO ? (uint32_t)c * (uint32_t)vol + cell(x0 + hx - 1, y0 + hy - 1) : own;
    }
    const int home = (ty + 1) * HT_HX + tx + 1; // this lane's cell
    cplx<T> *const mine = fld[w];
    const cplx<T> *const f = on ? op.in(r) : nullptr;

    cplx<T> cur[3], nxt[3], halo[2], carry[3];
    cplx<RL> lreg[PL];
    auto load_links = [&](uint32_t p) {
        if constexpr (WHOLE) {
            if (t < HT_L)
#pragma unroll
                for (int k = 0; k < PL; ++k) lreg[k] = get(u + lsrc[0] + (int64_t)k * vol + p);
        } else {
#pragma unroll
            for (int k = 0; k < PL; ++k) lreg[k] = get(u + lsrc[k] + p);
        }
    };
    auto store_links = [&](int buf) {
        if constexpr (WHOLE) {
            if (t < HT_L) {
                mat3<T> m;
#pragma unroll
                for (int k = 0; k < 6; ++k) m.m[k] = {(T)lreg[k].re, (T)lreg[k].im};
                su3_row3(m);
#pragma unroll
                for (int k = 0; k < 9; ++k) put(&lnk[buf][ldst + k * lstep], cplx<RL>{(RL)m.m[k].re, (RL)m.m[k].im});
            }
        } else {
#pragma unroll
            for (int k = 0; k < PL; ++k) put(&lnk[buf][t + k * HT_THREADS], lreg[k]);
        }
    };
    auto load_halo = [&](uint32_t p) {
#pragma unroll
        for (int k = 0; k < 2; ++k) halo[k] = get(at32(f, hsrc[k] + p));
    };
    auto store_plane = [&](const cplx<T> (&v)[3]) {
#pragma unroll
        for (int c = 0; c < 3; ++c) put(mine + c * HT_CELLS + home, v[c]);
#pragma unroll
        for (int k = 0; k < 2; ++k) put(mine + hdst[k], halo[k]);
    };
    {
        // first plane, and the hop from the plane below it
        const uint32_t p = plane * (uint32_t)b.z0, pm = plane * (uint32_t)(b.z0 > 0 ? b.z0 - 1 : g.n2 - 1);
        load_links(p);
        if (on) {
            cplx<RL> l[NE];
            cplx<T> below[3];
#pragma unroll
            for (int e = 0; e < NE; ++e) l[e] = get(u + (int64_t)(18 + e) * vol + own + pm);
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                below[c] = get(at32(f + (int64_t)c * vol, own + pm));
                cur[c] = get(at32(f + (int64_t)c * vol, own + p));
            }
            load_halo(p);
            clear(carry);
            hop_bwd(hop_link<NE, RL, T>(l), below, carry);
            store_plane(cur);
        }
        store_links(0);
    }
    __syncthreads();
    T ia2[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) ia2[i] = T(1.0 / (g.a[i + 1] * g.a[i + 1]));
    const T dsum = T(1.0 / (g.a[1] * g.a[1]) + 1.0 / (g.a[2] * g.a[2]) + 1.0 / (g.a[3] * g.a[3]));
    double nrm = 0;
#pragma unroll 1
    for (int kz = 0; kz < b.nz; ++kz) {
        const int z = b.z0 + kz;
        const uint32_t p = plane * (uint32_t)z, pn = plane * (uint32_t)(z + 1 < g.n2 ? z + 1 : 0);
        const bool more = kz + 1 < b.nz;
        const cplx<RL> *L = lnk[kz & 1];
        typename OP::pre own_values;
        if (on) {
#pragma unroll
            for (int c = 0; c < 3; ++c) nxt[c] = get(at32(f + (int64_t)c * vol, own + pn));
            if (more) load_halo(pn);
            op.load(r, vol, own + p, own_values);
        }
        if (more) load_links(pn);
        if (on) {
            cplx<T> hop[3], h[3], v[3];
            clear(hop);
            clear(h);
            // hop += h / a_i^2 once both neighbours of a direction are in h
            auto add = [&](T c2) {
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    hop[c].re = fmx(c2, h[c].re, hop[c].re);
                    hop[c].im = fmx(c2, h[c].im, hop[c].im);
                }
                pin(hop);
                clear(h);
                __builtin_amdgcn_sched_barrier(0);
            };
            auto cellv = [&](int d) {
#pragma unroll
                for (int c = 0; c < 3; ++c) v[c] = get(mine + c * HT_CELLS + home + d);
            };
            auto lds_link = [&](int at, int stride) {
                cplx<RL> l[NS];
#pragma unroll
                for (int e = 0; e < NS; ++e) l[e] = get(L + at + e * stride);
                return hop_link<NS, RL, T>(l);
            };
            const int lx = tx + 1 + (HT_X + 1) * ty, ly = NS * HT_LX + tx + HT_X * (ty + 1);
            cellv(1);
            hop_fwd(lds_link(lx, HT_LX), v, h);
            pin(h);
            __builtin_amdgcn_sched_barrier(0);
            cellv(-1);
            hop_bwd(lds_link(lx - 1, HT_LX), v, h);
            add(ia2[0]);
            cellv(HT_HX);
            hop_fwd(lds_link(ly, HT_LY), v, h);
            pin(h);
            __builtin_amdgcn_sched_barrier(0);
            cellv(-HT_HX);
            hop_bwd(lds_link(ly - HT_X, HT_LY), v, h);
            add(ia2[1]);
            const mat3<T> uz = lds_link(NS * (HT_LX + HT_LY) + lane, HT_LZ);
            hop_fwd(uz, nxt, carry);
#pragma unroll
            for (int c = 0; c < 3; ++c) h[c] = carry[c];
            add(ia2[2]);
            clear(carry);
            hop_bwd(uz, cur, carry);
            pin(carry);
            if (valid) op.use(r, vol, own + p, own_values, cur, hop, dsum, nrm);
        }
        if (more) {
            // every lane's reads of this plane come before the writes of the
            // next one; other wavefronts read only the other link buffer, the
            // one written here was last read before the previous barrier
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            if (on) {
#pragma unroll
                for (int c = 0; c < 3; ++c) cur[c] = nxt[c];
                store_plane(cur);
            }
            store_links((kz + 1) & 1);
            __syncthreads();
        }
    }
    if (on && OP::NORM) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) nrm += __shfl_down(nrm, off, 64);
        if (lane == 0) op.sum(r, b.index, nrm);
    }
}

// The tiling of lattice g for nf slots.
inline hop_tiles hop_tiles_for(const geom &g, int nf)
{
    hop_tiles t{};
    t.ntx = (g.n0 + HT_X - 1) / HT_X;
    t.nty = (g.n1 + HT_Y - 1) / HT_Y;
    t.groups = (nf + HT_F - 1) / HT_F;
    const int64_t tiles = (int64_t)t.ntx * t.nty;
    // at least two blocks per CU, runs of at least four planes
    int nzr = (int)((2 * HT_CUS + tiles * t.groups - 1) / (tiles * t.groups));
    nzr = nzr < g.n2 / 4 ? nzr : g.n2 / 4;
    if (nzr < 1) nzr = 1;
    t.zc = (g.n2 + nzr - 1) / nzr;
    t.nzr = (g.n2 + t.zc - 1) / t.zc;
    return t;
}

inline unsigned hop_grid(const hop_tiles &t) { return (unsigned)t.ntx * (unsigned)t.nty * (unsigned)t.nzr * (unsigned)t.groups; }

enum hop_op { HOP_FP64, HOP_FP64_CHEB, HOP_FP32 }; // what a kernel computes

// Whether the tiles of lattice g are faster than the wave items of nrq_map.h for nf slots.
// The time of the tiles goes with the planes of a run times the rounds of blocks, one block per CU (half way
// between whole rounds and their exact number fits best); that of the wave items with their
// number, whatever part of their lanes is used, so that bands that fill 64 lanes badly favour
// the tiles and tiles that reach past the lattice the wave items.  plane_items are the wave items
// that cost as much as one plane of a tile on every CU: by operator, by rows that start on cache
// lines (n0 a multiple of 16) or do not, and by groups.  A block of wave items holds 16 slots in
// FP64 and 32 in FP32, so 24 and 36 slots leave part of it idle, and 48 fill it in FP64 only.
// Fitted to each operator taken alone both ways in CN steps of four solvers on 341 lattices of 10 to 112
// a side, 12, 24, 36 and 48 slots, both storages: against wave items everywhere steps are 1.12 times as
// fast in the mean and no less than 0.94 times.  us per step, wave items / tiles, 12 slots:
// FP64 Chebyshev 64^3 1497 / 1142, 90x62x58 2112 / 2099, 33x30x27 401 / 335, 32^3 238 / 271, 48x25x17
// 212 / 308; mixed Chebyshev 64^3 1001 / 759, 48^3 462 / 383, 8x81x27 437 / 210, 32^3 185 / 190,
// 90x62x58 1379 / 1459; GMRES 64^3 2071 / 1689, 40^3 613 / 646, 30x34x22 397 / 393.  With 48 slots
// mixed Chebyshev 48^3 2212 / 1731; FP64 Chebyshev 28^3 596 / 633, 48^3 2615 / 2489 and 48x25x17
// 610 / 663 (FP32 links), the line being between the last two.
// A group with idle wavefronts costs as much as a full one: tiles for at least 4/5 full
// groups (64^3 with 2 slots, mixed Chebyshev: 311 / 401).
inline bool hop_tiles_pay(const geom &g, const hop_tiles &t, int nf, hop_op op)
{
    static const double plane_items[3][2][NSLOT_GROUPS] = {
        {{1175, 1250, 1150, 1370}, {1250, 1165, 1400, 1650}}, // FP64
        {{1175, 1175, 1150, 1370}, {1360, 1175, 1375, 1650}}, // FP64 Chebyshev step
        {{675, 625, 350, 350}, {675, 550, 500, 500}},         // FP32
    };
    if (5 * nf < 4 * HT_F * t.groups || t.groups > NSLOT_GROUPS) return false;
    const int nc = op == HOP_FP32 ? 4 : 2; // fields per thread of the default wave items
    const lf_map mp = make_lf_map(g, 64, 8, 4, 1);
    const double items = (double)mp.nsb * ((nf + nc - 1) / nc);
    const double blocks = (double)hop_grid(t) / HT_CUS;
    const double per_plane = plane_items[op][g.n0 % HT_X != 0][t.groups - 1];
    return items > 0.5 * (std::ceil(blocks) + blocks) * (t.zc - 0.5) * per_plane;
}

} // namespace nrq
