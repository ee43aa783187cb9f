/*
 * kmc_kernels.hip -- marching-cubes kernels for gfx950 (CDNA4, wave64).
 *
 * The path is a memory-bound stencil followed by an ordered stream
 * emission; nothing here is a contraction, so nothing goes to MFMA.
 *
 * Classification is bit-sliced: a wave loads 64 consecutive nodes of a row,
 * compares them against every isolevel of the pass and turns each level's
 * predicate into a 64-bit chunk mask with one ballot.  Edge crossings are XORs
 * of (shifted) chunk masks, cell activity is OR & ~AND of the eight corner
 * masks, and every rank the ordered emission needs is a popcount.
 * Dense per-node work is therefore one load, one compare per level and one
 * ballot per level; only crossing edges and active cells do more.
 *
 * Passes: classify (values -> masks), count (per-row counts and in-row chunk
 * prefixes), scan (row prefixes), then the emit in chunk batches (kmc_emit.hip).
 * The tile-team emit here (each wave marching a band of rows through z with LDS
 * rings of masks) remains for volumes whose y or z exceed its lists' fields.
 *
 * Arithmetic follows Source/Core/Visualization/Mapper/MarchingCubes.cpp bit for
 * bit: the comparison double(v) > isolevel (:299-316), the FP64 clamp / ratio /
 * lerp of interpolate_vertex (:326-356), the float (p + min) * scale of the
 * callers (:169-173, :382-386) and the float cross product of Vector3::cross
 * (Source/Core/Matrix/Vector3.h:479-485).  The file is compiled with
 * -ffp-contract=off so that no multiply-add is fused.
 */
#include <hip/hip_runtime.h>
#include <algorithm>
#include <map>
#include <mutex>
#include "kmc_chunks.h"
#include "kmc_device.h"
#include "kmc_internal.h"
#include "kmc_job.h"

#pragma clang fp contract(off)

namespace kmc {

/* ------------------------------------------------------------------------- */
/* classification                                                              */
/* ------------------------------------------------------------------------- */

template <typename T>
struct Classify {
    /* bit l set iff double(v) > iso[l]  (MarchingCubes.cpp:306-313) */
    static __device__ __forceinline__ uint32_t bits(T v, const JobArgs& a)
    {
        const double d = (double)v;
        uint32_t r = 0;
#pragma unroll
        for (int l = 0; l < kMaxLevels; ++l)
            if (l < (int)a.nlev) r |= (d > a.iso[l] ? 1u : 0u) << l;
        return r;
    }
};

template <>
struct Classify<float> {
    /* For float data, double(v) > iso  <=>  v > thr with thr the largest
     * float not above iso (computed on the host; NaN for a NaN isolevel). */
    static __device__ __forceinline__ uint32_t bits(float v, const JobArgs& a)
    {
        uint32_t r = 0;
#pragma unroll
        for (int l = 0; l < kMaxLevels; ++l)
            if (l < (int)a.nlev) r |= (v > a.thr[l] ? 1u : 0u) << l;
        return r;
    }
};

/* ------------------------------------------------------------------------- */
/* tile-team emit                                                              */
/* ------------------------------------------------------------------------- */

/* The emit pass runs one independent team per wave: a team marches its own
 * unit (level, band, slab) in its own LDS region, so nothing in the emit pass
 * waits for another wave.  The LDS operations of one wave complete in issue
 * order; wave_sync only keeps the compiler from moving memory operations
 * across the points where lanes start reading what other lanes wrote. */

/* LDS arrays of one team (layout of lds_layout) and the shared case table. */
struct Team {
    const uint64_t* tri;  // [256] case table
    uint64_t* bits;       // [nslots][nrb][NC]
    uint32_t* wpv;        // [2][R+2][NC]
    uint64_t* act;        // [ncs][R+1][NC]
    uint32_t* pt;         // [ncs][R+1][NC]
    uint32_t* ap;         // [ncs][R+1][NC]
    uint32_t* crec;       // [ncs][fn_cap]
    float* fn;            // [ncs][fn_cap][3]
    uint32_t* vq;         // [queue_cap]
    uint32_t* tq;         // [queue_cap]
    uint32_t nrb, R, NC, fn_cap;
};

__device__ __forceinline__ Team make_team(const JobArgs& a, uint8_t* smem, uint32_t wave)
{
    const LdsLayout L = lds_layout(a);
    uint8_t* base = smem + kTableBytes + wave * a.team_stride;
    Team v;
    v.tri = (const uint64_t*)smem;
    v.bits = (uint64_t*)(base + L.off_bits);
    v.wpv = (uint32_t*)(base + L.off_wpv);
    v.act = (uint64_t*)(base + L.off_act);
    v.pt = (uint32_t*)(base + L.off_pt);
    v.ap = (uint32_t*)(base + L.off_ap);
    v.crec = (uint32_t*)(base + L.off_crec);
    v.fn = (float*)(base + L.off_fn);
    v.vq = (uint32_t*)(base + L.off_vq);
    v.tq = (uint32_t*)(base + L.off_tq);
    v.nrb = L.nrb;
    v.R = a.R;
    v.NC = a.NC;
    v.fn_cap = a.fn_cap;
    return v;
}

/* The level a unit works on: its bit volume, prefix segments and outputs. */
struct Level {
    const uint64_t* bits;    // [nz][ny][NC] chunk masks of the level
    const uint64_t* pre_v;   // prefixes of per-node-row vertex counts
    const uint64_t* pre_t;   // prefixes of per-cell-row triangle counts
    uint64_t bv, bt;         // first prefix of each segment (outputs index from 0)
    double iso;
    float* coords;
    float* normals;
    uint32_t* conn;
    uint64_t cap_v, cap_t;
};

__device__ __forceinline__ Level level_of(const JobArgs& a, uint32_t l)
{
    Level L;
    L.bits = a.bitvol + (uint64_t)l * ((uint64_t)a.nz * a.ny * a.NC);
    L.pre_v = a.prefix + (uint64_t)(l * 2 + 0) * a.nrows;
    L.pre_t = a.prefix + (uint64_t)(l * 2 + 1) * a.nrows;
    L.bv = L.pre_v[0];
    L.bt = L.pre_t[0];
    L.iso = a.iso[0];
    L.coords = a.coords[0];
    L.normals = a.normals[0];
    L.conn = a.conn[0];
    L.cap_v = a.cap_vertices[0];
    L.cap_t = a.cap_triangles[0];
#pragma unroll
    for (int k = 1; k < kMaxLevels; ++k) {
        if (k == (int)l) {
            L.iso = a.iso[k];
            L.coords = a.coords[k];
            L.normals = a.normals[k];
            L.conn = a.conn[k];
            L.cap_v = a.cap_vertices[k];
            L.cap_t = a.cap_triangles[k];
        }
    }
    return L;
}

/* Ring slot of node slice s (s >= -2): any 3 consecutive slices get distinct
 * slots. */
template <int M>
__device__ __forceinline__ uint32_t bslot(int s) { return (uint32_t)(s + 3) % 3u; }

/* Ring slot of cell slice zc (VertexNormal keeps two cell slices). */
template <int M>
__device__ __forceinline__ uint32_t cslot(int zc) { return M == kModeVertex ? ((uint32_t)zc & 1u) : 0u; }

/* Row of chunk masks: slot sl, LDS row r (node row y = y0 - 1 + r). */
__device__ __forceinline__ const uint64_t* brow(const Team& v, uint32_t sl, uint32_t r)
{
    return v.bits + (sl * v.nrb + r) * v.NC;
}
/* Window vertex chunk prefixes of window slice ws (0: node slice z-1, 1: z)
 * of tile z, window row w.  The two slots hold node slices by parity, so
 * slice z's prefixes of step z are slice z-1's of step z+1. */
__device__ __forceinline__ uint32_t* wrow(const Team& v, int z, uint32_t ws, uint32_t w)
{
    const uint32_t slot = (uint32_t)(z - 1 + (int)ws) & 1u;
    return v.wpv + (slot * (v.R + 2) + w) * v.NC;
}
/* Cell data index: cell slot cs, cell row j (cell row y0 - 1 + j), chunk c. */
__device__ __forceinline__ uint32_t cidx(const Team& v, uint32_t cs, uint32_t j, uint32_t c)
{
    return (cs * (v.R + 1) + j) * v.NC + c;
}

/* Bits of chunk c of a row of NC chunks shifted so that bit i holds node x+1. */
__device__ __forceinline__ uint64_t shift_next(const uint64_t* row, uint32_t c, uint32_t NC)
{
    return (row[c] >> 1) | ((c + 1 < NC ? row[c + 1] : 0ull) << 63);
}

struct Cross { uint64_t x, y, z; };

/* Crossing edges owned by the nodes of chunk c of window row w (node row
 * y0-1+w) of window slice ws (node slice z-1+ws).  z-edges reach slice
 * z+ws, whose masks the ring holds. */
template <int M>
__device__ __forceinline__ Cross window_cross(const JobArgs& a, const Team& v, int z, int y0,
                                              uint32_t ws, uint32_t w, uint32_t c)
{
    Cross k;
    const int s = z - 1 + (int)ws;
    const int y = y0 - 1 + (int)w;
    if (s < 0 || s >= (int)a.nz || y < 0 || y >= (int)a.ny) { k.x = k.y = k.z = 0; return k; }
    const uint64_t* row = brow(v, bslot<M>(s), w);
    const uint64_t b = row[c];
    k.x = (b ^ shift_next(row, c, a.NC)) & valid_mask(c, a.nx - 1);
    k.y = (y + 1 < (int)a.ny) ? ((b ^ brow(v, bslot<M>(s), w + 1)[c]) & valid_mask(c, a.nx)) : 0ull;
    k.z = (s + 1 < (int)a.nz) ? ((b ^ brow(v, bslot<M>(s + 1), w)[c]) & valid_mask(c, a.nx)) : 0ull;
    return k;
}

/* The eight corner masks of the cells of chunk c, cell row cy (node rows cy,
 * cy+1), cell slice cz (node slices cz, cz+1), shifted so that bit i is
 * corner k of cell x = 64c + i (corner order of MarchingCubes.cpp:187-194). */
struct Corners { uint64_t c[8]; };

template <int M>
__device__ __forceinline__ Corners corners_at(const JobArgs& a, const Team& v, int y0, uint32_t c, int cy, int cz)
{
    const uint32_t r = (uint32_t)(cy - y0 + 1);
    const uint64_t* r0 = brow(v, bslot<M>(cz), r);
    const uint64_t* r1 = brow(v, bslot<M>(cz), r + 1);
    const uint64_t* r2 = brow(v, bslot<M>(cz + 1), r);
    const uint64_t* r3 = brow(v, bslot<M>(cz + 1), r + 1);
    Corners k;
    k.c[0] = r0[c]; k.c[1] = shift_next(r0, c, a.NC); k.c[3] = r1[c]; k.c[2] = shift_next(r1, c, a.NC);
    k.c[4] = r2[c]; k.c[5] = shift_next(r2, c, a.NC); k.c[7] = r3[c]; k.c[6] = shift_next(r3, c, a.NC);
    return k;
}

__device__ __forceinline__ uint32_t corner_index(const Corners& k, uint32_t i)
{
    uint32_t ci = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) ci |= (uint32_t)((k.c[q] >> i) & 1ull) << q;
    return ci;
}

/* Cube index of cell (cx, cy, cz) from the mask ring (y0: first band row). */
template <int M>
__device__ __forceinline__ uint32_t cube_index_at(const Team& v, int y0, uint32_t cx, int cy, int cz)
{
    const uint32_t r = (uint32_t)(cy - y0 + 1);
    const uint64_t* b00 = brow(v, bslot<M>(cz), r);
    const uint64_t* b01 = brow(v, bslot<M>(cz), r + 1);
    const uint64_t* b10 = brow(v, bslot<M>(cz + 1), r);
    const uint64_t* b11 = brow(v, bslot<M>(cz + 1), r + 1);
    const uint32_t c0 = cx >> 6, i0 = cx & 63u;
    const uint32_t c1 = (cx + 1) >> 6, i1 = (cx + 1) & 63u;
    uint32_t ci = 0;
    ci |= (uint32_t)((b00[c0] >> i0) & 1ull) << 0;
    ci |= (uint32_t)((b00[c1] >> i1) & 1ull) << 1;
    ci |= (uint32_t)((b01[c1] >> i1) & 1ull) << 2;
    ci |= (uint32_t)((b01[c0] >> i0) & 1ull) << 3;
    ci |= (uint32_t)((b10[c0] >> i0) & 1ull) << 4;
    ci |= (uint32_t)((b10[c1] >> i1) & 1ull) << 5;
    ci |= (uint32_t)((b11[c1] >> i1) & 1ull) << 6;
    ci |= (uint32_t)((b11[c0] >> i0) & 1ull) << 7;
    return ci;
}

/* Cube index of cell (cx, cy, cz) read from the level's bit volume in memory
 * (for cells whose node slices have left the mask ring). */
__device__ __forceinline__ uint32_t cube_index_mem(const JobArgs& a, const uint64_t* bits, uint32_t cx, int cy, int cz)
{
    const uint64_t* b00 = bits + ((uint64_t)cz * a.ny + (uint64_t)cy) * a.NC;
    const uint64_t* b01 = b00 + a.NC;
    const uint64_t* b10 = b00 + (uint64_t)a.ny * a.NC;
    const uint64_t* b11 = b10 + a.NC;
    const uint32_t c0 = cx >> 6, i0 = cx & 63u;
    const uint32_t c1 = (cx + 1) >> 6, i1 = (cx + 1) & 63u;
    uint32_t ci = 0;
    ci |= (uint32_t)((b00[c0] >> i0) & 1ull) << 0;
    ci |= (uint32_t)((b00[c1] >> i1) & 1ull) << 1;
    ci |= (uint32_t)((b01[c1] >> i1) & 1ull) << 2;
    ci |= (uint32_t)((b01[c0] >> i0) & 1ull) << 3;
    ci |= (uint32_t)((b10[c0] >> i0) & 1ull) << 4;
    ci |= (uint32_t)((b10[c1] >> i1) & 1ull) << 5;
    ci |= (uint32_t)((b11[c1] >> i1) & 1ull) << 6;
    ci |= (uint32_t)((b11[c0] >> i0) & 1ull) << 7;
    return ci;
}

/* ------------------------------------------------------------------------- */
/* grid-stride ranges                                                          */
/* ------------------------------------------------------------------------- */

/* (Contiguous parts per XCD -- workgroups reach the eight XCDs round-robin,
 * each with an L2 of its own -- measured 3 % slower on the whole call than
 * this plain interleave: the emission lost more than count gained.) */
struct Span { uint64_t lo, first, end, step; };

/* Grid-stride walk over [b, e) in units of `units` items per workgroup
 * (`unit`: this thread's or wave's place in its workgroup). */
__device__ __forceinline__ Span grid_span(uint64_t b, uint64_t e, uint32_t units, uint32_t unit)
{
    Span sp;
    sp.lo = b;
    sp.first = b + (uint64_t)blockIdx.x * units + unit;
    sp.end = e;
    sp.step = (uint64_t)gridDim.x * units;
    return sp;
}

/* ------------------------------------------------------------------------- */
/* wave scan                                                                   */
/* ------------------------------------------------------------------------- */

/* In-place exclusive scan of n u32 values in LDS by one wave; returns the
 * total (the same in every lane). */
__device__ __forceinline__ uint32_t wave_exclusive_scan(uint32_t* p, uint32_t n)
{
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t carry = 0;
    for (uint32_t g = 0; g < n; g += 64) {
        const uint32_t i = g + lane;
        const uint32_t x = i < n ? p[i] : 0u;
        const uint32_t inc = wave_incl_scan(x);
        if (i < n) p[i] = carry + inc - x;
        carry += __shfl(inc, 63);
    }
    return carry;
}

/* ------------------------------------------------------------------------- */
/* slice loading                                                               */
/* ------------------------------------------------------------------------- */

/* Bring the chunk masks of node rows y0-1 .. y0+R+1 of node slices
 * s_lo .. s_hi of the level into their ring slots; rows and slices outside
 * the volume are zero.  For one slice the rows are contiguous both in the
 * bit volume and in LDS, so the copy is a flat range per slice; a lane's
 * loads are all issued before its stores. */
template <int M>
__device__ void load_slices(const JobArgs& a, const Team& v, const Level& L, int s_lo, int s_hi, int y0)
{
    if (s_hi < s_lo) return;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t nseg = v.nrb * a.NC;              // elements of one slice
    const uint32_t total = (uint32_t)(s_hi - s_lo + 1) * nseg;
    const uint32_t e_lo = (y0 - 1 < 0) ? a.NC : 0u;
    const int rows_left = (int)a.ny - (y0 - 1);
    const uint32_t e_hi = (rows_left >= (int)v.nrb ? v.nrb : (uint32_t)(rows_left > 0 ? rows_left : 0)) * a.NC;
    const uint64_t slice_words = (uint64_t)a.ny * a.NC;
    const int64_t row0 = (int64_t)(y0 - 1) * a.NC;
    constexpr int kB = 4;
    /* element i = b0 + 64u + lane is element e of slice s_lo + si */
    uint32_t si = 0, e = lane;
    while (e >= nseg) { e -= nseg; ++si; }
    for (uint32_t b0 = 0; b0 < total; b0 += 64u * kB) {
        uint64_t val[kB];
        uint32_t dst[kB];
#pragma unroll
        for (int u = 0; u < kB; ++u) {
            const uint32_t i = b0 + 64u * u + lane;
            const int s = s_lo + (int)si;
            const bool ok = i < total && s >= 0 && s < (int)a.nz && e >= e_lo && e < e_hi;
            val[u] = ok ? L.bits[(uint64_t)((int64_t)s * (int64_t)slice_words + row0 + (int64_t)e)] : 0ull;
            dst[u] = i < total ? bslot<M>(s) * nseg + e : ~0u;
            e += 64u;
            while (e >= nseg) { e -= nseg; ++si; }
        }
#pragma unroll
        for (int u = 0; u < kB; ++u)
            if (dst[u] != ~0u) v.bits[dst[u]] = val[u];
    }
}

/* ------------------------------------------------------------------------- */
/* per-tile counts and prefixes (lanes on (row, chunk))                        */
/* ------------------------------------------------------------------------- */

/* Totals of a tile: vertices it emits, triangles of its cell slice (halo row
 * included) and triangles of the halo row. */
struct TileTotals { uint32_t nv, nt, halo; };

/* Tile z: window vertex counts per chunk of window slices 0, 1 (node slices
 * z-1, z), rows 1..R+1 (for output ranks), and active cells / triangle
 * counts of cell slice z-1, cell rows j0..R (j = 0: the halo row y0-1, only
 * with VertexNormal); then exclusive prefixes -- window prefixes per slice
 * and triangle prefixes.  ws_v: window slice whose vertices the tile emits.
 * Lanes cover 64 >> cshift rows of 1 << cshift chunk lanes. */
template <int M>
__device__ TileTotals tile_prefixes(const JobArgs& a, const Team& v, int z, int y0, uint32_t ws_v, bool ranks,
                                    bool first)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t sub = lane >> a.cshift, cl = lane & ((1u << a.cshift) - 1u);
    const uint32_t G = 64u >> a.cshift, CS = 1u << a.cshift;
    const uint32_t nwr = a.R + 2;
    constexpr bool halo = M == kModeVertex;
    constexpr bool dup = M == kModeDup;
    const uint32_t j0 = halo ? 0u : 1u;
    const int zc = z - 1;
    const uint32_t cs = cslot<M>(zc);
    const bool wranks = ranks && !dup;
    /* window rows 1..R+1 of window slice 1 (and of slice 0 at a unit's first
     * step; later it is the previous step's slice 1) */
    if (wranks) {
        for (uint32_t ws = first ? 0u : 1u; ws < 2u; ++ws) {
            for (uint32_t w = 1 + sub; w < nwr; w += G) {
                uint32_t* dst = wrow(v, z, ws, w);
                for (uint32_t c = cl; c < a.NC; c += CS) {
                    const Cross k = window_cross<M>(a, v, z, y0, ws, w, c);
                    dst[c] = (uint32_t)(__popcll(k.x) + __popcll(k.y) + __popcll(k.z));
                }
            }
        }
    }
    for (uint32_t j = sub; j <= a.R; j += G) {
        const int y = y0 - 1 + (int)j;
        const bool live = j >= j0 && zc >= 0 && zc + 1 < (int)a.nz && y >= 0 && y + 1 < (int)a.ny;
        for (uint32_t c = cl; c < a.NC; c += CS) {
            uint64_t act = 0;
            uint32_t cnt = 0;
            if (live) {
                const Corners k = corners_at<M>(a, v, y0, c, y, zc);
                uint64_t o = 0, an = ~0ull;
#pragma unroll
                for (int q = 0; q < 8; ++q) { o |= k.c[q]; an &= k.c[q]; }
                act = (o & ~an) & valid_mask(c, a.nx - 1);
                uint64_t m = act;
                while (m) {
                    const uint32_t i = (uint32_t)__ffsll((unsigned long long)m) - 1u;
                    m &= m - 1ull;
                    cnt += (uint32_t)(v.tri[corner_index(k, i)] >> 60);
                }
            }
            v.act[cidx(v, cs, j, c)] = act;
            v.pt[cidx(v, cs, j, c)] = cnt;
            if (halo) v.ap[cidx(v, cs, j, c)] = (uint32_t)__popcll(act);
        }
    }
    wave_sync();
    if (halo) (void)wave_exclusive_scan(v.ap + cidx(v, cs, 0, 0), (a.R + 1) * a.NC);
    if (wranks) {
        for (uint32_t ws = first ? 0u : 1u; ws < 2u; ++ws)
            (void)wave_exclusive_scan(wrow(v, z, ws, 1), (nwr - 1) * a.NC);
    }
    TileTotals t;
    t.nt = uniform(wave_exclusive_scan(v.pt + cidx(v, cs, 0, 0), (a.R + 1) * a.NC));
    wave_sync();
    t.nv = wranks ? uniform(wrow(v, z, ws_v, a.R + 1)[0] - wrow(v, z, ws_v, 1)[0]) : 0u;
    t.halo = halo ? uniform(v.pt[cidx(v, cs, 1, 0)]) : 0u;
    return t;
}

/* ------------------------------------------------------------------------- */
/* vertex coordinates and normals                                              */
/* ------------------------------------------------------------------------- */

/* Coordinates of the shared vertex on the edge of node (x,y,z) along axis,
 * interpolated low -> high as calculate_isopoints does (:406,420,434). */
template <typename T>
__device__ __forceinline__ void node_edge_coords(const JobArgs& a, const T* vol, double iso,
                                                 uint32_t x, uint32_t y, uint32_t z, uint32_t axis, float out[3])
{
    interpolate<T>(a, vol, iso, x, y, z, x + (axis == 0), y + (axis == 1), z + (axis == 2), out);
}

/* Output bases of tile (z, band): vertex prefixes of node rows (z-1, y0),
 * (z-1, y0+R), (z, y0), (z, y0+R) and the triangle prefix of cell row
 * (y0, z-1), relative to the first row of their segment; one lane loads each
 * and every lane gets all five. */
struct Bases { uint64_t v[4]; uint64_t t; };

__device__ __forceinline__ Bases tile_bases(const JobArgs& a, const Level& L, int z, int y0)
{
    const uint32_t lane = threadIdx.x & 63u;
    const bool in = z < (int)a.nz, next = (uint32_t)y0 + a.R < a.ny;
    const uint64_t row = (uint64_t)z * a.ny + (uint64_t)y0;
    const uint64_t prow = (uint64_t)(z - 1) * a.ny + (uint64_t)y0;
    const uint64_t* p = nullptr;
    uint64_t b = 0;
    if (lane == 0 && z > 0) { p = L.pre_v + prow; b = L.bv; }
    if (lane == 1 && z > 0 && next) { p = L.pre_v + prow + a.R; b = L.bv; }
    if (lane == 2 && in) { p = L.pre_v + row; b = L.bv; }
    if (lane == 3 && in && next) { p = L.pre_v + row + a.R; b = L.bv; }
    if (lane == 4 && in) { p = L.pre_t + row; b = L.bt; }
    const uint64_t x = p ? *p - b : 0ull;
    Bases B;
    B.v[0] = readlane64(x, 0);
    B.v[1] = readlane64(x, 1);
    B.v[2] = readlane64(x, 2);
    B.v[3] = readlane64(x, 3);
    B.t = readlane64(x, 4);
    return B;
}

/* Rank within its tile row range of the vertex on (node x of band row k (0..R)
 * of node slice s in {z-1, z}, axis): rows 0..R-1 rank from the band's first
 * row, row R (first row of the next band) from its own start. */
template <int M>
__device__ __forceinline__ uint32_t tile_rank(const JobArgs& a, const Team& v, int z, int y0,
                                              uint32_t x, uint32_t k, int s, uint32_t axis)
{
    const uint32_t ws = (uint32_t)(s - z + 1), w = k + 1;
    const uint32_t c = x >> 6, i = x & 63u;
    const Cross e = window_cross<M>(a, v, z, y0, ws, w, c);
    const uint64_t lo = (1ull << i) - 1ull;
    const uint32_t start = wrow(v, z, ws, k == a.R ? a.R + 1 : 1)[0];
    uint32_t r = wrow(v, z, ws, w)[c] - start;
    r += __popcll(e.x & lo) + __popcll(e.y & lo) + __popcll(e.z & lo);
    if (axis >= 1) r += (uint32_t)((e.x >> i) & 1ull);
    if (axis >= 2) r += (uint32_t)((e.y >> i) & 1ull);
    return r;
}

/* VertexNormal of the vertex on (x,y,zv,axis): the float sum, in triangle
 * order, of the unnormalized face normals of the triangles that use it --
 * the order of calculate_normals_on_vertex (:569-605).  Incident cells are
 * visited in cell scan order and triangles in table order; cube indices come
 * from the bit volume and every face normal is recomputed from interpolated
 * coordinates (used when the face normals of a cell slice did not fit in
 * LDS). */
template <typename T>
__device__ void vertex_normal_direct(const JobArgs& a, const Team& v, const Level& L, const T* vol,
                                     uint32_t x, uint32_t y, int zv, uint32_t axis, float n[3])
{
    n[0] = 0.0f; n[1] = 0.0f; n[2] = 0.0f;
    const uint32_t around = around_nibbles(axis);
    for (int q = 0; q < 4; ++q) {
        int cx, cy, cz;
        around_cell(axis, q, (int)x, (int)y, zv, cx, cy, cz);
        if (cx < 0 || cy < 0 || cz < 0) continue;
        if (cx + 1 >= (int)a.nx || cy + 1 >= (int)a.ny || cz + 1 >= (int)a.nz) continue;
        const uint32_t ci = cube_index_mem(a, L.bits, (uint32_t)cx, cy, cz);
        const uint64_t w = v.tri[ci];
        const int nt = (int)(w >> 60);
        const uint32_t me = (around >> (4 * q)) & 0xFu;
        for (int t = 0; t < nt; ++t) {
            const uint32_t e0 = (uint32_t)((w >> (12 * t)) & 0xF);
            const uint32_t e1 = (uint32_t)((w >> (12 * t + 8)) & 0xF);
            const uint32_t e2 = (uint32_t)((w >> (12 * t + 4)) & 0xF);
            if (e0 != me && e1 != me && e2 != me) continue;
            float p[3][3], fn[3];
            const uint32_t es[3] = { e0, e1, e2 };
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const uint32_t o = edge_owner(es[j]);
                node_edge_coords<T>(a, vol, L.iso, (uint32_t)cx + (o & 1u), (uint32_t)(cy + (int)((o >> 1) & 1u)),
                                    (uint32_t)(cz + (int)((o >> 2) & 1u)), o >> 3, p[j]);
            }
            face_normal(p[0], p[1], p[2], fn);
            n[0] = n[0] + fn[0];
            n[1] = n[1] + fn[1];
            n[2] = n[2] + fn[2];
        }
    }
}

/* The same sum from the face normals the triangle phase kept in LDS for cell
 * slices zv-1 and zv (band rows and the halo row above the band).  Every cell
 * around a crossing edge is active; its record, at its active-cell rank (the
 * active-cell prefix of its (cell row, chunk) + the active cells before it
 * in the chunk), holds its cube index and the rank of its first triangle. */
template <int M>
__device__ void vertex_normal_ring(const JobArgs& a, const Team& v, int y0, uint32_t x, uint32_t y, int zv,
                                   uint32_t axis, float n[3])
{
    n[0] = 0.0f; n[1] = 0.0f; n[2] = 0.0f;
    const uint32_t around = around_nibbles(axis);
    for (int q = 0; q < 4; ++q) {
        int cx, cy, cz;
        around_cell(axis, q, (int)x, (int)y, zv, cx, cy, cz);
        if (cx < 0 || cy < 0 || cz < 0) continue;
        if (cx + 1 >= (int)a.nx || cy + 1 >= (int)a.ny || cz + 1 >= (int)a.nz) continue;
        const uint32_t cs = (uint32_t)cz & 1u, j = (uint32_t)(cy - y0 + 1);
        const uint32_t c = (uint32_t)cx >> 6, i = (uint32_t)cx & 63u;
        const uint32_t d = cidx(v, cs, j, c);
        const uint32_t rank = v.ap[d] + (uint32_t)__popcll(v.act[d] & ((1ull << i) - 1ull));
        const uint32_t rc = v.crec[cs * v.fn_cap + rank];
        const uint32_t base = rc >> 8;
        const uint64_t w = v.tri[rc & 0xFFu];
        const int nt = (int)(w >> 60);
        const uint32_t me = (around >> (4 * q)) & 0xFu;
        const float* f = v.fn + (size_t)cs * v.fn_cap * 3u;
        for (int t = 0; t < nt; ++t) {
            const uint32_t e0 = (uint32_t)((w >> (12 * t)) & 0xF);
            const uint32_t e1 = (uint32_t)((w >> (12 * t + 8)) & 0xF);
            const uint32_t e2 = (uint32_t)((w >> (12 * t + 4)) & 0xF);
            if (e0 != me && e1 != me && e2 != me) continue;
            const float* g = f + 3u * (base + (uint32_t)t);
            n[0] = n[0] + g[0];
            n[1] = n[1] + g[1];
            n[2] = n[2] + g[2];
        }
    }
}

/* Emit tile (z, band): the vertices of window slice ws_v (shared-vertex
 * modes, when out_vert) and the triangles of cell slice z-1 (when out_tri),
 * through two LDS work queues whose entry index is the output rank.  With
 * VertexNormal the triangles of the halo row are processed too and, when
 * keep_fn, every face normal is kept in the cell slice's ring slot; ring_ok:
 * both slots hold all their face normals. */
template <typename T, int M>
__device__ void emit_tile(const JobArgs& a, const Team& v, const Level& L, const Bases& B, const T* vol, int z,
                          int y0, uint32_t ws_v, bool out_vert, bool out_tri, const TileTotals& tt, bool keep_fn,
                          bool ring_ok)
{
    constexpr bool vn = M == kModeVertex;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t sub = lane >> a.cshift, cl = lane & ((1u << a.cshift) - 1u);
    const uint32_t G = 64u >> a.cshift, CS = 1u << a.cshift;
    const uint32_t nv_all = out_vert ? tt.nv : 0u;
    const uint32_t nt_all = tt.nt;
    const uint32_t Q = a.queue_cap;
    const int zc = z - 1;
    const int zv = z - 1 + (int)ws_v;
    const uint32_t cs = cslot<M>(zc);

    /* triangles of cell slice z-1 (with VertexNormal first, so that their face
     * normals are in LDS before the vertices below read them) */
    for (uint32_t w0 = 0; w0 < nt_all; w0 += Q) {
        for (uint32_t j = sub; j <= a.R; j += G) {
            for (uint32_t c = cl; c < a.NC; c += CS) {
                uint64_t m = v.act[cidx(v, cs, j, c)];
                if (!m) continue;
                const Corners k = corners_at<M>(a, v, y0, c, y0 - 1 + (int)j, zc);
                uint32_t r = v.pt[cidx(v, cs, j, c)];
                /* with the face normals kept, each active cell also records its first
                 * triangle and cube index at its active-cell rank */
                const bool rec = vn && keep_fn && w0 == 0;
                uint32_t ai = rec ? v.ap[cidx(v, cs, j, c)] : 0u;
                while (m) {
                    const uint32_t i = (uint32_t)__ffsll((unsigned long long)m) - 1u;
                    m &= m - 1ull;
                    const uint32_t ci = corner_index(k, i);
                    const uint32_t nt = (uint32_t)(v.tri[ci] >> 60);
                    const uint32_t x = c * 64u + i;
                    if (rec) v.crec[cs * v.fn_cap + ai++] = r << 8 | ci;
                    for (uint32_t t = 0; t < nt; ++t, ++r)
                        if (r >= w0 && r - w0 < Q) v.tq[r - w0] = x | (j << 20) | (t << 25);
                }
            }
        }
        wave_sync();
        const uint32_t ntq = (nt_all - w0) < Q ? (nt_all - w0) : Q;
        for (uint32_t q = lane; q < ntq; q += 64u) {
            const uint32_t e = v.tq[q];
            const uint32_t x = e & 0xFFFFFu, j = (e >> 20) & 0x1Fu, t = (e >> 25) & 7u;
            const uint32_t rank = w0 + q;                           // rank in the tile, halo row included
            const uint64_t tri = B.t + (uint64_t)(rank - tt.halo);
            const bool write = out_tri && j >= 1 && tri < L.cap_t;
            if (!write && !keep_fn) continue;
            const int y = y0 - 1 + (int)j;
            const uint32_t ci = cube_index_at<M>(v, y0, x, y, zc);
            const uint64_t w = v.tri[ci];
            const uint32_t eds[3] = { (uint32_t)((w >> (12 * t)) & 0xF), (uint32_t)((w >> (12 * t + 8)) & 0xF),
                                      (uint32_t)((w >> (12 * t + 4)) & 0xF) };
            float p[3][3], nn[3];
            if constexpr (M == kModeDup) {
                /* extract_surfaces_with_duplication: table orientation (:206-228) */
#pragma unroll
                for (int jj = 0; jj < 3; ++jj) {
                    const uint32_t qq = edge_ends(eds[jj]);
                    interpolate<T>(a, vol, L.iso,
                                   x + (qq & 1u), (uint32_t)y + ((qq >> 1) & 1u), (uint32_t)zc + ((qq >> 2) & 1u),
                                   x + ((qq >> 4) & 1u), (uint32_t)y + ((qq >> 5) & 1u),
                                   (uint32_t)zc + ((qq >> 6) & 1u), p[jj]);
                }
                face_normal(p[0], p[1], p[2], nn);
                float* co = L.coords + 9 * tri;
#pragma unroll
                for (int jj = 0; jj < 3; ++jj) {
                    co[3 * jj + 0] = p[jj][0];
                    co[3 * jj + 1] = p[jj][1];
                    co[3 * jj + 2] = p[jj][2];
                }
                L.normals[3 * tri + 0] = nn[0];
                L.normals[3 * tri + 1] = nn[1];
                L.normals[3 * tri + 2] = nn[2];
                continue;
            }
            if (write) {
                /* connect_isopoints: vertex ids of the three edges (:493-514) */
                uint32_t id[3];
#pragma unroll
                for (int jj = 0; jj < 3; ++jj) {
                    const uint32_t o = edge_owner(eds[jj]);
                    const uint32_t dx = o & 1u, dy = (o >> 1) & 1u, dz = (o >> 2) & 1u, ax = o >> 3;
                    const uint32_t kk = j - 1 + dy;
                    const uint32_t rk = tile_rank<M>(a, v, z, y0, x + dx, kk, zc + (int)dz, ax);
                    const uint32_t sel = (dz << 1) | (kk == a.R ? 1u : 0u);
                    const uint64_t b = sel == 0 ? B.v[0] : sel == 1 ? B.v[1] : sel == 2 ? B.v[2] : B.v[3];
                    id[jj] = (uint32_t)(b + rk);
                }
                L.conn[3 * tri + 0] = id[0];
                L.conn[3 * tri + 1] = id[1];
                L.conn[3 * tri + 2] = id[2];
            }
            if (vn && !keep_fn) continue;
            /* calculate_normals_on_polygon (:531-559); with VertexNormal the same face
             * normal is what calculate_normals_on_vertex sums */
#pragma unroll
            for (int jj = 0; jj < 3; ++jj) {
                const uint32_t o = edge_owner(eds[jj]);
                node_edge_coords<T>(a, vol, L.iso, x + (o & 1u), (uint32_t)(y + (int)((o >> 1) & 1u)),
                                    (uint32_t)(zc + (int)((o >> 2) & 1u)), o >> 3, p[jj]);
            }
            face_normal(p[0], p[1], p[2], nn);
            if constexpr (vn) {
                float* g = v.fn + ((size_t)cs * v.fn_cap + rank) * 3u;
                g[0] = nn[0]; g[1] = nn[1]; g[2] = nn[2];
            } else {
                L.normals[3 * tri + 0] = nn[0];
                L.normals[3 * tri + 1] = nn[1];
                L.normals[3 * tri + 2] = nn[2];
            }
        }
        wave_sync();
    }

    /* vertices of window slice ws_v, band rows */
    for (uint32_t w0 = 0; w0 < nv_all; w0 += Q) {
        const uint32_t start = wrow(v, z, ws_v, 1)[0];
        for (uint32_t k = sub; k < a.R && y0 + (int)k < (int)a.ny; k += G) {
            for (uint32_t c = cl; c < a.NC; c += CS) {
                const Cross e = window_cross<M>(a, v, z, y0, ws_v, k + 1, c);
                uint64_t m = e.x | e.y | e.z;
                uint32_t r = wrow(v, z, ws_v, k + 1)[c] - start;
                while (m) {
                    const uint32_t i = (uint32_t)__ffsll((unsigned long long)m) - 1u;
                    m &= m - 1ull;
                    const uint32_t base = (c * 64u + i) | (k << 20);
                    if ((e.x >> i) & 1ull) { if (r >= w0 && r - w0 < Q) v.vq[r - w0] = base; ++r; }
                    if ((e.y >> i) & 1ull) { if (r >= w0 && r - w0 < Q) v.vq[r - w0] = base | (1u << 26); ++r; }
                    if ((e.z >> i) & 1ull) { if (r >= w0 && r - w0 < Q) v.vq[r - w0] = base | (2u << 26); ++r; }
                }
            }
        }
        wave_sync();
        const uint32_t nvq = (nv_all - w0) < Q ? (nv_all - w0) : Q;
        for (uint32_t q = lane; q < nvq; q += 64u) {
            const uint32_t e = v.vq[q];
            const uint32_t x = e & 0xFFFFFu, k = (e >> 20) & 0x3Fu, axis = (e >> 26) & 3u;
            const uint64_t vid = (ws_v == 1 ? B.v[2] : B.v[0]) + (uint64_t)(w0 + q);
            if (vid >= L.cap_v) continue;
            const uint32_t y = (uint32_t)y0 + k;
            float p[3];
            node_edge_coords<T>(a, vol, L.iso, x, y, (uint32_t)zv, axis, p);
            L.coords[3 * vid + 0] = p[0];
            L.coords[3 * vid + 1] = p[1];
            L.coords[3 * vid + 2] = p[2];
            if constexpr (vn) {
                float nn[3];
                if (ring_ok) vertex_normal_ring<M>(a, v, y0, x, y, zv, axis, nn);
                else vertex_normal_direct<T>(a, v, L, vol, x, y, zv, axis, nn);
                L.normals[3 * vid + 0] = nn[0];
                L.normals[3 * vid + 1] = nn[1];
                L.normals[3 * vid + 2] = nn[2];
            }
        }
        wave_sync();
    }
}

/* Stage the case table in the workgroup's LDS (shared by its teams). */
__device__ void stage_table(uint8_t* smem)
{
    uint64_t* tri = (uint64_t*)smem;
    for (uint32_t i = threadIdx.x; i < 256; i += kEmitBlock) tri[i] = d_tri[i];
    __syncthreads();
}

/* ------------------------------------------------------------------------- */
/* classify pass: values -> bit volume                                         */
/* ------------------------------------------------------------------------- */

/* Predicate of level l for a value (double(v) > iso[l]). */
template <typename T>
__device__ __forceinline__ bool above(T v, const JobArgs& a, int l) { return (double)v > a.iso[l]; }
template <>
__device__ __forceinline__ bool above<float>(float v, const JobArgs& a, int l) { return v > a.thr[l]; }

/* Classification of node row `row` of a job (the single-volume pass). */
template <typename T, int NLEV>
__device__ __forceinline__ void classify_row(const JobArgs& a, uint64_t row)
{
    const uint32_t lane = threadIdx.x & 63u;
    const T* src = (const T*)a.values + row * a.nx;
    const uint64_t z = row / a.ny, y = row - z * a.ny;
    constexpr uint32_t kBatch = 16;
    for (uint32_t c0 = 0; c0 < a.NC; c0 += 64) {
        uint32_t lo[NLEV], hi[NLEV];
#pragma unroll
        for (int l = 0; l < NLEV; ++l) { lo[l] = 0; hi[l] = 0; }
        const uint32_t cend = (a.NC - c0) < 64u ? (a.NC - c0) : 64u;
        for (uint32_t cb = 0; cb < cend; cb += kBatch) {
            T val[kBatch];
#pragma unroll
            for (uint32_t i = 0; i < kBatch; ++i) {
                const uint32_t x = (c0 + cb + i) * 64u + lane;
                val[i] = (cb + i < cend && x < a.nx) ? __builtin_nontemporal_load(src + x) : T(0);   // read once
            }
#pragma unroll
            for (uint32_t i = 0; i < kBatch; ++i) {
                if (cb + i < cend) {
                    const bool in = (c0 + cb + i) * 64u + lane < a.nx;
                    const bool mine = lane == cb + i;
#pragma unroll
                    for (int l = 0; l < NLEV; ++l) {
                        const uint64_t m = __ballot(in && above<T>(val[i], a, l));
                        lo[l] = mine ? (uint32_t)m : lo[l];
                        hi[l] = mine ? (uint32_t)(m >> 32) : hi[l];
                    }
                }
            }
        }
        /* the 8-level instance also serves passes of 5..7 levels: store only
         * the pass's own levels.  Nontemporal stores: the masks' writes,
         * mixed into the volume's read stream, cost more than their bytes
         * (measured: 384 MiB of mask stores add ~180 us to a 4 GiB read, 25 us
         * less with the nontemporal hint) */
        if (lane < cend) {
#pragma unroll
            for (int l = 0; l < NLEV; ++l)
                if (NLEV < 8 || l < (int)a.nlev)
                    __builtin_nontemporal_store(((uint64_t)hi[l] << 32) | lo[l],
                                                &a.bitvol[(((uint64_t)l * a.nz + z) * a.ny + y) * a.NC + c0 + lane]);
        }
    }
}

/* Classification of 16 chunks from q0 on, then of every step-th such run below
 * q1, q = row * NC + chunk: the chunks of consecutive rows follow each other,
 * so that short rows share a wave's loads, and the masks of consecutive rows are
 * contiguous (one 128-byte store per level). */
template <typename T, int NLEV>
__device__ __forceinline__ void classify_chunks(const JobArgs& a, uint64_t q0, uint64_t q1, uint64_t step)
{
    const uint32_t lane = threadIdx.x & 63u;
    const T* vals = (const T*)a.values;
    const uint64_t level_words = (uint64_t)a.nz * a.ny * a.NC;
    constexpr uint32_t kBatch = 16;
    for (; q0 < q1; q0 += step) {
        const uint32_t wn = (q1 - q0) < kBatch ? (uint32_t)(q1 - q0) : kBatch;
        uint64_t row = q0 / a.NC;
        uint32_t c = (uint32_t)(q0 - row * a.NC);
        T val[kBatch];
        uint32_t cs[kBatch];
#pragma unroll
        for (uint32_t i = 0; i < kBatch; ++i) {
            cs[i] = c;
            const uint32_t x = c * 64u + lane;
            val[i] = (i < wn && x < a.nx) ? __builtin_nontemporal_load(vals + row * a.nx + x) : T(0);   // read once
            if (++c == a.NC) { c = 0; ++row; }
        }
        uint32_t lo[NLEV], hi[NLEV];
#pragma unroll
        for (int l = 0; l < NLEV; ++l) { lo[l] = 0; hi[l] = 0; }
#pragma unroll
        for (uint32_t i = 0; i < kBatch; ++i) {
            const bool in = i < wn && cs[i] * 64u + lane < a.nx;
            const bool mine = lane == i;
#pragma unroll
            for (int l = 0; l < NLEV; ++l) {
                const uint64_t m = __ballot(in && above<T>(val[i], a, l));
                lo[l] = mine ? (uint32_t)m : lo[l];
                hi[l] = mine ? (uint32_t)(m >> 32) : hi[l];
            }
        }
        /* the 8-level instance also serves passes of 5..7 levels: store only
         * the pass's own levels */
        if (lane < wn) {
#pragma unroll
            for (int l = 0; l < NLEV; ++l)
                if (NLEV < 8 || l < (int)a.nlev)
                    __builtin_nontemporal_store(((uint64_t)hi[l] << 32) | lo[l],
                                                &a.bitvol[(uint64_t)l * level_words + q0 + lane]);
        }
    }
}

/* Streams the volume once.  Each wave owns whole rows: its lanes load 64
 * consecutive nodes per chunk (one coalesced access), the comparison against
 * level l is a ballot (v_cmp into a lane mask), and the mask is parked in
 * lane c of a register by a lane-select; the masks of up to 64 chunks of a
 * row leave with one coalesced 64-bit store per level.  NLEV is the number of
 * levels, a compile-time constant so that nothing is guarded per level. */
template <typename T, int NLEV>
__global__ __launch_bounds__(kBlock) void k_classify(JobArgs a)
{
    const uint64_t nrows = (uint64_t)a.ny * a.nz;
    const uint64_t wave_id = (uint64_t)blockIdx.x * kWaves + uniform(threadIdx.x >> 6);   // uniform: scalar
    const uint64_t nwaves = ((uint64_t)gridDim.x * kBlock) >> 6;
    for (uint64_t row = wave_id; row < nrows; row += nwaves) classify_row<T, NLEV>(a, row);
}

/* The same for many short rows (classify_by_runs), 16 chunks of consecutive rows a
 * wave: 256^3 float 23.5 us a row a wave, 15.0 so. */
template <typename T, int NLEV>
__global__ __launch_bounds__(kBlock) void k_classify_runs(JobArgs a)
{
    const uint64_t wave = (uint64_t)blockIdx.x * kWaves + uniform(threadIdx.x >> 6);   // uniform: scalar
    classify_chunks<T, NLEV>(a, wave * 16, a.nrows * a.NC, (uint64_t)gridDim.x * kWaves * 16);
}

/* Node q of a dword of 8- or 16-bit values (little-endian: the first node
 * in the low bits). */
template <typename T>
__device__ __forceinline__ T dword_node(uint32_t d, uint32_t q)
{
    if constexpr (sizeof(T) == 1) return (T)(uint8_t)(d >> (8u * q));
    else return (T)(uint16_t)(d >> (16u * q));
}

/* Classification of an 8- or 16-bit volume whose rows are whole dwords (nx
 * a multiple of P = 4 / sizeof(T), the values 4-byte aligned).  A lane loads
 * one dword, P nodes, so that a wave load moves 256 bytes as a float row's
 * does (one node a lane would move 64 or 128); the lane's P comparisons are
 * bits (lane mod LPC) * P + q of its chunk's mask word, which an OR over the
 * chunk's LPC = 64 / P lanes assembles.  Work items are (row, segment of 64
 * dwords), 16 consecutive ones per wave iteration, their loads in flight
 * together; the wave's item indices are scalars. */
/* Items [i0, i1) of a job in the packed classification, item = row * nseg +
 * segment: 16 consecutive ones at a time from i0 on, then every istep-th
 * batch of 16 (i0, i1 and istep the same on all of the wave's lanes). */
template <typename T, int NLEV>
__device__ __forceinline__ void classify_packed_items(const JobArgs& a, uint64_t i0, uint64_t i1, uint64_t istep)
{
    static_assert(sizeof(T) <= 2, "8- and 16-bit values");
    constexpr uint32_t P = 4 / sizeof(T), LPC = 64 / P;
    constexpr uint32_t kBatch = 16;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t nd = a.nx / P;
    const uint32_t nseg = (nd + 63) / 64;
    const uint64_t level_words = (uint64_t)a.nz * a.ny * a.NC;
    const uint32_t* vals = (const uint32_t*)a.values;
    for (; i0 < i1; i0 += istep) {
        uint64_t row = i0 / nseg;
        uint32_t seg = (uint32_t)(i0 - row * nseg);
        uint32_t d[kBatch];
#pragma unroll
        for (uint32_t i = 0; i < kBatch; ++i) {
            const uint32_t k = seg * 64u + lane;
            d[i] = (i0 + i < i1 && k < nd) ? __builtin_nontemporal_load(vals + row * nd + k) : 0u;   // read once
            if (++seg == nseg) { seg = 0; ++row; }
        }
        row = i0 / nseg;
        seg = (uint32_t)(i0 - row * nseg);
#pragma unroll
        for (uint32_t i = 0; i < kBatch; ++i) {
            if (i0 + i < i1) {
                const bool valid = seg * 64u + lane < nd;
                const uint32_t c = seg * P + lane / LPC;
                const uint32_t sh = (lane % LPC) * P;
#pragma unroll
                for (int l = 0; l < NLEV; ++l) {
                    if (NLEV == 8 && l >= (int)a.nlev) break;   // the 8-level instance serves 5..7 levels
                    uint32_t bits = 0;
#pragma unroll
                    for (uint32_t q = 0; q < P; ++q) bits |= (valid && above<T>(dword_node<T>(d[i], q), a, l) ? 1u : 0u) << q;
                    /* OR over the chunk's lanes: each contributes its P bits */
                    uint32_t lo = sh < 32u ? bits << sh : 0u, hi = sh >= 32u ? bits << (sh - 32u) : 0u;
#pragma unroll
                    for (uint32_t m = 1; m < LPC; m <<= 1) {
                        lo |= (uint32_t)__shfl_xor((int)lo, (int)m);
                        hi |= (uint32_t)__shfl_xor((int)hi, (int)m);
                    }
                    if (lane % LPC == 0 && c < a.NC)
                        __builtin_nontemporal_store((uint64_t)hi << 32 | lo,
                                                    &a.bitvol[(uint64_t)l * level_words + row * a.NC + c]);
                }
            }
            if (++seg == nseg) { seg = 0; ++row; }
        }
    }
}

/* Whether job a's values load a dword of nodes per lane: 8- or 16-bit
 * values, rows of whole dwords, 4-byte aligned. */
template <typename T>
__device__ __host__ __forceinline__ bool packed_rows(const JobArgs& a)
{
    return sizeof(T) <= 2 && a.nx % (4 / sizeof(T)) == 0 && ((uintptr_t)a.values & 3u) == 0;
}

template <typename T, int NLEV>
__global__ __launch_bounds__(kBlock) void k_classify_packed(JobArgs a)
{
    const uint64_t nseg = (a.nx / (4 / sizeof(T)) + 63) / 64;
    const uint64_t items = (uint64_t)a.ny * a.nz * nseg;
    const uint64_t wave_id = (uint64_t)blockIdx.x * kWaves + uniform(threadIdx.x >> 6);
    const uint64_t nwaves = (uint64_t)gridDim.x * kWaves;
    classify_packed_items<T, NLEV>(a, wave_id * 16, items, nwaves * 16);
}

/* Index j with start[j] <= g < start[j+1] (start has n+1 ascending entries). */
__device__ __forceinline__ uint32_t find_job(const uint64_t* start, uint32_t n, uint64_t g)
{
    uint32_t lo = 0, hi = n;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (start[mid] <= g) lo = mid; else hi = mid;
    }
    return lo;
}

/* Classify pass of a batch of jobs sharing the value type T: a job's workgroups
 * (front_blocks) walk its chunks in steps of them all, 16 consecutive chunks a
 * wave, so that every wave has 16 loads in flight and they sweep the job in address
 * order (one contiguous range of rows per wave took 199 us on 14 volumes of 32
 * .. 256 per axis, 186 MB).  kWide: some job has more than four levels (the
 * eight-level instance's registers would otherwise halve the waves per SIMD of
 * every batch). */
template <typename T, bool kWide>
__global__ __launch_bounds__(kBlock) void k_classify_batch(const JobArgs* jobs, const BlockRef* refs)
{
    const BlockRef ref = refs[blockIdx.x];
    const JobArgs& a = jobs[ref.job];
    const uint64_t wave = (uint64_t)ref.block * kWaves + uniform(threadIdx.x >> 6);   // uniform: scalar
    const uint64_t step = (uint64_t)ref.blocks * kWaves * 16;
    if constexpr (sizeof(T) <= 2) {
        if (packed_rows<T>(a)) {
            const uint64_t items = a.nrows * ((a.nx / (4 / sizeof(T)) + 63) / 64);
            switch (a.nlev) {
            case 1: classify_packed_items<T, 1>(a, wave * 16, items, step); break;
            case 2: classify_packed_items<T, 2>(a, wave * 16, items, step); break;
            case 3: classify_packed_items<T, 3>(a, wave * 16, items, step); break;
            case 4: classify_packed_items<T, 4>(a, wave * 16, items, step); break;
            default:
                if constexpr (kWide) classify_packed_items<T, 8>(a, wave * 16, items, step);
                break;
            }
            return;
        }
    }
    const uint64_t chunks = a.nrows * a.NC;
    switch (a.nlev) {
    case 1: classify_chunks<T, 1>(a, wave * 16, chunks, step); break;
    case 2: classify_chunks<T, 2>(a, wave * 16, chunks, step); break;
    case 3: classify_chunks<T, 3>(a, wave * 16, chunks, step); break;
    case 4: classify_chunks<T, 4>(a, wave * 16, chunks, step); break;
    default:
        if constexpr (kWide) classify_chunks<T, 8>(a, wave * 16, chunks, step);
        break;
    }
}

/* ------------------------------------------------------------------------- */
/* count pass: per-row counts from the bit volume                              */
/* ------------------------------------------------------------------------- */

/* (y, z) of node row g + sub of a wave that walks row groups g = g0, g0 +
 * step, ... (g0 and step are the same on all of the wave's lanes): the
 * group's first row advances by the step's quotient and remainder by ny,
 * instead of a division of every row index. */
struct RowWalk { uint32_t yg, zg, qs, rs; };

__device__ __forceinline__ RowWalk row_walk(const JobArgs& a, uint64_t g0, uint64_t step)
{
    RowWalk w;
    const uint64_t g = uniform64(g0), s = uniform64(step);
    w.zg = (uint32_t)(g / a.ny);
    w.yg = (uint32_t)(g - (uint64_t)w.zg * a.ny);
    w.qs = (uint32_t)(s / a.ny);
    w.rs = (uint32_t)(s - (uint64_t)w.qs * a.ny);
    return w;
}

__device__ __forceinline__ void row_at(const JobArgs& a, const RowWalk& w, uint32_t sub, uint32_t& y, uint32_t& z)
{
    y = w.yg + sub;
    z = w.zg;
    if (y >= a.ny) {
        /* sub < 64: one wrap when ny >= 64 */
        if (a.ny >= 64u) {
            y -= a.ny;
            ++z;
        } else {
            z += y / a.ny;
            y %= a.ny;
        }
    }
}

__device__ __forceinline__ void row_next(const JobArgs& a, RowWalk& w)
{
    w.yg += w.rs;
    w.zg += w.qs;
    if (w.yg >= a.ny) {
        w.yg -= a.ny;
        ++w.zg;
    }
}

/* x of the lane d below within its DPP row of 16 lanes (0 for the row's
 * first d lanes): row_shr:d. */
template <int D>
__device__ __forceinline__ uint32_t row_shr(uint32_t x)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x110 + D, 0xf, 0xf, true);
}

/* Exclusive scan of x over the CS lanes of each row group (CS a power of two;
 * group cl = lane mod CS).  Groups of up to 16 lanes lie inside one DPP row:
 * the steps are row shifts, with no LDS round trip. */
__device__ __forceinline__ uint32_t group_excl_scan(uint32_t x, uint32_t cl, uint32_t CS, uint32_t& total)
{
    uint32_t inc = x;
    if (CS <= 16) {
        if (CS > 1) { const uint32_t t = row_shr<1>(inc); inc += cl >= 1 ? t : 0u; }
        if (CS > 2) { const uint32_t t = row_shr<2>(inc); inc += cl >= 2 ? t : 0u; }
        if (CS > 4) { const uint32_t t = row_shr<4>(inc); inc += cl >= 4 ? t : 0u; }
        if (CS > 8) { const uint32_t t = row_shr<8>(inc); inc += cl >= 8 ? t : 0u; }
    } else {
        for (uint32_t d = 1; d < CS; d <<= 1) {
            const uint32_t t = __shfl_up(inc, d, (int)CS);
            if (cl >= d) inc += t;
        }
    }
    total = __shfl(inc, (int)CS - 1, (int)CS);
    return inc - x;
}

/* Triangles of a chunk's cells.  The table cuts each loop of n crossed edges into
 * n - 2 triangles, so a cell of E crossed edges and L loops has E - 2 L.  The
 * edges are twelve popcounts; more than one loop takes a face with all four
 * edges crossed or two opposite corners that differ from all their neighbours,
 * and only those cells are looked up: fewer[] holds 2 (L - 1).  A lookup per
 * active cell runs each wave as long as its fullest chunk takes (512^3: 43 us, so
 * 27; 256^3 7.9 and 5.5; 14 volumes of up to 256^3 in a batch 42 and 33). */
__device__ __forceinline__ uint32_t chunk_triangles(const RowChunk& o, const uint8_t* fewer)
{
    int n = -2 * __popcll(o.act);
    uint32_t multi[2];
    /* 32 cells at a time, one after the other: half the registers */
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int d = 32 * h;
        const uint32_t m = (uint32_t)(o.act >> d);
        /* the x + 1 corners: the next bits, the last one's from the next chunk */
        const uint32_t nx = h ? o.next : 0u;
        const uint32_t k0 = (uint32_t)(o.k0 >> d), k1 = (uint32_t)(o.k0 >> (d + 1)) | nx << 31;
        const uint32_t k3 = (uint32_t)(o.k3 >> d), k2 = (uint32_t)(o.k3 >> (d + 1)) | (nx >> 1) << 31;
        const uint32_t k4 = (uint32_t)(o.k4 >> d), k5 = (uint32_t)(o.k4 >> (d + 1)) | (nx >> 2) << 31;
        const uint32_t k7 = (uint32_t)(o.k7 >> d), k6 = (uint32_t)(o.k7 >> (d + 1)) | (nx >> 3) << 31;
        const uint32_t x0 = (k0 ^ k1) & m, x1 = (k3 ^ k2) & m, x2 = (k4 ^ k5) & m, x3 = (k7 ^ k6) & m;
        const uint32_t y0 = (k0 ^ k3) & m, y1 = (k1 ^ k2) & m, y2 = (k4 ^ k7) & m, y3 = (k5 ^ k6) & m;
        const uint32_t z0 = (k0 ^ k4) & m, z1 = (k1 ^ k5) & m, z2 = (k3 ^ k7) & m, z3 = (k2 ^ k6) & m;
        n += __popc(x0) + __popc(x1) + __popc(x2) + __popc(x3);
        n += __popc(y0) + __popc(y1) + __popc(y2) + __popc(y3);
        n += __popc(z0) + __popc(z1) + __popc(z2) + __popc(z3);
        /* three crossed edges of a face: the fourth is crossed too */
        uint32_t w = (x0 & x1 & y0) | (x2 & x3 & y2) | (x0 & x2 & z0) | (x1 & x3 & z2) | (y0 & y2 & z0) | (y1 & y3 & z1);
        w |= ((x0 & y0 & z0) & (x3 & y3 & z3)) | ((x0 & y1 & z1) & (x3 & y2 & z2));
        w |= ((x1 & y1 & z3) & (x2 & y2 & z0)) | ((x1 & y0 & z2) & (x2 & y3 & z1));
        multi[h] = w;
        __builtin_amdgcn_sched_barrier(0);
    }
    uint64_t w = (uint64_t)multi[1] << 32 | multi[0];
    while (w) {
        const uint32_t i = (uint32_t)__ffsll((unsigned long long)w) - 1u;
        w &= w - 1ull;
        n -= fewer[corner_pairs(o, i)];
    }
    return (uint32_t)n;
}

/* Counts of node rows [r0, r1) of a job: one row group of 64 >> cshift rows
 * per wave iteration, one lane per 64-node chunk, no LDS window and no
 * barrier.  Per row: the crossing edges its nodes own and the triangles of
 * cell row (y, z-1); with a.vpc / a.tpc also each chunk's exclusive prefix of
 * both within its row.  POP: triangles by chunk_triangles, else by a lookup per
 * active cell; tab is the table of either (LDS). */
template <int NLEV, bool POP>
__device__ __forceinline__ void count_rows_t(const JobArgs& a, const uint8_t* tab, uint64_t r0, uint64_t r1,
                                             uint64_t wave_first, uint64_t wave_step)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t sub = lane >> a.cshift, cl = lane & ((1u << a.cshift) - 1u);
    const uint32_t G = 64u >> a.cshift, CS = 1u << a.cshift;
    const uint64_t level_words = (uint64_t)a.nz * a.ny * a.NC;
    const bool chunk_prefixes = a.vpc != nullptr;
    RowWalk rw = row_walk(a, r0 + wave_first * G, wave_step * G);
    for (uint64_t g = r0 + wave_first * G; g < r1; g += wave_step * G, row_next(a, rw)) {
        const uint64_t r = g + sub;
        const bool ok = r < r1;
        uint32_t y, z;
        row_at(a, rw, sub, y, z);
        const uint32_t nl = NLEV ? (uint32_t)NLEV : a.nlev;
#pragma unroll
        for (uint32_t l = 0; l < nl; ++l) {
            const uint64_t* lev = a.bitvol + (uint64_t)l * level_words;
            uint32_t vc = 0, tc = 0;
            for (uint32_t c0 = 0; c0 < a.NC; c0 += CS) {
                const uint32_t c = c0 + cl;
                uint32_t cv = 0, ct = 0;
                if (ok && c < a.NC) {
                    RowChunk o;
                    row_chunk(a, lev, y, z, c, o);
                    cv = (uint32_t)(__popcll(o.x) + __popcll(o.y) + __popcll(o.z));
                    if constexpr (POP) {
                        if (o.act) ct = chunk_triangles(o, tab);
                    } else {
                        uint64_t m = o.act;
                        while (m) {
                            const uint32_t i = (uint32_t)__ffsll((unsigned long long)m) - 1u;
                            m &= m - 1ull;
                            ct += tab[corner_pairs(o, i)];
                        }
                    }
                }
                if (chunk_prefixes) {
                    /* both counts in one scan: a chunk holds at most 192
                     * crossing edges and 320 triangles, a group of at most 64
                     * chunks sums below 2^16 in each half */
                    uint32_t s;
                    const uint32_t e = group_excl_scan(cv | ct << 16, cl, CS, s);
                    if (ok && c < a.NC) {
                        const uint64_t w = (uint64_t)l * level_words + r * a.NC + c;
                        /* coalesced stream of prefixes: nontemporal (measured
                         * faster).  Rows of at most 64 chunks are one group,
                         * so the packed scan result is the chunk's in-row
                         * prefix pair */
                        const uint32_t hv = cv ? kHalfBusy : 0u, ht = ct ? kWordBusy : 0u;
                        if (a.NC <= 64) {
                            __builtin_nontemporal_store(e | hv | ht, &a.vpc[w]);
                        } else {
                            __builtin_nontemporal_store((vc + (e & 0xFFFFu)) | hv << 16, &a.vpc[w]);
                            __builtin_nontemporal_store((tc + (e >> 16)) | ht, &a.tpc[w]);
                        }
                    }
                    vc += s & 0xFFFFu;
                    tc += s >> 16;
                } else {
                    vc += cv;
                    tc += ct;
                }
            }
            if (!chunk_prefixes) {
                /* sum over the CS lanes of each row group */
                for (uint32_t d = CS >> 1; d >= 1; d >>= 1) {
                    vc += __shfl_xor(vc, (int)d);
                    tc += __shfl_xor(tc, (int)d);
                }
            }
            if (ok && cl == 0) {
                a.counts[(uint64_t)(l * 2 + 0) * a.nrows + r] = vc;
                a.counts[(uint64_t)(l * 2 + 1) * a.nrows + r] = tc;
            }
        }
    }
}

/* Level count as a compile-time constant where it is small, so that the loads
 * of all levels can be in flight together. */
template <bool POP>
__device__ __forceinline__ void count_rows(const JobArgs& a, const uint8_t* tab, uint64_t r0, uint64_t r1,
                                           uint64_t wave_first, uint64_t wave_step)
{
    switch (a.nlev) {
    case 1:
        /* a plain pass of one level has a kernel of its own (k_count_level) */
        if constexpr (POP) count_rows_t<1, POP>(a, tab, r0, r1, wave_first, wave_step);
        break;
    case 2: count_rows_t<2, POP>(a, tab, r0, r1, wave_first, wave_step); break;
    case 3: count_rows_t<3, POP>(a, tab, r0, r1, wave_first, wave_step); break;
    case 4: count_rows_t<4, POP>(a, tab, r0, r1, wave_first, wave_step); break;
    default: count_rows_t<0, POP>(a, tab, r0, r1, wave_first, wave_step); break;
    }
}

/* Per swap_pairs(cube index) (the index corner_pairs gives) 2 (loops - 1), the
 * cell's crossed edges less its triangles, less 2; without POP its triangles. */
template <bool POP>
__device__ __forceinline__ void stage_counts(uint8_t* tab)
{
    for (uint32_t i = threadIdx.x; i < 256; i += kBlock) {
        const uint32_t c = swap_pairs(i), lo = c & 15u, hi = c >> 4, nt = (uint32_t)(d_tri[c] >> 60);
        const uint32_t edges = __popc(lo ^ ((lo >> 1) | (lo & 1u) << 3)) + __popc(hi ^ ((hi >> 1) | (hi & 1u) << 3)) +
                               __popc(lo ^ hi);
        tab[i] = (uint8_t)(!POP ? nt : (edges ? edges - nt - 2u : 0u));
    }
    __syncthreads();
}

/* Row groups of 64 >> cshift rows as the units. */
template <bool POP, int NLEV>
__device__ __forceinline__ void count_job(const JobArgs& a, uint8_t* tab)
{
    stage_counts<POP>(tab);
    const uint64_t G = 64u >> a.cshift, groups = (a.nrows + G - 1) / G;
    const Span sp = grid_span(0, groups, kWaves, uniform(threadIdx.x >> 6));
    const uint64_t r1 = sp.end * G < a.nrows ? sp.end * G : a.nrows;
    if constexpr (NLEV == 1) count_rows_t<1, POP>(a, tab, sp.lo * G, r1, sp.first - sp.lo, sp.step);
    else count_rows<POP>(a, tab, sp.lo * G, r1, sp.first - sp.lo, sp.step);
}

/* One level: 74 VGPRs, six waves per SIMD without a spill. */
__global__ __launch_bounds__(kBlock) void k_count_level(JobArgs a)
{
    __shared__ uint8_t tab[256];
    count_job<true, 1>(a, tab);
}

/* Several levels, all their loads in flight: seven waves per SIMD (at most 72
 * VGPRs).  With chunk_triangles and four waves, mostly empty chunks, whose time is
 * load latency, lose more than full ones gain (1024^3 at three levels: 357 -> 390
 * us with smooth fields, 432 -> 413 with rough ones). */
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(7))) void k_count(JobArgs a)
{
    __shared__ uint8_t tab[256];
    count_job<false, 0>(a, tab);
}

/* Count pass of a batch: a job's workgroups walk its row groups in steps of them
 * all. */
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(5))) void k_count_batch(const JobArgs* jobs,
                                                                                              const BlockRef* refs)
{
    const BlockRef ref = refs[blockIdx.x];
    const JobArgs& a = jobs[ref.job];
    const uint64_t wave = (uint64_t)ref.block * kWaves;
    __shared__ uint8_t tab[256];
    stage_counts<true>(tab);
    count_rows<true>(a, tab, 0, a.nrows, wave + uniform(threadIdx.x >> 6), (uint64_t)ref.blocks * kWaves);
}

/* ------------------------------------------------------------------------- */
/* tile-team emit pass                                                         */
/* ------------------------------------------------------------------------- */

/* One unit: level l of band b over steps zs .. ze-1 (with VertexNormal one
 * more step after the last node slice).  Tile z emits the triangles of cell
 * slice z-1 and the vertices of node slice z, or of node slice z-1 with
 * VertexNormal: their normals sum face normals of cell slices z-2 and z-1,
 * both then in the face-normal ring (a first unit step without output fills
 * in z-2).  The mask ring holds node slices z-1 .. z+1 and takes one new
 * slice per step. */
template <typename T, int M>
__device__ void emit_unit(const JobArgs& a, const Team& v, uint64_t unit)
{
    const T* vol = (const T*)a.values;
    const uint64_t per_level = (uint64_t)a.nb * a.nslabs;
    const uint32_t l = (uint32_t)(unit / per_level);
    const uint64_t rem = unit - (uint64_t)l * per_level;
    const uint32_t slab = (uint32_t)(rem / a.nb);
    const uint32_t band = (uint32_t)(rem - (uint64_t)slab * a.nb);
    const int y0 = (int)(band * a.R);
    const int zs = (int)(slab * a.slab);
    const int ze = min(zs + (int)a.slab, (int)a.nz);
    constexpr bool vn = M == kModeVertex;
    const int zend = (vn && ze == (int)a.nz) ? ze + 1 : ze;
    const uint32_t ws_v = vn ? 0u : 1u;
    const Level L = level_of(a, l);

    /* VertexNormal first prepares cell slice zs-2 (node slices zs-2, zs-1) */
    load_slices<M>(a, v, L, vn ? zs - 2 : zs - 1, vn ? zs : zs + 1, y0);
    uint32_t ovf = 0;   // bit cs: the face normals of cell slot cs did not fit
    wave_sync();
    if (vn && zs >= 2) {
        const TileTotals t = tile_prefixes<M>(a, v, zs - 1, y0, ws_v, false, true);
        const bool keep = t.nt <= v.fn_cap;
        ovf = keep ? 0u : (1u << cslot<M>(zs - 2));
        Bases B;
        B.v[0] = B.v[1] = B.v[2] = B.v[3] = 0;
        B.t = 0;
        emit_tile<T, M>(a, v, L, B, vol, zs - 1, y0, ws_v, false, false, t, keep, false);
        wave_sync();
    }
    for (int z = zs; z < zend; ++z) {
        if (vn || z > zs) load_slices<M>(a, v, L, z + 1, z + 1, y0);
        const Bases B = tile_bases(a, L, z, y0);
        wave_sync();
        const TileTotals t = tile_prefixes<M>(a, v, z, y0, ws_v, true, z == zs);
        bool keep = false;
        if (vn) {
            const uint32_t bit = 1u << cslot<M>(z - 1);
            keep = t.nt <= v.fn_cap;
            ovf = keep ? (ovf & ~bit) : (ovf | bit);
        }
        emit_tile<T, M>(a, v, L, B, vol, z, y0, ws_v, true, true, t, keep, ovf == 0);
        wave_sync();   // the next step overwrites a mask slot and the cell data
    }
}

/* Persistent workgroups of `teams` one-wave teams (the other waves only help
 * stage the table): team w of workgroup g takes units g * teams + w, then
 * strides by all teams of the grid; neighbouring teams take neighbouring
 * bands of the same slab and level. */
template <typename T, int M>
__global__ __launch_bounds__(kEmitBlock) void k_emit(JobArgs a)
{
    extern __shared__ __align__(16) uint8_t smem[];
    stage_table(smem);
    const uint32_t wave = uniform(threadIdx.x >> 6);
    if (wave >= a.teams) return;
    const Team v = make_team(a, smem, wave);
    const uint64_t step = (uint64_t)gridDim.x * a.teams;
    for (uint64_t u = (uint64_t)blockIdx.x * a.teams + wave; u < a.nunits; u += step) emit_unit<T, M>(a, v, u);
}

/* Emit pass of a batch of jobs sharing the value type T and the mode: the
 * units of all jobs in one sequence, taken by persistent teams.  Every job of
 * the launch has the same team_stride. */
template <typename T, int M>
__global__ __launch_bounds__(kEmitBlock) void k_emit_batch(const JobArgs* jobs, const uint64_t* unit_start, uint32_t njobs,
                                                            uint32_t teams)
{
    extern __shared__ __align__(16) uint8_t smem[];
    stage_table(smem);
    const uint32_t wave = uniform(threadIdx.x >> 6);
    if (wave >= teams) return;
    const uint64_t total = unit_start[njobs];
    const uint64_t step = (uint64_t)gridDim.x * teams;
    for (uint64_t g = (uint64_t)blockIdx.x * teams + wave; g < total; g += step) {
        const uint32_t j = uniform(find_job(unit_start, njobs, g));
        const JobArgs& a = jobs[j];
        const Team v = make_team(a, smem, wave);
        emit_unit<T, M>(a, v, g - unit_start[j]);
    }
}

__device__ __forceinline__ void stage_table_block(uint64_t* tri)
{
    for (uint32_t i = threadIdx.x; i < 256; i += kBlock) tri[i] = d_tri[i];
    __syncthreads();
}

/* ------------------------------------------------------------------------- */
/* SlicePlane: classification by a plane, emit with per-vertex colours         */
/* ------------------------------------------------------------------------- */

/* The plane's value at (x, y, z) as SlicePlane::substitute_plane_equation
 * evaluates it (SlicePlane.cpp:936-971): c0*x + c1*y + c2*z + c3, left to right
 * in float, node indices converted to float. */
__device__ __forceinline__ float plane_at(const float c[4], float x, float y, float z)
{
    float s = c[0] * x;
    s = s + c[1] * y;
    s = s + c[2] * z;
    return s + c[3];
}

/* Bit i of chunk c of row (y, z): plane(64c+i, y, z) > 0.0f
 * (calculate_table_index, SlicePlane.cpp:802-818).  Nothing is read: one node
 * row per wave, one ballot per 64 nodes, the masks of up to 64 chunks parked
 * in lanes and stored together. */
__global__ __launch_bounds__(kBlock) void k_classify_plane(JobArgs a)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t nrows = (uint64_t)a.ny * a.nz;
    const uint64_t wave_id = (uint64_t)blockIdx.x * kWaves + uniform(threadIdx.x >> 6);   // uniform: scalar
    const uint64_t nwaves = ((uint64_t)gridDim.x * kBlock) >> 6;
    for (uint64_t row = wave_id; row < nrows; row += nwaves) {
        const uint64_t z = row / a.ny, y = row - z * a.ny;
        const float fy = (float)y, fz = (float)z;
        for (uint32_t c0 = 0; c0 < a.NC; c0 += 64) {
            const uint32_t cend = (a.NC - c0) < 64u ? (a.NC - c0) : 64u;
            uint64_t mine = 0;
            for (uint32_t i = 0; i < cend; ++i) {
                const uint32_t x = (c0 + i) * 64u + lane;
                const uint64_t m = __ballot(x < a.nx && plane_at(a.plane, (float)x, fy, fz) > 0.0f);
                mine = lane == i ? m : mine;
            }
            if (lane < cend) a.bitvol[row * a.NC + c0 + lane] = mine;
        }
    }
}

/* interpolate_value<T> (SlicePlane.cpp:1001-1026): the value at ratio r along
 * the edge, computed in the types C++ gives values[i0] + r * (values[i1] -
 * values[i0]) for T (integer promotion and unsigned wrap-around of the
 * difference, a float product, double only for double data). */
template <typename T>
__device__ __forceinline__ double slice_value(T va, T vb, float r)
{
    return va + r * (vb - va);
}

/* Math::Round (Utility/Math.h:110-114): half away from zero, in double. */
__device__ __forceinline__ int round_half_away(float a) { return a >= 0 ? (int)(a + 0.5) : -(int)(0.5 - a); }

__device__ __forceinline__ float clampf(float a, float lo, float hi) { return a <= lo ? lo : (a <= hi ? a : hi); }

/* Colour-map entry s in [0,1] floats: from the device table (3 bytes an entry) or
 * from a copy in LDS, divided once per workgroup instead of six times a corner. */
struct GlobalColors {
    const uint8_t* t;
    __device__ __forceinline__ void operator()(uint32_t s, float c[3]) const
    {
#pragma unroll
        for (int k = 0; k < 3; ++k) c[k] = (float)t[3 * s + k] / 255.0f;
    }
};
struct LdsColors {
    const float* t;
    __device__ __forceinline__ void operator()(uint32_t s, float c[3]) const
    {
#pragma unroll
        for (int k = 0; k < 3; ++k) c[k] = t[3 * s + k];
    }
};

/* ColorMap::at (ColorMap.cpp:1043-1054): the two table entries around the
 * value, mixed by RGBColor::Mix (RGBColor.cpp:23-31) in [0,1] floats,
 * x*(1-t) + y*t, and rounded back to bytes.  A NaN position (an empty range)
 * takes the first entry. */
template <typename C>
__device__ __forceinline__ void color_at(const JobArgs& a, const C& tab, float value, uint8_t rgb[3])
{
    const float lo = a.crange[0], hi = a.crange[1];
    const float v0 = clampf(value, lo, hi);
    const float rr = (float)(a.cres - 1);
    float v = (v0 - lo) / (hi - lo) * rr;
    if (!(v >= 0.0f)) v = 0.0f;
    const uint32_t s0 = (uint32_t)v;
    const uint32_t s1 = (s0 + 1 < a.cres - 1) ? s0 + 1 : a.cres - 1;
    const float t = v - (float)s0;
    float c0[3], c1[3];
    tab(s0, c0);
    tab(s1, c1);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float p = c0[k] * (1 - t);
        const float q = c1[k] * t;
        rgb[k] = (uint8_t)round_half_away(clampf(p + q, 0.0f, 1.0f) * 255.0f);
    }
}

/* One triangle of extract_plane<T> (SlicePlane.cpp:165-280): per edge in the
 * order (T[i], T[i+2], T[i+1]) its plane crossing in table orientation
 * (interpolate_vertex :981-990, float), (p + min) * scale, and the colour of
 * the value interpolated at the same ratio; the normal is
 * -(v2 - v0) x (v1 - v0). */
template <typename T, typename C, typename Sink>
__device__ __forceinline__ void slice_triangle_values(const JobArgs& a, const uint64_t* tri, uint64_t rec, uint32_t ci,
                                                      const C& colors, Sink& out)
{
    const T* vol = (const T*)a.values;
    const uint32_t x = (uint32_t)(rec & 0xFFFFFu), y = (uint32_t)((rec >> 20) & 0xFFFFFu);
    const uint32_t zc = (uint32_t)((rec >> 40) & 0xFFFFFu), t = (uint32_t)(rec >> 60);
    const uint64_t w = tri[ci];
    const uint32_t eds[3] = { (uint32_t)((w >> (12 * t)) & 0xF), (uint32_t)((w >> (12 * t + 8)) & 0xF),
                              (uint32_t)((w >> (12 * t + 4)) & 0xF) };
    const uint64_t line = a.nx, slice = (uint64_t)a.nx * a.ny;
    /* the six values in flight before any arithmetic */
    const T* cell = vol + x + y * line + zc * slice;
    T va[3], vb[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const uint32_t qq = edge_ends(eds[j]);
        va[j] = cell[(qq & 1u) + (qq & 2u ? line : 0) + (qq & 4u ? slice : 0)];
        vb[j] = cell[((qq >> 4) & 1u) + (qq & 32u ? line : 0) + (qq & 64u ? slice : 0)];
    }
    float p[3][3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const uint32_t qq = edge_ends(eds[j]);
        const uint32_t ax = x + (qq & 1u), ay = y + ((qq >> 1) & 1u), az = zc + ((qq >> 2) & 1u);
        const uint32_t bx = x + ((qq >> 4) & 1u), by = y + ((qq >> 5) & 1u), bz = zc + ((qq >> 6) & 1u);
        const float fa[3] = { (float)ax, (float)ay, (float)az };
        const float fb[3] = { (float)bx, (float)by, (float)bz };
        const float f0 = plane_at(a.plane, fa[0], fa[1], fa[2]);
        const float f1 = plane_at(a.plane, fb[0], fb[1], fb[2]);
        float r = f0 / (f1 - f0);
        r = r < 0 ? -r : r;
        const float s = 1.0f - r;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float u = s * fa[k];
            const float v = r * fb[k];
            const float q = (u + v) + a.minc[k];
            p[j][k] = q * a.sc[k];
        }
        uint8_t rgb[3];
        color_at(a, colors, (float)slice_value<T>(va[j], vb[j], r), rgb);
        out.vertex(j, p[j], rgb);
    }
    const float d1x = p[2][0] - p[0][0], d1y = p[2][1] - p[0][1], d1z = p[2][2] - p[0][2];
    const float d2x = p[1][0] - p[0][0], d2y = p[1][1] - p[0][1], d2z = p[1][2] - p[0][2];
    const float nn[3] = { -(d1y * d2z - d1z * d2y), -(d1z * d2x - d1x * d2z), -(d1x * d2y - d1y * d2x) };
    out.normal(nn);
}

/* Where a triangle's corners (coordinates, colour) and normal go: arrays of
 * 9, 9 and 3 elements a triangle, from element 0 of triangle 0. */
template <typename F, typename B>
struct SliceSink {
    F* co;
    F* no;
    B* cl;
    __device__ __forceinline__ void vertex(int j, const float p[3], const uint8_t rgb[3])
    {
        co[3 * j + 0] = p[0];
        co[3 * j + 1] = p[1];
        co[3 * j + 2] = p[2];
        cl[3 * j + 0] = rgb[0];
        cl[3 * j + 1] = rgb[1];
        cl[3 * j + 2] = rgb[2];
    }
    __device__ __forceinline__ void normal(const float n[3])
    {
        no[0] = n[0];
        no[1] = n[1];
        no[2] = n[2];
    }
};

/* Triangle `id` of the output, written by its own thread. */
template <typename T>
__device__ __forceinline__ void slice_triangle(const JobArgs& a, const uint64_t* tri, uint64_t id, uint64_t rec,
                                               uint32_t ci)
{
    SliceSink<float, uint8_t> out{ a.coords[0] + 9 * id, a.normals[0] + 3 * id, a.colors + 9 * id };
    slice_triangle_values<T>(a, tri, rec, ci, GlobalColors{ a.ctable }, out);
}

/* Triangles of the planes the thresholds do not serve, from their chunk masks
 * (slice_triangle's table indexed as corner_pairs gives the case). */
template <typename T>
__global__ __launch_bounds__(kBlock) void k_slice_triangles(JobArgs a)
{
    struct SliceLds {
        ListLds l;
        uint64_t m[4][kChunks];      // k0, k3, k4, k7 of each chunk
        uint64_t key[kChunks];       // 64 c | y << 20 | z << 40 of each chunk's first cell
        uint32_t next[kChunks];
    };
    __shared__ uint64_t tri[256];
    __shared__ SliceLds lds[kWaves];
    for (uint32_t i = threadIdx.x; i < 256; i += kBlock) tri[i] = d_tri[swap_pairs(i)];
    __syncthreads();
    SliceLds& s = lds[threadIdx.x >> 6];
    const uint32_t lane = threadIdx.x & 63u;
    const EmitLevel L = emit_level(a, 0, blockIdx.x);
    busy_chunks<false, kChunks>(a, L, s.l.q, [&](uint32_t n) {
        list_triangles(a, L, tri, s.l, n, [&](uint64_t, uint32_t y, uint32_t z, uint32_t c, uint64_t) {
            const CellMasks o = load_cells(a, L, y, z, c);
            s.m[0][lane] = o.k0;
            s.m[1][lane] = o.k3;
            s.m[2][lane] = o.k4;
            s.m[3][lane] = o.k7;
            s.next[lane] = o.next;
            s.key[lane] = (uint64_t)(c * 64u) | (uint64_t)y << 20 | (uint64_t)(z - 1) << 40;
            return o.act;
        }, [&](uint32_t q, uint32_t i) { return corner_pairs_at(s.m, s.next, q, i); },
        [](uint32_t, uint32_t, uint32_t, uint32_t) {}, [&](uint32_t cnt, uint32_t rank) {
            for (uint32_t j = lane; j < cnt; j += 64) {
                const uint32_t e = s.l.tl[j], cell = s.l.cell[e & 63u], q = cell & 63u;
                const uint64_t rec = (s.key[q] + ((cell >> 6) & 63u)) | (uint64_t)(e >> 6) << 60;
                slice_triangle<T>(a, tri, s.l.out[q] + (rank + j), rec, cell >> 12);
            }
        });
    });
}

/* SlicePlane without classifying every node.  Along a node row (y, z) the
 * plane value plane_at(c, x, y, z) is monotone in x -- each float operation
 * is monotone in its operand, rounding included -- so the nodes above the
 * plane are x >= t (c0 > 0; c0 == 0 with t = 0 or nx) or x < t (c0 < 0) for
 * one threshold t per node row, found by bisection on the same float
 * expression.  A cell row's active cells are then the one run
 * [min t - 1, max t - 1] over its four node rows, cut by the points t - 1
 * and t of each row into at most nine runs of one cube index.  Counts per
 * cell row, a scan, then one thread per triangle.  The host takes this path
 * when the plane is finite at the volume's eight corners (and so, being
 * monotone in each coordinate, everywhere inside). */
__device__ __forceinline__ bool above_thr(int dir, int32_t t, int32_t x) { return dir < 0 ? x < t : x >= t; }

__global__ __launch_bounds__(kBlock) void k_slice_thresholds(JobArgs a, int32_t* thr)
{
    const int dir = a.plane[0] > 0.0f ? 1 : (a.plane[0] < 0.0f ? -1 : 0);
    const uint64_t nrows = (uint64_t)a.ny * a.nz, step = (uint64_t)gridDim.x * kBlock;
    for (uint64_t row = (uint64_t)blockIdx.x * kBlock + threadIdx.x; row < nrows; row += step) {
        const uint32_t z = (uint32_t)(row / a.ny), y = (uint32_t)(row - (uint64_t)z * a.ny);
        const float fy = (float)y, fz = (float)z;
        int32_t t;
        if (dir == 0) {
            t = plane_at(a.plane, 0.0f, fy, fz) > 0.0f ? 0 : (int32_t)a.nx;
        } else {
            /* the first x whose node is above (c0 > 0) or not above (c0 < 0) */
            uint32_t lo = 0, hi = a.nx;
            while (lo < hi) {
                const uint32_t mid = (lo + hi) >> 1;
                const bool up = plane_at(a.plane, (float)mid, fy, fz) > 0.0f;
                if (up == (dir > 0)) hi = mid; else lo = mid + 1;
            }
            t = (int32_t)lo;
        }
        thr[row] = t;
    }
}

/* The active cells of cell row (y, z) as nine runs [b[i], b[i + 1]) of one
 * cube index each (ci(i)): the breakpoints t - 1 and t of the four node rows,
 * clamped to [lo, hi + 1] and sorted, so that coinciding or outside points
 * give empty runs.  Every index is static, so the runs stay in registers. */
struct SliceRuns {
    int32_t b[10];
    int32_t t[4];   // thresholds of node rows (y,z), (y+1,z), (y,z+1), (y+1,z+1)
    int dir;
    __device__ __forceinline__ uint32_t ci(int i) const;
};

__device__ __forceinline__ uint32_t slice_cube_index(int dir, const int32_t t[4], int32_t x)
{
    /* corners 0..7: (x,y,z) (x+1,y,z) (x+1,y+1,z) (x,y+1,z) and the same at z+1;
     * t: node rows (y,z), (y+1,z), (y,z+1), (y+1,z+1) */
    return (uint32_t)above_thr(dir, t[0], x) | (uint32_t)above_thr(dir, t[0], x + 1) << 1 |
           (uint32_t)above_thr(dir, t[1], x + 1) << 2 | (uint32_t)above_thr(dir, t[1], x) << 3 |
           (uint32_t)above_thr(dir, t[2], x) << 4 | (uint32_t)above_thr(dir, t[2], x + 1) << 5 |
           (uint32_t)above_thr(dir, t[3], x + 1) << 6 | (uint32_t)above_thr(dir, t[3], x) << 7;
}

__device__ __forceinline__ uint32_t SliceRuns::ci(int i) const { return slice_cube_index(dir, t, b[i]); }

__device__ __forceinline__ void order2(int32_t& p, int32_t& q)
{
    const int32_t lo = p < q ? p : q, hi = p < q ? q : p;
    p = lo;
    q = hi;
}

/* Returns false when the cell row has no active cell. */
__device__ __forceinline__ bool slice_runs(const JobArgs& a, const int32_t* thr, uint32_t y, uint32_t z, SliceRuns& r)
{
    r.dir = a.plane[0] < 0.0f ? -1 : 1;
    const uint64_t r0 = (uint64_t)z * a.ny + y;
    int32_t* t = r.t;
    t[0] = thr[r0];
    t[1] = thr[r0 + 1];
    t[2] = thr[r0 + a.ny];
    t[3] = thr[r0 + a.ny + 1];
    const int32_t tmin = min(min(t[0], t[1]), min(t[2], t[3]));
    const int32_t tmax = max(max(t[0], t[1]), max(t[2], t[3]));
    const int32_t lo = max(tmin - 1, 0), hi = min(tmax - 1, (int32_t)a.nx - 2);
    if (lo > hi) return false;
    int32_t* b = r.b;
    b[0] = lo;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        b[1 + 2 * k] = min(max(t[k] - 1, lo), hi + 1);
        b[2 + 2 * k] = min(max(t[k], lo), hi + 1);
    }
    b[9] = hi + 1;
    /* sorting network of b[1..8] (19 comparators) */
    order2(b[1], b[3]); order2(b[2], b[4]); order2(b[5], b[7]); order2(b[6], b[8]);
    order2(b[1], b[5]); order2(b[2], b[6]); order2(b[3], b[7]); order2(b[4], b[8]);
    order2(b[1], b[2]); order2(b[3], b[4]); order2(b[5], b[6]); order2(b[7], b[8]);
    order2(b[3], b[5]); order2(b[4], b[6]);
    order2(b[2], b[5]); order2(b[4], b[7]);
    order2(b[2], b[3]); order2(b[4], b[5]); order2(b[6], b[7]);
    return true;
}

__global__ __launch_bounds__(kBlock) void k_slice_row_counts(JobArgs a, const int32_t* thr, uint32_t* counts)
{
    __shared__ uint8_t ntri[256];
    for (uint32_t i = threadIdx.x; i < 256; i += kBlock) ntri[i] = (uint8_t)(d_tri[i] >> 60);
    __syncthreads();
    const uint64_t ncr = (uint64_t)(a.ny - 1) * (a.nz - 1), step = (uint64_t)gridDim.x * kBlock;
    for (uint64_t cr = (uint64_t)blockIdx.x * kBlock + threadIdx.x; cr < ncr; cr += step) {
        const uint32_t z = (uint32_t)(cr / (a.ny - 1)), y = (uint32_t)(cr - (uint64_t)z * (a.ny - 1));
        SliceRuns r;
        uint32_t c = 0;
        if (slice_runs(a, thr, y, z, r)) {
#pragma unroll
            for (int i = 0; i < 9; ++i) c += (uint32_t)(r.b[i + 1] - r.b[i]) * ntri[r.ci(i)];
        }
        counts[cr] = c;
    }
}

/* The cell rows of the first and the last triangle of every unit of 64
 * triangles (unit u: triangles 64u .. min(64u + 63, n - 1)), written by the
 * rows that hold them: one writer each. */
__global__ __launch_bounds__(kBlock) void k_slice_unit_rows(uint64_t ncr, const uint32_t* counts, const uint64_t* prefix,
                                                           uint64_t n, uint64_t* first, uint64_t* last)
{
    const uint64_t step = (uint64_t)gridDim.x * kBlock;
    for (uint64_t cr = (uint64_t)blockIdx.x * kBlock + threadIdx.x; cr < ncr; cr += step) {
        const uint32_t c = counts[cr];
        if (!c) continue;
        const uint64_t p = prefix[cr], e = p + c;   // the row's triangles [p, e)
        for (uint64_t u = p >> 6; (u << 6) < e; ++u) {
            const uint64_t f = u << 6, l = f + 63 < n ? f + 63 : n - 1;
            if (f >= p) first[u] = cr;
            if (l >= p && l < e) last[u] = cr;
        }
    }
}

/* Colour maps of up to this many entries are staged in LDS by the run emit. */
constexpr uint32_t kSliceLdsColors = 1024;

/* One thread per triangle.  A wave's 64 triangles lie in the cell rows
 * between those of its first and last (k_slice_unit_rows); each lane bisects
 * that short range (of at most 64 rows in registers, one row a lane), then walks
 * its row's runs to its cell and table index.  Instruction issue bounds it:
 * divisions are kept out of the runs, the rows and the colours (640 x 704 x 768
 * float: 66 us with them, 54.6 without).
 * The wave's 64 triangles are consecutive in the output: their coordinates,
 * normals and colours are assembled in LDS and written as whole 16-byte
 * words. */
template <typename T, bool kLdsColors>
__global__ __launch_bounds__(kBlock) void k_slice_triangles_runs(JobArgs a, const int32_t* thr, const uint64_t* prefix,
                                                                const uint64_t* unit_first, const uint64_t* unit_last)
{
    __shared__ uint64_t tri[256];
    __shared__ __align__(16) float stage[kWaves][9 * 64 + 3 * 64 + 9 * 64 / 4];   // coords, normals, colours
    extern __shared__ __align__(16) uint8_t smem[];
    float* ctab = (float*)smem;
    if (kLdsColors)
        for (uint32_t i = threadIdx.x; i < a.cres; i += kBlock) GlobalColors{ a.ctable }(i, ctab + 3 * i);
    stage_table_block(tri);
    const uint64_t n = a.toff[1];
    const uint32_t lane = threadIdx.x & 63u;
    float* sc = stage[threadIdx.x >> 6];
    float* sn = sc + 9 * 64;
    uint8_t* scl = (uint8_t*)(sn + 3 * 64);
    const Span sp = grid_span(0, n, kBlock, threadIdx.x);
    for (uint64_t gw = sp.first - lane; gw < n; gw += sp.step) {   // wave-uniform
        const uint64_t lo = uniform64(unit_first[gw >> 6]), hi = uniform64(unit_last[gw >> 6]);
        const uint64_t g = gw + lane;
        const uint32_t cells = a.ny - 1;   // cell rows of a slice
        uint32_t y, z, k;                  // the lane's cell row, its triangle in it
        if (hi - lo < 64) {
            /* where each row's triangles start, from gw: only the first row's may lie before */
            const int32_t start = lo + lane <= hi ? (int32_t)(prefix[lo + lane] - gw) : INT32_MAX;
            uint32_t row = 0;
#pragma unroll
            for (uint32_t d = 32; d >= 1; d >>= 1)
                if (__shfl(start, (int)(row + d)) <= (int32_t)lane) row += d;
            k = lane - (uint32_t)__shfl(start, (int)row);
            z = lo >> 32 ? (uint32_t)(lo / cells) : (uint32_t)lo / cells;
            y = (uint32_t)(lo - (uint64_t)z * cells) + row;
            if (y >= cells) {
                /* row < 64: one wrap where a slice has as many rows */
                const uint32_t over = cells >= 64u ? 1u : y / cells;
                y -= over * cells;
                z += over;
            }
        } else {
            uint64_t l = lo, h = hi;
            while (l < h) {
                const uint64_t mid = (l + h + 1) >> 1;
                if (prefix[mid] <= g) l = mid; else h = mid - 1;
            }
            z = (uint32_t)(l / cells);
            y = (uint32_t)(l - (uint64_t)z * cells);
            k = (uint32_t)(g - prefix[l]);
        }
        if (g < n) {
            SliceRuns r;
            slice_runs(a, thr, y, z, r);   // the row has triangles, so active cells
            uint32_t x = 0, ci = 0, per = 1;
            bool found = false;
#pragma unroll
            for (int i = 0; i < 9; ++i) {
                const uint32_t ci_i = r.ci(i);
                const uint32_t nt = (uint32_t)(tri[ci_i] >> 60);
                const uint32_t m = (uint32_t)(r.b[i + 1] - r.b[i]) * nt;
                if (!found) {
                    if (k < m) {
                        x = (uint32_t)r.b[i];
                        per = nt;
                        ci = ci_i;
                        found = true;
                    } else {
                        k -= m;
                    }
                }
            }
            const uint32_t t = k % per;
            x += k / per;
            const uint64_t rec = (uint64_t)x | (uint64_t)y << 20 | (uint64_t)z << 40 | (uint64_t)t << 60;
            SliceSink<float, uint8_t> out{ sc + 9 * lane, sn + 3 * lane, scl + 9 * lane };
            if (kLdsColors)
                slice_triangle_values<T>(a, tri, rec, ci, LdsColors{ ctab }, out);
            else
                slice_triangle_values<T>(a, tri, rec, ci, GlobalColors{ a.ctable }, out);
        }
        wave_sync();
        /* the wave's output: triangles gw .. gw + cnt - 1 (9 * gw floats and
         * bytes from the array starts: 16-byte aligned when cnt is 64) */
        const uint32_t cnt = n - gw < 64 ? (uint32_t)(n - gw) : 64u;
        float* co = a.coords[0] + 9 * gw;
        float* no = a.normals[0] + 3 * gw;
        uint8_t* cl = a.colors + 9 * gw;
        if (cnt == 64) {
            for (uint32_t i = lane; i < 9 * 64 / 4; i += 64) ((float4*)co)[i] = ((const float4*)sc)[i];
            if (lane < 3 * 64 / 4) ((float4*)no)[lane] = ((const float4*)sn)[lane];
            if (lane < 9 * 64 / 16) ((uint4*)cl)[lane] = ((const uint4*)scl)[lane];
        } else {
            for (uint32_t i = lane; i < 9 * cnt; i += 64) co[i] = sc[i];
            for (uint32_t i = lane; i < 3 * cnt; i += 64) no[i] = sn[i];
            for (uint32_t i = lane; i < 9 * cnt; i += 64) cl[i] = scl[i];
        }
        wave_sync();
    }
}

/* ------------------------------------------------------------------------- */
/* row-count scan                                                              */
/* ------------------------------------------------------------------------- */

constexpr uint32_t kScanPer = 16;                      // elements per thread
constexpr uint32_t kScanTile = kScanPer * kBlock;      // elements per block

/* Four counts in one load; an array's base is aligned to one count only. */
struct __attribute__((packed, aligned(4))) Count4 {
    uint32_t x, y, z, w;
};

/* Sum of each kScanTile segment of each of the narr count arrays; a whole segment's
 * loads are in flight at once (one at a time, 256^3: 6.7 us, so 3.0). */
__global__ __launch_bounds__(kBlock) void k_scan_partials(const uint32_t* counts, uint64_t n, uint32_t nseg, uint64_t* partials)
{
    __shared__ uint64_t sh[kWaves];
    const uint32_t arr = blockIdx.x / nseg, seg = blockIdx.x - arr * nseg;
    const uint32_t* src = counts + (uint64_t)arr * n;
    const uint64_t b = (uint64_t)seg * kScanTile;
    uint64_t s = 0;
    if (b + kScanTile <= n) {
        Count4 v[kScanPer / 4];
#pragma unroll
        for (uint32_t i = 0; i < kScanPer / 4; ++i) v[i] = ((const Count4*)(src + b))[i * kBlock + threadIdx.x];
#pragma unroll
        for (uint32_t i = 0; i < kScanPer / 4; ++i) s += ((uint64_t)v[i].x + v[i].y) + ((uint64_t)v[i].z + v[i].w);
    } else {
        for (uint64_t g = b + threadIdx.x; g < n; g += kBlock) s += src[g];
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) s += (uint64_t)__shfl_xor((unsigned long long)s, d);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t t = 0;
        for (int w = 0; w < kWaves; ++w) t += sh[w];
        partials[blockIdx.x] = t;
    }
}

/* In place: partials of each array become their exclusive prefix, and the
 * grand total of array arr goes to totals[arr].  One workgroup. */
__global__ __launch_bounds__(kBlock) void k_scan_mid(uint64_t* partials, uint32_t nseg, uint32_t narr, uint64_t* totals)
{
    __shared__ uint64_t sh[kWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (uint32_t arr = 0; arr < narr; ++arr) {
        uint64_t* p = partials + (uint64_t)arr * nseg;
        uint64_t carry = 0;
        for (uint32_t b0 = 0; b0 < nseg; b0 += kScanTile) {
            const uint32_t b = b0 + threadIdx.x * kScanPer;
            uint64_t vals[kScanPer];
            uint64_t s = 0;
#pragma unroll
            for (uint32_t i = 0; i < kScanPer; ++i) {
                vals[i] = b + i < nseg ? p[b + i] : 0ull;
                s += vals[i];
            }
            uint64_t incl = s;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const uint64_t t = (uint64_t)__shfl_up((unsigned long long)incl, d);
                if (lane >= d) incl += t;
            }
            if (lane == 63) sh[wave] = incl;
            __syncthreads();
            uint64_t run = carry;
            uint64_t all = 0;
            for (int w = 0; w < kWaves; ++w) {
                if (w < wave) run += sh[w];
                all += sh[w];
            }
            run += incl - s;
#pragma unroll
            for (uint32_t i = 0; i < kScanPer; ++i) {
                if (b + i < nseg) p[b + i] = run;
                run += vals[i];
            }
            carry += all;
            __syncthreads();
        }
        if (threadIdx.x == 0) totals[arr] = carry;
    }
}

/* Two prefixes in one store, likewise. */
struct __attribute__((packed, aligned(8))) Prefix2 {
    uint64_t x, y;
};

/* Sum over the block's threads (the same in every thread). */
__device__ __forceinline__ uint64_t block_sum(uint64_t s, uint64_t* sh)
{
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) s += (uint64_t)__shfl_xor((unsigned long long)s, d);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    uint64_t t = 0;
    for (int w = 0; w < kWaves; ++w) t += sh[w];
    __syncthreads();
    return t;
}

/* Exclusive prefix of each count array.  Where a workgroup's segment starts:
 * kScanCounts sums all counts before it (few segments: the whole scan is this
 * one kernel), kScanPartials the segments' sums before it, kScanScanned reads
 * the scanned sum (so many segments that summing them per workgroup would
 * cost more than a kernel).  Launches are what a small scan costs: 65536
 * counts took 15 us in three kernels, 8 in two. */
enum : int { kScanCounts = 0, kScanPartials = 1, kScanScanned = 2 };

template <int kFrom>
__global__ __launch_bounds__(kBlock) void k_scan_apply(const uint32_t* counts, uint64_t n, uint32_t nseg,
                                                       const uint64_t* partials, uint64_t* prefix, uint64_t* totals)
{
    __shared__ uint64_t sh[kWaves];
    const uint32_t arr = blockIdx.x / nseg, seg = blockIdx.x - arr * nseg;
    const uint32_t* src = counts + (uint64_t)arr * n;
    uint64_t* dst = prefix + (uint64_t)arr * n;
    uint64_t base = 0;
    if constexpr (kFrom == kScanCounts) {
        /* four segments' loads in flight: the sum waits for memory once per four */
        uint64_t before = 0;
        for (uint32_t s0 = 0; s0 < seg; s0 += 4) {
            Count4 v[4][4];
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
#pragma unroll
                for (uint32_t i = 0; i < 4; ++i)
                    v[j][i] = s0 + j < seg ? ((const Count4*)(src + (s0 + j) * kScanTile))[i * kBlock + threadIdx.x] : Count4{};
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
#pragma unroll
                for (uint32_t i = 0; i < 4; ++i) before += ((uint64_t)v[j][i].x + v[j][i].y) + ((uint64_t)v[j][i].z + v[j][i].w);
        }
        base = block_sum(before, sh);
    } else if constexpr (kFrom == kScanPartials) {
        uint64_t before = 0;
        for (uint32_t i = threadIdx.x; i < seg; i += kBlock) before += partials[(uint64_t)arr * nseg + i];
        base = block_sum(before, sh);
    } else {
        base = partials[blockIdx.x];
    }
    const uint64_t b = (uint64_t)seg * kScanTile + (uint64_t)threadIdx.x * kScanPer;
    uint32_t vals[kScanPer];
    uint64_t s = 0;
    /* a thread's 16 counts are contiguous: 16-byte loads where they lie
     * inside the array */
    const bool whole = b + kScanPer <= n;
    if (whole) {
#pragma unroll
        for (uint32_t i = 0; i < kScanPer; i += 4) {
            const Count4 v = *(const Count4*)(src + b + i);
            vals[i] = v.x;
            vals[i + 1] = v.y;
            vals[i + 2] = v.z;
            vals[i + 3] = v.w;
        }
    } else {
#pragma unroll
        for (uint32_t i = 0; i < kScanPer; ++i) {
            const uint64_t g = b + i;
            vals[i] = g < n ? src[g] : 0u;
        }
    }
#pragma unroll
    for (uint32_t i = 0; i < kScanPer; ++i) s += vals[i];
    /* exclusive scan of s across the block */
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint64_t incl = s;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint64_t t = (uint64_t)__shfl_up((unsigned long long)incl, d);
        if (lane >= d) incl += t;
    }
    if (lane == 63) sh[wave] = incl;
    __syncthreads();
    uint64_t run = base;
    for (int w = 0; w < wave; ++w) run += sh[w];
    run += incl - s;
    /* the last segment's last thread ends at the array's total */
    if (kFrom != kScanScanned && seg == nseg - 1 && threadIdx.x == kBlock - 1) totals[arr] = run + s;
    if (whole) {
#pragma unroll
        for (uint32_t i = 0; i < kScanPer; i += 2) {
            Prefix2 o;
            o.x = run;
            run += vals[i];
            o.y = run;
            run += vals[i + 1];
            *(Prefix2*)(dst + b + i) = o;
        }
    } else {
#pragma unroll
        for (uint32_t i = 0; i < kScanPer; ++i) {
            const uint64_t g = b + i;
            if (g < n) dst[g] = run;
            run += vals[i];
        }
    }
}

/* ------------------------------------------------------------------------- */
/* min / max                                                                   */
/* ------------------------------------------------------------------------- */

/* GetMinMaxValues<T> (StructuredVolumeObject.cpp:66-88) is a serial scan
 * min = v < min ? v : min seeded with the first value: NaNs never replace the
 * running extreme, and a NaN first value is never replaced.  The parallel form
 * reduces the non-NaN values and applies the first-value rule at the end. */
template <typename T>
__device__ __forceinline__ bool is_nan_val(T) { return false; }
template <> __device__ __forceinline__ bool is_nan_val<float>(float v) { return v != v; }
template <> __device__ __forceinline__ bool is_nan_val<double>(double v) { return v != v; }

/* Running extreme with the reference's tie rule: on equal values the earlier
 * index wins (only observable for float +0/-0). */
constexpr uint32_t kMinMaxParts = 2048;   // at most so many partial results of the first pass
static_assert(kMinMaxParts % kBlock == 0, "the final merge gives every thread the same number of parts");

template <typename T>
struct Extreme {
    T mn, mx;
    uint64_t imn, imx;
    uint32_t valid;
};

template <typename T>
__device__ __forceinline__ void merge_extreme(Extreme<T>& a, const Extreme<T>& b)
{
    if (!b.valid) return;
    if (!a.valid) { a = b; return; }
    if (b.mn < a.mn || (!(a.mn < b.mn) && b.imn < a.imn)) { a.mn = b.mn; a.imn = b.imn; }
    if (b.mx > a.mx || (!(a.mx > b.mx) && b.imx < a.imx)) { a.mx = b.mx; a.imx = b.imx; }
}

template <typename T>
__device__ __forceinline__ void take_value(Extreme<T>& e, T v, uint64_t i)
{
    if (is_nan_val<T>(v)) return;
    if (!e.valid) { e.mn = v; e.mx = v; e.imn = i; e.imx = i; e.valid = 1; return; }
    if (v < e.mn) { e.mn = v; e.imn = i; }
    if (v > e.mx) { e.mx = v; e.imx = i; }
}

/* Block-wide merge of the threads' extremes; thread 0 gets the result. */
template <typename T>
__device__ __forceinline__ Extreme<T> block_extreme(Extreme<T> e)
{
    __shared__ Extreme<T> sh[kBlock];
    sh[threadIdx.x] = e;
    __syncthreads();
    for (uint32_t s = kBlock / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) {
            Extreme<T> x = sh[threadIdx.x];
            merge_extreme(x, sh[threadIdx.x + s]);
            sh[threadIdx.x] = x;
        }
        __syncthreads();
    }
    return sh[0];
}

/* Streams the volume with 16-byte loads, kU of them in flight per thread;
 * each thread visits its elements in increasing index order, so strict
 * comparisons keep the first occurrence, and merges break ties by index. */
template <typename T>
__global__ __launch_bounds__(kBlock) void k_minmax_partial(const T* vol, uint64_t n, Extreme<T>* parts)
{
    constexpr uint32_t V = 16 / sizeof(T);
    constexpr uint32_t kU = 4;
    Extreme<T> e;
    e.mn = T(0); e.mx = T(0); e.imn = 0; e.imx = 0; e.valid = 0;
    const uint64_t tid = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    const uint64_t nth = (uint64_t)gridDim.x * kBlock;
    const bool aligned = ((uintptr_t)vol & 15u) == 0;
    const uint64_t nvec = aligned ? n / V : 0;
    const uint4* vp = (const uint4*)vol;
    for (uint64_t b = tid; b < nvec; b += nth * kU) {
        uint4 r[kU];
#pragma unroll
        for (uint32_t u = 0; u < kU; ++u) {
            const uint64_t idx = b + u * nth;
            r[u] = idx < nvec ? vp[idx] : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (uint32_t u = 0; u < kU; ++u) {
            const uint64_t idx = b + u * nth;
            if (idx < nvec) {
                T vals[V];
                __builtin_memcpy(vals, &r[u], 16);
#pragma unroll
                for (uint32_t k = 0; k < V; ++k) take_value(e, vals[k], idx * V + k);
            }
        }
    }
    for (uint64_t i = nvec * V + tid; i < n; i += nth) take_value(e, vol[i], i);
    const Extreme<T> r = block_extreme(e);
    if (threadIdx.x == 0) parts[blockIdx.x] = r;
}

/* GetMinMaxValues<T> of an unstructured volume (UnstructuredVolumeObject.cpp:
 * 123-141): the first value of the array, then every connection entry in
 * order.  Position 0 is vol[0], position p >= 1 is vol[conn[p - 1]]; each
 * thread visits its positions in increasing order. */
template <typename T>
__global__ __launch_bounds__(kBlock) void k_minmax_gather_partial(const T* vol, const uint32_t* conn, uint64_t nconn,
                                                                  Extreme<T>* parts)
{
    Extreme<T> e;
    e.mn = T(0); e.mx = T(0); e.imn = 0; e.imx = 0; e.valid = 0;
    const uint64_t tid = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    const uint64_t nth = (uint64_t)gridDim.x * kBlock;
    for (uint64_t p = tid; p <= nconn; p += nth) take_value(e, p == 0 ? vol[0] : vol[conn[p - 1]], p);
    const Extreme<T> r = block_extreme(e);
    if (threadIdx.x == 0) parts[blockIdx.x] = r;
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_minmax_final(const T* vol, const Extreme<T>* parts, uint32_t nparts, double* out)
{
    Extreme<T> e;
    e.mn = T(0); e.mx = T(0); e.imn = 0; e.imx = 0; e.valid = 0;
    const T first = vol[0];
    /* all parts of a thread in flight before the first is merged */
    constexpr uint32_t kPer = kMinMaxParts / kBlock;
    Extreme<T> p[kPer];
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) {
        const uint32_t i = threadIdx.x + k * kBlock;
        p[k] = parts[i < nparts ? i : 0u];
        if (i >= nparts) p[k].valid = 0;
    }
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) merge_extreme(e, p[k]);
    const Extreme<T> r = block_extreme(e);
    if (threadIdx.x == 0) {
        Extreme<T> f = r;
        if (is_nan_val<T>(first) || !f.valid) { f.mn = first; f.mx = first; }
        out[0] = (double)f.mn;
        out[1] = (double)f.mx;
    }
}

/* ------------------------------------------------------------------------- */
/* host-side launch wrappers                                                   */
/* ------------------------------------------------------------------------- */

/* Emit workgroups that fit on the device at once for this LDS size
 * (persistent grid); remembered per (kernel, LDS size). */
template <typename K>
uint32_t resident_blocks(K kernel, uint32_t lds_bytes, int block = kEmitBlock)
{
    static std::mutex mu;
    static std::map<std::pair<const void*, uint32_t>, uint32_t> known;
    const std::pair<const void*, uint32_t> key((const void*)kernel, lds_bytes);
    {
        std::lock_guard<std::mutex> lk(mu);
        auto it = known.find(key);
        if (it != known.end()) return it->second;
    }
    int cus = 0, dev = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) {
        (void)hipGetLastError();
        cus = 256;
    }
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, block, lds_bytes) != hipSuccess || per_cu <= 0) {
        (void)hipGetLastError();
        per_cu = 1;
    }
    const uint32_t n = (uint32_t)(cus * per_cu);
    std::lock_guard<std::mutex> lk(mu);
    known[key] = n;
    return n;
}

template <typename T>
hipError_t launch_emit_t(const JobArgs& a, uint32_t lds_bytes, hipStream_t st)
{
    const uint64_t teams = (a.nunits + a.teams - 1) / a.teams;
    switch (emit_mode(a)) {
    case kModeDup: {
        const uint64_t grid = std::min<uint64_t>(teams, resident_blocks(k_emit<T, kModeDup>, lds_bytes));
        hipLaunchKernelGGL((k_emit<T, kModeDup>), dim3((uint32_t)grid), dim3(kEmitBlock), lds_bytes, st, a);
        break;
    }
    case kModePolygon: {
        const uint64_t grid = std::min<uint64_t>(teams, resident_blocks(k_emit<T, kModePolygon>, lds_bytes));
        hipLaunchKernelGGL((k_emit<T, kModePolygon>), dim3((uint32_t)grid), dim3(kEmitBlock), lds_bytes, st, a);
        break;
    }
    default: {
        const uint64_t grid = std::min<uint64_t>(teams, resident_blocks(k_emit<T, kModeVertex>, lds_bytes));
        hipLaunchKernelGGL((k_emit<T, kModeVertex>), dim3((uint32_t)grid), dim3(kEmitBlock), lds_bytes, st, a);
        break;
    }
    }
    return hipGetLastError();
}

template <typename T>
hipError_t launch_classify_packed_t(const JobArgs& a, hipStream_t st)
{
    constexpr uint32_t P = 4 / sizeof(T);
    const uint64_t items = (uint64_t)a.ny * a.nz * ((a.nx / P + 63) / 64);
    uint64_t blocks = (items + 16 * kWaves - 1) / (16 * kWaves);
    if (blocks > (1u << 20)) blocks = 1u << 20;
    const dim3 g((uint32_t)blocks), b(kBlock);
    switch (a.nlev) {
    case 1: hipLaunchKernelGGL((k_classify_packed<T, 1>), g, b, 0, st, a); break;
    case 2: hipLaunchKernelGGL((k_classify_packed<T, 2>), g, b, 0, st, a); break;
    case 3: hipLaunchKernelGGL((k_classify_packed<T, 3>), g, b, 0, st, a); break;
    case 4: hipLaunchKernelGGL((k_classify_packed<T, 4>), g, b, 0, st, a); break;
    default: hipLaunchKernelGGL((k_classify_packed<T, 8>), g, b, 0, st, a); break;
    }
    return hipGetLastError();
}

template <typename T>
hipError_t launch_classify_t(const JobArgs& a, hipStream_t st)
{
    if constexpr (sizeof(T) <= 2) {
        /* rows of whole dwords: one dword of nodes per lane */
        if (packed_rows<T>(a)) return launch_classify_packed_t<T>(a, st);
    }
    if (classify_by_runs(a, sizeof(T))) {
        const uint64_t want = ((a.nrows * a.NC + 15) / 16 + kWaves - 1) / kWaves;
        const dim3 g((uint32_t)std::min<uint64_t>(want, 1u << 20)), b(kBlock);
        switch (a.nlev) {
        case 1: hipLaunchKernelGGL((k_classify_runs<T, 1>), g, b, 0, st, a); break;
        case 2: hipLaunchKernelGGL((k_classify_runs<T, 2>), g, b, 0, st, a); break;
        case 3: hipLaunchKernelGGL((k_classify_runs<T, 3>), g, b, 0, st, a); break;
        case 4: hipLaunchKernelGGL((k_classify_runs<T, 4>), g, b, 0, st, a); break;
        default: hipLaunchKernelGGL((k_classify_runs<T, 8>), g, b, 0, st, a); break;
        }
        return hipGetLastError();
    }
    /* one node row per wave: consecutive workgroups sweep the volume in
     * address order (measured faster than waves that take several rows) */
    const uint64_t rows = (uint64_t)a.ny * a.nz;
    uint64_t blocks = (rows + kWaves - 1) / kWaves;
    if (blocks > (1u << 20)) blocks = 1u << 20;
    const dim3 g((uint32_t)blocks), b(kBlock);
    switch (a.nlev) {
    case 1: hipLaunchKernelGGL((k_classify<T, 1>), g, b, 0, st, a); break;
    case 2: hipLaunchKernelGGL((k_classify<T, 2>), g, b, 0, st, a); break;
    case 3: hipLaunchKernelGGL((k_classify<T, 3>), g, b, 0, st, a); break;
    case 4: hipLaunchKernelGGL((k_classify<T, 4>), g, b, 0, st, a); break;
    default: hipLaunchKernelGGL((k_classify<T, 8>), g, b, 0, st, a); break;
    }
    return hipGetLastError();
}

hipError_t launch_classify(int dtype, const JobArgs& a, hipStream_t st)
{
    switch (dtype) {
    case 0: return launch_classify_t<int8_t>(a, st);
    case 1: return launch_classify_t<int16_t>(a, st);
    case 2: return launch_classify_t<int32_t>(a, st);
    case 3: return launch_classify_t<int64_t>(a, st);
    case 4: return launch_classify_t<uint8_t>(a, st);
    case 5: return launch_classify_t<uint16_t>(a, st);
    case 6: return launch_classify_t<uint32_t>(a, st);
    case 7: return launch_classify_t<uint64_t>(a, st);
    case 8: return launch_classify_t<float>(a, st);
    default: return launch_classify_t<double>(a, st);
    }
}

hipError_t launch_count(const JobArgs& a, hipStream_t st)
{
    const uint64_t G = 64u >> a.cshift;
    uint64_t blocks = ((a.nrows + G - 1) / G + kWaves - 1) / kWaves;
    if (blocks > 16384) blocks = 16384;
    if (a.nlev == 1) hipLaunchKernelGGL(k_count_level, dim3((uint32_t)blocks), dim3(kBlock), 0, st, a);
    else hipLaunchKernelGGL(k_count, dim3((uint32_t)blocks), dim3(kBlock), 0, st, a);
    return hipGetLastError();
}

/* Grid of a flat per-item kernel: up to 8 resident workgroups per CU. */
static uint32_t flat_blocks(uint64_t items)
{
    const uint64_t b = (items + kBlock - 1) / kBlock;
    return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(b, 256 * 8));
}

hipError_t launch_classify_plane(const JobArgs& a, hipStream_t st)
{
    const uint64_t rows = (uint64_t)a.ny * a.nz;
    uint64_t blocks = (rows + kWaves - 1) / kWaves;
    if (blocks > (1u << 20)) blocks = 1u << 20;
    hipLaunchKernelGGL(k_classify_plane, dim3((uint32_t)blocks), dim3(kBlock), 0, st, a);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_slice_emit_t(const JobArgs& a, hipStream_t st)
{
    hipLaunchKernelGGL((k_slice_triangles<T>), dim3(a.eblocks), dim3(kBlock), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_slice_runs_front(const JobArgs& a, int32_t* thr, uint32_t* counts, hipStream_t st)
{
    const uint64_t rows = (uint64_t)a.ny * a.nz, ncr = (uint64_t)(a.ny - 1) * (a.nz - 1);
    hipLaunchKernelGGL(k_slice_thresholds, dim3(flat_blocks(rows)), dim3(kBlock), 0, st, a, thr);
    if (ncr) hipLaunchKernelGGL(k_slice_row_counts, dim3(flat_blocks(ncr)), dim3(kBlock), 0, st, a, thr, counts);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_slice_runs_emit_t(const JobArgs& a, const int32_t* thr, const uint32_t* counts,
                                    const uint64_t* prefix, uint64_t* units, hipStream_t st)
{
    const uint64_t nt = a.toff[1], ncr = (uint64_t)(a.ny - 1) * (a.nz - 1), nunits = (nt + 63) / 64;
    if (!nt) return hipSuccess;
    uint64_t* first = units;
    uint64_t* last = units + nunits;
    hipLaunchKernelGGL(k_slice_unit_rows, dim3(flat_blocks(ncr)), dim3(kBlock), 0, st, ncr, counts, prefix, nt, first,
                       last);
    /* as many workgroups as fit at once: 1.6 rounds of them would take two */
    const uint64_t want = (nt + kBlock - 1) / kBlock;
    const uint32_t lds = a.cres <= kSliceLdsColors ? 3 * sizeof(float) * a.cres : 0;
    if (lds)
        hipLaunchKernelGGL((k_slice_triangles_runs<T, true>),
                           dim3((uint32_t)std::min<uint64_t>(want, resident_blocks(k_slice_triangles_runs<T, true>, lds, kBlock))),
                           dim3(kBlock), lds, st, a, thr, prefix, first, last);
    else
        hipLaunchKernelGGL((k_slice_triangles_runs<T, false>),
                           dim3((uint32_t)std::min<uint64_t>(want, resident_blocks(k_slice_triangles_runs<T, false>, 0, kBlock))),
                           dim3(kBlock), 0, st, a, thr, prefix, first, last);
    return hipGetLastError();
}

hipError_t launch_slice_runs_emit(int dtype, const JobArgs& a, const int32_t* thr, const uint32_t* counts,
                                  const uint64_t* prefix, uint64_t* units, hipStream_t st)
{
    switch (dtype) {
    case 0: return launch_slice_runs_emit_t<int8_t>(a, thr, counts, prefix, units, st);
    case 1: return launch_slice_runs_emit_t<int16_t>(a, thr, counts, prefix, units, st);
    case 2: return launch_slice_runs_emit_t<int32_t>(a, thr, counts, prefix, units, st);
    case 3: return launch_slice_runs_emit_t<int64_t>(a, thr, counts, prefix, units, st);
    case 4: return launch_slice_runs_emit_t<uint8_t>(a, thr, counts, prefix, units, st);
    case 5: return launch_slice_runs_emit_t<uint16_t>(a, thr, counts, prefix, units, st);
    case 6: return launch_slice_runs_emit_t<uint32_t>(a, thr, counts, prefix, units, st);
    case 7: return launch_slice_runs_emit_t<uint64_t>(a, thr, counts, prefix, units, st);
    case 8: return launch_slice_runs_emit_t<float>(a, thr, counts, prefix, units, st);
    default: return launch_slice_runs_emit_t<double>(a, thr, counts, prefix, units, st);
    }
}

hipError_t launch_slice_emit(int dtype, const JobArgs& a, hipStream_t st)
{
    switch (dtype) {
    case 0: return launch_slice_emit_t<int8_t>(a, st);
    case 1: return launch_slice_emit_t<int16_t>(a, st);
    case 2: return launch_slice_emit_t<int32_t>(a, st);
    case 3: return launch_slice_emit_t<int64_t>(a, st);
    case 4: return launch_slice_emit_t<uint8_t>(a, st);
    case 5: return launch_slice_emit_t<uint16_t>(a, st);
    case 6: return launch_slice_emit_t<uint32_t>(a, st);
    case 7: return launch_slice_emit_t<uint64_t>(a, st);
    case 8: return launch_slice_emit_t<float>(a, st);
    default: return launch_slice_emit_t<double>(a, st);
    }
}

hipError_t launch_emit(int dtype, const JobArgs& a, uint32_t lds_bytes, hipStream_t st)
{
    switch (dtype) {
    case 0: return launch_emit_t<int8_t>(a, lds_bytes, st);
    case 1: return launch_emit_t<int16_t>(a, lds_bytes, st);
    case 2: return launch_emit_t<int32_t>(a, lds_bytes, st);
    case 3: return launch_emit_t<int64_t>(a, lds_bytes, st);
    case 4: return launch_emit_t<uint8_t>(a, lds_bytes, st);
    case 5: return launch_emit_t<uint16_t>(a, lds_bytes, st);
    case 6: return launch_emit_t<uint32_t>(a, lds_bytes, st);
    case 7: return launch_emit_t<uint64_t>(a, lds_bytes, st);
    case 8: return launch_emit_t<float>(a, lds_bytes, st);
    default: return launch_emit_t<double>(a, lds_bytes, st);
    }
}

template <typename T>
hipError_t launch_classify_batch_t(const JobArgs* jobs, const BlockRef* refs, uint32_t nrefs, uint32_t max_levels, hipStream_t st)
{
    if (max_levels > 4) hipLaunchKernelGGL((k_classify_batch<T, true>), dim3(nrefs), dim3(kBlock), 0, st, jobs, refs);
    else hipLaunchKernelGGL((k_classify_batch<T, false>), dim3(nrefs), dim3(kBlock), 0, st, jobs, refs);
    return hipGetLastError();
}

hipError_t launch_classify_batch(int dtype, const JobArgs* jobs, const BlockRef* refs, uint32_t nrefs, uint32_t max_levels,
                                 hipStream_t st)
{
    switch (dtype) {
    case 0: return launch_classify_batch_t<int8_t>(jobs, refs, nrefs, max_levels, st);
    case 1: return launch_classify_batch_t<int16_t>(jobs, refs, nrefs, max_levels, st);
    case 2: return launch_classify_batch_t<int32_t>(jobs, refs, nrefs, max_levels, st);
    case 3: return launch_classify_batch_t<int64_t>(jobs, refs, nrefs, max_levels, st);
    case 4: return launch_classify_batch_t<uint8_t>(jobs, refs, nrefs, max_levels, st);
    case 5: return launch_classify_batch_t<uint16_t>(jobs, refs, nrefs, max_levels, st);
    case 6: return launch_classify_batch_t<uint32_t>(jobs, refs, nrefs, max_levels, st);
    case 7: return launch_classify_batch_t<uint64_t>(jobs, refs, nrefs, max_levels, st);
    case 8: return launch_classify_batch_t<float>(jobs, refs, nrefs, max_levels, st);
    default: return launch_classify_batch_t<double>(jobs, refs, nrefs, max_levels, st);
    }
}

hipError_t launch_count_batch(const JobArgs* jobs, const BlockRef* refs, uint32_t nrefs, hipStream_t st)
{
    hipLaunchKernelGGL(k_count_batch, dim3(nrefs), dim3(kBlock), 0, st, jobs, refs);
    return hipGetLastError();
}

template <typename T, int M>
hipError_t launch_emit_batch_m(const JobArgs* jobs, const uint64_t* unit_start, uint32_t njobs, uint64_t units,
                               uint32_t lds_bytes, uint32_t teams, hipStream_t st)
{
    const uint64_t grid = std::min<uint64_t>((units + teams - 1) / teams,
                                             resident_blocks(k_emit_batch<T, M>, lds_bytes));
    hipLaunchKernelGGL((k_emit_batch<T, M>), dim3((uint32_t)grid), dim3(kEmitBlock), lds_bytes, st, jobs, unit_start,
                       njobs, teams);
    return hipGetLastError();
}

/* Every pass of a batch group shares the value type T and the emit mode. */
template <typename T>
hipError_t launch_emit_batch_t(int mode, const JobArgs* jobs, const uint64_t* unit_start, uint32_t njobs,
                               uint64_t units, uint32_t lds_bytes, uint32_t teams, hipStream_t st)
{
    switch (mode) {
    case kModeDup: return launch_emit_batch_m<T, kModeDup>(jobs, unit_start, njobs, units, lds_bytes, teams, st);
    case kModePolygon: return launch_emit_batch_m<T, kModePolygon>(jobs, unit_start, njobs, units, lds_bytes, teams, st);
    default: return launch_emit_batch_m<T, kModeVertex>(jobs, unit_start, njobs, units, lds_bytes, teams, st);
    }
}

hipError_t launch_emit_batch(int dtype, int mode, const JobArgs* jobs, const uint64_t* unit_start, uint32_t njobs,
                             uint64_t units, uint32_t lds_bytes, uint32_t teams, hipStream_t st)
{
    switch (dtype) {
    case 0: return launch_emit_batch_t<int8_t>(mode, jobs, unit_start, njobs, units, lds_bytes, teams, st);
    case 1: return launch_emit_batch_t<int16_t>(mode, jobs, unit_start, njobs, units, lds_bytes, teams, st);
    case 2: return launch_emit_batch_t<int32_t>(mode, jobs, unit_start, njobs, units, lds_bytes, teams, st);
    case 3: return launch_emit_batch_t<int64_t>(mode, jobs, unit_start, njobs, units, lds_bytes, teams, st);
    case 4: return launch_emit_batch_t<uint8_t>(mode, jobs, unit_start, njobs, units, lds_bytes, teams, st);
    case 5: return launch_emit_batch_t<uint16_t>(mode, jobs, unit_start, njobs, units, lds_bytes, teams, st);
    case 6: return launch_emit_batch_t<uint32_t>(mode, jobs, unit_start, njobs, units, lds_bytes, teams, st);
    case 7: return launch_emit_batch_t<uint64_t>(mode, jobs, unit_start, njobs, units, lds_bytes, teams, st);
    case 8: return launch_emit_batch_t<float>(mode, jobs, unit_start, njobs, units, lds_bytes, teams, st);
    default: return launch_emit_batch_t<double>(mode, jobs, unit_start, njobs, units, lds_bytes, teams, st);
    }
}

/* Segments up to which a workgroup sums all counts before its own (one CU reads a
 * segment's 16 KiB in 1.1 us: 2 segments 5.4 us, 16 segments 17-21, in two
 * kernels 8 and a launch), and up to which it sums the segments' sums. */
constexpr uint32_t kScanDirect = 4, kScanSummed = 4096;

hipError_t launch_scan(const uint32_t* counts, uint64_t n, uint32_t narr, uint64_t* partials,
                       uint64_t* prefix, uint64_t* totals, hipStream_t st)
{
    const uint32_t nseg = (uint32_t)((n + kScanTile - 1) / kScanTile);
    const dim3 g(nseg * narr), b(kBlock);
    if (nseg <= kScanDirect) {
        hipLaunchKernelGGL(k_scan_apply<kScanCounts>, g, b, 0, st, counts, n, nseg, partials, prefix, totals);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(k_scan_partials, g, b, 0, st, counts, n, nseg, partials);
    if (nseg <= kScanSummed) {
        hipLaunchKernelGGL(k_scan_apply<kScanPartials>, g, b, 0, st, counts, n, nseg, partials, prefix, totals);
    } else {
        hipLaunchKernelGGL(k_scan_mid, dim3(1), b, 0, st, partials, nseg, narr, totals);
        hipLaunchKernelGGL(k_scan_apply<kScanScanned>, g, b, 0, st, counts, n, nseg, partials, prefix, totals);
    }
    return hipGetLastError();
}

uint32_t scan_partials_needed(uint64_t n, uint32_t narr)
{
    return (uint32_t)((n + kScanTile - 1) / kScanTile) * narr;
}

template <typename T>
hipError_t launch_minmax_t(const void* vol, uint64_t n, void* scratch, double* out, hipStream_t st)
{
    /* a small volume in workgroups of one load a thread: 64^3 floats are 256, and
     * the final merge then reads one part a thread, not eight */
    const uint64_t want = (n + (uint64_t)kBlock * (16 / sizeof(T)) - 1) / ((uint64_t)kBlock * (16 / sizeof(T)));
    const uint32_t nparts = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(want, kMinMaxParts));
    Extreme<T>* parts = (Extreme<T>*)scratch;
    hipLaunchKernelGGL((k_minmax_partial<T>), dim3(nparts), dim3(kBlock), 0, st, (const T*)vol, n, parts);
    hipLaunchKernelGGL((k_minmax_final<T>), dim3(1), dim3(kBlock), 0, st, (const T*)vol, parts, nparts, out);
    return hipGetLastError();
}

hipError_t launch_minmax(int dtype, const void* vol, uint64_t n, void* scratch, double* out, hipStream_t st)
{
    switch (dtype) {
    case 0: return launch_minmax_t<int8_t>(vol, n, scratch, out, st);
    case 1: return launch_minmax_t<int16_t>(vol, n, scratch, out, st);
    case 2: return launch_minmax_t<int32_t>(vol, n, scratch, out, st);
    case 3: return launch_minmax_t<int64_t>(vol, n, scratch, out, st);
    case 4: return launch_minmax_t<uint8_t>(vol, n, scratch, out, st);
    case 5: return launch_minmax_t<uint16_t>(vol, n, scratch, out, st);
    case 6: return launch_minmax_t<uint32_t>(vol, n, scratch, out, st);
    case 7: return launch_minmax_t<uint64_t>(vol, n, scratch, out, st);
    case 8: return launch_minmax_t<float>(vol, n, scratch, out, st);
    default: return launch_minmax_t<double>(vol, n, scratch, out, st);
    }
}

size_t minmax_scratch_bytes() { return kMinMaxParts * sizeof(Extreme<double>) + 64; }

template <typename T>
hipError_t launch_minmax_gather_t(const void* vol, const uint32_t* conn, uint64_t nconn, void* scratch, double* out,
                                  hipStream_t st)
{
    const uint32_t nparts = kMinMaxParts;
    Extreme<T>* parts = (Extreme<T>*)scratch;
    hipLaunchKernelGGL((k_minmax_gather_partial<T>), dim3(nparts), dim3(kBlock), 0, st, (const T*)vol, conn, nconn,
                       parts);
    hipLaunchKernelGGL((k_minmax_final<T>), dim3(1), dim3(kBlock), 0, st, (const T*)vol, parts, nparts, out);
    return hipGetLastError();
}

hipError_t launch_minmax_gather(int dtype, const void* vol, const uint32_t* conn, uint64_t nconn, void* scratch,
                                double* out, hipStream_t st)
{
    switch (dtype) {
    case 0: return launch_minmax_gather_t<int8_t>(vol, conn, nconn, scratch, out, st);
    case 1: return launch_minmax_gather_t<int16_t>(vol, conn, nconn, scratch, out, st);
    case 2: return launch_minmax_gather_t<int32_t>(vol, conn, nconn, scratch, out, st);
    case 3: return launch_minmax_gather_t<int64_t>(vol, conn, nconn, scratch, out, st);
    case 4: return launch_minmax_gather_t<uint8_t>(vol, conn, nconn, scratch, out, st);
    case 5: return launch_minmax_gather_t<uint16_t>(vol, conn, nconn, scratch, out, st);
    case 6: return launch_minmax_gather_t<uint32_t>(vol, conn, nconn, scratch, out, st);
    case 7: return launch_minmax_gather_t<uint64_t>(vol, conn, nconn, scratch, out, st);
    case 8: return launch_minmax_gather_t<float>(vol, conn, nconn, scratch, out, st);
    default: return launch_minmax_gather_t<double>(vol, conn, nconn, scratch, out, st);
    }
}

}  // namespace kmc
