/*
 * kmc_device.h -- device code shared by the kernel sources: the case table,
 * the interpolation and face normal of the reference, wave helpers, cell
 * geometry and the chunk masks of the bit volume.
 */
#pragma once
#include <hip/hip_runtime.h>
#include "kmc_job.h"
#include "mc_tables.h"

#pragma clang fp contract(off)

namespace kmc {

static __constant__ uint64_t d_tri[256] = { KMC_TABLE_WORDS };

/* Emit modes, a template parameter so that each kernel carries only its own
 * path: duplicated vertices, shared vertices with PolygonNormal, shared
 * vertices with VertexNormal. */
enum : int { kModeDup = 0, kModePolygon = 1, kModeVertex = 2 };

__host__ __device__ inline int emit_mode(const JobArgs& a) { return a.dup ? kModeDup : (a.vnormal ? kModeVertex : kModePolygon); }

/* ------------------------------------------------------------------------- */
/* interpolation and normals                                                   */
/* ------------------------------------------------------------------------- */

template <typename T>
__device__ __forceinline__ void interpolate_values(const JobArgs& a, double iso, T value_a, T value_b,
                                                   uint32_t ax, uint32_t ay, uint32_t az,
                                                   uint32_t bx, uint32_t by, uint32_t bz, float out[3]);

/* interpolate_vertex<T> + (p + min_coord) * scale_factor for the edge from
 * node a to node b (integer node coordinates). */
template <typename T>
__device__ __forceinline__ void interpolate(const JobArgs& a, const T* vol, double iso,
                                            uint32_t ax, uint32_t ay, uint32_t az,
                                            uint32_t bx, uint32_t by, uint32_t bz, float out[3])
{
    const uint64_t line = a.nx, slice = (uint64_t)a.nx * a.ny;
    const uint64_t ia = ax + ay * line + az * slice;
    const uint64_t ib = bx + by * line + bz * slice;
    interpolate_values<T>(a, iso, vol[ia], vol[ib], ax, ay, az, bx, by, bz, out);
}

/* The interpolation of interpolate() from the two node values. */
template <typename T>
__device__ __forceinline__ void interpolate_values(const JobArgs& a, double iso, T value_a, T value_b,
                                                   uint32_t ax, uint32_t ay, uint32_t az,
                                                   uint32_t bx, uint32_t by, uint32_t bz, float out[3])
{
    double va = (double)value_a;
    double vb = (double)value_b;
    va = va <= a.minv ? a.minv : (va <= a.maxv ? va : a.maxv);
    vb = vb <= a.minv ? a.minv : (vb <= a.maxv ? vb : a.maxv);
    double r = (iso - va) / (vb - va);
    r = r < 0 ? -r : r;
    const double s = 1.0 - r;
    const double pa[3] = { (double)(float)ax, (double)(float)ay, (double)(float)az };
    const double pb[3] = { (double)(float)bx, (double)(float)by, (double)(float)bz };
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const double t0 = s * pa[k];
        const double t1 = r * pb[k];
        const float p = (float)(t0 + t1);
        const float q = p + a.minc[k];
        out[k] = q * a.sc[k];
    }
}

__device__ __forceinline__ void face_normal(const float v0[3], const float v1[3], const float v2[3], float n[3])
{
    const float d1x = v1[0] - v0[0], d1y = v1[1] - v0[1], d1z = v1[2] - v0[2];
    const float d2x = v2[0] - v0[0], d2y = v2[1] - v0[1], d2z = v2[2] - v0[2];
    const float p0 = d1y * d2z, p1 = d1z * d2y;
    const float p2 = d1z * d2x, p3 = d1x * d2z;
    const float p4 = d1x * d2y, p5 = d1y * d2x;
    n[0] = p0 - p1;
    n[1] = p2 - p3;
    n[2] = p4 - p5;
}

/* ------------------------------------------------------------------------- */
/* wave helpers                                                                */
/* ------------------------------------------------------------------------- */

/* The LDS operations of one wave complete in issue order; wave_sync only keeps
 * the compiler from moving memory operations across the points where lanes
 * start reading what other lanes wrote. */
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ uint32_t uniform(uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }

__device__ __forceinline__ uint64_t uniform64(uint64_t x)
{
    return (uint64_t)uniform((uint32_t)(x >> 32)) << 32 | uniform((uint32_t)x);
}

__device__ __forceinline__ uint64_t readlane64(uint64_t x, int k)
{
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, k);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), k);
    return (uint64_t)hi << 32 | lo;
}

/* Set bits of the wave mask m on the lanes below this one (v_mbcnt). */
__device__ __forceinline__ uint32_t lanes_below(uint64_t m)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t t = __shfl_up(x, d);
        if (lane >= d) x += t;
    }
    return x;
}

/* Mask of the nodes x < limit inside chunk c. */
__device__ __forceinline__ uint64_t valid_mask(uint32_t c, uint32_t limit)
{
    const uint32_t x0 = c * 64u;
    if (limit <= x0) return 0ull;
    const uint32_t n = limit - x0;
    return n >= 64u ? ~0ull : ((1ull << n) - 1ull);
}

/* ------------------------------------------------------------------------- */
/* cell geometry                                                               */
/* ------------------------------------------------------------------------- */

/* Owner node offset (dx, dy, dz) and axis of local edge e, packed as
 * dx | dy << 1 | dz << 2 | axis << 3 (connect_isopoints, :493-504), five
 * bits per edge. */
__device__ __forceinline__ uint32_t edge_owner(uint32_t e)
{
    constexpr uint64_t kOwner =
        (0x00ull << 0) | (0x09ull << 5) | (0x02ull << 10) | (0x08ull << 15) | (0x04ull << 20) | (0x0Dull << 25) |
        (0x06ull << 30) | (0x0Cull << 35) | (0x10ull << 40) | (0x11ull << 45) | (0x13ull << 50) | (0x12ull << 55);
    return (uint32_t)(kOwner >> (5 * e)) & 31u;
}

/* Table-orientation endpoints of local edge e as two corner offsets packed
 * bit0 x, bit1 y, bit2 z, first endpoint in the low nibble
 * (MarchingCubesTable.cpp:276-290), eight bits per edge. */
__device__ __forceinline__ uint32_t edge_ends(uint32_t e)
{
    constexpr uint64_t kLo = 0x4667755402233110ull;   // edges 0..7
    constexpr uint32_t kHi = 0x62735140u;             // edges 8..11
    return e < 8 ? (uint32_t)(kLo >> (8 * e)) & 0xFFu : (kHi >> (8 * (e - 8))) & 0xFFu;
}

/* The four cells around the edge of node (x, y, zv) along axis, in scan
 * order: offsets across the edge are -1/0 along the other two axes (low axis
 * first); the edge's local id in cell q is the q-th nibble of `around`. */
__device__ __forceinline__ void around_cell(uint32_t axis, int q, int x, int y, int zv, int& cx, int& cy, int& cz)
{
    const int lo = (q & 1) ? 0 : -1, hi = (q & 2) ? 0 : -1;
    cx = x + (axis == 0 ? 0 : lo);
    cy = y + (axis == 0 ? lo : (axis == 1 ? 0 : hi));
    cz = zv + (axis == 2 ? 0 : hi);
}

__device__ __forceinline__ uint32_t around_nibbles(uint32_t axis)
{
    return axis == 0 ? 0x0246u : (axis == 1 ? 0x3175u : 0x89BAu);
}

/* ------------------------------------------------------------------------- */
/* chunks of the bit volume                                                    */
/* ------------------------------------------------------------------------- */

/* Crossing edges and active cells of chunk c of node row (y, z) of one level,
 * read straight from the bit volume `lev` (coalesced across the lanes of a
 * row, neighbours from L1/L2).  x/y/z: crossing edges owned by the row's
 * nodes; act: active cells of cell row (y, z-1); k0/k3/k4/k7: the masks of
 * the cells' four node rows (bit i of kq is corner q of cell x = 64c + i; the
 * x+1 corners 1, 2, 5, 6 are the next bits of the same masks); next: bit 0 of
 * the next chunk's word of those four rows (corners 1, 2, 5, 6 of cell 63). */
struct RowChunk {
    uint64_t x, y, z, act;
    uint64_t k0, k3, k4, k7;
    uint32_t next;
};

__device__ __forceinline__ void row_chunk(const JobArgs& a, const uint64_t* lev, uint32_t y, uint32_t z, uint32_t c,
                                          RowChunk& o)
{
    const uint64_t slice_words = (uint64_t)a.ny * a.NC;
    const bool has_up = y + 1 < a.ny, has_next = z + 1 < a.nz, has_cells = z >= 1 && has_up;
    /* Every load is issued (no branch around it): a neighbour row outside the
     * volume is read as the row itself, which makes its crossings (b ^ u,
     * b ^ n0) zero, and the cells are masked out below.  The next chunk of a
     * row's last chunk is read as the chunk itself: its bit 0 lands only on
     * bit 63 of the shifted words and of `next`, i.e. on node / cell 64c + 63,
     * which lies at or past nx - 1 in a row's last chunk, so valid_mask(c,
     * nx - 1) clears it from x and act (and corner_pairs reads `next` only for
     * an active cell 63). */
    const uint64_t* row = lev + (uint64_t)z * slice_words + (uint64_t)y * a.NC;
    const uint64_t* up = has_up ? row + a.NC : row;
    const uint64_t* nz = has_next ? row + slice_words : row;
    const uint64_t* pr = has_cells ? row - slice_words : row;
    const uint64_t* pu = has_cells ? pr + a.NC : row;
    const uint32_t cn = c + 1 < a.NC ? c + 1 : c;
    const uint64_t b = row[c], b1 = row[cn];
    const uint64_t u = up[c], u1 = up[cn];
    const uint64_t n0 = nz[c];
    const uint64_t p = pr[c], p1 = pr[cn];
    const uint64_t q = pu[c], q1 = pu[cn];
    const uint64_t c4 = b, c5 = (b >> 1) | (b1 << 63);
    const uint64_t c7 = u, c6 = (u >> 1) | (u1 << 63);
    const uint64_t c1 = (p >> 1) | (p1 << 63), c2 = (q >> 1) | (q1 << 63);
    const uint64_t vx = valid_mask(c, a.nx - 1), vn = valid_mask(c, a.nx);
    o.x = (b ^ c5) & vx;
    o.y = (b ^ u) & vn;
    o.z = (b ^ n0) & vn;
    const uint64_t or_ = p | c1 | c2 | q | c4 | c5 | c6 | c7;
    const uint64_t an = p & c1 & c2 & q & c4 & c5 & c6 & c7;
    o.act = has_cells ? (or_ & ~an) & vx : 0ull;
    o.k0 = p;
    o.k3 = q;
    o.k4 = c4;
    o.k7 = c7;
    o.next = (uint32_t)(p1 & 1ull) | (uint32_t)(q1 & 1ull) << 1 | (uint32_t)(b1 & 1ull) << 2 |
             (uint32_t)(u1 & 1ull) << 3;
}

/* The cube index with bits 2, 3 and bits 6, 7 swapped (an involution). */
__device__ __forceinline__ uint32_t swap_pairs(uint32_t c)
{
    return (c & 0x33u) | ((c & 0x44u) << 1) | ((c & 0x88u) >> 1);
}

/* swap_pairs(cube index) of cell i of a chunk: the corners (x, x+1) of each of
 * the cell's four node rows are two adjacent bits of that row's mask (k0, k3,
 * k4, k7), taken as one 2-bit window; for cell 63 the x+1 bits come from the
 * next chunk (o.next). */
__device__ __forceinline__ uint32_t corner_pairs(const RowChunk& o, uint32_t i)
{
    if (i == 63u) {
        return (uint32_t)(o.k0 >> 63) | (o.next & 1u) << 1 | (uint32_t)(o.k3 >> 63) << 2 |
               ((o.next >> 1) & 1u) << 3 | (uint32_t)(o.k4 >> 63) << 4 | ((o.next >> 2) & 1u) << 5 |
               (uint32_t)(o.k7 >> 63) << 6 | ((o.next >> 3) & 1u) << 7;
    }
    const uint32_t p0 = (uint32_t)(o.k0 >> i) & 3u, p3 = (uint32_t)(o.k3 >> i) & 3u;
    const uint32_t p4 = (uint32_t)(o.k4 >> i) & 3u, p7 = (uint32_t)(o.k7 >> i) & 3u;
    return p0 | p3 << 2 | p4 << 4 | p7 << 6;
}

}  // namespace kmc
