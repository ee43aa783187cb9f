/*
 * kmc_emit.hip -- emit of a pass in chunk batches (gfx950, wave64).
 *
 * After the count pass and the scan, the output position of everything a
 * 64-node chunk holds is known: row prefix + chunk prefix within the row.  A
 * wave walks its share of a level's (row, chunk) slots (kmc_plan.h), queues the
 * chunks that hold something in LDS and works on 32, 48 or 64 of them at a time:
 * each lane takes one chunk's masks, the wave lists the chunks' active cells or
 * crossing edges in LDS, and the listed items are produced one per lane -- every lane
 * busy whatever the chunks hold; only the vertex normals need more than the
 * outputs written (face normals and cell records).
 *
 * Output order: cells in scan order, triangles in table order
 * (extract_surfaces_with_duplication,
 * Source/Core/Visualization/Mapper/MarchingCubes.cpp:155-243).
 */
#include <hip/hip_runtime.h>
#include <algorithm>
#include <type_traits>
#include "kmc_chunks.h"
#include "kmc_device.h"
#include "kmc_internal.h"
#include "kmc_job.h"

#pragma clang fp contract(off)

namespace kmc {

namespace {

/* The cases as the cells' lanes need them, indexed by swap_pairs(cube index)
 * (corner_pairs).  edges: the crossing edges (bit e: edge e).  tri: the
 * triangle count in the top nibble and, 12 bits a triangle, its corners in
 * output order (T[i], T[i+2], T[i+1]) as ranks among the case's crossing
 * edges. */
struct EdgeEnds {
    float x, y, z;          // offset of the first end from the cell's first node
    uint32_t at;            // first end << 6 | second end << 19 | second end above the first << 3 | axis bits
};

struct alignas(16) CaseLds {
    uint64_t tri[256];
    EdgeEnds ends[12];
    uint16_t edges[256];
};

/* The tables, evaluated at compile time (a workgroup only copies them); the
 * edges in their table orientation (MarchingCubesTable.cpp:276-290). */
constexpr uint64_t kTableWords[256] = { KMC_TABLE_WORDS };

constexpr uint32_t bits_below(uint32_t m, uint32_t e)
{
    uint32_t n = 0;
    for (uint32_t k = 0; k < e; ++k) n += (m >> k) & 1u;
    return n;
}

constexpr CaseLds make_cases()
{
    CaseLds t{};
    for (uint32_t i = 0; i < 256; ++i) {
        const uint64_t w = kTableWords[(i & 0x33u) | ((i & 0x44u) << 1) | ((i & 0x88u) >> 1)];
        const uint32_t n = 3u * (uint32_t)(w >> 60);
        uint32_t m = 0;
        for (uint32_t k = 0; k < n; ++k) m |= 1u << ((w >> (4 * k)) & 0xFu);
        uint64_t o = w & 0xFull << 60;
        for (uint32_t k = 0; k < n; ++k) {
            const uint32_t c = k % 3, from = c == 1 ? k + 1 : c == 2 ? k - 1 : k;
            o |= (uint64_t)bits_below(m, (uint32_t)(w >> (4 * from)) & 0xFu) << (4 * k);
        }
        t.tri[i] = o;
        t.edges[i] = (uint16_t)m;
    }
    for (uint32_t e = 0; e < 12; ++e) {
        const uint32_t o = e < 8 ? (uint32_t)(0x4667755402233110ull >> (8 * e)) & 0xFFu
                                 : (0x62735140u >> (8 * (e - 8))) & 0xFFu;   // edge_ends
        const uint32_t p = o & 7u, q = o >> 4, axis = p ^ q;
        t.ends[e] = EdgeEnds{ (float)(p & 1u), (float)((p >> 1) & 1u), (float)(p >> 2),
                              p << 6 | q << 19 | ((q & axis) ? 8u : 0u) | axis };
    }
    return t;
}

static __constant__ CaseLds d_cases_dup = make_cases();

__device__ __forceinline__ void stage_cases(CaseLds& t, const CaseLds& from)
{
    static_assert(sizeof(CaseLds) % 16 == 0, "copied in 16-byte words");
    for (uint32_t i = threadIdx.x; i < sizeof(CaseLds) / 16; i += kBlock) ((uint4*)&t)[i] = ((const uint4*)&from)[i];
    __syncthreads();
}

/* LDS of one wave of the duplicated triangles: 9.1 kB with values of up to 32
 * bits, so that four workgroups fit a CU's 160 KiB; 11.1 kB with 64 bits, three. */
constexpr uint32_t kDupCells = 320;      // active cells listed at once (a chunk has at most 64)
constexpr uint32_t kVerts = 236;         // edge crossings of the up to 64 cells in work (a cell has at most 12)

struct CellPos { float x, y, z; };         // exact: coordinates lie below 2^24

template <typename T>
struct CellLds {
    uint32_t q[kChunks + 64];    // busy queue: at most kChunks - 1 left over and 64 new
    uint64_t m[4][kChunks];      // k0, k3, k4, k7 of each chunk (RowChunk)
    uint64_t out[kChunks];       // output id - batch rank of each chunk's triangles (its first array's address with
    uint64_t out2[kChunks];      // duplicated vertices, the second one's here)
    uint64_t key[kChunks];       // 64 c | y << 20 | z << 40 of each chunk's first cell
    CellPos cpos[64];            // the cells in work
    uint32_t next[kChunks];
    float p[kVerts][3];          // crossing points of the cells in work
    uint16_t el[kVerts];         // crossing: cell | edge << 6
    uint16_t cells[kDupCells];   // chunk | cell << 6
    union {
        T v[8 * 64];             // node values of the cells in work (corner offset bits x, y, z)
        uint32_t tl[320];        // then their triangles: three crossings | chunk << 24
    };
};

/* Floats in device memory, for pointers that come out of LDS. */
using GlobalFloats = __attribute__((address_space(1))) float*;

/* Two neighbouring values (one load). */
template <typename T>
__device__ __forceinline__ void load_pair(const T* p, T& a, T& b)
{
    struct __attribute__((packed, aligned(sizeof(T)))) Pair { T a, b; };
    const Pair v = *(const Pair*)p;
    a = v.a;
    b = v.b;
}

/* A node value in the interpolation's clamp range (interpolate_vertex,
 * MarchingCubes.cpp:335-341).  With kFloatClamp the range's ends are floats,
 * in order, and so is every value of T: the clamp is then done on floats, and
 * a NaN becomes the upper end as in the reference's comparisons. */
template <typename T, bool kFloatClamp>
__device__ __forceinline__ double clamped(const JobArgs& a, T value)
{
    if constexpr (kFloatClamp) {
        return (double)fmaxf(fminf((float)value, a.fmaxv), a.fminv);
    } else {
        const double v = (double)value;
        return v <= a.minv ? a.minv : (v <= a.maxv ? v : a.maxv);
    }
}

/* Crossing point of a grid edge: interpolate_vertex<T> and the callers' (p +
 * min_coord) * scale (interpolate_values).  With 0 <= r <= 1 the sums (1 - r)
 * p + r p of the two axes along which both ends have the same coordinate p are
 * p itself (p is an integer below 2^24: the double sum is within a few 2^-53 p
 * of p, and rounds to the float p), so only the edge's own axis is evaluated;
 * any other r takes the general form. */
template <typename T, bool kFloatClamp>
__device__ __forceinline__ void crossing_point(const JobArgs& a, double iso, T value_a, T value_b, const EdgeEnds& e,
                                               const CellPos& c, float out[3])
{
    const double va = clamped<T, kFloatClamp>(a, value_a), vb = clamped<T, kFloatClamp>(a, value_b);
    double r = (iso - va) / (vb - va);
    r = r < 0 ? -r : r;
    const double s = 1.0 - r;
    const bool ax = (e.at & 1u) != 0, ay = (e.at & 2u) != 0, az = (e.at & 4u) != 0;
    const double dir = (e.at & 8u) ? 1.0 : -1.0;
    float p[3] = { c.x + e.x, c.y + e.y, c.z + e.z };
    if (__builtin_expect(r <= 1.0, 1)) {
        const double ia = (double)(ax ? p[0] : (ay ? p[1] : p[2]));
        const double t0 = s * ia;
        const double t1 = r * (ia + dir);
        const float f = (float)(t0 + t1);
        p[0] = ax ? f : p[0];
        p[1] = ay ? f : p[1];
        p[2] = az ? f : p[2];
    } else {
        const bool on[3] = { ax, ay, az };
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const double ia = (double)p[k];
            const double t0 = s * ia;
            const double t1 = r * (on[k] ? ia + dir : ia);
            p[k] = (float)(t0 + t1);
        }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float q = p[k] + a.minc[k];
        out[k] = q * a.sc[k];
    }
}

/* A cell in work: its chunk, position, case and node values. */
template <typename T>
struct CellItem {
    uint32_t chunk, edges, nt;
    uint64_t tri;
    bool first;             // of its chunk
    CellPos pos;
    T v[8];
};

/* Cell k of the list of ncells; nothing (no crossing, no triangle) past it. */
template <typename T>
__device__ __forceinline__ void fetch_cell(const JobArgs& a, const CaseLds& tab, const CellLds<T>& s, uint32_t k,
                                           uint32_t ncells, CellItem<T>& o)
{
    o.chunk = o.edges = o.nt = 0;
    o.tri = 0;
    o.first = false;
    if (k >= ncells) return;
    const uint32_t cell = s.cells[k];
    const uint32_t q = cell & 63u, i = cell >> 6;
    const uint64_t key = s.key[q];
    const uint32_t x = (uint32_t)(key & 0xFFFFFu) + i, y = (uint32_t)((key >> 20) & 0xFFFFFu), z = (uint32_t)(key >> 40);
    const uint64_t line = a.nx, slice = (uint64_t)a.nx * a.ny;
    const T* src = (const T*)a.values + (x + y * line + z * slice);
    load_pair(src, o.v[0], o.v[1]);
    load_pair(src + line, o.v[2], o.v[3]);
    load_pair(src + slice, o.v[4], o.v[5]);
    load_pair(src + slice + line, o.v[6], o.v[7]);
    o.pos = CellPos{ (float)x, (float)y, (float)z };
    o.chunk = q;
    o.first = k == 0 || (s.cells[k - 1] & 63u) != q;
    const uint32_t pi = corner_pairs_at(s.m, s.next, q, i);
    o.tri = tab.tri[pi];
    o.edges = tab.edges[pi];
    o.nt = (uint32_t)(o.tri >> 60);
}

/* s_waitcnt vmcnt(0), the other counters at their maximum. */
constexpr int kWaitVm0 = 0x0F70;

/* The n queued chunks' cells, up to 64 in work at a time, one per lane: their
 * node values are loaded as four pairs, their edge crossings listed and
 * computed one per lane into s.p, and their triangles listed in s.tl; then
 * emit(count, rank) produces the outputs of the `count` listed triangles, rank
 * being the first one's rank in the batch.  place(chunk, d) is called before a
 * chunk's first triangle: the output id of its triangles is d + rank. */
template <typename T, typename P, typename F>
__device__ __forceinline__ void chunk_triangles(const JobArgs& a, const EmitLevel& L, double iso, const CaseLds& tab,
                                                CellLds<T>& s, uint32_t n, P&& place, F&& emit)
{
    /* types whose values are all floats */
    constexpr bool kFloat = sizeof(T) <= 2 || std::is_same<T, float>::value;
    const uint32_t lane = threadIdx.x & 63u;
    uint64_t act = 0;
    if (lane < n) {
        uint64_t r;
        uint32_t y, z, c;
        chunk_place(a, L, s.q[lane], r, y, z, c);
        const CellMasks o = load_cells(a, L, y, z, c);
        const uint64_t w = r * a.NC + c;
        act = o.act;
        s.m[0][lane] = o.k0;
        s.m[1][lane] = o.k3;
        s.m[2][lane] = o.k4;
        s.m[3][lane] = o.k7;
        s.next[lane] = o.next;
        s.key[lane] = (uint64_t)(c * 64u) | (uint64_t)y << 20 | (uint64_t)(z - 1) << 40;
        s.out[lane] = (L.pt[r] - L.t0) + triangles_before(a, L, w);
    }
    const uint32_t incl = wave_incl_scan((uint32_t)__popcll(act));
    const uint32_t excl = incl - (uint32_t)__popcll(act);
    const uint32_t total = uniform((uint32_t)__builtin_amdgcn_readlane((int)incl, 63));
    uint32_t rank = 0;
    for (uint32_t start = 0; start < total;) {
        /* chunks whose cells fit the list */
        const uint64_t fit = __ballot(excl >= start && incl - start <= kDupCells && act != 0);
        const uint32_t stop = uniform((uint32_t)__builtin_amdgcn_readlane((int)incl, 63 - __builtin_clzll(fit)));
        list_bits(act, excl, start, fit, total > 8 * n, s.cells);
        wave_sync();
        const uint32_t ncells = stop - start;
        CellItem<T> cur;
        fetch_cell<T>(a, tab, s, lane, ncells, cur);
        for (uint32_t k0 = 0; k0 < ncells;) {
            /* triangles in the high, crossings in the low half; the cells
             * whose crossings fit s.p are taken */
            const uint32_t mine = (uint32_t)__popc(cur.edges) | cur.nt << 16;
            const uint32_t inc = wave_incl_scan(mine);
            const uint64_t take = __ballot(k0 + lane < ncells && (inc & 0xFFFFu) <= kVerts);
            const uint32_t ntake = (uint32_t)__popcll(take);
            const uint32_t both = uniform((uint32_t)__builtin_amdgcn_readlane((int)inc, (int)ntake - 1));
            const uint32_t ne = both & 0xFFFFu, ntri = both >> 16;
            const uint32_t e0 = (inc - mine) & 0xFFFFu, t0 = (inc - mine) >> 16;
            if (lane < ntake) {
                uint32_t m = cur.edges, p = e0;
                while (m) {
                    const uint32_t e = (uint32_t)__ffs(m) - 1u;
                    m &= m - 1u;
                    s.el[p++] = (uint16_t)(lane | e << 6);
                }
                /* the chunk's first cell turns its output base into base - rank */
                if (cur.first) place(cur.chunk, s.out[cur.chunk] - (uint64_t)(rank + t0));
                s.cpos[lane] = cur.pos;
#pragma unroll
                for (int j = 0; j < 8; ++j) s.v[j * 64 + lane] = cur.v[j];
            }
            wave_sync();
            /* the next cells' values are in flight during the crossings, and
             * here before this step's stores: vector memory operations
             * complete in issue order, so a wait for loads issued after the
             * stores would wait for the stores too */
            CellItem<T> nxt;
            fetch_cell<T>(a, tab, s, k0 + ntake + lane, ncells, nxt);
            for (uint32_t j = lane; j < ne; j += 64) {
                const uint32_t w = s.el[j], c = w & 63u;
                const EdgeEnds e = tab.ends[w >> 6];
                const T va = s.v[(e.at & 0x1FFFu & ~63u) + c], vb = s.v[(e.at >> 13 & ~63u) + c];
                float pt[3];
                if (kFloat && a.fclamp)
                    crossing_point<T, kFloat>(a, iso, va, vb, e, s.cpos[c], pt);
                else
                    crossing_point<T, false>(a, iso, va, vb, e, s.cpos[c], pt);
                s.p[j][0] = pt[0];
                s.p[j][1] = pt[1];
                s.p[j][2] = pt[2];
            }
            wave_sync();
            __builtin_amdgcn_s_waitcnt(kWaitVm0);
            if (lane < ntake) {
                const uint32_t at = e0 * 0x010101u + (cur.chunk << 24);
                for (uint32_t t = 0; t < cur.nt; ++t) {
                    const uint32_t w = (uint32_t)(cur.tri >> (12 * t));
                    s.tl[t0 + t] = at + ((w & 0xFu) | (w & 0xF0u) << 4 | (w & 0xF00u) << 8);
                }
            }
            wave_sync();
            emit(ntri, rank);
            wave_sync();
            rank += ntri;
            k0 += ntake;
            cur = nxt;
        }
        start = stop;
    }
}

/* ------------------------------------------------------------------------- */
/* duplicated vertices                                                         */
/* ------------------------------------------------------------------------- */

template <typename T>
__device__ __forceinline__ void dup_level(const JobArgs& a, uint32_t l, uint32_t block, const CaseLds& tab, CellLds<T>& s)
{
    if (!a.cap_triangles[l]) return;       // a level without outputs
    const uint32_t lane = threadIdx.x & 63u;
    const EmitLevel L = emit_level(a, l, block);
    const double iso = a.iso[l];
    float* coords = a.coords[l];
    float* normals = a.normals[l];
    const uint32_t lane_k = lane / 3, lane_c = lane - 3 * lane_k;
    busy_chunks<false, kChunks>(a, L, s.q, [&](uint32_t n) {
        chunk_triangles<T>(a, L, iso, tab, s, n, [&](uint32_t q, uint64_t d) {
            s.out[q] = (uint64_t)(coords + 9 * d);
            s.out2[q] = (uint64_t)(normals + 3 * d);
        }, [&](uint32_t cnt, uint32_t rank) {
            /* a corner per lane: the stores of a wave are contiguous */
            uint32_t c = lane_c;
            for (uint32_t k = lane_k; k < cnt;) {
                const uint32_t t = s.tl[k];
                const float* p = s.p[(t >> (8 * c)) & 255u];
                GlobalFloats co = (GlobalFloats)(s.out[t >> 24] + (36u * (rank + k) + 12u * c));
                co[0] = p[0];
                co[1] = p[1];
                co[2] = p[2];
                /* 64 corners on: 21 triangles and one corner */
                k += c == 2 ? 22u : 21u;
                c = c == 2 ? 0u : c + 1u;
            }
            for (uint32_t k = lane; k < cnt; k += 64) {
                const uint32_t t = s.tl[k];
                float nn[3];
                face_normal(s.p[t & 255u], s.p[(t >> 8) & 255u], s.p[(t >> 16) & 255u], nn);
                GlobalFloats no = (GlobalFloats)(s.out2[t >> 24] + 12u * (rank + k));
                no[0] = nn[0];
                no[1] = nn[1];
                no[2] = nn[2];
            }
        });
    });
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_dup(JobArgs a)
{
    __shared__ CaseLds tab;
    __shared__ CellLds<T> s[kWaves];
    stage_cases(tab, d_cases_dup);
    dup_level<T>(a, blockIdx.y, blockIdx.x, tab, s[threadIdx.x >> 6]);
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_dup_batch(const JobArgs* jobs, const BlockRef* refs)
{
    __shared__ CaseLds tab;
    __shared__ CellLds<T> s[kWaves];
    const BlockRef r = refs[blockIdx.x];
    const JobArgs& a = jobs[r.job];
    stage_cases(tab, d_cases_dup);
    dup_level<T>(a, r.level, r.block, tab, s[threadIdx.x >> 6]);
}

/* ------------------------------------------------------------------------- */
/* shared vertices: coordinates                                                */
/* ------------------------------------------------------------------------- */

/* Crossing edges of a wave's chunks, listed in output order (nodes in scan
 * order, x, y, z edge of each), and produced one per lane. */
constexpr uint32_t kPointList = 512;     // crossings listed at once (a chunk has at most 192)

/* N: chunks worked on at a time. */
template <uint32_t N>
struct PointLds {
    uint32_t q[N + 64];          // busy queue: at most N - 1 left over and 64 new
    uint64_t key[N];             // 64 c | y << 20 | z << 40 of each chunk's first node
    uint64_t out[N];             // output id - batch rank of each chunk's vertices
    uint16_t el[kPointList];     // chunk | node << 6 | axis << 12
};

/* The vertices of the n queued chunks: emit(first, count, rank) for runs of
 * listed ones, s.el[0 .. count); a vertex's id is s.out[chunk] + its rank.
 * chunk(row, y, z, chunk of the row) is called on a lane of its own each. */
template <uint32_t N, typename C, typename F>
__device__ __forceinline__ void chunk_points(const JobArgs& a, const EmitLevel& L, PointLds<N>& s, uint32_t n, C&& chunk,
                                             F&& emit)
{
    const uint32_t lane = threadIdx.x & 63u;
    uint64_t mx = 0, my = 0, mz = 0, base = 0;
    if (lane < n) {
        uint64_t r;
        uint32_t y, z, c;
        chunk_place(a, L, s.q[lane], r, y, z, c);
        /* row_chunk's crossings alone: a neighbour row outside the volume is
         * read as the row itself */
        const uint64_t* row = L.bits + r * a.NC;
        uint64_t b, b1;
        load_words(row + c, b, b1);
        const uint64_t u = (y + 1 < a.ny ? row + a.NC : row)[c];
        const uint64_t nz = (z + 1 < a.nz ? row + (uint64_t)a.ny * a.NC : row)[c];
        const uint64_t vn = valid_mask(c, a.nx);
        mx = (b ^ (b >> 1 | b1 << 63)) & valid_mask(c, a.nx - 1);
        my = (b ^ u) & vn;
        mz = (b ^ nz) & vn;
        base = (L.pv[r] - L.v0) + (L.vp[r * a.NC + c] & prefix_mask(a));
        s.key[lane] = (uint64_t)(c * 64u) | (uint64_t)y << 20 | (uint64_t)z << 40;
        chunk(r, y, z, c);
    }
    const uint32_t cnt = (uint32_t)(__popcll(mx) + __popcll(my) + __popcll(mz));
    const uint32_t incl = wave_incl_scan(cnt);
    const uint32_t excl = incl - cnt;
    const uint32_t total = uniform((uint32_t)__builtin_amdgcn_readlane((int)incl, 63));
    if (lane < n) s.out[lane] = base - (uint64_t)excl;
    for (uint32_t start = 0; start < total;) {
        const uint64_t fit = __ballot(excl >= start && incl - start <= kPointList && cnt != 0);
        const uint32_t stop = uniform((uint32_t)__builtin_amdgcn_readlane((int)incl, 63 - __builtin_clzll(fit)));
        if (total > 16 * n) {
            /* dense: chunk after chunk, a node per lane (list_bits) */
            for (uint64_t f = fit; f; f &= f - 1) {
                const int q = __builtin_ctzll(f);
                const uint64_t x = readlane64(mx, q), y = readlane64(my, q), z = readlane64(mz, q);
                uint32_t p = (uint32_t)__builtin_amdgcn_readlane((int)excl, q) - start + lanes_below(x) + lanes_below(y) +
                             lanes_below(z);
                const uint32_t e = (uint32_t)q | lane << 6;
                if (__builtin_amdgcn_inverse_ballot_w64(x)) s.el[p++] = (uint16_t)e;
                if (__builtin_amdgcn_inverse_ballot_w64(y)) s.el[p++] = (uint16_t)(e | 1u << 12);
                if (__builtin_amdgcn_inverse_ballot_w64(z)) s.el[p] = (uint16_t)(e | 2u << 12);
            }
        } else if ((fit >> lane) & 1ull) {
            uint64_t m = mx | my | mz;
            uint32_t p = excl - start;
            while (m) {
                const uint32_t i = (uint32_t)__ffsll((unsigned long long)m) - 1u;
                m &= m - 1ull;
                const uint32_t e = lane | i << 6;
                if ((mx >> i) & 1ull) s.el[p++] = (uint16_t)e;
                if ((my >> i) & 1ull) s.el[p++] = (uint16_t)(e | 1u << 12);
                if ((mz >> i) & 1ull) s.el[p++] = (uint16_t)(e | 2u << 12);
            }
        }
        wave_sync();
        emit(stop - start, start);
        wave_sync();
        start = stop;
    }
}

/* A vertex in flight. */
template <typename T>
struct PointItem {
    uint32_t x, y, z, axis;
    uint64_t id;
    T va, vb;
};

template <typename T>
__device__ __forceinline__ void fetch_point(const JobArgs& a, const PointLds<64>& s, uint32_t j, uint32_t rank, PointItem<T>& o)
{
    const uint32_t e = s.el[j], q = e & 63u;
    const uint64_t key = s.key[q];
    o.x = (uint32_t)(key & 0xFFFFFu) + ((e >> 6) & 63u);
    o.y = (uint32_t)((key >> 20) & 0xFFFFFu);
    o.z = (uint32_t)(key >> 40);
    o.axis = e >> 12;
    o.id = s.out[q] + (rank + j);
    const uint64_t line = a.nx, slice = (uint64_t)a.nx * a.ny;
    const T* src = (const T*)a.values + (o.x + o.y * line + o.z * slice);
    o.va = src[0];
    o.vb = src[o.axis == 0 ? 1ull : (o.axis == 1 ? line : slice)];
}

/* Its coordinates, interpolated low -> high (calculate_isopoints, :365-437). */
template <typename T>
__device__ __forceinline__ void store_point(const JobArgs& a, double iso, float* coords, const PointItem<T>& o)
{
    constexpr bool kFloat = sizeof(T) <= 2 || std::is_same<T, float>::value;
    const EdgeEnds e{ 0.0f, 0.0f, 0.0f, 8u | 1u << o.axis };
    const CellPos c{ (float)o.x, (float)o.y, (float)o.z };
    float p[3];
    if (kFloat && a.fclamp)
        crossing_point<T, kFloat>(a, iso, o.va, o.vb, e, c, p);
    else
        crossing_point<T, false>(a, iso, o.va, o.vb, e, c, p);
    float* co = coords + 3 * o.id;
    co[0] = p[0];
    co[1] = p[1];
    co[2] = p[2];
}

template <typename T>
__device__ __forceinline__ void points_level(const JobArgs& a, uint32_t l, uint32_t block, PointLds<64>& s)
{
    if (!a.cap_vertices[l]) return;        // a level without outputs
    const uint32_t lane = threadIdx.x & 63u;
    const EmitLevel L = emit_level(a, l, block);
    const double iso = a.iso[l];
    float* coords = a.coords[l];
    busy_chunks<true, 64>(a, L, s.q, [&](uint32_t n) {
        chunk_points(a, L, s, n, [](uint64_t, uint32_t, uint32_t, uint32_t) {}, [&](uint32_t cnt, uint32_t rank) {
            /* two vertices a lane, their values in flight together; lanes
             * past the end fetch the last one and store nothing */
            for (uint32_t j = lane; j < cnt + lane; j += 128) {
                PointItem<T> p0, p1;
                fetch_point<T>(a, s, j < cnt ? j : cnt - 1, rank, p0);
                fetch_point<T>(a, s, j + 64 < cnt ? j + 64 : cnt - 1, rank, p1);
                if (j < cnt) store_point<T>(a, iso, coords, p0);
                if (j + 64 < cnt) store_point<T>(a, iso, coords, p1);
            }
        });
    });
}

template <typename T>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(7))) void k_points(JobArgs a)
{
    __shared__ PointLds<64> s[kWaves];
    points_level<T>(a, blockIdx.y, blockIdx.x, s[threadIdx.x >> 6]);
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_points_batch(const JobArgs* jobs, const BlockRef* refs)
{
    __shared__ PointLds<64> s[kWaves];
    const BlockRef r = refs[blockIdx.x];
    const JobArgs& a = jobs[r.job];
    points_level<T>(a, r.level, r.block, s[threadIdx.x >> 6]);
}

/* ------------------------------------------------------------------------- */
/* shared vertices: triangles                                                  */
/* ------------------------------------------------------------------------- */

/* Crossing edges of one chunk of a node row: the id of its first vertex and
 * the x / y / z edge masks of its nodes. */
struct RowCross {
    uint64_t x, y, z;
    uint32_t base;           // vertex ids are 32-bit, as the connections are
    uint32_t next;           // bits 0, 1: the x and y edge of the next chunk's first node
};

struct FaceCases {
    uint64_t tri[256];       // by pair index: corners in output order (edges), count in the top nibble
    uint16_t edge[12];       // owner row (dy | dz << 1) << 4 | dx << 3 | axis
    uint16_t pad[4];
};

constexpr FaceCases make_face_cases()
{
    FaceCases t{};
    for (uint32_t i = 0; i < 256; ++i) {
        const uint64_t w = kTableWords[(i & 0x33u) | ((i & 0x44u) << 1) | ((i & 0x88u) >> 1)];
        uint64_t o = w & 0xFull << 60;
        for (uint32_t k = 0; k < 3u * (uint32_t)(w >> 60); ++k) {
            const uint32_t c = k % 3, from = c == 1 ? k + 1 : c == 2 ? k - 1 : k;
            o |= ((w >> (4 * from)) & 0xFull) << (4 * k);
        }
        t.tri[i] = o;
    }
    constexpr uint64_t kOwner =
        (0x00ull << 0) | (0x09ull << 5) | (0x02ull << 10) | (0x08ull << 15) | (0x04ull << 20) | (0x0Dull << 25) |
        (0x06ull << 30) | (0x0Cull << 35) | (0x10ull << 40) | (0x11ull << 45) | (0x13ull << 50) | (0x12ull << 55);
    for (uint32_t e = 0; e < 12; ++e) {   // edge_owner: dx | dy << 1 | dz << 2 | axis << 3
        const uint32_t o = (uint32_t)(kOwner >> (5 * e)) & 31u;
        t.edge[e] = (uint16_t)((o >> 1 & 3u) << 4 | (o & 1u) << 3 | o >> 3);
    }
    return t;
}

static __constant__ FaceCases d_face_cases = make_face_cases();

/* Node rows (y, z), (y + 1, z), (y, z + 1), (y + 1, z + 1) of a chunk's cells;
 * 144 bytes, so that lanes reading one row of different chunks spread over the
 * LDS banks. */
struct ChunkRows {
    RowCross r[4];
    uint32_t pad[4];
};

struct FaceLds {
    ListLds l;
    uint64_t k0[kChunks];        // mask of each chunk's first node row
    uint64_t act[kChunks];       // active cells (VertexNormal)
    uint32_t tri0[kChunks];      // id of each chunk's first triangle (32-bit, VertexNormal)
    ChunkRows row[kChunks];
};

/* corner_pairs of cell i of a chunk: the first corner's bit and the crossings
 * of the edges that lead from it to the others. */
__device__ __forceinline__ uint32_t pair_of(const FaceLds& s, uint32_t q, uint32_t i)
{
    const RowCross* r = s.row[q].r;
    const uint32_t c0 = (uint32_t)(s.k0[q] >> i) & 1u;
    const uint32_t c1 = c0 ^ ((uint32_t)(r[0].x >> i) & 1u), c3 = c0 ^ ((uint32_t)(r[0].y >> i) & 1u);
    const uint32_t c4 = c0 ^ ((uint32_t)(r[0].z >> i) & 1u), c2 = c3 ^ ((uint32_t)(r[1].x >> i) & 1u);
    const uint32_t c7 = c3 ^ ((uint32_t)(r[1].z >> i) & 1u), c5 = c4 ^ ((uint32_t)(r[2].x >> i) & 1u);
    const uint32_t c6 = c7 ^ ((uint32_t)(r[3].x >> i) & 1u);
    return c0 | c1 << 1 | c3 << 2 | c2 << 3 | c4 << 4 | c5 << 5 | c7 << 6 | c6 << 7;
}

/* The cells of cell row (y, z - 1), chunk c, and the crossing edges of its four
 * node rows (all in the volume): eight mask rows, five of them with their next
 * word. */
__device__ __forceinline__ CellMasks load_row_cross(const JobArgs& a, const EmitLevel& L, uint32_t y, uint32_t z,
                                                    uint32_t c, ChunkRows& o)
{
    const uint64_t sw = (uint64_t)a.ny * a.NC, r0 = (uint64_t)(z - 1) * a.ny + y, r2 = r0 + a.ny;
    const uint64_t* p = L.bits + r0 * a.NC + c;
    const uint64_t* q = p + sw;
    const uint64_t* u = z + 1 < a.nz ? q + sw : q;      // a row past the volume is read as the one before it
    const uint32_t y2 = y + 2 < a.ny ? 2 * a.NC : a.NC;
    uint64_t m00, n00, m10, n10, m20, n20, m01, n01, m11, n11;
    load_words(p, m00, n00);
    load_words(p + a.NC, m10, n10);
    load_words(p + y2, m20, n20);
    load_words(q, m01, n01);
    load_words(q + a.NC, m11, n11);
    const uint64_t m21 = q[y2], m02 = u[0], m12 = u[a.NC];
    uint64_t v0, v1, v2, v3;
    load_words(L.pv + r0, v0, v1);
    load_words(L.pv + r2, v2, v3);
    const uint32_t* vp = L.vp + r0 * a.NC + c;
    const uint32_t mask = prefix_mask(a);
    const uint32_t e0 = vp[0] & mask, e1 = vp[a.NC] & mask, e2 = vp[sw] & mask, e3 = vp[sw + a.NC] & mask;
    const uint64_t vx = valid_mask(c, a.nx - 1), vn = valid_mask(c, a.nx);
    auto cross = [&](RowCross& k, uint64_t b, uint64_t b1, uint64_t up, uint64_t nz, uint64_t pre, uint32_t e,
                     uint32_t next) {
        k.x = (b ^ (b >> 1 | b1 << 63)) & vx;
        k.y = (b ^ up) & vn;
        k.z = (b ^ nz) & vn;
        k.base = (uint32_t)(pre - L.v0) + e;
        k.next = next;
    };
    /* x and y edge of the first node of the next chunk (read for a cell 63 only,
     * whose node x + 1 it is; its x edge needs a node after it) */
    const uint64_t has = 64ull * (c + 1) + 1 < a.nx ? 1ull : 0ull;
    auto next_bits = [&](uint64_t b1, uint64_t up1) {
        return (uint32_t)((b1 ^ b1 >> 1) & has) | (uint32_t)((b1 ^ up1) & 1ull) << 1;
    };
    cross(o.r[0], m00, n00, m10, m01, v0, e0, next_bits(n00, n10));
    cross(o.r[1], m10, n10, m20, m11, v1, e1, next_bits(n10, n20));
    cross(o.r[2], m01, n01, m11, m02, v2, e2, next_bits(n01, n11));
    cross(o.r[3], m11, n11, m21, m12, v3, e3, 0u);
    return cell_masks(a, c, m00, n00, m10, n10, m01, n01, m11, n11);
}

/* Vertex id on the edge along `axis` of node i (0 .. 64) of a row's chunk: its
 * first vertex + the crossing edges of the nodes before i and of node i's
 * lower axes. */
__device__ __forceinline__ uint32_t cross_rank(const RowCross& o, uint32_t i, uint32_t axis)
{
    const uint64_t lo = i ? ~0ull >> (64u - i) : 0ull;
    const uint32_t r = o.base + (uint32_t)(__popcll(o.x & lo) + __popcll(o.y & lo) + __popcll(o.z & lo));
    const uint32_t bx = i < 64u ? (uint32_t)(o.x >> i) & 1u : o.next & 1u;
    const uint32_t by = i < 64u ? (uint32_t)(o.y >> i) & 1u : o.next >> 1;
    return r + (axis >= 1 ? bx : 0u) + (axis >= 2 ? by : 0u);
}

/* A triangle in flight: its vertices and their coordinates. */
struct FaceItem {
    uint64_t id;
    uint32_t v[3];
    float p[3][3];
};

__device__ __forceinline__ void fetch_face(const FaceCases& tab, const FaceLds& s, const float* coords,
                                           uint32_t cell, uint32_t t, uint32_t rank, FaceItem& o)
{
    const uint32_t q = cell & 63u, i = (cell >> 6) & 63u;
    o.id = s.l.out[q] + rank;
    const uint32_t w = (uint32_t)(tab.tri[cell >> 12] >> (12 * t));
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const uint32_t d = tab.edge[(w >> (4 * j)) & 0xFu];
        o.v[j] = cross_rank(s.row[q].r[d >> 4], i + ((d >> 3) & 1u), d & 7u);
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const float* c = coords + 3 * (uint64_t)o.v[j];
        o.p[j][0] = c[0];
        o.p[j][1] = c[1];
        o.p[j][2] = c[2];
    }
}

/* Every triangle of shared vertices: its connectivity (connect_isopoints,
 * :439-521) and the face normal of its vertices' coordinates -- the
 * PolygonNormal output (calculate_normals_on_polygon, :531-559) or, with
 * VertexNormal, kept in a.fn for the per-vertex sums, which find it through
 * the chunk's active cells (a.act) and their first triangles and cases
 * (a.crec). */
template <int M>
__device__ __forceinline__ void faces_level(const JobArgs& a, uint32_t l, uint32_t block, const FaceCases& tab, FaceLds& s)
{
    if (!a.cap_triangles[l]) return;       // a level without outputs
    const uint32_t lane = threadIdx.x & 63u;
    const EmitLevel L = emit_level(a, l, block);
    const float* coords = a.coords[l];
    uint32_t* conn = a.conn[l];
    float* normals = M == kModeVertex ? a.fn + 3 * a.toff[l] : a.normals[l];
    uint64_t* act_l = M == kModeVertex ? a.act + (uint64_t)l * (a.nrows * a.NC) : nullptr;
    uint32_t* crec = M == kModeVertex ? a.crec + a.toff[l] : nullptr;
    busy_chunks<false, kChunks>(a, L, s.l.q, [&](uint32_t n) {
        list_triangles(a, L, tab.tri, s.l, n, [&](uint64_t r, uint32_t y, uint32_t z, uint32_t c, uint64_t base) {
            const CellMasks o = load_row_cross(a, L, y, z, c, s.row[lane]);
            s.k0[lane] = o.k0;
            if constexpr (M == kModeVertex) {
                act_l[r * a.NC + c] = o.act;
                s.act[lane] = o.act;
                s.tri0[lane] = (uint32_t)base;
            }
            return o.act;
        }, [&](uint32_t q, uint32_t i) { return pair_of(s, q, i); }, [&](uint32_t q, uint32_t i, uint32_t pi, uint32_t rank) {
            /* first triangle relative to the chunk's first, and the case */
            if constexpr (M == kModeVertex) {
                const uint32_t t0 = s.tri0[q], ord = (uint32_t)__popcll(s.act[q] & ((1ull << i) - 1ull));
                crec[t0 + ord] = ((uint32_t)s.l.out[q] + rank - t0) | pi << 16;
            }
        }, [&](uint32_t cnt, uint32_t rank) {
            /* (two triangles a lane, their loads in flight together, are
             * slower: 349 us to 317 on the 512^3 CT volume) */
            for (uint32_t j = lane; j < cnt; j += 64) {
                const uint32_t e = s.l.tl[j];
                FaceItem o;
                fetch_face(tab, s, coords, s.l.cell[e & 63u], e >> 6, rank + j, o);
                uint32_t* k = conn + 3 * o.id;
                k[0] = o.v[0];
                k[1] = o.v[1];
                k[2] = o.v[2];
                float nn[3];
                face_normal(o.p[0], o.p[1], o.p[2], nn);
                float* no = normals + 3 * o.id;
                no[0] = nn[0];
                no[1] = nn[1];
                no[2] = nn[2];
            }
        });
    });
}

__device__ __forceinline__ void stage_face_cases(FaceCases& t)
{
    static_assert(sizeof(FaceCases) % 16 == 0, "copied in 16-byte words");
    for (uint32_t i = threadIdx.x; i < sizeof(FaceCases) / 16; i += kBlock) ((uint4*)&t)[i] = ((const uint4*)&d_face_cases)[i];
    __syncthreads();
}

template <int M>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(5))) void k_faces(JobArgs a)
{
    __shared__ __attribute__((aligned(16))) FaceCases tab;
    __shared__ FaceLds s[kWaves];
    stage_face_cases(tab);
    faces_level<M>(a, blockIdx.y, blockIdx.x, tab, s[threadIdx.x >> 6]);
}

template <int M>
__global__ __launch_bounds__(kBlock) void k_faces_batch(const JobArgs* jobs, const BlockRef* refs)
{
    __shared__ __attribute__((aligned(16))) FaceCases tab;
    __shared__ FaceLds s[kWaves];
    const BlockRef r = refs[blockIdx.x];
    const JobArgs& a = jobs[r.job];
    stage_face_cases(tab);
    faces_level<M>(a, r.level, r.block, tab, s[threadIdx.x >> 6]);
}

/* ------------------------------------------------------------------------- */
/* shared vertices: vertex normals                                             */
/* ------------------------------------------------------------------------- */

/* Triangles (table order, a bit each) of a case that use an edge. */
struct UseCases { uint8_t use[256][12]; };

constexpr UseCases make_use_cases()
{
    UseCases t{};
    for (uint32_t i = 0; i < 256; ++i) {
        const uint64_t w = kTableWords[(i & 0x33u) | ((i & 0x44u) << 1) | ((i & 0x88u) >> 1)];
        for (uint32_t k = 0; k < 3u * (uint32_t)(w >> 60); ++k) t.use[i][(w >> (4 * k)) & 0xFu] |= (uint8_t)(1u << (k / 3));
    }
    return t;
}

static __constant__ UseCases d_use_cases = make_use_cases();

/* A cell row around a chunk of nodes: the active cells of the chunk, its first
 * triangle, and that of the chunk before it, whose cell 63 is the x - 1 cell
 * of node 0. */
struct RowCells {
    uint64_t act;
    uint32_t tri0, prev_tri0;
};

/* The cell rows (y - 1, z - 1), (y, z - 1), (y - 1, z), (y, z) of a chunk; 72
 * bytes, so that lanes reading one row of different chunks spread over the LDS
 * banks.  info: 8 bits a row, the active cells of the chunk before it without
 * its cell 63, and bit 7 set when the row lies in the volume. */
struct ChunkCells {
    RowCells r[4];
    uint32_t info, pad;
};

constexpr uint32_t kNormalChunks = 48;

struct NormalLds {
    PointLds<kNormalChunks> p;
    ChunkCells row[kNormalChunks];
};

/* VertexNormal: the float sum, in triangle order, of the face normals of the
 * triangles that use the vertex (calculate_normals_on_vertex, :569-605) -- the
 * four cells around its edge in cell scan order and each cell's triangles in
 * table order.  A cell's record (a.crec) gives its case and first triangle;
 * the face normals of the first two triangles of every cell are loaded
 * together (most cells have one or two), further ones after.  A slot without
 * a triangle adds +0, which changes no partial sum: the sum starts at +0 and a
 * float sum is -0 only when both terms are. */
struct NormalItem {
    uint32_t around, rec[4], t0[4], m[4];
    bool in[4];
    uint64_t id;
    float f[4][2][3];
};

/* The vertex's cells and their records (loads issued). */
__device__ __forceinline__ void fetch_cells(const JobArgs& a, const NormalLds& s, const uint32_t* crec, uint32_t j,
                                            uint32_t rank, NormalItem& o)
{
    const uint32_t e = s.p.el[j], q = e & 63u, i = (e >> 6) & 63u, axis = e >> 12;
    const uint32_t c64 = (uint32_t)(s.p.key[q] & 0xFFFFFu);
    o.around = around_nibbles(axis);
    o.id = s.p.out[q] + (rank + j);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        int dx, dy, dz;
        around_cell(axis, k, 0, 0, 0, dx, dy, dz);
        const uint32_t row = (uint32_t)((dy + 1) | (dz + 1) << 1);
        const RowCells& r = s.row[q].r[row];
        const uint32_t info = s.row[q].info >> (8 * row);
        const int ci = (int)i + dx;
        o.in[k] = (info & 128u) && (int)c64 + ci >= 0 && c64 + (uint32_t)(ci + 1) < a.nx;
        const uint64_t below = (1ull << (ci & 63)) - 1ull;
        o.t0[k] = ci >= 0 ? r.tri0 : r.prev_tri0;
        const uint32_t at = o.t0[k] + (ci >= 0 ? (uint32_t)__popcll(r.act & below) : info & 127u);
        o.rec[k] = crec[o.in[k] ? at : 0u];
    }
}

/* The first two face normals of every cell (loads issued). */
__device__ __forceinline__ void fetch_faces(const UseCases& use, const float* fn, NormalItem& o)
{
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        o.m[k] = o.in[k] ? (uint32_t)use.use[(o.rec[k] >> 16) & 255u][(o.around >> (4 * k)) & 0xFu] : 0u;
        o.t0[k] += o.rec[k] & 0xFFFFu;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            o.f[k][u][0] = o.f[k][u][1] = o.f[k][u][2] = 0.0f;
            if (o.m[k]) {
                const uint32_t t = (uint32_t)__ffs(o.m[k]) - 1u;
                o.m[k] &= o.m[k] - 1u;
                const float* p = fn + 3 * (uint64_t)(o.t0[k] + t);
                o.f[k][u][0] = p[0];
                o.f[k][u][1] = p[1];
                o.f[k][u][2] = p[2];
            }
        }
    }
}

__device__ __forceinline__ void store_normal(const float* fn, NormalItem& o, float* normals)
{
    /* the starting +0 comes from an opaque move, so that the compiler does not
     * fold the first addition into the first load's branch (which would wait
     * for that load alone) */
    float zero;
    asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
    float n[3] = { zero, zero, zero };
#pragma unroll
    for (int k = 0; k < 4; ++k) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            n[0] = n[0] + o.f[k][u][0];
            n[1] = n[1] + o.f[k][u][1];
            n[2] = n[2] + o.f[k][u][2];
        }
        while (o.m[k]) {   // further triangles of the cell that use the edge (rare)
            const uint32_t t = (uint32_t)__ffs(o.m[k]) - 1u;
            o.m[k] &= o.m[k] - 1u;
            const float* p = fn + 3 * (uint64_t)(o.t0[k] + t);
            n[0] = n[0] + p[0];
            n[1] = n[1] + p[1];
            n[2] = n[2] + p[2];
        }
    }
    float* no = normals + 3 * o.id;
    no[0] = n[0];
    no[1] = n[1];
    no[2] = n[2];
}

__device__ __forceinline__ void normals_level(const JobArgs& a, uint32_t l, uint32_t block, const UseCases& use, NormalLds& s)
{
    if (!a.cap_vertices[l]) return;        // a level without outputs
    const uint32_t lane = threadIdx.x & 63u;
    const EmitLevel L = emit_level(a, l, block);
    float* normals = a.normals[l];
    const bool triangles = a.cap_triangles[l] != 0;   // without one no cell of the volume is active
    const float* fn = a.fn + 3 * a.toff[l];
    const uint32_t* crec = triangles ? a.crec + a.toff[l] : (const uint32_t*)L.bits;   // read, not used, without one
    const uint64_t* act_l = a.act + (uint64_t)l * (a.nrows * a.NC);
    const uint32_t* tri_pre = a.NC <= 64 ? L.vp : L.tp;   // packed: triangles in the high half of vp
    const uint32_t sh = a.NC <= 64 ? 16u : 0u, mask = prefix_mask(a);
    busy_chunks<true, kNormalChunks>(a, L, s.p.q, [&](uint32_t n) {
        chunk_points(a, L, s.p, n, [&](uint64_t r, uint32_t y, uint32_t z, uint32_t c) {
            /* cell row (cy, cz) is kept at node row (cy, cz + 1): node rows r -
             * 1, r and the same of the next slice; the words of this chunk and
             * the one before it in one load each (node row r >= 1 wherever a
             * row below or a chunk before is used) */
            const bool y0 = triangles && y >= 1, y1 = triangles && y + 1 < a.ny, z0 = z >= 1, z1 = z + 1 < a.nz;
            uint32_t info = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const bool in = (k & 1 ? y1 : y0) && (k & 2 ? z1 : z0);
                const uint64_t cr = in ? r - (k & 1 ? 0 : 1) + (k & 2 ? a.ny : 0) : r;
                const uint64_t w = cr * a.NC + c, w1 = w ? w - 1 : 0;
                const uint32_t base = (uint32_t)(L.pt[cr] - L.t0);
                uint64_t act1, act;
                load_words(act_l + w1, act1, act);
                uint32_t e1, e;
                load_pair(tri_pre + w1, e1, e);
                e1 = base + (e1 >> sh & mask);
                e = base + (e >> sh & mask);
                if (w == 0) { act = act1; e = e1; }
                RowCells o;
                o.act = act;
                o.tri0 = e;
                o.prev_tri0 = e1;
                s.row[lane].r[k] = o;
                info |= ((uint32_t)__popcll(act1 & ~(1ull << 63)) | (in ? 128u : 0u)) << (8 * k);
            }
            s.row[lane].info = info;
        }, [&](uint32_t cnt, uint32_t rank) {
            for (uint32_t j = lane; j < cnt; j += 64) {
                NormalItem o;
                fetch_cells(a, s, crec, j, rank, o);
                fetch_faces(use, fn, o);
                store_normal(fn, o, normals);
            }
        });
    });
}

__device__ __forceinline__ void stage_use_cases(UseCases& t)
{
    static_assert(sizeof(UseCases) % 16 == 0, "copied in 16-byte words");
    for (uint32_t i = threadIdx.x; i < sizeof(UseCases) / 16; i += kBlock) ((uint4*)&t)[i] = ((const uint4*)&d_use_cases)[i];
    __syncthreads();
}

__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(6))) void k_normals(JobArgs a)
{
    __shared__ __attribute__((aligned(16))) UseCases use;
    __shared__ NormalLds s[kWaves];
    stage_use_cases(use);
    normals_level(a, blockIdx.y, blockIdx.x, use, s[threadIdx.x >> 6]);
}

__global__ __launch_bounds__(kBlock) void k_normals_batch(const JobArgs* jobs, const BlockRef* refs)
{
    __shared__ __attribute__((aligned(16))) UseCases use;
    __shared__ NormalLds s[kWaves];
    const BlockRef r = refs[blockIdx.x];
    const JobArgs& a = jobs[r.job];
    stage_use_cases(use);
    normals_level(a, r.level, r.block, use, s[threadIdx.x >> 6]);
}

/* Workgroups of each kernel that a CU holds: by LDS k_dup dup_blocks and k_faces 5,
 * by registers k_points 7 and k_normals 5 or more. */
constexpr uint32_t kPointBlocks = 7, kFaceBlocks = 5, kNormalBlocks = 5;

template <typename T>
hipError_t launch_chunk_emit_t(JobArgs a, hipStream_t st, hipEvent_t* marks)
{
    static_assert((160u << 10) / (sizeof(CaseLds) + kWaves * sizeof(CellLds<T>)) == dup_blocks(sizeof(T)), "workgroups a CU holds");
    const dim3 b(kBlock);
    uint64_t nv = 0, nt = 0;
    for (uint32_t l = 0; l < a.nlev; ++l) { nv += a.cap_vertices[l]; nt += a.cap_triangles[l]; }
    /* each kernel's waves by the workgroups of it that a CU holds */
    auto grid = [&](uint32_t per_cu, uint64_t items) {
        plan_emit(a, emit_steps(a), per_cu, items);
        return dim3(a.eblocks, a.nlev);
    };
    if (!a.dup) hipLaunchKernelGGL((k_points<T>), grid(kPointBlocks, nv), b, 0, st, a);
    if (marks) (void)hipEventRecord(marks[0], st);
    switch (emit_mode(a)) {
    case kModeDup: hipLaunchKernelGGL((k_dup<T>), grid(dup_blocks(sizeof(T)), nt), b, 0, st, a); break;
    case kModePolygon: hipLaunchKernelGGL((k_faces<kModePolygon>), grid(kFaceBlocks, nt), b, 0, st, a); break;
    default: hipLaunchKernelGGL((k_faces<kModeVertex>), grid(kFaceBlocks, nt), b, 0, st, a); break;
    }
    if (marks) (void)hipEventRecord(marks[1], st);
    if (a.vnormal) hipLaunchKernelGGL(k_normals, grid(kNormalBlocks, nv), b, 0, st, a);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_chunk_emit_batch_t(int mode, const JobArgs* jobs, const BlockRef* refs, uint32_t nrefs, hipStream_t st)
{
    const dim3 g(nrefs), b(kBlock);
    if (mode != kModeDup) hipLaunchKernelGGL((k_points_batch<T>), g, b, 0, st, jobs, refs);
    switch (mode) {
    case kModeDup: hipLaunchKernelGGL((k_dup_batch<T>), g, b, 0, st, jobs, refs); break;
    case kModePolygon: hipLaunchKernelGGL((k_faces_batch<kModePolygon>), g, b, 0, st, jobs, refs); break;
    default: hipLaunchKernelGGL((k_faces_batch<kModeVertex>), g, b, 0, st, jobs, refs); break;
    }
    if (mode == kModeVertex) hipLaunchKernelGGL(k_normals_batch, g, b, 0, st, jobs, refs);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_chunk_emit(int dtype, const JobArgs& a, hipStream_t st, hipEvent_t* marks)
{
    switch (dtype) {
    case 0: return launch_chunk_emit_t<int8_t>(a, st, marks);
    case 1: return launch_chunk_emit_t<int16_t>(a, st, marks);
    case 2: return launch_chunk_emit_t<int32_t>(a, st, marks);
    case 3: return launch_chunk_emit_t<int64_t>(a, st, marks);
    case 4: return launch_chunk_emit_t<uint8_t>(a, st, marks);
    case 5: return launch_chunk_emit_t<uint16_t>(a, st, marks);
    case 6: return launch_chunk_emit_t<uint32_t>(a, st, marks);
    case 7: return launch_chunk_emit_t<uint64_t>(a, st, marks);
    case 8: return launch_chunk_emit_t<float>(a, st, marks);
    default: return launch_chunk_emit_t<double>(a, st, marks);
    }
}

hipError_t launch_chunk_emit_batch(int dtype, int mode, const JobArgs* jobs, const BlockRef* refs, uint32_t nrefs,
                                   hipStream_t st)
{
    switch (dtype) {
    case 0: return launch_chunk_emit_batch_t<int8_t>(mode, jobs, refs, nrefs, st);
    case 1: return launch_chunk_emit_batch_t<int16_t>(mode, jobs, refs, nrefs, st);
    case 2: return launch_chunk_emit_batch_t<int32_t>(mode, jobs, refs, nrefs, st);
    case 3: return launch_chunk_emit_batch_t<int64_t>(mode, jobs, refs, nrefs, st);
    case 4: return launch_chunk_emit_batch_t<uint8_t>(mode, jobs, refs, nrefs, st);
    case 5: return launch_chunk_emit_batch_t<uint16_t>(mode, jobs, refs, nrefs, st);
    case 6: return launch_chunk_emit_batch_t<uint32_t>(mode, jobs, refs, nrefs, st);
    case 7: return launch_chunk_emit_batch_t<uint64_t>(mode, jobs, refs, nrefs, st);
    case 8: return launch_chunk_emit_batch_t<float>(mode, jobs, refs, nrefs, st);
    default: return launch_chunk_emit_batch_t<double>(mode, jobs, refs, nrefs, st);
    }
}

}  // namespace kmc
