/*
 * kmc_emit.hip -- emit of a pass in chunk batches (gfx950, wave64).
 *
 * After the count pass and the scan, the output position of everything a
 * 64-node chunk holds is known: row prefix + chunk prefix within the row.  A
 * wave walks the (row, chunk) pairs of one level, queues the chunks that hold
 * something in LDS and works on 64 of them at a time: each lane takes one
 * chunk's masks, the wave lists the chunks' active cells in LDS, and the
 * listed triangles are produced one per lane -- every lane busy whatever the
 * chunks hold, nothing but the outputs written.
 *
 * Output order: cells in scan order, triangles in table order
 * (extract_surfaces_with_duplication,
 * Source/Core/Visualization/Mapper/MarchingCubes.cpp:155-243).
 */
#include <hip/hip_runtime.h>
#include <algorithm>
#include <type_traits>
#include "kmc_device.h"
#include "kmc_internal.h"
#include "kmc_job.h"

#pragma clang fp contract(off)

namespace kmc {

namespace {

/* One level of a pass; the same on all lanes. */
struct EmitLevel {
    const uint64_t* bits;    // [nz][ny][NC] chunk masks
    const uint32_t* vp;      // in-row chunk prefixes (chunk_prefix)
    const uint32_t* tp;
    const uint32_t* cv;      // row counts: crossing edges, triangles
    const uint32_t* ct;
    const uint64_t* pv;      // row prefixes
    const uint64_t* pt;
    uint64_t v0, t0;         // first prefix of each (outputs index from 0)
};

__device__ __forceinline__ EmitLevel emit_level(const JobArgs& a, uint32_t l)
{
    const uint64_t words = (uint64_t)l * (a.nrows * a.NC);
    EmitLevel L;
    L.bits = a.bitvol + words;
    L.vp = a.vpc + words;
    L.tp = a.tpc + words;
    L.cv = a.counts + (uint64_t)(l * 2 + 0) * a.nrows;
    L.ct = a.counts + (uint64_t)(l * 2 + 1) * a.nrows;
    L.pv = a.prefix + (uint64_t)(l * 2 + 0) * a.nrows;
    L.pt = a.prefix + (uint64_t)(l * 2 + 1) * a.nrows;
    L.v0 = L.pv[0];
    L.t0 = L.pt[0];
    return L;
}

/* Calls batch(n) for every group of n <= N chunks of the level with a
 * crossing edge (V) or a triangle (!V), their entries, row | chunk << 40,
 * in q[0 .. n) (q: N + 64 entries).  A wave
 * takes units of a.erows rows x up to 64 chunks; the prefixes of kScan units
 * are in flight together, since the test of a unit is one dependent load.
 * Across a batch only the units' busy masks stay live (scalars). */
constexpr uint32_t kScan = 4;

template <bool V, uint32_t N, typename F>
__device__ __forceinline__ void busy_chunks(const JobArgs& a, const EmitLevel& L, uint64_t* q, F&& batch)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t wave = (uint64_t)blockIdx.x * kWaves + uniform(threadIdx.x >> 6), nwaves = (uint64_t)a.eblocks * kWaves;
    const uint32_t sub = lane >> a.cshift;
    const uint64_t step = nwaves * a.erows;
    const bool packed = a.NC <= 64;        // vertices in the low, triangles in the high half of vpc
    const uint32_t* pre = V || packed ? L.vp : L.tp;
    const uint32_t* row_end = V ? L.cv : L.ct;
    const uint32_t sh = V || !packed ? 0u : 16u, mask = packed ? 0xFFFFu : ~0u;
    uint32_t qn = 0;
    for (uint32_t c0 = 0; c0 < a.NC; c0 += 64) {
        const uint32_t c = c0 + (lane & ((1u << a.cshift) - 1u));
        const bool in = sub < a.erows && c < a.NC;
        const bool row_last = c + 1 == a.NC;
        for (uint64_t r0 = wave * a.erows; r0 < a.nrows; r0 += step * kScan) {
            uint32_t p0[kScan], p1[kScan];
#pragma unroll
            for (uint32_t k = 0; k < kScan; ++k) {
                const uint64_t r = r0 + k * step + sub;
                p0[k] = p1[k] = 0u;
                if (in && r < a.nrows) {
                    const uint64_t w = r * a.NC + c;
                    p0[k] = (pre[w] >> sh) & mask;
                    p1[k] = row_last ? row_end[r] : (pre[w + 1] >> sh) & mask;
                }
            }
            uint64_t busy[kScan];
#pragma unroll
            for (uint32_t k = 0; k < kScan; ++k) busy[k] = __ballot(p0[k] != p1[k]);
#pragma unroll 1
            for (uint32_t k = 0; k < kScan; ++k) {
                uint64_t bm = busy[0];
#pragma unroll
                for (uint32_t j = 1; j < kScan; ++j) bm = k == j ? busy[j] : bm;
                if ((bm >> lane) & 1ull) q[qn + lanes_below(bm)] = (r0 + k * step + sub) | (uint64_t)c << 40;
                qn += (uint32_t)__popcll(bm);
                const bool end = r0 + step * kScan >= a.nrows && k == kScan - 1;
                while (qn >= N || (end && qn)) {
                    wave_sync();
                    const uint32_t n = qn < N ? qn : N;
                    batch(n);
                    wave_sync();
                    /* the rest (at most 63) moves to the front */
                    qn -= n;
                    const uint64_t rest = q[N + lane];
                    wave_sync();
                    if (lane < qn) q[lane] = rest;
                    wave_sync();
                }
            }
        }
    }
}

/* Row and slice of row index r. */
__device__ __forceinline__ void row_yz(const JobArgs& a, uint64_t r, uint32_t& y, uint32_t& z)
{
    if (a.nrows <= 0xFFFFFFFFull) {
        z = (uint32_t)r / a.ny;
        y = (uint32_t)r - z * a.ny;
    } else {
        const uint64_t zz = r / a.ny;
        z = (uint32_t)zz;
        y = (uint32_t)(r - zz * a.ny);
    }
}

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

/* The tables, evaluated at compile time (a workgroup only copies them).  M:
 * table orientation of the edges with duplicated vertices (:276-290 of
 * MarchingCubesTable.cpp), else low to high. */
constexpr uint64_t kTableWords[256] = { KMC_TABLE_WORDS };

constexpr uint32_t bits_below(uint32_t m, uint32_t e)
{
    uint32_t n = 0;
    for (uint32_t k = 0; k < e; ++k) n += (m >> k) & 1u;
    return n;
}

constexpr CaseLds make_cases(bool table_edges)
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
        const uint32_t first = table_edges ? p : p & q, second = table_edges ? q : p | q;
        t.ends[e] = EdgeEnds{ (float)(first & 1u), (float)((first >> 1) & 1u), (float)(first >> 2),
                              first << 6 | second << 19 | ((second & axis) ? 8u : 0u) | axis };
    }
    return t;
}

static __constant__ CaseLds d_cases_dup = make_cases(true);

__device__ __forceinline__ void stage_cases(CaseLds& t, const CaseLds& from)
{
    static_assert(sizeof(CaseLds) % 16 == 0, "copied in 16-byte words");
    for (uint32_t i = threadIdx.x; i < sizeof(CaseLds) / 16; i += kBlock) ((uint4*)&t)[i] = ((const uint4*)&from)[i];
    __syncthreads();
}

/* LDS of one wave of the triangle kernels: 9.6 kB with values of up to 32
 * bits, so that four workgroups fit a CU's 160 KiB. */
constexpr uint32_t kChunks = 32;         // chunks worked on at a time
constexpr uint32_t kCellList = 320;      // active cells listed at once (a chunk has at most 64)
constexpr uint32_t kVerts = 236;         // edge crossings of the up to 64 cells in work (a cell has at most 12)

struct CellPos { float x, y, z; };         // exact: coordinates lie below 2^24

template <typename T>
struct CellLds {
    uint64_t q[kChunks + 64];    // busy queue: at most kChunks - 1 left over and 64 new
    uint64_t m[4][kChunks];      // k0, k3, k4, k7 of each chunk (RowChunk)
    uint64_t out[kChunks];       // output id - batch rank of each chunk's triangles (its first array's address with
    uint64_t out2[kChunks];      // duplicated vertices, the second one's here)
    uint64_t key[kChunks];       // 64 c | y << 20 | z << 40 of each chunk's first cell
    CellPos cpos[64];            // the cells in work
    uint32_t next[kChunks];
    float p[kVerts][3];          // crossing points of the cells in work
    uint16_t el[kVerts];         // crossing: cell | edge << 6
    uint16_t cells[kCellList];   // chunk | cell << 6
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
    RowChunk m;
    m.k0 = s.m[0][q];
    m.k3 = s.m[1][q];
    m.k4 = s.m[2][q];
    m.k7 = s.m[3][q];
    m.next = s.next[q];
    const uint32_t pi = corner_pairs(m, i);
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
        const uint64_t e = s.q[lane];
        const uint64_t r = e & 0xFFFFFFFFFFull;
        const uint32_t c = (uint32_t)(e >> 40);
        uint32_t y, z;
        row_yz(a, r, y, z);
        RowChunk o;
        row_chunk(a, L.bits, y, z, c, o);
        const uint64_t w = r * a.NC + c;
        act = o.act;
        s.m[0][lane] = o.k0;
        s.m[1][lane] = o.k3;
        s.m[2][lane] = o.k4;
        s.m[3][lane] = o.k7;
        s.next[lane] = o.next;
        s.key[lane] = (uint64_t)(c * 64u) | (uint64_t)y << 20 | (uint64_t)(z - 1) << 40;
        s.out[lane] = (L.pt[r] - L.t0) + (a.NC <= 64 ? L.vp[w] >> 16 : L.tp[w]);
    }
    const uint32_t incl = wave_incl_scan((uint32_t)__popcll(act));
    const uint32_t excl = incl - (uint32_t)__popcll(act);
    const uint32_t total = uniform((uint32_t)__builtin_amdgcn_readlane((int)incl, 63));
    uint32_t rank = 0;
    for (uint32_t start = 0; start < total;) {
        /* chunks whose cells fit the list */
        const uint64_t fit = __ballot(excl >= start && incl - start <= kCellList && act != 0);
        const uint32_t stop = uniform((uint32_t)__builtin_amdgcn_readlane((int)incl, 63 - __builtin_clzll(fit)));
        if ((fit >> lane) & 1ull) {
            uint64_t m = act;
            uint32_t p = excl - start;
            while (m) {
                const uint32_t i = (uint32_t)__ffsll((unsigned long long)m) - 1u;
                m &= m - 1ull;
                s.cells[p++] = (uint16_t)(lane | i << 6);
            }
        }
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
__device__ __forceinline__ void dup_level(const JobArgs& a, uint32_t l, const CaseLds& tab, CellLds<T>& s)
{
    if (!a.cap_triangles[l]) return;       // a level without outputs
    const uint32_t lane = threadIdx.x & 63u;
    const EmitLevel L = emit_level(a, l);
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
    dup_level<T>(a, blockIdx.y, tab, s[threadIdx.x >> 6]);
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_dup_batch(const JobArgs* jobs)
{
    __shared__ CaseLds tab;
    __shared__ CellLds<T> s[kWaves];
    const JobArgs& a = jobs[blockIdx.z];
    if (blockIdx.y >= a.nlev || blockIdx.x >= a.eblocks) return;
    stage_cases(tab, d_cases_dup);
    dup_level<T>(a, blockIdx.y, tab, s[threadIdx.x >> 6]);
}

template <typename T>
hipError_t launch_dup_t(const JobArgs& a, hipStream_t st)
{
    hipLaunchKernelGGL((k_dup<T>), dim3(a.eblocks, a.nlev), dim3(kBlock), 0, st, a);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_dup_batch_t(const JobArgs* jobs, uint32_t njobs, uint32_t blocks, uint32_t levels, hipStream_t st)
{
    constexpr uint32_t kMaxJobs = 32768;   // of one grid's z
    for (uint32_t j = 0; j < njobs; j += kMaxJobs)
        hipLaunchKernelGGL((k_dup_batch<T>), dim3(blocks, levels, std::min(kMaxJobs, njobs - j)), dim3(kBlock), 0, st,
                           jobs + j);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_dup(int dtype, const JobArgs& a, hipStream_t st)
{
    switch (dtype) {
    case 0: return launch_dup_t<int8_t>(a, st);
    case 1: return launch_dup_t<int16_t>(a, st);
    case 2: return launch_dup_t<int32_t>(a, st);
    case 3: return launch_dup_t<int64_t>(a, st);
    case 4: return launch_dup_t<uint8_t>(a, st);
    case 5: return launch_dup_t<uint16_t>(a, st);
    case 6: return launch_dup_t<uint32_t>(a, st);
    case 7: return launch_dup_t<uint64_t>(a, st);
    case 8: return launch_dup_t<float>(a, st);
    default: return launch_dup_t<double>(a, st);
    }
}

hipError_t launch_dup_batch(int dtype, const JobArgs* jobs, uint32_t njobs, uint32_t blocks, uint32_t levels,
                            hipStream_t st)
{
    switch (dtype) {
    case 0: return launch_dup_batch_t<int8_t>(jobs, njobs, blocks, levels, st);
    case 1: return launch_dup_batch_t<int16_t>(jobs, njobs, blocks, levels, st);
    case 2: return launch_dup_batch_t<int32_t>(jobs, njobs, blocks, levels, st);
    case 3: return launch_dup_batch_t<int64_t>(jobs, njobs, blocks, levels, st);
    case 4: return launch_dup_batch_t<uint8_t>(jobs, njobs, blocks, levels, st);
    case 5: return launch_dup_batch_t<uint16_t>(jobs, njobs, blocks, levels, st);
    case 6: return launch_dup_batch_t<uint32_t>(jobs, njobs, blocks, levels, st);
    case 7: return launch_dup_batch_t<uint64_t>(jobs, njobs, blocks, levels, st);
    case 8: return launch_dup_batch_t<float>(jobs, njobs, blocks, levels, st);
    default: return launch_dup_batch_t<double>(jobs, njobs, blocks, levels, st);
    }
}

}  // namespace kmc
