/*
 * kmc_chunks.h -- device code of the chunk-batch emit: the walk over a level's
 * busy chunks and the listing of their triangles.
 */
#pragma once
#include "kmc_device.h"
#include "kmc_plan.h"

#pragma clang fp contract(off)

namespace kmc {

/* One level of a pass; the same on all lanes. */
struct EmitLevel {
    const uint64_t* bits;    // [nz][ny][NC] chunk masks
    const uint32_t* vp;      // in-row chunk prefixes
    const uint32_t* tp;
    const uint64_t* pv;      // row prefixes
    const uint64_t* pt;
    uint64_t v0, t0;         // first prefix of each (outputs index from 0)
    uint32_t wave;           // this wave among the level's
};

__device__ __forceinline__ EmitLevel emit_level(const JobArgs& a, uint32_t l, uint32_t block)
{
    const uint64_t words = (uint64_t)l * (a.nrows * a.NC);
    EmitLevel L;
    L.bits = a.bitvol + words;
    L.vp = a.vpc + words;
    L.tp = a.tpc + words;
    L.pv = a.prefix + (uint64_t)(l * 2 + 0) * a.nrows;
    L.pt = a.prefix + (uint64_t)(l * 2 + 1) * a.nrows;
    L.v0 = L.pv[0];
    L.t0 = L.pt[0];
    L.wave = block * (uint32_t)kWaves + uniform(threadIdx.x >> 6);
    return L;
}

/* A chunk's in-row prefix among the bits of its word (kHalfBusy, kWordBusy). */
__device__ __forceinline__ uint32_t prefix_mask(const JobArgs& a) { return a.NC <= 64 ? kHalfBusy - 1u : kWordBusy - 1u; }

__device__ __forceinline__ uint32_t triangles_before(const JobArgs& a, const EmitLevel& L, uint64_t w)
{
    return (a.NC <= 64 ? L.vp[w] >> 16 : L.tp[w]) & prefix_mask(a);
}

/* Calls batch(n) for every group of n <= N chunks of the level with a
 * crossing edge (V) or a triangle (!V), queued in q[0 .. n) (emit_queued;
 * chunk_place tells where they lie; q: N + 64 entries).  The words of kScan units
 * are in flight together, since the test of a unit is one dependent load.
 * Across a batch only a bit per unit stays live in a lane. */
constexpr uint32_t kScan = 4;

template <bool V, uint32_t N, typename F>
__device__ __forceinline__ void busy_chunks(const JobArgs& a, const EmitLevel& L, uint32_t* q, F&& batch)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t nwaves = a.ewaves, words = a.nrows * a.NC;
    const bool packed = a.NC <= 64;        // vertices in the low, triangles in the high half of vpc
    const uint32_t* pre = V || packed ? L.vp : L.tp;
    const uint32_t bit = V && packed ? kHalfBusy : kWordBusy;
    const uint32_t wave = L.wave;
    uint32_t qn = 0, step = 0;
    for (uint64_t u0 = wave < a.ewaves ? wave : a.eunits; u0 < a.eunits; u0 += nwaves * kScan, step += kScan) {
        uint32_t p[kScan];
        /* (opaque, so that nothing made of it stays in a register over the batches) */
        uint32_t slot = lane;
        asm volatile("" : "+v"(slot));
        const bool on = lane_piece(a, slot) < a.eparts && lane_chunk(a, slot) < a.NC;
        /* a unit's first piece, whole rows: lanes lie `off` words on from it */
        const uint64_t piece = (uint64_t)a.NC << (a.plog - a.eshift);
        const uint64_t off = lane_piece(a, slot) * (a.edist * piece) + lane_row(a, slot) * a.NC + lane_chunk(a, slot);
        /* steps left: most walks of a small volume have one or two */
        uint32_t n_left = 1;
#pragma unroll
        for (uint32_t k = 1; k < kScan; ++k) n_left += u0 + k * nwaves < a.eunits ? 1u : 0u;
#pragma unroll
        for (uint32_t k = 0; k < kScan; ++k) {
            p[k] = 0u;
            if (k < n_left) {
                const uint64_t u = u0 + k * nwaves;
                uint64_t w = u * (a.ehop * piece) + off;
                if (a.esegs > 1) {
                    const EmitSlot s = emit_slot(a, u, slot);
                    w = s.chunk < a.NC ? s.row * a.NC + s.chunk : words;
                }
                if (on && w < words) p[k] = pre[w];
            }
        }
        uint32_t busy = 0;
#pragma unroll
        for (uint32_t k = 0; k < kScan; ++k) busy |= (p[k] & bit) ? 1u << k : 0u;
        const bool last = u0 + nwaves * kScan >= a.eunits;
#pragma unroll 1
        for (uint32_t k = 0; k < n_left; ++k) {
            const uint64_t bm = __ballot((busy >> k) & 1u);
            if ((bm >> lane) & 1ull) q[qn + lanes_below(bm)] = emit_queued(step + k, lane);
            qn += (uint32_t)__popcll(bm);
            const bool end = last && k == n_left - 1;
            while (qn >= N || (end && qn)) {
                wave_sync();
                const uint32_t n = qn < N ? qn : N;
                batch(n);
                wave_sync();
                /* the rest (at most 63) moves to the front */
                qn -= n;
                const uint32_t rest = q[N + lane];
                wave_sync();
                if (lane < qn) q[lane] = rest;
                wave_sync();
            }
        }
    }
}

/* Row, its y and z, and chunk of the row of a queued slot of this wave. */
__device__ __forceinline__ void chunk_place(const JobArgs& a, const EmitLevel& L, uint32_t queued, uint64_t& r, uint32_t& y, uint32_t& z, uint32_t& c)
{
    const EmitSlot s = emit_slot(a, emit_unit(a, L.wave, queued), queued & 63u);
    r = s.row;
    c = s.chunk;
    row_place(a, r, y, z);
}

/* Lists the set bits of the masks of lanes `fit` as lane | bit << 6, each lane's
 * from list[excl - start] on.  Dense masks one after the other, a bit per lane
 * (about 10 instructions a mask); sparse ones all at once, each lane walking
 * its own (as many per bit of the fullest mask). */
__device__ __forceinline__ void list_bits(uint64_t mask, uint32_t excl, uint32_t start, uint64_t fit, bool dense,
                                          uint16_t* list)
{
    const uint32_t lane = threadIdx.x & 63u;
    if (dense) {
        for (uint64_t f = fit; f; f &= f - 1) {
            const int q = __builtin_ctzll(f);
            const uint64_t m = readlane64(mask, q);
            const uint32_t p = (uint32_t)__builtin_amdgcn_readlane((int)excl, q) - start + lanes_below(m);
            if (__builtin_amdgcn_inverse_ballot_w64(m)) list[p] = (uint16_t)((uint32_t)q | lane << 6);
        }
    } else if ((fit >> lane) & 1ull) {
        uint64_t m = mask;
        uint32_t p = excl - start;
        while (m) {
            const uint32_t i = (uint32_t)__ffsll((unsigned long long)m) - 1u;
            m &= m - 1ull;
            list[p++] = (uint16_t)(lane | i << 6);
        }
    }
}

/* Two neighbouring mask words in one load.  A row's last chunk has no next
 * one: its second word is the next row's or lies in the 16 bytes allocated past
 * the bit volume, and only reaches node / cell 64c + 63, which is at or past nx
 * - 1 there. */
__device__ __forceinline__ void load_words(const uint64_t* p, uint64_t& a, uint64_t& b)
{
    struct __attribute__((packed, aligned(8))) Words { uint64_t a, b; };
    const Words v = *(const Words*)p;
    a = v.a;
    b = v.b;
}

/* The cells of chunk c of cell row (y, z - 1), which lies in the volume: active
 * cells, the masks of their four node rows and the next chunk's first node of
 * each (RowChunk's act, k0, k3, k4, k7, next). */
struct CellMasks {
    uint64_t act, k0, k3, k4, k7;
    uint32_t next;
};

__device__ __forceinline__ CellMasks cell_masks(const JobArgs& a, uint32_t c, uint64_t k0, uint64_t n0, uint64_t k3,
                                                uint64_t n3, uint64_t k4, uint64_t n4, uint64_t k7, uint64_t n7)
{
    CellMasks o;
    const uint64_t c1 = k0 >> 1 | n0 << 63, c2 = k3 >> 1 | n3 << 63, c5 = k4 >> 1 | n4 << 63, c6 = k7 >> 1 | n7 << 63;
    o.act = ((k0 | c1 | c2 | k3 | k4 | c5 | c6 | k7) & ~(k0 & c1 & c2 & k3 & k4 & c5 & c6 & k7)) & valid_mask(c, a.nx - 1);
    o.k0 = k0;
    o.k3 = k3;
    o.k4 = k4;
    o.k7 = k7;
    o.next = (uint32_t)(n0 & 1ull) | (uint32_t)(n3 & 1ull) << 1 | (uint32_t)(n4 & 1ull) << 2 | (uint32_t)(n7 & 1ull) << 3;
    return o;
}

__device__ __forceinline__ CellMasks load_cells(const JobArgs& a, const EmitLevel& L, uint32_t y, uint32_t z, uint32_t c)
{
    const uint64_t* p = L.bits + ((uint64_t)(z - 1) * a.ny + y) * a.NC + c;
    const uint64_t* q = p + (uint64_t)a.ny * a.NC;
    uint64_t k0, n0, k3, n3, k4, n4, k7, n7;
    load_words(p, k0, n0);
    load_words(p + a.NC, k3, n3);
    load_words(q, k4, n4);
    load_words(q + a.NC, k7, n7);
    return cell_masks(a, c, k0, n0, k3, n3, k4, n4, k7, n7);
}

/* corner_pairs of cell i of a chunk whose masks lie in LDS. */
template <uint32_t N>
__device__ __forceinline__ uint32_t corner_pairs_at(const uint64_t (&m)[4][N], const uint32_t (&next)[N], uint32_t q,
                                                    uint32_t i)
{
    RowChunk o;
    o.k0 = m[0][q];
    o.k3 = m[1][q];
    o.k4 = m[2][q];
    o.k7 = m[3][q];
    o.next = next[q];
    return corner_pairs(o, i);
}

/* ------------------------------------------------------------------------- */
/* triangles of queued chunks, one per lane                                    */
/* ------------------------------------------------------------------------- */

constexpr uint32_t kChunks = 32;         // chunks worked on at a time
constexpr uint32_t kCellList = 192;      // active cells listed at once (a chunk has at most 64)

/* LDS of one wave.  Kept small: the kernels built on it wait for memory, and
 * run the faster the more waves a CU holds. */
struct ListLds {
    uint64_t out[kChunks];       // output id of each chunk's first triangle, then that id - its batch rank
    uint32_t q[kChunks + 64];    // busy queue: at most kChunks - 1 left over and 64 new
    uint32_t cell[64];           // the cells in work: chunk | cell << 6 | pair index << 12
    uint16_t cells[kCellList];   // chunk | cell << 6
    uint16_t tl[320];            // their triangles: cell in work | t << 6
};

/* The triangles of the n queued chunks.  masks(row, y, z, chunk of the row, id
 * of the first triangle) gives each chunk's active cells, on a lane of its own;
 * pair(chunk, cell) a cell's case as corner_pairs gives it; cell_of(chunk, cell,
 * case, batch rank of its first triangle) is called for each active cell; and
 * emit(count, batch rank) for up to 320 listed triangles at a time, s.tl[0 ..
 * count).  A triangle's output id is s.out[chunk] + its batch rank (in cell_of
 * and emit).  tri: case table by pair, the triangle count in the top nibble. */
template <typename C, typename P, typename K, typename F>
__device__ __forceinline__ void list_triangles(const JobArgs& a, const EmitLevel& L, const uint64_t* tri, ListLds& s,
                                               uint32_t n, C&& masks, P&& pair, K&& cell_of, F&& emit)
{
    const uint32_t lane = threadIdx.x & 63u;
    uint64_t act = 0;
    if (lane < n) {
        uint64_t r;
        uint32_t y, z, c;
        chunk_place(a, L, s.q[lane], r, y, z, c);
        const uint64_t w = r * a.NC + c;
        const uint64_t base = (L.pt[r] - L.t0) + triangles_before(a, L, w);
        act = masks(r, y, z, c, base);
        s.out[lane] = base;
    }
    const uint32_t incl = wave_incl_scan((uint32_t)__popcll(act));
    const uint32_t excl = incl - (uint32_t)__popcll(act);
    const uint32_t total = uniform((uint32_t)__builtin_amdgcn_readlane((int)incl, 63));
    uint32_t done = 0;                     // triangles emitted
    for (uint32_t start = 0; start < total;) {
        /* chunks whose cells fit the list */
        const uint64_t fit = __ballot(excl >= start && incl - start <= kCellList && act != 0);
        const uint32_t stop = uniform((uint32_t)__builtin_amdgcn_readlane((int)incl, 63 - __builtin_clzll(fit)));
        list_bits(act, excl, start, fit, total > 8 * n, s.cells);
        wave_sync();
        const uint32_t ncells = stop - start;
        for (uint32_t k0 = 0; k0 < ncells; k0 += 64) {
            const uint32_t k = k0 + lane;
            uint32_t cell = 0, q = 0, pi = 0, nt = 0;
            bool first = false;
            if (k < ncells) {
                cell = s.cells[k];
                q = cell & 63u;
                first = k == 0 || (s.cells[k - 1] & 63u) != q;
                pi = pair(q, cell >> 6);
                nt = (uint32_t)(tri[pi] >> 60);
            }
            const uint32_t inc = wave_incl_scan(nt);
            const uint32_t at = inc - nt;
            if (first) s.out[q] -= (uint64_t)(done + at);
            wave_sync();
            if (k < ncells) {
                cell_of(q, cell >> 6, pi, done + at);
                s.cell[lane] = cell | pi << 12;
                for (uint32_t t = 0; t < nt; ++t) s.tl[at + t] = (uint16_t)(lane | t << 6);
            }
            const uint32_t cnt = uniform((uint32_t)__builtin_amdgcn_readlane((int)inc, 63));
            wave_sync();
            emit(cnt, done);
            wave_sync();
            done += cnt;
        }
        start = stop;
    }
}

}  // namespace kmc
