/*
 * kmc_job.h -- the argument block of one extraction job and the layout of
 * the per-workgroup LDS state, shared by host launch code and kernels.
 *
 * A job is one structured volume with up to kMaxLevels isolevels extracted in
 * the same pass (each level yields its own surface, identical to what a
 * separate kvs::MarchingCubes call at that level would return).
 *
 * Geometry of the work decomposition (all in reference scan order, x fastest):
 *   - a *band* is R consecutive node rows [y0, y0+R) spanning the full x range;
 *   - a *tile* (z, b) is band b at step z.  It emits the triangles of the
 *     cells of band b at cell slice z-1 and the vertices of the crossing edges
 *     whose low node lies in the band at node slice z (or z-1 with
 *     VertexNormal, whose normals need the face normals of the cells on both
 *     sides of a slice).  Tiles in (z, b) order enumerate vertices in node
 *     scan order x {x,y,z}-edge and triangles in cell scan order, which is the
 *     order of calculate_isopoints and connect_isopoints /
 *     extract_surfaces_with_duplication in
 *     Source/Core/Visualization/Mapper/MarchingCubes.cpp:155-243,365-521;
 *   - a *unit* is one level of one band over a slab of `slab` consecutive
 *     steps.  The emit pass runs one unit at a time per wave (a *team*): the
 *     wave marches z through its unit with its own LDS region, keeping a ring
 *     of node-slice classification masks (one new slice loaded per step) and,
 *     with VertexNormal, a ring of the face normals of the last two cell
 *     slices.  Teams never wait for each other.
 *
 * Passes of one job: classify (stream the values once, write the bit volume),
 * count (per-row vertex / triangle counts and in-row chunk prefixes from the
 * bit volume), scan (row prefixes), emit (outputs at the prefixes; raw values
 * are read again only at the endpoints of crossing edges).  The emit works
 * on batches of chunks (kmc_emit.hip) unless y or z exceeds 2^20, when the tile
 * teams below do it.
 *
 * Within a slice, the classification bits of 64 consecutive nodes of a row
 * are held as one 64-bit mask per level (a *chunk*), built with one wave
 * ballot; edge crossings and cell activity are then bitwise operations on
 * chunks, and ranks are popcounts.
 */
#pragma once
#include <stdint.h>

namespace kmc {

constexpr int kMaxLevels = 8;
constexpr uint32_t kBitSlack = 16;   // bytes allocated past a bit volume (read, not used: load_words)
constexpr int kBlock = 256;          // threads per workgroup of the dense passes (4 waves of 64)
constexpr int kWaves = kBlock / 64;
constexpr int kEmitTeams = 4;        // emit workgroup: 4 independent one-wave teams
constexpr int kEmitBlock = 64 * kEmitTeams;
constexpr uint32_t kTableBytes = 256 * 8;   // case table at the start of the emit workgroup's LDS

/* In-row prefixes of a chunk: rows of at most 64 chunks keep both in a word of vpc,
 * vertices in the low and triangles in the high half, longer rows one in vpc and one in
 * tpc.  At most 63 chunks of 192 and 320 come before a chunk of such a row (14 and 15
 * bits), 2^14 of any row (23 bits): the top bit of each half, or word, says whether
 * the chunk itself has any. */
constexpr uint32_t kHalfBusy = 1u << 15, kWordBusy = 1u << 31;

struct JobArgs {
    const void* values;
    uint32_t nx, ny, nz;
    uint32_t R;        // node rows per band (emit tiles)
    uint32_t nb;       // number of bands, ceil(ny / R)
    uint32_t NC;       // 64-node chunks per row, ceil(nx / 64)
    uint32_t cshift;   // lanes are split into 64 >> cshift rows of (1 << cshift) chunk lanes
                       // (1 << cshift = the power of two >= min(NC, 64))
    uint32_t nlev;     // isolevels in this pass
    uint32_t slab;     // steps marched by one unit
    uint32_t nslabs;   // units per band, ceil(nz / slab)
    uint32_t dup;      // 1: duplicated vertices (per-triangle output)
    uint32_t vnormal;  // 1: VertexNormal (only without duplication)
    uint32_t queue_cap;
    uint32_t fn_cap;   // face normals held per cell slice (VertexNormal)
    uint32_t team_stride;  // bytes of LDS per team (>= the team layout's size)
    uint32_t teams;        // teams per emit workgroup (<= kEmitTeams; fewer when a team's LDS is large)
    uint64_t nunits;   // nlev * nb * nslabs
    // chunk-batch emit (kmc_plan.h): log2 of the chunk lanes of a row and of the
    // lanes of a piece; pieces per row and per unit; a level's units; pieces from
    // a unit to the next and between those of a unit; the waves that share a
    // level's units and their workgroups
    uint32_t eshift, plog, esegs, eparts;
    uint64_t eunits, ehop, edist;
    uint32_t ewaves, eblocks;
    double seg_inverse, ny_inverse;   // 1 / esegs, 1 / ny (div_by)
    uint64_t nrows;    // nz * ny: counts and prefixes are kept per node row
    double minv, maxv; // clamp range of the interpolation (volume min/max)
    float fminv, fmaxv;    // the same as floats ...
    uint32_t fclamp;       // ... 1: exactly, and minv <= maxv
    float minc[3];     // min object coordinate
    float sc[3];       // (max - min) / ncells, per axis (float ops, host side)
    double iso[kMaxLevels];
    float thr[kMaxLevels];    // float32 data: v > thr  <=>  double(v) > iso
    // counts[(l*2 + k) * nrows + z*ny + y], k = 0: vertices owned by node row
    // (y, z); k = 1: triangles of cell row (y, z-1)
    uint32_t* counts;
    // exclusive prefixes, same layout
    const uint64_t* prefix;
    // classification bit volume: bitvol[((l * nz + z) * ny + y) * NC + c] is the
    // 64-bit mask of nodes x in [64c, 64c+64) of row y, slice z, level l
    uint64_t* bitvol;
    // optional, same layout as bitvol: per chunk the exclusive prefix within its
    // row of the vertex counts (vpc) and of the triangle counts of cell row
    // (y, z-1) (tpc), and whether the chunk has any (chunk_words); written by the
    // count pass when non-null
    uint32_t* vpc;
    uint32_t* tpc;
    // VertexNormal: per triangle its face normal, per active cell its case and
    // first triangle (kmc_emit.hip); level l's start at toff[l]
    float* fn;
    uint32_t* crec;
    // VertexNormal: active cells of cell row (y, z-1), bit volume layout, written
    // for chunks with one
    uint64_t* act;
    uint64_t toff[kMaxLevels + 1];
    // per-level outputs
    float* coords[kMaxLevels];
    float* normals[kMaxLevels];
    uint32_t* conn[kMaxLevels];
    uint64_t cap_vertices[kMaxLevels];   // capacity in coordinate triples
    uint64_t cap_triangles[kMaxLevels];
    // SlicePlane: nodes classify by the plane's sign instead of their values;
    // each vertex gets the colour of the value interpolated along its edge
    float plane[4];            // coefficients: plane(x,y,z) = plane[0]*x + plane[1]*y + plane[2]*z + plane[3]
    const uint8_t* ctable;     // colour map table, 3 bytes per entry (device)
    uint32_t cres;             // entries of ctable
    float crange[2];           // colour map range
    uint8_t* colors;           // one RGB per vertex (9 bytes per triangle)
};

/* LDS layout of one team (one level); sizes in bytes, offsets 16-byte
 * aligned, relative to the team's region.  Node slices live in a ring of
 * 3 mask slots (slices z-1 .. z+1), each holding node rows y0-1 .. y0+R+1.  Window vertex
 * prefixes cover node slices z-1 and z and node rows y0-1 .. y0+R; cell data
 * cover cell slice z-1, cell rows y0-1 .. y0+R-1 (row 0 is the halo row of
 * the band above, used for face normals only), in a ring of 2 cell slices
 * with VertexNormal. */
struct LdsLayout {
    uint32_t nrb;       // mask rows held per slice: y0-1 .. y0+R+1
    uint32_t nslots;    // node-slice mask slots
    uint32_t ncs;       // cell-slice slots
    uint32_t off_bits;  // uint64 [nslots][nrb][NC]         classification masks
    uint32_t off_wpv;   // uint32 [2][R+2][NC]              window vertex chunk prefixes
    uint32_t off_act;   // uint64 [ncs][R+1][NC]            active cells
    uint32_t off_pt;    // uint32 [ncs][R+1][NC]            triangle chunk prefixes
    uint32_t off_ap;    // uint32 [ncs][R+1][NC]            active-cell chunk prefixes (VertexNormal)
    uint32_t off_crec;  // uint32 [ncs][fn_cap]             per active cell: first triangle << 8 | cube index
    uint32_t off_fn;    // float  [ncs][fn_cap][3]          face normals (VertexNormal)
    uint32_t off_vq;    // uint32 [queue_cap]               vertex work queue
    uint32_t off_tq;    // uint32 [queue_cap]               triangle work queue
    uint32_t bytes;
};

#if defined(__HIPCC__)
__host__ __device__
#endif
inline uint32_t align16(uint32_t x) { return (x + 15u) & ~15u; }

#if defined(__HIPCC__)
__host__ __device__
#endif
inline LdsLayout lds_layout(const JobArgs& a)
{
    LdsLayout L;
    const uint32_t R = a.R, NC = a.NC;
    L.nrb = R + 3;
    L.nslots = 3u;
    L.ncs = a.vnormal ? 2u : 1u;
    uint32_t o = 0;
    L.off_bits = o;  o = align16(o + L.nslots * L.nrb * NC * 8u);
    L.off_wpv = o;   o = align16(o + 2u * (R + 2) * NC * 4u);
    L.off_act = o;   o = align16(o + L.ncs * (R + 1) * NC * 8u);
    L.off_pt = o;    o = align16(o + L.ncs * (R + 1) * NC * 4u);
    L.off_ap = o;    o = align16(o + (a.vnormal ? L.ncs * (R + 1) * NC * 4u : 0u));
    L.off_crec = o;  o = align16(o + (a.vnormal ? L.ncs * a.fn_cap * 4u : 0u));
    L.off_fn = o;    o = align16(o + (a.vnormal ? L.ncs * a.fn_cap * 12u : 0u));
    L.off_vq = o;    o = align16(o + a.queue_cap * 4u);
    L.off_tq = o;    o = align16(o + a.queue_cap * 4u);
    L.bytes = o;
    return L;
}

/* LDS of an emit workgroup of `teams` teams, team_stride bytes apart. */
#if defined(__HIPCC__)
__host__ __device__
#endif
inline uint32_t emit_lds_bytes(uint32_t team_stride, uint32_t teams) { return kTableBytes + teams * team_stride; }

}  // namespace kmc
