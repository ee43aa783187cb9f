/*
 * kmc_plan.h -- how the slots (node row, 64-node chunk) of a level are dealt to
 * the waves of the chunk-batch emit, which form classifies a volume, and how a
 * batch's workgroups are dealt to its passes.  Plain C++, shared by the host's
 * planning, the kernels and the host-side tests.
 *
 * A *piece* is a run of up to 16 lanes' slots: 8 or 16 chunks of a row, or all
 * chunks of one or more short rows.  A *unit*, what a wave looks at in one step,
 * is a.eparts pieces, side by side or equal distances apart over the level.  Wave w
 * takes units w, w + waves, w + 2 waves, ...; a slot is known to its wave by
 * the step and the lane alone, so 32 bits name it in volumes of any number of rows.
 */
#pragma once
#include <stdint.h>
#include <algorithm>
#include <vector>
#include "kmc_job.h"

#if defined(__HIPCC__)
#define KMC_HD __host__ __device__
#else
#define KMC_HD
#endif

namespace kmc {

/* x / d of integers through the double 1 / d, without an integer division's 20
 * instructions (100 in 64 bits): (x + 1/2) / d lies at least 1 / (2 d) off every
 * integer, and the product is off by less than x / d * 2^-51.  x / d * d stays
 * below 2^45 here: rows are at most 2^40, and parts of rows as few as masks fit
 * a device. */
KMC_HD inline uint64_t div_by(uint64_t x, double inverse) { return (uint64_t)(((double)x + 0.5) * inverse); }

/* What a lane looks at: the piece of the unit, the row of the piece and the chunk of
 * the row's part.  Pieces from a.eparts on, chunks past the row and rows past the
 * last hold nothing. */
KMC_HD inline uint32_t lane_piece(const JobArgs& a, uint32_t lane) { return lane >> a.plog; }
KMC_HD inline uint32_t lane_row(const JobArgs& a, uint32_t lane) { return (lane & ((1u << a.plog) - 1u)) >> a.eshift; }
KMC_HD inline uint32_t lane_chunk(const JobArgs& a, uint32_t lane) { return lane & ((1u << a.eshift) - 1u); }

struct EmitSlot {
    uint64_t row;
    uint32_t chunk;
};

KMC_HD inline EmitSlot emit_slot(const JobArgs& a, uint64_t unit, uint32_t lane)
{
    EmitSlot s;
    uint64_t group = unit * a.ehop + lane_piece(a, lane) * a.edist;
    s.chunk = lane_chunk(a, lane);
    if (a.esegs > 1) {
        const uint64_t piece = group;
        group = div_by(piece, a.seg_inverse);
        s.chunk += (uint32_t)(piece - group * a.esegs) << a.eshift;
    }
    s.row = (group << (a.plog - a.eshift)) + lane_row(a, lane);
    return s;
}

/* A slot as its wave queues it, and the unit that it came from. */
KMC_HD inline uint32_t emit_queued(uint32_t step, uint32_t lane) { return step << 6 | lane; }

KMC_HD inline uint64_t emit_unit(const JobArgs& a, uint32_t wave, uint32_t queued)
{
    return wave + (uint64_t)(queued >> 6) * a.ewaves;
}

/* Node row -> (y, z). */
KMC_HD inline void row_place(const JobArgs& a, uint64_t row, uint32_t& y, uint32_t& z)
{
    z = (uint32_t)div_by(row, a.ny_inverse);
    y = (uint32_t)row - z * a.ny;
}

/* The largest prime <= n (n >= 2). */
inline uint32_t prime_below(uint32_t n)
{
    for (;; --n) {
        bool prime = n >= 2;
        for (uint32_t d = 2; prime && (uint64_t)d * d <= n; ++d) prime = n % d != 0;
        if (prime) return n;
    }
}

/* Wave steps of 64 (row, chunk) pairs that a pass's levels hold. */
inline uint64_t emit_steps(const JobArgs& a)
{
    const uint64_t G = 64u >> a.cshift;
    return std::max(1u, a.nlev) * ((a.nrows + G - 1) / G * ((a.NC + 63) / 64));
}

/* Waves of a launch: as many as the device holds of the kernel at once, and up
 * to eight times that while each still has four full steps -- the later ones
 * even out a large pass (1024^3 float turbulence, three levels, triangles /
 * normals: 1666 / 1240 us with one time, 1367 / 1205 with two, 1250 / 1129
 * with eight, 1277 / 1162 with sixteen; a half-filled round costs: 512^3 CT
 * triangles 287 us with one time, 338 with 1.6) -- and no more than one per 32
 * outputs, but as many as leave none a walk of more than 16 steps: a small
 * surface in a large volume is all walking (a sphere of radius 4 in 1024^3,
 * vertex normals: 3390 us a call by outputs alone, 995 with 32 steps, 890 with 16). */
constexpr uint64_t kEmitRounds = 8, kEmitItems = 32, kEmitWalk = 16;

/* Workgroups of the duplicated triangles' kernel that a CU's LDS holds, by the size of
 * the values it stages (kmc_emit.hip checks it).  A grid for four of them where three
 * fit takes a round and a third: 512^3 double CT 770 us a call, so 705. */
constexpr uint32_t dup_blocks(uint32_t value_size) { return value_size == 8 ? 3u : 4u; }

/* Split of the chunk-batch emit (rows planned; a.nlev set) of a pass whose emit
 * shares its launch with others, `all` being the sum of their emit_steps, for a
 * kernel of which a CU holds per_cu workgroups and that produces `items` outputs
 * (0: not known yet).
 *
 * A wave takes 64 slots a step, but at most a quarter of its share of the pass:
 * four steps far apart even the waves out (256^3 blobs, duplicated: 26 us, 36
 * with two steps).  Where every chunk holds many outputs there is nothing to
 * even out, and two steps keep the batches full (320 x 288 x 256 CT, vertices:
 * 38 us, 42 with four).  Rows of 64 chunks and more are cut down to 8 of them a
 * step: few rows of full chunks are long chains of work (9000 x 40 x 33 blobs,
 * vertex normals: 270 us a call with a row's 64 chunks a step, 190 with 16, 146
 * with 8).
 *
 * Pieces far apart share a sheet out (a plane of one z in 1024^3, vertex normals:
 * 1184 us a call with pieces side by side, 943 so), pieces side by side share
 * cache lines of neighbouring rows and slices, which counts where those of a
 * slice do not stay in the L2 (1024^3 turbulence, three levels: 4150 us side by
 * side, 4670 far apart; 512^3 CT 820 and 812): side by side only in volumes of
 * 2^22 slots and more a level with an output in every sixth of them, and in rows
 * that are cut anyway (6000 x 150 x 120 blobs, vertex normals: 224 and 244).
 *
 * The number of waves is made prime where they take several steps, so that no period of
 * the rows meets the same waves again and again (a plane of one y in 1024^3, whose rows
 * lie 1024 apart: 128 of 32768 waves had all of it, 2990 us a call, 1360 so). */
inline void plan_emit(JobArgs& a, uint64_t all, uint32_t per_cu = 4, uint64_t items = 0)
{
    const uint64_t own = emit_steps(a), nlev = std::max(1u, a.nlev), slots = a.nrows * a.NC;
    const uint64_t resident = 256ull * kWaves * per_cu;
    uint64_t waves = resident * std::min(kEmitRounds, std::max<uint64_t>(1, all / 4 / resident));
    if (items) waves = std::min(waves, std::max<uint64_t>(256, std::max(items / kEmitItems, all / kEmitWalk)));
    else waves = std::max(waves, std::min(2 * resident, all / 4));   // a batch's uneven passes even out by themselves
    const uint64_t want = std::max<uint64_t>(1, (waves * own + all - 1) / all / nlev);   // waves per level
    const uint64_t steps = items > 4 * nlev * slots ? 2 : 4;
    a.eshift = std::min(a.cshift, 4u);
    a.plog = 4;
    a.eparts = 4;
    auto segs = [&] { return (a.NC + (1u << a.eshift) - 1) >> a.eshift; };
    auto pieces = [&] { return (((a.nrows - 1) >> (a.plog - a.eshift)) + 1) * segs(); };
    while (pieces() / a.eparts < steps * want && (a.eparts > 1 || a.plog > a.eshift)) {
        if (a.eparts > 1) a.eparts >>= 1;
        else --a.plog;
    }
    if (pieces() / a.eparts < 8 * want && a.NC >= 64) a.plog = a.eshift = 3;
    a.esegs = segs();
    a.seg_inverse = 1.0 / a.esegs;
    a.ny_inverse = 1.0 / a.ny;
    a.eunits = (pieces() + a.eparts - 1) / a.eparts | 1;   // odd: the pieces of a unit meet no period of the rows either
    const bool far = a.NC < 64 && (slots < 1u << 22 || (items && items / nlev < slots / 6));
    a.ehop = far ? 1 : a.eparts;
    a.edist = far ? a.eunits : 1;
    /* (a step's number has 26 bits in the queue) */
    const uint64_t least = (a.eunits >> 25) + 1;
    a.eblocks = (uint32_t)std::max<uint64_t>(1, (std::max(least, std::min(a.eunits, want)) + kWaves - 1) / kWaves);
    a.ewaves = a.eblocks * (uint32_t)kWaves;
    if (a.eunits > a.ewaves) a.ewaves = prime_below(a.ewaves);
}

/* Classification: 16 chunks of consecutive rows a wave (runs) or a row a wave.  A row
 * a wave leaves short rows few loads in flight, and with more rows than the device
 * holds waves that is what it waits for; runs spend some instructions per chunk
 * and level and store their masks in shorter pieces.  Row / run form, us:
 *   float, one level, 65536 rows of 4 / 8 / 12 / 16 chunks  25.2 / 30.2 / 39.0, 16.6 / 26.9 / 36.9; 86.8 and 87.3 at 2 GiB
 *   three levels, 4 / 5 / 6 / 12 chunks  28.6 / 30.6 / 32.4 / 45.9 and 25.0 / 29.8 / 34.4 / 61.8
 *   double, one level, 4 / 5 / 6 / 8 chunks  27.2 / 32.2 / 34.6 / 43.8 and 24.9 / 30.0 / 34.6 / 46.0
 *   uint16 (odd rows), three levels, 3 / 4 / 6 / 8 chunks  38.7 / 43.6 / 56.6 / 67.5 and 31.1 / 41.5 / 56.9 / 75.4
 *   five levels, 262144 rows of 4 chunks  float 300 and 351, double 163 and 183 (at 2^28 bytes a volume of 3 chunks 7 % slower, of 2 faster)
 *   one level, 1024 .. 8192 rows: the same within 0.5 us, uint16 6.6 and 7.5 */
inline bool classify_by_runs(const JobArgs& a, uint32_t value_size)
{
    constexpr uint32_t most[3][5] = { { 8, 6, 4, 2, 2 }, { 12, 6, 5, 4, 2 }, { 5, 5, 5, 4, 2 } };   // by levels, the last for five and more
    return a.nrows > 8192 && a.NC <= most[value_size <= 2 ? 0 : value_size / 4][std::min(a.nlev, 5u) - 1];
}

/* One workgroup of a launch over a batch's passes: its pass, its level (emit) and
 * which of the pass's (level's) workgroups it is. */
struct BlockRef {
    uint32_t job, level, block, blocks;
};

inline void add_blocks(std::vector<BlockRef>& out, uint32_t job, uint32_t level, uint64_t blocks)
{
    for (uint32_t i = 0; i < blocks; ++i) out.push_back(BlockRef{ job, level, i, (uint32_t)blocks });
}

/* Workgroups of a batch's front passes: as many as each pass has work for, or some
 * 16384 in all, dealt by that work.  (The same number for every pass left one
 * 512^3 volume among 255 of 32^3 to 64 workgroups: duplicated vertices, 645 us a run
 * when rows were cut evenly over all waves, 1707 so.) */
constexpr uint64_t kFrontBlocks = 16384;

inline std::vector<BlockRef> front_blocks(const std::vector<uint64_t>& wants)
{
    uint64_t sum = 0;
    for (uint64_t w : wants) sum += w;
    std::vector<BlockRef> out;
    for (uint32_t j = 0; j < wants.size(); ++j)
        add_blocks(out, j, 0, sum <= kFrontBlocks ? wants[j] : std::max<uint64_t>(1, wants[j] * kFrontBlocks / sum));
    return out;
}

/* Workgroups that a pass's classification (16 chunks a wave at a time) and count
 * (row groups of 64 >> cshift rows) have work for. */
inline uint64_t classify_blocks(const JobArgs& a) { return (a.nrows * a.NC + 16 * kWaves - 1) / (16 * kWaves); }

inline uint64_t count_blocks(const JobArgs& a)
{
    const uint64_t G = 64u >> a.cshift;
    return ((a.nrows + G - 1) / G + kWaves - 1) / kWaves;
}

}  // namespace kmc
