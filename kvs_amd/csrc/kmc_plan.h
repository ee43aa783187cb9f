/*
 * kmc_plan.h -- how the slots (node row, 64-node chunk) of a level are dealt to
 * the waves of the chunk-batch emit.  Plain C++, shared by the host's planning,
 * the kernels and the host-side tests.
 *
 * A *unit* is what a wave looks at in one step, a slot per lane: a.erows node rows
 * of up to 64 chunks, or one of the a.esegs parts of a longer row.  Wave w takes
 * units w, w + waves, w + 2 waves, ...; a slot is known to its wave by the step
 * and the lane alone, so 32 bits name it in volumes of any number of rows.
 */
#pragma once
#include <stdint.h>
#include <algorithm>
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

KMC_HD inline uint32_t emit_waves(const JobArgs& a) { return a.eblocks * (uint32_t)kWaves; }

/* First row and first chunk of a unit; the same on all lanes of its wave. */
struct EmitPart {
    uint64_t row;
    uint32_t chunk;
};

KMC_HD inline EmitPart emit_part(const JobArgs& a, uint64_t unit)
{
    EmitPart p;
    uint64_t group = unit;
    p.chunk = 0;
    if (a.esegs > 1) {
        group = div_by(unit, a.seg_inverse);
        p.chunk = (uint32_t)(unit - group * a.esegs) << a.cshift;
    }
    p.row = group * a.erows;
    return p;
}

/* Row of the unit and chunk of the row that a lane looks at.  Rows from a.erows on,
 * and slots past the row's chunks or the last row, hold nothing. */
KMC_HD inline uint32_t lane_row(const JobArgs& a, uint32_t lane) { return lane >> a.cshift; }
KMC_HD inline uint32_t lane_chunk(const JobArgs& a, uint32_t lane) { return lane & ((1u << a.cshift) - 1u); }

/* A slot as its wave queues it, and the unit that it came from. */
KMC_HD inline uint32_t emit_queued(uint32_t step, uint32_t lane) { return step << 6 | lane; }

KMC_HD inline uint64_t emit_unit(const JobArgs& a, uint32_t wave, uint32_t queued)
{
    return wave + (uint64_t)(queued >> 6) * emit_waves(a);
}

/* Node row -> (y, z). */
KMC_HD inline void row_place(const JobArgs& a, uint64_t row, uint32_t& y, uint32_t& z)
{
    z = (uint32_t)div_by(row, a.ny_inverse);
    y = (uint32_t)row - z * a.ny;
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
 * outputs.  A wave takes as many rows at a time as its lanes hold, but at most a
 * quarter of its share of the pass: a surface lies in few neighbouring rows, and
 * four steps far apart even the waves out (256^3 blobs, duplicated: 26 us, 36
 * with two steps).  Where every chunk holds many outputs there is nothing to
 * even out, and two steps keep the batches full (320 x 288 x 256 CT, vertices:
 * 38 us, 42 with four). */
constexpr uint64_t kEmitRounds = 8, kEmitItems = 32;

/* Split of the chunk-batch emit (rows planned; a.nlev set) of a pass whose emit
 * shares its launch with others, `all` being the sum of their emit_steps, for a
 * kernel of which a CU holds per_cu workgroups and that produces `items` outputs
 * (0: not known yet). */
inline void plan_emit(JobArgs& a, uint64_t all, uint32_t per_cu = 4, uint64_t items = 0)
{
    const uint64_t own = emit_steps(a), nlev = std::max(1u, a.nlev);
    const uint64_t resident = 256ull * kWaves * per_cu;
    uint64_t waves = resident * std::min(kEmitRounds, std::max<uint64_t>(1, all / 4 / resident));
    if (items) waves = std::min(waves, std::max<uint64_t>(256, items / kEmitItems));
    else waves = std::max(waves, std::min(2 * resident, all / 4));   // a batch's uneven passes even out by themselves
    const uint64_t want = std::max<uint64_t>(1, (waves * own + all - 1) / all / nlev);   // waves per level
    const uint64_t steps = items > 4 * nlev * a.nrows * a.NC ? 2 : 4;
    a.erows = 64u >> a.cshift;
    while (a.erows > 1 && a.nrows / a.erows < steps * want) a.erows >>= 1;
    a.esegs = (a.NC + 63) / 64;
    a.seg_inverse = 1.0 / a.esegs;
    a.ny_inverse = 1.0 / a.ny;
    a.eunits = (a.nrows + a.erows - 1) / a.erows * a.esegs;
    /* (a step's number has 26 bits in the queue) */
    const uint64_t least = (a.eunits >> 26) + 1;
    a.eblocks = (uint32_t)std::max<uint64_t>(1, (std::max(least, std::min(a.eunits, want)) + kWaves - 1) / kWaves);
}

}  // namespace kmc
