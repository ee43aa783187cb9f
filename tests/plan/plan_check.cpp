/* Host program over the emit's plan (kmc_plan.h): plan_check slots | places | large | shares | unequal. */
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>
#include "kmc_plan.h"

using namespace kmc;

static JobArgs volume(uint32_t nx, uint32_t ny, uint32_t nz, uint32_t nlev)
{
    JobArgs a;
    std::memset(&a, 0, sizeof(a));
    a.nx = nx;
    a.ny = ny;
    a.nz = nz;
    a.nlev = nlev;
    a.NC = (nx + 63) / 64;
    while ((1u << a.cshift) < a.NC && a.cshift < 6) ++a.cshift;
    a.nrows = (uint64_t)ny * nz;
    return a;
}

/* Waves of a level that a set of rows falls to. */
template <typename F>
static uint64_t waves_of(const JobArgs& a, F&& has)
{
    std::vector<bool> met(a.ewaves);
    for (uint64_t u = 0; u < a.eunits; ++u)
        for (uint32_t lane = 0; lane < 64; ++lane) {
            const EmitSlot s = emit_slot(a, u, lane);
            if (lane_piece(a, lane) >= a.eparts || s.row >= a.nrows || s.chunk >= a.NC) continue;
            uint32_t y, z;
            row_place(a, s.row, y, z);
            if (has(s.chunk, y, z)) { met[u % a.ewaves] = true; break; }
        }
    uint64_t n = 0;
    for (bool b : met) n += b;
    return n;
}

static void fail(const char* what, const JobArgs& a)
{
    std::printf("%s: %u x %u x %u, %u levels\n", what, a.nx, a.ny, a.nz, a.nlev);
    std::exit(1);
}

/* What a wave queues for lane `lane` of its step comes back as the slot it looked at. */
static void check_slot(const JobArgs& a, uint32_t wave, uint64_t step, uint32_t lane)
{
    if (step >> 26) fail("step number does not fit the queue", a);
    const uint64_t unit = wave + step * a.ewaves;
    const EmitSlot s = emit_slot(a, unit, lane);
    const uint32_t queued = emit_queued((uint32_t)step, lane);
    const EmitSlot t = emit_slot(a, emit_unit(a, wave, queued), queued & 63u);
    if (s.row != t.row || s.chunk != t.chunk) fail("queued slot", a);
    if (s.row >= a.nrows || s.chunk >= a.NC) return;
    uint32_t y, z;
    row_place(a, t.row, y, z);
    if (y >= a.ny || z >= a.nz || (uint64_t)z * a.ny + y != s.row) fail("row of the slot", a);
}

/* Every slot of a small volume belongs to exactly one wave, step and lane. */
static void slots()
{
    const uint32_t shapes[][3] = { { 2, 1, 1 }, { 2, 70, 3 }, { 64, 9, 7 }, { 65, 33, 5 }, { 300, 40, 11 }, { 1024, 30, 4 }, { 1100, 40, 11 }, { 2000, 90, 70 }, { 4032, 9, 8 },
                                   { 4096, 5, 3 }, { 4097, 5, 3 }, { 9000, 7, 2 }, { 17, 700, 600 }, { 1024, 512, 520 } };
    for (auto& d : shapes)
        for (uint32_t nlev = 1; nlev <= 3; nlev += 2)
            for (uint64_t items : { 0ull, 1ull, 5000ull, 100000000ull }) {
                JobArgs a = volume(d[0], d[1], d[2], nlev);
                plan_emit(a, emit_steps(a), 5, items);
                std::vector<int> seen(a.nrows * a.NC, 0);
                for (uint32_t wave = 0; wave < a.ewaves; ++wave)
                    for (uint64_t step = 0; wave + step * a.ewaves < a.eunits; ++step)
                        for (uint32_t lane = 0; lane < 64; ++lane) {
                            check_slot(a, wave, step, lane);
                            const EmitSlot s = emit_slot(a, wave + step * a.ewaves, lane);
                            if (lane_piece(a, lane) < a.eparts && s.row < a.nrows && s.chunk < a.NC) ++seen[s.row * a.NC + s.chunk];
                        }
                for (int n : seen)
                    if (n != 1) fail("a slot is not looked at exactly once", a);
            }
}

/* row_place at the rows where the quotient steps, against the integer division. */
static void places()
{
    for (uint64_t ny : { 1u, 2u, 3u, 7u, 1000u, 65537u, 699049u, (1u << 20) - 1u, 1u << 20 }) {
        const uint64_t last = (1u << 20) - 1;
        JobArgs a = volume(2, (uint32_t)ny, 1u << 20, 1);
        plan_emit(a, emit_steps(a));
        for (uint64_t k = 0; k < 1u << 20; k += k < 64 ? 1 : 1 + k / 61)
            for (uint64_t row : { (uint64_t)k * ny, k * ny + ny / 2, k * ny + ny - 1, (last - k) * ny, (last - k) * ny + ny - 1 }) {
                uint32_t y, z;
                row_place(a, row, y, z);
                if (z != row / ny || y != row % ny) fail("row_place", a);
            }
    }
    for (uint32_t nx : { 4097u, 9000u, 500000u, 1u << 20 }) {
        JobArgs a = volume(nx, 1000, 1000, 1);
        plan_emit(a, emit_steps(a));
        for (uint64_t group = 0; group < 1ull << 31; group += 1 + group / 1000)
            for (uint32_t seg : { 0u, a.esegs / 2, a.esegs - 1 }) {
                const uint64_t piece = group * a.esegs + seg, unit = a.edist == 1 ? piece / a.eparts : piece;
                const EmitSlot t = emit_slot(a, unit, a.edist == 1 ? (uint32_t)(piece % a.eparts) << a.plog : 0);
                if (t.row != group << (a.plog - a.eshift) || t.chunk != seg << a.eshift) fail("emit_slot", a);
            }
    }
}

/* Volumes of more than 2^32 rows and chunks. */
static void large()
{
    const uint32_t shapes[][3] = { { 2, 65537, 65537 }, { 2, 65536, 65537 }, { 65, 1u << 20, 4096 }, { 64, 1u << 20, 1u << 20 },
                                   { 1u << 20, 1024, 1025 } };
    for (auto& d : shapes)
        for (uint64_t items : { 0ull, 1ull, 1000000000ull }) {
            JobArgs a = volume(d[0], d[1], d[2], 1);
            plan_emit(a, emit_steps(a), 4, items);
            const uint64_t last = a.nrows - 1, at = 1ull << 32;
            for (uint64_t row : { (uint64_t)0, at / a.NC - 1, at / a.NC, at - 1, at, at + 131072, last })
                for (uint32_t chunk : { 0u, a.NC / 2, a.NC - 1 }) {
                    if (row > last) continue;
                    const uint32_t rows = a.plog - a.eshift;
                    const uint64_t piece = (row >> rows) * a.esegs + (chunk >> a.eshift);
                    const uint64_t unit = a.edist == 1 ? piece / a.eparts : piece % a.eunits;
                    const uint64_t part = a.edist == 1 ? piece % a.eparts : piece / a.eunits;
                    const uint32_t wave = (uint32_t)(unit % a.ewaves);
                    const uint32_t lane = (uint32_t)part << a.plog | (uint32_t)(row & ((1u << rows) - 1u)) << a.eshift |
                                          (chunk & ((1u << a.eshift) - 1u));
                    const uint64_t step = unit / a.ewaves;
                    check_slot(a, wave, step, lane);
                    const EmitSlot s = emit_slot(a, emit_unit(a, wave, emit_queued((uint32_t)step, lane)), lane);
                    if (lane > 63 || s.row != row || s.chunk != chunk) fail("slot past 2^32", a);
                }
        }
}

/* Walks stay short whatever the outputs, and planes of one coordinate fall to many waves. */
static void shares()
{
    for (uint32_t e : { 256u, 512u, 1024u })
        for (uint64_t items : { 1ull, 1000ull, 100000ull }) {
            JobArgs a = volume(e, e, e, 1);
            plan_emit(a, emit_steps(a), 5, items);
            if (a.eunits * a.eparts << a.plog > 2 * kEmitWalk * 64 * a.ewaves && a.ewaves >= 256) fail("long walks", a);
        }
    for (uint32_t e : { 512u, 1000u, 1024u }) {
        JobArgs a = volume(e, e, e, 1);
        plan_emit(a, emit_steps(a), 4, 2ull * (e - 1) * (e - 1));
        if (waves_of(a, [&](uint32_t, uint32_t, uint32_t z) { return z == e / 2; }) < e / 3) fail("plane of one z", a);
        if (waves_of(a, [&](uint32_t, uint32_t y, uint32_t) { return y == e / 2; }) < e / 3) fail("plane of one y", a);
    }
    JobArgs a = volume(9000, 40, 33, 1);
    plan_emit(a, emit_steps(a), 5, 100000);
    if (waves_of(a, [&](uint32_t c, uint32_t y, uint32_t z) { return c >= 40 && c < 100 && y == 20 && z > 10 && z < 30; }) < 100)
        fail("long rows", a);
}

/* A large volume among small ones keeps its share of a batch's workgroups. */
static void unequal()
{
    for (uint32_t small : { 0u, 1u, 13u, 255u, 5000u }) {
        std::vector<JobArgs> jobs(1, volume(512, 512, 512, 1));
        jobs.resize(small + 1, volume(32, 32, 32, 1));
        for (int count = 0; count < 2; ++count) {
            std::vector<uint64_t> wants;
            uint64_t sum = 0;
            for (const JobArgs& a : jobs) {
                wants.push_back(count ? count_blocks(a) : classify_blocks(a));
                sum += wants.back();
            }
            const std::vector<BlockRef> refs = front_blocks(wants);
            std::vector<uint64_t> has(jobs.size(), 0);
            for (const BlockRef& r : refs) {
                if (r.block != has[r.job] || r.block >= r.blocks || r.blocks > wants[r.job]) fail("workgroups of a job", jobs[r.job]);
                ++has[r.job];
            }
            for (uint64_t n : has)
                if (n == 0) fail("a job without a workgroup", jobs[0]);
            if (refs.size() > kFrontBlocks + jobs.size()) fail("too many workgroups", jobs[0]);
            if (has[0] * sum * 2 < wants[0] * std::min(sum, kFrontBlocks)) fail("the large volume's share", jobs[0]);
        }
    }
}

int main(int argc, char** argv)
{
    if (argc < 2) return 2;
    if (!std::strcmp(argv[1], "slots")) slots();
    else if (!std::strcmp(argv[1], "large")) large();
    else if (!std::strcmp(argv[1], "places")) places();
    else if (!std::strcmp(argv[1], "shares")) shares();
    else if (!std::strcmp(argv[1], "unequal")) unequal();
    else return 2;
    std::printf("ok\n");
    return 0;
}
