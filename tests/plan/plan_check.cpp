/* Host program over the emit's plan (kmc_plan.h): plan_check slots | places | large. */
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

static void fail(const char* what, const JobArgs& a)
{
    std::printf("%s: %u x %u x %u, %u levels\n", what, a.nx, a.ny, a.nz, a.nlev);
    std::exit(1);
}

struct Slot {
    uint64_t row;
    uint32_t chunk;
};

static Slot slot_of(const JobArgs& a, uint64_t unit, uint32_t lane)
{
    const EmitPart p = emit_part(a, unit);
    return { p.row + lane_row(a, lane), p.chunk + lane_chunk(a, lane) };
}

/* What a wave queues for lane `lane` of its step comes back as the slot it looked at. */
static void check_slot(const JobArgs& a, uint32_t wave, uint64_t step, uint32_t lane)
{
    if (step >> 26) fail("step number does not fit the queue", a);
    const uint64_t unit = wave + step * emit_waves(a);
    const Slot s = slot_of(a, unit, lane);
    const uint32_t queued = emit_queued((uint32_t)step, lane);
    const Slot t = slot_of(a, emit_unit(a, wave, queued), queued & 63u);
    if (s.row != t.row || s.chunk != t.chunk) fail("queued slot", a);
    if (s.row >= a.nrows || s.chunk >= a.NC) return;
    uint32_t y, z;
    row_place(a, t.row, y, z);
    if (y >= a.ny || z >= a.nz || (uint64_t)z * a.ny + y != s.row) fail("row of the slot", a);
}

/* Every slot of a small volume belongs to exactly one wave, step and lane. */
static void slots()
{
    const uint32_t shapes[][3] = { { 2, 1, 1 }, { 2, 70, 3 }, { 64, 9, 7 }, { 65, 33, 5 }, { 300, 40, 11 }, { 1024, 30, 4 },
                                   { 4096, 5, 3 }, { 4097, 5, 3 }, { 9000, 7, 2 } };
    for (auto& d : shapes)
        for (uint32_t nlev = 1; nlev <= 3; nlev += 2)
            for (uint64_t items : { 0ull, 1ull, 5000ull, 10000000ull }) {
                JobArgs a = volume(d[0], d[1], d[2], nlev);
                plan_emit(a, emit_steps(a), 5, items);
                std::vector<int> seen(a.nrows * a.NC, 0);
                for (uint32_t wave = 0; wave < emit_waves(a); ++wave)
                    for (uint64_t step = 0; wave + step * emit_waves(a) < a.eunits; ++step)
                        for (uint32_t lane = 0; lane < 64; ++lane) {
                            check_slot(a, wave, step, lane);
                            const Slot s = slot_of(a, wave + step * emit_waves(a), lane);
                            if (lane_row(a, lane) < a.erows && s.row < a.nrows && s.chunk < a.NC) ++seen[s.row * a.NC + s.chunk];
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
                const EmitPart p = emit_part(a, group * a.esegs + seg);
                if (p.row != group * a.erows || p.chunk != seg << a.cshift) fail("emit_part", a);
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
                    const uint64_t unit = row / a.erows * a.esegs + (chunk >> a.cshift);
                    const uint32_t wave = (uint32_t)(unit % emit_waves(a));
                    const uint32_t lane = (uint32_t)(row % a.erows) << a.cshift | (chunk & ((1u << a.cshift) - 1u));
                    const uint64_t step = unit / emit_waves(a);
                    check_slot(a, wave, step, lane);
                    const Slot s = slot_of(a, emit_unit(a, wave, emit_queued((uint32_t)step, lane)), lane);
                    if (unit >= a.eunits || s.row != row || s.chunk != chunk) fail("slot past 2^32", a);
                }
        }
}

int main(int argc, char** argv)
{
    if (argc < 2) return 2;
    if (!std::strcmp(argv[1], "slots")) slots();
    else if (!std::strcmp(argv[1], "large")) large();
    else if (!std::strcmp(argv[1], "places")) places();
    else return 2;
    std::printf("ok\n");
    return 0;
}
