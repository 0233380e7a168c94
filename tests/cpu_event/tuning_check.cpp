// The caller's tuning and what a run makes of it (gegs_amd/csrc/event.hpp
// config_of, tuning_of, pick_shape, split_tail): a tuning read and set again
// leaves every run's chunks, grid and short-run path as they were, and tables
// that split photons get a tail with the stacks they need.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstring>

#include "../../gegs_amd/csrc/event.hpp"

namespace gegs {
float lds_env[LDS_FLOATS];
}
using namespace gegs;

static int fails = 0;
static void check(bool ok, const char *what) {
    if (ok) return;
    printf("failed: %s\n", what);
    fails++;
}

// chunks, grid, short-run path and tail of a run under cfg
static void shape(EventConfig cfg, bool head, uint32_t p, uint32_t e, uint32_t g, bool direct, const char *what) {
    pick_shape(cfg, head);
    check(cfg.photon_chunk == p && cfg.electron_chunk == e && cfg.grid == g && cfg.direct == direct, what);
}

int main() {
    const EventConfig d;
    shape(d, false, 96, 12, 512, true, "default, phantom");
    shape(d, true, 32, 8, 512, true, "default, head");
    const gegs_tuning r = tuning_of(d);
    check(r.photon_chunk == 0 && r.electron_chunk == 0 && r.grid == 0, "what the run picks reads as 0");
    check(r.block == 256 && r.inject == 6u << 20 && r.tail_particles == 1u << 18 && r.sweep_streams == 2, "defaults filled in");
    shape(config_of(r), false, 96, 12, 512, true, "read and set again, phantom");
    shape(config_of(r), true, 32, 8, 512, true, "read and set again, head");
    gegs_tuning z{};
    shape(config_of(z), false, 96, 12, 512, true, "all zero");
    // one field of the caller's: the others stay the run's, and short runs sweep
    z.photon_chunk = 7;
    shape(config_of(z), false, 7, 12, 512, false, "photon chunk alone");
    const gegs_tuning z2 = tuning_of(config_of(z));
    check(z2.photon_chunk == 7 && z2.electron_chunk == 0 && z2.grid == 0, "photon chunk alone, read");
    shape(config_of(z2), true, 7, 8, 512, false, "photon chunk alone, read and set again");
    gegs_tuning s = r;
    s.sweep_streams = 1;
    shape(config_of(s), false, 96, 12, 512, false, "one stream");
    s.sweep_streams = 2;
    shape(config_of(s), false, 96, 12, 512, true, "and back");
    gegs_tuning t = r;
    t.tail_particles = 0xFFFFFFFFu;
    check(config_of(t).tail == 0 && tuning_of(config_of(t)).tail_particles == 0xFFFFFFFFu, "no tail");
    gegs_tuning a{};
    a.block = 128; a.grid = 77; a.photon_grid = 5; a.electron_grid = 6; a.photon_chunk = 0xFFFFFFFFu;
    a.electron_chunk = 3; a.inject = 10; a.threshold = 20; a.sweeps_per_graph = 2; a.flight_block = 512;
    a.refill_min = 9; a.refill_slots = 128; a.sweep_streams = 1; a.tail_particles = 99; a.capacity = 12345;
    const gegs_tuning b = tuning_of(config_of(a));
    check(memcmp(&a, &b, sizeof(a)) == 0, "every field given reads back");
    // photons split n ways: stacks n times as deep, past 8 for 8/n of the particles
    for (uint32_t n : {1u, 2u, 3u, 8u, 9u, 32u, 16384u}) {
        EventConfig c;
        split_tail(c, n);
        check(c.tail == (n <= 8u ? d.tail : d.tail * 8u / n) && c.tail_depth == (int)(40u * n), "split tail");
        check((uint64_t)tail_threads(c) * (uint64_t)c.tail_depth <= 8ull * tail_threads(d) * 40u * 3u / 2u, "split tail's memory");
    }
    for (uint32_t n : {16385u, 262145u, 0x7FFFFFFFu}) {
        EventConfig c;
        split_tail(c, n);
        check(c.tail == 0, "split too far for a tail");
    }
    EventConfig few;
    few.tail = 64;
    split_tail(few, 1);
    check(few.tail == 64 && few.tail_depth == 40, "a caller's short tail, unsplit");
    if (!fails) printf("ok\n");
    return fails != 0;
}
