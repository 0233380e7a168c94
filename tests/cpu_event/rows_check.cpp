// Dose rows of the plain kernel's batches where memory is short
// (gegs_amd/csrc/plain.hpp reserve_rows), with an allocator that refuses more
// than a given number of rows.
#include <hip/hip_runtime.h>

#include <cstdio>

#include "../../gegs_amd/csrc/event.hpp"

namespace gegs {
float lds_env[LDS_FLOATS];
}
using namespace gegs;

static int fails = 0;

static void expect(uint32_t want, size_t nvox, size_t held, size_t free, uint32_t limit, uint32_t rows, bool ok) {
    uint32_t got = 0, held_rows = 0;
    const hipError_t e = reserve_rows(got, want, nvox, held, free, [&](uint32_t n) {
        if (n > limit) return hipErrorInvalidValue;
        held_rows = n;
        return hipSuccess;
    });
    if ((e == hipSuccess) == ok && got == rows && (!ok || held_rows == rows)) return;
    printf("failed: want %u of %zu voxels, held %zu, free %zu, limit %u: %u rows (%u had), error %d\n", want, nvox, held, free,
           limit, got, held_rows, (int)e);
    fails++;
}

int main() {
    const size_t vox = 1638400, row = vox * 8, GiB = (size_t)1 << 30;
    expect(10, vox, 0, 200 * GiB, 1u << 30, 10, true);                 // all of them
    expect(1, vox, 0, 0, 1u << 30, 1, true);                           // one row is always tried
    expect(1310, vox, 0, 200 * GiB, 1u << 30, 1310, true);
    expect(1310, vox, 0, 4 * GiB, 1u << 30, (uint32_t)(2 * GiB / row), true);          // half of what is free
    expect(1310, vox, 2 * GiB, 4 * GiB, 1u << 30, (uint32_t)(3 * GiB / row), true);    // held rows count as free
    expect(1310, vox, 2 * GiB, 2 * GiB, 1u << 30, (uint32_t)(2 * GiB / row), true);    // a repeated run keeps its rows
    expect(1310, vox, 2 * GiB, 0, 1u << 30, (uint32_t)(2 * GiB / row), true);
    expect(1310, vox, 0, 200 * GiB, 500, 328, true);                   // refused twice: 1310, 655, 328
    expect(1310, vox, 0, 200 * GiB, 1, 1, true);                       // down to one row
    expect(1310, vox, 0, 200 * GiB, 0, 1, false);                      // and not even that
    expect(7, vox, 0, 200 * GiB, 5, 4, true);
    expect(2, vox, 0, 3 * row, 0, 1, false);
    if (!fails) printf("ok\n");
    return fails != 0;
}
