// The copy of results to host buffers (gegs_amd/csrc/readback.hpp) over a
// stand-in of the runtime calls that it makes, which fail when told to.
#include <atomic>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorInvalidHandle = 400 };
typedef void *hipStream_t;
typedef int *hipEvent_t;
enum { hipEventDisableTiming = 2, hipMemcpyDeviceToHost = 2 };

static int host_mallocs_ok = 1 << 30, events_ok = 1 << 30;   // calls that succeed before they fail
static std::atomic<int> staged{0}, plain{0}, null_events{0};
static int live_events = 0, live_host = 0;
static hipError_t last = hipSuccess;

static hipError_t hipHostMalloc(void **p, size_t n) {
    if (host_mallocs_ok-- <= 0) return last = hipErrorOutOfMemory;
    *p = malloc(n);
    live_host++;
    return hipSuccess;
}
static hipError_t hipHostFree(void *p) {
    free(p);
    live_host--;
    return hipSuccess;
}
static hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    if (events_ok-- <= 0) return last = hipErrorOutOfMemory;
    *e = new int(0);
    live_events++;
    return hipSuccess;
}
static hipError_t hipEventDestroy(hipEvent_t e) {
    delete e;
    live_events--;
    return hipSuccess;
}
static hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
static hipError_t hipSetDevice(int) { return hipSuccess; }
static hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    if (!e) {
        null_events++;
        return hipErrorInvalidHandle;
    }
    return hipSuccess;
}
static hipError_t hipEventSynchronize(hipEvent_t e) { return e ? hipSuccess : hipErrorInvalidHandle; }
static hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, int, hipStream_t) {
    memcpy(d, s, n);
    staged++;
    return hipSuccess;
}
static hipError_t hipMemcpy(void *d, const void *s, size_t n, int) {
    memcpy(d, s, n);
    plain++;
    return hipSuccess;
}

#include "../../gegs_amd/csrc/readback.hpp"
using namespace gegs;

static int fails = 0;
static void check(bool ok, const char *what) {
    if (ok) return;
    printf("failed: %s\n", what);
    fails++;
}

// one copy of n arrays; true when it succeeds, left no error and the bytes are right
static bool copies(ReadStage &st, int n, size_t bytes) {
    std::vector<std::vector<unsigned char>> in(n), out(n);
    std::vector<void *> d;
    std::vector<const void *> s;
    for (int k = 0; k < n; ++k) {
        in[k].resize(bytes);
        out[k].assign(bytes, 0);
        for (size_t i = 0; i < bytes; ++i) in[k][i] = (unsigned char)(i * 31u + (i >> 11) + (size_t)k * 7u + 1u);
        d.push_back(out[k].data());
        s.push_back(in[k].data());
    }
    staged = plain = 0;
    if (read_back(st, 0, nullptr, d.data(), s.data(), n, bytes) != hipSuccess || last != hipSuccess) return false;
    return in == out;
}

int main() {
    const size_t MiB = (size_t)1 << 20;
    {
        ReadStage st;
        check(copies(st, 2, 32768) && plain == 2 && !st.mem, "two small arrays: plain copies, no pinned memory");
        check(copies(st, 1, MiB) && plain == 1 && !st.mem, "one slot's worth: plain copy");
        check(copies(st, 2, MiB / 2) && plain == 2 && !st.mem, "one slot's worth together: plain copies");
        check(copies(st, 2, MiB / 2 + 8) && plain == 0 && staged == 2, "past one slot: staged");
        check(copies(st, 1, MiB + 8) && staged == 2, "one array past one slot: staged");
        check(copies(st, 2, 13 * MiB + 24) && staged == 28, "two doses: staged");
        check(copies(st, 0, 13 * MiB), "no array asked for");
        st.release();
    }
    {   // no pinned memory: plain copies, and the slots once there is some
        ReadStage st;
        host_mallocs_ok = 0;
        check(copies(st, 2, 3 * MiB) && plain == 2, "no pinned memory");
        host_mallocs_ok = 1;
        check(copies(st, 2, 3 * MiB) && staged == 6, "pinned memory again");
        host_mallocs_ok = 1 << 30;
        st.release();
    }
    for (int made = 0; made < ReadStage::SLOTS; ++made) {   // an event fails half way: no null event is used, now or later
        ReadStage st;
        events_ok = made;
        check(copies(st, 2, 3 * MiB) && plain == 2, "no event to be had");
        check(copies(st, 2, 3 * MiB) && plain == 2, "still no event");
        events_ok = 1 << 30;
        check(copies(st, 2, 3 * MiB) && staged == 6, "events again");
        st.release();
    }
    check(null_events == 0, "null events recorded");
    check(live_events == 0 && live_host == 0, "released");
    if (!fails) printf("ok\n");
    return fails != 0;
}
