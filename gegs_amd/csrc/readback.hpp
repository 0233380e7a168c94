// Results of a run from device memory into the caller's pageable buffers.
// Included after the HIP runtime's header.
#pragma once
#include <cstddef>
#include <cstring>
#include <thread>

namespace gegs {

// Pinned slots and their events: 8 MiB per context, made at the first use.
struct ReadStage {
    static constexpr int SLOTS = 8;
    static constexpr size_t BYTES = (size_t)1 << 20;
    unsigned char *mem = nullptr;
    hipEvent_t done[SLOTS] = {};

    // False where the runtime gives no pinned memory or no event (its error
    // is taken back: the caller has another way to copy); what was made
    // stays, the rest is tried again at the next call.
    bool ready() {
        if (!mem) {
            void *p = nullptr;
            if (hipHostMalloc(&p, SLOTS * BYTES) != hipSuccess) {
                (void)hipGetLastError();
                return false;
            }
            mem = static_cast<unsigned char *>(p);
        }
        for (int k = 0; k < SLOTS; ++k)
            if (!done[k] && hipEventCreateWithFlags(&done[k], hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                done[k] = nullptr;
                return false;
            }
        return true;
    }
    void release() {
        if (mem) (void)hipHostFree(mem);
        mem = nullptr;
        for (int k = 0; k < SLOTS; ++k) {
            if (done[k]) (void)hipEventDestroy(done[k]);
            done[k] = nullptr;
        }
    }
};

// Copies n arrays of `bytes` bytes each.  A copy of a dose spends
// most of its time on the host: the transfer into pinned memory runs at the
// link's rate, while moving it on into pages that the caller never touched
// is bound by one core.  Here up to SLOTS host threads take the pieces
// in turn, each through its own pinned slot, so the transfers of some pieces
// run beside the host copies of the others (two doses of 13 MB on the
// 128x128x100 CT: 1.9 -> 1.2 ms of a run).  Results of at most one slot
// together take a plain copy (16^3 water, 500 histories: a run of 0.50 ms with
// a slot and a helper, 0.44 ms without), and so do all where there are no
// slots.  The device's work on the arrays must be complete.
inline hipError_t read_back(ReadStage &stage, int device, hipStream_t stream, void *const *dst, const void *const *src,
                            int n, size_t bytes) {
    constexpr int SLOTS = ReadStage::SLOTS;
    constexpr size_t BYTES = ReadStage::BYTES;
    const size_t pieces = (bytes + BYTES - 1) / BYTES;
    const size_t total = pieces * (size_t)n;
    if ((size_t)n * bytes <= BYTES || !stage.ready()) {
        for (int k = 0; k < n; ++k) {
            const hipError_t e = hipMemcpy(dst[k], src[k], bytes, hipMemcpyDeviceToHost);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    hipError_t err[SLOTS] = {};
    auto work = [&](int slot) {
        hipError_t e = hipSetDevice(device);
        for (size_t i = (size_t)slot; i < total && e == hipSuccess; i += SLOTS) {
            const size_t at = i % pieces * BYTES, len = bytes - at < BYTES ? bytes - at : BYTES;
            unsigned char *mem = stage.mem + slot * BYTES;
            e = hipMemcpyAsync(mem, (const unsigned char *)src[i / pieces] + at, len, hipMemcpyDeviceToHost, stream);
            if (e == hipSuccess) e = hipEventRecord(stage.done[slot], stream);
            if (e == hipSuccess) e = hipEventSynchronize(stage.done[slot]);
            if (e == hipSuccess) memcpy((unsigned char *)dst[i / pieces] + at, mem, len);
        }
        err[slot] = e;
    };
    std::thread helper[SLOTS - 1];
    int started = 0;
    try {
        while (started < SLOTS - 1 && (size_t)(started + 1) < total) {
            helper[started] = std::thread(work, started + 1);
            ++started;
        }
    } catch (...) {   // no thread to be had: this one takes the slots left
    }
    work(0);
    for (int k = started + 1; k < SLOTS; ++k) work(k);
    for (int k = 0; k < started; ++k) helper[k].join();
    for (int k = 0; k < SLOTS; ++k)
        if (err[k] != hipSuccess) return err[k];
    return hipSuccess;
}

}  // namespace gegs
