// Staged copies between the device and pageable host memory.
//
// The runtime copies pageable memory through its own staging buffer on one
// thread: 17.6 GB/s to the host and 28.9 GB/s to the device, where the link
// carries 57 GB/s to or from pinned memory.  The stored tensor, its J/K
// contraction and the four-index transformation move N^4 doubles per call and
// were bound by that.  Here the array goes through up to six pinned slots of 8 MiB: the
// calling thread keeps the copy engine busy, and a few helper threads move the
// slots to or from the caller's array (one thread moves 31 GB/s at most), a
// sixteenth of a slot at a time, so that the first slot is soon full and the
// last soon empty.  The stored tensor of (H2O)4 6-31G (58 MB) took 3.5 ms
// through the runtime, 2.1 with slots of 1 MiB, 1.6 with 4, 1.5 with 8; its
// J/K 2.4, 2.2, 1.6 and 1.5; a transformation of 85 MB each way 8.9, 5.8, 4.1
// and 4.0 ms.  Four helpers did as well as eight.
// The helpers live for one call (their start costs about 0.1 ms, so arrays
// below STAGE_MIN keep the runtime's copy, as does pinned memory, which needs
// no staging).
#include "mmd_hostcopy.h"
#include "mmd_helpers.h"

#include <atomic>
#include <stdint.h>
#include <string.h>
#include <thread>

namespace mmd {

namespace {

constexpr size_t SLOT_BYTES = STAGE_SLOT_BYTES;
constexpr int PARTS = 16;                           // of a slot
constexpr size_t PART_BYTES = SLOT_BYTES / PARTS;
constexpr size_t STAGE_MIN = (size_t)12 << 20;

bool pageable(const void* p)
{
    hipPointerAttribute_t a;
    const hipError_t e = hipPointerGetAttributes(&a, p);
    if (e != hipSuccess) {
        (void)hipGetLastError();   // unknown to the runtime: ordinary memory
        return true;
    }
    return a.type == hipMemoryTypeUnregistered;
}

}  // namespace

HostStage::~HostStage()
{
    hipError_t e = drain();
    if (broken) e = hipStreamSynchronize(broken);
    if (nslots) pool_give_slots(nslots, slot, e == hipSuccess);
}

// Slots for an array of `bytes`, two at least; false: copy without.
bool HostStage::prepare(size_t bytes)
{
    const size_t n = (bytes + SLOT_BYTES - 1) / SLOT_BYTES;
    const int want = n < (size_t)SLOTS ? (int)n : SLOTS;
    if (nslots < want) nslots += pool_take_slots(want - nslots, slot + nslots);
    return nslots >= 2;
}

// Waits for copies that still read or write slots.
hipError_t HostStage::drain()
{
    hipError_t r = hipSuccess;
    for (int s = 0; s < nslots; ++s) {
        if (!busy[s]) continue;
        const hipError_t e = hipEventSynchronize(slot[s].ev);
        if (e != hipSuccess) r = e;
        busy[s] = false;
    }
    return r;
}

hipError_t HostStage::to_host(void* dst, const void* src, size_t bytes, hipStream_t st)
{
    if (bytes < STAGE_MIN || !pageable(dst) || !prepare(bytes)) {
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st);
        return e == hipSuccess ? hipStreamSynchronize(st) : e;
    }
    hipError_t err = drain();
    if (err != hipSuccess) return err;
    const int n = (int)((bytes + SLOT_BYTES - 1) / SLOT_BYTES);
    const int ns = nslots, half = ns < n ? (ns + 1) / 2 : n;   // no slot is used twice where all chunks fit
    auto size_of = [&](int i) { return i + 1 < n ? SLOT_BYTES : bytes - (size_t)i * SLOT_BYTES; };
    const int64_t parts = (int64_t)((bytes + PART_BYTES - 1) / PART_BYTES);
    // bytes of a slot's chunks up to and including chunk i
    auto through = [&](int i) { return (int64_t)(i / ns) * (int64_t)SLOT_BYTES + (int64_t)size_of(i); };
    std::atomic<int> ready{0};
    std::atomic<int64_t> ticket{0}, emptied[SLOTS];
    std::atomic<bool> stop{false};
    for (auto& x : emptied) x = 0;
    Helpers helpers([&] {
        for (int64_t k = ticket++; k < parts; k = ticket++) {
            const int i = (int)(k / PARTS), s = i % ns;
            const size_t in = (size_t)(k % PARTS) * PART_BYTES, at = (size_t)k * PART_BYTES;
            const size_t len = bytes - at < PART_BYTES ? bytes - at : PART_BYTES;
            while (ready.load(std::memory_order_acquire) <= i) {
                if (stop) return;
                std::this_thread::yield();
            }
            memcpy((char*)dst + at, slot[s].p + in, len);
            emptied[s].fetch_add((int64_t)len, std::memory_order_release);
        }
    });
    if (helpers.n == 0) {
        err = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st);
        return err == hipSuccess ? hipStreamSynchronize(st) : err;
    }
    // copies up to half the slots ahead of the wait, so that the engine runs
    // while the helpers empty the other half
    int next = 0;
    for (int i = 0; i < n && err == hipSuccess; ++i) {
        for (; next < n && next < i + half && err == hipSuccess; ++next) {
            const int s = next % ns;
            if (next >= ns)
                while (emptied[s].load(std::memory_order_acquire) < through(next - ns)) std::this_thread::yield();
            err = hipMemcpyAsync(slot[s].p, (const char*)src + (size_t)next * SLOT_BYTES,
                                 size_of(next), hipMemcpyDeviceToHost, st);
            if (err == hipSuccess) err = hipEventRecord(slot[s].ev, st);
            if (err == hipSuccess) busy[s] = true;
        }
        if (err == hipSuccess) err = hipEventSynchronize(slot[i % ns].ev);
        if (err == hipSuccess) {
            busy[i % ns] = false;
            ready.store(i + 1, std::memory_order_release);
        }
    }
    if (err != hipSuccess) {
        stop = true;
        broken = st;
    }
    helpers.join();
    return err;
}

hipError_t HostStage::to_device(void* dst, const void* src, size_t bytes, hipStream_t st)
{
    if (bytes < STAGE_MIN || !pageable(src) || !prepare(bytes))
        return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st);
    hipError_t err = drain();
    if (err != hipSuccess) return err;
    const int n = (int)((bytes + SLOT_BYTES - 1) / SLOT_BYTES);
    const int ns = nslots, half = ns < n ? (ns + 1) / 2 : n;   // no slot is used twice where all chunks fit
    auto size_of = [&](int i) { return i + 1 < n ? SLOT_BYTES : bytes - (size_t)i * SLOT_BYTES; };
    const int64_t parts = (int64_t)((bytes + PART_BYTES - 1) / PART_BYTES);
    auto through = [&](int i) { return (int64_t)(i / ns) * (int64_t)SLOT_BYTES + (int64_t)size_of(i); };
    std::atomic<int> freed{ns};
    std::atomic<int64_t> ticket{0}, filled[SLOTS];
    std::atomic<bool> stop{false};
    for (auto& x : filled) x = 0;
    Helpers helpers([&] {
        for (int64_t k = ticket++; k < parts; k = ticket++) {
            const int i = (int)(k / PARTS), s = i % ns;
            const size_t in = (size_t)(k % PARTS) * PART_BYTES, at = (size_t)k * PART_BYTES;
            const size_t len = bytes - at < PART_BYTES ? bytes - at : PART_BYTES;
            while (freed.load(std::memory_order_acquire) <= i) {
                if (stop) return;
                std::this_thread::yield();
            }
            memcpy(slot[s].p + in, (const char*)src + at, len);
            filled[s].fetch_add((int64_t)len, std::memory_order_release);
        }
    });
    if (helpers.n == 0) return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st);
    for (int i = 0; i < n && err == hipSuccess; ++i) {
        const int s = i % ns;
        while (filled[s].load(std::memory_order_acquire) < through(i)) std::this_thread::yield();
        err = hipMemcpyAsync((char*)dst + (size_t)i * SLOT_BYTES, slot[s].p, size_of(i),
                             hipMemcpyHostToDevice, st);
        if (err == hipSuccess) err = hipEventRecord(slot[s].ev, st);
        if (err == hipSuccess) busy[s] = true;
        const int back = i - (half - 1);   // half the slots in flight, half with the helpers
        if (err == hipSuccess && back >= 0 && back + ns < n) {
            err = hipEventSynchronize(slot[back % ns].ev);
            busy[back % ns] = false;
            freed.store(back + 1 + ns, std::memory_order_release);
        }
    }
    if (err != hipSuccess) {
        stop = true;
        broken = st;
    }
    helpers.join();
    return err;
}

}  // namespace mmd
