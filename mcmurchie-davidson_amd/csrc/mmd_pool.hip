// What the tensor calls keep between calls, per device.
//
// Pinned memory is cheap to allocate and dear to touch first: a new slot costs
// a host thread 0.36 ms per MiB of page faults, 17 ms for six slots on one
// thread.  With slots and N^4 buffers of each context's own the first stored
// tensor of every new molecule paid that ((H2O)4 6-31G 8.0 ms against 1.53 for
// a second one, (H2O)3 3.5 against 0.65), and eight live molecules of 64
// functions held 2.1 GB; from here it takes 1.55 and 0.73 ms, and they hold 512
// MB at most.
#include "mmd_pool.h"

#include <algorithm>
#include <mutex>

namespace mmd {

std::recursive_mutex& device_alloc_mutex();

namespace {

// What is kept of a device: buffers of at most KEEP_BUFFER bytes, the latest
// KEEP_COUNT that make up at most KEEP_BYTES, and the slots of two calls at once.
constexpr size_t KEEP_BUFFER = (size_t)256 << 20;
constexpr size_t KEEP_BYTES = (size_t)512 << 20;
constexpr int KEEP_COUNT = 4;
constexpr int KEEP_SLOTS = 12;
constexpr int DEVICES = 64;

struct Buffer {
    double* p;
    size_t n;
};
// Plain memory, left to the end of the process: the runtime may be gone before
// the process's statics are destroyed.
struct Kept {
    Buffer buffers[KEEP_COUNT];   // the one given back last at the end
    int nbuffers;
    StageSlot slots[KEEP_SLOTS];
    int nslots;
};
Kept g_kept[DEVICES];
// Guards g_kept alone, for a few instructions: a call that finds what it needs
// does not wait for another thread's allocation or graph capture.  Taken after
// device_alloc_mutex() where both are held.
std::mutex g_kept_mutex;

int current_device()
{
    int d = 0;
    return hipGetDevice(&d) == hipSuccess && d >= 0 && d < DEVICES ? d : 0;
}

void free_slots(int n, const StageSlot* s)
{
    if (n == 0) return;
    std::lock_guard<std::recursive_mutex> lk(device_alloc_mutex());
    for (int i = 0; i < n; ++i) {
        if (s[i].ev) (void)hipEventDestroy(s[i].ev);
        if (s[i].p) (void)hipHostFree(s[i].p);
    }
}

void free_buffers(int n, const Buffer* b)
{
    if (n == 0) return;   // nor wait for another thread's capture
    std::lock_guard<std::recursive_mutex> lk(device_alloc_mutex());
    for (int i = 0; i < n; ++i) (void)hipFree(b[i].p);
}

}  // namespace

int pool_take_slots(int want, StageSlot* s)
{
    int got = 0;
    {
        Kept& k = g_kept[current_device()];
        std::lock_guard<std::mutex> lk(g_kept_mutex);
        while (got < want && k.nslots > 0) s[got++] = k.slots[--k.nslots];
    }
    if (got == want) return got;
    std::lock_guard<std::recursive_mutex> lk(device_alloc_mutex());
    for (; got < want; ++got) {
        StageSlot x;
        if (hipEventCreateWithFlags(&x.ev, hipEventDisableTiming) != hipSuccess) x.ev = nullptr;
        else if (hipHostMalloc((void**)&x.p, STAGE_SLOT_BYTES, hipHostMallocDefault) != hipSuccess) x.p = nullptr;
        if (!x.ev || !x.p) {
            (void)hipGetLastError();
            free_slots(1, &x);
            break;
        }
        s[got] = x;
    }
    return got;
}

void pool_give_slots(int n, const StageSlot* s, bool keep)
{
    int taken = 0;
    if (keep) {
        Kept& k = g_kept[current_device()];
        std::lock_guard<std::mutex> lk(g_kept_mutex);
        // last one first: the next call of the size takes them in the same order
        // (in turned order J/K of 58 MB took 1611 us, so 1598)
        const int room = KEEP_SLOTS - k.nslots;
        taken = n < room ? n : room;
        for (int i = taken - 1; i >= 0; --i) k.slots[k.nslots++] = s[i];
    }
    if (taken < n) free_slots(n - taken, s + taken);
}

bool pool_release(int device)
{
    if (device < 0 || device >= DEVICES) return false;
    Kept k;
    {
        std::lock_guard<std::mutex> lk(g_kept_mutex);
        k = g_kept[device];
        g_kept[device].nbuffers = g_kept[device].nslots = 0;
    }
    free_buffers(k.nbuffers, k.buffers);
    free_slots(k.nslots, k.slots);
    return k.nbuffers > 0 || k.nslots > 0;
}

hipError_t device_malloc(void** p, size_t bytes)
{
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipErrorOutOfMemory) return e;
    (void)hipGetLastError();
    if (!pool_release(current_device())) return e;
    e = hipMalloc(p, bytes);
    if (e != hipSuccess) (void)hipGetLastError();
    return e;
}

hipError_t Tensor4::reserve(size_t doubles)
{
    device = current_device();
    {
        // the smallest kept buffer that is large enough
        Kept& k = g_kept[device];
        std::lock_guard<std::mutex> lk(g_kept_mutex);
        int best = -1;
        for (int i = 0; i < k.nbuffers; ++i)
            if (k.buffers[i].n >= doubles && (best < 0 || k.buffers[i].n < k.buffers[best].n)) best = i;
        if (best >= 0) {
            p = k.buffers[best].p;
            n = k.buffers[best].n;
            std::copy(k.buffers + best + 1, k.buffers + k.nbuffers--, k.buffers + best);
            return hipSuccess;
        }
    }
    std::lock_guard<std::recursive_mutex> lk(device_alloc_mutex());
    const hipError_t e = device_malloc((void**)&p, std::max<size_t>(1, doubles) * sizeof(double));
    if (e == hipSuccess) n = doubles;
    else p = nullptr;
    return e;
}

Tensor4::~Tensor4()
{
    if (!p) return;
    const Buffer mine{p, n};
    if (!idle || n > KEEP_BUFFER / sizeof(double)) {
        free_buffers(1, &mine);
        return;
    }
    // the latest ones stay, this one first of all
    Buffer drop[KEEP_COUNT];
    int ndrop;
    {
        Kept& k = g_kept[device];
        std::lock_guard<std::mutex> lk(g_kept_mutex);
        size_t total = n;
        int stay = 0;
        while (stay < k.nbuffers && stay < KEEP_COUNT - 1
               && (total += k.buffers[k.nbuffers - 1 - stay].n) <= KEEP_BYTES / sizeof(double))
            ++stay;
        ndrop = k.nbuffers - stay;
        std::copy(k.buffers, k.buffers + ndrop, drop);
        std::copy(k.buffers + ndrop, k.buffers + k.nbuffers, k.buffers);
        k.buffers[stay] = mine;
        k.nbuffers = stay + 1;
    }
    free_buffers(ndrop, drop);
}

}  // namespace mmd
