// Memory that large-tensor calls share: N^4 device buffers and pinned staging
// slots, kept per device between calls, whoever makes them.
//
// A molecule has a context of its own and makes its stored tensor once, so
// what a context allocates for it is paid for on every geometry and held as
// long as the molecule is.  First calls on new contexts, with buffers and slots
// of their own and from here: see mmd_pool.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace mmd {

constexpr size_t STAGE_SLOT_BYTES = (size_t)8 << 20;

// One pinned slot of STAGE_SLOT_BYTES and the event of the copy that uses it.
struct StageSlot {
    char* p = nullptr;
    hipEvent_t ev = nullptr;
};

// Up to `want` slots for the current device into s; the number it got (kept
// ones first, then new ones while they can be allocated).
int pool_take_slots(int want, StageSlot* s);
// Gives n slots back, which nothing uses any more; or frees them (keep false).
void pool_give_slots(int n, const StageSlot* s, bool keep);

// Frees what the pool keeps on `device`; true if there was anything.
bool pool_release(int device);
// hipMalloc on the current device, tried again without what the pool keeps
// when the device is out of memory.  The caller holds device_alloc_mutex().
hipError_t device_malloc(void** p, size_t bytes);

// An N^4 buffer for the length of a call.  The caller says when the work on it
// has been waited for (done); a call that ends early frees the buffer, which
// waits for the device.
class Tensor4 {
public:
    Tensor4() = default;
    Tensor4(const Tensor4&) = delete;
    Tensor4& operator=(const Tensor4&) = delete;
    ~Tensor4();
    hipError_t reserve(size_t doubles);   // once; contents undefined
    void done() { idle = true; }
    double* p = nullptr;

private:
    size_t n = 0;
    int device = 0;
    bool idle = false;
};

}  // namespace mmd
