// Copies of large arrays between the device and ordinary (pageable) host
// memory, through pinned slots and helper threads.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace mmd {

// The pinned slots of one context, allocated by its first large copy and freed
// with it.  Not for use by two threads at once (neither is a context).
class HostStage {
public:
    HostStage() = default;
    HostStage(const HostStage&) = delete;
    HostStage& operator=(const HostStage&) = delete;
    ~HostStage();
    // After the work queued on st; returns when dst is complete.
    hipError_t to_host(void* dst, const void* src, size_t bytes, hipStream_t st);
    // Returns when src has been read; dst is complete for later work on st.
    hipError_t to_device(void* dst, const void* src, size_t bytes, hipStream_t st);

private:
    static constexpr int SLOTS = 6;
    bool prepare();
    hipError_t drain();
    char* slots = nullptr;
    hipEvent_t ev[SLOTS] = {};
    bool busy[SLOTS] = {};
};

}  // namespace mmd
