// Copies of large arrays between the device and ordinary (pageable) host
// memory, through pinned slots and helper threads.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include "mmd_pool.h"

namespace mmd {

// The copies of one call: its slots come from the device's pool at the first
// large copy, as many as the array fills, and go back when the call ends.
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
    // The caller has waited for st since.
    void done()
    {
        for (bool& b : busy) b = false;
    }

private:
    static constexpr int SLOTS = 6;
    bool prepare(size_t bytes);
    hipError_t drain();
    StageSlot slot[SLOTS];
    int nslots = 0;
    bool busy[SLOTS] = {};
    hipStream_t broken = nullptr;   // where a copy failed: one without its event may still run there
};

}  // namespace mmd
