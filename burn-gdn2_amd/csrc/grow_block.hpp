// Device memory of a layer that grows on demand.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <vector>

namespace gdn2 {

// Device memory that grows on demand.  The kernels of a captured graph read and
// write the block they were recorded with, however many larger calls follow, so
// a block that a recorded call uses is kept until its owner is destroyed when it
// is outgrown; others are freed.
class GrowBlock {
  public:
    void *ptr() const { return ptr_; }
    size_t bytes() const { return bytes_; }
    // Room for `need` bytes.  recording: the call is being captured (nothing may
    // be waited for or freed then; whether it may allocate is the capture's mode).
    hipError_t ensure(size_t need, bool recording) {
        if (need > bytes_) {
            if (ptr_ && (recorded_ || recording)) {
                kept_.push_back(ptr_);
            } else if (ptr_) {
                hipError_t e = hipDeviceSynchronize();
                if (e == hipSuccess) e = hipFree(ptr_);
                if (e != hipSuccess) return e;
            }
            ptr_ = nullptr;
            bytes_ = 0;
            recorded_ = false;
            const hipError_t e = hipMalloc(&ptr_, need);
            if (e != hipSuccess) {
                ptr_ = nullptr;
                return e;
            }
            bytes_ = need;
        }
        recorded_ = recorded_ || recording;
        return hipSuccess;
    }
    void destroy() {
        for (void *p : kept_) (void)hipFree(p);
        kept_.clear();
        if (ptr_) (void)hipFree(ptr_);
        ptr_ = nullptr;
        bytes_ = 0;
        recorded_ = false;
    }

  private:
    void *ptr_ = nullptr;
    size_t bytes_ = 0;
    bool recorded_ = false; // a captured graph holds ptr_
    std::vector<void *> kept_;
};

// Whether calls on a stream are being captured (one that can't be asked counts
// as captured: its blocks are then kept).
inline bool stream_recording(hipStream_t s) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(s, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone;
}

}  // namespace gdn2
