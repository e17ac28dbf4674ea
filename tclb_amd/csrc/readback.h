// readback.h -- fields from the device to the caller's memory, through
// staging that a lattice or a batch keeps between reads.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <functional>
#include <mutex>

namespace tclbx {

// Two device buffers and two pinned host buffers of at most CHUNK bytes (or
// one unit, where that is more), grown to what the reads so far needed and
// freed with their owner.  A field is read in chunks: while one is evaluated
// and copied to its pinned buffer, a few threads of this call copy the one
// before into the caller's memory.  Reads of at most DIRECT bytes are
// evaluated into the pinned buffer itself.  One read at a time; a second
// thread's waits.
//
// A large read is bound by the host link and by the first touch of the
// caller's pages, which several threads share; a small one by calls.  Against
// a device allocation per read and a copy to pageable memory (U of d3q19 256^3,
// 403 MB, 38.0 -> 9.6 ms; of 256x128x128 9.7 -> 2.9; of 128x96x64, 19 MB,
// 1.09 -> 0.67; of d2q9 1024x256, 6 MB, 403 -> 311 us; of 128x32 70 -> 22 us).
class Readback {
public:
    Readback() = default;
    ~Readback();
    Readback(const Readback&) = delete;
    Readback& operator=(const Readback&) = delete;

    static constexpr size_t CHUNK = size_t(16) << 20, DIRECT = size_t(128) << 10;

    // Reads `units` units (rows, layers) of `unit_bytes` bytes each into out:
    // eval(first, count, dst) launches on `stream` what writes the units
    // [first, first + count) to the device address dst.
    void read(size_t units, size_t unit_bytes, void* out, hipStream_t stream,
              const std::function<hipError_t(size_t, size_t, double*)>& eval);

private:
    void reserve(size_t bytes, bool device);
    std::mutex m_;
    char* dev_ = nullptr;     // two buffers of dev_cap_ bytes, one after the other
    char* pinned_ = nullptr;  // two of pinned_cap_ bytes
    hipEvent_t done_[2] = {nullptr, nullptr};
    size_t dev_cap_ = 0, pinned_cap_ = 0;
};

}  // namespace tclbx
