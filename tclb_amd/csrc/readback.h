// readback.h -- fields from the device to the caller's memory, through
// staging that a lattice or a batch keeps between reads.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <functional>
#include <mutex>

namespace tclbx {

// Two pinned host buffers of at most CHUNK bytes each, grown to what the reads
// so far needed and freed with their owner; the field kernels write to them
// over the host link.  A field is read in chunks: while one is evaluated into
// its buffer, a few threads of this call copy the one before into the caller's
// memory.  One read at a time; a second thread's waits.
//
// A large read is bound by the host link and by the first touch of the
// caller's pages, which several threads share; a small one by calls.  Against
// a device allocation per read and a copy to pageable memory, U of d3q19 256^3
// (403 MB) 38.2 -> 8.7 ms, of 256x128x96 (75 MB) 7.5 -> 2.0, of 128x96x64 (19
// MB) 1.38 -> 0.62, of 61x48x57 (4 MB) 0.29 -> 0.20.  The first read of a
// lattice also pays for the pinned memory: 256^3 8.7 to 9.8 ms (38), 128x96x64
// 1.0 to 1.2 (1.4 to 2.2), 61x48x57 0.26 to 0.75 (0.28 to 0.58, by the
// runtime), 32^3 95 us (62).  Through device buffers and copies on the stream
// the steady reads took 10.5, 2.6, 0.67 and 0.25 ms, and the first of a
// process, which sets up the copies, up to 7 ms (now 1 to 2).
class Readback {
public:
    Readback() = default;
    ~Readback();
    Readback(const Readback&) = delete;
    Readback& operator=(const Readback&) = delete;

    static constexpr size_t CHUNK = size_t(16) << 20;

    // A box of nx x ny x nz nodes of node_bytes bytes each into out:
    // eval(x, y, z, nx, ny, nz, dst) launches on `stream` what writes the part
    // of the box from (x, y, z) on, of that size, to the device address dst.
    using Eval = std::function<hipError_t(int, int, int, int, int, int, double*)>;
    void read(int nx, int ny, int nz, size_t node_bytes, void* out, hipStream_t stream, const Eval& eval);

private:
    // `units` units of unit_bytes (at most CHUNK) bytes each: eval(first, count, dst)
    void read_units(size_t units, size_t unit_bytes, char* out, hipStream_t stream,
                    const std::function<hipError_t(int, int, double*)>& eval);
    std::mutex m_;
    char* pinned_ = nullptr;
    hipEvent_t done_[2] = {nullptr, nullptr};
    size_t cap_ = 0;
};

}  // namespace tclbx
