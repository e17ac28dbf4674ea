// readback.cpp -- see readback.h.
#include "readback.h"

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <system_error>
#include <thread>
#include <vector>

#include "lattice.h"

namespace tclbx {

namespace {
// copies split over the calling thread and some of its own
class Copier {
public:
    explicit Copier(unsigned threads) {
        workers_.reserve(threads);
        try {
            for (unsigned i = 1; i < threads; i++) workers_.emplace_back([this, i] { work(i); });
        } catch (const std::system_error&) {
            // no more threads to be had: the copies are split over those there are
        }
        std::lock_guard<std::mutex> l(m_);
        parts_ = (unsigned)workers_.size() + 1;
    }
    ~Copier() {
        {
            std::lock_guard<std::mutex> l(m_);
            stop_ = true;
        }
        go_.notify_all();
        for (auto& t : workers_) t.join();
    }
    void copy(char* dst, const char* src, size_t n) {
        {
            std::lock_guard<std::mutex> l(m_);
            dst_ = dst;
            src_ = src;
            n_ = n;
            left_ = parts_ - 1;
            turn_++;
        }
        go_.notify_all();
        part(0);
        std::unique_lock<std::mutex> l(m_);
        done_.wait(l, [&] { return left_ == 0; });
    }

private:
    // pages of the destination go whole to one thread
    void part(unsigned i) {
        const size_t each = (n_ / parts_ + 4096) / 4096 * 4096, a = std::min(n_, i * each);
        std::memcpy(dst_ + a, src_ + a, std::min(each, n_ - a));
    }
    void work(unsigned i) {
        unsigned seen = 0;
        std::unique_lock<std::mutex> l(m_);
        for (;;) {
            go_.wait(l, [&] { return stop_ || turn_ != seen; });
            if (stop_) return;
            seen = turn_;
            l.unlock();
            part(i);
            l.lock();
            if (--left_ == 0) done_.notify_one();
        }
    }
    std::vector<std::thread> workers_;
    std::mutex m_;
    std::condition_variable go_, done_;
    char* dst_ = nullptr;
    const char* src_ = nullptr;
    size_t n_ = 0;
    unsigned parts_ = 1, left_ = 0, turn_ = 0;
    bool stop_ = false;
};
}  // namespace

Readback::~Readback() {
    if (dev_) (void)hipFree(dev_);
    if (pinned_) (void)hipHostFree(pinned_);
    for (hipEvent_t e : done_)
        if (e) (void)hipEventDestroy(e);
}

// buffers of at least `bytes`: powers of two up to CHUNK, so that a region
// that grows from read to read does not allocate on each.  Both buffers of a
// kind are one allocation: the first read of a lattice pays for it.
void Readback::reserve(size_t bytes, bool device) {
    size_t want = 4096;
    while (want < bytes && want < CHUNK) want *= 2;
    want = std::max(want, bytes);
    if (pinned_cap_ < bytes) {
        pinned_cap_ = 0;
        if (pinned_) (void)hipHostFree(pinned_);
        pinned_ = nullptr;
        hip_check(hipHostMalloc((void**)&pinned_, 2 * want, hipHostMallocDefault), "hipHostMalloc(field staging)");
        pinned_cap_ = want;
    }
    if (device && dev_cap_ < bytes) {
        dev_cap_ = 0;
        if (dev_) (void)hipFree(dev_);
        dev_ = nullptr;
        hip_check(hipMalloc((void**)&dev_, 2 * want), "hipMalloc(field staging)");
        dev_cap_ = want;
    }
}

void Readback::read(size_t units, size_t unit_bytes, void* out, hipStream_t stream,
                    const std::function<hipError_t(size_t, size_t, double*)>& eval) {
    const size_t total = units * unit_bytes;
    if (total == 0) return;
    std::lock_guard<std::mutex> one(m_);
    if (total <= DIRECT) {
        reserve(total, false);
        hip_check(eval(0, units, (double*)pinned_), "field kernel");
        hip_check(hipStreamSynchronize(stream), "read field");
        std::memcpy(out, pinned_, total);
        return;
    }
    // four chunks, of 1 MB at least, so that small fields overlap too
    const size_t chunk = std::max(unit_bytes, std::min(CHUNK, std::max(CHUNK / 16, total / 4)));
    const size_t per = std::min(units, chunk / unit_bytes), chunks = (units + per - 1) / per;
    reserve(per * unit_bytes, true);
    for (hipEvent_t& e : done_)
        if (!e) hip_check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "event create");
    struct Drain {  // also a read that fails leaves nothing behind that writes to the buffers
        hipStream_t s;
        ~Drain() { (void)hipStreamSynchronize(s); }
    } drain{stream};
    // a thread for every 2 MB (for every 512 kB: U of 1024x256 400 us, not 311)
    Copier copier((unsigned)std::min<size_t>(8, 1 + total / (size_t(2) << 20)));
    const auto start = [&](size_t c) {
        const size_t b = c & 1, first = c * per, n = std::min(per, units - first);
        hip_check(eval(first, n, (double*)(dev_ + b * dev_cap_)), "field kernel");
        hip_check(hipMemcpyAsync(pinned_ + b * pinned_cap_, dev_ + b * dev_cap_, n * unit_bytes, hipMemcpyDeviceToHost, stream), "read field");
        hip_check(hipEventRecord(done_[b], stream), "event record");
    };
    start(0);
    for (size_t c = 0; c < chunks; c++) {
        if (c + 1 < chunks) start(c + 1);
        const size_t b = c & 1, first = c * per, n = std::min(per, units - first);
        hip_check(hipEventSynchronize(done_[b]), "read field");
        copier.copy((char*)out + first * unit_bytes, pinned_ + b * pinned_cap_, n * unit_bytes);
    }
}

}  // namespace tclbx
