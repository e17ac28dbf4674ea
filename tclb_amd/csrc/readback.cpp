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
constexpr size_t SMALL = size_t(128) << 10, HUGE_PAGE = size_t(2) << 20;

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
    if (pinned_) (void)hipHostFree(pinned_);
    for (hipEvent_t e : done_)
        if (e) (void)hipEventDestroy(e);
}

// in layers, in the rows of each layer where one is larger than a chunk, or in
// the nodes of each row
void Readback::read(int nx, int ny, int nz, size_t node_bytes, void* out, hipStream_t stream, const Eval& eval) {
    const size_t row = nx * node_bytes, layer = row * ny;
    char* const to = (char*)out;
    if (layer == 0 || nz <= 0) return;
    std::lock_guard<std::mutex> one(m_);
    if (nz > 1 && layer <= CHUNK) {
        read_units(nz, layer, to, stream, [&](int z, int n, double* d) { return eval(0, 0, z, nx, ny, n, d); });
        return;
    }
    for (int z = 0; z < nz; z++) {
        if (row <= CHUNK) {
            read_units(ny, row, to + layer * z, stream, [&](int y, int n, double* d) { return eval(0, y, z, nx, n, 1, d); });
            continue;
        }
        for (int y = 0; y < ny; y++)
            read_units(nx, node_bytes, to + layer * z + row * y, stream,
                       [&](int x, int n, double* d) { return eval(x, y, z, n, 1, 1, d); });
    }
}

void Readback::read_units(size_t units, size_t unit_bytes, char* out, hipStream_t stream,
                          const std::function<hipError_t(int, int, double*)>& eval) {
    const size_t total = units * unit_bytes;
    // four chunks, of 1 MB at least, so that small fields overlap too
    const size_t chunk = std::max(unit_bytes, std::min(CHUNK, std::max(CHUNK / 16, total / 4)));
    const size_t per = std::min(units, chunk / unit_bytes), chunks = (units + per - 1) / per;
    // Both buffers in one allocation, whole huge pages unless small: in 4 kB
    // pages the allocation and the first copy out of it cost about 0.5 ms each
    // per 2 MB.  Sized by the chunk, not by the units that fit in it, so that a
    // smaller field after a larger one fits.
    const size_t need = chunks == 1 ? total : 2 * chunk, page = need > SMALL ? HUGE_PAGE : 4096;
    if (cap_ < need) {
        const size_t want = (need + page - 1) / page * page;
        cap_ = 0;
        if (pinned_) (void)hipHostFree(pinned_);
        pinned_ = nullptr;
        hip_check(hipHostMalloc((void**)&pinned_, want, hipHostMallocDefault), "hipHostMalloc(field staging)");
        cap_ = want;
    }
    if (chunks == 1) {
        hip_check(eval(0, (int)units, (double*)pinned_), "field kernel");
        hip_check(hipStreamSynchronize(stream), "read field");
        std::memcpy(out, pinned_, total);
        return;
    }
    for (hipEvent_t& e : done_)
        if (!e) hip_check(hipEventCreateWithFlags(&e, hipEventDisableTiming | hipEventReleaseToSystem), "event create");
    struct Drain {  // also a read that fails leaves nothing behind that writes to the buffers
        hipStream_t s;
        ~Drain() { (void)hipStreamSynchronize(s); }
    } drain{stream};
    // a thread for every 2 MB (for every 512 kB: U of 1024x256 400 us, not 311)
    Copier copier((unsigned)std::min<size_t>(8, 1 + total / (size_t(2) << 20)));
    const auto buffer = [&](size_t c) { return pinned_ + (c & 1) * per * unit_bytes; };
    const auto start = [&](size_t c) {
        const size_t first = c * per, n = std::min(per, units - first);
        hip_check(eval((int)first, (int)n, (double*)buffer(c)), "field kernel");
        hip_check(hipEventRecord(done_[c & 1], stream), "event record");
    };
    start(0);
    for (size_t c = 0; c < chunks; c++) {
        if (c + 1 < chunks) start(c + 1);
        const size_t first = c * per, n = std::min(per, units - first);
        hip_check(hipEventSynchronize(done_[c & 1]), "read field");
        copier.copy(out + first * unit_bytes, buffer(c), n * unit_bytes);
    }
}

}  // namespace tclbx
