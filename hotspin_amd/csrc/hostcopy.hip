// hostcopy.hip -- staged copies from device to pageable host memory (hostcopy.hpp).
#include "hostcopy.hpp"

#include <string.h>

#include <algorithm>
#include <atomic>
#include <exception>
#include <map>
#include <new>
#include <thread>

std::shared_ptr<HostStage> HostStage::get() {
    static std::mutex mu;
    static std::map<int, std::weak_ptr<HostStage>> stages;
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) return nullptr;
    try {
        std::lock_guard<std::mutex> lk(mu);
        std::weak_ptr<HostStage>& w = stages[device];
        std::shared_ptr<HostStage> s = w.lock();
        if (!s) {
            s = std::make_shared<HostStage>();
            s->device_ = device;
            w = s;
        }
        return s;
    } catch (const std::bad_alloc&) {
        return nullptr;
    }
}

HostStage::~HostStage() {
    for (hipEvent_t e : ev_)
        if (e) (void)hipEventDestroy(e);
    if (pin_) (void)hipHostFree(pin_);
}

bool HostStage::ready() {
    if (pin_) return true;
    for (hipEvent_t& e : ev_)
        if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
            e = nullptr;
            (void)hipGetLastError();
            return false;
        }
    void* p = nullptr;
    if (hipHostMalloc(&p, 2 * kWorkers * kChunk, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    pin_ = static_cast<unsigned char*>(p);
    return true;
}

// Memory the runtime does not know: pinned, managed and device memory it copies
// to directly.
static bool pageable(const void* host) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, host) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return a.type == hipMemoryTypeUnregistered;
}

hipError_t HostStage::out(void* host, const void* dev, size_t bytes, hipStream_t st, size_t worth) {
    // hipStreamPerThread would be another stream in each worker
    if (bytes >= kLeast && st != hipStreamPerThread && std::thread::hardware_concurrency() >= 2 * kWorkers &&
        pageable(host)) {
        int device = -1;
        std::unique_lock<std::mutex> lk(mu_, std::try_to_lock);
        if (lk.owns_lock() && hipGetDevice(&device) == hipSuccess && device == device_ && (pin_ || bytes >= worth) &&
            ready())
            return staged(static_cast<unsigned char*>(host), static_cast<const unsigned char*>(dev), bytes, st);
    }
    const hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st);
    return e != hipSuccess ? e : hipStreamSynchronize(st);
}

hipError_t HostStage::staged(unsigned char* host, const unsigned char* dev, size_t bytes, hipStream_t st) {
    const size_t nch = (bytes + kChunk - 1) / kChunk;
    std::atomic<size_t> next{0};
    std::atomic<int> err{hipSuccess};
    auto run = [&](int w) {
        auto check = [&](hipError_t e) {
            int ok = hipSuccess;
            if (e != hipSuccess) err.compare_exchange_strong(ok, e);
            return e == hipSuccess;
        };
        if (!check(hipSetDevice(device_))) return;
        unsigned char* buf[2] = {pin_ + 2 * w * kChunk, pin_ + (2 * w + 1) * kChunk};
        hipEvent_t* ev = ev_ + 2 * w;
        size_t at[2] = {0, 0}, len[2] = {0, 0};  // the chunk in flight to each buffer
        auto land = [&](int b) {
            if (!len[b]) return true;
            if (!check(hipEventSynchronize(ev[b]))) return false;
            memcpy(host + at[b], buf[b], len[b]);
            len[b] = 0;
            return true;
        };
        for (int b = 0;; b ^= 1) {
            if (!land(b)) return;
            const size_t c = err.load() == hipSuccess ? next.fetch_add(1) : nch;
            if (c >= nch) {
                land(b ^ 1);
                return;
            }
            at[b] = c * kChunk;
            const size_t n = std::min(kChunk, bytes - at[b]);
            if (!check(hipMemcpyAsync(buf[b], dev + at[b], n, hipMemcpyDeviceToHost, st)) ||
                !check(hipEventRecord(ev[b], st)))
                return;
            len[b] = n;
        }
    };
    std::thread th[kWorkers];
    for (int w = 1; w < kWorkers; w++) {
        try {
            th[w] = std::thread(run, w);
        } catch (const std::exception&) {
            break;  // the workers there are take every chunk
        }
    }
    run(0);
    for (std::thread& t : th)
        if (t.joinable()) t.join();
    if (err.load() != hipSuccess) (void)hipStreamSynchronize(st);  // nothing in flight to the buffers
    return (hipError_t)err.load();
}
