// hostcopy.hpp -- copies from device arrays to ordinary host memory.
//
// hipMemcpyAsync to pageable memory runs one thread through the runtime's own
// staging buffer: 100 MB into a fresh array take 9.7 ms (10 GB/s), of which the
// link needs 1.8; the rest is the host's memcpy and the first touch of the
// destination's pages, which several threads share.  HostStage::out moves
// chunks through pinned buffers, two per worker, so that one worker's memcpy
// overlaps the transfers of the others: 2.8 ms for 100 MB, 0.57 against 1.12 for
// 19 MB.  A chunk costs about 16 us beside its transfer (4 workers, 100 MB:
// 13.2 ms with 128 KB chunks, 4.8 with 512 KB, 2.8 with 2 MB), and 8 workers are
// no faster than 4.  Uploads gain nothing below 32 MB (19 MB: 0.62 ms against
// 0.54) and stay with the runtime, and so do copies to pinned memory, which it
// moves in one transfer (20 MB: 0.36 ms against 0.66 through the chunks, 106 MB:
// 1.86 against 2.71).
#pragma once

#include <hip/hip_runtime.h>

#include <memory>
#include <mutex>

class HostStage {
  public:
    HostStage() = default;
    HostStage(const HostStage&) = delete;
    HostStage& operator=(const HostStage&) = delete;
    ~HostStage();
    // Copies in order on st (a stream of the current device) and returns when
    // the host memory is written.  Makes the buffers if there are none yet and the
    // copy has `worth` bytes: fresh ones cost up to 2 ms where the runtime has
    // to pin their pages, which a solver's many reads pay once.
    hipError_t out(void* host, const void* dev, size_t bytes, hipStream_t st, size_t worth = 0);
    // The current device's stage, one for all who hold it (the buffers, 16 MB,
    // go when the last lets go); null if there is none to be had.
    static std::shared_ptr<HostStage> get();

  private:
    static constexpr int kWorkers = 4;                // the caller's thread included
    static constexpr size_t kChunk = size_t(2) << 20;
    static constexpr size_t kLeast = size_t(8) << 20;  // smaller copies go to the runtime
    std::mutex mu_;                 // held by the copy that uses the buffers; another goes to the runtime
    int device_ = 0;
    unsigned char* pin_ = nullptr;  // kWorkers x 2 chunks, allocated on first use
    hipEvent_t ev_[2 * kWorkers] = {};
    bool ready();
    hipError_t staged(unsigned char* host, const unsigned char* dev, size_t bytes, hipStream_t st);
};
