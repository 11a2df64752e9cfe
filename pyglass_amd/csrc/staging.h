// Copies of large host arrays to the device, through pinned buffers that two
// threads fill in turn with the copies of what they filled before.  The
// runtime's own copy of pageable memory reaches 30 GB/s here and the link 57:
// an index of 500,000 x 128 (256 MB of rows, 64 MB of graph) loads in 11.2 ms,
// 42 by hipMemcpy.  Filling takes two threads (one 12.6 ms for 256 MB, two 5.9,
// four 6.7).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>

namespace glass_hip {

class Stager {
public:
    // Copies go through `stream`, which has to outlive the object.  A stream of
    // their own would be a hardware queue more, 3 ms the first few times in a
    // process, and the link carries one copy at a time anyway.
    explicit Stager(hipStream_t stream) : stream_(stream) {}
    Stager(const Stager &) = delete;
    Stager &operator=(const Stager &) = delete;
    ~Stager() {
        for (hipEvent_t e : sent_)
            if (e) (void)hipEventDestroy(e);
        if (host_) (void)hipHostFree(host_);
    }

    // Returns once dst (device memory) holds the `bytes` at src.  One call at
    // a time per object.
    hipError_t upload(void *dst, const void *src, size_t bytes) {
        if (bytes < (state_ == 1 ? 4 * kPiece : kWorth) || !ready()) return hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice);
        int device = 0;
        if (hipError_t e = hipGetDevice(&device)) return e;
        std::atomic<size_t> next{0};
        std::atomic<int> failed{hipSuccess};
        auto work = [&](int lane) {
            hipError_t e = hipSetDevice(device);
            for (int turn = 0; e == hipSuccess && failed == hipSuccess; ++turn) {
                const size_t at = next.fetch_add(kPiece);
                if (at >= bytes) break;
                const size_t n = std::min(kPiece, bytes - at);
                const int b = 2 * lane + (turn & 1);
                uint8_t *buf = host_ + b * kPiece;
                if (turn >= 2) e = hipEventSynchronize(sent_[b]);
                if (e != hipSuccess) break;
                std::memcpy(buf, (const uint8_t *)src + at, n);
                e = hipMemcpyAsync((uint8_t *)dst + at, buf, n, hipMemcpyHostToDevice, stream_);
                if (e == hipSuccess) e = hipEventRecord(sent_[b], stream_);
            }
            if (e != hipSuccess) failed = e;
        };
        std::thread other;
        try {
            other = std::thread([&] { work(1); });
        } catch (const std::system_error &) {  // this thread copies it all
        }
        work(0);
        if (other.joinable()) other.join();
        const hipError_t last = hipStreamSynchronize(stream_);
        return failed != hipSuccess ? (hipError_t)failed.load() : last;
    }

private:
    // A first load pays for touching the pinned pages, 0.4 ms per MB, a later
    // one for small copies.  Loads of 70,000 and 500,000 x 128, first in a
    // process / later, ms: pieces of 1 MB 7.8 / 2.5 and 18.1 / 13.3, of 2 MB
    // 8.3 / 2.3 and 16.6 / 11.2, of 4 MB 9.9 / 2.3 and 17.3 / 10.5; hipMemcpy
    // 11.9 / 4.9 and 50.5 / 42.2.
    static constexpr size_t kPiece = (size_t)2 << 20;
    // The first copy that pays for that: 33 MB of rows load first in 9.0 ms with
    // it and 7.6 without, later in 2.3 and 2.5; 75 MB about even at first.
    static constexpr size_t kWorth = (size_t)32 << 20;
    hipStream_t stream_;
    uint8_t *host_ = nullptr;  // two pieces for each of two threads, pinned
    hipEvent_t sent_[4] = {nullptr, nullptr, nullptr, nullptr};
    int state_ = 0;  // 0 not tried, 1 ready, 2 not available

    bool ready() {
        if (state_ == 0) {
            state_ = hipHostMalloc((void **)&host_, 4 * kPiece, hipHostMallocDefault) == hipSuccess ? 1 : 2;
            for (hipEvent_t &e : sent_)
                if (state_ == 1 && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) state_ = 2;
            if (state_ == 2) (void)hipGetLastError();
        }
        return state_ == 1;
    }
};

}  // namespace glass_hip
