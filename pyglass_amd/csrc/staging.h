// Copies of large host arrays to the device, through pinned buffers that two
// threads fill in turn with the copies of what they filled before.  The
// runtime's own copy of pageable memory reaches 30 GB/s here and the link 57:
// 256 MB take 9.1 ms by hipMemcpy and 5.9 ms by two threads with two 4 MB
// buffers each, set-up included (one thread 12.6, four 6.7, eight 10.3).
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
    Stager() = default;
    Stager(const Stager &) = delete;
    Stager &operator=(const Stager &) = delete;
    ~Stager() {
        for (Lane &ln : lanes_) {
            for (hipEvent_t e : ln.sent)
                if (e) (void)hipEventDestroy(e);
            if (ln.stream) (void)hipStreamDestroy(ln.stream);
            if (ln.host) (void)hipHostFree(ln.host);
        }
    }

    // Returns once dst (device memory) holds the `bytes` at src.  One call at
    // a time per object.
    hipError_t upload(void *dst, const void *src, size_t bytes) {
        if (bytes < (state_ == 1 ? 2 * kPiece : kWorth) || !ready()) return hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice);
        int device = 0;
        if (hipError_t e = hipGetDevice(&device)) return e;
        std::atomic<size_t> next{0};
        std::atomic<int> failed{hipSuccess};
        auto work = [&](Lane &ln) {
            hipError_t e = hipSetDevice(device);
            for (int turn = 0; e == hipSuccess && failed == hipSuccess; ++turn) {
                const size_t at = next.fetch_add(kPiece);
                if (at >= bytes) break;
                const size_t n = std::min(kPiece, bytes - at);
                uint8_t *buf = ln.host + (turn & 1) * kPiece;
                if (turn >= 2) e = hipEventSynchronize(ln.sent[turn & 1]);
                if (e != hipSuccess) break;
                std::memcpy(buf, (const uint8_t *)src + at, n);
                e = hipMemcpyAsync((uint8_t *)dst + at, buf, n, hipMemcpyHostToDevice, ln.stream);
                if (e == hipSuccess) e = hipEventRecord(ln.sent[turn & 1], ln.stream);
            }
            const hipError_t last = hipStreamSynchronize(ln.stream);
            if (e == hipSuccess) e = last;
            if (e != hipSuccess) failed = e;
        };
        std::thread other;
        try {
            other = std::thread([&] { work(lanes_[1]); });
        } catch (const std::system_error &) {  // this thread copies it all
        }
        work(lanes_[0]);
        if (other.joinable()) other.join();
        return (hipError_t)failed.load();
    }

private:
    static constexpr size_t kPiece = (size_t)4 << 20;
    // the first copy that pays for making buffers and streams: an index of
    // 14 MB of rows loads in 1.53 ms with and 1.34 without, one of 38 MB in
    // 2.17 and 2.35
    static constexpr size_t kWorth = (size_t)32 << 20;
    struct Lane {
        uint8_t *host = nullptr;  // two pieces, pinned
        hipStream_t stream = nullptr;
        hipEvent_t sent[2] = {nullptr, nullptr};
    };
    Lane lanes_[2];
    int state_ = 0;  // 0 not tried, 1 ready, 2 not available

    bool ready() {
        if (state_ == 0) {
            state_ = 1;
            for (Lane &ln : lanes_) {
                if (hipHostMalloc((void **)&ln.host, 2 * kPiece, hipHostMallocDefault) != hipSuccess ||
                    hipStreamCreateWithFlags(&ln.stream, hipStreamNonBlocking) != hipSuccess)
                    state_ = 2;
                for (hipEvent_t &e : ln.sent)
                    if (state_ == 1 && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) state_ = 2;
                if (state_ == 2) {
                    (void)hipGetLastError();
                    break;
                }
            }
        }
        return state_ == 1;
    }
};

}  // namespace glass_hip
