// clustering.cpp's device path over a stand-in for the HIP runtime with two
// devices, on the CPU: "device" memory is host memory, every stream and event
// belongs to the device that was current when it was made, and work queued on
// one while another device is current fails the program.  Kernels are plain
// loops.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "glass_hip.h"
#include "glass_hip_internal.h"

namespace {

int g_current = 0, g_live = 0;

struct Owned {
    int device;
};

Owned *own() {
    ++g_live;
    return new Owned{g_current};
}

void disown(void *p) {
    --g_live;
    delete (Owned *)p;
}

void check(const void *p, const char *what) {
    if (p && ((const Owned *)p)->device != g_current) {
        std::printf("%s of device %d used while device %d is current\n", what, ((const Owned *)p)->device, g_current);
        std::exit(1);
    }
}

}  // namespace

extern "C" {
hipError_t hipGetDevice(int *d) {
    *d = g_current;
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) { return (*p = std::malloc(n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void *p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = (hipStream_t)own();
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    disown(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = (hipEvent_t)own();
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    disown(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    check(e, "event");
    check(s, "stream");
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
}

namespace glass_hip {

int set_error(int code, const char *msg) {
    std::printf("error: %s\n", msg);
    return code;
}
int exception_status() noexcept { return -1; }
void gen_random(std::mt19937 &, int32_t *addr, int32_t size, int32_t) {
    for (int32_t i = 0; i < size; ++i) addr[i] = i;
}

size_t AssignScratch::bytes(int32_t, int32_t) { return 16; }
void AssignScratch::place(void *, int32_t, int32_t) {}

hipError_t launch_cluster_norms(const float *, int32_t, int32_t, const AssignScratch &, hipStream_t s) {
    check(s, "stream");
    return hipSuccess;
}
hipError_t launch_cluster_assign(const float *x, int32_t n, int32_t d, const float *cent, int32_t k, int32_t *ids,
                                 const AssignScratch &, hipStream_t s) {
    check(s, "stream");
    for (int32_t i = 0; i < n; ++i) {
        float best = 1e30f;
        for (int32_t c = 0; c < k; ++c) {
            const float t = x[(int64_t)i * d] - cent[(int64_t)c * d];
            if (t * t < best) {
                best = t * t;
                ids[i] = c;
            }
        }
    }
    return hipSuccess;
}
hipError_t launch_cluster_dist(const float *, int32_t, int32_t, const float *, float *, hipStream_t s) {
    check(s, "stream");
    return hipSuccess;
}
hipError_t launch_cluster_update(const float *, int32_t, int32_t, const int32_t *, int32_t, float *, hipStream_t s) {
    check(s, "stream");
    return hipSuccess;
}
hipError_t launch_cluster_gather(const float *x, const int32_t *rows, int32_t m, int32_t d, float *out, hipStream_t s) {
    check(s, "stream");
    for (int32_t i = 0; i < m; ++i) std::memcpy(out + (int64_t)i * d, x + (int64_t)rows[i] * d, 4 * (size_t)d);
    return hipSuccess;
}

}  // namespace glass_hip

int main() {
    constexpr int32_t kDim = 40000, kRows = 300;  // pieces of 64 rows
    std::vector<float> x((size_t)kRows * kDim);
    for (int32_t i = 0; i < kRows; ++i) x[(size_t)i * kDim] = (float)(i % 3);
    std::vector<int32_t> ids(kRows);
    glass_hip_clustering *c = nullptr;
    if (glass_hip_clustering_create(3, 1, "random", &c) || glass_hip_clustering_fit(c, x.data(), kRows, kDim)) return 2;
    for (int device : {0, 1, 1, 0}) {
        g_current = device;
        for (int32_t n : {kRows, 64}) {
            std::fill(ids.begin(), ids.end(), -1);
            if (glass_hip_clustering_predict(c, x.data(), n, kDim, ids.data())) return 3;
            for (int32_t i = 0; i < n; ++i)
                if (ids[i] != i % 3) return 4;
        }
        if (g_live != 3) return 5;  // a stream and two events, whichever device has them
    }
    glass_hip_clustering_free(c);
    return g_live == 0 ? 0 : 6;
}
