// k-means (glass::Clustering, glass/algorithms/clustering.hpp): the engine the
// PQ8 trainer and the Clustering object of the C ABI share.  Seeding and the
// centroid update follow the reference step by step on the host (both are
// order-dependent: every k-means++ pick depends on the previous one, and a
// centroid is a float sum over its rows in row order) for PQ8's small
// sub-spaces; the Clustering object's sweeps, updates and distances run on
// the GPU (cluster_kernels.hip).
//
// Float steps are those of the reference as GCC -Ofast compiles it:
//   distances     helpa::l2_fp32_fp32 (l2 below, l2_helpa on the device)
//   seeding total in double: 8 floats per step into 4 lanes,
//                 a_l += d[8b+l] + d[8b+4+l], (a1 + a3) + (a0 + a2), one
//                 4-wide step (d1 + d3) + (d0 + d2), then one by one
//   centroid      sum * (1.0f / float(count))  (reciprocal math)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <random>
#include <string>
#include <vector>

#include "../../include/glass_hip.h"
#include "glass_hip_internal.h"

namespace glass_hip {
namespace km {

float l2(const float *x, const float *y, int32_t d) {
    const int32_t da = d / 16 * 16;
    float A = 0.0f;
    if (da > 0) {
        float a[16] = {0};
        for (int32_t i = 0; i < da; i += 16)
            for (int l = 0; l < 16; ++l) {
                const float t = x[i + l] - y[i + l];
                a[l] = std::fma(t, t, a[l]);
            }
        float b[8], c[4];
        for (int l = 0; l < 8; ++l) b[l] = a[l + 8] + a[l];
        for (int l = 0; l < 4; ++l) c[l] = b[l + 4] + b[l];
        A = (c[0] + c[2]) + (c[1] + c[3]);
    }
    float T = 0.0f;
    int32_t i = da;
    if (d - i >= 8) {
        float u[4];
        for (int l = 0; l < 4; ++l) {
            const float t0 = x[i + l] - y[i + l], t1 = x[i + 4 + l] - y[i + 4 + l];
            u[l] = t1 * t1 + t0 * t0;
        }
        T = (u[1] + u[3]) + (u[0] + u[2]);
        i += 8;
    }
    if (d - i >= 4) {
        float q[4];
        for (int l = 0; l < 4; ++l) {
            const float t = x[i + l] - y[i + l];
            q[l] = t * t;
        }
        T = T + ((q[1] + q[3]) + (q[0] + q[2]));
        i += 4;
    }
    for (; i < d; ++i) {
        const float t = x[i] - y[i];
        T = std::fma(t, t, T);
    }
    return A + T;
}

namespace {

double seed_total(const float *d, int32_t n) {
    double S = 0.0;
    int32_t i = 0;
    if (n >= 8) {
        double a[4] = {0.0, 0.0, 0.0, 0.0};
        for (; i + 8 <= n; i += 8)
            for (int l = 0; l < 4; ++l) a[l] = a[l] + ((double)d[i + 4 + l] + (double)d[i + l]);
        S = (a[1] + a[3]) + (a[0] + a[2]);
    }
    if (n - i >= 4) {
        S = S + (((double)d[i + 1] + (double)d[i + 3]) + ((double)d[i] + (double)d[i + 2]));
        i += 4;
    }
    for (; i < n; ++i) S = S + (double)d[i];
    return S;
}

}  // namespace

std::vector<int32_t> sample_rows(int32_t n) {
    const int32_t m = std::min(n - 1, 100000);  // kSampleNum (clustering.hpp:24,75)
    std::vector<int32_t> samples(std::max(m, 1));
    std::mt19937 rng;
    gen_random(rng, samples.data(), m, n);
    samples.resize(std::max(m, 0));
    return samples;
}

std::vector<int32_t> random_picks(int32_t m, int32_t k) {
    std::mt19937 r;
    std::vector<int32_t> idx(k);
    gen_random(r, idx.data(), k, m);
    return idx;
}

int kmeanspp_picks(int32_t m, int32_t k, const std::function<int(int32_t, float *)> &dist_to,
                   std::vector<int32_t> &picked) {
    std::mt19937 r;
    std::uniform_real_distribution<> dart_dist(0, 1);
    std::uniform_int_distribution<int32_t> first(0, m - 1);
    std::vector<float> dist(std::max(m, 1)), fresh(std::max(m, 1));
    const int32_t init_id = first(r);
    picked.assign(1, init_id);
    if (int e = dist_to(init_id, dist.data())) return e;
    bool sum_flag = false;
    while ((int32_t)picked.size() < k) {
        double dart = dart_dist(r);
        const double sum = seed_total(dist.data(), m);
        if (sum < 1e-6) sum_flag = true;
        dart *= sum;
        double prefix = 0.0;
        int32_t pivot = 0;
        for (int32_t i = 0; i < m; ++i) {
            pivot = i;
            const double next = prefix + (double)dist[i];
            if (dart >= prefix && dart < next) break;
            prefix = next;
        }
        if (std::find(picked.begin(), picked.end(), pivot) != picked.end() && !sum_flag) continue;
        picked.push_back(pivot);
        if (int e = dist_to(pivot, fresh.data())) return e;
        for (int32_t i = 0; i < m; ++i) dist[i] = std::min(dist[i], fresh[i]);
    }
    return 0;
}

// Lloyd steps: compute_dist + find_index, update_mediods (clustering.hpp:198-256)
void fit_host(const float *rows, int32_t n, int32_t d, int32_t k, int32_t epochs, float *centroids) {
    const std::vector<int32_t> samples = sample_rows(n);
    const int32_t m = (int32_t)samples.size();
    std::vector<float> tr((size_t)d * std::max(m, 1));
    for (int32_t i = 0; i < m; ++i) std::memcpy(&tr[(size_t)d * i], rows + (int64_t)d * samples[i], 4 * (size_t)d);
    std::vector<int32_t> picks;
    (void)kmeanspp_picks(
        m, k,
        [&](int32_t p, float *out) {
            for (int32_t i = 0; i < m; ++i) out[i] = l2(&tr[(size_t)d * p], &tr[(size_t)d * i], d);
            return 0;
        },
        picks);
    for (int32_t c = 0; c < k; ++c) std::memcpy(centroids + (size_t)d * c, &tr[(size_t)d * picks[c]], 4 * (size_t)d);
    std::vector<int32_t> idx(std::max(m, 1)), cnt(k);
    std::vector<float> nm((size_t)d * k);
    for (int32_t e = 0; e < epochs; ++e) {
        for (int32_t i = 0; i < m; ++i) {
            float best = HUGE_VALF;
            idx[i] = -1;
            for (int32_t c = 0; c < k; ++c) {
                const float v = l2(&tr[(size_t)d * i], centroids + (size_t)d * c, d);
                if (v < best) {
                    best = v;
                    idx[i] = c;
                }
            }
        }
        std::fill(nm.begin(), nm.end(), 0.0f);
        std::fill(cnt.begin(), cnt.end(), 0);
        for (int32_t i = 0; i < m; ++i) {
            if (idx[i] < 0) continue;  // no centroid compares less than +inf (NaN rows)
            cnt[idx[i]]++;
            float *to = &nm[(size_t)d * idx[i]];
            const float *from = &tr[(size_t)d * i];
            for (int32_t j = 0; j < d; ++j) to[j] += from[j];
        }
        for (int32_t c = 0; c < k; ++c) {
            if (cnt[c] == 0) continue;
            const float rcp = 1.0f / (float)cnt[c];
            for (int32_t j = 0; j < d; ++j) nm[(size_t)d * c + j] *= rcp;
        }
        std::copy(nm.begin(), nm.end(), centroids);
    }
}

}  // namespace km

namespace {

// One device allocation that the arrays of a call are placed in.
struct Arena {
    uint8_t *p = nullptr;
    size_t used = 0;
    Arena() = default;
    Arena(const Arena &) = delete;
    Arena &operator=(const Arena &) = delete;
    ~Arena() {
        if (p) (void)hipFree(p);
    }
    size_t add(size_t bytes) {  // offset of the next array
        const size_t at = used;
        used += (bytes + 255) / 256 * 256;
        return at;
    }
    hipError_t alloc() { return hipMalloc((void **)&p, std::max<size_t>(used, 1)); }
    template <typename T>
    T *at(size_t offset) const {
        return (T *)(p + offset);
    }
};

int hip_fail(hipError_t e, const char *what) {
    std::string msg = std::string(what) + " failed: " + hipGetErrorString(e);
    return set_error(e == hipErrorOutOfMemory ? GLASS_HIP_ENOMEM : GLASS_HIP_EDEVICE, msg.c_str());
}

#define CL_TRY(expr)                                    \
    do {                                                \
        hipError_t _e = (expr);                         \
        if (_e != hipSuccess) return hip_fail(_e, #expr); \
    } while (0)

// Clustering::fit with everything but the seeding's picks on the device.  The
// sample is gathered there too unless it is a small part of the rows.
int fit_device(const float *rows, int32_t n, int32_t d, int32_t k, int32_t epochs, bool kmeanspp, float *centroids) {
    const std::vector<int32_t> samples = km::sample_rows(n);
    const int32_t m = (int32_t)samples.size();
    const bool whole = (int64_t)n <= 4 * (int64_t)m;
    Arena a;
    const size_t o_all = a.add(whole ? 4 * (size_t)n * d : 0), o_rows = a.add(4 * (size_t)std::max(m, k)),
                 o_x = a.add(4 * (size_t)m * d), o_cent = a.add(4 * (size_t)k * d), o_ids = a.add(4 * (size_t)m),
                 o_dist = a.add(4 * (size_t)m),
                 o_scratch = a.add(filter_pays(m, d, k) ? AssignScratch::bytes(m, k) : 0);
    CL_TRY(a.alloc());
    float *x = a.at<float>(o_x), *cent = a.at<float>(o_cent);
    int32_t *idx = a.at<int32_t>(o_rows), *ids = a.at<int32_t>(o_ids);
    AssignScratch s;
    s.place(a.p + o_scratch, m, k);
    if (whole) {
        CL_TRY(hipMemcpy(a.at<float>(o_all), rows, 4 * (size_t)n * d, hipMemcpyHostToDevice));
        CL_TRY(hipMemcpy(idx, samples.data(), 4 * (size_t)m, hipMemcpyHostToDevice));
        CL_TRY(launch_cluster_gather(a.at<float>(o_all), idx, m, d, x, nullptr));
    } else {
        std::vector<float> tr((size_t)d * m);
        for (int32_t i = 0; i < m; ++i) std::memcpy(&tr[(size_t)d * i], rows + (int64_t)d * samples[i], 4 * (size_t)d);
        CL_TRY(hipMemcpy(x, tr.data(), 4 * (size_t)m * d, hipMemcpyHostToDevice));
    }
    std::vector<int32_t> picks;
    if (kmeanspp) {
        float *dist = a.at<float>(o_dist);
        const int e = km::kmeanspp_picks(
            m, k,
            [&](int32_t p, float *out) -> int {
                CL_TRY(launch_cluster_dist(x, m, d, x + (int64_t)p * d, dist, nullptr));
                CL_TRY(hipMemcpy(out, dist, 4 * (size_t)m, hipMemcpyDeviceToHost));
                return 0;
            },
            picks);
        if (e) return e;
    } else {
        picks = km::random_picks(m, k);
    }
    CL_TRY(hipMemcpy(idx, picks.data(), 4 * (size_t)k, hipMemcpyHostToDevice));
    CL_TRY(launch_cluster_gather(x, idx, k, d, cent, nullptr));
    CL_TRY(launch_cluster_norms(x, m, d, s, nullptr));
    for (int32_t e = 0; e < epochs; ++e) {
        CL_TRY(launch_cluster_assign(x, m, d, cent, k, ids, s, nullptr));
        CL_TRY(launch_cluster_update(x, m, d, ids, k, cent, nullptr));
    }
    CL_TRY(hipMemcpy(centroids, cent, 4 * (size_t)k * d, hipMemcpyDeviceToHost));
    return GLASS_HIP_OK;
}

// A clustering object's stream and events, made by the first call that has
// pieces to overlap and kept with it (making them takes 0.05 ms, and 3 the
// first few times in a process); one call at a time.  They belong to the
// device that was current then: a call under another one makes its own.
struct Device {
    std::mutex mu;
    int index = -1;
    hipStream_t stream = nullptr;
    hipEvent_t done[2] = {nullptr, nullptr};
    ~Device() { release(); }
    void release() {
        for (hipEvent_t &e : done) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
        if (stream) (void)hipStreamDestroy(stream);
        stream = nullptr;
    }
    int make() {  // for the current device
        int current = 0;
        CL_TRY(hipGetDevice(&current));
        if (current != index) release();
        index = current;
        if (!stream) CL_TRY(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
        for (hipEvent_t &e : done)
            if (!e) CL_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        return GLASS_HIP_OK;
    }
};

// Nearest centroid of every row.  More than 24 MB of rows go to the device in
// pieces of about 16 MB while the piece before is worked on: the copy bounds the
// call.  Fewer go in one: 35,000 x 128 (18 MB) to 16 and 1,000 clusters take 630
// and 850 us in two pieces, 595 and 840 in one, and the first call of a process
// 5.5 ms, 2.2 in one: a stream is another hardware queue.  200,000 x 96 (77 MB)
// to 1,000: 3,090 in pieces, 3,700 in one.
int predict_device(Device &dev, const float *cent, int32_t k, int32_t d, const float *x, int32_t n, int32_t *ids) {
    const int64_t piece = std::max<int64_t>(64, ((int64_t)4 << 20) / d / 64 * 64);
    const int32_t rows = (int64_t)n * d <= (6 << 20) ? n : (int32_t)std::min<int64_t>(n, piece);
    const int32_t bufs = n > rows ? 2 : 1;
    if (bufs > 1)
        if (const int r = dev.make()) return r;
    const hipStream_t stream = bufs > 1 ? dev.stream : nullptr;
    Arena a;
    const size_t o_x = a.add(4 * (size_t)rows * d * bufs), o_cent = a.add(4 * (size_t)k * d),
                 o_ids = a.add(4 * (size_t)n),
                 o_scratch = a.add(filter_pays(rows, d, k) ? AssignScratch::bytes(rows, k) : 0);
    CL_TRY(a.alloc());
    struct Drain {  // before the arena goes; freeing it waits for the null stream
        hipStream_t s;
        ~Drain() {
            if (s) (void)hipStreamSynchronize(s);
        }
    } drain{stream};
    float *dc = a.at<float>(o_cent);
    int32_t *di = a.at<int32_t>(o_ids);
    AssignScratch s;
    int32_t turn = 0;
    for (int64_t at = 0; at < n; at += rows, ++turn) {
        const int32_t c = (int32_t)std::min<int64_t>(rows, n - at);
        const int32_t b = turn % bufs;
        float *dx = a.at<float>(o_x) + (size_t)b * rows * d;
        if (turn >= 2) CL_TRY(hipEventSynchronize(dev.done[b]));
        CL_TRY(hipMemcpy(dx, x + at * d, 4 * (size_t)c * d, hipMemcpyHostToDevice));
        if (turn == 0) CL_TRY(hipMemcpy(dc, cent, 4 * (size_t)k * d, hipMemcpyHostToDevice));
        s.place(a.p + o_scratch, c, k);
        CL_TRY(launch_cluster_norms(dx, c, d, s, stream));
        CL_TRY(launch_cluster_assign(dx, c, d, dc, k, di + at, s, stream));
        if (bufs > 1) CL_TRY(hipEventRecord(dev.done[b], stream));
    }
    // a copy that waits for work in flight takes 60 us longer than a wait and a
    // copy, and 8 us less where that work is short
    if (stream || filter_pays(rows, d, k)) CL_TRY(hipStreamSynchronize(stream));
    CL_TRY(hipMemcpy(ids, di, 4 * (size_t)n, hipMemcpyDeviceToHost));
    return GLASS_HIP_OK;
}

}  // namespace
}  // namespace glass_hip

using namespace glass_hip;

struct glass_hip_clustering {
    int32_t k = 0, epochs = 10, dim = 0;
    bool kmeanspp = false;
    std::vector<float> centroids;
    mutable Device dev;
};

extern "C" {

int glass_hip_clustering_create(int32_t n_cluster, int32_t epochs, const char *init, glass_hip_clustering **out) {
    try {
        if (!out || n_cluster < 1 || epochs < 0) return set_error(GLASS_HIP_EINVAL, "bad clustering arguments");
        const std::string in = init ? init : "random";
        if (in != "random" && in != "kmeans++")
            return set_error(GLASS_HIP_EINVAL, "init must be \"random\" or \"kmeans++\"");
        auto *c = new glass_hip_clustering;
        c->k = n_cluster;
        c->epochs = epochs;
        c->kmeanspp = in == "kmeans++";
        *out = c;
        return GLASS_HIP_OK;
    } catch (...) {
        return exception_status();
    }
}

void glass_hip_clustering_free(glass_hip_clustering *c) { delete c; }

int glass_hip_clustering_fit(glass_hip_clustering *c, const float *data, int32_t n, int32_t dim) {
    try {
        if (!c || !data || dim <= 0) return set_error(GLASS_HIP_EINVAL, "bad clustering input");
        // the fit samples min(n - 1, 100000) rows; random seeding draws k
        // distinct ones of them (GenRandom's draws are modulo their difference)
        if (n < 2 || (!c->kmeanspp && std::min(n - 1, 100000) <= c->k))
            return set_error(GLASS_HIP_EINVAL, "too few sampled rows for the number of clusters");
        std::vector<float> cent((size_t)c->k * dim);
        if (const int r = fit_device(data, n, dim, c->k, c->epochs, c->kmeanspp, cent.data())) return r;
        c->centroids.swap(cent);
        c->dim = dim;
        return GLASS_HIP_OK;
    } catch (...) {
        return exception_status();
    }
}

int glass_hip_clustering_predict(const glass_hip_clustering *c, const float *data, int32_t n, int32_t dim,
                                 int32_t *ids) {
    try {
        if (!c || !data || !ids || n < 0) return set_error(GLASS_HIP_EINVAL, "bad clustering input");
        if (c->dim == 0) return set_error(GLASS_HIP_ESTATE, "clustering not fitted");
        if (dim != c->dim) {
            char msg[96];
            std::snprintf(msg, sizeof(msg), "data has dim %d, the centroids %d", dim, c->dim);
            return set_error(GLASS_HIP_EINVAL, msg);
        }
        if (n == 0) return GLASS_HIP_OK;
        std::lock_guard<std::mutex> lk(c->dev.mu);
        return predict_device(c->dev, c->centroids.data(), c->k, dim, data, n, ids);
    } catch (...) {
        return exception_status();
    }
}

int glass_hip_clustering_transform(const glass_hip_clustering *c, float *data, int32_t n, int32_t dim) {
    try {
        std::vector<int32_t> ids(std::max(n, 1));
        if (int r = glass_hip_clustering_predict(c, data, n, dim, ids.data())) return r;
        for (int32_t i = 0; i < n; ++i) {
            if (ids[i] < 0) continue;  // a row with no nearest centroid is left as it is
            const float *ctr = &c->centroids[(size_t)dim * ids[i]];
            for (int32_t j = 0; j < dim; ++j) data[(int64_t)dim * i + j] -= ctr[j];
        }
        return GLASS_HIP_OK;
    } catch (...) {
        return exception_status();
    }
}

int glass_hip_clustering_centroids(const glass_hip_clustering *c, float *out, int32_t *n_cluster, int32_t *dim) {
    try {
        if (!c) return set_error(GLASS_HIP_EINVAL, "null clustering");
        if (n_cluster) *n_cluster = c->k;
        if (dim) *dim = c->dim;
        if (out && c->dim) std::copy(c->centroids.begin(), c->centroids.end(), out);
        return GLASS_HIP_OK;
    } catch (...) {
        return exception_status();
    }
}

}  // extern "C"
