// k-means kernels: nearest centroids (Clustering::compute_dist + find_index,
// glass/algorithms/clustering.hpp:198-232), the centroid update
// (clustering.hpp:234-256) and the distances of k-means++ seeding
// (clustering.hpp:138-196).  Every result is bit-equal to the reference's.
#include <algorithm>

#include "glass_hip_internal.h"

namespace glass_hip {

namespace {

// helpa::l2_fp32_fp32 for any d (x86/l2_impl.hpp:14-18,50-71 with
// ref/l2_ref.hpp:7-15), rounded as GCC -Ofast compiles it for the reference:
// the 16-lane body accumulates fma(t, t, a_l) for elements l, l+16, ... and
// reduces b_i = a_(i+8) + a_i, c_i = b_(i+4) + b_i, (c0 + c2) + (c1 + c3);
// the tail of d mod 16 elements takes one 8-wide step (squares rounded,
// u_i = s_(i+4) + s_i, (u1 + u3) + (u0 + u2)), one 4-wide step
// ((s1 + s3) + (s0 + s2), added), then fused multiply-adds; body + tail.
// C rows y, y + d, ... at once: out[c] is x's distance to the c-th.
template <int C, typename Y>
__device__ __forceinline__ void l2_helpa(const float *x, Y y, int32_t d, float (&out)[C]) {
    const int32_t da = d / 16 * 16;
    float A[C], T[C];
#pragma unroll
    for (int c = 0; c < C; ++c) A[c] = T[c] = 0.0f;
    if (da > 0) {
        float a[C][16];
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int l = 0; l < 16; ++l) a[c][l] = 0.0f;
        for (int32_t i = 0; i < da; i += 16) {
#pragma unroll
            for (int c = 0; c < C; ++c)
#pragma unroll
                for (int l = 0; l < 16; ++l) {
                    const float t = x[i + l] - y[(int64_t)c * d + i + l];
                    a[c][l] = fmaf(t, t, a[c][l]);
                }
        }
#pragma unroll
        for (int c = 0; c < C; ++c) {
            float b[8], q[4];
#pragma unroll
            for (int l = 0; l < 8; ++l) b[l] = a[c][l + 8] + a[c][l];
#pragma unroll
            for (int l = 0; l < 4; ++l) q[l] = b[l + 4] + b[l];
            A[c] = (q[0] + q[2]) + (q[1] + q[3]);
        }
    }
    int32_t i = da;
    if (d - i >= 8) {
#pragma unroll
        for (int c = 0; c < C; ++c) {
            float u[4];
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                const float t0 = x[i + l] - y[(int64_t)c * d + i + l];
                const float t1 = x[i + 4 + l] - y[(int64_t)c * d + i + 4 + l];
                u[l] = t1 * t1 + t0 * t0;
            }
            T[c] = (u[1] + u[3]) + (u[0] + u[2]);
        }
        i += 8;
    }
    if (d - i >= 4) {
#pragma unroll
        for (int c = 0; c < C; ++c) {
            float q[4];
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                const float t = x[i + l] - y[(int64_t)c * d + i + l];
                q[l] = t * t;
            }
            T[c] = T[c] + ((q[1] + q[3]) + (q[0] + q[2]));
        }
        i += 4;
    }
    for (; i < d; ++i) {
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const float t = x[i] - y[(int64_t)c * d + i];
            T[c] = fmaf(t, t, T[c]);
        }
    }
#pragma unroll
    for (int c = 0; c < C; ++c) out[c] = A[c] + T[c];
}

// ---------------------------------------------------------------------------
// Nearest centroids.  The reference's distance is a chain of n * k * d
// subtractions and fused multiply-adds in a fixed order, which no matrix
// instruction gives; but only the index of the least one is asked for.  So
//   filter   a_ij = |c_j|^2 - 2 x_i.c_j on the matrix cores, keeping per row
//            the least value, its index and the second least value;
//   decide   where the two differ by more than both roundings can move them,
//            the least one's index is the reference's answer;
//   exact    the other rows, in the reference's order.
// With u = 2^-24, S = (|x| + max |c|)^2: the reference's value is within
// (d + 16) u S of |x - c|^2 and a_ij + |x|^2 within (d + 4) u S, so a gap above
// (4d + 40) u S decides; 5 (d + 16) u S is asked for.  Rows whose S is not in
// [1e-28, 1e36] (underflow, overflow, infinities, NaN) go to the exact kernel.

// The squared norm of every row, one wave per row; its maximum as float bits
// (NaN compares above everything) where `most` is given.
__global__ __launch_bounds__(256) void cluster_norms_kernel(const float *x, int32_t n, int32_t d, float *out,
                                                            uint32_t *most) {
    const int l = threadIdx.x & 63;
    for (int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); i < n; i += (int64_t)gridDim.x * 4) {
        float s = 0.0f;
        for (int32_t j = l; j < d; j += 64) s = fmaf(x[i * d + j], x[i * d + j], s);
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
        if (l == 0) {
            out[i] = s;
            if (most) atomicMax(most, __float_as_uint(s) & 0x7fffffffu);
        }
    }
}

struct Best {
    float m1, m2;  // the least and the second least value
    int32_t i1;    // the least one's index
};

__device__ __forceinline__ Best better(Best a, Best b) {
    const bool lt = b.m1 < a.m1;
    Best r;
    r.m1 = lt ? b.m1 : a.m1;
    r.i1 = lt ? b.i1 : a.i1;
    r.m2 = fminf(lt ? a.m1 : b.m1, lt ? b.m2 : a.m2);
    return r;
}

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kRows = 64;    // rows per workgroup
constexpr int kCents = 256;  // centroids per step: 64 for each of its 4 waves
constexpr int kDims = 16;    // dimensions staged at a time
constexpr int kLd = 20;      // floats per staged row: 16 lanes' 16-byte reads fall on distinct banks

// Bound by the matrix cores: a wave's 64 centroids x 64 rows take 32 MFMAs
// (2,048 cycles) per 16 dimensions against 8 16-byte LDS reads, and the two
// least values cost 6 vector instructions per product, hidden under them.
// Centroids are the MFMA's rows, so that a lane holds 16 centroids' products
// of one data row and keeps their least two to itself until the end; an
// 64-row tile leaves 1,563 workgroups for 100,000 rows, six per CU.
// 100k x 128 rows, 1,024 centroids: 8,080 us per sweep by one thread per row, now
// 328 us here (80 TFLOP/s) and 50 us in the kernels around it.
__global__ __launch_bounds__(256) void cluster_filter_kernel(const float *x, int32_t n, int32_t d, const float *cent,
                                                             int32_t k, const float *c2, int32_t tiles, float *m1,
                                                             float *m2, int32_t *i1) {
    __shared__ __align__(16) float sa[kCents * kLd], sb[kRows * kLd], sc[kCents];
    __shared__ Best best[4][kRows];
    const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
    const int h = l >> 5, li = l & 31;
    const int64_t row0 = (int64_t)blockIdx.x * kRows;
    const int t0 = blockIdx.y * tiles;
    const int col = tid & 15, sub = tid >> 4;  // staged element: dimension col of row sub + 16 q
    Best b[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) b[j] = Best{__builtin_inff(), __builtin_inff(), -1};
    for (int t = t0; t < t0 + tiles && t * kCents < k; ++t) {
        const int c0 = t * kCents;
        f32x16 acc[2][2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
        float ra[16], rb[4];
        auto fetch = [&](int kc) __attribute__((always_inline)) {
            const bool in = kc + col < d;
            const int at = in ? kc + col : 0;
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int c = c0 + sub + 16 * q;
                const float v = cent[(int64_t)(c < k ? c : k - 1) * d + at];
                ra[q] = in ? v : 0.0f;
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int64_t r = row0 + sub + 16 * q;
                const float v = x[(r < n ? r : n - 1) * d + at];
                rb[q] = in ? v : 0.0f;
            }
        };
        fetch(0);
        __syncthreads();  // the last step's reads of sc are done
        sc[tid] = c0 + tid < k ? c2[c0 + tid] : __builtin_inff();
        for (int kc = 0; kc < d; kc += kDims) {
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 16; ++q) sa[(sub + 16 * q) * kLd + col] = ra[q];
#pragma unroll
            for (int q = 0; q < 4; ++q) sb[(sub + 16 * q) * kLd + col] = rb[q];
            __syncthreads();
            if (kc + kDims < d) fetch(kc + kDims);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                // dimensions 8s + 4h .. 8s + 4h + 3: MFMA e multiplies 8s + e and 8s + 4 + e
                float4 va[2], vb[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    va[i] = *(const float4 *)&sa[(wv * 64 + i * 32 + li) * kLd + 8 * s + 4 * h];
                    vb[i] = *(const float4 *)&sb[(i * 32 + li) * kLd + 8 * s + 4 * h];
                }
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j) {
                            const float ae = e == 0 ? va[i].x : e == 1 ? va[i].y : e == 2 ? va[i].z : va[i].w;
                            const float be = e == 0 ? vb[j].x : e == 1 ? vb[j].y : e == 2 ? vb[j].z : vb[j].w;
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(ae, be, acc[i][j], 0, 0, 0);
                        }
            }
        }
        // element r of a product: centroid 8 (r / 4) + 4h + r % 4, row li
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const float4 cc = *(const float4 *)&sc[wv * 64 + i * 32 + 8 * g + 4 * h];
                const float cs[4] = {cc.x, cc.y, cc.z, cc.w};
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const float a = fmaf(-2.0f, acc[i][j][4 * g + e], cs[e]);
                        const bool lt = a < b[j].m1;
                        b[j].m2 = fminf(b[j].m2, fmaxf(b[j].m1, a));
                        b[j].i1 = lt ? c0 + wv * 64 + i * 32 + 8 * g + e : b[j].i1;
                        b[j].m1 = fminf(b[j].m1, a);
                    }
            }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        b[j].i1 += 4 * h;
        const Best o = Best{__shfl_xor(b[j].m1, 32), __shfl_xor(b[j].m2, 32), __shfl_xor(b[j].i1, 32)};
        if (h == 0) best[wv][j * 32 + li] = better(b[j], o);
    }
    __syncthreads();
    if (tid < kRows && row0 + tid < n) {
        const Best r = better(better(best[0][tid], best[1][tid]), better(best[2][tid], best[3][tid]));
        const int64_t at = (int64_t)blockIdx.y * n + row0 + tid;
        m1[at] = r.m1;
        m2[at] = r.m2;
        i1[at] = r.i1;
    }
}

__global__ __launch_bounds__(256) void cluster_decide_kernel(int32_t n, int32_t d, int32_t splits, const float *x2,
                                                             const uint32_t *c2max, const float *m1, const float *m2,
                                                             const int32_t *i1, int32_t *ids, int32_t *list,
                                                             int32_t *count) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    Best b = Best{m1[i], m2[i], i1[i]};
    for (int32_t s = 1; s < splits; ++s)
        b = better(b, Best{m1[(int64_t)s * n + i], m2[(int64_t)s * n + i], i1[(int64_t)s * n + i]});
    const float r = sqrtf(x2[i]) + sqrtf(__uint_as_float(*c2max));
    const float S = r * r;
    const bool sure = S >= 1e-28f && S <= 1e36f && b.m2 - b.m1 > 5.0f * (float)(d + 16) * 0x1p-24f * S;
    if (sure) {
        ids[i] = b.i1;
    } else {
        list[atomicAdd(count, 1)] = (int32_t)i;
    }
}

constexpr int32_t kNone = 0x7fffffff;

// The first of the least distances so far; kNone while none compared less
// than infinity.
struct Near {
    float v = __builtin_inff();
    int32_t j = kNone;
    __device__ __forceinline__ void next(float v2, int32_t j2) {  // j2 above all before
        j = v2 < v ? j2 : j;
        v = v2 < v ? v2 : v;
    }
    __device__ __forceinline__ void join(float v2, int32_t j2) {  // another's, over other centroids
        const bool t = v2 < v || (v2 == v && j2 < j);
        v = t ? v2 : v;
        j = t ? j2 : j;
    }
};

// Each listed row's (every row's where list is null) first nearest centroid in
// the reference's order, in one of two forms.  Few rows take a workgroup each,
// a thread per centroid: a row is short work then, and there are no others to
// share the centroids with.  Many are taken 64 to a workgroup, a row per lane,
// and its waves take four centroids at a time in turn: those are the same for
// all lanes, so they come through scalar loads, and a row's elements are read
// once for four of them.  The first form is bound by its lanes' reads of one
// centroid each (0.5 ps per dimension), the second by the chain of a wave's
// 16-dimension steps (1 us each) until the rows fill the device.  20,000 rows x
// 128 that the filter cannot decide, 1,024 centroids: 1,380 us by rows, 470 by
// tiles; 1,000 of them: 70 and 400.
__global__ __launch_bounds__(256) void cluster_exact_kernel(const float *x, int32_t n, int32_t d, const float *cent,
                                                            int32_t k, const int32_t *list, const int32_t *count,
                                                            int32_t *ids) {
    __shared__ float near_v[4][64];
    __shared__ int32_t near_j[4][64];
    const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
    const int32_t rows = list ? *count : n;
    if (exact_by_row_ps(rows, d, k) > exact_by_tile_ps(rows, d, k)) {
        typedef const __attribute__((address_space(4))) float *Scalar;
        const Scalar sc = (Scalar)cent;
        for (int32_t at = blockIdx.x * 64; at < rows; at += gridDim.x * 64) {
            const int32_t r = at + l < rows ? at + l : rows - 1;
            const int32_t row = list ? list[r] : r;
            const float *xi = x + (int64_t)row * d;
            Near b;
            for (int32_t j = 4 * wv; j < k; j += 16) {
                if (j + 4 <= k) {
                    float v[4];
                    l2_helpa<4>(xi, sc + (int64_t)j * d, d, v);
#pragma unroll
                    for (int c = 0; c < 4; ++c) b.next(v[c], j + c);
                } else {
                    for (int32_t c = j; c < k; ++c) {
                        float v[1];
                        l2_helpa<1>(xi, sc + (int64_t)c * d, d, v);
                        b.next(v[0], c);
                    }
                }
            }
            __syncthreads();
            near_v[wv][l] = b.v;
            near_j[wv][l] = b.j;
            __syncthreads();
            if (wv == 0 && at + l < rows) {
                for (int w = 1; w < 4; ++w) b.join(near_v[w][l], near_j[w][l]);
                ids[row] = b.j == kNone ? -1 : b.j;
            }
        }
        return;
    }
    for (int32_t i = blockIdx.x; i < rows; i += gridDim.x) {
        const int32_t row = list ? list[i] : i;
        const float *xi = x + (int64_t)row * d;
        Near b;
        for (int32_t j = tid; j < k; j += 256) {
            float v[1];
            l2_helpa<1>(xi, cent + (int64_t)j * d, d, v);
            b.next(v[0], j);
        }
        for (int o = 32; o > 0; o >>= 1) b.join(__shfl_xor(b.v, o), __shfl_xor(b.j, o));
        __syncthreads();
        if (l == 0) {
            near_v[wv][0] = b.v;
            near_j[wv][0] = b.j;
        }
        __syncthreads();
        if (tid == 0) {
            for (int w = 1; w < 4; ++w) b.join(near_v[w][0], near_j[w][0]);
            ids[row] = b.j == kNone ? -1 : b.j;
        }
    }
}

// k-means++ seeding (clustering.hpp:138-196): distance of every row to one
// picked row, as the symmetric computer evaluates it (picked row first).
__global__ void cluster_dist_kernel(const float *x, int32_t n, int32_t d, const float *pivot, float *out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float v[1];
    l2_helpa<1>(pivot, x + i * d, d, v);
    out[i] = v[0];
}

// update_mediods (clustering.hpp:234-256): a centroid is the float sum of its
// rows in row order, times 1.0f / count; one without rows is zero.  One
// workgroup per centroid lists its rows in order, 1,024 ids at a time, and
// every thread then adds one dimension of them: the order is serial by
// definition, so the parallelism is in centroids and dimensions, and the loads
// of 16 rows are in flight at once.  100k x 128, 1,024 centroids: 90 us, 4 ms on
// the host with the copies there and back.
__global__ __launch_bounds__(256) void cluster_update_kernel(const float *x, int32_t n, int32_t d, const int32_t *ids,
                                                             float *cent) {
    constexpr int kList = 2048;
    __shared__ int32_t list[kList];
    __shared__ int32_t found[4];
    const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63;
    const int32_t c = blockIdx.x;
    for (int32_t j0 = 0; j0 < d; j0 += 256) {
        const int32_t j = j0 + tid;
        float sum = 0.0f;
        int32_t total = 0;
        int len = 0;
        int32_t next[4];
        auto fetch = [&](int32_t base) __attribute__((always_inline)) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int32_t r = base + wv * 256 + q * 64 + l;
                next[q] = r < n ? ids[r] : -1;
            }
        };
        fetch(0);
        for (int32_t base = 0; base < n; base += 1024) {
            unsigned long long m[4];
            int mine = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                m[q] = __ballot(next[q] == c);
                mine += __popcll(m[q]);
            }
            if (base + 1024 < n) fetch(base + 1024);
            if (l == 0) found[wv] = mine;
            __syncthreads();
            int at = len;
            for (int w = 0; w < wv; ++w) at += found[w];
            len += found[0] + found[1] + found[2] + found[3];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if ((m[q] >> l) & 1ull)
                    list[at + __popcll(m[q] & ((1ull << l) - 1ull))] = base + wv * 256 + q * 64 + l;
                at += __popcll(m[q]);
            }
            __syncthreads();
            if (len > kList - 1024 || base + 1024 >= n) {
                if (j < d) {
                    int i = 0;
                    for (; i + 16 <= len; i += 16) {
                        float v[16];
#pragma unroll
                        for (int q = 0; q < 16; ++q) v[q] = x[(int64_t)list[i + q] * d + j];
#pragma unroll
                        for (int q = 0; q < 16; ++q) sum += v[q];
                    }
                    for (; i < len; ++i) sum += x[(int64_t)list[i] * d + j];
                }
                total += len;
                len = 0;
                __syncthreads();
            }
        }
        if (j < d) cent[(int64_t)c * d + j] = total ? sum * (1.0f / (float)total) : sum;
    }
}

__global__ void cluster_gather_kernel(const float *x, const int32_t *rows, int32_t m, int32_t d, float *out) {
    const int64_t total = (int64_t)m * d;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = i / d;
        out[i] = x[(int64_t)rows[r] * d + (i - r * d)];
    }
}

int32_t cent_tiles(int32_t k) { return (k + kCents - 1) / kCents; }

// Workgroups along the centroids: enough that four per CU are there when the
// rows alone do not give them.
int32_t filter_splits(int32_t n, int32_t k) {
    const int32_t blocks = (n + kRows - 1) / kRows;
    const int32_t want = (1024 + blocks - 1) / blocks;
    return want < cent_tiles(k) ? want : cent_tiles(k);
}

// The exact kernel's workgroups for up to n rows in either form.
int32_t exact_blocks(int32_t n) { return std::max(std::min(n, 1024), std::min((n + 63) / 64, 4096)); }

}  // namespace

// Fewer rows are split further, so the layout for fewer rows can be the larger
// one: with b = ceil(c / 64) workgroups, the splits times the rows c are at most
// (1023 + b) / b * 64 b, and at most cent_tiles times the rows.
size_t AssignScratch::bytes(int32_t n, int32_t k) {
    const size_t blocks = ((size_t)n + kRows - 1) / kRows;
    const size_t part = std::min((size_t)cent_tiles(k) * n, (1023 + blocks) * kRows);
    return 4 * (2 * (size_t)n + (size_t)k + 3 * part + 2);
}

void AssignScratch::place(void *p, int32_t n, int32_t k) {
    const size_t part = (size_t)filter_splits(n, k) * n;
    x2 = (float *)p;
    c2 = x2 + n;
    m1 = c2 + k;
    m2 = m1 + part;
    i1 = (int32_t *)(m2 + part);
    list = i1 + part;
    count = list + n;
    c2max = (uint32_t *)(count + 1);
}

hipError_t launch_fill_i32(int32_t *p, int64_t n, int32_t v, hipStream_t stream);

hipError_t launch_cluster_norms(const float *x, int32_t n, int32_t d, const AssignScratch &s, hipStream_t stream) {
    if (!filter_pays(n, d, (int32_t)(s.m1 - s.c2))) return hipSuccess;  // nothing reads them; c2 has k words
    hipLaunchKernelGGL(cluster_norms_kernel, dim3((n + 3) / 4 < 8192 ? (n + 3) / 4 : 8192), dim3(256), 0, stream, x, n,
                       d, s.x2, (uint32_t *)nullptr);
    return hipGetLastError();
}

hipError_t launch_cluster_assign(const float *x, int32_t n, int32_t d, const float *cent, int32_t k, int32_t *ids,
                                 const AssignScratch &s, hipStream_t stream) {
    if (!filter_pays(n, d, k)) {
        hipLaunchKernelGGL(cluster_exact_kernel, dim3(exact_blocks(n)), dim3(256), 0, stream, x, n, d, cent, k,
                           (const int32_t *)nullptr, (const int32_t *)nullptr, ids);
        return hipGetLastError();
    }
    const int32_t splits = filter_splits(n, k);
    const int32_t tiles = (cent_tiles(k) + splits - 1) / splits;
    // count and c2max are neighbours
    if (hipError_t e = launch_fill_i32(s.count, 2, 0, stream)) return e;
    hipLaunchKernelGGL(cluster_norms_kernel, dim3((k + 3) / 4 < 8192 ? (k + 3) / 4 : 8192), dim3(256), 0, stream, cent,
                       k, d, s.c2, s.c2max);
    hipLaunchKernelGGL(cluster_filter_kernel, dim3((n + kRows - 1) / kRows, splits), dim3(256), 0, stream, x, n, d,
                       cent, k, s.c2, tiles, s.m1, s.m2, s.i1);
    hipLaunchKernelGGL(cluster_decide_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, n, d, splits, s.x2, s.c2max,
                       s.m1, s.m2, s.i1, ids, s.list, s.count);
    hipLaunchKernelGGL(cluster_exact_kernel, dim3(exact_blocks(n)), dim3(256), 0, stream, x, n, d, cent, k, s.list,
                       s.count, ids);
    return hipGetLastError();
}

hipError_t launch_cluster_dist(const float *x, int32_t n, int32_t d, const float *pivot, float *out,
                               hipStream_t stream) {
    hipLaunchKernelGGL(cluster_dist_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, x, n, d, pivot, out);
    return hipGetLastError();
}

hipError_t launch_cluster_update(const float *x, int32_t n, int32_t d, const int32_t *ids, int32_t k, float *cent,
                                 hipStream_t stream) {
    hipLaunchKernelGGL(cluster_update_kernel, dim3(k), dim3(256), 0, stream, x, n, d, ids, cent);
    return hipGetLastError();
}

hipError_t launch_cluster_gather(const float *x, const int32_t *rows, int32_t m, int32_t d, float *out,
                                 hipStream_t stream) {
    const int64_t blocks = ((int64_t)m * d + 255) / 256;
    hipLaunchKernelGGL(cluster_gather_kernel, dim3((unsigned)(blocks < 16384 ? blocks : 16384)), dim3(256), 0, stream,
                       x, rows, m, d, out);
    return hipGetLastError();
}

}  // namespace glass_hip
