// Bilinear queries into the jagged per-Gaussian texel tensor and the adjoint
// w.r.t. the texels.  Forward semantics: texture_sample.cu:11-36 (no uv clamp,
// replicate padding on the integer coordinates).  Coordinates the reference
// would read out of bounds (h*u <= -1) are clamped to the first texel.
#include "gstex_common.hpp"
#include "gstex_kernels.hpp"

namespace gstex {

__device__ __forceinline__ void sample_taps(int h, int w, int start, float u, float v, int num_texels,
                                            float wt[4], int row[4]) {
    const float tu = (float)h * u, tv = (float)w * v;
    int iu = f2i_trunc(tu), iv = f2i_trunc(tv);
    const float fu = tu - (float)iu, fv = tv - (float)iv;
    const int ju = max(min(iu + 1, h - 1), 0), jv = max(min(iv + 1, w - 1), 0);
    iu = max(min(iu, h - 1), 0);
    iv = max(min(iv, w - 1), 0);
    wt[0] = (1.f - fu) * (1.f - fv);
    wt[1] = (1.f - fu) * fv;
    wt[2] = fu * (1.f - fv);
    wt[3] = fu * fv;
    const int lim = num_texels - 1;
    row[0] = min(max(start + iu * w + iv, 0), lim);
    row[1] = min(max(start + iu * w + jv, 0), lim);
    row[2] = min(max(start + ju * w + iv, 0), lim);
    row[3] = min(max(start + ju * w + jv, 0), lim);
}

// One thread per query.  CM is the channel count, or 0 for a runtime count: the
// exact counts read a tap as one wide load, so a query makes 4 gathers instead
// of 4 C (each gather instruction of a wave touches up to 64 cache lines, which
// is what bounds this kernel).  4M queries of 3 channels over 2M texels:
// 135 us with a gather per value, 93 with one per tap.
template <int CM>
__global__ __launch_bounds__(256) void k_sample_forward(int q, int channels, int num_texels,
                                                        const int* __restrict__ dims,
                                                        const float* __restrict__ uvs,
                                                        const float* __restrict__ texture,
                                                        float* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= q) return;
    const int C = CM ? CM : channels;
    float wt[4];
    int row[4];
    sample_taps(dims[3 * i], dims[3 * i + 1], dims[3 * i + 2], uvs[2 * i], uvs[2 * i + 1],
                num_texels, wt, row);
    if constexpr (CM != 0) {
        float t[4][CM];
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int c = 0; c < CM; ++c) t[k][c] = texture[(size_t)row[k] * CM + c];
#pragma unroll
        for (int c = 0; c < CM; ++c)
            out[(size_t)i * CM + c] =
                wt[0] * t[0][c] + wt[1] * t[1][c] + wt[2] * t[2][c] + wt[3] * t[3][c];
    } else {
        for (int c = 0; c < C; ++c)
            out[(size_t)i * C + c] = wt[0] * texture[(size_t)row[0] * C + c] +
                                     wt[1] * texture[(size_t)row[1] * C + c] +
                                     wt[2] * texture[(size_t)row[2] * C + c] +
                                     wt[3] * texture[(size_t)row[3] * C + c];
    }
}

// Taps that clamp onto one texel (every tap of a 1x1 chart, the far edge of
// larger ones) are added once with their summed weight; a zero weight marks
// a tap with nothing to add.
__device__ __forceinline__ void merge_taps(float wt[4], const int row[4]) {
#pragma unroll
    for (int k = 1; k < 4; ++k) {
#pragma unroll
        for (int j = 0; j < k; ++j) {
            if (wt[k] != 0.f && wt[j] != 0.f && row[k] == row[j]) {
                wt[j] += wt[k];
                wt[k] = 0.f;
            }
        }
    }
}

// Query keys for the adjoint: the bucket of 2^kSampleBucketShift texels that
// holds the query's chart start (clamped into the texture), and its index.
// With C <= 4 the query is also packed into one 32-byte record (u, v, start,
// h | w << 16, the C cotangents), read in query order here so that the
// sorted pass gathers one record per query instead of three arrays.  A chart
// side of 2^16 or more does not fit the packing; such a record is marked
// (h | w << 16 = 0xffffffff) and that query reads the original arrays.
constexpr int kSampleBucketShift = 8;
constexpr uint32_t kSampleUnpacked = 0xffffffffu;

__global__ __launch_bounds__(256) void k_sample_keys(int q, int C, int num_texels,
                                                     const int* __restrict__ dims,
                                                     const float* __restrict__ uvs,
                                                     const float* __restrict__ v_out,
                                                     uint32_t* __restrict__ keys,
                                                     uint32_t* __restrict__ idx,
                                                     float4* __restrict__ rec) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= q) return;
    const int h = dims[3 * i], w = dims[3 * i + 1], start = dims[3 * i + 2];
    keys[i] = (uint32_t)min(max(start, 0), num_texels) >> kSampleBucketShift;
    idx[i] = (uint32_t)i;
    if (rec != nullptr) {
        const bool fits = h >= 0 && w >= 0 && h < 65536 && w < 65536;
        const uint32_t hw = fits ? ((uint32_t)h | ((uint32_t)w << 16)) : kSampleUnpacked;
        float g[4] = {0.f, 0.f, 0.f, 0.f};
        for (int c = 0; c < C; ++c) g[c] = v_out[(size_t)i * C + c];
        rec[2 * (size_t)i] = make_float4(uvs[2 * i], uvs[2 * i + 1], __int_as_float(start),
                                         __uint_as_float(hw));
        rec[2 * (size_t)i + 1] = make_float4(g[0], g[1], g[2], g[3]);
    }
}

// v_texture += sum over queries of weight * v_output, over the queries sorted
// by chart-start bucket: a workgroup takes kSampleRange consecutive sorted
// queries, whose charts lie in one contiguous run of texels starting at the
// first query's bucket.  Their taps are added into an LDS window over that run
// (taps past the window go straight to HBM), and the window is flushed with
// one atomic per value it received.  Each thread takes kSamplePer
// consecutive queries, so the lanes of a wave fall on different charts.
constexpr int kSamplePer = 16;
constexpr int kSampleRange = 256 * kSamplePer;
constexpr int kSampleWindow = 8192;  // floats (32 KiB)

// One query's adds: the taps of channel value g(c) into the window or HBM.
template <int CM, typename G>
__device__ __forceinline__ void sample_scatter(int C, int num_texels, int h, int w, int start,
                                               float u, float v, const G& g, long long base,
                                               float* win, float* v_texture, int& hi) {
    float wt[4];
    int row[4];
    sample_taps(h, w, start, u, v, num_texels, wt, row);
    merge_taps(wt, row);
#pragma unroll
    for (int c = 0; c < (CM ? CM : C); ++c) {
        const float gc = g(c);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const float add = wt[t] * gc;
            if (add == 0.f) continue;
            const long long at = (long long)row[t] * C + c;
            const long long off = at - base;
            if (off >= 0 && off < kSampleWindow) {
                atomicAdd(win + off, add);
                hi = max(hi, (int)off + 1);
            } else {
                unsafeAtomicAdd(v_texture + at, add);
            }
        }
    }
}

// CM 1..4: that many channels, through the packed records; 0: a runtime count,
// from the original arrays.  With records a thread takes its queries four at a
// time, the four gathers in flight together, and the exact count keeps the
// cotangents in registers (an index at run time put them in scratch memory):
// 4M queries of 3 channels, 141 -> 117 us.
template <int CM>
__global__ __launch_bounds__(256) void k_sample_backward_sorted(
    int q, int channels, int num_texels, const uint32_t* __restrict__ keys_sorted,
    const uint32_t* __restrict__ idx_sorted, const float4* __restrict__ rec,
    const int* __restrict__ dims, const float* __restrict__ uvs, const float* __restrict__ v_out,
    float* __restrict__ v_texture) {
    __shared__ float win[kSampleWindow];
    __shared__ int used;
    const int C = CM ? CM : channels;
    const int first = blockIdx.x * kSampleRange;
    const int last = min(first + kSampleRange, q);
    for (int k = threadIdx.x; k < kSampleWindow; k += blockDim.x) win[k] = 0.f;
    if (threadIdx.x == 0) used = 0;
    __syncthreads();
    const long long base = ((long long)keys_sorted[first] << kSampleBucketShift) * C;
    int hi = 0;  // past the last window value this thread touched
    const int k0 = first + threadIdx.x * kSamplePer, k1 = min(k0 + kSamplePer, last);
    auto from_arrays = [&](int i) {
        const float* g = v_out + (size_t)i * C;
        sample_scatter<CM>(
            C, num_texels, dims[3 * i], dims[3 * i + 1], dims[3 * i + 2], uvs[2 * i],
            uvs[2 * i + 1], [&](int c) { return g[c]; }, base, win, v_texture, hi);
    };
    if constexpr (CM == 0) {
        for (int k = k0; k < k1; ++k) from_arrays((int)idx_sorted[k]);
    } else {
        constexpr int kTake = 4;
        for (int k = k0; k < k1; k += kTake) {
            int id[kTake];
            float4 a[kTake], b[kTake];
#pragma unroll
            for (int j = 0; j < kTake; ++j) id[j] = (int)idx_sorted[min(k + j, k1 - 1)];
#pragma unroll
            for (int j = 0; j < kTake; ++j) {
                a[j] = rec[2 * (size_t)id[j]];
                b[j] = rec[2 * (size_t)id[j] + 1];
            }
#pragma unroll
            for (int j = 0; j < kTake; ++j) {
                if (k + j >= k1) break;
                const uint32_t hw = __float_as_uint(a[j].w);
                if (hw == kSampleUnpacked) {
                    from_arrays(id[j]);
                    continue;
                }
                const float g4[4] = {b[j].x, b[j].y, b[j].z, b[j].w};
                sample_scatter<CM>(
                    C, num_texels, (int)(hw & 0xffffu), (int)(hw >> 16), __float_as_int(a[j].z),
                    a[j].x, a[j].y, [&](int c) { return g4[c]; }, base, win, v_texture, hi);
            }
        }
    }
    atomicMax(&used, hi);
    __syncthreads();
    const int n = used;
    for (int k = threadIdx.x; k < n; k += blockDim.x) {
        const float val = win[k];
        if (val != 0.f) unsafeAtomicAdd(v_texture + base + k, val);
    }
}

hipError_t sample_forward(int q, int C, int num_texels, const int* dims, const float* uvs,
                          const float* texture, float* out, hipStream_t s) {
    if (q <= 0 || C <= 0) return hipSuccess;
    const int g = (q + 255) / 256;
    switch (C) {
        case 1: k_sample_forward<1><<<g, 256, 0, s>>>(q, C, num_texels, dims, uvs, texture, out); break;
        case 2: k_sample_forward<2><<<g, 256, 0, s>>>(q, C, num_texels, dims, uvs, texture, out); break;
        case 3: k_sample_forward<3><<<g, 256, 0, s>>>(q, C, num_texels, dims, uvs, texture, out); break;
        case 4: k_sample_forward<4><<<g, 256, 0, s>>>(q, C, num_texels, dims, uvs, texture, out); break;
        default: k_sample_forward<0><<<g, 256, 0, s>>>(q, C, num_texels, dims, uvs, texture, out);
    }
    return hipGetLastError();
}

static size_t up256(size_t b) { return (b + 255) & ~(size_t)255; }

size_t sample_backward_workspace_bytes(int q) {
    if (q <= 0) return 256;
    return 4 * up256(sizeof(uint32_t) * (size_t)q) + up256(32 * (size_t)q) +
           sort_u32_pairs_workspace_bytes(q) + 256;
}

hipError_t sample_backward(int q, int C, int num_texels, const int* dims, const float* uvs,
                           const float* v_out, float* v_texture, void* ws, size_t ws_bytes,
                           hipStream_t s) {
    hipError_t e = fill_f32(v_texture, (size_t)num_texels * (size_t)C, 0.f, s);
    if (e != hipSuccess || q <= 0 || C <= 0) return e;
    if (ws_bytes < sample_backward_workspace_bytes(q)) return hipErrorInvalidValue;
    char* p = static_cast<char*>(ws);
    const size_t a = up256(sizeof(uint32_t) * (size_t)q);
    uint32_t* keys = (uint32_t*)p;
    uint32_t* idx = (uint32_t*)(p + a);
    uint32_t* keys_s = (uint32_t*)(p + 2 * a);
    uint32_t* idx_s = (uint32_t*)(p + 3 * a);
    float4* rec = (float4*)(p + 4 * a);
    void* rws = p + 4 * a + up256(32 * (size_t)q);
    const size_t rws_bytes = ws_bytes - 4 * a - up256(32 * (size_t)q);
    // records only when the cotangents fit them
    if (C > 4) rec = nullptr;
    k_sample_keys<<<(q + 255) / 256, 256, 0, s>>>(q, C, num_texels, dims, uvs, v_out, keys, idx,
                                                  rec);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int end_bit = 32 - __builtin_clz(((unsigned)num_texels >> kSampleBucketShift) | 1u);
    e = sort_u32_pairs(q, keys, idx, keys_s, idx_s, end_bit, rws, rws_bytes, s);
    if (e != hipSuccess) return e;
    const int g = (q + kSampleRange - 1) / kSampleRange;
#define GSTEX_SAMPLE_BWD(CM)                                                                  \
    k_sample_backward_sorted<CM><<<g, 256, 0, s>>>(q, C, num_texels, keys_s, idx_s, rec, dims, \
                                                   uvs, v_out, v_texture)
    switch (C) {
        case 1: GSTEX_SAMPLE_BWD(1); break;
        case 2: GSTEX_SAMPLE_BWD(2); break;
        case 3: GSTEX_SAMPLE_BWD(3); break;
        case 4: GSTEX_SAMPLE_BWD(4); break;
        default: GSTEX_SAMPLE_BWD(0);
    }
#undef GSTEX_SAMPLE_BWD
    return hipGetLastError();
}

}  // namespace gstex
