// Row moves of the cache's tiers: join, keep, gather, append and scatter of token rows.
//
// A cache update moves rows of many small tensors (keys, values, codes, meta, positions,
// importance) the same way; as one library launch per tensor and step it is bound by the
// launches and their host work, ~100 a generated token.  Here one launch takes up to
// kRowsMaxJobs tensors.  A workgroup owns a run of token rows of one job and one (batch, head)
// -- about kRowsUnits units of up to 16 bytes, four a thread -- and resolves the source or
// destination rows of a list once before its threads move them: for KEEP a search of the
// ascending list, first among 1024 samples of it in LDS, so that a list of that size costs one
// trip to memory and a prompt's 16 thousand five instead of fourteen.  Rows that follow each
// other on both sides (codes and meta appended to a tier) are one range, cut into units
// whatever the row's length: 2-byte scale rows would otherwise go 2 bytes a thread.
// Cache updates, one tensor at a time -> this: a 16k prompt of 8 heads 517 -> 119 us (its
// launches here 33 us before tiles by units and the sampled search, 26 after); a 2 x 2-head
// bfloat16 layer's prompt and 12 tokens with promotions 13.3 -> 4.4 ms.
#include "rows.h"

#include <algorithm>

#include "akv_common.h"

namespace akv {
namespace {
constexpr int kRowsUnits = 1024;  // units of a workgroup: four a thread
constexpr int kRowsList = 256;    // most rows of a workgroup that a list places
constexpr int kRowsSamples = 1024;

template <typename T>
__device__ __forceinline__ void copy_unit(const char *s, char *d) {
    *(T *)d = *(const T *)s;
}
__device__ __forceinline__ float widen1(const char *s, int dt, int i) { return load_as_f32(s, i, dt); }
}  // namespace

__global__ __launch_bounds__(256) void rows_move_kernel(const RowsParams p) {
    __shared__ int64_t rows[kRowsList];
    __shared__ int sample[kRowsSamples];
    const akv_rows_job &j = p.job[blockIdx.y];
    const int tile = p.tile[blockIdx.y];
    const int64_t t0 = (int64_t)blockIdx.x * tile;
    if (t0 >= j.n) return;
    const int nt = (int)min((int64_t)tile, j.n - t0);
    const bool same = j.map == AKV_ROWS_SAME;
    if (!same) {
        const bool keep = j.map == AKV_ROWS_KEEP;
        const int64_t step = (p.n_idx + kRowsSamples - 1) / kRowsSamples;
        const int ns = keep && p.n_idx > 0 ? (int)((p.n_idx + step - 1) / step) : 0;
        for (int k = threadIdx.x; k < ns; k += 256) sample[k] = (int)(p.idx[k * step] - k * step);
        __syncthreads();
        if (threadIdx.x < (unsigned)nt) {
            const int64_t t = t0 + threadIdx.x;
            int64_t r;
            if (keep) {  // the t-th row that is not in the ascending list
                int a = 0, b = ns;  // samples at or below t
                while (a < b) {
                    const int mid = (a + b) / 2;
                    if (sample[mid] <= t) a = mid + 1;
                    else b = mid;
                }
                // entries idx[i] with idx[i] - i <= t lie before it
                int64_t lo = a > 0 ? (a - 1) * step + 1 : 0, hi = a > 0 ? min(p.n_idx, a * step) : 0;
                while (lo < hi) {
                    const int64_t mid = (lo + hi) / 2;
                    if (p.idx[mid] - mid <= t) lo = mid + 1;
                    else hi = mid;
                }
                r = t + lo;
            } else {
                r = p.idx[t];
            }
            rows[threadIdx.x] = (r >= 0 && r < j.limit) ? r : -1;
        }
        __syncthreads();
    }
    const int unit = p.unit[blockIdx.y], per = (j.kind == AKV_ROWS_COPY ? j.row * j.elem : j.row) / unit;
    const int64_t nbh = (int64_t)j.B * j.H;
    for (int64_t bh = blockIdx.z; bh < nbh; bh += gridDim.z) {
        const int64_t b = bh / j.H, h = bh - b * j.H;
        const char *src = (const char *)j.src + b * j.src_b + h * j.src_h;
        char *dst = (char *)j.dst + b * j.dst_b + h * j.dst_h;
        for (int u = threadIdx.x; u < nt * per; u += 256) {
            const int t = u / per, c = u - t * per;
            const int64_t r = same ? t0 + t : rows[t];
            if (r < 0) continue;
            const int64_t st = j.map == AKV_ROWS_SCATTER ? t0 + t : r, dt = j.map == AKV_ROWS_SCATTER ? r : t0 + t;
            const char *s = src + st * j.src_t;
            char *d = dst + dt * j.dst_t;
            if (j.kind == AKV_ROWS_COPY) {
                const int o = c * unit;
                if (unit == 16) copy_unit<u4>(s + o, d + o);
                else if (unit == 4) copy_unit<uint32_t>(s + o, d + o);
                else if (unit == 2) copy_unit<uint16_t>(s + o, d + o);
                else copy_unit<unsigned char>(s + o, d + o);
            } else if (j.kind == AKV_ROWS_WIDEN) {
                float *o = (float *)d + c * unit;
                if (unit == 8) {
                    const u4 x = *(const u4 *)(s + 16 * c);
                    float v[8];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const uint32_t w = x[i];
                        v[2 * i] = j.src_dt == AKV_DT_F16 ? (float)as_h2(w)[0] : __builtin_bit_cast(float, w << 16);
                        v[2 * i + 1] = j.src_dt == AKV_DT_F16 ? (float)as_h2(w)[1] : __builtin_bit_cast(float, w & 0xFFFF0000u);
                    }
                    *(f4 *)o = (f4){v[0], v[1], v[2], v[3]};
                    *(f4 *)(o + 4) = (f4){v[4], v[5], v[6], v[7]};
                } else {
                    o[0] = widen1(s, j.src_dt, c) * j.value;
                }
            } else if (j.kind == AKV_ROWS_FILL) {
                ((float *)d)[c] = j.value;
            } else {  // AKV_ROWS_COUNT: consecutive integers
                const int64_t v = j.start + j.step * dt;
                if (j.elem == 8) ((int64_t *)d)[c] = v;
                else ((int32_t *)d)[c] = (int32_t)v;
            }
        }
    }
}

// The widest unit that rows, strides and pointers of a job allow.
static int rows_unit(const akv_rows_job &j) {
    const uint64_t al = (uint64_t)(uintptr_t)j.src | (uint64_t)j.src_b | (uint64_t)j.src_h | (uint64_t)j.src_t |
                        (uint64_t)(uintptr_t)j.dst | (uint64_t)j.dst_b | (uint64_t)j.dst_h | (uint64_t)j.dst_t;
    if (j.kind == AKV_ROWS_COPY) {
        const uint64_t a = al | (uint64_t)j.row * (uint64_t)j.elem;
        return (a & 15) == 0 ? 16 : (a & 3) == 0 ? 4 : (a & 1) == 0 ? 2 : 1;
    }
    if (j.kind == AKV_ROWS_WIDEN && j.src_dt != AKV_DT_F32 && j.value == 1.0f && j.row % 8 == 0 && (al & 15) == 0) return 8;
    return 1;
}

hipError_t rows_move_launch(const akv_rows_job *jobs, int n_jobs, const int64_t *idx, int64_t n_idx, hipStream_t s) {
    RowsParams p;
    p.idx = idx;
    p.n_idx = n_idx;
    int n = 0;
    int64_t tiles = 0, nbh = 0;
    for (int i = 0; i < n_jobs; ++i) {
        akv_rows_job j = jobs[i];
        if (j.n == 0 || j.B == 0 || j.H == 0) continue;
        if (j.map == AKV_ROWS_SAME) j.n = j.kind == AKV_ROWS_COPY || j.kind == AKV_ROWS_WIDEN ? std::min(j.n, j.limit) : j.n;
        int unit = rows_unit(j);
        const int64_t bytes = (int64_t)j.row * j.elem;
        if (j.kind == AKV_ROWS_COPY && j.map == AKV_ROWS_SAME && j.src_t == bytes && j.dst_t == bytes) {
            // one range of n * bytes, as rows of one unit (the row stride need not be aligned)
            const uint64_t al = (uint64_t)(uintptr_t)j.src | (uint64_t)j.src_b | (uint64_t)j.src_h |
                                (uint64_t)(uintptr_t)j.dst | (uint64_t)j.dst_b | (uint64_t)j.dst_h | (uint64_t)(j.n * bytes);
            unit = (al & 15) == 0 ? 16 : (al & 3) == 0 ? 4 : (al & 1) == 0 ? 2 : 1;
            j.n = j.n * bytes / unit;
            j.row = unit;
            j.elem = 1;
            j.src_t = j.dst_t = unit;
        }
        const int per = (j.kind == AKV_ROWS_COPY ? j.row * j.elem : j.row) / unit;
        const int tile = std::max(1, std::min(kRowsUnits / per, j.map == AKV_ROWS_SAME ? kRowsUnits : kRowsList));
        p.job[n] = j;
        p.unit[n] = unit;
        p.tile[n++] = tile;
        tiles = std::max(tiles, (j.n + tile - 1) / tile);
        nbh = std::max(nbh, (int64_t)j.B * j.H);
    }
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(rows_move_kernel, dim3((unsigned)tiles, (unsigned)n, (unsigned)std::min(nbh, (int64_t)65535)),
                       dim3(256), 0, s, p);
    return hipGetLastError();
}

}  // namespace akv
