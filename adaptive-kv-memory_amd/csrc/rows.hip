// Row moves of the cache's tiers: join, keep, gather, append and scatter of token rows.
//
// A cache update moves rows of many small tensors (keys, values, codes, meta, positions,
// importance) the same way; as one library launch per tensor and step it is bound by the
// launches and their host work, ~100 a generated token.  Here one launch takes up to
// kRowsMaxJobs tensors.  A workgroup owns 64 token rows of one job and one (batch, head):
// its first wave resolves the 64 source or destination rows once (a binary search of the
// sorted list for KEEP), then 256 threads move the rows in units of up to 16 bytes.
// Cache updates, one tensor at a time -> this: a 16k prompt of 8 heads 517 -> 164 us; a 2 x
// 2-head bfloat16 layer's prompt and 12 tokens with promotions 13.3 -> 5.4 ms.
#include "rows.h"

#include <algorithm>

#include "akv_common.h"

namespace akv {
namespace {
constexpr int kRowsTile = 64;

template <typename T>
__device__ __forceinline__ void copy_unit(const char *s, char *d) {
    *(T *)d = *(const T *)s;
}
__device__ __forceinline__ float widen1(const char *s, int dt, int i) { return load_as_f32(s, i, dt); }
}  // namespace

__global__ __launch_bounds__(256) void rows_move_kernel(const RowsParams p) {
    __shared__ int64_t rows[kRowsTile];
    const akv_rows_job &j = p.job[blockIdx.y];
    const int64_t t0 = (int64_t)blockIdx.x * kRowsTile;
    if (t0 >= j.n) return;
    const int nt = (int)min((int64_t)kRowsTile, j.n - t0);
    if (threadIdx.x < (unsigned)nt) {
        const int64_t t = t0 + threadIdx.x;
        int64_t r = t;
        if (j.map == AKV_ROWS_KEEP) {  // the t-th row that is not in the ascending list
            int64_t lo = 0, hi = p.n_idx;  // entries idx[i] with idx[i] - i <= t lie before it
            while (lo < hi) {
                const int64_t mid = (lo + hi) / 2;
                if (p.idx[mid] - mid <= t) lo = mid + 1;
                else hi = mid;
            }
            r = t + lo;
        } else if (j.map != AKV_ROWS_SAME) {
            r = p.idx[t];
        }
        rows[threadIdx.x] = (r >= 0 && r < j.limit) ? r : -1;
    }
    __syncthreads();
    const int unit = p.unit[blockIdx.y], per = (j.kind == AKV_ROWS_COPY ? j.row * j.elem : j.row) / unit;
    const int64_t nbh = (int64_t)j.B * j.H;
    for (int64_t bh = blockIdx.z; bh < nbh; bh += gridDim.z) {
        const int64_t b = bh / j.H, h = bh - b * j.H;
        const char *src = (const char *)j.src + b * j.src_b + h * j.src_h;
        char *dst = (char *)j.dst + b * j.dst_b + h * j.dst_h;
        for (int u = threadIdx.x; u < nt * per; u += 256) {
            const int t = u / per, c = u - t * per;
            const int64_t r = rows[t];
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
        const akv_rows_job &j = jobs[i];
        if (j.n == 0 || j.B == 0 || j.H == 0) continue;
        p.job[n] = j;
        p.unit[n++] = rows_unit(j);
        tiles = std::max(tiles, (j.n + kRowsTile - 1) / kRowsTile);
        nbh = std::max(nbh, (int64_t)j.B * j.H);
    }
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(rows_move_kernel, dim3((unsigned)tiles, (unsigned)n, (unsigned)std::min(nbh, (int64_t)65535)),
                       dim3(256), 0, s, p);
    return hipGetLastError();
}

}  // namespace akv
