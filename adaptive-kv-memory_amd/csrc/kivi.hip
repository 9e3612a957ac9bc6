// KIVI overflow rows: quantize, pack, append and dequantize in one pass over the tokens.
//
// HBM-bound.  The tokens that leave the residual window are read once; their codes, float32
// (and float16) scales and zeros go straight into the tier's rows, and their dequantized
// float16 values into the view the update returns (no working copy: a later view dequantizes
// the packed rows again, which reads an eighth of it at 2 bits).  A thread owns 8
// channels of kTok tokens (16-byte loads, all in flight), the lanes of a group reduce min /
// max by shuffles, and every thread dequantizes the codes it has just made from registers.
// Before, each tensor went through a float32 copy, a quantize, five slice copies into the
// zero-filled tier, a dequantize and a concatenation: 4,097 tokens x 32 heads of 128, K and V
// at 2 bits, 226 -> 61-67 us an update (this launch 43-46 us, 3.3 TB/s; the divisions, one an
// element in the reference's arithmetic, cost about as much as the stores).
#include "kivi.h"

#include <algorithm>

#include "akv_common.h"

namespace akv {
namespace {
constexpr int kTok = 4, kThreads = 256;

// The arithmetic of the group layouts on float32 input: scale = max((max - min) / maxv, 1e-10),
// codes = clamp(rint((x - min) / scale)), NaN codes 0.
__device__ __forceinline__ float group_scale(float mn, float mx, float maxv) {
    const float s = (mx - mn) / maxv;
    return s != s ? s : fmaxf(s, 1e-10f);
}
__device__ __forceinline__ uint32_t group_code(float x, float zero, float scale, float maxv) {
    const float q = rintf((x - zero) / scale);
    return q != q ? 0u : (uint32_t)fminf(fmaxf(q, 0.f), maxv);
}
__device__ __forceinline__ void put_codes(const uint32_t (&c)[8], int bits, unsigned char *d) {
    if (bits == 8) {
        u2 w = {0u, 0u};
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i / 4] |= c[i] << (8 * (i & 3));
        *(u2 *)d = w;
    } else if (bits == 4) {
        uint32_t w = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) w |= ((c[2 * i] << 4) | c[2 * i + 1]) << (8 * i);
        *(uint32_t *)d = w;
    } else {
        uint32_t w = 0;
#pragma unroll
        for (int i = 0; i < 2; ++i) w |= ((c[4 * i] << 6) | (c[4 * i + 1] << 4) | (c[4 * i + 2] << 2) | c[4 * i + 3]) << (8 * i);
        *(uint16_t *)d = (uint16_t)w;
    }
}
}  // namespace

template <int IN, int D>
__global__ __launch_bounds__(kThreads) void kivi_append_kernel(const KiviParams p) {
    constexpr int CG = D / 8, PER = kThreads / CG;  // lanes of a token, tokens of one pass
    const akv_kivi_side &s = p.side[blockIdx.z];
    const int cg = threadIdx.x % CG, tr = threadIdx.x / CG;
    const int64_t bh = blockIdx.y, b = bh / p.H, h = bh - b * p.H;
    const int64_t t0 = (int64_t)blockIdx.x * PER * kTok + tr;
    const int G = p.group_size, ng = (D + G - 1) / G, row = ng * G * s.bits / 8;
    const bool pad = G > D;
    const int LG = pad ? CG : G / 8;
    const float maxv = (float)((1 << s.bits) - 1);
    const char *src = (const char *)s.src + b * s.src_b + h * s.src_h;
    u4 x[kTok][IN == AKV_DT_F32 ? 2 : 1];
#pragma unroll
    for (int i = 0; i < kTok; ++i) {
        const u4 *q = (const u4 *)(src + min(t0 + (int64_t)i * PER, p.n - 1) * s.src_t) + cg * (IN == AKV_DT_F32 ? 2 : 1);
        x[i][0] = q[0];
        if constexpr (IN == AKV_DT_F32) x[i][1] = q[1];
    }
#pragma unroll
    for (int i = 0; i < kTok; ++i) {
        const int64_t t = t0 + (int64_t)i * PER;
        float v[8], mn = INFINITY, mx = -INFINITY;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if constexpr (IN == AKV_DT_F32) {
                const uint32_t w = x[i][e / 4][e & 3];
                v[e] = __builtin_bit_cast(float, w);
            } else {
                const uint32_t w = x[i][0][e / 2];
                if constexpr (IN == AKV_DT_F16) v[e] = (float)as_h2(w)[e & 1];
                else v[e] = __builtin_bit_cast(float, (e & 1) ? w & 0xFFFF0000u : w << 16);
            }
            mn = fminf(mn, v[e]);
            mx = fmaxf(mx, v[e]);
        }
        for (int o = 1; o < LG; o <<= 1) {
            mn = fminf(mn, __shfl_xor(mn, o));
            mx = fmaxf(mx, __shfl_xor(mx, o));
        }
        if (pad) {  // the group's channels past D are zeros
            mn = fminf(mn, 0.f);
            mx = fmaxf(mx, 0.f);
        }
        if (t >= p.n) continue;  // after the shuffles
        const float sc = group_scale(mn, mx, maxv);
        const int64_t at = bh * s.cap + s.row0 + t;
        uint32_t c[8];
        h8 y;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            c[e] = group_code(v[e], mn, sc, maxv);
            const float m = (float)c[e] * sc;
            v[e] = m + mn;
            y[e] = (_Float16)v[e];
        }
        unsigned char *cr = (unsigned char *)s.codes + at * row;
        put_codes(c, s.bits, cr + cg * s.bits);
        if (pad) {
            const uint32_t z = group_code(0.f, mn, sc, maxv);
            const uint32_t zs[8] = {z, z, z, z, z, z, z, z};
            put_codes(zs, s.bits, cr + (CG + cg) * s.bits);
        }
        if (cg % LG == 0) {
            const int64_t m = at * ng + cg / LG;
            ((float *)s.scale)[m] = sc;
            ((float *)s.zero)[m] = mn;
            if (s.scale16) {
                ((_Float16 *)s.scale16)[m] = (_Float16)sc;
                ((_Float16 *)s.zero16)[m] = (_Float16)mn;
            }
        }
        if (s.view) {
            const int64_t o = (bh * s.view_rows + s.row0 + t) * D + 8 * cg;
            if (p.view_dt == AKV_DT_F16) *(h8 *)((_Float16 *)s.view + o) = y;
            else {
                float *f = (float *)s.view + o;
                *(f4 *)f = (f4){(float)y[0], (float)y[1], (float)y[2], (float)y[3]};
                *(f4 *)(f + 4) = (f4){(float)y[4], (float)y[5], (float)y[6], (float)y[7]};
            }
        }
    }
    // rows [row0 + n, zero_to) of a new tier read as zeros
    for (int64_t r = s.row0 + p.n + (int64_t)blockIdx.x * kThreads + threadIdx.x; r < s.zero_to;
         r += (int64_t)gridDim.x * kThreads) {
        const int64_t at = bh * s.cap + r;
        for (int i = 0; i < row / 8; ++i) ((u2 *)((unsigned char *)s.codes + at * row))[i] = (u2){0u, 0u};
        for (int g = 0; g < ng; ++g) {
            ((float *)s.scale)[at * ng + g] = ((float *)s.zero)[at * ng + g] = 0.f;
            if (s.scale16) ((_Float16 *)s.scale16)[at * ng + g] = ((_Float16 *)s.zero16)[at * ng + g] = (_Float16)0.f;
        }
    }
}

hipError_t kivi_append_launch(const KiviParams &p, int n_sides, hipStream_t s) {
    if (p.n == 0 || p.B == 0 || p.H == 0) return hipSuccess;
    const int per = kThreads / (p.D / 8) * kTok;
    const dim3 grid((unsigned)((p.n + per - 1) / per), (unsigned)((int64_t)p.B * p.H), (unsigned)n_sides);
#define AKV_KIVI(in)                                                                                  \
    if (p.D == 64) hipLaunchKernelGGL((kivi_append_kernel<in, 64>), grid, dim3(kThreads), 0, s, p);   \
    else hipLaunchKernelGGL((kivi_append_kernel<in, 128>), grid, dim3(kThreads), 0, s, p)
    if (p.in_dt == AKV_DT_F32) { AKV_KIVI(AKV_DT_F32); }
    else if (p.in_dt == AKV_DT_F16) { AKV_KIVI(AKV_DT_F16); }
    else { AKV_KIVI(AKV_DT_BF16); }
#undef AKV_KIVI
    return hipGetLastError();
}

}  // namespace akv
