// Quantize + pack for every form that quant_fast_kernel (quant.hip) does not take:
// float16 / bfloat16 / float32 input, K blocks of any length, outlier channels, and the
// per-token-group layouts.  Same per-op rounding as quant_kernel (quant.hip), which
// remains for inputs off a 16-byte boundary and for KVQuantizer's layout.
//
// One wave holds a 32-token tile of one tensor in registers, one 16-byte load per token
// and 8 channels (two at float32).  A lane is (channel group of 8, token group); K
// statistics go over a lane's tokens and then across the token groups, V statistics
// over a lane's channels and then across the group's lanes; the packed rows leave
// through LDS as contiguous stores.  What bounds the kernels at sizes that fill the GPU is
// memory.  Measured against quant_kernel, which loads single elements and gives a block one
// wave: one block of 16,255 float16 tokens x 8 heads 42.1 ms -> 10 us of statistics (3.3
// TB/s) + 29 us of encoding; 3,969 float32 tokens x 32 heads in groups of 128 143 -> 26 us
// (2.7 TB/s); 32-token float16 blocks with one outlier channel, 15,872 tokens x 128 heads
// 2.43 -> 0.35 ms, and their channel choice (outlier_select_kernel) 1.18 -> 0.21 ms.
//
// K statistics of a block, by its length T:
//   T <= 32           in the wave (block = tile);
//   longer            a workgroup of 4 waves walks the block (the tile stays in registers
//                     when T <= 128, else the second walk reads it again from L2);
//   T > 512 with fewer than 512 such blocks and a workspace: that would leave most CUs
//                     idle, so kstat_kernel writes min / max partials of chunks of the
//                     block, and workgroups of 8 tiles reduce them (in LDS) before they
//                     encode.
#include <atomic>

#include "akv_common.h"
#include "quant.h"

namespace akv {

namespace {

template <int IN> constexpr int kInWords = IN == AKV_DT_F32 ? 8 : 4;  // dwords of 8 elements
constexpr int kTileWaves = 4;
constexpr int kEncTiles = 8;        // tiles per workgroup when a long block's statistics are precomputed
constexpr int kLongT = 512;         // blocks longer than this may use the workspace
constexpr int kStatTokens = 512;    // tokens per statistics chunk (at least)
constexpr int kStatWaves = 16;      // a wave a tile of a chunk: every load of the chunk in flight at once
constexpr int kMaxChunks = 64;

// K statistics sources of qtile_kernel
constexpr int kKNone = 0, kKTile = 1, kKBlock = 2, kKPartials = 3, kKGroups = 4;

template <int DT>
__device__ __forceinline__ float rnd(float x) {
    if (DT == AKV_DT_F16) return (float)(_Float16)x;
    if (DT == AKV_DT_BF16) return bf16_to_f32(f32_to_bf16_rne(x));
    return x;
}
// scale of a (min, max) pair with the arithmetic dtype's roundings; NaN stays
template <int DT>
__device__ __forceinline__ float scale_of(float mn, float mx, float maxv, float lo) {
    const float s = rnd<DT>(rnd<DT>(mx - mn) / maxv);
    return s != s ? s : fmaxf(s, lo);
}
template <int DT>
__device__ __forceinline__ uint32_t code_of(float x, float zero, float scale, float maxv) {
    float q = rnd<DT>(x - zero);
    q = rnd<DT>(q / scale);
    q = rintf(q);
    if (q != q) return 0u;  // NaN -> 0
    return (uint32_t)fminf(fmaxf(q, 0.0f), maxv);
}

template <int IN>
__device__ __forceinline__ float elem(const uint32_t *w, int i) {
    if (IN == AKV_DT_F16) return (float)as_h2(w[i / 2])[i & 1];
    if (IN == AKV_DT_BF16) return __builtin_bit_cast(float, (i & 1) ? w[i / 2] & 0xFFFF0000u : w[i / 2] << 16);
    return __builtin_bit_cast(float, w[i]);
}

__device__ __forceinline__ int64_t src_token(const QuantParams &p, int b, int64_t t) {
    return p.sel ? min(max(p.sel[(int64_t)b * p.n_sel + t], (int64_t)0), p.n_src - 1) : t;
}

// Lane roles of a tile: 8 channels 8 cg .. of tokens TPL tg .. TPL tg + TPL - 1.
template <int D>
struct Tile {
    static constexpr int CG = D / 8, TG = 64 / CG, TPL = 32 / TG;
};

// The tile of tokens [tok0, tok0 + nv): invalid rows repeat the first (min / max unchanged).
template <int IN, int D>
__device__ __forceinline__ void load_tile(const QuantParams &p, const void *x, int b, int64_t bh, int64_t tok0, int nv,
                                          int cg, int tg, uint32_t (&w)[Tile<D>::TPL][kInWords<IN>]) {
#pragma unroll
    for (int i = 0; i < Tile<D>::TPL; ++i) {
        const int tl = Tile<D>::TPL * tg + i;
        const int64_t off = (bh * p.n_src + src_token(p, b, tok0 + (tl < nv ? tl : 0))) * D + 8 * cg;
#pragma unroll
        for (int k = 0; k < kInWords<IN> / 4; ++k) {
            const u4 v = *((const u4 *)((const char *)x + off * (IN == AKV_DT_F32 ? 4 : 2)) + k);
#pragma unroll
            for (int j = 0; j < 4; ++j) w[i][4 * k + j] = v[j];
        }
    }
}

// Outlier channels of the tile's block: their values leave as float16 and read as zero below.
template <int IN, int D>
__device__ __forceinline__ void take_outliers(const int64_t *oidx, int n_out, void *odata, int64_t row0, int nv, int cg,
                                              int tg, uint32_t (&w)[Tile<D>::TPL][kInWords<IN>], bool store) {
    for (int j = 0; j < n_out; ++j) {
        const int d = (int)oidx[j];
        if (d / 8 != cg) continue;
        const int c = d & 7;
#pragma unroll
        for (int i = 0; i < Tile<D>::TPL; ++i) {
            const int tl = Tile<D>::TPL * tg + i;
            float v = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) v = e == c ? elem<IN>(w[i], e) : v;
            if (store && tl < nv) ((_Float16 *)odata)[(row0 + tl) * n_out + j] = (_Float16)v;
#pragma unroll
            for (int k = 0; k < kInWords<IN>; ++k) {
                const uint32_t m = IN == AKV_DT_F32 ? (k == c ? 0u : ~0u)
                                                    : (k != c / 2 ? ~0u : (c & 1) ? 0x0000FFFFu : 0xFFFF0000u);
                w[i][k] &= m;
            }
        }
    }
}

// min / max of the lane's 8 channels over its tokens
template <int IN, int D>
__device__ __forceinline__ void lane_minmax(const uint32_t (&w)[Tile<D>::TPL][kInWords<IN>], float (&mn)[8], float (&mx)[8]) {
    if constexpr (IN == AKV_DT_F16) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            h2 a = {(_Float16)INFINITY, (_Float16)INFINITY}, c = {-(_Float16)INFINITY, -(_Float16)INFINITY};
#pragma unroll
            for (int i = 0; i < Tile<D>::TPL; ++i) {
                a = __builtin_elementwise_min(a, as_h2(w[i][j]));
                c = __builtin_elementwise_max(c, as_h2(w[i][j]));
            }
            mn[2 * j] = fminf(mn[2 * j], (float)a[0]);
            mn[2 * j + 1] = fminf(mn[2 * j + 1], (float)a[1]);
            mx[2 * j] = fmaxf(mx[2 * j], (float)c[0]);
            mx[2 * j + 1] = fmaxf(mx[2 * j + 1], (float)c[1]);
        }
    } else {
#pragma unroll
        for (int i = 0; i < Tile<D>::TPL; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float v = elem<IN>(w[i], e);
                mn[e] = fminf(mn[e], v);
                mx[e] = fmaxf(mx[e], v);
            }
    }
}
// across the lanes that share the channels
template <int D>
__device__ __forceinline__ void wave_minmax(float (&mn)[8], float (&mx)[8]) {
#pragma unroll
    for (int o = Tile<D>::CG; o < 64; o <<= 1)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            mn[e] = fminf(mn[e], __shfl_xor(mn[e], o));
            mx[e] = fmaxf(mx[e], __shfl_xor(mx[e], o));
        }
}

template <int SB>
__device__ __forceinline__ void put_codes(const uint32_t (&v)[8], unsigned char *dst) {
    if (SB == 8) {
        u2 w = {0u, 0u};
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i / 4] |= (v[i] & 0xFFu) << (8 * (i & 3));
        *(u2 *)dst = w;
    } else if (SB == 4) {
        uint32_t w = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) w |= ((v[2 * i] << 4) | v[2 * i + 1]) << (8 * i);
        *(uint32_t *)dst = w;
    } else if (SB == 2) {
        uint32_t w = 0;
#pragma unroll
        for (int i = 0; i < 2; ++i)
            w |= ((v[4 * i] << 6) | (v[4 * i + 1] << 4) | (v[4 * i + 2] << 2) | v[4 * i + 3]) << (8 * i);
        *(uint16_t *)dst = (uint16_t)w;
    } else {
        uint32_t W = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) W |= v[i] << (21 - 3 * i);
        dst[0] = (unsigned char)(W >> 16);
        dst[1] = (unsigned char)(W >> 8);
        dst[2] = (unsigned char)W;
    }
}

// Codes of 8 channels in float16 arithmetic with at most 4 bits: the reciprocal form of
// quant_fast_kernel (r = 1 / scale in float32, equal codes for every float16 pair).
__device__ __forceinline__ void codes_f16(const uint32_t *w, const uint32_t (&nz)[4], const float (&r)[8], float maxv,
                                          uint32_t (&v)[8]) {
    const h2 k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
    const h2 hic = {(_Float16)(1024.0f + maxv), (_Float16)(1024.0f + maxv)};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t q = as_u32(as_h2(w[j]) + as_h2(nz[j]));
        uint32_t d = 0;
        asm volatile("v_fma_mixlo_f16 %0, %1, %2, 0 op_sel_hi:[1,0,0]" : "+v"(d) : "v"(q), "v"(r[2 * j]));
        asm volatile("v_fma_mixhi_f16 %0, %1, %2, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(d) : "v"(q), "v"(r[2 * j + 1]));
        h2 u = as_h2(d) + k1024;
        u = __builtin_elementwise_max(u, k1024);
        u = __builtin_elementwise_min(u, hic);
        v[2 * j] = as_u32(u) & 0x3FFu;
        v[2 * j + 1] = (as_u32(u) >> 16) & 0x3FFu;
    }
}

// nbytes (a multiple of 8) of staged rows to their contiguous destination (8-byte aligned)
__device__ __forceinline__ void copy_rows(const unsigned char *st, unsigned char *dst, int nbytes, int lane) {
    if (((uintptr_t)dst & 15u) == 0) {
        const int n16 = nbytes & ~15;
        for (int o = 16 * lane; o < n16; o += 1024) *(u4 *)(dst + o) = *(const u4 *)(st + o);
        if ((nbytes & 8) && lane == 0) *(u2 *)(dst + n16) = *(const u2 *)(st + n16);
    } else {
        for (int o = 8 * lane; o < nbytes; o += 512) *(u2 *)(dst + o) = *(const u2 *)(st + o);
    }
}

constexpr int kStageCodes = 32 * 128, kStageMeta = 2 * 32 * 4 * 4;

// Encode a K tile whose lane holds its channels' scale and zero.
template <int IN, int D, int SB>
__device__ __forceinline__ void encode_k(const uint32_t (&w)[Tile<D>::TPL][kInWords<IN>], const float (&sc)[8],
                                         const float (&ze)[8], float maxv, int cg, int tg, unsigned char *st) {
    constexpr int ROW = D * SB / 8;
    uint32_t nz[4] = {0, 0, 0, 0};
    float r[8] = {};
    if (IN == AKV_DT_F16 && SB <= 4) {
#pragma unroll
        for (int j = 0; j < 4; ++j) nz[j] = as_u32((h2){(_Float16)ze[2 * j], (_Float16)ze[2 * j + 1]}) ^ 0x80008000u;
#pragma unroll
        for (int e = 0; e < 8; ++e) r[e] = 1.0f / sc[e];
    }
#pragma unroll
    for (int i = 0; i < Tile<D>::TPL; ++i) {
        uint32_t v[8];
        if constexpr (IN == AKV_DT_F16 && SB <= 4) codes_f16(w[i], nz, r, maxv, v);
        else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = code_of<IN>(elem<IN>(w[i], e), ze[e], sc[e], maxv);
        }
        put_codes<SB>(v, st + (Tile<D>::TPL * tg + i) * ROW + cg * SB);
    }
}

// Per-token groups of LG lanes (G channels; `pad`: the group's channels past D are zeros).
template <int IN, int D, int SB>
__device__ __forceinline__ void encode_groups(const uint32_t (&w)[Tile<D>::TPL][kInWords<IN>], int LG, bool pad,
                                              float maxv, float lo, bool small, int cg, int tg, int rowb, int ng,
                                              unsigned char *st, float *meta) {
#pragma unroll
    for (int i = 0; i < Tile<D>::TPL; ++i) {
        float mn, mx;
        if constexpr (IN == AKV_DT_F16) {
            h2 a = {(_Float16)INFINITY, (_Float16)INFINITY};  // (min, -max)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const h2 x = as_h2(w[i][j]);
                const h2 lo2 = {x[0], -x[0]}, hi2 = {x[1], -x[1]};
                a = __builtin_elementwise_min(a, __builtin_elementwise_min(lo2, hi2));
            }
            for (int o = 1; o < LG; o <<= 1)
                a = __builtin_elementwise_min(a, as_h2((uint32_t)__shfl_xor((int)as_u32(a), o)));
            mn = (float)a[0];
            mx = -(float)a[1];
        } else {
            mn = INFINITY;
            mx = -INFINITY;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float x = elem<IN>(w[i], e);
                mn = fminf(mn, x);
                mx = fmaxf(mx, x);
            }
            for (int o = 1; o < LG; o <<= 1) {
                mn = fminf(mn, __shfl_xor(mn, o));
                mx = fmaxf(mx, __shfl_xor(mx, o));
            }
        }
        if (pad) {
            mn = fminf(mn, 0.f);
            mx = fmaxf(mx, 0.f);
        }
        const int tl = Tile<D>::TPL * tg + i;
        const float s = scale_of<IN>(mn, mx, maxv, lo);
        if (cg % LG == 0) {
            meta[tl * ng + cg / LG] = s;
            meta[128 + tl * ng + cg / LG] = mn;
        }
        uint32_t v[8];
        if (IN == AKV_DT_F16 && small) {
            const uint32_t z = as_u32((h2){(_Float16)mn, (_Float16)mn}) ^ 0x80008000u;
            const float r = 1.0f / s;
            const uint32_t nz[4] = {z, z, z, z};
            const float r8[8] = {r, r, r, r, r, r, r, r};
            codes_f16(w[i], nz, r8, maxv, v);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = code_of<IN>(elem<IN>(w[i], e), mn, s, maxv);
        }
        put_codes<SB>(v, st + tl * rowb + cg * SB);
        if (pad) {
            const uint32_t c0 = code_of<IN>(0.f, mn, s, maxv);
            const uint32_t v0[8] = {c0, c0, c0, c0, c0, c0, c0, c0};
            put_codes<SB>(v0, st + tl * rowb + (Tile<D>::CG + cg) * SB);
        }
    }
}

template <int DT>
__device__ __forceinline__ void store_meta(void *dst, int64_t i, float v) {
    if (DT == AKV_DT_F16) ((_Float16 *)dst)[i] = (_Float16)v;
    else if (DT == AKV_DT_BF16) ((uint16_t *)dst)[i] = f32_to_bf16_rne(v);
    else ((float *)dst)[i] = v;
}

__device__ __forceinline__ int64_t block_end(const QuantParams &p, int64_t blk) { return min((blk + 1) * p.T, p.n_sel); }

// K tile: encode with the lane's statistics, copy out, and (meta) write the block's scale / zero
template <int IN, int D>
__device__ __forceinline__ void finish_k(const QuantParams &p, const uint32_t (&w)[Tile<D>::TPL][kInWords<IN>],
                                         const float (&sc)[8], const float (&ze)[8], int64_t bh, int64_t tok0, int nv,
                                         int cg, int tg, int lane, unsigned char *st) {
    const float maxv = (float)((1 << p.bits_k) - 1);
    if (p.bits_k == 2) encode_k<IN, D, 2>(w, sc, ze, maxv, cg, tg, st);
    else if (p.bits_k == 3) encode_k<IN, D, 3>(w, sc, ze, maxv, cg, tg, st);
    else if (p.bits_k == 4) encode_k<IN, D, 4>(w, sc, ze, maxv, cg, tg, st);
    else encode_k<IN, D, 8>(w, sc, ze, maxv, cg, tg, st);
    __builtin_amdgcn_wave_barrier();
    copy_rows(st, (unsigned char *)p.k_codes + (bh * p.n_sel + tok0) * p.k_row, nv * p.k_row, lane);
    __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ void put_kmeta(const QuantParams &p, const float (&sc)[8], const float (&ze)[8], int64_t row,
                                          int cg) {
    h8 s, z;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        s[e] = (_Float16)sc[e];
        z[e] = (_Float16)ze[e];
    }
    *(h8 *)((_Float16 *)p.k_scale + row * p.D + 8 * cg) = s;
    *(h8 *)((_Float16 *)p.k_zero + row * p.D + 8 * cg) = z;
}

}  // namespace

// grid (x: tiles / blocks / tile runs, H, B * tensors); ksrc: where K's statistics come from
template <int IN, int D>
__global__ __launch_bounds__(64 * kTileWaves) void qtile_kernel(const QuantParams p, int ksrc, int vgrp) {
    __shared__ __align__(16) unsigned char stage[kTileWaves][kStageCodes + kStageMeta];
    __shared__ float red[kTileWaves][2][D];
    using TL = Tile<D>;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int cg = lane % TL::CG, tg = lane / TL::CG;
    const int nt = (ksrc != kKNone) + vgrp;
    const int b = blockIdx.z / nt, h = blockIdx.y;
    const bool is_k = ksrc != kKNone && (int)blockIdx.z % nt == 0;
    const int64_t bh = (int64_t)b * p.H + h;
    unsigned char *st = stage[wave];
    uint32_t w[TL::TPL][kInWords<IN>];

    if (is_k && ksrc != kKGroups) {
        const float maxv = (float)((1 << p.bits_k) - 1);
        float mn[8], mx[8], sc[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            mn[e] = INFINITY;
            mx[e] = -INFINITY;
        }
        const int64_t *oidx = nullptr;
        if (ksrc == kKTile) {
            const int64_t blk = (int64_t)blockIdx.x * kTileWaves + wave;
            if (blk >= p.nblk) return;
            const int64_t t0 = blk * p.T;
            const int nv = (int)(block_end(p, blk) - t0);
            load_tile<IN, D>(p, p.k, b, bh, t0, nv, cg, tg, w);
            if (p.n_out) {
                oidx = p.k_oidx + ((int64_t)b * p.nblk + blk) * p.n_out;
                take_outliers<IN, D>(oidx, p.n_out, p.k_odata, bh * p.n_sel + t0, nv, cg, tg, w, true);
            }
            lane_minmax<IN, D>(w, mn, mx);
            wave_minmax<D>(mn, mx);
#pragma unroll
            for (int e = 0; e < 8; ++e) sc[e] = scale_of<IN>(mn[e], mx[e], maxv, p.lo);
            if (tg == 0) put_kmeta(p, sc, mn, bh * p.nblk + blk, cg);
            finish_k<IN, D>(p, w, sc, mn, bh, t0, nv, cg, tg, lane, st);
            return;
        }
        // a block per workgroup, or a run of kEncTiles tiles of a block whose partials are known
        const int tpb = (p.T + 31) / 32;
        const int runs = ksrc == kKPartials ? (tpb + kEncTiles - 1) / kEncTiles : 1;
        const int64_t blk = blockIdx.x / runs;
        if (blk >= p.nblk) return;
        const int64_t t0 = blk * p.T, t1 = block_end(p, blk);
        const int ntile = (int)((t1 - t0 + 31) / 32);
        const int first = ksrc == kKPartials ? (int)(blockIdx.x % runs) * kEncTiles : 0;
        const int last = ksrc == kKPartials ? min(first + kEncTiles, ntile) : ntile;
        if (first >= ntile) return;
        if (p.n_out) oidx = p.k_oidx + ((int64_t)b * p.nblk + blk) * p.n_out;
        auto tile_in = [&](int i, bool store) {
            const int64_t tok0 = t0 + 32 * (int64_t)i;
            const int nv = (int)min((int64_t)32, t1 - tok0);
            load_tile<IN, D>(p, p.k, b, bh, tok0, nv, cg, tg, w);
            if (oidx) take_outliers<IN, D>(oidx, p.n_out, p.k_odata, bh * p.n_sel + tok0, nv, cg, tg, w, store);
        };
        if (ksrc == kKPartials) {
            // thread = (statistic, channel) over the block's chunks
            const float *part = p.ws + (bh * p.nblk + blk) * p.nchunk * 2 * D;
            for (int i = threadIdx.x; i < 2 * D; i += 64 * kTileWaves) {
                float v = i < D ? INFINITY : -INFINITY;
#pragma unroll 8
                for (int c = 0; c < p.nchunk; ++c) {
                    const float x = part[(int64_t)c * 2 * D + i];
                    v = i < D ? fminf(v, x) : fmaxf(v, x);
                }
                red[0][i / D][i % D] = v;
            }
            __syncthreads();
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                mn[e] = red[0][0][8 * cg + e];
                mx[e] = red[0][1][8 * cg + e];
            }
            for (int j = 0; oidx && j < p.n_out; ++j) {  // their channel holds zeros only
                const int d = (int)oidx[j];
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (d == 8 * cg + e) mn[e] = mx[e] = 0.f;
            }
        } else {
            for (int i = wave; i < ntile; i += kTileWaves) {
                tile_in(i, true);
                lane_minmax<IN, D>(w, mn, mx);
            }
            wave_minmax<D>(mn, mx);
            if (tg == 0)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    red[wave][0][8 * cg + e] = mn[e];
                    red[wave][1][8 * cg + e] = mx[e];
                }
            __syncthreads();
#pragma unroll
            for (int e = 0; e < 8; ++e)
#pragma unroll
                for (int o = 0; o < kTileWaves; ++o) {
                    mn[e] = fminf(mn[e], red[o][0][8 * cg + e]);
                    mx[e] = fmaxf(mx[e], red[o][1][8 * cg + e]);
                }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) sc[e] = scale_of<IN>(mn[e], mx[e], maxv, p.lo);
        if (first == 0 && wave == 0 && tg == 0) put_kmeta(p, sc, mn, bh * p.nblk + blk, cg);
        const bool held = ksrc == kKBlock && ntile <= kTileWaves;  // the wave's one tile is in registers
        for (int i = first + wave; i < last; i += kTileWaves) {
            if (!held) tile_in(i, ksrc == kKPartials);
            const int64_t tok0 = t0 + 32 * (int64_t)i;
            finish_k<IN, D>(p, w, sc, mn, bh, tok0, (int)min((int64_t)32, t1 - tok0), cg, tg, lane, st);
        }
        return;
    }

    // ------------------------------------------- per-token groups: V, or K of the group layouts
    const void *x = is_k ? p.k : p.v;
    const int bits = is_k ? p.bits_k : p.bits_v, sb = is_k ? p.sbits_k : p.sbits_v;
    const int G = is_k ? p.G_k : p.G_v, rowb = is_k ? p.k_row : p.v_row, ng = p.pD / G;
    const int64_t tile = (int64_t)blockIdx.x * kTileWaves + wave;
    int64_t tok0, t1;
    const int64_t *oidx = nullptr;
    if (!is_k && p.n_out) {  // the tile lies in one block, whose outlier channels are known
        const int tpb = (p.T + 31) / 32;
        const int64_t blk = tile / tpb;
        if (blk >= p.nblk) return;
        tok0 = blk * p.T + 32 * (tile % tpb);
        t1 = block_end(p, blk);
        oidx = p.v_oidx + ((int64_t)b * p.nblk + blk) * p.n_out;
    } else {
        tok0 = 32 * tile;
        t1 = p.n_sel;
    }
    if (tok0 >= t1) return;
    const int nv = (int)min((int64_t)32, t1 - tok0);
    load_tile<IN, D>(p, x, b, bh, tok0, nv, cg, tg, w);
    if (oidx) take_outliers<IN, D>(oidx, p.n_out, p.v_odata, bh * p.n_sel + tok0, nv, cg, tg, w, true);
    const float maxv = (float)((1 << bits) - 1);
    const bool pad = p.pD > D;
    const int LG = pad ? TL::CG : G / 8;
    float *meta = (float *)(st + kStageCodes);
    if (sb == 2) encode_groups<IN, D, 2>(w, LG, pad, maxv, p.lo, true, cg, tg, rowb, ng, st, meta);
    else if (sb == 3) encode_groups<IN, D, 3>(w, LG, pad, maxv, p.lo, true, cg, tg, rowb, ng, st, meta);
    else if (sb == 4) encode_groups<IN, D, 4>(w, LG, pad, maxv, p.lo, true, cg, tg, rowb, ng, st, meta);
    else encode_groups<IN, D, 8>(w, LG, pad, maxv, p.lo, bits <= 4, cg, tg, rowb, ng, st, meta);
    __builtin_amdgcn_wave_barrier();
    copy_rows(st, (unsigned char *)(is_k ? p.k_codes : p.v_codes) + (bh * p.n_sel + tok0) * rowb, nv * rowb, lane);
    const int64_t m0 = (bh * p.n_sel + tok0) * ng;
    void *msc = is_k ? p.k_scale : p.v_scale, *mze = is_k ? p.k_zero : p.v_zero;
    for (int i = lane; i < nv * ng; i += 64) {
        if (p.meta_dt == AKV_DT_F16) {  // the affine tier's meta is float16 whatever the input
            store_meta<AKV_DT_F16>(msc, m0 + i, meta[i]);
            store_meta<AKV_DT_F16>(mze, m0 + i, meta[128 + i]);
        } else {
            store_meta<IN>(msc, m0 + i, meta[i]);
            store_meta<IN>(mze, m0 + i, meta[128 + i]);
        }
    }
}

// min / max partials of chunk c of a long block: grid (nblk * nchunk, H, B).  (An outlier
// channel's partials are not used: the encoder sets its statistics to zero.)  Bound by the
// latency of the index and row loads, so a wave takes one tile of the chunk, not four in turn:
// 16,255 tokens x 8 heads (33 MB) 17.7 -> 9.8 us.
template <int IN, int D>
__global__ __launch_bounds__(64 * kStatWaves) void kstat_kernel(const QuantParams p) {
    __shared__ float red[kStatWaves][2][D];
    using TL = Tile<D>;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int cg = lane % TL::CG, tg = lane / TL::CG;
    const int64_t blk = blockIdx.x / p.nchunk;
    const int c = (int)(blockIdx.x % p.nchunk), b = blockIdx.z;
    const int64_t bh = (int64_t)b * p.H + blockIdx.y;
    const int64_t t1 = block_end(p, blk), c0 = blk * p.T + (int64_t)c * p.chunk_tokens;
    const int64_t c1 = min(c0 + p.chunk_tokens, t1);
    float mn[8], mx[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        mn[e] = INFINITY;
        mx[e] = -INFINITY;
    }
    for (int64_t t = c0 + 32 * wave; t < c1; t += 32 * kStatWaves) {
        uint32_t w[TL::TPL][kInWords<IN>];
        load_tile<IN, D>(p, p.k, b, bh, t, (int)min((int64_t)32, c1 - t), cg, tg, w);
        lane_minmax<IN, D>(w, mn, mx);
    }
    wave_minmax<D>(mn, mx);
    if (tg == 0)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            red[wave][0][8 * cg + e] = mn[e];
            red[wave][1][8 * cg + e] = mx[e];
        }
    __syncthreads();
    float *part = p.ws + ((bh * p.nblk + blk) * p.nchunk + c) * 2 * D;
    for (int i = threadIdx.x; i < 2 * D; i += 64 * kStatWaves) {
        float v = red[0][i / D][i % D];
        for (int o = 1; o < kStatWaves; ++o)
            v = i < D ? fminf(v, red[o][i / D][i % D]) : fmaxf(v, red[o][i / D][i % D]);
        part[i] = v;
    }
}

// ------------------------------------------------------- outlier channels
// The n_out channels of a (batch, block) with the largest mean over heads of the L2 norm
// over the block's tokens (akv/affine_quantizer.py:76-80), ties to the lower index.  The
// squares of a (head, channel) are added in token order and the norms in head order: the
// sums of outlier_select_kernel (quant.hip), so near ties fall the same way.

namespace {

// cn[0..D): pick the n_out largest into oidx; one wave.  A NaN at the lowest index left is
// taken first and any other NaN never (the comparison v > best of a serial scan).
__device__ __forceinline__ void rank_channels(const float *cn, int D, int n_out, int64_t *oidx, int lane) {
    uint32_t taken = 0;  // bit i: channel lane + 64 i
    for (int j = 0; j < n_out; ++j) {
        uint64_t best = 0;  // (value, 255 - index): norms are >= +0 or NaN
        int head = D;       // lowest channel left
        bool head_nan = false;
        for (int i = 0; i < 2; ++i) {
            const int d = lane + 64 * i;
            if (d >= D || (taken >> i & 1u)) continue;
            const float v = cn[d];
            if (d < head) {
                head = d;
                head_nan = v != v;
            }
            if (v == v) {
                const uint64_t k = ((uint64_t)__builtin_bit_cast(uint32_t, v) << 8) | (uint32_t)(255 - d);
                best = k > best ? k : best;
            }
        }
        for (int o = 32; o; o >>= 1) {
            const uint64_t k = (uint64_t)__shfl_xor((unsigned long long)best, o);
            best = k > best ? k : best;
            const int hd = __shfl_xor(head, o), hn = __shfl_xor((int)head_nan, o);
            if (hd < head) {
                head = hd;
                head_nan = hn != 0;
            }
        }
        const int d = head_nan ? head : 255 - (int)(best & 255u);
        if (lane == 0) oidx[j] = d;
        if (d % 64 == lane) taken |= 1u << (d / 64);
    }
}

}  // namespace

// Blocks of any length without a workspace: a workgroup per (block, batch, tensor), a lane
// per (head, 8 channels) adding its tokens one after another, 8 loads in flight.
template <int IN, int D>
__global__ __launch_bounds__(256) void outlier_block_kernel(const QuantParams p) {
    constexpr int CG = D / 8, HS = 256 / CG;  // heads per pass
    __shared__ float ns[HS][D];
    __shared__ float cn[D];
    const int cg = threadIdx.x % CG, hs = threadIdx.x / CG;
    const int64_t blk = blockIdx.x;
    const int b = blockIdx.y;
    const bool is_k = p.k && blockIdx.z == 0;
    const void *x = is_k ? p.k : p.v;
    const int64_t t0 = blk * p.T, t1 = block_end(p, blk);
    float acc = 0.f;  // thread d < D: sum over the heads so far
    for (int h0 = 0; h0 < p.H; h0 += HS) {
        const int h = min(h0 + hs, p.H - 1);
        const int64_t bh = (int64_t)b * p.H + h;
        float ss[8] = {};
        for (int64_t t = t0; t < t1; t += 8) {
            uint32_t w[8][kInWords<IN>];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int64_t off = (bh * p.n_src + src_token(p, b, min(t + i, t1 - 1))) * D + 8 * cg;
#pragma unroll
                for (int k = 0; k < kInWords<IN> / 4; ++k) {
                    const u4 v = *((const u4 *)((const char *)x + off * (IN == AKV_DT_F32 ? 4 : 2)) + k);
#pragma unroll
                    for (int j = 0; j < 4; ++j) w[i][4 * k + j] = v[j];
                }
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if (t + i < t1)
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float v = elem<IN>(w[i], e);
                        ss[e] += v * v;
                    }
            }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) ns[hs][8 * cg + e] = sqrtf(ss[e]);
        __syncthreads();
        if (threadIdx.x < D)
            for (int i = 0; i < HS && h0 + i < p.H; ++i) acc += ns[i][threadIdx.x];
        __syncthreads();
    }
    if (threadIdx.x < D) cn[threadIdx.x] = acc / (float)p.H;
    __syncthreads();
    if (threadIdx.x < 64)
        rank_channels(cn, D, p.n_out, (is_k ? p.k_oidx : p.v_oidx) + ((int64_t)b * p.nblk + blk) * p.n_out, threadIdx.x);
}

// Long blocks: a workgroup per (head, half row of 64 channels; block; batch x tensor).  All 8
// waves square tiles of 256 tokens into LDS (double-buffered, the next tile's loads in
// flight), wave 0 adds them in token order, one channel per lane.  Bound by that chain of
// dependent adds: ~8 cycles per token (16k tokens: about 60 us; the lanes of
// outlier_block_kernel would wait for memory every 8 tokens).
constexpr int kNormTokens = 256;
template <int IN, int D>
__global__ __launch_bounds__(512) void outlier_norm_kernel(const QuantParams p) {
    extern __shared__ __align__(16) float sq[];  // [2][kNormTokens][64]
    constexpr int PT = kNormTokens / 64;         // tokens per thread and tile: 64 rows of 8 lanes
    const int half = blockIdx.x % (D / 64), h = blockIdx.x / (D / 64);
    const int64_t blk = blockIdx.y;
    const int nt = (p.k != nullptr) + (p.v != nullptr);
    const int b = blockIdx.z / nt;
    const bool is_k = p.k && blockIdx.z % nt == 0;
    const void *x = is_k ? p.k : p.v;
    const int tid = threadIdx.x, cg = tid % 8, row = tid / 8;
    const int64_t bh = (int64_t)b * p.H + h, t0 = blk * p.T, t1 = block_end(p, blk);
    uint32_t w[PT][kInWords<IN>];
    auto load = [&](int64_t t) {
#pragma unroll
        for (int i = 0; i < PT; ++i) {
            const int64_t tok = min(t + 64 * i + row, t1 - 1);
            const int64_t off = (bh * p.n_src + src_token(p, b, tok)) * D + 64 * half + 8 * cg;
#pragma unroll
            for (int k = 0; k < kInWords<IN> / 4; ++k) {
                const u4 v = *((const u4 *)((const char *)x + off * (IN == AKV_DT_F32 ? 4 : 2)) + k);
#pragma unroll
                for (int j = 0; j < 4; ++j) w[i][4 * k + j] = v[j];
            }
        }
    };
    float ss = 0.f;
    load(t0);
    int buf = 0;
    for (int64_t t = t0; t < t1; t += kNormTokens, buf ^= 1) {
        float *dst = sq + buf * kNormTokens * 64;
#pragma unroll
        for (int i = 0; i < PT; ++i) {
            f4 lo, hi;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float a = elem<IN>(w[i], e), c = elem<IN>(w[i], 4 + e);
                lo[e] = a * a;
                hi[e] = c * c;
            }
            float *r = dst + (64 * i + row) * 64 + 8 * cg;
            *(f4 *)r = lo;
            *(f4 *)(r + 4) = hi;
        }
        // one barrier per tile: wave 0 sums tile j while the others write tile j + 1 into the other
        // buffer, and reaches the next barrier only after its sum, before j + 2 reuses this one
        __syncthreads();
        if (t + kNormTokens < t1) load(t + kNormTokens);
        if (tid < 64) {
            const int n = (int)min((int64_t)kNormTokens, t1 - t);
            int i = 0;
            for (; i + 16 <= n; i += 16) {
                float v[16];
#pragma unroll
                for (int k = 0; k < 16; ++k) v[k] = dst[(i + k) * 64 + tid];
#pragma unroll
                for (int k = 0; k < 16; ++k) ss += v[k];
            }
            for (; i < n; ++i) ss += dst[i * 64 + tid];
        }
    }
    if (tid < 64) {
        float *norms = p.ws + p.norm_off;
        const int which = p.k && p.v ? (is_k ? 0 : 1) : 0;
        norms[((((int64_t)b * p.nblk + blk) * 2 + which) * p.H + h) * D + 64 * half + tid] = sqrtf(ss);
    }
}
template <int D>
__global__ __launch_bounds__(128) void outlier_rank_kernel(const QuantParams p) {
    __shared__ float cn[D];
    const int64_t blk = blockIdx.x;
    const int b = blockIdx.y, which = blockIdx.z;
    const bool is_k = p.k && which == 0;
    if (threadIdx.x < D) {
        const float *n = p.ws + p.norm_off + (((int64_t)b * p.nblk + blk) * 2 + which) * p.H * D + threadIdx.x;
        float acc = 0.f;
#pragma unroll 8
        for (int h = 0; h < p.H; ++h) acc += n[(int64_t)h * D];
        cn[threadIdx.x] = acc / (float)p.H;
    }
    __syncthreads();
    if (threadIdx.x < 64)
        rank_channels(cn, D, p.n_out, (is_k ? p.k_oidx : p.v_oidx) + ((int64_t)b * p.nblk + blk) * p.n_out, threadIdx.x);
}

// ------------------------------------------------------------- host side

// The tensors of the batch elements are the grid's last dimension: past its limit the call stays
// with quant_kernel, whose last dimension is the batch alone.
constexpr int64_t kGridYZ = 65535;

bool quant_tile_eligible(const QuantParams &p) {
    if ((int64_t)p.B * ((p.k != nullptr) + (p.v != nullptr)) > kGridYZ) return false;
    const uintptr_t al = (uintptr_t)p.k | (uintptr_t)p.v | (uintptr_t)p.k_codes | (uintptr_t)p.v_codes;
    const uintptr_t meta = p.k_mode == 0 ? (uintptr_t)p.k_scale | (uintptr_t)p.k_zero : 0;
    return ((al | meta) & 15u) == 0 && p.ar_dt == p.in_dt && !p.symmetric;
}

// Chunks of the long-block statistics (0: the block's own workgroup computes them).
int quant_stat_chunks(const QuantParams &p, int *tokens) {
    if (!p.k || p.k_mode != 0 || p.T <= kLongT || (int64_t)p.B * p.H * p.nblk >= 512) return 0;
    const int64_t T = p.T < p.n_sel ? p.T : p.n_sel;
    if (T <= kLongT) return 0;
    int64_t ct = kStatTokens;
    if (T > ct * kMaxChunks) ct = (T + kMaxChunks - 1) / kMaxChunks;
    ct = (ct + 127) / 128 * 128;
    *tokens = (int)ct;
    return (int)((T + ct - 1) / ct);
}

// Outlier norms go through the workspace for blocks longer than kLongT (a grid row each).
bool quant_norms_in_ws(const QuantParams &p) {
    return p.n_out > 0 && p.T > kLongT && p.n_sel > kLongT && p.nblk <= kGridYZ && (p.k || p.v);
}

template <int IN, int D>
static hipError_t launch_outliers(const QuantParams &p, hipStream_t s) {
    const unsigned nt = (p.k != nullptr) + (p.v != nullptr);
    if (p.ws && quant_norms_in_ws(p)) {
        constexpr int lds = 2 * kNormTokens * 64 * 4;  // 128 KiB
        static std::atomic<uint64_t> attr_devs{0};     // a bit per device index; racing threads both set it
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return e;
        const uint64_t bit = (dev >= 0 && dev < 64) ? 1ull << dev : 0ull;
        if (!bit || !(attr_devs.load(std::memory_order_acquire) & bit)) {
            e = hipFuncSetAttribute((const void *)outlier_norm_kernel<IN, D>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
            if (e != hipSuccess) return e;
            attr_devs.fetch_or(bit, std::memory_order_release);
        }
        hipLaunchKernelGGL((outlier_norm_kernel<IN, D>), dim3(p.H * (D / 64), (unsigned)p.nblk, p.B * nt), dim3(512), lds,
                           s, p);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        hipLaunchKernelGGL(outlier_rank_kernel<D>, dim3((unsigned)p.nblk, p.B, nt), dim3(128), 0, s, p);
    } else {
        hipLaunchKernelGGL((outlier_block_kernel<IN, D>), dim3((unsigned)p.nblk, p.B, nt), dim3(256), 0, s, p);
    }
    return hipGetLastError();
}

template <int IN, int D>
static hipError_t launch_tiles(const QuantParams &p, hipStream_t s) {
    if (p.n_out > 0) {
        const hipError_t e = launch_outliers<IN, D>(p, s);
        if (e != hipSuccess) return e;
    }
    const int vgrp = p.v ? 1 : 0;
    int ksrc = kKNone;
    int64_t gx = 0;
    const int64_t T = p.T < p.n_sel ? p.T : p.n_sel, tpb = (T + 31) / 32;
    if (p.k) {
        if (p.k_mode == 1) {
            ksrc = kKGroups;
            gx = (p.n_sel + 127) / 128;
        } else if (T <= 32) {
            ksrc = kKTile;
            gx = (p.nblk + kTileWaves - 1) / kTileWaves;
        } else if (p.nchunk > 0) {
            ksrc = kKPartials;
            gx = p.nblk * ((tpb + kEncTiles - 1) / kEncTiles);
            hipLaunchKernelGGL((kstat_kernel<IN, D>), dim3((unsigned)(p.nblk * p.nchunk), p.H, p.B),
                               dim3(64 * kStatWaves), 0, s, p);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
        } else {
            ksrc = kKBlock;
            gx = p.nblk;
        }
    }
    if (p.v) {
        const int64_t tiles = p.n_out ? p.nblk * tpb : (p.n_sel + 31) / 32;
        const int64_t g = (tiles + kTileWaves - 1) / kTileWaves;
        if (g > gx) gx = g;
    }
    hipLaunchKernelGGL((qtile_kernel<IN, D>), dim3((unsigned)gx, p.H, p.B * ((ksrc != kKNone) + vgrp)),
                       dim3(64 * kTileWaves), 0, s, p, ksrc, vgrp);
    return hipGetLastError();
}

hipError_t quant_tile_launch(const QuantParams &p, hipStream_t s) {
    if (!p.k && !p.v) return hipSuccess;
    QuantParams q = p;
    q.T = (int)(p.T < p.n_sel ? p.T : p.n_sel);  // one block either way when T >= n_sel
#define AKV_QT(in)                                                    \
    if (p.in_dt == in) return p.D == 128 ? launch_tiles<in, 128>(q, s) : launch_tiles<in, 64>(q, s);
    AKV_QT(AKV_DT_F16) AKV_QT(AKV_DT_BF16) AKV_QT(AKV_DT_F32)
#undef AKV_QT
    return hipErrorInvalidValue;
}

}  // namespace akv
