// Dequant / unpack to dense values, device bit-packing, and the importance
// update from materialised attention weights.
#include <atomic>

#include "akv_common.h"
#include "misc.h"

namespace akv {

// ------------------------------------------------------------------ dequant
// One thread per (row, 8-channel chunk).  AFFINE: fp16 codes*scale + zero with
// two roundings, then outlier channels replaced (akv/affine_quantizer.py:112-124,
// :178-189).  LEGACY: fp32 u*s + z or (u - maxv//2)*s cast to the output dtype
// (akv/triton_ops.py:657-713, akv/fused_attention.py:281-317).
__global__ __launch_bounds__(256) void dequant_kernel(const DequantParams p) {
    const int nch = p.D / 8;
    const int64_t task = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t rows = (int64_t)p.nbh * p.n_warm;
    if (task >= rows * nch) return;
    const int ch8 = (int)(task % nch);
    const int64_t bh = task / nch / p.n_warm, t = task / nch % p.n_warm;
    const int64_t row = bh * p.tok_stride + t;  // input row (bh, token)
    const int64_t blk = p.blk_of ? (int64_t)p.blk_of[t] : t / p.T;
    const int64_t orow = bh * p.out_tokens + (p.out_slot ? p.out_slot[t] : t);
    for (int which = 0; which < 2; ++which) {
        void *out = which == 0 ? p.k_out : p.v_out;
        if (!out) continue;
        const int bits = which == 0 ? p.bits_k : p.bits_v;
        const unsigned char *codes = (const unsigned char *)(which == 0 ? p.kc : p.vc) + row * (which == 0 ? p.kc_row : p.vc_row);
        const void *sc = which == 0 ? p.ks : p.vs;
        const void *ze = which == 0 ? p.kz : p.vz;
        float vals[8];
        for (int i = 0; i < 8; ++i) {
            const int d = 8 * ch8 + i;
            const uint32_t c = extract_code(codes, d, bits);
            if (p.kind == AKV_WARM_AFFINE) {
                int64_t mi;
                if (which == 0) mi = (bh * p.nblk + blk) * p.D + d;              // per channel, per block
                else mi = row * (p.D / p.Gv) + d / p.Gv;                          // per token, per group
                const _Float16 s = ((const _Float16 *)sc)[mi], z = ((const _Float16 *)ze)[mi];
                _Float16 v = (_Float16)c * s;
                v = v + z;
                vals[i] = (float)v;
            } else {
                const int64_t mi = row * p.lg + d / p.gs;
                const float s = load_as_f32(sc, mi, p.meta_dt);
                const int sym = p.sym_flags ? p.sym_flags[which] : p.legacy_sym;
                float v;
                if (sym) v = ((float)c - (float)(((1 << bits) - 1) / 2)) * s;  // maxv // 2
                else {
                    v = (float)c * s;
                    v = v + load_as_f32(ze, mi, p.meta_dt);
                }
                vals[i] = v;
            }
        }
        if (p.kind == AKV_WARM_AFFINE && p.n_out > 0) {
            const int64_t *oi = (which == 0 ? p.k_oidx : p.v_oidx) + ((bh / p.Hkv) * p.nblk + blk) * p.n_out;
            const _Float16 *od = (const _Float16 *)(which == 0 ? p.k_odata : p.v_odata) + row * p.n_out;
            for (int j = 0; j < p.n_out; ++j) {
                const int d = (int)oi[j];
                if (d / 8 == ch8) {
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        if (d % 8 == i) vals[i] = (float)od[j];
                }
            }
        }
        const int64_t o = orow * p.D + 8 * ch8;
        for (int i = 0; i < 8; ++i) {
            if (p.out_dt == AKV_DT_F16) ((_Float16 *)out)[o + i] = (_Float16)vals[i];
            else if (p.out_dt == AKV_DT_BF16) ((uint16_t *)out)[o + i] = f32_to_bf16_rne(vals[i]);
            else ((float *)out)[o + i] = vals[i];
        }
    }
}

// ------------------------------------------------------- dequant, whole chunks
// The same arithmetic for tiers whose rows, meta and outputs lie on vector boundaries
// (head_dim a multiple of 32, groups of a multiple of 8): a thread owns 8 channels of
// kDqTok tokens of one (batch, head) and one of K / V, with one load for the codes, one for
// the scales and zeros (K: 16 bytes each; V and legacy: one value of the chunk's group) and
// 16-byte stores; all its tokens' loads are in flight together.  HBM-bound: it writes what
// the view holds and reads a fraction of that.  Before, each code, scale and zero was a load
// of its own behind three 64-bit divisions per thread (dequant_kernel): 16,255 tokens x 8
// heads of K and V at 3 bits 101 -> 28 us (2.9 TB/s, scattered to their positions); 3,969
// tokens x 32 heads of legacy 2-bit rows 52 -> 12.8 us (2.9 TB/s).
namespace {
constexpr int kDqTok = 4;

// the 8 codes of chunk ch8 of a packed row whose start is 4-byte aligned (8 with 8 bits)
__device__ __forceinline__ void chunk_codes(const unsigned char *row, int ch8, int bits, uint32_t (&c)[8]) {
    if (bits == 4) {
        const uint32_t w = *(const uint32_t *)(row + 4 * ch8);
#pragma unroll
        for (int i = 0; i < 8; ++i) c[i] = (w >> (8 * (i / 2) + ((i & 1) ? 0 : 4))) & 15u;
    } else if (bits == 2) {
        const uint32_t w = *(const uint16_t *)(row + 2 * ch8);
#pragma unroll
        for (int i = 0; i < 8; ++i) c[i] = (w >> (8 * (i / 4) + 6 - 2 * (i & 3))) & 3u;
    } else if (bits == 3) {  // 3 bytes, in one or two aligned words of the row
        const int o = 3 * ch8;
        const uint32_t *w = (const uint32_t *)row + o / 4;
        const uint32_t lo = w[0], hi = (o & 3) > 1 ? w[1] : 0u;
        const uint32_t x = (uint32_t)((((uint64_t)hi << 32) | lo) >> (8 * (o & 3)));
        const uint32_t W = ((x & 0xFFu) << 16) | (x & 0xFF00u) | ((x >> 16) & 0xFFu);
#pragma unroll
        for (int i = 0; i < 8; ++i) c[i] = (W >> (21 - 3 * i)) & 7u;
    } else {
        const u2 w = *(const u2 *)(row + 8 * ch8);
#pragma unroll
        for (int i = 0; i < 8; ++i) c[i] = (w[i / 4] >> (8 * (i & 3))) & 0xFFu;
    }
}
template <int OUT>
__device__ __forceinline__ void store_chunk(void *out, int64_t o, const float (&v)[8]) {
    if (OUT == AKV_DT_F32) {
        *(f4 *)((float *)out + o) = (f4){v[0], v[1], v[2], v[3]};
        *(f4 *)((float *)out + o + 4) = (f4){v[4], v[5], v[6], v[7]};
    } else if (OUT == AKV_DT_F16) {
        h8 x;
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = (_Float16)v[i];
        *(h8 *)((_Float16 *)out + o) = x;
    } else {
        u4 x;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            x[i] = (uint32_t)f32_to_bf16_rne(v[2 * i]) | ((uint32_t)f32_to_bf16_rne(v[2 * i + 1]) << 16);
        *(u4 *)((uint16_t *)out + o) = x;
    }
}
}  // namespace

template <bool AFFINE, int OUT>
__global__ __launch_bounds__(256) void dequant_chunk_kernel(const DequantParams p) {
    const int nch = p.D / 8, per = 256 / nch;  // tokens of one pass of the workgroup
    const int ch8 = threadIdx.x % nch, tr = threadIdx.x / nch;
    const bool is_k = p.k_out && blockIdx.z == 0;
    void *out = is_k ? p.k_out : p.v_out;
    const int bits = is_k ? p.bits_k : p.bits_v, row_bytes = is_k ? p.kc_row : p.vc_row;
    const unsigned char *codes = (const unsigned char *)(is_k ? p.kc : p.vc);
    const void *sc = is_k ? p.ks : p.vs, *ze = is_k ? p.kz : p.vz;
    const int64_t bh = blockIdx.y, t0 = (int64_t)blockIdx.x * per * kDqTok + tr;
    if (tr >= per) return;
    const int sym = AFFINE ? 0 : p.sym_flags ? p.sym_flags[is_k ? 0 : 1] : p.legacy_sym;
    const float half_max = (float)(((1 << bits) - 1) / 2);
    uint32_t c[kDqTok][8];
    h8 s8[kDqTok], z8[kDqTok];
    float sf[kDqTok], zf[kDqTok];
    int64_t orow[kDqTok], blk[kDqTok];
#pragma unroll
    for (int i = 0; i < kDqTok; ++i) {
        const int64_t t = min(t0 + (int64_t)i * per, p.n_warm - 1), row = bh * p.tok_stride + t;
        orow[i] = bh * p.out_tokens + (p.out_slot ? p.out_slot[t] : t);
        chunk_codes(codes + row * row_bytes, ch8, bits, c[i]);
        if (AFFINE) {
            blk[i] = p.blk_of ? (int64_t)p.blk_of[t] : (int64_t)((uint32_t)t / (uint32_t)p.T);
            if (is_k) {
                const int64_t mi = (bh * p.nblk + blk[i]) * p.D + 8 * ch8;
                s8[i] = *(const h8 *)((const _Float16 *)sc + mi);
                z8[i] = *(const h8 *)((const _Float16 *)ze + mi);
            } else {
                const int64_t mi = row * (p.D / p.Gv) + 8 * ch8 / p.Gv;
                const _Float16 s = ((const _Float16 *)sc)[mi], z = ((const _Float16 *)ze)[mi];
                s8[i] = (h8){s, s, s, s, s, s, s, s};
                z8[i] = (h8){z, z, z, z, z, z, z, z};
            }
        } else {
            const int64_t mi = row * p.lg + 8 * ch8 / p.gs;
            sf[i] = load_as_f32(sc, mi, p.meta_dt);
            zf[i] = sym ? 0.f : load_as_f32(ze, mi, p.meta_dt);
        }
    }
#pragma unroll
    for (int i = 0; i < kDqTok; ++i) {
        const int64_t t = t0 + (int64_t)i * per;
        if (t >= p.n_warm) break;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (AFFINE) {
                _Float16 x = (_Float16)(uint16_t)c[i][e] * s8[i][e];
                x = x + z8[i][e];
                v[e] = (float)x;
            } else if (sym) {
                v[e] = ((float)c[i][e] - half_max) * sf[i];
            } else {
                const float x = (float)c[i][e] * sf[i];
                v[e] = x + zf[i];
            }
        }
        if (AFFINE && p.n_out > 0) {
            const int64_t *oi = (is_k ? p.k_oidx : p.v_oidx) + ((bh / p.Hkv) * p.nblk + blk[i]) * p.n_out;
            const _Float16 *od = (const _Float16 *)(is_k ? p.k_odata : p.v_odata) + (bh * p.tok_stride + t) * p.n_out;
            for (int j = 0; j < p.n_out; ++j) {
                const int d = (int)oi[j];
                if (d / 8 != ch8) continue;
                const float x = (float)od[j];
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (d % 8 == e) v[e] = x;
            }
        }
        store_chunk<OUT>(out, orow[i] * p.D + 8 * ch8, v);
    }
}

// Vector boundaries everywhere, a chunk inside one group, 32-bit token arithmetic.
static bool dequant_chunk_eligible(const DequantParams &p) {
    const uintptr_t al = (uintptr_t)p.kc | (uintptr_t)p.vc | (uintptr_t)p.ks | (uintptr_t)p.kz | (uintptr_t)p.k_out |
                         (uintptr_t)p.v_out;
    const int g = p.kind == AKV_WARM_AFFINE ? p.Gv : p.gs;
    return (al & 15u) == 0 && p.D % 32 == 0 && p.D <= 2048 && g % 8 == 0 && p.kc_row % 8 == 0 && p.vc_row % 8 == 0 &&
           p.nbh <= 65535 && p.n_warm < ((int64_t)1 << 31);
}

// ------------------------------------------------------------------ bitpack
// One thread per (row, group of 8 codes); bytes past the packed row are not written.
__global__ __launch_bounds__(256) void bitpack_kernel(const unsigned char *codes, unsigned char *packed, int64_t rows,
                                                      int dim, int bits, int prow) {
    const int ng = (dim + 7) / 8;
    const int64_t task = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (task >= rows * ng) return;
    const int64_t r = task / ng;
    const int g = (int)(task % ng);
    uint32_t c[8];
    for (int i = 0; i < 8; ++i) {
        const int d = 8 * g + i;
        c[i] = d < dim ? codes[r * dim + d] : 0u;
    }
    unsigned char out[8];
    int nb;
    if (bits == 4) {
        for (int i = 0; i < 4; ++i) out[i] = (unsigned char)(((c[2 * i] & 15u) << 4) | (c[2 * i + 1] & 15u));
        nb = 4;
    } else if (bits == 2) {
        for (int i = 0; i < 2; ++i)
            out[i] = (unsigned char)(((c[4 * i] & 3u) << 6) | ((c[4 * i + 1] & 3u) << 4) | ((c[4 * i + 2] & 3u) << 2) | (c[4 * i + 3] & 3u));
        nb = 2;
    } else {  // 3
        uint32_t W = 0;
        for (int i = 0; i < 8; ++i) W |= (c[i] & 7u) << (21 - 3 * i);
        out[0] = (unsigned char)(W >> 16);
        out[1] = (unsigned char)(W >> 8);
        out[2] = (unsigned char)W;
        nb = 3;
    }
    const int64_t base = (int64_t)g * nb;
    for (int i = 0; i < nb; ++i)
        if (base + i < prow) packed[r * prow + base + i] = out[i];
}

__global__ __launch_bounds__(256) void bitunpack_kernel(const unsigned char *packed, unsigned char *codes, int64_t rows,
                                                        int prow, int dim, int bits) {
    const int64_t task = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (task >= rows * dim) return;
    const int64_t r = task / dim;
    const int d = (int)(task % dim);
    codes[task] = (unsigned char)extract_code(packed + r * prow, d, bits);
}

// --------------------------------------------------------------- importance
// scores[n] = scores[n]*decay + imp[n], imp[n] = sum_{m >= m0} (sum_{b,h} attn[b,h,m,n]) / (B*H);
// with pool > 1 imp is first average-pooled over keys: (1/pool) sum_{j<pool} imp[n - pool/2 + j]
// (zero outside [0, N)).  A workgroup owns 256 keys; with pooling it also sums the
// pool - 1 keys of its halo into LDS, so each attention element is read about once.
constexpr int kImpTile = 256, kImpMaxPool = 64;
__device__ __forceinline__ float key_importance(const ImportanceParams &p, int64_t n) {
    if (n < 0 || n >= p.N) return 0.f;
    const float inv_bh = (float)(p.B * p.H);
    float imp = 0.f;
    for (int64_t m = p.m0; m < p.M; ++m) {
        float acc = 0.f;
        for (int64_t bh = 0; bh < p.B * p.H; ++bh) acc += load_as_f32(p.attn, (bh * p.M + m) * p.N + n, p.attn_dt);
        imp += acc / inv_bh;
    }
    return imp;
}
__global__ __launch_bounds__(kImpTile) void importance_kernel(const ImportanceParams p) {
    __shared__ float halo[kImpTile + kImpMaxPool];
    const int64_t n0 = (int64_t)blockIdx.x * kImpTile, n = n0 + threadIdx.x;
    float imp;
    if (p.pool > 1) {
        const int pad = p.pool / 2, width = kImpTile + p.pool - 1;
        for (int i = threadIdx.x; i < width; i += kImpTile) halo[i] = key_importance(p, n0 - pad + i);
        __syncthreads();
        imp = 0.f;
        for (int j = 0; j < p.pool; ++j) imp += halo[threadIdx.x + j];
        imp = imp / (float)p.pool;
        if (n >= p.N) imp = 0.f;  // pooled output is trimmed to the N keys
    } else {
        imp = key_importance(p, n);
    }
    if (n >= p.n_scores) return;
    float s = p.scores[n] * p.decay;
    s = s + imp;
    p.scores[n] = s;
}

// Without key pooling: a workgroup owns 64 keys and its RG waves split the (batch x
// head) rows into RG contiguous ranges, 8 loads in flight per lane.  The row loads of
// a wave cover 64 consecutive keys (256 coalesced bytes at fp32).  Sum order, per
// query row m >= m0: over the rows of a range, then over the ranges in range order,
// then divided by B*H; the per-query means are then added in query order -- the
// reference's association (mean over batch and heads, then the sum over queries),
// with the (batch, head) sum itself in another order than torch's reduction (fp32
// rounding may differ in the last bits).  RG = 16 when there are too few key tiles to
// fill the GPU with RG = 4.
constexpr int kImpKeys = 64;
template <int RG>
__global__ __launch_bounds__(64 * RG) void importance_rows_kernel(const ImportanceParams p) {
    __shared__ float part[RG][kImpKeys];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t n = (int64_t)blockIdx.x * kImpKeys + lane;
    const int64_t bhn = p.B * p.H, per = (bhn + RG - 1) / RG;
    const int64_t bh0 = min(bhn, per * w), bh1 = min(bhn, bh0 + per);
    float imp = 0.f;  // wave 0: the sum over queries of the per-query means
    for (int64_t m = p.m0; m < p.M; ++m) {
        float acc = 0.f;
        if (n < p.N) {
            int64_t bh = bh0;
            for (; bh + 8 <= bh1; bh += 8) {
                float x[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) x[j] = load_as_f32(p.attn, ((bh + j) * p.M + m) * p.N + n, p.attn_dt);
#pragma unroll
                for (int j = 0; j < 8; ++j) acc += x[j];
            }
            for (; bh < bh1; ++bh) acc += load_as_f32(p.attn, (bh * p.M + m) * p.N + n, p.attn_dt);
        }
        part[w][lane] = acc;
        __syncthreads();
        if (w == 0) {
            float tot = 0.f;
#pragma unroll
            for (int r = 0; r < RG; ++r) tot += part[r][lane];
            imp += tot / (float)bhn;
        }
        __syncthreads();  // part is rewritten for the next query row
    }
    if (w != 0 || n >= p.n_scores) return;
    if (n >= p.N) imp = 0.f;
    float sc = p.scores[n] * p.decay;
    sc = sc + imp;
    p.scores[n] = sc;
}

// Many query rows (a prefill's weights): the sum over queries is split across workgroups.
// HBM-bound: B*H*M*N weights are read once and everything else is small.  A wave owns
// 64 x kV consecutive keys of every 4th query of its workgroup's range, each lane one
// 16-byte load (kV keys) per (batch, head) row, 8 rows in flight; the four waves' sums and
// one partial row per workgroup go to a workspace that importance_finish_kernel adds,
// pools and folds into the scores.  Rows of odd length put the loads off 16 bytes, which
// global loads allow; the lane across the row's end loads the row's last kV keys instead and
// keeps those that are its own.  Per query the (batch, head) rows go to two accumulators
// in turn, then the mean, then the queries in blocks: the association of
// importance_rows_kernel with the query sum split.  32 heads x 256 queries x 8,191 keys in
// bf16 (134 MB): 299 -> 26.6 us (5.0 TB/s); with 7-key pooling 4,888 -> 28.4 us.
typedef u4 u4_any __attribute__((aligned(2)));
template <int DT>
struct ImpVec {
    static constexpr int kV = DT == AKV_DT_F32 ? 4 : 8;
    static __device__ __forceinline__ void add(u4 w, float (&acc)[kV]) {
        if constexpr (DT == AKV_DT_F32) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t e = w[i];  // a copy: __builtin_bit_cast of a vector's element reads element 0
                acc[i] += __builtin_bit_cast(float, e);
            }
        } else if constexpr (DT == AKV_DT_BF16) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                acc[2 * i] += __builtin_bit_cast(float, w[i] << 16);
                acc[2 * i + 1] += __builtin_bit_cast(float, w[i] & 0xFFFF0000u);
            }
        } else {
            const h8 x = __builtin_bit_cast(h8, w);
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[i] += (float)x[i];
        }
    }
};
constexpr int kImpWaves = 4, kImpMinQueries = 20, kImpMinPooledRows = 40;
template <int DT>
__global__ __launch_bounds__(64 * kImpWaves) void importance_part_kernel(const ImportanceParams p, float *part,
                                                                         int64_t q_per) {
    constexpr int kV = ImpVec<DT>::kV, kTile = 64 * kV, kSize = DT == AKV_DT_F32 ? 4 : 2;
    __shared__ float red[kImpWaves][kTile];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t n0 = (int64_t)blockIdx.x * kTile + lane * kV, base = min(n0, p.N - kV);
    const int64_t bhn = p.B * p.H, bh_bytes = p.M * p.N * kSize;
    const int64_t q0 = p.m0 + (int64_t)blockIdx.y * q_per, q1 = min(p.M, q0 + q_per);
    float imp[kV];
#pragma unroll
    for (int i = 0; i < kV; ++i) imp[i] = 0.f;
    for (int64_t m = q0 + w; m < q1; m += kImpWaves) {
        const char *row = (const char *)p.attn + (m * p.N + base) * kSize;
        float a0[kV], a1[kV];
#pragma unroll
        for (int i = 0; i < kV; ++i) a0[i] = a1[i] = 0.f;
        int64_t bh = 0;
        for (; bh + 8 <= bhn; bh += 8) {
            u4 x[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = *(const u4_any *)(row + (bh + j) * bh_bytes);
#pragma unroll
            for (int j = 0; j < 8; j += 2) {
                ImpVec<DT>::add(x[j], a0);
                ImpVec<DT>::add(x[j + 1], a1);
            }
        }
        for (; bh < bhn; ++bh) ImpVec<DT>::add(*(const u4_any *)(row + bh * bh_bytes), a0);
#pragma unroll
        for (int i = 0; i < kV; ++i) imp[i] += (a0[i] + a1[i]) / (float)bhn;
    }
#pragma unroll
    for (int i = 0; i < kV; ++i) red[w][lane * kV + i] = imp[i];
    __syncthreads();
    // entry (lane, i) is key base + i; a key two lanes hold is written by its owner
    for (int t = threadIdx.x; t < kTile; t += 64 * kImpWaves) {
        float s = red[0][t];
#pragma unroll
        for (int r = 1; r < kImpWaves; ++r) s += red[r][t];
        const int64_t own = (int64_t)blockIdx.x * kTile + t / kV * kV;
        const int64_t n = min(own, p.N - kV) + t % kV;
        if (own < p.N && n >= own) part[(int64_t)blockIdx.y * p.N + n] = s;
    }
}
// One workgroup per 64 scores: its 4 waves add the partials of a quarter of the query blocks
// each (8 loads in flight), over the tile and the pooling halo.
__global__ __launch_bounds__(256) void importance_finish_kernel(const ImportanceParams p, const float *part, int nq) {
    __shared__ float red[4][64 + kImpMaxPool];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t n0 = (int64_t)blockIdx.x * 64;
    const int pad = p.pool / 2, width = 64 + p.pool - 1, per = (nq + 3) / 4;
    const int c0 = min(nq, per * w), c1 = min(nq, c0 + per);
    for (int i = lane; i < width; i += 64) {
        const int64_t n = n0 - pad + i;
        float s = 0.f;
        if (n >= 0 && n < p.N) {
            int c = c0;
            for (; c + 8 <= c1; c += 8) {
                float x[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) x[j] = part[(int64_t)(c + j) * p.N + n];
#pragma unroll
                for (int j = 0; j < 8; ++j) s += x[j];
            }
            for (; c < c1; ++c) s += part[(int64_t)c * p.N + n];
        }
        red[w][i] = s;
    }
    __syncthreads();
    const int64_t n = n0 + lane;
    if (w != 0 || n >= p.n_scores) return;
    float imp = 0.f;
    for (int j = 0; j < p.pool; ++j) {
        float s = red[0][lane + j];
#pragma unroll
        for (int r = 1; r < 4; ++r) s += red[r][lane + j];
        imp += s;
    }
    if (p.pool > 1) imp = imp / (float)p.pool;
    if (n >= p.N) imp = 0.f;
    float sc = p.scores[n] * p.decay;
    sc = sc + imp;
    p.scores[n] = sc;
}

// ------------------------------------------------------------ demote selection
// One workgroup (1024 threads) per row; latency-bound, so few passes over the keys.  Scores
// become order-preserving 32-bit keys (-0 as +0, NaN above +inf, protected positions =
// +inf).  Wave w owns the contiguous elements [w seg, (w + 1) seg), 64 per slot; its keys
// are read once and kept on chip: slots 0-31 in registers, slots 32-63 in LDS (128 KiB;
// 64 registers of keys spill at 1024 threads).  Rows past 65,536 re-read the row.
//   1. smallest and largest finite key, finite and +inf counts (a selection that reaches
//      past the finite keys is settled here: the keys left are +inf and NaN alone);
//   2. a histogram of 2048 equal bins over that range finds the bin of the n-th smallest --
//      bins of the range, not of the leading bits, so that scores of one magnitude spread
//      over many bins instead of colliding on a few LDS addresses, and a row of equal
//      scores needs no histogram; lanes that share the first lane's bin add once;
//   3. at most 2048 keys of that bin go to a list, on which the remaining bits are refined;
//   4. the selected indices are written in ascending order (equal keys: lowest index
//      first) from per-wave counts and ballots.
// The radix select before it made four histogram passes over 64 slots whatever the row's
// length, with one LDS address per lane: uniform scores, 1 x 140 45 -> 7.5 us, 1 x 2,049
// 46 -> 9.0, 1 x 16,383 49 -> 19.7, 16 x 65,536 67 -> 53, 1 x 131,071 371 -> 150; equal
// scores (a prompt's, all new) 1 x 16,383 87 -> 11.7 us.  The promotion's form holds more state:
// past 8,192 scores it spills (38 VGPRs at 32 slots, 50 at 64; the demotion's spills none).
namespace {
__device__ __forceinline__ uint32_t order_key(float f) {
    uint32_t u = __builtin_bit_cast(uint32_t, f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return 0xFFFFFFFFu;  // NaN sorts after +inf
    if (u == 0x80000000u) u = 0u;                             // -0 == +0
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
constexpr uint32_t kKeyInf = 0xFF800000u;  // order_key(+inf)
constexpr int kSelRegSlots = 32, kSelBins = 2048, kSelList = 2048;
// LDS words: bins, list, per-wave scratch of the reductions and scans (5 x 16), then the LDS slots
constexpr int kSelHeadWords = kSelBins + kSelList + 5 * 16;
constexpr int sel_lds_bytes(int slots) {
    return 4 * (kSelHeadWords + (slots > kSelRegSlots ? (slots - kSelRegSlots) * 1024 : 0));
}
static_assert(sel_lds_bytes(64) <= 160 * 1024, "select keys exceed the LDS");
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x, int lane) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)x, o);
        if (lane >= o) x += y;
    }
    return x;
}
__device__ __forceinline__ uint32_t lanes_below(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
}  // namespace

// What a selection takes besides the row: of a demotion the protected ends, of a promotion
// the score update, the threshold and the most rows it may take.
struct SelectParams {
    const float *scores;
    int64_t len, n, pf, pl;
    int64_t *out;
    const float *previous;  // promotion: scores before this step (or NULL)
    float *proxy;           // promotion: updated scores (or NULL: `scores` as they are)
    float decay, fresh, threshold;
};

// SLOTS 0: the row stays in memory.  PROMOTE: the keys are inverted (the largest scores are
// the smallest keys, NaN smallest), n is the smaller of p.n and the scores above the
// threshold, and out starts with that count.
template <int SLOTS, bool PROMOTE>
__global__ __launch_bounds__(1024) void select_kernel(const SelectParams p) {
    const int64_t len = p.len, n = p.n, pl = PROMOTE ? 0 : p.pl, pf = PROMOTE ? 0 : p.pf;
    extern __shared__ __align__(16) uint32_t sel_lds[];
    uint32_t *hist = sel_lds, *list = hist + kSelBins, *red = list + kSelList, *key_lds = red + 5 * 16;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const float *srow = (PROMOTE && p.proxy ? p.proxy : p.scores) + (int64_t)blockIdx.x * len;
    int64_t *orow = PROMOTE ? p.out + 1 : p.out + (int64_t)blockIdx.x * n;
    // len < 2^31: positions in 32 bits
    const uint32_t L = (uint32_t)len, rec = (uint32_t)(len - pl > 0 ? len - pl : 0);
    const uint32_t first = (uint32_t)(pf < len ? pf : len);
    const int nslot = (int)((L + 1023u) / 1024u);
    const uint32_t i0 = (uint32_t)wave * 64u * (uint32_t)nslot + (uint32_t)lane;  // slot 0 of this lane
    auto raw_at = [&](int j) { return srow[min(i0 + 64u * (uint32_t)j, L - 1u)]; };
    auto to_key = [&](int j, float x) -> uint32_t {
        const uint32_t i = i0 + 64u * (uint32_t)j;
        if (i >= L) return 0xFFFFFFFFu;
        if (PROMOTE) return ~order_key(x);
        return (i < first || i >= rec) ? kKeyInf : order_key(x);
    };
    if (PROMOTE && p.proxy) {  // a thread reads back only the scores it writes
        for (int j = 0; j < nslot; ++j) {
            const uint32_t i = i0 + 64u * (uint32_t)j;
            if (i >= L) break;
            float x = __builtin_fabsf(p.scores[i]);
            if (p.previous) {
                const float a = p.decay * p.previous[i], b = p.fresh * x;
                x = a + b;
            }
            p.proxy[i] = x;
        }
    }
    uint32_t key_reg[SLOTS > 0 ? (SLOTS < kSelRegSlots ? SLOTS : kSelRegSlots) : 1];
    // f(slot, key) over this wave's slots
    auto each = [&](auto &&f) {
        if constexpr (SLOTS > 0) {
#pragma unroll
            for (int j = 0; j < (SLOTS < kSelRegSlots ? SLOTS : kSelRegSlots); ++j)
                if (j < nslot) f(j, key_reg[j]);
            if constexpr (SLOTS > kSelRegSlots)
                for (int j = kSelRegSlots; j < nslot; j += 8) {  // 8 reads in flight
                    uint32_t k[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) k[e] = key_lds[(min(j + e, nslot - 1) - kSelRegSlots) * 1024 + tid];
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (j + e < nslot) f(j + e, k[e]);
                }
        } else {
            for (int j = 0; j < nslot; j += 8) {  // 8 loads in flight; slots past the last hold no element
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = raw_at(min(j + e, nslot - 1));
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (j + e < nslot) f(j + e, to_key(j + e, x[e]));
            }
        }
    };
    if constexpr (SLOTS > 0) {
        constexpr int kR = SLOTS < kSelRegSlots ? SLOTS : kSelRegSlots;
        float x[kR];
#pragma unroll
        for (int j = 0; j < kR; ++j) x[j] = raw_at(min(j, nslot - 1));
#pragma unroll
        for (int j = 0; j < kR; ++j) key_reg[j] = to_key(j, x[j]);
        if constexpr (SLOTS > kSelRegSlots) {
            for (int j = kSelRegSlots; j < nslot; j += 8) {
                float y[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) y[e] = raw_at(min(j + e, nslot - 1));
#pragma unroll
                for (int e = 0; e < 8; ++e)  // a thread reads only its own LDS slots: no barrier
                    if (j + e < nslot) key_lds[(j + e - kSelRegSlots) * 1024 + tid] = to_key(j + e, y[e]);
            }
        }
    }
    uint32_t kmin = 0xFFFFFFFFu, kmax = 0u, n_fin = 0u, n_inf = 0u;
    each([&](int, uint32_t k) {
        const bool fin = k < kKeyInf;
        kmin = min(kmin, k);
        kmax = max(kmax, fin ? k : 0u);
        n_fin += fin;
        n_inf += k == kKeyInf;
    });
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        kmin = min(kmin, (uint32_t)__shfl_xor((int)kmin, o));
        kmax = max(kmax, (uint32_t)__shfl_xor((int)kmax, o));
        n_fin += (uint32_t)__shfl_xor((int)n_fin, o);
        n_inf += (uint32_t)__shfl_xor((int)n_inf, o);
    }
    if (lane == 0) {
        red[wave] = kmin;
        red[16 + wave] = kmax;
        red[32 + wave] = n_fin;
        red[48 + wave] = n_inf;
    }
    __syncthreads();
    n_fin = n_inf = 0u;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
        kmin = min(kmin, red[w]);
        kmax = max(kmax, red[16 + w]);
        n_fin += red[32 + w];
        n_inf += red[48 + w];
    }
    uint32_t want = (uint32_t)n;
    const uint32_t above = PROMOTE ? ~order_key(p.threshold) : 0u;  // keys below it, NaN apart, are above the threshold
    bool skip_nan = false;
    if (PROMOTE) {
        uint32_t c = 0;
        each([&](int j, uint32_t k) {
            c += (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(k < above && k != 0u));
        });
        if (lane == 0) red[64 + wave] = c;
        __syncthreads();
        c = 0;
#pragma unroll
        for (int w = 0; w < 16; ++w) c += red[64 + w];
        __syncthreads();  // red is written again below
        skip_nan = c <= want;  // all of them; else the largest, NaN among them
        want = min(want, c);
        if (tid == 0) p.out[0] = (int64_t)want;
        if (want == 0u) return;
    }
    uint32_t tau, take_eq;  // the n-th smallest key; how many elements equal to it to take
    if (skip_nan) {
        tau = above;
        take_eq = 0u;
    } else if (want > n_fin) {
        tau = want <= n_fin + n_inf ? kKeyInf : 0xFFFFFFFFu;
        take_eq = want - n_fin - (tau == kKeyInf ? 0u : n_inf);
    } else {
        // the key of rank k among those in [lo, lo + maxd], maxd < 2^bits
        uint32_t lo = kmin, maxd = kmax - kmin, k = want, n_list = 0;
        int bits = maxd ? 32 - __builtin_clz(maxd) : 0;
        bool listed = false;
        while (bits > 0) {
            const int shift = bits > 11 ? bits - 11 : 0;
            hist[tid] = 0u;
            hist[tid + 1024] = 0u;
            __syncthreads();
            auto add = [&](uint32_t key) {
                const uint32_t d = key - lo, bin = d >> shift;
                const bool in = d <= maxd;
                const uint64_t act = __builtin_amdgcn_ballot_w64(in);
                if (!act) return;
                const int l0 = (int)__builtin_ctzll(act);
                const bool same = in && bin == (uint32_t)__builtin_amdgcn_readlane((int)bin, l0);
                const uint64_t m = __builtin_amdgcn_ballot_w64(same);
                if (in && (!same || lane == l0)) atomicAdd(&hist[bin], same ? (uint32_t)__builtin_popcountll(m) : 1u);
            };
            if (listed) {
                for (uint32_t i = 0; i < n_list; i += 1024u)
                    add(i + (uint32_t)tid < n_list ? list[i + (uint32_t)tid] : lo - 1u);
            } else {
                each([&](int, uint32_t key) { add(key); });
            }
            __syncthreads();
            const uint32_t a = hist[2 * tid], b = hist[2 * tid + 1];
            uint32_t incl = wave_incl_scan(a + b, lane);
            if (lane == 63) red[wave] = incl;
            __syncthreads();
            for (int w = 0; w < wave; ++w) incl += red[w];
            const uint32_t excl = incl - a - b;
            if (excl < k && k <= incl) {  // one thread
                const bool hi = k > excl + a;
                red[64] = 2u * (uint32_t)tid + (hi ? 1u : 0u);
                red[65] = k - excl - (hi ? a : 0u);
                red[66] = hi ? b : a;
                red[67] = 0u;  // the list's length
            }
            __syncthreads();
            const uint32_t off = red[64] << shift, cnt = red[66];
            k = red[65];
            maxd = min(maxd - off, (1u << shift) - 1u);
            lo += off;
            bits = shift;
            if (bits > 0 && !listed && cnt <= (uint32_t)kSelList) {
                each([&](int, uint32_t key) {
                    const bool in = key - lo <= maxd;
                    const uint64_t m = __builtin_amdgcn_ballot_w64(in);
                    if (!m) return;
                    uint32_t base = 0;
                    if (lane == 0) base = atomicAdd(&red[67], (uint32_t)__builtin_popcountll(m));
                    base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
                    if (in) list[base + lanes_below(m)] = key;
                });
                listed = true;
                n_list = cnt;
            }
            __syncthreads();  // the list is written; red and hist may be written again
        }
        tau = lo;
        take_eq = k;
    }
    __syncthreads();
    uint32_t lt_run = 0, eq_run = 0;  // of this wave, then before its current slot
    auto is_eq = [&](int j, uint32_t key) { return key == tau && i0 + 64u * (uint32_t)j < L; };
    auto is_lt = [&](uint32_t key) { return key < tau && !(PROMOTE && skip_nan && key == 0u); };
    each([&](int j, uint32_t key) {
        lt_run += (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(is_lt(key)));
        eq_run += (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(is_eq(j, key)));
    });
    if (lane == 0) {
        red[wave] = lt_run;
        red[16 + wave] = eq_run;
    }
    __syncthreads();
    lt_run = eq_run = 0;
    for (int w = 0; w < wave; ++w) {
        lt_run += red[w];
        eq_run += red[16 + w];
    }
    each([&](int j, uint32_t key) {
        const bool lt = is_lt(key), eq = is_eq(j, key);
        const uint64_t ml = __builtin_amdgcn_ballot_w64(lt), me = __builtin_amdgcn_ballot_w64(eq);
        const uint32_t lt_before = lt_run + lanes_below(ml), eq_before = eq_run + lanes_below(me);
        if (lt || (eq && eq_before < take_eq))
            orow[lt_before + min(eq_before, take_eq)] = (int64_t)(i0 + 64u * (uint32_t)j);
        lt_run += (uint32_t)__builtin_popcountll(ml);
        eq_run += (uint32_t)__builtin_popcountll(me);
    });
}

template <bool PROMOTE>
static hipError_t select_dispatch(const SelectParams &p, int64_t rows, hipStream_t s) {
#define AKV_SEL(slots) \
    hipLaunchKernelGGL((select_kernel<slots, PROMOTE>), dim3((unsigned)rows), dim3(1024), sel_lds_bytes(slots), s, p)
    if (p.len <= 2 * 1024) AKV_SEL(2);
    else if (p.len <= 8 * 1024) AKV_SEL(8);
    else if (p.len <= 32 * 1024) AKV_SEL(32);
    else if (p.len <= 64 * 1024) {
        // raise the dynamic LDS cap above 64 KiB once per device (a bit per device index;
        // host threads that race here both set it, which is harmless)
        static std::atomic<uint64_t> attr_devs{0};
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return e;
        const uint64_t bit = (dev >= 0 && dev < 64) ? 1ull << dev : 0ull;
        if (!bit || !(attr_devs.load(std::memory_order_acquire) & bit)) {
            e = hipFuncSetAttribute((const void *)select_kernel<64, PROMOTE>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, sel_lds_bytes(64));
            if (e != hipSuccess) return e;
            attr_devs.fetch_or(bit, std::memory_order_release);
        }
        AKV_SEL(64);
    } else AKV_SEL(0);
#undef AKV_SEL
    return hipGetLastError();
}
hipError_t select_launch(const float *scores, int64_t rows, int64_t len, int64_t n, int64_t pf, int64_t pl,
                         int64_t *out, hipStream_t s) {
    if (rows <= 0 || n <= 0) return hipSuccess;
    SelectParams p{};
    p.scores = scores; p.len = len; p.n = n; p.pf = pf; p.pl = pl; p.out = out;
    return select_dispatch<false>(p, rows, s);
}
hipError_t promote_launch(const float *scores, const float *previous, float *proxy, int64_t n, float decay, float fresh,
                          float threshold, int64_t cap, int64_t *out, hipStream_t s) {
    SelectParams p{};
    p.scores = scores; p.len = n; p.n = cap < n ? cap : n; p.out = out;
    p.previous = previous; p.proxy = proxy; p.decay = decay; p.fresh = fresh; p.threshold = threshold;
    return select_dispatch<true>(p, 1, s);
}

hipError_t dequant_launch(const DequantParams &p, hipStream_t s) {
    const int64_t tasks = (int64_t)p.nbh * p.n_warm * (p.D / 8);
    if (tasks == 0 || (!p.k_out && !p.v_out)) return hipSuccess;
    if (dequant_chunk_eligible(p)) {
        const int per = 256 / (p.D / 8) * kDqTok;
        const dim3 grid((unsigned)((p.n_warm + per - 1) / per), (unsigned)p.nbh, (p.k_out != nullptr) + (p.v_out != nullptr));
#define AKV_DQ(aff, dt) hipLaunchKernelGGL((dequant_chunk_kernel<aff, dt>), grid, dim3(256), 0, s, p)
        if (p.kind == AKV_WARM_AFFINE) {
            if (p.out_dt == AKV_DT_F16) AKV_DQ(true, AKV_DT_F16);
            else AKV_DQ(true, AKV_DT_F32);
        } else if (p.out_dt == AKV_DT_F16) AKV_DQ(false, AKV_DT_F16);
        else if (p.out_dt == AKV_DT_BF16) AKV_DQ(false, AKV_DT_BF16);
        else AKV_DQ(false, AKV_DT_F32);
#undef AKV_DQ
        return hipGetLastError();
    }
    hipLaunchKernelGGL(dequant_kernel, dim3((unsigned)((tasks + 255) / 256)), dim3(256), 0, s, p);
    return hipGetLastError();
}
hipError_t bitpack_launch(const void *codes, void *packed, int64_t rows, int dim, int bits, int prow, hipStream_t s) {
    const int64_t tasks = rows * ((dim + 7) / 8);
    if (tasks == 0) return hipSuccess;
    hipLaunchKernelGGL(bitpack_kernel, dim3((unsigned)((tasks + 255) / 256)), dim3(256), 0, s,
                       (const unsigned char *)codes, (unsigned char *)packed, rows, dim, bits, prow);
    return hipGetLastError();
}
hipError_t bitunpack_launch(const void *packed, void *codes, int64_t rows, int prow, int dim, int bits, hipStream_t s) {
    const int64_t tasks = rows * dim;
    if (tasks == 0) return hipSuccess;
    hipLaunchKernelGGL(bitunpack_kernel, dim3((unsigned)((tasks + 255) / 256)), dim3(256), 0, s,
                       (const unsigned char *)packed, (unsigned char *)codes, rows, prow, dim, bits);
    return hipGetLastError();
}
__global__ void zero_fill_kernel(u4 *p, int64_t n16) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = (u4){0u, 0u, 0u, 0u};
}
hipError_t zero_fill_launch(void *p, int64_t bytes, hipStream_t s) {
    const int64_t n16 = bytes / 16;
    if (n16 <= 0) return hipSuccess;
    const int64_t blocks = (n16 + 255) / 256;
    hipLaunchKernelGGL(zero_fill_kernel, dim3((unsigned)(blocks < 1024 ? blocks : 1024)), dim3(256), 0, s, (u4 *)p, n16);
    return hipGetLastError();
}
// Streaming read of `bytes` (a multiple of 16) in 16-byte non-temporal loads over a
// grid-stride loop, the loads XORed into a value that is stored only if it equals a
// sentinel: the bandwidth a read-once kernel of that size reaches on this GPU.
__global__ __launch_bounds__(256) void stream_read_kernel(const u4 *__restrict__ x, int64_t n16, uint32_t *sink) {
    u4 acc = {0u, 0u, 0u, 0u};
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += (int64_t)gridDim.x * blockDim.x)
        acc ^= __builtin_nontemporal_load(x + i);
    const uint32_t r = acc[0] ^ acc[1] ^ acc[2] ^ acc[3];
    if (r == 0x5A17C0DEu) sink[0] = r;
}
hipError_t stream_read_launch(const void *p, int64_t bytes, uint32_t *sink, hipStream_t s) {
    const int64_t n16 = bytes / 16;
    if (n16 <= 0) return hipSuccess;
    // 2048 workgroups of 256 threads: the fastest of 1024-8192 for 73 MB - 1 GB reads
    hipLaunchKernelGGL(stream_read_kernel, dim3(2048), dim3(256), 0, s, (const u4 *)p, n16, sink);
    return hipGetLastError();
}
// Query blocks of importance_part_kernel (0: the one-launch kernels); about four workgroups
// per compute unit, each wave at least one query.  On the device the split (5.8-7.1 us at any
// count up to 16) passes the one launch at 8 query rows without pooling (6.5-8.7 us; 11-15 at
// 16, ~0.55 a row) and at ~12 (batch, head, query) rows with it (~0.3 us a row: 10.8 us at 32,
// 20.5 at 64); but an eager call with a workspace and a second launch costs 12.2 us of host time
// against 10.6, so the lines lie where the one launch takes longer than that.  A captured call takes
// the same lines, though only the device's time counts there.
static int64_t importance_q_blocks(const ImportanceParams &p, int64_t *q_per) {
    const int64_t q = p.M - p.m0, kv = p.attn_dt == AKV_DT_F32 ? 4 : 8;
    if ((p.pool > 1 ? p.B * p.H * q < kImpMinPooledRows : q < kImpMinQueries) || p.N < kv || p.n_scores == 0) return 0;
    const int64_t tiles = (p.N + 64 * kv - 1) / (64 * kv);
    const int64_t want = max((int64_t)1, min((q + kImpWaves - 1) / kImpWaves, 1024 / tiles));
    *q_per = ((q + want - 1) / want + kImpWaves - 1) / kImpWaves * kImpWaves;
    const int64_t nq = (q + *q_per - 1) / *q_per;
    return nq <= 65535 ? nq : 0;
}
int64_t importance_workspace_bytes(const ImportanceParams &p) {
    int64_t q_per;
    return importance_q_blocks(p, &q_per) * p.N * 4;
}
hipError_t importance_launch(const ImportanceParams &p, float *part, hipStream_t s) {
    if (p.n_scores == 0) return hipSuccess;
    int64_t q_per = 0;
    const int64_t nq = part ? importance_q_blocks(p, &q_per) : 0;
    if (nq > 0) {
        const int64_t kv = p.attn_dt == AKV_DT_F32 ? 4 : 8;
        const dim3 grid((unsigned)((p.N + 64 * kv - 1) / (64 * kv)), (unsigned)nq);
#define AKV_IMP(dt) hipLaunchKernelGGL(importance_part_kernel<dt>, grid, dim3(64 * kImpWaves), 0, s, p, part, q_per)
        if (p.attn_dt == AKV_DT_F32) AKV_IMP(AKV_DT_F32);
        else if (p.attn_dt == AKV_DT_F16) AKV_IMP(AKV_DT_F16);
        else AKV_IMP(AKV_DT_BF16);
#undef AKV_IMP
        hipLaunchKernelGGL(importance_finish_kernel, dim3((unsigned)((p.n_scores + 63) / 64)), dim3(256), 0, s, p,
                           part, (int)nq);
        return hipGetLastError();
    }
    if (p.pool <= 1) {
        const unsigned tiles = (unsigned)((p.n_scores + kImpKeys - 1) / kImpKeys);
        const int64_t rows = p.B * p.H * (p.M - p.m0);
        if (tiles >= 512 || rows < 64) hipLaunchKernelGGL(importance_rows_kernel<4>, dim3(tiles), dim3(256), 0, s, p);
        else hipLaunchKernelGGL(importance_rows_kernel<16>, dim3(tiles), dim3(1024), 0, s, p);
    } else {
        hipLaunchKernelGGL(importance_kernel, dim3((unsigned)((p.n_scores + 255) / 256)), dim3(256), 0, s, p);
    }
    return hipGetLastError();
}

}  // namespace akv
