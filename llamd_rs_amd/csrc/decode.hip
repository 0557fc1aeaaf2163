// decode.hip -- the pieces of a whole-token decode step around the
// quantized matvecs: embedding row and attention over the KV cache (QK-norm,
// RoPE and the cache store are in norm.hip, beside the norms they fuse with). Each reproduces the reference CPU path's f32
// operations in its order, so a step is bit-identical to
// crates/llamd-runtime/src/layer.rs:forward (single token, single sequence).
//
// The token and position are read from device memory (not kernel
// arguments), so a step's launches do not change from token to token.
#include <algorithm>

#include "common.hpp"
#include "exact_sum.hpp"
#include "expf_ref.h"
#include "launch.hpp"
#include "q8k_wave.hpp"
#include "row_scale.hpp"

namespace llamd {
namespace {

// One row of a ggml-layout Q6_K table, dequantized as dequantize_q6_k
// (crates/llamd-quant/src/lib.rs:181-226): y = (f16(d) * sc) * (q - 32), all
// products exact in f32. get_rows of the dequantized table
// (crates/llamd-cpu/src/lib.rs:211-224). One wave per 256-value block; lane
// (half h, l) writes elements l, l+32, l+64, l+96 of half h.
// Sequence s = blockIdx.y reads its token at tok[s * tok_stride] (tok null:
// tok_fixed) and writes row s of out.
__global__ __launch_bounds__(64) void embed_q6k(const uint8_t *table, const int32_t *tok,
                                                int tok_stride, int tok_fixed, int blocks,
                                                float *out) {
    const int b = blockIdx.x, lane = threadIdx.x, sq = blockIdx.y;
    const int token = tok ? tok[(size_t)sq * tok_stride] : tok_fixed;
    out += (size_t)sq * blocks * 256;
    const uint8_t *blk = table + ((size_t)token * blocks + b) * 210;
    const int half = lane >> 5, l = lane & 31;
    const uint8_t *ql = blk + half * 64, *qh = blk + 128 + half * 32;
    const int8_t *sc = (const int8_t *)(blk + 192 + half * 8);
    const float d = f16_bits_to_f32((uint16_t)(blk[208] | (blk[209] << 8)));
    const int is = l / 16;
    const uint8_t h = qh[l], lo0 = ql[l], lo1 = ql[l + 32];
    const int q1 = ((lo0 & 0x0F) | ((h >> 0) & 3) << 4) - 32;
    const int q2 = ((lo1 & 0x0F) | ((h >> 2) & 3) << 4) - 32;
    const int q3 = ((lo0 >> 4) | ((h >> 4) & 3) << 4) - 32;
    const int q4 = ((lo1 >> 4) | ((h >> 6) & 3) << 4) - 32;
    float *y = out + (size_t)b * 256 + half * 128;
    y[l] = d * (float)sc[is] * (float)q1;
    y[l + 32] = d * (float)sc[is + 2] * (float)q2;
    y[l + 64] = d * (float)sc[is + 4] * (float)q3;
    y[l + 96] = d * (float)sc[is + 6] * (float)q4;
}

constexpr int ATT_MAX_KV = 16384;  // positions whose logits fit in LDS

// attend (crates/llamd-runtime/src/attention.rs:73-125), one workgroup per
// query head (kv head h / (n_head / n_head_kv)), n_kv = pos + 1:
//   logit_t = (sum_d q[d] k_t[d], in order from 0) * scale       one lane per t
//   max; e_t = expf(logit_t - max)                                all lanes
//   sum_t e_t in order from 0; inv = 1 / sum                      one lane
//   out[d] = sum_t (e_t * inv) v_t[d] in order from 0             one lane per d
// Sequence s = blockIdx.y: n_kv = pos_p[s * pos_stride] + 1 (pos_p null:
// n_kv_fixed), q / out row s, its cache slice at s * cache_seq_stride. An
// n_kv outside 1..ATT_MAX_KV writes NaN.
__global__ __launch_bounds__(256) void attend_decode(const float *q, const float *kc,
                                                     const float *vc, const int32_t *pos_p,
                                                     int n_head, int n_head_kv, int hd, float scale,
                                                     float *out, int n_kv_fixed, int pos_stride,
                                                     size_t cache_seq_stride) {
    __shared__ float lg[ATT_MAX_KV];
    __shared__ float qs[256];
    __shared__ float red[4];
    __shared__ uint64_t tab[32];
    const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int sq = blockIdx.y;
    const int n_kv = pos_p ? pos_p[(size_t)sq * pos_stride] + 1 : n_kv_fixed;
    q += (size_t)sq * n_head * hd;
    out += (size_t)sq * n_head * hd;
    kc += (size_t)sq * cache_seq_stride;
    vc += (size_t)sq * cache_seq_stride;
    if (n_kv < 1 || n_kv > ATT_MAX_KV) {
        for (int d = tid; d < hd; d += 256) out[h * hd + d] = __builtin_nanf("");
        return;
    }
    const int kv_dim = n_head_kv * hd, kvh = h / (n_head / n_head_kv);
    if (wave == 0) expf_ref_tab_fill(tab);
    for (int d = tid; d < hd; d += 256) qs[d] = q[h * hd + d];
    __syncthreads();
    float mx = -INFINITY;
    for (int t = tid; t < n_kv; t += 256) {
        const float *kr = kc + (size_t)t * kv_dim + kvh * hd;
        float dot = 0.0f;
        for (int d = 0; d < hd; d += 4) {
            const float4 k4 = *(const float4 *)(kr + d);
            dot = dot + qs[d] * k4.x;
            dot = dot + qs[d + 1] * k4.y;
            dot = dot + qs[d + 2] * k4.z;
            dot = dot + qs[d + 3] * k4.w;
        }
        const float l = dot * scale;
        lg[t] = l;
        mx = fmaxf(mx, l);  // f32::max fold: NaN-ignoring, order-free
    }
    mx = wave_reduce(mx, -INFINITY, [](float a, float b) { return fmaxf(a, b); });
    if (lane == 0) red[wave] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    for (int t = tid; t < n_kv; t += 256) lg[t] = expf_ref_tab(lg[t] - mx, tab);
    __syncthreads();
    if (tid == 0) {
        float sum = 0.0f;
        for (int t = 0; t < n_kv; ++t) sum = sum + lg[t];
        red[0] = __fdiv_rn(1.0f, sum);
    }
    __syncthreads();
    const float inv = red[0];
    for (int d = tid; d < hd; d += 256) {
        const float *vr = vc + (size_t)kvh * hd + d;
        float acc = 0.0f;
        int t = 0;
        for (; t + 8 <= n_kv; t += 8) {
            float vv[8];  // eight loads in flight, then the eight ordered adds
#pragma unroll
            for (int j = 0; j < 8; ++j) vv[j] = vr[(size_t)(t + j) * kv_dim];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float w = lg[t + j] * inv;
                acc = acc + w * vv[j];
            }
        }
        for (; t < n_kv; ++t) {
            const float w = lg[t] * inv;
            acc = acc + w * vr[(size_t)t * kv_dim];
        }
        out[h * hd + d] = acc;
    }
}

// Norm + RoPE of one head (hd values from src) into dst in LDS, as
// qk_norm_rope_store does: (x * scale) * w, then a*cos - b*sin and
// a*sin + b*cos on the halves. One wave; w null skips the norm.
__device__ void head_norm_rope(const float *src, const float *w, const float2 *row, int hd,
                               float eps, float *sq, float *buf, float *dst) {
    const int lane = threadIdx.x & 63, half = hd / 2;
    // every global value this wave needs, loaded before any is used (hd <= 256)
    float xv[4], wv[4];
    float2 cv[2];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int d = lane + WAVE * j;
        xv[j] = d < hd ? src[d] : 0.0f;
        wv[j] = d < hd && w ? w[d] : 1.0f;
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int i = lane + WAVE * j;
        cv[j] = i < half ? row[i] : make_float2(0.0f, 0.0f);
    }
    float scale = 1.0f;
    if (w) {
        // the sum of squares in order by lane 0 (row_scale_wave's fold)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (lane + WAVE * j < hd) sq[lane + WAVE * j] = xv[j] * xv[j];
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        if (lane == 0) {
            float sum = 0.0f;
            for (int d = 0; d < hd; d += 32) {
                float4 v[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] = *(const float4 *)(sq + d + 4 * j);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    sum = sum + v[j].x;
                    sum = sum + v[j].y;
                    sum = sum + v[j].z;
                    sum = sum + v[j].w;
                }
            }
            const float mean = __fdiv_rn(sum, (float)hd);
            scale = __fdiv_rn(1.0f, sqrt_rn(mean + eps));
        }
        scale = __shfl(scale, 0, WAVE);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int d = lane + WAVE * j;
        if (d < hd) buf[d] = w ? (xv[j] * scale) * wv[j] : xv[j];
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int i = lane + WAVE * j;
        if (i < half) {
            const float a = buf[i], b = buf[i + half];
            dst[i] = a * cv[j].x - b * cv[j].y;
            dst[i + half] = a * cv[j].y + b * cv[j].x;
        }
    }
}

// One decode step's attention block after the Q/K/V matvecs, two query
// heads (hd = 128) per workgroup -- one 256-value Q8_K block of the output:
//   1. per head: QK-norm + RoPE of Q (wave 0 of the head's 256 threads) and
//      of this position's K, plus its V (wave 1); the first query head of
//      each kv group also appends K and V to the cache. The other workgroups
//      of the group use their own copy of the same values for position pos,
//      so no workgroup waits on another.
//   2. attention exactly as attend_decode: the logits' dot products in
//      order, the max, expf_ref, the in-order sum, 1 / sum, the in-order
//      weighted V sum.
//   3. Q8_K of the workgroup's 256 outputs (quantize_q8_k bits) for the O
//      projection, and the f32 outputs if `out` is set.
// Cached K and V rows reach LDS in chunks of ATT_CHUNK positions with
// coalesced loads (all of a chunk's loads in flight at once; the first
// chunk's while the norms run): one thread per position then folds its K
// row, and one per dimension its V column, from LDS.
// Bit-identical to qk_norm_rope_store + attend_decode + q8k_quantize.
constexpr int ATT_HD = 128;
constexpr int ATT_CHUNK = 64;
constexpr int ATT_KS = ATT_HD + 4;  // padded K row in LDS (fewer bank conflicts)

// Staging of cached K or V positions [c0, c0 + ATT_CHUNK) below pos into LDS
// for the workgroup's nkv kv slots (512 threads): each thread loads its
// float4s first (ATT_PER at most), then stores them.
constexpr int ATT_PER = 2 * ATT_CHUNK * (ATT_HD / 4) / 512;
// a native vector (HIP's float4 struct copies stayed in scratch memory here)
typedef float att_f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void att_stage_load(att_f4 (&r)[ATT_PER], const float *cache, int c0,
                                               int pos, int nkv, int h0, int group, int kv_dim) {
    constexpr int C = ATT_CHUNK, D4 = ATT_HD / 4;
    const int np = min(C, pos - c0), last = np > 0 ? np - 1 : 0;
#pragma unroll
    for (int k = 0; k < ATT_PER; ++k) {
        const int i = threadIdx.x + 512 * k;  // over [slot][t][d4]
        const int sl = i / (C * D4), t = min((i / D4) % C, last), d4 = i % D4;
        // a slot past nkv reads slot 0's row again (same lines; never stored)
        const int kh = (h0 + (sl < nkv ? sl : 0)) / group;
        r[k] = *(const att_f4 *)(cache + (size_t)(c0 + t) * kv_dim + (size_t)kh * ATT_HD + 4 * d4);
    }
}

__device__ __forceinline__ void att_stage_store(const att_f4 (&r)[ATT_PER], float *dst, int stride,
                                                int c0, int pos, int nkv) {
    constexpr int C = ATT_CHUNK, D4 = ATT_HD / 4;
    const int np = min(C, pos - c0);
#pragma unroll
    for (int k = 0; k < ATT_PER; ++k) {
        const int i = threadIdx.x + 512 * k;
        const int sl = i / (C * D4), t = (i / D4) % C, d4 = i % D4;
        if (sl < nkv && t < np) *(att_f4 *)(dst + ((size_t)sl * C + t) * stride + 4 * d4) = r[k];
    }
}

// Up to two regions of a later launch's weights to read into L2 under the
// attention (n0 pieces of b0 bytes from p0, then n1 of b1 from p1).
struct AttPrefetch {
    const uint8_t *p0, *p1;
    unsigned b0, b1;
    int n0, n1;
};

__global__ __launch_bounds__(512) void attend_fused(
    const float *q_raw, const float *k_raw, const float *v_raw, const float *qw, const float *kw,
    const float2 *cs, const int32_t *pos_p, int n_head, int n_head_kv, float eps, float scale,
    int max_kv, float *kc, float *vc, int8_t *oq, float *od, float *out, AttPrefetch pf) {
    constexpr int HD = ATT_HD, C = ATT_CHUNK, KS = ATT_KS;
    if (blockIdx.x >= n_head / 2) {
        // a prefetch workgroup: one piece of a later launch's weights into
        // this XCD's L2 (piece i of a region goes to the workgroup of this
        // launch that shares XCD i % 8 with the later launch's workgroup i),
        // read and dropped; no result depends on it
        const int i = blockIdx.x - n_head / 2;
        const bool r0 = i < pf.n0;
        const uint8_t *base = r0 ? pf.p0 + (size_t)i * pf.b0 : pf.p1 + (size_t)(i - pf.n0) * pf.b1;
        const unsigned pf_bytes = r0 ? pf.b0 : pf.b1;
        const uint4 *src = (const uint4 *)base;
        const unsigned n16 = pf_bytes / 16;
        uint32_t acc = 0;
        for (unsigned i = threadIdx.x; i < n16; i += 512) {
            const uint4 q = src[i];
            acc ^= q.x ^ q.y ^ q.z ^ q.w;
        }
        if (acc == 0x9E3779B9u && pf_bytes == 1u) od[0] = 0.0f;  // never (pf_bytes % 16 == 0): keeps the loads
        return;
    }
    extern __shared__ __align__(16) float dyn[];  // lg [2][max_kv] | K [nkv][C][KS] | V [nkv][C][HD]
    __shared__ __align__(16) float qs[2][HD], kn[2][HD], vn[2][HD];
    __shared__ __align__(16) float sq[2][2][HD], buf[2][2][HD];
    __shared__ __align__(16) float ov[256];
    __shared__ float red[2][4];
    __shared__ uint64_t tab[2][32];
    const int grp = threadIdx.x >> 8, tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6;
    const int h0 = blockIdx.x * 2, h = h0 + grp, group = n_head / n_head_kv;
    const int kvh = h / group, kv_dim = n_head_kv * HD, pos = pos_p[0], n_kv = pos + 1;
    const int nkv = group >= 2 ? 1 : 2;   // distinct kv heads of the two query heads
    const int slot = nkv == 1 ? 0 : grp;  // this head's K / V staging slot
    const int lgs = (max_kv + 3) & ~3;    // logits row stride (float4-aligned)
    float *lg = dyn + (size_t)grp * lgs;
    float *kst = dyn + (size_t)2 * lgs;
    float *vst = kst + (size_t)nkv * C * KS;
    const float2 *row = cs + (size_t)pos * (HD / 2);

    att_f4 sk[ATT_PER], sv[ATT_PER];
    if (pos > 0) {
        att_stage_load(sk, kc, 0, pos, nkv, h0, group, kv_dim);
        att_stage_load(sv, vc, 0, pos, nkv, h0, group, kv_dim);
    }
    if (wave == 0) {
        head_norm_rope(q_raw + (size_t)h * HD, qw, row, HD, eps, sq[grp][0], buf[grp][0], qs[grp]);
    } else if (wave == 1) {
        const float v0 = v_raw[(size_t)kvh * HD + lane], v1 = v_raw[(size_t)kvh * HD + WAVE + lane];
        head_norm_rope(k_raw + (size_t)kvh * HD, kw, row, HD, eps, sq[grp][1], buf[grp][1], kn[grp]);
        vn[grp][lane] = v0;
        vn[grp][WAVE + lane] = v1;
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        if (h % group == 0)
            for (int d = lane; d < HD; d += WAVE) {
                kc[(size_t)pos * kv_dim + (size_t)kvh * HD + d] = kn[grp][d];
                vc[(size_t)pos * kv_dim + (size_t)kvh * HD + d] = vn[grp][d];
            }
    } else if (wave == 2) {
        expf_ref_tab_fill(tab[grp]);
    }
    if (pos > 0) {
        att_stage_store(sk, kst, KS, 0, pos, nkv);
        att_stage_store(sv, vst, HD, 0, pos, nkv);
    }
    __syncthreads();

    // logits: one thread per position, q . k in order from 0; 32 values of
    // q and of the row read from LDS per step, then their 32 ordered adds
    const auto qdot = [&](const float *kr) {
        float dot = 0.0f;
#pragma unroll
        for (int d0 = 0; d0 < HD; d0 += 32) {
            float4 k4[8], q4[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                k4[j] = *(const float4 *)(kr + d0 + 4 * j);
                q4[j] = *(const float4 *)(&qs[grp][d0 + 4 * j]);
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                dot = dot + q4[j].x * k4[j].x;
                dot = dot + q4[j].y * k4[j].y;
                dot = dot + q4[j].z * k4[j].z;
                dot = dot + q4[j].w * k4[j].w;
            }
        }
        return dot;
    };
    float mx = -INFINITY;
    for (int c0 = 0; c0 < n_kv; c0 += C) {
        if (c0 > 0) {
            // later chunks (long contexts): every thread stages, then folds
            if (c0 < pos) att_stage_load(sk, kc, c0, pos, nkv, h0, group, kv_dim);
            __syncthreads();
            if (c0 < pos) att_stage_store(sk, kst, KS, c0, pos, nkv);
            __syncthreads();
        }
        const int t = c0 + tid;
        if (tid < C && t < n_kv) {
            const float dot = t < pos ? qdot(kst + ((size_t)slot * C + tid) * KS) : qdot(kn[grp]);
            const float l = dot * scale;
            lg[t] = l;
            mx = fmaxf(mx, l);  // f32::max fold: NaN-ignoring, order-free
        }
    }
    mx = wave_reduce(mx, -INFINITY, [](float a, float b) { return fmaxf(a, b); });
    if (lane == 0) red[grp][wave] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[grp][0], red[grp][1]), fmaxf(red[grp][2], red[grp][3]));
    for (int t = tid; t < n_kv; t += 256) lg[t] = expf_ref_tab(lg[t] - mx, tab[grp]);
    __syncthreads();
    if (tid == 0) {
        float sum = 0.0f;
        int t = 0;
        for (; t + 32 <= n_kv; t += 32) {
            float4 e[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) e[j] = *(const float4 *)(lg + t + 4 * j);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                sum = sum + e[j].x;
                sum = sum + e[j].y;
                sum = sum + e[j].z;
                sum = sum + e[j].w;
            }
        }
        for (; t < n_kv; ++t) sum = sum + lg[t];
        red[grp][0] = __fdiv_rn(1.0f, sum);
    }
    __syncthreads();
    const float inv = red[grp][0];

    // the weighted V sum, one thread per dimension, in position order; the
    // first chunk was staged with K
    float acc = 0.0f;
    for (int c0 = 0; c0 < pos; c0 += C) {
        if (c0 > 0) {
            att_stage_load(sv, vc, c0, pos, nkv, h0, group, kv_dim);
            __syncthreads();
            att_stage_store(sv, vst, HD, c0, pos, nkv);
            __syncthreads();
        }
        if (tid < HD) {
            const int np = min(C, pos - c0);
            const float *vr = vst + (size_t)slot * C * HD + tid;
            int t = 0;
            for (; t + 8 <= np; t += 8) {
                // the 8 values and their 8 weights read together, then the
                // ordered adds (lg + c0 + t is 16-byte aligned)
                float vv[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) vv[j] = vr[(size_t)(t + j) * HD];
                const float4 l0 = *(const float4 *)(lg + c0 + t), l1 = *(const float4 *)(lg + c0 + t + 4);
                const float ll[8] = {l0.x, l0.y, l0.z, l0.w, l1.x, l1.y, l1.z, l1.w};
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float w = ll[j] * inv;
                    acc = acc + w * vv[j];
                }
            }
            for (; t < np; ++t) {
                const float w = lg[c0 + t] * inv;
                acc = acc + w * vr[(size_t)t * HD];
            }
        }
    }
    if (tid < HD) {
        const float w = lg[pos] * inv;
        acc = acc + w * vn[grp][tid];
        ov[grp * HD + tid] = acc;
        if (out) out[(size_t)h * HD + tid] = acc;
    }
    __syncthreads();
    if (threadIdx.x < WAVE) {
        const float4 v4 = *(const float4 *)(ov + 4 * lane);
        const float v[4] = {v4.x, v4.y, v4.z, v4.w};
        quantize_wave(v, lane, oq + (size_t)blockIdx.x * QK_K, od + blockIdx.x, nullptr);
    }
}

// ---- attention split over the GPU -------------------------------------------
// attend_fused and attend_decode give a head one workgroup that walks its
// positions, so their cost grows by 50-70 ns per position. Here the same
// arithmetic runs in one or two launches, for any number of sequences (Q
// normed and rotated and K, V already in the cache):
//  - attend_scores (past a.fuse positions): a workgroup takes 64 positions of
//    one kv head, one wave per query head of its group, one lane per position.
//    The K rows are staged in LDS once for the group; the wave's q comes
//    through the scalar cache into SGPRs, so the in-order 128-term dot reads
//    LDS once per four terms.
//  - attend_mix: a workgroup per head and slice of DS dimensions: the logits
//    (read, or formed from K rows staged in LDS), their max (order free), e_t =
//    expf(logit_t - max), the in-order sum of e_t (one lane, or past
//    ATT_SERIAL terms exact_sum_nonneg: the reference's bits from a
//    workgroup-wide certificate), w_t = e_t * (1 / sum), then out[d] =
//    sum_t w_t * v_t[d] in position order.
// The last sum is one dependent chain of n_kv adds per output and bounds the
// kernel. So the folding waves (one lane per dimension) do nothing but read
// four products and add them: other waves load V a few chunks ahead, multiply
// by the weights and hand chunks of products over in LDS, transposed so that a
// lane's four next products are one read. What is left is the chain itself, 3.6
// ns per position, and 1-1.5 ns of waiting for the products; a barrier per
// 32 positions instead of 128 (64 for all 128 dimensions in one workgroup) costs
// another 2-4 ns. The last chunk ends with its last 32 positions (one sequence of
// 20: 8.1, 7.5 us a call; of 150 11.9, 11.0).
// The same operations in the same order as attend_decode (and the reference,
// attention.rs:73-125): the same bits.
constexpr int AS_POS = 64;          // positions per block of attend_scores
constexpr int AS_MAX_GROUP = 16;    // query heads per kv head
constexpr int ATT_SERIAL = 320;     // e_t that one lane adds
constexpr int ATT_FEW = 56;         // positions that one wave takes (att_few)

typedef const __attribute__((address_space(4))) float *att_cptr;

struct AttArgs {
    const float *q, *kc, *vc;
    const int32_t *pos_p;     // n_kv = pos_p[s * pos_stride] + 1 (null: n_kv_fixed)
    float *scores;            // [nseq][n_head][cap]
    float *out;               // [nseq][n_head * HD]
    size_t seq_stride;        // floats between two sequences' caches
    int pos_stride, n_kv_fixed, n_head, n_head_kv, cap, fuse, grid_y;
    float scale;
};

__device__ __forceinline__ int att_n_kv(const AttArgs &a, int s) {
    return a.pos_p ? a.pos_p[(size_t)s * a.pos_stride] + 1 : a.n_kv_fixed;
}

// One word of each of q's 64-byte lines, so that the scalar cache holds them
// when the dot products read the rest.
template <int HD>
__device__ __forceinline__ void att_touch(att_cptr q) {
#pragma unroll
    for (int d = 0; d < HD; d += 16) asm volatile("" ::"s"(q[d]));
}

template <int HD>
__global__ __launch_bounds__(64 * AS_MAX_GROUP) void attend_scores(AttArgs a) {
    constexpr int KS = HD + 4;  // padded row: conflict-free 16-byte reads
    __shared__ __align__(16) float ks[AS_POS * KS];
    const int group = a.n_head / a.n_head_kv, nt = 64 * group;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = blockIdx.x % a.n_head_kv, s = blockIdx.x / a.n_head_kv;
    const int n_kv = att_n_kv(a, s), kv_dim = a.n_head_kv * HD;
    if (n_kv <= a.fuse || n_kv > a.cap) return;
    const int head = s * a.n_head + g * group + wave;
    const att_cptr q = (att_cptr)(a.q + (size_t)head * HD);
    const float *kc = a.kc + (size_t)s * a.seq_stride + (size_t)g * HD;
    for (int t0 = blockIdx.y * AS_POS; t0 < n_kv; t0 += a.grid_y * AS_POS) {
        const int np = min(AS_POS, n_kv - t0);
        __syncthreads();  // the previous block's rows are read
        for (int i0 = tid; i0 < np * (HD / 4); i0 += 4 * nt) {
            att_f4 r[4];  // four loads in flight; those past the block re-read its last row
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int i = i0 + k * nt, t = min(i / (HD / 4), np - 1);
                r[k] = *(const att_f4 *)(kc + (size_t)(t0 + t) * kv_dim + 4 * (i % (HD / 4)));
            }
            if (t0 == (int)blockIdx.y * AS_POS && i0 == tid) att_touch<HD>(q);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int i = i0 + k * nt, t = i / (HD / 4);
                if (t < np) *(att_f4 *)(ks + t * KS + 4 * (i % (HD / 4))) = r[k];
            }
        }
        __syncthreads();
        const float *kr = ks + lane * KS;
        float dot = 0.0f;
#pragma unroll
        for (int d0 = 0; d0 < HD; d0 += 16) {
            att_f4 k4[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) k4[j] = *(const att_f4 *)(kr + d0 + 4 * j);
#pragma unroll
            for (int j = 0; j < 16; ++j) dot = dot + q[d0 + j] * k4[j / 4][j % 4];
        }
        if (lane < np) a.scores[(size_t)head * a.cap + t0 + lane] = dot * a.scale;
    }
}

// The logit of one position for one head, q through the scalar cache.
template <int HD>
__device__ __forceinline__ float att_logit(const float *qp, const float *kr, float scale) {
    att_cptr q = (att_cptr)qp;
    asm volatile("" : "+s"(q));  // read again for each position: 128 registers otherwise
    float dot = 0.0f;
#pragma unroll
    for (int d0 = 0; d0 < HD; d0 += 32) {
        att_f4 k4[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) k4[j] = *(const att_f4 *)(kr + d0 + 4 * j);
#pragma unroll
        for (int j = 0; j < 32; ++j) dot = dot + q[d0 + j] * k4[j / 4][j % 4];
    }
    return dot * scale;
}

// in-order sum of lg[0..n) from 0 by the workgroup, in pieces of what
// exact_sum_nonneg takes: the running sum is the next piece's first term
template <int NT>
__device__ __forceinline__ float att_sum(const float *lg, int n, ExactSumLds &xl) {
    constexpr int MOST = NT * XSUM_M < XSUM_MAX_N ? NT * XSUM_M : XSUM_MAX_N;
    float sum = 0.0f;
    for (int base = 0; base < n;) {
        const bool cont = base > 0;
        const int cnt = min(MOST, n - base + (cont ? 1 : 0));
        const float first = sum;
        const float *e = lg + base - (cont ? 1 : 0);
        const int m = xsum_run(cnt, NT), j0 = threadIdx.x * m;
        float v[XSUM_M];
#pragma unroll
        for (int k = 0; k < XSUM_M; ++k) {
            const int j = j0 + k;
            v[k] = (k < m && j < cnt) ? (cont && j == 0 ? first : e[j]) : 0.0f;
        }
        sum = exact_sum_nonneg(v, cnt, NT, xl, [e, cont, first](int j) { return cont && j == 0 ? first : e[j]; });
        base += cnt - (cont ? 1 : 0);
    }
    return sum;
}

// (n_kv past cap: a batched caller's position beyond its slice.) attend_decode's
// sequence with the logits formed again, cap positions at a time.
template <int HD, int DS, int NT>
__device__ __forceinline__ void att_beyond_cap(const AttArgs &a, const float *q, const float *kc, const float *vc,
                               int kv_dim, int n_kv, float *lg, float *red, const uint64_t *tab,
                               float *out) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float mx = -INFINITY;
    for (int t = tid; t < n_kv; t += NT)
        mx = fmaxf(mx, att_logit<HD>(q, kc + (size_t)t * kv_dim, a.scale));
    mx = wave_reduce(mx, -INFINITY, [](float x, float y) { return fmaxf(x, y); });
    if (lane == 0) red[wave] = mx;
    __syncthreads();
    for (int w = 0; w < NT / 64; ++w) mx = fmaxf(mx, red[w]);
    float sum = 0.0f, inv = 0.0f, acc = 0.0f;
    for (int pass = 0; pass < 2; ++pass) {
        for (int c0 = 0; c0 < n_kv; c0 += a.cap) {
            const int np = min(a.cap, n_kv - c0);
            __syncthreads();
            for (int t = tid; t < np; t += NT)
                lg[t] = expf_ref_tab(att_logit<HD>(q, kc + (size_t)(c0 + t) * kv_dim, a.scale) - mx, tab);
            __syncthreads();
            if (pass == 0) {
                if (tid == 0)
                    for (int t = 0; t < np; ++t) sum = sum + lg[t];
            } else if (tid < DS) {
                for (int t = 0; t < np; ++t) {
                    const float w = lg[t] * inv;
                    acc = acc + w * vc[(size_t)(c0 + t) * kv_dim + tid];
                }
            }
        }
        if (pass == 0) {
            if (tid == 0) red[0] = __fdiv_rn(1.0f, sum);
            __syncthreads();
            inv = red[0];
        }
    }
    if (tid < DS) out[tid] = acc;
}

// e_t summed in order from 0 by one lane, 32 read per step. The e_t up to the
// next multiple of 32 are +0.0, which leaves the sum as it is (it is never
// -0.0), so the last step needs no terms one by one (20 terms: 0.4 us less).
__device__ __forceinline__ float att_sum_serial(const float *lg, int n) {
    float sum = 0.0f;
    int t = 0;
    for (; t + 32 <= n; t += 32) {
        att_f4 e[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) e[j] = *(const att_f4 *)(lg + t + 4 * j);
#pragma unroll
        for (int j = 0; j < 32; ++j) sum = sum + e[j / 4][j % 4];
    }
    if (t < n) {
        att_f4 e[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) e[j] = *(const att_f4 *)(lg + t + 4 * j);
#pragma unroll
        for (int j = 0; j < 32; ++j) {
            if (j && j % 8 == 0 && t + j >= n) break;
            sum = sum + e[j / 4][j % 4];
        }
    }
    return sum;
}

// A sequence of up to ATT_FEW positions, without chunks: wave 0 takes a position
// a lane; the DS / 64 waves after it, which fold, have the V rows in flight
// meanwhile. (us a call, with chunks and without, 32 query / 4 kv heads: one
// sequence of 1 position 5.3, 4.0; of 20 5.5, 4.2; of 48 5.7, 4.8; 32 of 20 13.7,
// 9.3. From about 56 on a wave that reads the K rows by itself is behind: 16 of 64
// 6.8, 7.4.)
template <int HD, int DS>
__device__ __forceinline__ void att_few(const float *q, const float *kc, const float *vc, int kv_dim,
                                        int n_kv, float scale, float *lg, const uint64_t *tab, float *out) {
    constexpr int A = 8;
    static_assert(ATT_FEW <= 64 && ATT_FEW % A == 0, "a lane per position");
    const int lane = threadIdx.x & 63, d = (int)threadIdx.x - 64;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const bool folds = wave > 0 && wave <= DS / 64;
    float v[ATT_FEW], l = -INFINITY, mx = 0.0f;
    if (folds) {
#pragma unroll
        for (int t0 = 0; t0 < ATT_FEW; t0 += A)
            if (t0 < n_kv)  // (rows past the last re-read it, unused)
#pragma unroll
                for (int t = t0; t < t0 + A; ++t) v[t] = vc[(size_t)min(t, n_kv - 1) * kv_dim + d];
    } else if (wave == 0) {
        l = att_logit<HD>(q, kc + (size_t)min(lane, n_kv - 1) * kv_dim, scale);
        // f32::max fold: NaN ignoring, order free (the last row taken again changes nothing)
        mx = wave_reduce(l, -INFINITY, [](float x, float y) { return fmaxf(x, y); });
    }
    __syncthreads();  // tab
    if (wave == 0) {
        const float e = expf_ref_tab(l - mx, tab);
        float sum = 0.0f;
        for (int t = 0; t < n_kv; ++t)
            sum = sum + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(e), t));
        lg[lane] = e * __fdiv_rn(1.0f, sum);
    }
    __syncthreads();
    if (!folds) return;
    float acc = 0.0f;
#pragma unroll
    for (int t0 = 0; t0 < ATT_FEW; t0 += A)
        if (t0 < n_kv)
#pragma unroll
            for (int t = t0; t < t0 + A; ++t) {
                const float w = lg[t] * v[t];
                acc = t < n_kv ? acc + w : acc;
            }
    out[d] = acc;
}

// The logits of every position into lg, from K rows staged 64 * TILES at a
// time in `ks` (16-byte units of row t at unit u ^ t: conflict-free reads of one
// unit by 64 rows); returns this thread's share of their max.
template <int HD, int NT, int TILES>
__device__ __forceinline__ float att_logits_here(const float *q, const float *kc, int kv_dim, int n_kv,
                                                 float scale, float *lg, float *ks) {
    constexpr int U = HD / 4, ROWS = 64 * TILES, PER = (ROWS * U + NT - 1) / NT;
    const int tid = threadIdx.x;
    float mx = -INFINITY;
    for (int t0 = 0; t0 < n_kv; t0 += ROWS) {
        const int last = min(ROWS, n_kv - t0) - 1;
        if (t0) __syncthreads();  // the previous rows are read
        att_f4 r[PER];
        // loads at clamped rows (all in flight together)
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            if (NT * k > last * U + U - 1) break;
            const int i = tid + NT * k, t = min(i / U, last);
            r[k] = *(const att_f4 *)(kc + (size_t)(t0 + t) * kv_dim + 4 * (i % U));
        }
        if (t0 == 0) att_touch<HD>((att_cptr)q);
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            if (NT * k > last * U + U - 1) break;
            const int i = tid + NT * k, t = i / U;
            if (t <= last) *(att_f4 *)(ks + 4 * (t * U + ((i % U) ^ (t % U)))) = r[k];
        }
        __syncthreads();
        if (tid < ROWS) {
            att_cptr qc = (att_cptr)q;
            float dot = 0.0f;
#pragma unroll
            for (int u0 = 0; u0 < U; u0 += 8) {
                att_f4 k4[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) k4[j] = *(const att_f4 *)(ks + 4 * (tid * U + ((u0 + j) ^ (tid % U))));
#pragma unroll
                for (int j = 0; j < 32; ++j) dot = dot + qc[4 * u0 + j] * k4[j / 4][j % 4];
            }
            if (tid <= last) {
                const float l = dot * scale;
                lg[t0 + tid] = l;
                mx = fmaxf(mx, l);
            }
        }
    }
    return mx;
}

// WIDE: a CU to a workgroup: wave 0 folds and the producers are on the other
// three SIMDs (wave % 4 != 0), so nothing competes with the chain for its
// SIMD. Else DS / 64 folding waves, then the producers, several workgroups to
// a CU.
template <int DS, int NP, bool WIDE>
constexpr int am_threads = WIDE ? 64 * (1 + (NP + 2) / 3 * 3 + (NP - 1) / 3) : DS + 64 * NP;
// Positions per chunk: one 4 x 4 piece of products per producer thread, or two
// where several workgroups share the CU (a barrier and a hand-over per 128
// positions of 64 dimensions or 64 of 128, instead of half).
template <int DS, int NP, bool WIDE>
constexpr int am_chunk = (WIDE ? 1 : 2) * 1024 * NP / DS;

// ONE: forms the logits of any number of positions; else attend_scores has formed
// those of more than a.fuse.
template <int HD, int DS, int NP, bool WIDE, int TILES, bool ONE>
__global__ __launch_bounds__((am_threads<DS, NP, WIDE>)) void attend_mix(AttArgs a) {
    constexpr int NF = DS / 64, NT = am_threads<DS, NP, WIDE>, NW = NT / 64;
    constexpr int CH = am_chunk<DS, NP, WIDE>, HALF = CH / 2, D4 = DS / 4;
    static_assert(!WIDE || NF == 1, "the wide form folds on one wave");
    static_assert(NW <= 16 && CH % 32 == 0, "the workgroup's size, whole reads of a chunk");
    // weights [cap, rounded up to 128], then 2 chunks of products or 64 * TILES K rows
    extern __shared__ __align__(16) float dyn[];
    __shared__ ExactSumLds xl;
    __shared__ uint64_t tab[32];
    __shared__ float red[16];
    __shared__ float inv1;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // a kv head's heads and slices on every n_head_kv-th workgroup, so that
    // the XCD they share reads that kv head's V only
    constexpr int SL = HD / DS;
    const int g = blockIdx.x % a.n_head_kv, r = blockIdx.x / a.n_head_kv;
    const int h = g * (a.n_head / a.n_head_kv) + r / SL, sd = (r % SL) * DS, s = blockIdx.y;
    const int kv_dim = a.n_head_kv * HD;
    int n_kv = att_n_kv(a, s);
    const float *q = a.q + ((size_t)s * a.n_head + h) * HD;
    const float *kc = a.kc + (size_t)s * a.seq_stride + (size_t)g * HD;
    const float *vc = a.vc + (size_t)s * a.seq_stride + (size_t)g * HD + sd;
    float *out = a.out + ((size_t)s * a.n_head + h) * HD + sd;
    if (n_kv < 1 || n_kv > ATT_MAX_KV) {
        if (tid < DS) out[tid] = __builtin_nanf("");
        return;
    }
    float *lg = dyn, *buf = dyn + (a.cap + 127) / 128 * 128;
    if (wave == NW - 1) expf_ref_tab_fill(tab);
    if (n_kv > a.cap) {
        __syncthreads();
        att_beyond_cap<HD, DS, NT>(a, q, kc, vc, kv_dim, n_kv, lg, red, tab, out);
        return;
    }
    if (n_kv <= ATT_FEW) {
        att_few<HD, DS>(q, kc, vc, kv_dim, n_kv, a.scale, lg, tab, out);
        return;
    }
    // (the loops of this form fold slower where the compiler knows n_kv > ATT_FEW:
    // 13 sequences of 1000 30.2 us, 28.0)
    if constexpr (!WIDE && !ONE) asm volatile("" : "+s"(n_kv));
    const int nc = (n_kv + CH - 1) / CH;
    // a producer thread's piece of a chunk: positions 4 t4 .. 4 t4 + 3, dimensions
    // 4 d4 .. 4 d4 + 3
    const int pw = WIDE ? (wave >> 2) * 3 + (wave & 3) - 1 : wave - NF;
    const bool folds = WIDE ? wave == 0 : wave < NF;
    const bool produces = WIDE ? (wave & 3) != 0 && pw < NP : !folds;
    const int piece = pw * 64 + lane, t4 = piece / D4, d4 = piece % D4;
    att_f4 va[4], vb[4];
    const float *vp = vc + 4 * d4;
    const auto vload = [&](att_f4 (&v)[4], int t0) {  // from position t0 + 4 t4
        const int t = t0 + 4 * t4;
        if (t0 + CH <= n_kv) {
            const float *p = vp + (size_t)t * kv_dim;
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = *(const att_f4 *)(p + (size_t)i * kv_dim);
        } else {  // rows past the last re-read it, unused
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = *(const att_f4 *)(vp + (size_t)min(t + i, n_kv - 1) * kv_dim);
        }
    };
    // the two register sets: both halves of a chunk, or two chunks
    constexpr int STEP = WIDE ? CH : HALF;
    if (produces) {
        vload(va, 0);
        if (!WIDE || nc > 1) vload(vb, STEP);
    }
    // the logits and their max (f32::max fold: NaN ignoring, order free)
    float mx = -INFINITY;
    if (ONE || n_kv <= a.fuse) {
        mx = att_logits_here<HD, NT, TILES>(q, kc, kv_dim, n_kv, a.scale, lg, buf);
    } else {
        const float *sc = a.scores + ((size_t)s * a.n_head + h) * a.cap;
        for (int t = tid; t < n_kv; t += NT) {
            const float l = sc[t];
            lg[t] = l;
            mx = fmaxf(mx, l);
        }
    }
    mx = wave_reduce(mx, -INFINITY, [](float x, float y) { return fmaxf(x, y); });
    if (lane == 0) red[wave] = mx;
    __syncthreads();
    mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) mx = fmaxf(mx, red[w]);
    for (int t = tid; t < n_kv; t += NT) lg[t] = expf_ref_tab(lg[t] - mx, tab);
    if (tid >= n_kv % 32 && tid < 32 && n_kv % 32) lg[n_kv / 32 * 32 + tid] = 0.0f;  // (att_sum_serial)
    __syncthreads();
    if (n_kv <= ATT_SERIAL) {
        if (tid == 0) inv1 = __fdiv_rn(1.0f, att_sum_serial(lg, n_kv));
    } else {
        const float sum = att_sum<NT>(lg, n_kv, xl);
        if (tid == 0) inv1 = __fdiv_rn(1.0f, sum);
    }
    __syncthreads();
    const float inv = inv1;

    // products of chunk c into its buffer; positions past the last add +0.0,
    // which leaves every sum as it is (a sum from +0.0 is never -0.0)
    const auto produce = [&](const att_f4 (&v)[4], int c, int half) {
        const int t0 = c * CH + half * HALF, t = t0 + 4 * t4;
        const att_f4 e = *(const att_f4 *)(lg + t);
        att_f4 p[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float w = e[i] * inv;
#pragma unroll
            for (int j = 0; j < 4; ++j) p[j][i] = w * v[i][j];
        }
        if (t0 + CH > n_kv) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) p[j][i] = t + i < n_kv ? p[j][i] : 0.0f;
        }
        // dimension 4 d4 + j in slot j * D4 + d4: a wave's stores are contiguous
        float *dst = buf + (c & 1) * (CH * DS) + half * (HALF * DS) + t4 * DS * 4 + d4 * 4;
#pragma unroll
        for (int j = 0; j < 4; ++j) *(att_f4 *)(dst + j * D4 * 4) = p[j];
    };
    // Chunk c is folded between barriers c and c + 1, while chunk c + 1 goes
    // into the other buffer. The folding and the producing waves have loops of
    // their own (a shared loop's register merges would wait for the loads in
    // flight).
    if (folds) {
        __builtin_amdgcn_s_setprio(3);
        float acc = 0.0f;
        // 32 products ahead of the 32 being added
        att_f4 p[2][8];
        const auto read = [&](const float *src, int k) {
#pragma unroll
            for (int i = 0; i < 8; ++i) p[k & 1][i] = *(const att_f4 *)(src + (8 * k + i) * DS * 4);
            __builtin_amdgcn_sched_barrier(0);
        };
        const auto add = [&](int k) {
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc = acc + p[k & 1][i][e];
        };
        // the last chunk ends with its last 32 positions; zeros follow
        const int left = n_kv - (nc - 1) * CH, full = left > CH - 32 ? nc : nc - 1;
        for (int c = 0; c < full; ++c) {
            __syncthreads();
            const float *src = buf + (c & 1) * (CH * DS) + tid * 4;
            read(src, 0);
#pragma unroll
            for (int k = 0; k < CH / 32; ++k) {
                if (k + 1 < CH / 32) read(src, k + 1);
                add(k);
            }
        }
        if (full < nc) {
            __syncthreads();
            const float *src = buf + (full & 1) * (CH * DS) + tid * 4;
#pragma unroll 1
            for (int t = 0; t < left; t += 32, src += 32 * DS) {
                read(src, 0);
                add(0);
            }
        }
        out[(tid % D4) * 4 + tid / D4] = acc;
    } else if (produces) {
        if constexpr (WIDE) {
            produce(va, 0, 0);
            if (nc > 2) vload(va, 2 * CH);
            for (int c = 0; c < nc; c += 2) {
                __syncthreads();
                if (c + 1 >= nc) break;
                produce(vb, c + 1, 0);
                if (c + 3 < nc) vload(vb, (c + 3) * CH);
                __syncthreads();
                if (c + 2 >= nc) break;
                produce(va, c + 2, 0);
                if (c + 4 < nc) vload(va, (c + 4) * CH);
            }
        } else {
            for (int c = 0; c < nc; ++c) {
                if (c) __syncthreads();
                produce(va, c, 0);
                if (c + 1 < nc) vload(va, (c + 1) * CH);
                produce(vb, c, 1);
                if (c + 1 < nc) vload(vb, (c + 1) * CH + HALF);
            }
            __syncthreads();
        }
    } else {
        for (int c = 0; c < nc; ++c) __syncthreads();
    }
}

}  // namespace

int launch_embed_q6k(const void *table, const int32_t *tok, int blocks, float *out, hipStream_t st,
                     int nseq, int tok_stride, int tok_fixed) {
    if (blocks <= 0 || nseq <= 0) return -1;
    hipLaunchKernelGGL(embed_q6k, dim3(blocks, nseq), dim3(64), 0, st, (const uint8_t *)table, tok,
                       tok_stride, tok_fixed, blocks, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int attend_max_kv() { return ATT_MAX_KV; }

namespace {
size_t g_fused_lds = 0;  // the dynamic LDS attend_fused may use (raised by prepare)
}

namespace {
size_t fused_lds(int n_head, int n_head_kv, int max_kv) {
    const int nkv = n_head / n_head_kv >= 2 ? 1 : 2;
    return (size_t)2 * ((max_kv + 3) & ~3) * 4 + (size_t)nkv * ATT_CHUNK * (ATT_KS + ATT_HD) * 4;
}
}  // namespace

bool attend_fused_fits(int n_head, int n_head_kv, int hd, int max_kv) {
    if (hd != ATT_HD || n_head_kv <= 0 || n_head % n_head_kv || n_head % 2 || max_kv <= 0) return false;
    return fused_lds(n_head, n_head_kv, max_kv) + 24 * 1024 <= 160 * 1024;
}

int attend_fused_prepare(int n_head, int n_head_kv, int hd, int max_kv) {
    if (!attend_fused_fits(n_head, n_head_kv, hd, max_kv)) return -1;
    const size_t lds = fused_lds(n_head, n_head_kv, max_kv);
    if (lds <= g_fused_lds) return 0;
    if (hipFuncSetAttribute((const void *)attend_fused, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)lds) != hipSuccess)
        return -1;
    g_fused_lds = lds;
    return 0;
}

int launch_attend_fused(const float *q, const float *k, const float *v, const float *qw,
                        const float *kw, const float2 *cs, const int32_t *pos, int n_head,
                        int n_head_kv, int hd, float eps, float scale, int max_kv, float *kc,
                        float *vc, int8_t *oq, float *od, float *out, hipStream_t st,
                        const void *pf0, size_t b0, int n0, const void *pf1, size_t b1, int n1) {
    if (!attend_fused_fits(n_head, n_head_kv, hd, max_kv)) return -1;
    const size_t lds = fused_lds(n_head, n_head_kv, max_kv);
    if (lds > g_fused_lds) return -1;  // attend_fused_prepare first
    // the pieces of region 1 start on XCD 0 again: region 0 is padded to a
    // multiple of 8 workgroups
    AttPrefetch pf{(const uint8_t *)pf0, (const uint8_t *)pf1, (unsigned)b0, (unsigned)b1, n0, n1};
    if (!pf0 || b0 % 16 || b0 > (1u << 30) || n0 < 0 || (n_head / 2) % 8) pf.n0 = 0;
    if (!pf1 || b1 % 16 || b1 > (1u << 30) || n1 < 0 || pf.n0 % 8 || (n_head / 2) % 8) pf.n1 = 0;
    hipLaunchKernelGGL(attend_fused, dim3(n_head / 2 + pf.n0 + pf.n1), dim3(512), lds, st, q, k, v,
                       qw, kw, cs, pos, n_head, n_head_kv, eps, scale, max_kv, kc, vc, oq, od, out,
                       pf);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

namespace {
size_t split_lds(int cap, int hd, int ds, int chunk, int tiles) {
    return (size_t)(cap + 127) / 128 * 128 * 4 + std::max(2 * chunk * ds * 4, tiles * 64 * hd * 4);
}

template <int HD, int DS, int NP, bool WIDE, int TILES, bool ONE = false>
int launch_mix(const AttArgs &a, int nseq, hipStream_t st) {
    constexpr int CH = am_chunk<DS, NP, WIDE>;
    // the largest cache's dynamic LDS, allowed once per kernel
    static const hipError_t ok = hipFuncSetAttribute((const void *)attend_mix<HD, DS, NP, WIDE, TILES, ONE>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize,
                                                     (int)split_lds(ATT_MAX_KV, HD, DS, CH, TILES));
    if (ok != hipSuccess) return -1;
    hipLaunchKernelGGL((attend_mix<HD, DS, NP, WIDE, TILES, ONE>), dim3(a.n_head * (HD / DS), nseq),
                       dim3(am_threads<DS, NP, WIDE>), split_lds(a.cap, HD, DS, CH, TILES), st, a);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
}  // namespace

bool attend_split_fits(int n_head, int n_head_kv, int hd, int max_kv) {
    return (hd == 64 || hd == 128) && n_head_kv > 0 && n_head_kv <= 65535 && n_head > 0 &&
           n_head % n_head_kv == 0 && n_head / n_head_kv <= AS_MAX_GROUP && max_kv > 0 &&
           max_kv <= ATT_MAX_KV;
}

namespace {
// The most positions that the one-launch form is chosen for (launch_attend_split).
constexpr int ATT_ONE_LAUNCH = 256;
int split_expect(int cap, int expect) { return expect <= 0 || expect > cap ? cap : expect; }
}  // namespace

size_t attend_split_scores(int n_head, int cap, int nseq, int expect) {
    return split_expect(cap, expect) <= ATT_ONE_LAUNCH ? 0 : (size_t)nseq * n_head * cap;
}

int launch_attend_split(const float *q, const float *kc, const float *vc, const int32_t *pos,
                        int n_head, int n_head_kv, int hd, float scale, int cap, float *scores,
                        float *out, hipStream_t st, int nseq, int n_kv_fixed, int pos_stride,
                        size_t cache_seq_stride, int expect) {
    if (!attend_split_fits(n_head, n_head_kv, hd, cap) || nseq <= 0 || nseq > 65535) return -1;
    expect = split_expect(cap, expect);
    if (!scores && expect > ATT_ONE_LAUNCH) return -1;
    AttArgs a{};
    a.q = q;
    a.kc = kc;
    a.vc = vc;
    a.pos_p = pos;
    a.scores = scores;
    a.out = out;
    a.seq_stride = cache_seq_stride;
    a.pos_stride = pos_stride;
    a.n_kv_fixed = n_kv_fixed;
    a.n_head = n_head;
    a.n_head_kv = n_head_kv;
    a.cap = cap;
    a.scale = scale;
    const int heads = nseq * n_head;
    // us per call with the Q8_K behind it, 32 query / 4 kv heads of 128
    // (attend_decode alone, then this): 1 sequence of 250 positions 15.2, 13.2;
    // 1000: 49, 16.8; 4100: 278, 34.5; 8192: 544, 56; 13 of up to 1000: 88, 29;
    // 16 of up to 2000: 185, 49; of up to 40: 10.5, 8.9.
    if (expect <= ATT_ONE_LAUNCH) {
        // short caches: one launch of small workgroups that form the logits
        // themselves (at 300 positions the second launch already pays)
        if (hd == 64) return launch_mix<64, 64, 4, false, 2, true>(a, nseq, st);
        return heads <= 128 ? launch_mix<128, 64, 4, false, 2, true>(a, nseq, st)
                            : launch_mix<128, 128, 4, false, 1, true>(a, nseq, st);
    }
    a.fuse = 64;
    // 16 waves a CU (at most 2048 workgroups), which take several blocks each
    // where there are more: a slice may be mostly empty, and each workgroup that
    // finds nothing to do still costs its launch (us with 2048 workgroups of 8
    // waves, then 512: 16 sequences of 100 positions in slices of 2048 19.7, 13.3;
    // of 2000 54, 51; 1 of 8192 56, 56. With 256, 16 of 4096 147 against 135).
    // Slices of up to 1024 may have 32 a CU, one round (13 of 1000 28.8, 29.3 with 512).
    const int blocks = (expect + AS_POS - 1) / AS_POS, pairs = n_head_kv * nseq;
    const int most = std::min(2048, (blocks <= 16 ? 8192 : 4096) / (n_head / n_head_kv));
    a.grid_y = std::min(blocks, (most + pairs - 1) / pairs);
    // kv heads and sequences first: where only the first blocks find positions,
    // their workgroups are on all XCDs, not on one or two (16 of 80 in slices of
    // 2048, 16 query / 8 kv heads: 18.0, 9.4; 13 of 1000 28.7, 28.0)
    const dim3 grid(pairs, a.grid_y), block(64 * (n_head / n_head_kv));
    if (hd == 128) hipLaunchKernelGGL(attend_scores<128>, grid, block, 0, st, a);
    else hipLaunchKernelGGL(attend_scores<64>, grid, block, 0, st, a);
    if (hipGetLastError() != hipSuccess) return -1;
    // a CU to a workgroup while every one finds its own (1..4 sequences of
    // 1000: 16.8-18.3 us, 17.2-18.7 with the small workgroups); then small
    // workgroups on 64 dimensions up to one per CU and dimension half (8 of
    // 500: 16.9, 18.9 with all 128 dimensions; of 2000 34, 41) where a CU's LDS
    // holds two of them, then on all (13 of 1000: 28.9, 36 with 64; 8 in slices
    // of 8192, with 64 and with 128 dimensions: 20 positions 13.4, 8.9; 500 24.5,
    // 19.5; 8000 162, 129)
    if (hd == 64)
        return heads <= 128 ? launch_mix<64, 64, 8, true, 1>(a, nseq, st)
                            : launch_mix<64, 64, 4, false, 1>(a, nseq, st);
    if (heads <= 128) return launch_mix<128, 64, 8, true, 1>(a, nseq, st);
    const bool two = 2 * (split_lds(cap, 128, 64, am_chunk<64, 4, false>, 1) + sizeof(ExactSumLds) + 1024) <= 160 * 1024;
    return heads <= 256 && two ? launch_mix<128, 64, 4, false, 1>(a, nseq, st)
                               : launch_mix<128, 128, 4, false, 1>(a, nseq, st);
}

int launch_attend_decode(const float *q, const float *kc, const float *vc, const int32_t *pos,
                         int n_head, int n_head_kv, int hd, float scale, float *out,
                         hipStream_t st, int nseq, int n_kv_fixed, int pos_stride,
                         size_t cache_seq_stride) {
    if (hd <= 0 || hd % 4 || hd > 256 || n_head_kv <= 0 || n_head % n_head_kv || nseq <= 0)
        return -1;
    hipLaunchKernelGGL(attend_decode, dim3(n_head, nseq), dim3(256), 0, st, q, kc, vc, pos, n_head,
                       n_head_kv, hd, scale, out, n_kv_fixed, pos_stride, cache_seq_stride);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace llamd
