// q6k_mv.hip -- Q6_K x Q8_K matrix-vector kernels for gfx950 (CDNA4, wave64).
//
// WHAT IS COMPUTED. For every row r, exactly the reference's
// dot_q6k_q8k (crates/llamd-quant/src/dot.rs:138-196): per 256-weight block
// the eight integer lane sums
//     aux32[c] = sum over groups j of sc[j] * sum_{e in j, e mod 8 == c} (q_e - 32) * a_e
// then the ordered float epilogue sums[c] += (f16(d) * a.d) * aux32[c]
// (no FMA), block after block, and finally sums[0] + ... + sums[7] in order.
// The integer part is exact whatever the association, and the float part is
// performed in the reference's order, so the result is BIT-IDENTICAL to the
// CPU path, not merely within REDUCTION.
//
// HOW, ON CDNA4. The integer part runs on the matrix cores. One wave owns a
// 16-row tile; per block and per class c it issues
//     D = v_mfma_i32_16x16x32_i8(A_c, B_c, K_c)
// with
//   B_c[k][n] = code of weight e = 8k + c of row n   (K = the 32 class-c weights,
//               unpacked in registers from the tiled layout, host/layout.cpp)
//   A_c[j][k] = a_e if k / 2 == j else 0             (M = the 16 scale groups:
//               weight e = 8k + c lies in group e / 16 = k / 2)
//   K_c       = A_c x (-32)                           (the code offset, from a
//               second MFMA against a constant, once per block and class)
// so D[j][n] = sum_{e in group j, class c} (q_e - 32) a_e for all 16 groups at
// once. Each lane then holds 4 groups of one row and applies their int8 scales
// with 4 integer multiply-adds; a cross-lane add over the 4 lanes of a row
// gives aux32[c]. HBM traffic is the 210 bytes per 256 weights of the format
// plus the activation, read with three coalesced 16-byte loads per lane per
// block; the 16x redundancy of the masked MFMA costs nothing because the
// matrix cores are >50x faster than HBM can feed this op.
#include "common.hpp"
#include "expf_ref.h"
#include "launch.hpp"
#include "q6k_tile.hpp"
#include "q8k_wave.hpp"
#include "route.hpp"

namespace llamd {
namespace {

// Up to three weight matrices ("segments") share one launch and one
// activation set: gate and up of the same experts, or Q, K and V. Items are
// numbered segment by segment; within a segment, item = slot * tiles + tile.
struct MvSeg {
    const uint8_t *w;         // tiled Q6_K base (expert 0)
    float *y;                 // [n_slots][rows]
    int rows, tiles, first;   // first: index of the segment's first item
};

// The fields every launch reads come first and together, so the kernel's
// prologue fetches them from the kernarg segment in one go before the first
// weight load; the other segments, the routing prologue's and the arg-max
// fields follow.
struct MvParams {
    MvSeg seg0;               // 32 B
    const int8_t *aq;         // Q8_K quants, [n_act][blocks*256]
    const float *ad;          // Q8_K scales, [n_act][blocks]
    const int32_t *ids;       // slot -> expert (nullptr: slot -> expert 0)
    size_t expert_stride;     // bytes between experts' tiled matrices
    int items, blocks;        // items over all segments; 256-blocks per row
    int n_slots, act_per_slot;  // > 0: slot i uses activation i / act_per_slot; 0: activation 0
    MvSeg seg1, seg2;
    int n_seg;
    // routing prologue (ROUTE): wave 0 of every workgroup routes on the exact
    // router logits and takes slot -> expert from its own selection;
    // workgroup 0 publishes ids / weights for the kernels after it
    const float *route_l;     // [n_expert]
    int n_expert, n_used;
    int32_t *ids_out;
    float *w_out;
    int *stats;               // [2] calls (+1 each, both counters)
    // optional per-tile arg-max candidates (one segment): [n_slots][tiles]
    float *amax_v;
    int *amax_i;
    // optional in-kernel clock (llamd_hip_kernel_clock): the launch's record
    unsigned long long *clk;
};

// In-kernel clock: wave w (flat index over the grid) stores its start at
// clk[w] and its end at clk[CLOCK_WAVES + w], s_memrealtime ticks, with plain
// vector stores (one writer per word: no contention, no atomics). The start
// is read first thing and both are stored on every exit of the kernel, so
// the record's pointer is not needed before the kernel's first loads.
constexpr int CLOCK_WAVES = 1024;
template <int WAVES_PER_WG>
struct ClockEnd {
    unsigned long long *r;  // the launch's record (null: no clock)
    unsigned long long t0;
    __device__ ~ClockEnd() {
        const int w = (int)(blockIdx.x * WAVES_PER_WG + (threadIdx.x >> 6));
        if (r && w < CLOCK_WAVES && (threadIdx.x & 63) == 0) {
            r[w] = t0;
            r[CLOCK_WAVES + w] = __builtin_amdgcn_s_memrealtime();
        }
    }
};

// One (slot, 16-row tile) item per KS waves of a 4-wave (KS = 8: 8-wave) workgroup; wave kc of
// the item takes blocks [kc*bpc, (kc+1)*bpc) with the next block's loads in
// flight while the current one is computed. With KS > 1 the per-block terms
// meet in LDS and are folded in block order -- the same additions in the same
// order as a single wave walking every block, so splitting K changes the
// latency, never the bits.
//
// The fields the first loads depend on come as leading scalar arguments,
// which gfx950 preloads into SGPRs at dispatch (kernarg preload): the first
// weight and activation loads issue without waiting for the kernarg segment.
//
// PX is MvParams, or MvLite for the plain matvec (one segment, no routing
// prologue, no arg-max): a 40-byte block instead of 216 bytes, since the
// size of the kernarg segment shows in the launch cost of a small matvec.
struct MvLite {
    float *y;
    size_t expert_stride;
    unsigned long long *clk;
    int rows, n_slots;
};
__device__ __forceinline__ MvParams expand_params(const MvParams &p) { return p; }
__device__ __forceinline__ MvParams expand_params(const MvLite &l) {
    MvParams p = {};
    p.seg0.y = l.y;
    p.seg0.rows = l.rows;
    p.expert_stride = l.expert_stride;
    p.clk = l.clk;
    p.n_slots = l.n_slots;
    p.n_seg = 1;
    return p;
}

template <int KS, bool ROUTE = false, int NSEG = 1, bool AMAX = false, class PX = MvParams>
__global__ __launch_bounds__(KS > 4 ? 64 * KS : 256) void q6k_mv_b1(
    const uint8_t *w0, const int8_t *aq0, const float *ad0, const int32_t *ids0, int blocks0,
    int tiles0, int items0, int act_per_slot0, PX px) {
    const unsigned long long t_start = __builtin_amdgcn_s_memrealtime();
    MvParams p = expand_params(px);
    p.seg0.w = w0;
    p.aq = aq0;
    p.ad = ad0;
    p.ids = ids0;
    p.blocks = blocks0;
    p.seg0.tiles = tiles0;
    p.items = items0;
    p.act_per_slot = act_per_slot0;
    constexpr int IPW = KS >= 4 ? 1 : 4 / KS;   // items per workgroup
    constexpr int MAXB = 16;                    // blocks per row held in LDS (KS > 1)
    __shared__ float terms[KS > 1 ? IPW : 1][KS > 1 ? MAXB : 1][TILE_ROWS][8];
    const int lane = threadIdx.x & 63;
    // the parameter block's fields that the item's segment and the weight
    // address need, fetched in one batch up front (not one dependent scalar
    // load after another)
    if constexpr (NSEG > 1)
        asm volatile("" ::"s"(p.seg1.w), "s"(p.seg1.first), "s"(p.seg1.tiles), "s"(p.seg2.w),
                     "s"(p.seg2.first), "s"(p.seg2.tiles), "s"(p.expert_stride), "s"(p.seg0.y),
                     "s"(p.seg0.rows));
    else
        asm volatile("" ::"s"(p.expert_stride), "s"(p.seg0.y), "s"(p.seg0.rows));
    const ClockEnd<(KS > 4 ? KS : 4)> clock_end{p.clk, t_start};
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
    const int kc = wave % KS;
    const int local = wave / KS;
    const int item = blockIdx.x * IPW + local;
    const bool live = item < p.items;
    // the item's segment, chosen with scalar selects (no indexed kernarg load)
    // field by field (a whole-struct select becomes an indexed stack copy)
    MvSeg sgm = p.seg0;
    sgm.first = 0;  // segment 0 always starts the item numbering
    if constexpr (NSEG > 1) {
        const bool in1 = item >= px.seg1.first;
        const bool in2 = NSEG > 2 && item >= px.seg2.first;
        sgm.w = in2 ? px.seg2.w : in1 ? px.seg1.w : sgm.w;
        sgm.y = in2 ? px.seg2.y : in1 ? px.seg1.y : sgm.y;
        sgm.rows = in2 ? px.seg2.rows : in1 ? px.seg1.rows : sgm.rows;
        sgm.tiles = in2 ? px.seg2.tiles : in1 ? px.seg1.tiles : sgm.tiles;
        sgm.first = in2 ? px.seg2.first : in1 ? px.seg1.first : 0;
    }
    const int pos = item - sgm.first;
    const int slot = live ? pos / sgm.tiles : 0;
    const int t = live ? pos - slot * sgm.tiles : 0;
    const int n = lane & 15;
    const int s = lane >> 4;
    const MaskSel msel = mask_selectors(n, (n >> 2) == s);  // lane carries group n's mask

    int expert;
    if constexpr (ROUTE) {
        // wave 0 routes; the workgroup's other waves wait for its choice
        __shared__ RouteLds rsh;
        if (wave == 0) {
            float l[RW];
#pragma unroll
            for (int j = 0; j < RW; ++j) {
                const int i = lane + WAVE * j;
                l[j] = i < p.n_expert ? p.route_l[i] : 0.0f;
            }
            const bool writer = blockIdx.x == 0;
            route_finish(l, p.n_expert, p.n_used, true, rsh, writer ? p.ids_out : nullptr,
                         writer ? p.w_out : nullptr, nullptr);
            if (writer && lane == 0 && p.stats) {
                p.stats[0] += 1;
                p.stats[1] += 1;
            }
        }
        __syncthreads();
        expert = live ? rsh.sorted[slot] : 0;
    } else {
        expert = (live && p.ids) ? p.ids[slot] : 0;
    }
    const int act = p.act_per_slot ? slot / p.act_per_slot : 0;
    const int8_t *aq = p.aq + (size_t)act * p.blocks * QK_K;
    const float *ad = p.ad + (size_t)act * p.blocks;
    // (without ids, expert 0: no kernarg-segment field on the way to the first load)
    const uint8_t *wexp = (ROUTE || p.ids) ? sgm.w + (size_t)expert * p.expert_stride : sgm.w;
    const uint8_t *seg0 = wexp + (size_t)t * p.blocks * SEG_BYTES;

    const int bpc = (p.blocks + KS - 1) / KS;
    const int b0 = kc * bpc;
    const int b1 = min(p.blocks, b0 + bpc);

    float se = 0.0f, so = 0.0f;  // classes 2s and 2s+1 of row n
    if (live && b0 < b1) {
        // two register sets in ping-pong: the next block's loads are in
        // flight while the current block is computed, with no copies
        BlockRegs ra, rb;
        auto load = [&](BlockRegs &r, int bb) {
            load_block(r, seg0 + (size_t)bb * SEG_BYTES, aq, ad, bb, lane, n);
        };
        auto terms_of = [&](const BlockRegs &r, float &te, float &to) {
            block_terms(r, msel, te, to);
        };
        load(ra, b0);
        for (int b = b0; b < b1; b += 2) {
            if (b + 1 < b1) load(rb, b + 1);
            float te, to;
            terms_of(ra, te, to);
            consume_terms<KS>(b, te, to, se, so, terms[local], n, s);
            if (b + 1 >= b1) break;
            if (b + 2 < b1) load(ra, b + 2);
            terms_of(rb, te, to);
            consume_terms<KS>(b + 1, te, to, se, so, terms[local], n, s);
        }
    }
    if constexpr (KS > 1) {
        __syncthreads();
        if (!live || kc != 0) return;
        // fold in block order, classes 2s and 2s+1 on lane (n, s)
        for (int b = 0; b < p.blocks; ++b) {
            se = se + terms[local][b][n][2 * s];
            so = so + terms[local][b][n][2 * s + 1];
        }
    } else {
        if (!live) return;
    }
    // lane (n, 0) adds the eight class sums in class order (dot.rs:195)
    float cls[8];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        cls[2 * q] = __shfl(se, n + 16 * q, WAVE);
        cls[2 * q + 1] = __shfl(so, n + 16 * q, WAVE);
    }
    const int row = t * TILE_ROWS + n;
    float tot = -0.0f;
#pragma unroll
    for (int c = 0; c < 8; ++c) tot = tot + cls[c];
    if (s == 0 && row < sgm.rows) sgm.y[(size_t)slot * sgm.rows + row] = tot;
    if constexpr (AMAX) {
        // this tile's arg-max candidate for the LM head (argmax_final reduces
        // the tiles): the largest non-NaN logit, lowest row on ties
        const bool ok = s == 0 && row < sgm.rows && !isnan(tot);
        float bv = ok ? tot : -INFINITY;
        int bi = ok ? row : 0x7FFFFFFF;
        argmax_step(bv, bi, dpp<DPP_XOR1>(-INFINITY, bv), dpp<DPP_XOR1>(0x7FFFFFFF, bi));
        argmax_step(bv, bi, dpp<DPP_XOR2>(-INFINITY, bv), dpp<DPP_XOR2>(0x7FFFFFFF, bi));
        argmax_step(bv, bi, dpp<DPP_HALF_MIRROR>(-INFINITY, bv), dpp<DPP_HALF_MIRROR>(0x7FFFFFFF, bi));
        argmax_step(bv, bi, dpp<DPP_MIRROR>(-INFINITY, bv), dpp<DPP_MIRROR>(0x7FFFFFFF, bi));
        if (lane == 0) {
            p.amax_v[(size_t)slot * sgm.tiles + t] = bv;
            p.amax_i[(size_t)slot * sgm.tiles + t] = bi;
        }
    }
}

// Down projection and expert combine in one workgroup per 16-row tile: wave e
// computes the tile for routed expert ids[e] on activation e (all of its
// blocks, next block's loads in flight), then wave 0 adds the experts in
// routing order, out = res + (((0 + w0*y0) + w1*y1) + ...) (layer.rs:245-258,
// 281-287). No cross-workgroup traffic: the combine reads LDS.
struct DownParams {
    const uint8_t *w;
    size_t expert_stride;
    const int32_t *ids;
    const int8_t *aq;     // [n_slots][blocks*256]  (act == nullptr)
    const float *ad;      // [n_slots][blocks]
    const float *weights; // [n_slots] routing weights
    const float *res;     // [rows] or nullptr
    float *out;           // [rows]
    int rows, tiles, blocks, n_slots;
};

__global__ __launch_bounds__(1024) void q6k_down_combine(DownParams p) {
    asm volatile("" ::"s"(p.w), "s"(p.expert_stride), "s"(p.ids), "s"(p.aq), "s"(p.ad),
                 "s"(p.weights), "s"(p.res), "s"(p.out), "s"(p.rows), "s"(p.blocks), "s"(p.n_slots));
    __shared__ float ys[16][TILE_ROWS];
    const int lane = threadIdx.x & 63;
    const int e = threadIdx.x >> 6;
    const int t = blockIdx.x;
    const int n = lane & 15, s = lane >> 4;
    const MaskSel msel = mask_selectors(n, (n >> 2) == s);
    float se = 0.0f, so = 0.0f;
    BlockRegs ra, rb;
    {
        const uint8_t *seg0 = p.w + (size_t)p.ids[e] * p.expert_stride + (size_t)t * p.blocks * SEG_BYTES;
        const int8_t *aq = p.aq + (size_t)e * p.blocks * QK_K;
        const float *ad = p.ad + (size_t)e * p.blocks;
        load_block(ra, seg0, aq, ad, 0, lane, n);
        for (int b = 0; b < p.blocks; b += 2) {
            if (b + 1 < p.blocks) load_block(rb, seg0 + (size_t)(b + 1) * SEG_BYTES, aq, ad, b + 1, lane, n);
            float te, to;
            block_terms(ra, msel, te, to);
            se = se + te;
            so = so + to;
            if (b + 1 >= p.blocks) break;
            if (b + 2 < p.blocks) load_block(ra, seg0 + (size_t)(b + 2) * SEG_BYTES, aq, ad, b + 2, lane, n);
            block_terms(rb, msel, te, to);
            se = se + te;
            so = so + to;
        }
    }
    float cls[8];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        cls[2 * q] = __shfl(se, n + 16 * q, WAVE);
        cls[2 * q + 1] = __shfl(so, n + 16 * q, WAVE);
    }
    if (s == 0) {
        float tot = -0.0f;
#pragma unroll
        for (int c = 0; c < 8; ++c) tot = tot + cls[c];
        ys[e][n] = tot;
    }
    __syncthreads();
    if (e == 0 && lane < TILE_ROWS) {
        const int row = t * TILE_ROWS + lane;
        if (row < p.rows) {
            float acc = 0.0f;
            for (int q = 0; q < p.n_slots; ++q) {
                const float prod = p.weights[q] * ys[q][lane];
                acc = acc + prod;
            }
            p.out[row] = p.res ? p.res[row] + acc : acc;
        }
    }
}

// Device dequantization of the tiled layout back to f32, element order of
// crates/llamd-quant/src/lib.rs:181-226 (d * sc first, then * (q - 32)).
// One wave per segment; out is [rows][blocks*256].
__global__ __launch_bounds__(256) void q6k_dequant_tiled(const uint8_t *w, int rows, int tiles,
                                                         int blocks, float *out) {
    const int lane = threadIdx.x & 63;
    const int item = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (item >= tiles * blocks) return;
    const int t = item / blocks, b = item - t * blocks;
    const uint8_t *seg = w + (size_t)item * SEG_BYTES;
    const int n = lane & 15, s = lane >> 4;
    const int row = t * TILE_ROWS + n;
    const uint4 q0 = *(const uint4 *)(seg + 16 * lane);
    const uint4 q1 = *(const uint4 *)(seg + SEG_PART + 16 * lane);
    const uint4 q2 = *(const uint4 *)(seg + 2 * SEG_PART + 16 * lane);
    const uint32_t scw = *(const uint32_t *)(seg + SEG_SC + 4 * lane);
    const float d = f16_bits_to_f32(*(const uint16_t *)(seg + SEG_D + 2 * n));
    const uint32_t nib[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
    const uint32_t hb[4] = {q2.x, q2.y, q2.z, q2.w};
    if (row >= rows) return;
    float *o = out + (size_t)row * blocks * QK_K + (size_t)b * QK_K;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const uint64_t codes = (uint64_t)unpack_codes(nib, hb, c);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int m = 8 * s + k;           // class element index
            const int e = 8 * m + c;           // weight index in the block
            const int grp = e >> 4;            // = 4 s + k / 2
            const int sc = (int8_t)((scw >> (8 * (grp - 4 * s))) & 0xFF);
            const int q = (int)((codes >> (8 * k)) & 0x3F) - 32;
            o[e] = d * (float)sc * (float)q;
        }
    }
}


// ---- batched / expert-grouped: up to 16 tokens per MFMA ---------------------
//
// For many tokens against one weight tile, the scale is folded into the
// weights instead of into the masked activation: per class c,
//     w'_k = sc[group(k)] * (q_k - 32)  in [-4064, 4096]
// is split into two int8 digits w' = 64 * hi + lo (lo = w' & 63, hi = w' >> 6)
// and two MFMAs against the 16 tokens' class-c activations give
//     aux32[c] = 64 * (A_hi x B) + (A_lo x B)
// exactly, for 16 rows x 16 tokens at once. The float epilogue per (row,
// token) is the reference's, so every output is again bit-identical to
// dot_q6k_q8k on that token's activation.
//
// Work: one wave per (16-token chunk, or two, of one group; 16-row tile t). A
// group is one expert and its run of sorted pairs (moe_group's records); the LM
// head at batch 16 is one group of 16 tokens. Activations are read in the
// token-chunked layout (q8k_wave.hpp).
struct BatchParams {
    const uint8_t *w;
    size_t expert_stride;
    const int32_t *pair_out;     // output row of each sorted pair (nullptr: identity)
    const int8_t *act_q;         // token-chunked Q8_K quants (q8k_wave.hpp)
    const float *act_d;          // their scales
    float *y;                    // y[pair_out * ldy + row]
    float *amax_v;               // optional per-(token, tile) arg-max candidates
    int *amax_i;                 //   [token][tiles] (single group only)
    int ldy, rows, tiles, blocks;
    int single_count;            // sub_info == nullptr: one group, expert 0, this many tokens
    const GroupItem *sub_info;   // each chunk's record (launch_moe_group)
    const GroupItem *twin_info;  // each twin's
    const GroupItem *wide_info;  // each wide unit's (q6k_mv_batched_wide)
    // optional second matrix of the same shape on the same activations (gate
    // and up in one launch): items from items_per_mat on use w2 / y2
    const uint8_t *w2;
    float *y2;
    int items_per_mat;
    // n_segs > 0 (single group only): up to three matrices of their own row
    // counts on the same activations in one launch (Q, K and V of a batch);
    // segment i's items start at item segs[i].first
    int n_segs;
    struct Seg {
        const uint8_t *w;
        float *y;
        int rows, tiles, first, items;
    } segs[3];
};

// The work item of this wave and the parameters it runs with: the second
// matrix's items are the first's, offset by items_per_mat. The item is the same
// for the whole wave, so its addresses stay in SGPRs (twins 168 -> 154 registers);
// SEGS false: grouped calls, which have no segments to choose from. Together 512
// tokens 258.6 -> 248.6 us a call, 45 104.7 -> 102.3, a layer of 16 sequences
// 109.4 -> 107.2.
template <bool SEGS>
__device__ __forceinline__ int batch_item(const BatchParams &p, BatchParams &q, int item) {
    q = p;
    if (SEGS && p.n_segs > 0) {
        // the item's segment, chosen with scalar selects
        BatchParams::Seg sg = p.segs[0];
        if (p.n_segs > 1 && item >= p.segs[1].first) sg = p.segs[1];
        if (p.n_segs > 2 && item >= p.segs[2].first) sg = p.segs[2];
        q.w = sg.w;
        q.y = sg.y;
        q.rows = q.ldy = sg.rows;
        q.tiles = sg.tiles;
        q.items_per_mat = sg.items;
        return item - sg.first;
    }
    if (p.w2 && item >= p.items_per_mat) {
        item -= p.items_per_mat;
        q.w = p.w2;
        q.y = p.y2;
    }
    return item;
}

typedef short s16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ s16x2 as_s16x2(uint32_t v) { return __builtin_bit_cast(s16x2, v); }
__device__ __forceinline__ uint32_t as_u32(s16x2 v) { return __builtin_bit_cast(uint32_t, v); }

// Per-block constants of the fold: this lane's 4 scales as int16 pairs, and
// 128 - 32 * scale likewise (so sc * (q - 32) + 128 is one packed multiply-add).
struct FoldScales {
    s16x2 sc[4], off[4];
};

__device__ __forceinline__ FoldScales fold_scales(uint32_t scw) {
    FoldScales f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const short v = (short)(int8_t)((scw >> (8 * j)) & 0xFF);
        f.sc[j] = s16x2{v, v};
        f.off[j] = s16x2{(short)(128 - 32 * v), (short)(128 - 32 * v)};
    }
    return f;
}

// w' = sc * (q - 32) for the lane's 8 class-c weights (codes: one byte each,
// weight kk uses scale kk / 2), split into int8 digits w' = 256 * hi + lo with
// lo in [-128, 127] and hi in [-16, 16]. One packed 16-bit multiply-add per
// two weights gives v = w' + 128 in [-3936, 4224]; the high byte of v is hi
// (arithmetic: floor(v / 256)) and its low byte, minus 128, is lo -- as a
// byte, the low byte with its top bit flipped. Byte permutes gather the
// 8-byte MFMA operands straight from the 16-bit lanes.
__device__ __forceinline__ void fold_digits(uint64_t codes, const FoldScales &f, long &lo8,
                                            long &hi8) {
    const uint32_t c0 = (uint32_t)codes, c1 = (uint32_t)(codes >> 32);
    const uint32_t w[4] = {__builtin_amdgcn_perm(0u, c0, 0x0C010C00u),
                           __builtin_amdgcn_perm(0u, c0, 0x0C030C02u),
                           __builtin_amdgcn_perm(0u, c1, 0x0C010C00u),
                           __builtin_amdgcn_perm(0u, c1, 0x0C030C02u)};
    uint32_t v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = as_u32(as_s16x2(w[j]) * f.sc[j] + f.off[j]);
    lo8 = (long)((uint64_t)(__builtin_amdgcn_perm(v[1], v[0], 0x06040200u) ^ 0x80808080u) |
                 ((uint64_t)(__builtin_amdgcn_perm(v[3], v[2], 0x06040200u) ^ 0x80808080u) << 32));
    hi8 = (long)((uint64_t)__builtin_amdgcn_perm(v[1], v[0], 0x07050301u) |
                 ((uint64_t)__builtin_amdgcn_perm(v[3], v[2], 0x07050301u) << 32));
}


// The outputs of tile_block's sums: y, and the tile's arg-max candidates.
template <int NC>
__device__ __forceinline__ void batched_store(const BatchParams &p, const float (&sums)[NC][8][4], int lane,
                                              int t, int st0, int cnt, int start) {
    const int n = lane & 15, s = lane >> 4;
#pragma unroll
    for (int u = 0; u < NC; ++u) {
        const int tok = 16 * (st0 + u) + n;  // this lane's token (B operand / output column)
        const bool tok_ok = tok < cnt;       // slots past the last token hold no data;
                                             // their columns are never stored
        float bv = -INFINITY;  // arg-max candidate of this lane's rows (lowest row on ties)
        int bi = 0x7FFFFFFF;
        if (tok_ok) {
            const int pos = start + tok;
            const int orow = p.pair_out ? p.pair_out[pos] : pos;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = t * TILE_ROWS + 4 * s + v;
                if (row < p.rows) {
                    float tot = -0.0f;
#pragma unroll
                    for (int c = 0; c < 8; ++c) tot = tot + sums[u][c][v];
                    p.y[(size_t)orow * p.ldy + row] = tot;
                    if (!isnan(tot)) argmax_step(bv, bi, tot, row);
                }
            }
        }
        if (p.amax_v) {
            // combine the 4 lanes (s = 0..3) of each token: lanes n, n+16, n+32, n+48
            argmax_step(bv, bi, __shfl_xor(bv, 16, WAVE), __shfl_xor(bi, 16, WAVE));
            argmax_step(bv, bi, __shfl_xor(bv, 32, WAVE), __shfl_xor(bi, 32, WAVE));
            if (s == 0 && tok_ok) {
                p.amax_v[(size_t)tok * p.tiles + t] = bv;
                p.amax_i[(size_t)tok * p.tiles + t] = bi;
            }
        }
    }
}

// One block of a tile against NC chunks whose planes lie in LDS at aq (this
// lane's 16 bytes of the first plane; chunks CHUNK_BLOCK_BYTES apart): the
// integer dots of all 8 classes and the reference's ordered sums.
struct TileRegs {
    uint4 q0, q1, q2;
    uint32_t scw;
    uint2 dw;
};
__device__ __forceinline__ void tile_load(TileRegs &r, const uint8_t *sg, int lane) {
    r.q0 = *(const uint4 *)(sg + 16 * lane);
    r.q1 = *(const uint4 *)(sg + SEG_PART + 16 * lane);
    r.q2 = *(const uint4 *)(sg + 2 * SEG_PART + 16 * lane);
    r.scw = *(const uint32_t *)(sg + SEG_SC + 4 * lane);
    r.dw = *(const uint2 *)(sg + SEG_D + 8 * (lane >> 4));  // f16 d of rows 4s..4s+3
}

__device__ __forceinline__ long plane_half(v4i v, int h) {
    return (long)((uint64_t)(uint32_t)v[2 * h] | ((uint64_t)(uint32_t)v[2 * h + 1] << 32));
}

template <int NC>
__device__ __forceinline__ void tile_block(const TileRegs &r, const float (&adb)[NC], const int8_t *aq,
                                           float (&sums)[NC][8][4]) {
    const uint32_t nib[8] = {r.q0.x, r.q0.y, r.q0.z, r.q0.w, r.q1.x, r.q1.y, r.q1.z, r.q1.w};
    const uint32_t hb[4] = {r.q2.x, r.q2.y, r.q2.z, r.q2.w};
    const FoldScales fs = fold_scales(r.scw);
    const float d4[4] = {f16_bits_to_f32((uint16_t)(r.dw.x & 0xFFFF)), f16_bits_to_f32((uint16_t)(r.dw.x >> 16)),
                         f16_bits_to_f32((uint16_t)(r.dw.y & 0xFFFF)), f16_bits_to_f32((uint16_t)(r.dw.y >> 16))};
    float dd[NC][4];
#pragma unroll
    for (int u = 0; u < NC; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) dd[u][v] = d4[v] * adb[u];
    const v4i zero = {0, 0, 0, 0};
    v4i act[2][NC], dh[2][NC], dl[2][NC];
    const auto read = [&](int P) {
#pragma unroll
        for (int u = 0; u < NC; ++u) act[P & 1][u] = *(const v4i *)(aq + u * CHUNK_BLOCK_BYTES + 1024 * P);
    };
    // class c's MFMAs are issued before class c - 1's results are used
    const auto dots = [&](int c) {
        long a_lo, a_hi;
        fold_digits((uint64_t)unpack_codes(nib, hb, c), fs, a_lo, a_hi);
#pragma unroll
        for (int u = 0; u < NC; ++u) {
            const long av = plane_half(act[(c >> 1) & 1][u], c & 1);
            dh[c & 1][u] = __builtin_amdgcn_mfma_i32_16x16x32_i8(a_hi, av, zero, 0, 0, 0);
            dl[c & 1][u] = __builtin_amdgcn_mfma_i32_16x16x32_i8(a_lo, av, zero, 0, 0, 0);
        }
    };
    read(0);
    dots(0);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        if ((c & 1) == 0 && c + 2 < 8) read((c >> 1) + 1);
        if (c + 1 < 8) dots(c + 1);
#pragma unroll
        for (int u = 0; u < NC; ++u)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int aux = dh[c & 1][u][v] * 256 + dl[c & 1][u][v];
                sums[u][c][v] = sums[u][c][v] + dd[u][v] * (float)aux;
            }
    }
}

// ---- REDUCTION-tolerance batched kernels (LLAMD_HIP_REDUCTION) ----------------
//
// The same operands and digits as tile_block, but the MFMAs of all 8
// classes of a block accumulate into one pair of digit accumulators: the
// block's integer dot sum_c aux32[c] is exact in int32 (|.| < 2^27), and the
// float epilogue is one convert and one fused multiply-add per (row, token,
// block) instead of the reference's eight ordered class sums. Only the float
// rounding differs from dot_q6k_q8k (nb products and additions per row
// instead of 8 nb and the 8-term class sum), so outputs are within REDUCTION,
// not bit-identical. Because the partial sums may now be added in any order,
// K is split over KS waves of one workgroup (a shorter dependent chain of
// block loads per wave, KS times the waves in flight), met in LDS.

// The dynamic LDS of the staged kernels below.
extern __shared__ uint4 g_act_lds[];

// The digit operands of the 64-deep MFMA of classes 2 P and 2 P + 1.
__device__ __forceinline__ void fold_pair(const uint32_t nib[8], const uint32_t hb[4], int P,
                                          const FoldScales &fs, v4i &lo, v4i &hi) {
    long l[2], h[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) fold_digits((uint64_t)unpack_codes(nib, hb, 2 * P + i), fs, l[i], h[i]);
    lo = v4i{(int)l[0], (int)(l[0] >> 32), (int)l[1], (int)(l[1] >> 32)};
    hi = v4i{(int)h[0], (int)(h[0] >> 32), (int)h[1], (int)(h[1] >> 32)};
}

// The lane's partial sums (4 rows x NC chunks) over blocks [b0, b1) of tile t.
// LDSA: the chunk's quants are read from g_act_lds (same layout).
template <int NC, bool LDSA = false>
__device__ __forceinline__ void fast_tile_range(const BatchParams &p, int lane, int t, int sub0,
                                                int expert, int b0, int b1, float acc[2][4]) {
    const int n = lane & 15, s = lane >> 4;
    const uint8_t *seg = p.w + (size_t)expert * p.expert_stride + (size_t)t * p.blocks * SEG_BYTES;
    const size_t chunk_q = (size_t)p.blocks * CHUNK_BLOCK_BYTES, chunk_d = (size_t)p.blocks * CHUNK_TOKENS;
    const int8_t *aq = LDSA ? (const int8_t *)g_act_lds + 16 * lane
                            : p.act_q + (size_t)sub0 * chunk_q + 16 * lane;
    const float *ad = p.act_d + (size_t)sub0 * chunk_d + n;
    // planes of two classes one ahead of their MFMAs, across blocks (past the
    // range's last block the loads re-read it, unused)
    const int last = b1 - 1;
    v4i act[2][NC];
    auto aload = [&](int b, int P) {
#pragma unroll
        for (int u = 0; u < NC; ++u)
            act[P % 2][u] = *(const v4i *)(aq + u * chunk_q + (size_t)min(b, last) * CHUNK_BLOCK_BYTES + 1024 * P);
    };
    aload(b0, 0);
    struct W {
        uint4 q0, q1, q2;
        uint32_t scw;
        uint2 dw;
        float adb[NC];
    };
    auto wload = [&](W &r, int b) {
        const uint8_t *sg = seg + (size_t)b * SEG_BYTES;
        r.q0 = *(const uint4 *)(sg + 16 * lane);
        r.q1 = *(const uint4 *)(sg + SEG_PART + 16 * lane);
        r.q2 = *(const uint4 *)(sg + 2 * SEG_PART + 16 * lane);
        r.scw = *(const uint32_t *)(sg + SEG_SC + 4 * lane);
        r.dw = *(const uint2 *)(sg + SEG_D + 8 * s);  // f16 d of rows 4s..4s+3
#pragma unroll
        for (int u = 0; u < NC; ++u) r.adb[u] = ad[u * chunk_d + (size_t)b * CHUNK_TOKENS];
    };
    auto compute = [&](const W &r, int b) {
        const uint32_t nib[8] = {r.q0.x, r.q0.y, r.q0.z, r.q0.w, r.q1.x, r.q1.y, r.q1.z, r.q1.w};
        const uint32_t hb[4] = {r.q2.x, r.q2.y, r.q2.z, r.q2.w};
        const FoldScales fs = fold_scales(r.scw);
        const v4i zero = {0, 0, 0, 0};
        v4i ah[NC], al[NC];
#pragma unroll
        for (int u = 0; u < NC; ++u) ah[u] = al[u] = zero;
#pragma unroll
        for (int P = 0; P < 4; ++P) {
            aload(P + 1 < 4 ? b : b + 1, (P + 1) % 4);
            v4i a_lo, a_hi;
            fold_pair(nib, hb, P, fs, a_lo, a_hi);
#pragma unroll
            for (int u = 0; u < NC; ++u) {
                ah[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a_hi, act[P % 2][u], ah[u], 0, 0, 0);
                al[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a_lo, act[P % 2][u], al[u], 0, 0, 0);
            }
        }
        const float d4[4] = {f16_bits_to_f32((uint16_t)(r.dw.x & 0xFFFF)), f16_bits_to_f32((uint16_t)(r.dw.x >> 16)),
                             f16_bits_to_f32((uint16_t)(r.dw.y & 0xFFFF)), f16_bits_to_f32((uint16_t)(r.dw.y >> 16))};
#pragma unroll
        for (int u = 0; u < NC; ++u)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int aux = ah[u][v] * 256 + al[u][v];
                acc[u][v] = __builtin_fmaf(d4[v] * r.adb[u], (float)aux, acc[u][v]);
            }
    };
    if constexpr (LDSA) {
        // the planes come from LDS (lgkmcnt), so the next block's weights can
        // be in flight a whole block ahead without a plane's wait also waiting
        // for them; the scheduling barriers keep the compiler from sinking
        // those loads back to their first use
        W ra, rb;
        wload(ra, b0);
        for (int b = b0; b < b1; b += 2) {
            wload(rb, min(b + 1, last));
            __builtin_amdgcn_sched_barrier(0);
            compute(ra, b);
            if (b + 1 >= b1) break;
            wload(ra, min(b + 2, last));
            __builtin_amdgcn_sched_barrier(0);
            compute(rb, b + 1);
        }
    } else {
        for (int b = b0; b < b1; ++b) {
            W r;
            wload(r, b);
            compute(r, b);
        }
    }
}

// KS waves per work item (4 / KS items per workgroup). TWIN: the items are
// twins (moe_group's twin records), else 16-token chunks (chunk records, or
// the single group).
// LDSA: one 16-token chunk for the whole grid (the LM head at batch <= 16):
// each workgroup first copies the chunk's quants (blocks x 4 KiB, dynamic
// LDS) once, so the class-plane loads of every block read LDS instead of
// going through the vector memory path (they outnumber the weight loads).
template <int KS, bool TWIN, bool LDSA = false>
__global__ __launch_bounds__(256) void q6k_mv_batched_fast(BatchParams pk) {
    constexpr int IPW = 4 / KS;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int kc = wave % KS;
    const int n = lane & 15, s = lane >> 4;
    int item = (int)blockIdx.x * IPW + wave / KS;
    BatchParams p = pk;
    if (p.w2 && item >= p.items_per_mat) {
        item -= p.items_per_mat;
        p.w = p.w2;
        p.y = p.y2;
    }
    bool live = item < p.items_per_mat;  // the grid's rounding to whole workgroups
    int t = 0, sub = 0, st = 0, cnt = 0, start = 0, expert = 0, nc = 1;
    if (live) {
        t = item % p.tiles;
        const int unit = item / p.tiles;
        if (p.sub_info) {
            const GroupItem it = TWIN ? p.twin_info[unit] : p.sub_info[unit];  // expert -1: spare
            live = it.expert >= 0;
            st = it.st;
            sub = it.sub;
            cnt = it.count;
            start = it.start;
            expert = it.expert;
            nc = TWIN && it.twin2 ? 2 : 1;
        } else {
            cnt = p.single_count;
            sub = st = unit;
            live = unit < (cnt + 15) / 16;
        }
    }
    const int bpc = (p.blocks + KS - 1) / KS;
    const int b0 = kc * bpc, b1 = min(p.blocks, b0 + bpc);
    float acc[2][4] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
    if constexpr (LDSA) {
        const int n16 = p.blocks * CHUNK_BLOCK_BYTES / 16;
        const uint4 *src = (const uint4 *)p.act_q;
        for (int i = threadIdx.x; i < n16; i += blockDim.x) g_act_lds[i] = src[i];
        __syncthreads();
        if (live && b0 < b1) fast_tile_range<1, true>(p, lane, t, 0, expert, b0, b1, acc);
    } else if (live && b0 < b1) {
        if (nc == 2) fast_tile_range<2>(p, lane, t, sub, expert, b0, b1, acc);
        else fast_tile_range<1>(p, lane, t, sub, expert, b0, b1, acc);
    }
    if constexpr (KS > 1) {
        // every wave reaches the barrier (no early return above)
        __shared__ float part[4][2][4][WAVE];
        if (kc != 0) {
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int v = 0; v < 4; ++v) part[wave][u][v][lane] = acc[u][v];
        }
        __syncthreads();
        if (kc != 0) return;
#pragma unroll
        for (int k = 1; k < KS; ++k)
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[u][v] += part[wave + k][u][v][lane];
    }
    if (!live) return;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        if (u >= nc) break;
        const int tok = 16 * (st + u) + n;  // this lane's token
        const bool tok_ok = tok < cnt;
        float bv = -INFINITY;  // arg-max candidate of this lane's rows (lowest row on ties)
        int bi = 0x7FFFFFFF;
        int nan_row = 0;       // a NaN logit in the tile voids the tile's certificate
        if (tok_ok) {
            const int pos = start + tok;
            const int orow = p.pair_out ? p.pair_out[pos] : pos;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = t * TILE_ROWS + 4 * s + v;
                if (row < p.rows) {
                    p.y[(size_t)orow * p.ldy + row] = acc[u][v];
                    if (!isnan(acc[u][v])) argmax_step(bv, bi, acc[u][v], row);
                    else nan_row = 1;
                }
            }
        }
        if (p.amax_v) {
            // the 4 lanes (s = 0..3) of each token: lanes n, n+16, n+32, n+48
            argmax_step(bv, bi, __shfl_xor(bv, 16, WAVE), __shfl_xor(bi, 16, WAVE));
            argmax_step(bv, bi, __shfl_xor(bv, 32, WAVE), __shfl_xor(bi, 32, WAVE));
            nan_row |= __shfl_xor(nan_row, 16, WAVE);
            nan_row |= __shfl_xor(nan_row, 32, WAVE);
            if (s == 0 && tok_ok) {
                p.amax_v[(size_t)tok * p.tiles + t] = bv;
                p.amax_i[(size_t)tok * p.tiles + t] = nan_row ? -1 : bi;
            }
        }
    }
}



// The grouped kernel with the activations staged in LDS. A workgroup's 4
// waves are 4 tiles of one unit (tiles % 4 == 0), so they read the same
// chunks: per block, the unit's NC x 4 KiB of class planes are copied once
// into LDS by direct global-to-LDS loads (1 KiB per wave instruction, no
// registers), double-buffered, and every wave reads its planes from LDS. The
// next block's planes and weights are in flight while the current block is
// computed; one barrier per block hands the buffer over.
using lds_ptr = __attribute__((address_space(3))) void *;

// One group of tokens against few tiles (Q, K, V or an output projection of a few
// sequences): a workgroup per (chunk, tile), wave P on classes 2P and 2P + 1
// alone. Each class's sum stays with one wave, block after block, and one
// thread per output adds the eight in class order, so the bits are those of
// q6k_mv_batched_staged; the chip gets four times the waves, each with a quarter
// of the chain (launch_one_group has the figures).
__global__ __launch_bounds__(256) void q6k_mv_batched_classes(BatchParams pk) {
    __shared__ float part[8][4][64];  // [class][v][lane]
    const int lane = threadIdx.x & 63, P = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    BatchParams p;
    const int item = batch_item<true>(pk, p, (int)blockIdx.x);
    const int t = item % p.tiles, chunk = item / p.tiles;
    if (CHUNK_TOKENS * chunk >= p.single_count) return;
    const uint8_t *seg = p.w + (size_t)t * p.blocks * SEG_BYTES;
    const int8_t *aq = p.act_q + (size_t)chunk * p.blocks * CHUNK_BLOCK_BYTES + 1024 * P + 16 * lane;
    const float *ad = p.act_d + (size_t)chunk * p.blocks * CHUNK_TOKENS + (lane & 15);
    struct Regs {
        uint2 nib;
        uint32_t hb, scw;
        uint2 dw;
        v4i a;
        float ad;
    };
    constexpr int B = 4;  // blocks per batch of loads, two batches in turn
    Regs ra[B], rb[B];
    const auto load = [&](Regs (&r)[B], int b0) {
#pragma unroll
        for (int k = 0; k < B; ++k) {
            const int b = min(b0 + k, p.blocks - 1);
            const uint8_t *sg = seg + (size_t)b * SEG_BYTES;
            r[k].nib = *(const uint2 *)(sg + (P >> 1) * SEG_PART + 16 * lane + 8 * (P & 1));
            r[k].hb = *(const uint32_t *)(sg + 2 * SEG_PART + 16 * lane + 4 * P);
            r[k].scw = *(const uint32_t *)(sg + SEG_SC + 4 * lane);
            r[k].dw = *(const uint2 *)(sg + SEG_D + 8 * (lane >> 4));
            r[k].a = *(const v4i *)(aq + (size_t)b * CHUNK_BLOCK_BYTES);
            r[k].ad = ad[b * CHUNK_TOKENS];
        }
    };
    float sums[2][4] = {};
    const auto add = [&](const Regs (&r)[B], int b0) {
#pragma unroll
        for (int k = 0; k < B; ++k) {
            if (b0 + k < p.blocks) {
                const uint32_t nib[8] = {r[k].nib.x, r[k].nib.y}, hb[4] = {r[k].hb};
                const FoldScales fs = fold_scales(r[k].scw);
                const uint16_t dh[4] = {(uint16_t)(r[k].dw.x & 0xFFFF), (uint16_t)(r[k].dw.x >> 16),
                                        (uint16_t)(r[k].dw.y & 0xFFFF), (uint16_t)(r[k].dw.y >> 16)};
                const v4i zero = {0, 0, 0, 0};
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    long a_lo, a_hi;
                    fold_digits((uint64_t)unpack_codes(nib, hb, j), fs, a_lo, a_hi);
                    const long av = plane_half(r[k].a, j);
                    const v4i hi = __builtin_amdgcn_mfma_i32_16x16x32_i8(a_hi, av, zero, 0, 0, 0);
                    const v4i lo = __builtin_amdgcn_mfma_i32_16x16x32_i8(a_lo, av, zero, 0, 0, 0);
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int aux = hi[v] * 256 + lo[v];
                        sums[j][v] = sums[j][v] + f16_bits_to_f32(dh[v]) * r[k].ad * (float)aux;
                    }
                }
            }
        }
    };
    load(ra, 0);
    for (int b = 0; b < p.blocks; b += 2 * B) {
        load(rb, b + B);
        add(ra, b);
        load(ra, b + 2 * B);
        add(rb, b + B);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) part[2 * P + j][v][lane] = sums[j][v];
    __syncthreads();
    // wave v stores the rows 4s + v
    const int tok = 16 * chunk + (lane & 15), row = t * TILE_ROWS + 4 * (lane >> 4) + P;
    if (tok < p.single_count && row < p.rows) {
        float tot = -0.0f;
#pragma unroll
        for (int c = 0; c < 8; ++c) tot = tot + part[c][P][lane];
        p.y[(size_t)(p.pair_out ? p.pair_out[tok] : tok) * p.ldy + row] = tot;
    }
}

// A twin's (or chunk's) planes staged in LDS for 4 tiles, as in
// q6k_mv_batched_fast_staged below: a plane is read from L2 once per 4 tiles
// instead of once per tile, and the loop keeps no planes in flight in registers
// (512 tokens, skewed routing: 282 -> 262 us a call; 2000: 775 -> 727; still
// bound by vector issue, the fold per twin and the ordered sums per chunk).
template <int NC, bool PF = false>
__device__ __forceinline__ void exact_tile_staged(const BatchParams &p, const GroupItem &it, int lane, int wave,
                                                  int t) {
    const size_t chunk_q = (size_t)p.blocks * CHUNK_BLOCK_BYTES, chunk_d = (size_t)p.blocks * CHUNK_TOKENS;
    const uint8_t *seg = p.w + (size_t)it.expert * p.expert_stride + (size_t)t * p.blocks * SEG_BYTES;
    const int8_t *gq = p.act_q + (size_t)it.sub * chunk_q + 1024 * wave + 16 * lane;
    const float *ad = p.act_d + (size_t)it.sub * chunk_d + (lane & 15);
    int8_t *lds = (int8_t *)g_act_lds;  // [2][NC][4096]
    auto stage = [&](int b) {           // plane `wave` of each chunk
#pragma unroll
        for (int u = 0; u < NC; ++u)
            __builtin_amdgcn_global_load_lds((const void *)(gq + u * chunk_q + (size_t)b * CHUNK_BLOCK_BYTES),
                                             (lds_ptr)(lds + ((b & 1) * NC + u) * CHUNK_BLOCK_BYTES + 1024 * wave),
                                             16, 0, 0);
    };
    float sums[NC][8][4];
#pragma unroll
    for (int u = 0; u < NC; ++u)
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int v = 0; v < 4; ++v) sums[u][c][v] = 0.0f;
    struct R {
        TileRegs t;
        float adb[NC];
    } ra, rb;
    const int last = p.blocks - 1;
    const auto load = [&](R &r, int b) {
        tile_load(r.t, seg + (size_t)b * SEG_BYTES, lane);
#pragma unroll
        for (int u = 0; u < NC; ++u) r.adb[u] = ad[u * chunk_d + (size_t)b * CHUNK_TOKENS];
    };
    // block b's planes (and weights) have landed, and the other buffer is read
    const auto handover = [&]() {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    };
    stage(0);
    if constexpr (PF) {
        load(ra, 0);
        // the next block's weights in flight too, where registers allow
        for (int b = 0; b < p.blocks; b += 2) {
            handover();
            if (b < last) stage(b + 1);
            load(rb, min(b + 1, last));
            __builtin_amdgcn_sched_barrier(0);
            tile_block<NC>(ra.t, ra.adb, lds + 16 * lane, sums);
            if (b == last) break;
            handover();
            if (b + 1 < last) stage(b + 2);
            load(ra, min(b + 2, last));
            __builtin_amdgcn_sched_barrier(0);
            tile_block<NC>(rb.t, rb.adb, lds + NC * CHUNK_BLOCK_BYTES + 16 * lane, sums);
        }
    } else {
        for (int b = 0; b < p.blocks; ++b) {
            load(ra, b);
            handover();
            if (b < last) stage(b + 1);
            tile_block<NC>(ra.t, ra.adb, lds + (b & 1) * NC * CHUNK_BLOCK_BYTES + 16 * lane, sums);
        }
    }
    batched_store<NC>(p, sums, lane, t, it.st, it.count, it.start);
}

// A group of T <= 2 tokens against a tile, as q6k_mv_b1 does it: the masked
// activations and the scales after the MFMA, so nothing is folded into the
// weights and no token slot is idle (about 110 and 170 vector instructions per
// block for 1 and 2 tokens, 330 for a 16-token chunk). The A operand of class c
// is this lane's 8 bytes of the chunk's plane, kept where they belong to scale
// group n.
template <int T>
__device__ __forceinline__ void few_tile(const BatchParams &p, const GroupItem &it, int lane, int t) {
    const int n = lane & 15, s = lane >> 4;
    const uint8_t *seg = p.w + (size_t)it.expert * p.expert_stride + (size_t)t * p.blocks * SEG_BYTES;
    const int8_t *aq = p.act_q + (size_t)it.sub * p.blocks * CHUNK_BLOCK_BYTES + 256 * s;
    const float *ad = p.act_d + (size_t)it.sub * p.blocks * CHUNK_TOKENS;
    const uint64_t mask = (n >> 2) == s ? 0xFFFFull << (16 * (n & 3)) : 0ull;
    struct Regs {
        uint4 q0, q1, q2;
        uint32_t scw;
        uint16_t dh;
        v4i a[T][4];
        float ad[T];
    } ra, rb;
    const auto load = [&](Regs &r, int b) {
        const uint8_t *sg = seg + (size_t)b * SEG_BYTES;
        r.q0 = *(const uint4 *)(sg + 16 * lane);
        r.q1 = *(const uint4 *)(sg + SEG_PART + 16 * lane);
        r.q2 = *(const uint4 *)(sg + 2 * SEG_PART + 16 * lane);
        r.scw = *(const uint32_t *)(sg + SEG_SC + 4 * lane);
        r.dh = *(const uint16_t *)(sg + SEG_D + 2 * n);
#pragma unroll
        for (int k = 0; k < T; ++k) {
#pragma unroll
            for (int P = 0; P < 4; ++P)
                r.a[k][P] = *(const v4i *)(aq + (size_t)b * CHUNK_BLOCK_BYTES + 1024 * P + 16 * k);
            r.ad[k] = ad[b * CHUNK_TOKENS + k];
        }
    };
    float se[T], so[T];  // classes 2s and 2s+1 of row n
#pragma unroll
    for (int k = 0; k < T; ++k) se[k] = so[k] = 0.0f;
    const auto add = [&](const Regs &r) {
        const uint32_t nib[8] = {r.q0.x, r.q0.y, r.q0.z, r.q0.w, r.q1.x, r.q1.y, r.q1.z, r.q1.w};
        const uint32_t hb[4] = {r.q2.x, r.q2.y, r.q2.z, r.q2.w};
        const v4i zero = {0, 0, 0, 0};
        const int sc0 = __builtin_amdgcn_sbfe(r.scw, 0, 8), sc1 = __builtin_amdgcn_sbfe(r.scw, 8, 8);
        const int sc2 = __builtin_amdgcn_sbfe(r.scw, 16, 8), sc3 = __builtin_amdgcn_sbfe(r.scw, 24, 8);
        int acc[T][8];
        v4i d[2][T];
        const auto dots = [&](int c) {
            const long codes = unpack_codes(nib, hb, c);
#pragma unroll
            for (int k = 0; k < T; ++k) {
                const long am = plane_half(r.a[k][c >> 1], c & 1) & (long)mask;
                const v4i kc = __builtin_amdgcn_mfma_i32_16x16x32_i8(am, NEG32_BYTES, zero, 0, 0, 0);
                d[c & 1][k] = __builtin_amdgcn_mfma_i32_16x16x32_i8(am, codes, kc, 0, 0, 0);
            }
        };
        dots(0);
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            if (c + 1 < 8) dots(c + 1);
#pragma unroll
            for (int k = 0; k < T; ++k) {
                int v = __mul24(sc0, d[c & 1][k][0]);
                v = __mul24(sc1, d[c & 1][k][1]) + v;
                v = __mul24(sc2, d[c & 1][k][2]) + v;
                acc[k][c] = __mul24(sc3, d[c & 1][k][3]) + v;
            }
        }
#pragma unroll
        for (int k = 0; k < T; ++k) {
            int ae, ao;
            reduce_classes(acc[k], ae, ao);
            const float dd = f16_bits_to_f32(r.dh) * r.ad[k];
            se[k] = se[k] + dd * (float)ae;
            so[k] = so[k] + dd * (float)ao;
        }
    };
    const int last = p.blocks - 1;
    load(ra, 0);
    for (int b = 0; b < p.blocks; b += 2) {
        load(rb, min(b + 1, last));
        add(ra);
        if (b == last) break;
        load(ra, min(b + 2, last));
        add(rb);
    }
    const int row = t * TILE_ROWS + n;
#pragma unroll
    for (int k = 0; k < T; ++k) {
        // lane (n, 0) adds the eight class sums in class order (dot.rs:195)
        float tot = -0.0f;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            tot = tot + __shfl(se[k], n + 16 * q, WAVE);
            tot = tot + __shfl(so[k], n + 16 * q, WAVE);
        }
        if (s == 0 && row < p.rows)
            p.y[(size_t)(p.pair_out ? p.pair_out[it.start + k] : it.start + k) * p.ldy + row] = tot;
    }
}

// (tiles % 4 == 0: the workgroup's 4 items share their twin, so its exits are
// uniform and no barrier is skipped by some waves only)
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3))) void q6k_mv_batched_twin_staged(BatchParams pk) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    BatchParams p;
    const int item = batch_item<false>(pk, p, (int)blockIdx.x * 4 + wave);
    if (item >= p.items_per_mat) return;
    const GroupItem it = p.twin_info[item / p.tiles];
    if (it.expert < 0) return;
    if (it.twin2) exact_tile_staged<2>(p, it, lane, wave, item % p.tiles);
    else exact_tile_staged<1>(p, it, lane, wave, item % p.tiles);
}

// The same by chunks on one group of tokens (LM head of 151936 rows, 16
// sequences: 75.7 -> 70.3 us a call; of 32003: 22.4 -> 20.9; QKV of 96 tokens
// 22.4 -> 21.0, of 512 61.7, 61.8; the whole chunk in LDS before the first
// block: 73.9, 23.2). Items count staged_slots(tiles) tiles to a chunk, so that a
// workgroup's four share their chunk; the waves past the last tile only stage
// (8200 rows, 40 sequences: 16.8 us; 17.8 by a wave per item, which reads its
// planes from L2 by itself).
__host__ __device__ constexpr int staged_slots(int tiles) { return (tiles + 3) & ~3; }

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 4))) void q6k_mv_batched_staged(BatchParams pk) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    BatchParams p;
    const int item = batch_item<true>(pk, p, (int)blockIdx.x * 4 + wave);
    const int chunk = item / staged_slots(p.tiles), t = item % staged_slots(p.tiles);
    if (CHUNK_TOKENS * chunk >= p.single_count) return;
    const GroupItem it = {0, chunk, chunk, t < p.tiles ? p.single_count : 0, 0, 0, 0, 0};
    exact_tile_staged<1, true>(p, it, lane, wave, min(t, p.tiles - 1));
}

// The same by chunks, for calls that leave most experts a token or two.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 4))) void q6k_mv_batched_few(BatchParams pk) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    BatchParams p;
    const int item = batch_item<false>(pk, p, (int)blockIdx.x * 4 + wave);
    if (item >= p.items_per_mat) return;
    const GroupItem it = p.sub_info[item / p.tiles];
    if (it.expert < 0) return;
    if (it.count == 1) few_tile<1>(p, it, lane, item % p.tiles);
    else if (it.count == 2) few_tile<2>(p, it, lane, item % p.tiles);
    else exact_tile_staged<1, true>(p, it, lane, wave, item % p.tiles);
}

template <int NC>
__device__ __forceinline__ void fast_tile_staged(const BatchParams &p, int lane, int wave, int t,
                                                 int sub0, int expert, float acc[2][4]) {
    const int n = lane & 15, s = lane >> 4;
    const uint8_t *seg = p.w + (size_t)expert * p.expert_stride + (size_t)t * p.blocks * SEG_BYTES;
    const size_t chunk_q = (size_t)p.blocks * CHUNK_BLOCK_BYTES, chunk_d = (size_t)p.blocks * CHUNK_TOKENS;
    const int8_t *gq = p.act_q + (size_t)sub0 * chunk_q;
    const float *ad = p.act_d + (size_t)sub0 * chunk_d + n;
    int8_t *lds = (int8_t *)g_act_lds;  // [2][NC][4096]
    constexpr int BUF = NC * CHUNK_BLOCK_BYTES;
    // this wave's share of a block's planes: NC KiB, one 16-byte piece per lane
    auto stage = [&](int b) {
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const int off = (wave * NC + i) * 1024;  // within the NC x 4 KiB
            const int u = off / CHUNK_BLOCK_BYTES, o = off % CHUNK_BLOCK_BYTES;
            __builtin_amdgcn_global_load_lds(
                (const void *)(gq + u * chunk_q + (size_t)b * CHUNK_BLOCK_BYTES + o + 16 * lane),
                (lds_ptr)(lds + (b & 1) * BUF + off), 16, 0, 0);
        }
    };
    struct W {
        uint4 q0, q1, q2;
        uint32_t scw;
        uint2 dw;
        float adb[NC];
    };
    auto wload = [&](W &r, int b) {
        const uint8_t *sg = seg + (size_t)b * SEG_BYTES;
        r.q0 = *(const uint4 *)(sg + 16 * lane);
        r.q1 = *(const uint4 *)(sg + SEG_PART + 16 * lane);
        r.q2 = *(const uint4 *)(sg + 2 * SEG_PART + 16 * lane);
        r.scw = *(const uint32_t *)(sg + SEG_SC + 4 * lane);
        r.dw = *(const uint2 *)(sg + SEG_D + 8 * s);
#pragma unroll
        for (int u = 0; u < NC; ++u) r.adb[u] = ad[u * chunk_d + (size_t)b * CHUNK_TOKENS];
    };
    auto compute = [&](const W &r, int b) {
        const int8_t *aq = lds + (b & 1) * BUF + 16 * lane;
        const uint32_t nib[8] = {r.q0.x, r.q0.y, r.q0.z, r.q0.w, r.q1.x, r.q1.y, r.q1.z, r.q1.w};
        const uint32_t hb[4] = {r.q2.x, r.q2.y, r.q2.z, r.q2.w};
        const FoldScales fs = fold_scales(r.scw);
        const v4i zero = {0, 0, 0, 0};
        v4i ah[NC], al[NC];
#pragma unroll
        for (int u = 0; u < NC; ++u) ah[u] = al[u] = zero;
#pragma unroll
        for (int P = 0; P < 4; ++P) {
            v4i a_lo, a_hi;
            fold_pair(nib, hb, P, fs, a_lo, a_hi);
#pragma unroll
            for (int u = 0; u < NC; ++u) {
                const v4i av = *(const v4i *)(aq + u * CHUNK_BLOCK_BYTES + 1024 * P);
                ah[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a_hi, av, ah[u], 0, 0, 0);
                al[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a_lo, av, al[u], 0, 0, 0);
            }
        }
        const float d4[4] = {f16_bits_to_f32((uint16_t)(r.dw.x & 0xFFFF)), f16_bits_to_f32((uint16_t)(r.dw.x >> 16)),
                             f16_bits_to_f32((uint16_t)(r.dw.y & 0xFFFF)), f16_bits_to_f32((uint16_t)(r.dw.y >> 16))};
#pragma unroll
        for (int u = 0; u < NC; ++u)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int aux = ah[u][v] * 256 + al[u][v];
                acc[u][v] = __builtin_fmaf(d4[v] * r.adb[u], (float)aux, acc[u][v]);
            }
    };
    // the block's planes must be in LDS (this wave's pieces landed, every
    // wave past the barrier) before any wave reads them; the barrier also
    // keeps a buffer from being refilled while a wave still reads it
    auto handover = [&]() {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    };
    const int last = p.blocks - 1;
    W ra, rb;
    stage(0);
    wload(ra, 0);
    handover();
    for (int b = 0; b < p.blocks; b += 2) {
        if (b + 1 <= last) stage(b + 1);
        wload(rb, min(b + 1, last));
        __builtin_amdgcn_sched_barrier(0);
        compute(ra, b);
        handover();
        if (b + 1 > last) break;
        if (b + 2 <= last) stage(b + 2);
        wload(ra, min(b + 2, last));
        __builtin_amdgcn_sched_barrier(0);
        compute(rb, b + 1);
        handover();
    }
}

// One wave per (unit, tile), 4 tiles of one unit per workgroup; TWIN as in
// q6k_mv_batched_fast. Dynamic LDS: 2 x (TWIN ? 2 : 1) x 4 KiB.
template <bool TWIN>
__global__ __launch_bounds__(256) void q6k_mv_batched_fast_staged(BatchParams pk) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n = lane & 15, s = lane >> 4;
    int item = (int)blockIdx.x * 4 + wave;
    BatchParams p = pk;
    if (p.w2 && item >= p.items_per_mat) {
        item -= p.items_per_mat;
        p.w = p.w2;
        p.y = p.y2;
    }
    // the workgroup's 4 items share their unit (tiles % 4 == 0), so these
    // exits are uniform over the workgroup and no barrier below is skipped
    // by some waves only
    if (item >= p.items_per_mat) return;
    const int t = item % p.tiles;
    const GroupItem it = TWIN ? p.twin_info[item / p.tiles] : p.sub_info[item / p.tiles];
    if (it.expert < 0) return;
    const int nc = TWIN && it.twin2 ? 2 : 1;
    float acc[2][4] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
    if (nc == 2) fast_tile_staged<2>(p, lane, wave, t, it.sub, it.expert, acc);
    else fast_tile_staged<1>(p, lane, wave, t, it.sub, it.expert, acc);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        if (u >= nc) break;
        const int tok = 16 * (it.st + u) + n;
        if (tok >= it.count) continue;
        const int pos = it.start + tok;
        const int orow = p.pair_out ? p.pair_out[pos] : pos;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int row = t * TILE_ROWS + 4 * s + v;
            if (row < p.rows) p.y[(size_t)orow * p.ldy + row] = acc[u][v];
        }
    }
}

// The grouped kernel for experts with many tokens: a workgroup takes up to
// WIDE_CHUNKS 16-token chunks of one expert (a unit) against 8 waves of one
// 16-row tile each. A wave folds a block of its tile into digits once (32
// registers) and runs them against every chunk, whose planes all 8 waves read
// from LDS (double-buffered direct global-to-LDS copies, one barrier per
// block), so the fold costs a quarter of what it costs a twin and a plane is
// read from L2 once per 128 rows. PAIR: waves 0..3 and 4..7 take the same rows
// of gate and up, and the output is silu(gate) * up (up through LDS).
// 128 registers: four waves a SIMD, so that folds, MFMAs and float epilogues
// of different waves overlap (two tiles a wave halve the LDS reads but leave
// two waves a SIMD: the same at 2000 tokens, 2-3% slower at 100-512; 16 chunks
// a unit leave one workgroup a CU: 453 us instead of 367 at 2000).
// At 2000 tokens the copies and stores alone take 65% of the time and the
// arithmetic alone 65%; gate + up 185 us, down 100 (traced 350 and 190 as twins).
// A unit's workgroups run on one XCD (workgroup i on XCD i % 8), which then
// reads the unit's planes and each weight once.
constexpr int WIDE_CHUNKS = GROUP_WIDE_CHUNKS;

template <bool PAIR>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4, 4))) void q6k_mv_batched_wide(
    BatchParams p, int row_groups) {
    __shared__ float ds[WIDE_MAX_BLOCKS][WIDE_CHUNKS * 16];
    __shared__ uint64_t tab[32];
    const int lane = threadIdx.x & 63, n = lane & 15, s = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = blockIdx.x / 8;
    const int unit = (q / row_groups) * 8 + blockIdx.x % 8, rg = q % row_groups;
    const GroupItem it = p.wide_info[unit];
    if (it.expert < 0) return;
    const int nc = it.twin2;
    const int t = PAIR ? rg * 4 + (wave & 3) : rg * 8 + wave;
    const bool live = t < p.tiles;  // (a wave past the last tile works on the last one and stores nothing)
    const uint8_t *seg = (PAIR && wave >= 4 ? p.w2 : p.w) + (size_t)it.expert * p.expert_stride +
                         (size_t)min(t, p.tiles - 1) * p.blocks * SEG_BYTES;
    const size_t chunk_q = (size_t)p.blocks * CHUNK_BLOCK_BYTES, chunk_d = (size_t)p.blocks * CHUNK_TOKENS;
    int8_t *lds = (int8_t *)g_act_lds;  // [2][WIDE_CHUNKS][4096]
    // plane wave % 4 of every second chunk of block b, 16 bytes a lane
    const int u0 = wave >> 2, po = 1024 * (wave & 3);
    const int8_t *gq = p.act_q + (size_t)(it.sub + u0) * chunk_q + po + 16 * lane;
    auto stage = [&](int b) {
#pragma unroll
        for (int u = 0; u < WIDE_CHUNKS; u += 2)
            if (u + u0 < nc)
                __builtin_amdgcn_global_load_lds(
                    (const void *)(gq + u * chunk_q + (size_t)b * CHUNK_BLOCK_BYTES),
                    (lds_ptr)(lds + ((b & 1) * WIDE_CHUNKS + u + u0) * CHUNK_BLOCK_BYTES + po), 16, 0, 0);
    };
    struct W {
        uint4 q0, q1, q2;
        uint32_t scw;
        uint2 dw;
    } w;
    auto wload = [&](int b) {
        const uint8_t *sg = seg + (size_t)b * SEG_BYTES;
        w.q0 = *(const uint4 *)(sg + 16 * lane);
        w.q1 = *(const uint4 *)(sg + SEG_PART + 16 * lane);
        w.q2 = *(const uint4 *)(sg + 2 * SEG_PART + 16 * lane);
        w.scw = *(const uint32_t *)(sg + SEG_SC + 4 * lane);
        w.dw = *(const uint2 *)(sg + SEG_D + 8 * s);  // f16 d of rows 4s..4s+3
    };
    stage(0);
    wload(0);
    // every block's scales of the unit's tokens
    for (int i = threadIdx.x; i < nc * (int)chunk_d; i += 512) {
        const int u = i / (int)chunk_d, r = i % (int)chunk_d;
        ds[r / 16][u * 16 + r % 16] = p.act_d[(size_t)it.sub * chunk_d + i];
    }
    if (PAIR && wave == 0) expf_ref_tab_fill(tab);
    float acc[WIDE_CHUNKS][4];
#pragma unroll
    for (int u = 0; u < WIDE_CHUNKS; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[u][v] = 0.0f;
    for (int b = 0; b < p.blocks; ++b) {
        v4i lo[4], hi[4];
        {
            const uint32_t nib[8] = {w.q0.x, w.q0.y, w.q0.z, w.q0.w, w.q1.x, w.q1.y, w.q1.z, w.q1.w};
            const uint32_t hb[4] = {w.q2.x, w.q2.y, w.q2.z, w.q2.w};
            const FoldScales fs = fold_scales(w.scw);
#pragma unroll
            for (int P = 0; P < 4; ++P) fold_pair(nib, hb, P, fs, lo[P], hi[P]);
        }
        const float d4[4] = {f16_bits_to_f32((uint16_t)(w.dw.x & 0xFFFF)), f16_bits_to_f32((uint16_t)(w.dw.x >> 16)),
                             f16_bits_to_f32((uint16_t)(w.dw.y & 0xFFFF)), f16_bits_to_f32((uint16_t)(w.dw.y >> 16))};
        // this wave's pieces of block b have landed (with its weights, used
        // above); past the barrier everyone's have, and the other buffer is read
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (b + 1 < p.blocks) {
            stage(b + 1);
            wload(b + 1);
        }
        __builtin_amdgcn_sched_barrier(0);
        const int8_t *aq = lds + (b & 1) * WIDE_CHUNKS * CHUNK_BLOCK_BYTES + 16 * lane;
#pragma unroll
        for (int u = 0; u < WIDE_CHUNKS; ++u) {
            if (u < nc) {
                const v4i zero = {0, 0, 0, 0};
                v4i ah = zero, al = zero;
#pragma unroll
                for (int P = 0; P < 4; ++P) {
                    const v4i av = *(const v4i *)(aq + u * CHUNK_BLOCK_BYTES + 1024 * P);
                    ah = __builtin_amdgcn_mfma_i32_16x16x64_i8(hi[P], av, ah, 0, 0, 0);
                    al = __builtin_amdgcn_mfma_i32_16x16x64_i8(lo[P], av, al, 0, 0, 0);
                }
                const float adb = ds[b][u * 16 + n];
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int aux = ah[v] * 256 + al[v];
                    acc[u][v] = __builtin_fmaf(d4[v] * adb, (float)aux, acc[u][v]);
                }
            }
        }
    }
    if constexpr (PAIR) {
        // up's sums to gate's waves, in the buffers of the planes
        __syncthreads();
        float4 *ex = (float4 *)g_act_lds + (wave & 3) * WIDE_CHUNKS * 64 + lane;
        if (wave >= 4) {
#pragma unroll
            for (int u = 0; u < WIDE_CHUNKS; ++u)
                if (u < nc) ex[u * 64] = make_float4(acc[u][0], acc[u][1], acc[u][2], acc[u][3]);
        }
        __syncthreads();
        if (wave >= 4) return;
#pragma unroll
        for (int u = 0; u < WIDE_CHUNKS; ++u)
            if (u < nc) {
                const float4 up = ex[u * 64];
                acc[u][0] = silu_ref(acc[u][0], tab) * up.x;
                acc[u][1] = silu_ref(acc[u][1], tab) * up.y;
                acc[u][2] = silu_ref(acc[u][2], tab) * up.z;
                acc[u][3] = silu_ref(acc[u][3], tab) * up.w;
            }
    }
    if (!live) return;
#pragma unroll
    for (int u = 0; u < WIDE_CHUNKS; ++u) {
        const int tok = 16 * (it.st + u) + n;
        if (u < nc && tok < it.count) {
            const int pos = it.start + tok;
            const int orow = p.pair_out ? p.pair_out[pos] : pos;
            // (p.rows % 16 == 0, rows 16-byte aligned: checked at launch)
            *(float4 *)(p.y + (size_t)orow * p.ldy + t * TILE_ROWS + 4 * s) =
                make_float4(acc[u][0], acc[u][1], acc[u][2], acc[u][3]);
        }
    }
}

// ---- LM head: certified arg-max over REDUCTION-tolerance logits -------------
//
// The fast batched kernel's logit F_r of row r and the reference's E_r are two
// roundings of the same real value T_r = sum_b dd_b * sum_c aux_b[c] (dd_b =
// f16(d_b) * a.d_b, the same float in both; aux integers exact in both):
//   |E_r - T_r| <= gamma_{nb+10} S_r  (8 class sums of nb rounded products,
//                                     then the 8-term class sum)
//   |F_r - T_r| <= gamma_{nb+1} S_r   (nb fused multiply-adds)
// with S_r = sum_b |dd_b| sum_c |aux_b[c]| <= 127 (1 + u) sum_b |a.d_b|
// |f16(d_b)| sum_e |sc(e)(q_e - 32)| <= 127 (1 + u) D_a M_r, since every Q8_K
// quant is at most 127 in magnitude; D_a = max_b |a.d_b| of the token and M_r
// the weights' own sum, bounded per tile by q6k_tile_bound. So
// |F_r - E_r| <= delta_t = 2 (2 nb + 12) u 127 D_a M_t (+ 2^-20 |F|, covering
// the bound's own float rounding) for every row r of tile t (u = 2^-24).
// Every row whose E_r could be the maximum then lies in a tile with
// F_t + delta_t >= L = max_t (F_t - delta_t), F_t the tile's largest F.

// One wave per tile.
__global__ __launch_bounds__(256) void q6k_tile_bound(const uint8_t *w, int tiles, int blocks,
                                                      float *mt) {
    const int lane = threadIdx.x & 63, t = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= tiles) return;
    const int n = lane & 15;
    float m = 0.0f;
    for (int b = 0; b < blocks; ++b) {
        const uint8_t *sg = w + ((size_t)t * blocks + b) * SEG_BYTES;
        const uint4 q0 = *(const uint4 *)(sg + 16 * lane);
        const uint4 q1 = *(const uint4 *)(sg + SEG_PART + 16 * lane);
        const uint4 q2 = *(const uint4 *)(sg + 2 * SEG_PART + 16 * lane);
        const uint32_t scw = *(const uint32_t *)(sg + SEG_SC + 4 * lane);
        const uint16_t dh = *(const uint16_t *)(sg + SEG_D + 2 * n);
        const uint32_t nib[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
        const uint32_t hb[4] = {q2.x, q2.y, q2.z, q2.w};
        // the lane's 64 weights of row n: class c, byte kk = weight 8 (8 s + kk) + c,
        // scale group 4 s + kk / 2 (byte kk / 2 of scw)
        int acc = 0;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const uint64_t codes = (uint64_t)unpack_codes(nib, hb, c);
#pragma unroll
            for (int kk = 0; kk < 8; ++kk) {
                const int q = (int)((codes >> (8 * kk)) & 0xFF) - 32;
                const int sc = __builtin_amdgcn_sbfe(scw, 8 * (kk >> 1), 8);
                acc += abs(sc * q);
            }
        }
        acc += __shfl_xor(acc, 16, WAVE);
        acc += __shfl_xor(acc, 32, WAVE);
        m += fabsf(f16_bits_to_f32(dh)) * (float)acc;  // acc <= 2^20: exact
    }
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) m = fmaxf(m, __shfl_xor(m, o, WAVE));
    if (lane == 0) mt[t] = m;
}

struct CertifyParams {
    const uint8_t *w;      // tiled Q6_K [rows x blocks]
    const int8_t *nq;      // [nseq][blocks * 256] natural Q8_K
    const float *nd;       // [nseq][blocks]
    const float *pv;       // [nseq][tiles] the fast kernel's tile candidates
    const int *pi;         //   (row, or -1: a NaN logit in the tile)
    const float *mt;       // [tiles] q6k_tile_bound
    float *logits;         // [nseq][rows]
    int32_t *ids;          // [nseq]
    int rows, tiles, blocks;
};

// One 1024-thread workgroup per token. Its tiles' candidates are read once
// (CERT_PT per thread kept in registers), the candidate tiles gathered in LDS,
// and their exact recomputation spread over the 16 waves by (tile, block):
// each wave computes one block's eight class terms of one tile into LDS (a
// single round trip to memory for up to 16 / blocks tiles), then one wave per
// tile folds them in block order, as dot_q6k_q8k does (the q6k_mv_b1 split-K
// fold).
constexpr int CERT_PT = 16;     // tiles per thread held in registers (beyond: re-read)
constexpr int CERT_CAP = 1024;  // candidate list; more (no certificate) -> every tile
constexpr int CERT_MAXB = 32;   // blocks per row (k <= 8192)

__global__ __launch_bounds__(1024) void lmhead_certify(CertifyParams p) {
    const int u = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = lane & 15, s = lane >> 4;
    const float *F = p.pv + (size_t)u * p.tiles;
    const int *FI = p.pi + (size_t)u * p.tiles;
    const float *ad = p.nd + (size_t)u * p.blocks;
    const int8_t *aq = p.nq + (size_t)u * p.blocks * QK_K;
    __shared__ float s_lo[16];
    __shared__ int s_bad[16];
    __shared__ int s_cand[CERT_CAP];
    __shared__ int s_ncand;
    // per round: entry e = (tile e / blocks, block e % blocks), CERT_MAXB / blocks tiles
    __shared__ float s_terms[CERT_MAXB][TILE_ROWS][8];
    if (tid == 0) s_ncand = 0;
    // 1. the certified lower bound L of the largest exact logit
    float fv[CERT_PT], dv[CERT_PT];
    float lo = -INFINITY;
    int bad = 0;
    float da, cst;
    {
        // all of the thread's loads in flight at once: unconditional, at a
        // clamped index, the out-of-range ones discarded afterwards
        int fi[CERT_PT];
        float mv[CERT_PT];
#pragma unroll
        for (int i = 0; i < CERT_PT; ++i) {
            const int t = min(tid + i * (int)blockDim.x, p.tiles - 1);
            fv[i] = F[t];
            mv[i] = p.mt[t];
            fi[i] = FI[t];
        }
        // D_a = max_b |a.d_b|: one load per lane (blocks <= 32), a wave max
        da = lane < p.blocks ? fabsf(ad[lane]) : 0.0f;
#pragma unroll
        for (int o = 1; o < WAVE; o <<= 1) da = fmaxf(da, __shfl_xor(da, o, WAVE));
        cst = 2.0f * (float)(2 * p.blocks + 12) * 0x1p-24f * 127.0f * da;
#pragma unroll
        for (int i = 0; i < CERT_PT; ++i) {
            if (tid + i * (int)blockDim.x >= p.tiles) continue;
            dv[i] = cst * mv[i] + 0x1p-20f * fabsf(fv[i]);
            if (!isfinite(fv[i]) || !isfinite(dv[i]) || fi[i] < 0) bad = 1;
            else lo = fmaxf(lo, fv[i] - dv[i]);
        }
    }
    for (int t = tid + CERT_PT * (int)blockDim.x; t < p.tiles; t += blockDim.x) {
        const float f = F[t], d = cst * p.mt[t] + 0x1p-20f * fabsf(f);
        if (!isfinite(f) || !isfinite(d) || FI[t] < 0) bad = 1;
        else lo = fmaxf(lo, f - d);
    }
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
        lo = fmaxf(lo, __shfl_xor(lo, o, WAVE));
        bad |= __shfl_xor(bad, o, WAVE);
    }
    if (lane == 0) { s_lo[wave] = lo; s_bad[wave] = bad; }
    __syncthreads();
    for (int w = 0; w < 16; ++w) { lo = fmaxf(lo, s_lo[w]); bad |= s_bad[w]; }
    // 2. the candidate tiles (tile 0 always: the reference's incumbent is row 0)
    if (!bad) {
        auto keep = [&](int t, float f, float d) {
            if (t == 0 || f + d >= lo) {
                const int at = atomicAdd(&s_ncand, 1);
                if (at < CERT_CAP) s_cand[at] = t;
            }
        };
#pragma unroll
        for (int i = 0; i < CERT_PT; ++i) {
            const int t = tid + i * (int)blockDim.x;
            if (t < p.tiles) keep(t, fv[i], dv[i]);
        }
        for (int t = tid + CERT_PT * (int)blockDim.x; t < p.tiles; t += blockDim.x)
            keep(t, F[t], cst * p.mt[t] + 0x1p-20f * fabsf(F[t]));
    }
    __syncthreads();
    const bool all = bad || s_ncand > CERT_CAP;
    const int total = all ? p.tiles : s_ncand;
    // 3. exact recomputation, (tile, block) pairs over the waves: up to
    // CERT_MAXB pairs per round, two per wave with both pairs' loads in
    // flight together (a round is one memory round trip)
    // tiles per round: a wave folds each (blocks <= CERT_MAXB, checked at launch)
    const int per = min(16, CERT_MAXB / p.blocks);
    const int pairs = per * p.blocks;
    const MaskSel msel = mask_selectors(n, (n >> 2) == s);
    float bv = -INFINITY;
    int bi = 0x7FFFFFFF;
    int nan0 = 0;
    for (int r0 = 0; r0 < total; r0 += per) {
        float se = 0.0f, so = 0.0f;
        for (int e0 = wave; e0 < pairs; e0 += 32) {
            BlockRegs r[2];
            bool ok[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int e = e0 + 16 * h;
                const int ci = r0 + e / p.blocks, b = e % p.blocks;
                ok[h] = e < pairs && ci < total;
                if (ok[h]) {
                    const int tt = all ? ci : s_cand[ci];
                    load_block(r[h], p.w + ((size_t)tt * p.blocks + b) * SEG_BYTES, aq, ad, b, lane, n);
                }
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (!ok[h]) continue;
                const int e = e0 + 16 * h;
                float te, to;
                block_terms(r[h], msel, te, to);
                const int slot = e;
                s_terms[slot][n][2 * s] = te;
                s_terms[slot][n][2 * s + 1] = to;
            }
        }
        __syncthreads();
        if (wave < per && r0 + wave < total) {
            const int tt = all ? r0 + wave : s_cand[r0 + wave];
            const int base = wave * p.blocks;
            for (int b = 0; b < p.blocks; ++b) {
                se = se + s_terms[base + b][n][2 * s];
                so = so + s_terms[base + b][n][2 * s + 1];
            }
            float cls[8];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                cls[2 * q] = __shfl(se, n + 16 * q, WAVE);
                cls[2 * q + 1] = __shfl(so, n + 16 * q, WAVE);
            }
            float tot = -0.0f;
#pragma unroll
            for (int c = 0; c < 8; ++c) tot = tot + cls[c];
            const int row = tt * TILE_ROWS + n;
            if (s == 0 && row < p.rows) {
                p.logits[(size_t)u * p.rows + row] = tot;
                if (!isnan(tot)) argmax_step(bv, bi, tot, row);
                if (row == 0 && isnan(tot)) nan0 = 1;
            }
        }
        __syncthreads();
    }
    wave_argmax(bv, bi, -INFINITY);
    nan0 = __ballot(nan0 != 0) != 0 ? 1 : 0;
    __shared__ float s_bv[16];
    __shared__ int s_bi[16], s_nan[16];
    if (lane == 0) { s_bv[wave] = bv; s_bi[wave] = bi; s_nan[wave] = nan0; }
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < 16; ++w) {
            argmax_step(bv, bi, s_bv[w], s_bi[w]);
            nan0 |= s_nan[w];
        }
        p.ids[u] = (nan0 || bi == 0x7FFFFFFF) ? 0 : bi;
    }
}

// y = W . Q8_K(x) with x in f32 (the long-context decode step's O
// projection, whose activation comes from the attention as f32): the bits of
// launch_q8k_quantize + q6k_mv_b1<8> in one launch. One 16-row tile per
// 8-wave workgroup; wave k quantizes the blocks it multiplies, [bpc k,
// bpc k + bpc), with quantize_wave into its own LDS rows while its weight
// loads are in flight; the per-block terms are folded in block order.
constexpr int F32X_MAX_BLOCKS = 16;

__global__ __launch_bounds__(512) void q6k_mv_f32x(const uint8_t *w, const float *x, float *y,
                                                   int rows, int blocks) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 15, s = lane >> 4;
    const int t = blockIdx.x;
    const int bpc = (blocks + 7) / 8;  // at most 2
    const int b0 = wave * bpc, b1 = min(blocks, b0 + bpc);
    __shared__ float terms[F32X_MAX_BLOCKS][TILE_ROWS][8];
    __shared__ __align__(16) int8_t lq[F32X_MAX_BLOCKS * QK_K];
    __shared__ float ld[F32X_MAX_BLOCKS];
    const uint8_t *seg = w + (size_t)t * blocks * SEG_BYTES;
    BlockRegs r[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
        if (i < bpc) load_weights(r[i], seg + (size_t)min(b0 + i, blocks - 1) * SEG_BYTES, lane, n);
    float4 xv[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
        if (i < bpc) xv[i] = *(const float4 *)(x + (size_t)min(b0 + i, blocks - 1) * QK_K + 4 * lane);
#pragma unroll
    for (int i = 0; i < 2; ++i)
        if (i < bpc && b0 + i < b1) {
            const float v[4] = {xv[i].x, xv[i].y, xv[i].z, xv[i].w};
            quantize_wave(v, lane, lq + (b0 + i) * QK_K, ld + b0 + i, nullptr);
        }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    const MaskSel msel = mask_selectors(n, (n >> 2) == s);
#pragma unroll
    for (int i = 0; i < 2; ++i)
        if (i < bpc && b0 + i < b1) {
            r[i].g = *(const uint4 *)(lq + (b0 + i) * QK_K + 16 * n);
            r[i].ad = ld[b0 + i];
            float te, to;
            block_terms(r[i], msel, te, to);
            terms[b0 + i][n][2 * s] = te;
            terms[b0 + i][n][2 * s + 1] = to;
        }
    __syncthreads();
    if (wave != 0) return;
    float se = 0.0f, so = 0.0f;
    for (int b = 0; b < blocks; ++b) {
        se = se + terms[b][n][2 * s];
        so = so + terms[b][n][2 * s + 1];
    }
    float cls[8];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        cls[2 * q] = __shfl(se, n + 16 * q, WAVE);
        cls[2 * q + 1] = __shfl(so, n + 16 * q, WAVE);
    }
    const int row = t * TILE_ROWS + n;
    float tot = -0.0f;
#pragma unroll
    for (int c = 0; c < 8; ++c) tot = tot + cls[c];
    if (s == 0 && row < rows) y[row] = tot;
}

}  // namespace

int g_tune_mv_ks = 0;
int g_tune_batched_twin = 1;
int g_tune_fast_ks = 0;
int g_tune_fast_lds = 1;

namespace {

// Fills the segment table for n matrices sharing `rows`-independent shapes.
void set_segments(MvParams &p, int n, const void *const *w, float *const *y, const int *rows,
                  int n_slots) {
    MvSeg *seg[3] = {&p.seg0, &p.seg1, &p.seg2};
    int first = 0;
    p.n_seg = n;
    for (int i = 0; i < n; ++i) {
        seg[i]->w = (const uint8_t *)w[i];
        seg[i]->y = y[i];
        seg[i]->rows = rows[i];
        seg[i]->tiles = (rows[i] + TILE_ROWS - 1) / TILE_ROWS;
        seg[i]->first = first;
        first += seg[i]->tiles * n_slots;
    }
    for (int i = n; i < 3; ++i) *seg[i] = p.seg0;
    p.items = first;
    p.n_slots = n_slots;
}

// q6k_mv_b1's preloaded leading arguments, then the whole parameter block
#define B1_ARGS(p) (p).seg0.w, (p).aq, (p).ad, (p).ids, (p).blocks, (p).seg0.tiles, (p).items, \
                   (p).act_per_slot, (p)
// ... or, for the plain matvec, the compact one
#define B1_LITE(p) (p).seg0.w, (p).aq, (p).ad, (p).ids, (p).blocks, (p).seg0.tiles, (p).items, \
                   (p).act_per_slot, MvLite{(p).seg0.y, (p).expert_stride, (p).clk, (p).seg0.rows, (p).n_slots}

template <int NSEG, bool AMAX = false>
void launch_b1_n(const MvParams &p, hipStream_t st) {
    const int items = p.items;
    // Measured on MI355X: eight waves per tile (one block each at k = 2048)
    // win while the grid is small -- 768 x 2048: 3.46 -> 3.17 us, 4096 x
    // 2048: 4.14 -> 3.82 us -- and lose from ~1000 tiles on (LM head 41 ->
    // 52 us), where four waves already fill the machine.
    // Short rows (at most 4 blocks, down's k = 768) in a large grid go the
    // other way: one wave per tile walks all of its blocks. 128 down
    // matrices [2048 x 768] in one grouped launch: 44.0 -> 29.9 us with one
    // wave per tile; 8 of them (1024 tiles): 3.80 -> 3.48 us; below ~1000
    // tiles four waves stay ahead (512 tiles: 2.98 vs 3.12 us).
    const int ks = g_tune_mv_ks ? g_tune_mv_ks
                                : (p.blocks > 4 && items <= 384 ? 8 : (p.blocks <= 4 && items >= 1024 ? 1 : 0));
    constexpr bool LITE = NSEG == 1 && !AMAX;
    if (p.blocks <= 16 && (ks == 4 || ks == 8 || ks == 0)) {
        if (ks == 8) {
            if constexpr (LITE)
                hipLaunchKernelGGL((q6k_mv_b1<8, false, 1, false, MvLite>), dim3(items), dim3(512), 0, st, B1_LITE(p));
            else
                hipLaunchKernelGGL((q6k_mv_b1<8, false, NSEG, AMAX>), dim3(items), dim3(512), 0, st, B1_ARGS(p));
        } else {
            // Measured on MI355X (gate/up/down/q_proj/LM-head shapes): four
            // waves per tile, each on a quarter of the row, beat one wave per
            // tile -- more loads in flight per tile and shorter per-wave
            // chains -- except for short rows in large grids (above).
            if constexpr (LITE)
                hipLaunchKernelGGL((q6k_mv_b1<4, false, 1, false, MvLite>), dim3(items), dim3(256), 0, st, B1_LITE(p));
            else
                hipLaunchKernelGGL((q6k_mv_b1<4, false, NSEG, AMAX>), dim3(items), dim3(256), 0, st, B1_ARGS(p));
        }
    } else {
        if constexpr (LITE)
            hipLaunchKernelGGL((q6k_mv_b1<1, false, 1, false, MvLite>), dim3((items + 3) / 4), dim3(256), 0, st, B1_LITE(p));
        else
            hipLaunchKernelGGL((q6k_mv_b1<1, false, NSEG, AMAX>), dim3((items + 3) / 4), dim3(256), 0, st, B1_ARGS(p));
    }
}

// llamd_hip_kernel_clock: slots [n][2] for the q6k_mv_b1 launches, in turn
unsigned long long *g_clk_slots = nullptr;
int g_clk_n = 0, g_clk_next = 0;

int launch_b1(const MvParams &pin, hipStream_t st) {
    MvParams p = pin;
    if (g_clk_slots) {
        p.clk = g_clk_slots + 2 * (size_t)CLOCK_WAVES * g_clk_next;
        g_clk_next = (g_clk_next + 1) % g_clk_n;
    }
    if (p.amax_v) launch_b1_n<1, true>(p, st);  // LM head: one segment, one slot
    else if (p.n_seg == 1) launch_b1_n<1>(p, st);
    else if (p.n_seg == 2) launch_b1_n<2>(p, st);
    else launch_b1_n<3>(p, st);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace

int launch_q6k_mv_b1(const void *w, size_t expert_stride, const int32_t *ids, const int8_t *aq,
                     const float *ad, float *y, int rows, int blocks, int n_slots, int act_per_slot,
                     hipStream_t st, const void *w_b, float *amax_v, int *amax_i) {
    if (amax_v && w_b) return -1;
    MvParams p = {};
    p.amax_v = amax_v;
    p.amax_i = amax_i;
    // with a second weight, its outputs follow the first's: y = [w | w_b]
    const void *ws[2] = {w, w_b};
    float *ys[2] = {y, y + (size_t)n_slots * rows};
    const int rs[2] = {rows, rows};
    set_segments(p, w_b ? 2 : 1, ws, ys, rs, n_slots);
    p.expert_stride = expert_stride;
    p.ids = ids;
    p.aq = aq;
    p.ad = ad;
    p.blocks = blocks;
    p.act_per_slot = act_per_slot;
    return launch_b1(p, st);
}

int launch_q6k_mv_x3(const void *const w[3], float *const y[3], const int rows[3], int n_mat,
                     const int8_t *aq, const float *ad, int blocks, hipStream_t st) {
    if (n_mat < 1 || n_mat > 3) return -1;
    MvParams p = {};
    set_segments(p, n_mat, w, y, rows, 1);
    p.aq = aq;
    p.ad = ad;
    p.blocks = blocks;
    return launch_b1(p, st);
}

int launch_q6k_mv_grouped_x2(const void *wa, const void *wb, size_t expert_stride,
                             const int32_t *ids, const int8_t *aq, const float *ad, float *oa,
                             float *ob, int rows, int blocks, int n_used, hipStream_t st,
                             int act_per_slot) {
    MvParams p = {};
    const void *ws[2] = {wa, wb};
    float *ys[2] = {oa, ob};
    const int rs[2] = {rows, rows};
    set_segments(p, 2, ws, ys, rs, n_used);
    p.expert_stride = expert_stride;
    p.ids = ids;
    p.aq = aq;
    p.ad = ad;
    p.blocks = blocks;
    p.act_per_slot = act_per_slot;
    return launch_b1(p, st);
}

int launch_q6k_mv_routed(const void *w, const void *w_b, size_t expert_stride,
                         const float *logits, int n_expert, int n_used, int32_t *ids_out,
                         float *w_out, int *stats, const int8_t *aq, const float *ad, float *y,
                         int rows, int blocks, hipStream_t st) {
    if (blocks > 16 || n_expert > ROUTE_MAX_EXPERTS || n_used > ROUTE_MAX_USED) return -1;
    MvParams p = {};
    const void *ws[2] = {w, w_b};
    float *ys[2] = {y, y + (size_t)n_used * rows};
    const int rs[2] = {rows, rows};
    set_segments(p, 2, ws, ys, rs, n_used);
    p.expert_stride = expert_stride;
    p.aq = aq;
    p.ad = ad;
    p.blocks = blocks;
    p.route_l = logits;
    p.n_expert = n_expert;
    p.n_used = n_used;
    p.ids_out = ids_out;
    p.w_out = w_out;
    p.stats = stats;
    hipLaunchKernelGGL((q6k_mv_b1<4, true, 2>), dim3(p.items), dim3(256), 0, st, B1_ARGS(p));
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

namespace {
// The exact kernels on one group of tokens in `chunks` chunks, items = tiles x
// chunks in all.
int launch_one_group(BatchParams &p, int chunks, long items, hipStream_t st) {
    // half a wave per SIMD or less (us per call with the norm and the quants, a
    // wave per item -> four: 320 items (5120 x 2048) 15.9 -> 14.4, 640 16.3 -> 16.8)
    if (items <= 512 && !p.amax_v) {
        hipLaunchKernelGGL(q6k_mv_batched_classes, dim3((unsigned)items), dim3(256), 0, st, p);
        return hipGetLastError() == hipSuccess ? 0 : -1;
    }
    long slots = 0;
    if (p.n_segs > 0) {
        for (int i = 0; i < p.n_segs; ++i) {
            p.segs[i].first = (int)slots;
            slots += p.segs[i].items = staged_slots(p.segs[i].tiles) * chunks;
        }
    } else {
        p.items_per_mat = staged_slots(p.tiles) * chunks;
        slots = p.w2 ? 2L * p.items_per_mat : p.items_per_mat;
    }
    hipLaunchKernelGGL(q6k_mv_batched_staged, dim3((unsigned)(slots / 4)), dim3(256), 2 * CHUNK_BLOCK_BYTES, st, p);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
}  // namespace

int launch_q6k_mv_batched(const void *w, size_t expert_stride, const GroupItem *records,
                          const int32_t *pair_out, const int8_t *act_q, const float *act_d, float *y,
                          int ldy, int rows, int blocks, int n_groups, int max_chunks, hipStream_t st,
                          float *amax_v, int *amax_i, const void *w2, float *y2, bool fast, bool few) {
    if (amax_v && records) return -1;
    // every item of the grids below indexes a record below max_chunks when
    // max_chunks >= n_groups (twins: ceil((max_chunks + n_groups) / 2) items)
    if (records && max_chunks < n_groups) return -1;
    if (max_chunks <= 0 || rows <= 0) return 0;
    BatchParams p = {};
    if (w2 && (!y2 || amax_v)) return -1;
    p.w2 = (const uint8_t *)w2;
    p.y2 = y2;
    p.sub_info = records;
    p.twin_info = records ? records + max_chunks : nullptr;
    p.single_count = n_groups;  // only read without records
    p.w = (const uint8_t *)w;
    p.expert_stride = expert_stride;
    p.pair_out = pair_out;
    p.act_q = act_q;
    p.act_d = act_d;
    p.y = y;
    p.amax_v = amax_v;
    p.amax_i = amax_i;
    p.ldy = ldy;
    p.rows = rows;
    p.tiles = (rows + TILE_ROWS - 1) / TILE_ROWS;
    p.blocks = blocks;
    // twins: sum of ceil(ch/2) <= (sum of ch + n_groups) / 2
    const bool twin = records && g_tune_batched_twin && (fast || !few);
    const long items = (long)p.tiles * (twin ? (max_chunks + n_groups + 1) / 2 : max_chunks);
    const long all = w2 ? 2 * items : items;
    p.items_per_mat = (int)items;
    if (fast) {
        // K split over ks waves (tune key fast_ks): one measured best on
        // MI355X for both the prefill and the LM head shapes
        const int ks = g_tune_fast_ks ? g_tune_fast_ks : 1;
        const unsigned grid = (unsigned)((all * ks + 3) / 4);
        const size_t lds = (size_t)blocks * CHUNK_BLOCK_BYTES;
        if (records && ks == 1 && p.tiles % 4 == 0 && g_tune_fast_lds) {
            const size_t slds = (size_t)2 * (twin ? 2 : 1) * CHUNK_BLOCK_BYTES;
            if (twin) hipLaunchKernelGGL(q6k_mv_batched_fast_staged<true>, dim3(grid), dim3(256), slds, st, p);
            else hipLaunchKernelGGL(q6k_mv_batched_fast_staged<false>, dim3(grid), dim3(256), slds, st, p);
        } else if (!records && n_groups <= CHUNK_TOKENS && lds <= 65536 && g_tune_fast_lds) {
            if (ks == 4) hipLaunchKernelGGL((q6k_mv_batched_fast<4, false, true>), dim3(grid), dim3(256), lds, st, p);
            else if (ks == 2) hipLaunchKernelGGL((q6k_mv_batched_fast<2, false, true>), dim3(grid), dim3(256), lds, st, p);
            else hipLaunchKernelGGL((q6k_mv_batched_fast<1, false, true>), dim3(grid), dim3(256), lds, st, p);
        } else if (ks == 4 && twin) hipLaunchKernelGGL((q6k_mv_batched_fast<4, true>), dim3(grid), dim3(256), 0, st, p);
        else if (ks == 4) hipLaunchKernelGGL((q6k_mv_batched_fast<4, false>), dim3(grid), dim3(256), 0, st, p);
        else if (ks == 2 && twin) hipLaunchKernelGGL((q6k_mv_batched_fast<2, true>), dim3(grid), dim3(256), 0, st, p);
        else if (ks == 2) hipLaunchKernelGGL((q6k_mv_batched_fast<2, false>), dim3(grid), dim3(256), 0, st, p);
        else if (twin) hipLaunchKernelGGL((q6k_mv_batched_fast<1, true>), dim3(grid), dim3(256), 0, st, p);
        else hipLaunchKernelGGL((q6k_mv_batched_fast<1, false>), dim3(grid), dim3(256), 0, st, p);
        return hipGetLastError() == hipSuccess ? 0 : -1;
    }
    if (!records) return launch_one_group(p, max_chunks, all, st);
    // (a layer's rows are multiples of 256)
    if (p.tiles % 4) return -1;
    if (twin) hipLaunchKernelGGL(q6k_mv_batched_twin_staged, dim3((unsigned)(all / 4)), dim3(256), 4 * CHUNK_BLOCK_BYTES, st, p);
    else hipLaunchKernelGGL(q6k_mv_batched_few, dim3((unsigned)(all / 4)), dim3(256), 2 * CHUNK_BLOCK_BYTES, st, p);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int q6k_wide_groups(int rows, bool pair) {
    const int tiles = (rows + TILE_ROWS - 1) / TILE_ROWS;
    return pair ? (tiles + 3) / 4 : (tiles + 7) / 8;  // four of gate and four of up, or eight
}

bool q6k_wide_fits(int rows, int blocks) { return rows % TILE_ROWS == 0 && blocks <= WIDE_MAX_BLOCKS; }

int launch_q6k_mv_batched_wide(const void *w, const void *w2, size_t expert_stride,
                               const GroupItem *records, const int32_t *pair_out,
                               const int8_t *act_q, const float *act_d, float *y, int rows,
                               int blocks, int n_groups, int max_chunks, hipStream_t st) {
    if (!q6k_wide_fits(rows, blocks) || (uintptr_t)y % 16 || max_chunks <= 0) return -1;
    BatchParams p = {};
    p.w = (const uint8_t *)w;
    p.w2 = (const uint8_t *)w2;
    p.expert_stride = expert_stride;
    p.wide_info = records + 2 * (size_t)max_chunks;
    p.pair_out = pair_out;
    p.act_q = act_q;
    p.act_d = act_d;
    p.y = y;
    p.ldy = p.rows = rows;
    p.tiles = rows / TILE_ROWS;
    p.blocks = blocks;
    const int row_groups = q6k_wide_groups(rows, w2 != nullptr);
    const int units = group_wide_units(n_groups, max_chunks);
    constexpr size_t lds = 2 * WIDE_CHUNKS * CHUNK_BLOCK_BYTES;
    if (w2) hipLaunchKernelGGL(q6k_mv_batched_wide<true>, dim3(units * row_groups), dim3(512), lds, st, p, row_groups);
    else hipLaunchKernelGGL(q6k_mv_batched_wide<false>, dim3(units * row_groups), dim3(512), lds, st, p, row_groups);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_q6k_mv_batched_x3(const void *const w[3], float *const y[3], const int rows[3], int n_mat,
                             const int8_t *act_q, const float *act_d, int blocks, int nseq,
                             hipStream_t st) {
    if (n_mat < 1 || n_mat > 3 || nseq <= 0 || blocks <= 0) return -1;
    BatchParams p = {};
    const int chunks = (nseq + CHUNK_TOKENS - 1) / CHUNK_TOKENS;
    int first = 0;
    p.n_segs = n_mat;
    for (int i = 0; i < n_mat; ++i) {
        auto &sg = p.segs[i];
        sg.w = (const uint8_t *)w[i];
        sg.y = y[i];
        sg.rows = rows[i];
        sg.tiles = (rows[i] + TILE_ROWS - 1) / TILE_ROWS;
        sg.first = first;
        sg.items = sg.tiles * chunks;
        first += sg.items;
    }
    p.w = p.segs[0].w;
    p.y = p.segs[0].y;
    p.rows = p.ldy = rows[0];
    p.tiles = p.segs[0].tiles;
    p.items_per_mat = p.segs[0].items;
    p.act_q = act_q;
    p.act_d = act_d;
    p.blocks = blocks;
    p.single_count = nseq;  // one group (expert 0) of nseq tokens
    return launch_one_group(p, chunks, first, st);
}

int launch_q6k_down_combine(const void *w, size_t expert_stride, const int32_t *ids,
                            const int8_t *aq, const float *ad, const float *weights,
                            const float *res, float *out, int rows, int blocks, int n_slots,
                            hipStream_t st) {
    if (n_slots <= 0 || n_slots > 16) return -1;
    DownParams p;
    p.w = (const uint8_t *)w;
    p.expert_stride = expert_stride;
    p.ids = ids;
    p.aq = aq;
    p.ad = ad;
    p.weights = weights;
    p.res = res;
    p.out = out;
    p.rows = rows;
    p.tiles = (rows + TILE_ROWS - 1) / TILE_ROWS;
    p.blocks = blocks;
    p.n_slots = n_slots;
    hipLaunchKernelGGL(q6k_down_combine, dim3(p.tiles), dim3(64 * n_slots), 0, st, p);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_q6k_dequant(const void *w, int rows, int blocks, float *out, hipStream_t st) {
    const int tiles = (rows + TILE_ROWS - 1) / TILE_ROWS;
    const int items = tiles * blocks;
    hipLaunchKernelGGL(q6k_dequant_tiled, dim3((items + 3) / 4), dim3(256), 0, st,
                       (const uint8_t *)w, rows, tiles, blocks, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace llamd

namespace llamd {

int launch_q6k_tile_bound(const void *w, int rows, int blocks, float *mt, hipStream_t st) {
    const int tiles = (rows + TILE_ROWS - 1) / TILE_ROWS;
    if (tiles <= 0 || blocks <= 0) return -1;
    hipLaunchKernelGGL(q6k_tile_bound, dim3((tiles + 3) / 4), dim3(256), 0, st, (const uint8_t *)w,
                       tiles, blocks, mt);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_q6k_mv_f32x(const void *w, const float *x, float *y, int rows, int blocks,
                       hipStream_t st) {
    if (!w || !x || !y || rows <= 0 || blocks <= 0 || blocks > F32X_MAX_BLOCKS) return -1;
    hipLaunchKernelGGL(q6k_mv_f32x, dim3((rows + TILE_ROWS - 1) / TILE_ROWS), dim3(512), 0, st,
                       (const uint8_t *)w, x, y, rows, blocks);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_lmhead_certify(const void *w, int rows, int blocks, int nseq, const int8_t *nq,
                          const float *nd, const float *pv, const int *pi, const float *mt,
                          float *logits, int32_t *ids, hipStream_t st) {
    if (rows <= 0 || blocks <= 0 || blocks > CERT_MAXB || nseq <= 0) return -1;
    CertifyParams p{(const uint8_t *)w, nq, nd, pv, pi, mt, logits, ids, rows,
                    (rows + TILE_ROWS - 1) / TILE_ROWS, blocks};
    hipLaunchKernelGGL(lmhead_certify, dim3(nseq), dim3(1024), 0, st, p);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace llamd

extern "C" int llamd_hip_kernel_clock(unsigned long long *d_slots, int n_slots) {
    if (d_slots && n_slots <= 0) return -1;
    llamd::g_clk_slots = d_slots;
    llamd::g_clk_n = d_slots ? n_slots : 0;
    llamd::g_clk_next = 0;
    return 0;
}
