// group.hip -- expert grouping for the prefill path.
//
// The design of the reference's moe_group.comp (crates/llamd-vulkan/shaders/
// moe_group.comp:37-82) on one gfx950 workgroup: a counting sort of the
// n_tok * n_used (token, slot) pairs by expert -- LDS histogram, prefix sum,
// scatter -- giving each expert a contiguous run of pairs. The order of pairs
// inside one expert's run depends on atomic arrival, which is harmless: each
// pair's result is computed independently and written to its own output row
// (the pair index), so the expert-major result equals the token-major one
// exactly, the property crates/llamd-testing/tests/vulkan_prefill.rs:268-333
// holds the reference's Vulkan path to.
//
// Outputs: slot_of_pair[p] = the chunk slot of pair p (an expert's 16-token chunks
// follow the expert before's; the j-th pair of an expert is token j % 16 of its
// chunk j / 16), pair_idx[i] = the pair index t * n_used + k at sorted position i,
// and a record per work item of the batched kernels (GroupItem, launch.hpp), which
// a wave reads in one load: one per chunk, records[max_chunks], then one per twin
// (two chunks of one expert), [max_chunks], then one per wide unit (up to
// GROUP_WIDE_CHUNKS chunks, fewer where units are few; an expert's chunks split
// evenly), [group_wide_units].
#include "common.hpp"
#include "launch.hpp"

namespace llamd {
namespace {

constexpr int GROUP_MAX_EXPERTS = 1024;

__global__ __launch_bounds__(1024) void moe_group(const int32_t *ids, int n_pairs, int n_expert,
                                                  GroupItem *records, int32_t *slot_of_pair,
                                                  int32_t *pair_idx, int max_chunks, int wide_few,
                                                  int max_sorted) {
    __shared__ int sub_lds[GROUP_MAX_EXPERTS];
    __shared__ int start_lds[GROUP_MAX_EXPERTS];
    __shared__ int hist[GROUP_MAX_EXPERTS];
    __shared__ int cursor[GROUP_MAX_EXPERTS];
    constexpr int PB = 8;
    const bool once = n_pairs <= PB * (int)blockDim.x;
    // the sorted pairs of a long prompt: scattered here, then written in order
    // (2000 tokens of 8: 18 -> 15 us; nothing to gain up to 8192 pairs)
    extern __shared__ int32_t sorted_lds[];
    int32_t *sorted = once || n_pairs > max_sorted ? nullptr : sorted_lds;
    __shared__ int totals[4];  // chunks, twins, pairs in a group, wide units
    const int tid = threadIdx.x;
    for (int e = tid; e < n_expert; e += blockDim.x) hist[e] = 0;
    __syncthreads();
    // a pair whose id is outside [0, n_expert) joins no group: its slot is -1,
    // which the chunk quantizers skip and the combine counts as no term
    // ids in batches of PB per thread, all of a batch's loads in flight
    // before its first atomic (one memory round trip per batch, not per id).
    // An id's place within its expert is what its count's increment returns;
    // it stays in a register, with the id, for the scatter below.
    int eid[PB], rank[PB];
    for (int base = 0; base < n_pairs; base += PB * (int)blockDim.x) {
#pragma unroll
        for (int k = 0; k < PB; ++k) {
            const int p = base + k * (int)blockDim.x + tid;
            eid[k] = p < n_pairs ? ids[p] : -1;
        }
#pragma unroll
        for (int k = 0; k < PB; ++k)
            if ((unsigned)eid[k] < (unsigned)n_expert) rank[k] = atomicAdd(&hist[eid[k]], 1);
    }
    __syncthreads();
    // exclusive prefix sums over experts (thread e owns expert e) of the
    // pair counts and of the 16-token chunk counts
    __shared__ int wsum_c[GROUP_MAX_EXPERTS / WAVE], wsum_s[GROUP_MAX_EXPERTS / WAVE],
        wsum_t[GROUP_MAX_EXPERTS / WAVE], wsum_q[GROUP_MAX_EXPERTS / WAVE], wsum_u[GROUP_MAX_EXPERTS / WAVE];
    const int lane = tid & 63, wave = tid >> 6;
    const int c = tid < n_expert ? hist[tid] : 0, ch = (c + 15) / 16, tw = (ch + 1) / 2;
    const int qu = (ch + 3) / 4;
    int wu = (ch + GROUP_WIDE_CHUNKS - 1) / GROUP_WIDE_CHUNKS;
    const int ic = wave_incl_sum_i(c), is = wave_incl_sum_i(ch), it = wave_incl_sum_i(tw);
    const int iu = wave_incl_sum_i(wu), iq = wide_few > 0 ? wave_incl_sum_i(qu) : 0;
    if (lane == WAVE - 1) {
        wsum_c[wave] = ic;
        wsum_s[wave] = is;
        wsum_t[wave] = it;
        wsum_q[wave] = iq;
        wsum_u[wave] = iu;
    }
    __syncthreads();
    int start = ic - c, sub = is - ch, tst = it - tw, ust = iu - wu;
    for (int w = 0; w < wave; ++w) {
        start += wsum_c[w];
        sub += wsum_s[w];
        tst += wsum_t[w];
        ust += wsum_u[w];
    }
    if (wide_few > 0) {
        // shorter wide units where those of 1, 2 or 4 chunks are few as well
        int s1 = 0, s2 = 0, s4 = 0, before = 0;
        for (int w = 0; WAVE * w < n_expert; ++w) {
            s1 += wsum_s[w];
            s2 += wsum_t[w];
            s4 += wsum_q[w];
            if (w < wave) before += wsum_q[w];
        }
        if (s1 <= wide_few) {
            wu = ch;
            ust = sub;
        } else if (s2 <= wide_few) {
            wu = tw;
            ust = tst;
        } else if (s4 <= wide_few) {
            wu = qu;
            ust = before + iq - qu;
        }
    }
    GroupItem *twin_info = records + max_chunks, *wide_info = twin_info + max_chunks;
    if (tid < n_expert) {
        sub_lds[tid] = sub;
        start_lds[tid] = start;
        cursor[tid] = 0;
        if (tid == n_expert - 1) {
            totals[0] = sub + ch;
            totals[1] = tst + tw;
            totals[2] = start + c;
            totals[3] = ust + wu;
        }
        for (int j = 0; j < ch; ++j)
            records[sub + j] = GroupItem{tid, j, sub + j, c, start, 0, 0, 0};
        for (int j = 0; j < tw; ++j)
            twin_info[tst + j] = GroupItem{tid, 2 * j, sub + 2 * j, c, start, 2 * j + 1 < ch, 0, 0};
        for (int j = 0, at = 0; j < wu; ++j) {
            const int nc = ch / wu + (j < ch % wu);
            wide_info[ust + j] = GroupItem{tid, at, sub + at, c, start, nc, 0, 0};
            at += nc;
        }
    }
    __syncthreads();
    // the records past the last chunk / twin / unit: no work (expert -1), so a
    // wave of the grid's spare items needs no other load to know it
    for (int i = totals[0] + tid; i < max_chunks; i += blockDim.x)
        records[i] = GroupItem{-1, 0, 0, 0, 0, 0, 0, 0};
    for (int i = totals[1] + tid; i < max_chunks; i += blockDim.x)
        twin_info[i] = GroupItem{-1, 0, 0, 0, 0, 0, 0, 0};
    for (int i = totals[3] + tid; i < group_wide_units(n_expert, max_chunks); i += blockDim.x)
        wide_info[i] = GroupItem{-1, 0, 0, 0, 0, 0, 0, 0};
    for (int base = 0; base < n_pairs; base += PB * (int)blockDim.x) {
        if (!once) {
            // more pairs than registers: the ids and their places again
#pragma unroll
            for (int k = 0; k < PB; ++k) {
                const int p = base + k * (int)blockDim.x + tid;
                eid[k] = p < n_pairs ? ids[p] : -1;
            }
#pragma unroll
            for (int k = 0; k < PB; ++k)
                if ((unsigned)eid[k] < (unsigned)n_expert) rank[k] = atomicAdd(&cursor[eid[k]], 1);
        }
#pragma unroll
        for (int k = 0; k < PB; ++k) {
            const int p = base + k * (int)blockDim.x + tid;
            if (p >= n_pairs) continue;
            const int e = eid[k];
            if ((unsigned)e >= (unsigned)n_expert) {
                slot_of_pair[p] = -1;
                continue;
            }
            const int j = rank[k];
            slot_of_pair[p] = (sub_lds[e] + j / 16) * 16 + j % 16;
            (sorted ? sorted : pair_idx)[start_lds[e] + j] = p;
        }
    }
    if (sorted) {
        __syncthreads();
        for (int i = tid; i < totals[2]; i += blockDim.x) pair_idx[i] = sorted[i];
    }
}

}  // namespace

int launch_moe_group(const int32_t *ids, int n_pairs, int n_expert, GroupItem *records,
                     int32_t *slot_of_pair, int32_t *pair_idx, hipStream_t st, int max_chunks,
                     int wide_few) {
    if (wide_few > n_expert) return -1;  // (group_wide_units)
    if (n_expert > GROUP_MAX_EXPERTS || n_expert <= 0 || max_chunks <= 0) return -1;
    const int max_sorted = 24576;
    const size_t lds = n_pairs > 8192 && n_pairs <= max_sorted ? (size_t)n_pairs * 4 : 0;
    static const hipError_t ok = hipFuncSetAttribute((const void *)moe_group, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                     max_sorted * 4);
    if (ok != hipSuccess) return -1;
    hipLaunchKernelGGL(moe_group, dim3(1), dim3(1024), lds, st, ids, n_pairs, n_expert, records,
                       slot_of_pair, pair_idx, max_chunks, wide_few, max_sorted);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace llamd
