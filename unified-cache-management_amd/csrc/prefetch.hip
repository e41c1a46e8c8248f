// Hit / miss / free-list bookkeeping of the GSA prefetch engine on the device:
// GSAPrefetchEngineC::RunOneBsPrefetch with GetHitAndMissBlock, RunPrefetchH2D
// and LoadKVToHBM (ucm/sparse/gsa/prefetch/src/kvcache_pre.cpp:206-322), one
// 256-thread workgroup per (request of the call, layer).
//
// The reference walks std::map / std::unordered_set containers with 16 OpenMP
// threads over the layers, requests one after the other.  Here a request's
// resident blocks are a row of plain arrays (slot s: cache block map_block[s],
// logical block map_idx[l][s]) and every step of the walk is a rank:
//   * a selected logical block is a hit if some slot holds it (each thread
//     scans the slots for one selection entry); misses keep their top-k order
//     (rank = misses before it, a ballot prefix);
//   * a free-list entry is eligible if its block is not (yet) in the hit set;
//     the i-th eligible entry, in free-list order, takes the i-th miss;
//   * the success table lists hits and served misses by logical index
//     ascending (rank = entries with a smaller index);
//   * the new free list is the blocks outside the hit set by block id ascending
//     (rank = such blocks with a smaller id).
// A few hundred integers per workgroup: latency-bound, like the selection.
#include "common.h"

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;

__device__ __forceinline__ unsigned lanes_below(unsigned long long mask)
{
    return __builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(mask >> 32),
                                     __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(mask), 0u));
}

// Rank of this thread among the threads (in thread order) whose predicate holds, and their number.
__device__ __forceinline__ int block_rank(bool pred, int* s_cnt, int& total)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned long long mask = __ballot(pred);
    int rank = static_cast<int>(lanes_below(mask));
    __syncthreads();                                   // s_cnt may still be read from the previous use
    if (lane == 0) { s_cnt[wave] = __popcll(mask); }
    __syncthreads();
    total = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        if (w < wave) { rank += s_cnt[w]; }
        total += s_cnt[w];
    }
    return rank;
}

// The first of list[0 .. n) that equals `x`, or -1; all kThreads entries of the list exist.  Sixteen entries per trip, their
// reads issued together, without an early exit: one entry per trip is one LDS latency per entry, four times in a
// row in this kernel (16 requests x 8 layers, 49 slots, 48 selected: 14.4 us that way, 9.4 this way).
__device__ __forceinline__ int first_equal(const int32_t* list, int n, int32_t x)
{
    int found = kThreads;
    for (int i0 = 0; i0 < n; i0 += 16) {
        int4 v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) { v[q] = *reinterpret_cast<const int4*>(&list[i0 + 4 * q]); }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int i = i0 + 4 * q;
            found = min(found, v[q].x == x ? i : kThreads);
            found = min(found, v[q].y == x ? i + 1 : kThreads);
            found = min(found, v[q].z == x ? i + 2 : kThreads);
            found = min(found, v[q].w == x ? i + 3 : kThreads);
        }
    }
    return found < n ? found : -1;
}

// grid: x = request of the call, y = layer
__global__ __launch_bounds__(kThreads) void prefetch_plan_kernel(
    const int32_t* __restrict__ map_block, const int32_t* __restrict__ map_len, int32_t* __restrict__ map_idx,
    int table_rows, int cap, const int32_t* __restrict__ topk_idx, int topk_stride,
    const int32_t* __restrict__ topk_len, const int32_t* __restrict__ rows, const int32_t* __restrict__ bs_index,
    int batch, int max_bs, int row_len, int32_t* __restrict__ free_block, int32_t* __restrict__ free_len,
    int32_t* __restrict__ success_blocks, int32_t* __restrict__ success_len, int32_t* __restrict__ load_blocks,
    int32_t* __restrict__ load_count, int32_t* __restrict__ miss_idxs, int32_t* __restrict__ miss_count)
{
    __shared__ __attribute__((aligned(16))) int32_t s_block[kThreads], s_idx[kThreads], s_miss[kThreads];
    __shared__ __attribute__((aligned(16))) int32_t s_ent_idx[2 * kThreads], s_ent_blk[2 * kThreads], s_succ[2 * kThreads];
    __shared__ __attribute__((aligned(16))) int s_hit[kThreads];
    __shared__ int s_cnt[kWaves];

    const int i = blockIdx.x, l = blockIdx.y, t = threadIdx.x;
    const size_t li = static_cast<size_t>(l) * batch + i;
    const int row = rows[i], b = bs_index[i];
    const int k = min(min(topk_len[i], topk_stride), kThreads);
    if (row < 0 || row >= table_rows || b < 0 || b >= max_bs || k <= 0) {   // (uniform) the reference skips such a request
        if (t == 0 && row >= 0 && row < table_rows) {
            load_count[static_cast<size_t>(l) * table_rows + row] = 0;
            miss_count[static_cast<size_t>(l) * table_rows + row] = 0;
        }
        return;
    }
    const size_t lb = static_cast<size_t>(l) * max_bs + b;
    const size_t lr = static_cast<size_t>(l) * table_rows + row;     // results stay with the request's row
    const int n = min(min(map_len[row], cap), kThreads);
    const int f = min(min(free_len[lb], row_len), kThreads);
    int32_t* idx_row = map_idx + (static_cast<size_t>(l) * table_rows + row) * cap;
    int32_t* free_row = free_block + lb * row_len;
    int32_t* succ_row = success_blocks + lb * row_len;

    s_block[t] = t < n ? map_block[static_cast<size_t>(row) * cap + t] : -1;
    s_idx[t] = t < n ? idx_row[t] : -1;
    s_hit[t] = 0;
    const int item = t < k ? topk_idx[li * topk_stride + t] : -1;
    const int free_id = t < f ? free_row[t] : -1;
    s_succ[t] = 0;
    s_succ[t + kThreads] = 0;
    __syncthreads();

    // 1. hits and misses of the selection
    const int hit_slot = first_equal(s_idx, n, item);
    if (t < k && hit_slot >= 0) { s_hit[hit_slot] = 1; }
    const bool is_hit = t < k && hit_slot >= 0, is_miss = t < k && hit_slot < 0;
    int n_hit_entries;
    const int hit_rank = block_rank(is_hit, s_cnt, n_hit_entries);
    const int miss_rank = t - hit_rank, n_miss = k - n_hit_entries;    // (of the first k threads, who did not hit)
    if (is_miss) {
        s_miss[miss_rank] = item;
        miss_idxs[lr * topk_stride + miss_rank] = item;
    }
    if (is_hit) { s_ent_idx[hit_rank] = item; s_ent_blk[hit_rank] = s_block[hit_slot]; }
    __syncthreads();                                   // s_hit, s_miss complete

    // 2. the free list serves the misses in order
    const int free_slot = first_equal(s_block, n, free_id);
    const bool eligible = t < f && n_miss > 0 && free_slot >= 0 && s_hit[free_slot] == 0;
    int n_eligible;
    const int el_rank = block_rank(eligible, s_cnt, n_eligible);
    const int n_load = min(min(n_eligible, n_miss), cap);   // (a free list that names a block twice could outnumber the slots)
    if (eligible && el_rank < n_load) {
        const int32_t want = s_miss[el_rank];
        load_blocks[lr * cap + el_rank] = free_id;
        s_hit[free_slot] = 1;
        s_idx[free_slot] = want;                          // the block now holds the missing logical block
        s_ent_idx[n_hit_entries + el_rank] = want;
        s_ent_blk[n_hit_entries + el_rank] = free_id;
    }
    __syncthreads();

    // 3. success table: by logical index ascending
    const int n_ent = n_hit_entries + n_load;
    for (int e = t; e < n_ent; e += kThreads) {
        const int32_t mine = s_ent_idx[e];
        int rank = 0;
        for (int u0 = 0; u0 < n_ent; u0 += 16) {
            int4 v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) { v[q] = *reinterpret_cast<const int4*>(&s_ent_idx[u0 + 4 * q]); }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int u = u0 + 4 * q;
                rank += (u < n_ent && v[q].x < mine) + (u + 1 < n_ent && v[q].y < mine) + (u + 2 < n_ent && v[q].z < mine) +
                        (u + 3 < n_ent && v[q].w < mine);
            }
        }
        s_succ[rank] = s_ent_blk[e];
    }
    __syncthreads();
    // (the reference zero-fills the whole row first)
    for (int p = t; p < row_len; p += kThreads) { succ_row[p] = p < 2 * kThreads ? s_succ[p] : 0; }

    // 4. new free list: blocks outside the hit set by block id ascending; map write-back
    const bool is_free = t < n && s_hit[t] == 0;
    if (is_free) {
        const int32_t mine = s_block[t];
        int rank = 0;
        for (int u0 = 0; u0 < n; u0 += 8) {
            int4 v[2], hit[2];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                v[q] = *reinterpret_cast<const int4*>(&s_block[u0 + 4 * q]);
                hit[q] = *reinterpret_cast<const int4*>(&s_hit[u0 + 4 * q]);
            }
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int u = u0 + 4 * q;
                rank += (u < n && hit[q].x == 0 && v[q].x < mine) + (u + 1 < n && hit[q].y == 0 && v[q].y < mine) +
                        (u + 2 < n && hit[q].z == 0 && v[q].z < mine) + (u + 3 < n && hit[q].w == 0 && v[q].w < mine);
            }
        }
        if (rank < row_len) { free_row[rank] = mine; }
    }
    int n_free;
    block_rank(is_free, s_cnt, n_free);
    if (t < n) { idx_row[t] = s_idx[t]; }
    if (t == 0) {
        free_len[lb] = n_free;
        success_len[lb] = max(n, 0) - n_free;
        load_count[lr] = n_load;
        miss_count[lr] = n_miss;
    }
}

}  // namespace

extern "C" int ucm_prefetch_plan(const int32_t* map_block, const int32_t* map_len, int32_t* map_idx, int table_rows,
                                 int cap, const int32_t* topk_idx, int topk_stride, const int32_t* topk_len,
                                 const int32_t* rows, const int32_t* bs_index, int batch, int n_layers, int max_bs,
                                 int row_len, int32_t* free_block, int32_t* free_len, int32_t* success_blocks,
                                 int32_t* success_len, int32_t* load_blocks, int32_t* load_count, int32_t* miss_idxs,
                                 int32_t* miss_count, ucm_stream_t stream)
{
    UCM_REQUIRE(batch >= 0 && n_layers > 0 && n_layers <= 65535, "ucm_prefetch_plan: batch=%d n_layers=%d", batch, n_layers);
    if (batch == 0) { return UCM_OK; }
    UCM_REQUIRE(map_block && map_len && map_idx && topk_idx && topk_len && rows && bs_index && free_block && free_len &&
                    success_blocks && success_len && load_blocks && load_count && miss_idxs && miss_count,
                "ucm_prefetch_plan: null pointer");
    UCM_REQUIRE(table_rows > 0 && max_bs > 0, "ucm_prefetch_plan: table_rows=%d max_bs=%d", table_rows, max_bs);
    UCM_SUPPORTED(cap >= 1 && cap <= kThreads && topk_stride >= 1 && topk_stride <= kThreads && row_len >= 1,
                  "ucm_prefetch_plan: cap=%d topk_stride=%d (1..%d resident blocks and selected blocks per request)", cap,
                  topk_stride, kThreads);
    hipLaunchKernelGGL(prefetch_plan_kernel, dim3(batch, n_layers), dim3(kThreads), 0, ucm::as_stream(stream), map_block,
                       map_len, map_idx, table_rows, cap, topk_idx, topk_stride, topk_len, rows, bs_index, batch, max_bs,
                       row_len, free_block, free_len, success_blocks, success_len, load_blocks, load_count, miss_idxs,
                       miss_count);
    UCM_LAUNCH_CHECK("ucm_prefetch_plan");
}
