// Block selection of one (layer, request) by a workgroup of one or four waves: the device
// function behind ucm_topk_windows / ucm_kvstar_topk (topk.hip) and behind the
// tail of the fused score + select kernel (score.hip).
//
// The request's scores become order-preserving 32-bit keys; every wave makes its share of
// them and leaves them in LDS, and one wave then holds all of them in registers (element i
// in lane i%64, register i/64).  Selection is a radix select,
// one bit per step from the top: the threshold T is grown greedily while at
// least k keys (the forced blocks' are the largest there are) are >= T, each count being a wave ballot + popcount.
// Candidates with key > T are all taken; of those with key == T the first
// `k - count(key > T)` in index order are taken, which is exactly where a
// stable descending sort leaves equal scores.  Output positions are ballot
// prefix counts in index order, so the result comes out sorted ascending with
// no sort at all, and the logical->physical block-table lookup is applied on
// the way out.
//
// What bounds it is latency: a wave alone issues an instruction in about ten cycles, and a chain of scalar results takes longer.
// So all loads stand together without a branch between them (a branch per register had each wait for the one before: 4700 of
// the 11 100 cycles of a request of 512 blocks), the compares of a step stand before their counts (42 cycles per register and
// step one after the other, 26 so), and four waves share the loads and the way out.  Alone, of 256, 512 and 1024 blocks: 3.7,
// 6.3 and 10.2 us as one wave with a register per 64 blocks throughout, 2.9, 4.1 and 5.0 us.  With the scores: 16 requests of up to
// 512 blocks 14.2 -> 12.6 us (fp32 table), one of 1024 14.3 -> 10.5, one of 256 8.0.  (Halving an interval between the lanes'
// maxima instead of going bit by bit takes half the steps, each nearly twice as long, and 1000 cycles to begin with.)
#pragma once

#include "common.h"

namespace ucm {

__device__ __forceinline__ unsigned ordered_key(float f)
{
    f = f + 0.0f;  // -0.0 -> +0.0, so that the two zeros tie like they do under operator>
    const int u = __float_as_int(f);
    return static_cast<unsigned>(u ^ ((u >> 31) | static_cast<int>(0x80000000u)));       // negative: all bits, else the sign bit
}

__device__ __forceinline__ unsigned lanes_below(unsigned long long mask)
{
    return __builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(mask >> 32),
                                     __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(mask), 0u));
}

// How many of the wave's keys are at least c: the compares of up to sixteen registers first, then their counts (one after the
// other, every count would wait for its own compare).
template <int kEpl>
__device__ __forceinline__ int count_at_least(const unsigned (&key)[kEpl], unsigned c)
{
    constexpr int kGroup = kEpl < 16 ? kEpl : 16;
    int cnt = 0;
#pragma unroll
    for (int g = 0; g < kEpl; g += kGroup) {
        unsigned long long m[kGroup];
#pragma unroll
        for (int j = 0; j < kGroup; ++j) { m[j] = __ballot(key[g + j] >= c); }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < kGroup; ++j) { cnt += __popcll(m[j]); }
    }
    return cnt;
}

// What one selection reads and writes; the same for every (layer, request) of a launch.
struct SelectArgs {
    const float* scores;            // layer 0; row x of layer l at scores[l * scores_layer_stride + x]
    int64_t scores_layer_stride;
    int64_t scores_rows;            // rows of a layer that may be read: a request outside them selects nothing
    const int32_t* seg_off;
    const int32_t* seg_len;
    const int32_t* topk_len;
    int n_req;
    int max_seg_len;                // the host's bound: a longer seg_len is cut there
    int start_w, end_w;
    int32_t* idx_out;
    int out_stride;
    int64_t idx_layer_stride;       // elements between two layers of idx_out / phys_out (dense: n_req * out_stride)
    int64_t cnt_layer_stride;       // elements between two layers of count_out / sparse_seq_lens (dense: n_req)
    int32_t* count_out;
    const int32_t* block_tables;
    int bt_stride;
    int32_t* phys_out;
    const int32_t* seq_lens;
    int block_size;
    int32_t* sparse_seq_lens;
};

// kHeapTies selects which blocks tied at the k-th score are kept.  false: the
// first ones in index order (std::stable_sort).  true: the ones KVStar's
// min-heap of (score, index) pairs ends up with
// (ucm/sparse/kvstar/retrieve/core/domain/retrieve_task/simd_compute_kernel.cpp:955-977:
// blocks arrive in index order, a full heap replaces its smallest pair only
// for a strictly greater score).  That process has a closed form: ties enter
// while fewer than k blocks with key >= T have arrived and leave, lowest index
// first, once per block above T that arrives later; so with P the shortest
// prefix holding k blocks >= T, g_P the blocks above T inside P and g those in
// the whole list, the ties kept are the ones of P whose rank among the ties is
// at least g - g_P.  Windows are not used with it (host checked).
//
// Called by all threads of a workgroup of kWaves waves (1 or 4) for request r of layer l; kEpl * 64 is the
// longest request the instance holds (longer ones are cut there: host checked).
//
// The request's own descriptors (length, first row, how many to keep) come from the caller, which may have fetched them
// long before.
//
// kCoherent: the scores were written by other workgroups of the SAME launch (device-scope stores that went through
// to memory); they are read with device-scope loads, which do not take a line that an L2 of another part of the
// chip may still hold in an older state - or they are all in this workgroup's LDS (`lds`, not null).
//
// scratch: select_scratch(kEpl) words of LDS that nothing else uses any more.
constexpr int select_scratch(int epl) { return 2 * 64 * epl + 64; }

template <int kEpl, bool kHeapTies, int kWaves, bool kCoherent = false>
__device__ __forceinline__ void select_blocks(const SelectArgs& a, int r, int l, int n, int64_t seg0, int k, unsigned* scratch,
                                              const float* lds = nullptr)
{
    constexpr int kThreads = kWaves * 64;
    constexpr int kPer = kEpl > kWaves ? kEpl / kWaves : 1;      // keys a thread makes
    const int tid = threadIdx.x, lane = tid & 63;
    const int start_w = a.start_w, end_w = a.end_w, out_stride = a.out_stride;
    const int64_t lr = static_cast<int64_t>(l) * a.cnt_layer_stride + r;
    const int64_t row_at = static_cast<int64_t>(l) * a.idx_layer_stride + static_cast<int64_t>(r) * out_stride;
    n = min(min(n, a.max_seg_len), min(out_stride, 64 * kEpl));  // host checked; clamp so nothing can run past a row
    if (a.block_tables) { n = min(n, a.bt_stride); }
    // a descriptor that came from device memory is followed only inside the scores of a layer
    if (seg0 < 0 || seg0 + max(n, 0) > a.scores_rows) { n = 0; }
    int32_t* out = a.idx_out + row_at;
    int32_t* pout = a.phys_out ? a.phys_out + row_at : nullptr;
    const int32_t* bt = a.block_tables ? a.block_tables + static_cast<size_t>(r) * a.bt_stride : nullptr;
    int count = 0;
    bool kept_all = false;

    if (n <= 0) {
        count = 0;
        kept_all = true;                         // nothing to drop: the request keeps its length
    } else if (start_w + end_w >= n || k >= n || k <= 0) {
        for (int i = tid; i < n; i += kThreads) {
            out[i] = i;
            if (pout) { pout[i] = bt[i]; }
        }
        count = n;
        kept_all = true;
    } else if (k < start_w + end_w) {
        // fewer slots than forced blocks: the first k of [0..start_w) ++ [n-end_w..n)
        for (int j = tid; j < k; j += kThreads) {
            const int idx = j < start_w ? j : n - end_w + (j - start_w);
            out[j] = idx;
            if (pout) { pout[j] = bt[idx]; }
        }
        count = k;
    } else {
        const int hi = n - end_w;                // candidates are start_w <= i < hi
        const float* s = a.scores + static_cast<int64_t>(l) * a.scores_layer_stride + seg0;
        // the block table's entries are fetched with the scores; without a table the loads read the row of indices
        // instead, and nothing uses them
        const int32_t* table = bt ? bt : out;
        unsigned *keys = scratch, *phys = scratch + 64 * kEpl;
        unsigned own_key[kPer], pv[kPer];        // (one wave alone goes on from these, without LDS)
        if (kEpl >= kWaves || tid < 64 * kEpl) {
            float sv[kPer];
            if (kCoherent && lds) {
#pragma unroll
                for (int j = 0; j < kPer; ++j) { sv[j] = lds[min(j * kThreads + tid, n - 1)]; }
            } else {
#pragma unroll
                for (int j = 0; j < kPer; ++j) {
                    const float* p = s + min(j * kThreads + tid, n - 1);
                    sv[j] = kCoherent ? __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : *p;
                }
            }
#pragma unroll
            for (int j = 0; j < kPer; ++j) { pv[j] = static_cast<unsigned>(table[min(j * kThreads + tid, n - 1)]); }
            asm volatile("" ::: "memory");
#pragma unroll
            for (int j = 0; j < kPer; ++j) {
                const int i = j * kThreads + tid;
                const unsigned forced = i < n ? 0xffffffffu : 0u;        // a forced block's key is above all, a place past the end's below
                own_key[j] = i >= start_w && i < hi ? ordered_key(sv[j]) : forced;
                keys[i] = own_key[j];
                if (kWaves > 1) { phys[i] = pv[j]; }
            }
        }
        // One wave finds the threshold; then up to four write out what is above it, each from its share of the elements (a
        // register's worth takes a wave 240 cycles, the two barriers 300).
        constexpr int kOutWaves = kWaves < kEpl ? kWaves : kEpl, kOwn = kEpl / kOutWaves;
        unsigned* shared = scratch + 2 * 64 * kEpl;      // the threshold, then the waves' counts
        const int wave = kOutWaves > 1 ? __builtin_amdgcn_readfirstlane(tid >> 6) : 0;
        if (kWaves > 1) {
            __syncthreads();
            if (tid >= kOutWaves * 64) { return; }
        }
        unsigned T = 0xffffffffu;
        if (kOutWaves == 1 || wave == 0) {
            const int m = k - start_w - end_w;           // free picks among the candidates
            bool exact = false;
            unsigned key[kEpl];
#pragma unroll
            for (int j = 0; j < kEpl; ++j) { key[j] = kWaves == 1 ? own_key[kWaves == 1 ? j : 0] : keys[j * 64 + lane]; }
            if (m > 0) {
                T = 0;
#pragma unroll 1
                for (int bit = 31; bit >= 0; --bit) {
                    const unsigned c = T | (1u << bit);
                    const int cnt = count_at_least<kEpl>(key, c);
                    if (cnt >= k) { T = c; }
                    // exactly k keys at or above c: they are the selection, and no lower bit can change that
                    if (cnt == k) { exact = true; T = c - 1u; break; }
                }
            }
            if (!exact) {
                // T is the k-th largest key and others hold the same (or no candidate is to be taken at all): the ones that are kept
                // get the largest key there is, the others the smallest
                const int greater = T == 0xffffffffu ? 0 : count_at_least<kEpl>(key, T + 1u) - start_w - end_w;
                int tie_lo = 0, tie_hi = m - greater;    // ranks (among the ties) that are kept
                if (kHeapTies) {
                    // walk the list in index order up to the m-th block with key >= T
                    int seen = 0, g_p = 0;
#pragma unroll
                    for (int j = 0; j < kEpl; ++j) {
                        const unsigned long long ge_mask = __ballot(key[j] >= T && key[j] != 0u);
                        const unsigned long long gt_mask = __ballot(key[j] > T);
                        const int c = __popcll(ge_mask);
                        if (seen < m) {
                            if (seen + c >= m) {
                                // lane holding the m-th one: the (m - seen)-th set bit of ge_mask
                                const bool is_pth = ((ge_mask >> lane) & 1ull) && seen + static_cast<int>(lanes_below(ge_mask)) + 1 == m;
                                const unsigned long long pm = __ballot(is_pth);
                                const int p_lane = __ffsll(static_cast<long long>(pm)) - 1;
                                const unsigned long long upto = p_lane >= 63 ? ~0ull : ((2ull << p_lane) - 1ull);
                                g_p += __popcll(gt_mask & upto);
                            } else {
                                g_p += __popcll(gt_mask);
                            }
                        }
                        seen += c;
                    }
                    tie_lo = greater - g_p;              // one tie left per block above T that came after P
                    tie_hi = m - g_p;                    // ties inside P
                }
                int ties_seen = 0;
#pragma unroll
                for (int j = 0; j < kEpl; ++j) {
                    const int i = j * 64 + lane;
                    const bool eq = key[j] == T && i >= start_w && i < hi;
                    const unsigned long long eq_mask = __ballot(eq);
                    const int rank = ties_seen + static_cast<int>(lanes_below(eq_mask));
                    if (eq) { keys[i] = rank >= tie_lo && rank < tie_hi ? 0xffffffffu : 0u; }
                    ties_seen += __popcll(eq_mask);
                }
                T = min(T, 0xfffffffeu);
                if (kWaves == 1) {
#pragma unroll
                    for (int j = 0; j < kPer; ++j) { own_key[j] = keys[j * 64 + lane]; }
                }
            }
            if (kOutWaves > 1 && lane == 0) { shared[0] = T; }
        }
        if (kOutWaves > 1) {
            __syncthreads();
            T = __builtin_amdgcn_readfirstlane(shared[0]);
        }
        // (a trip takes up to four registers' worth of elements, whose LDS reads then stand together)
        static_assert(kWaves > 1 || kEpl <= 4, "one wave alone keeps its keys in registers: one trip");
        constexpr int kTrip = kOwn < 4 ? kOwn : 4;
        int mine = 0, pos = 0;
        if (kOutWaves > 1) {
#pragma unroll 1
            for (int j0 = 0; j0 < kOwn; j0 += kTrip) {
#pragma unroll
                for (int u = 0; u < kTrip; ++u) { mine += __popcll(__ballot(keys[(wave * kOwn + j0 + u) * 64 + lane] > T)); }
            }
            if (lane == 0) { shared[1 + wave] = static_cast<unsigned>(mine); }
            __syncthreads();
#pragma unroll
            for (int w = 0; w < kOutWaves; ++w) {
                const int c = __builtin_amdgcn_readfirstlane(shared[1 + w]);
                pos += w < wave ? c : 0;
                count += c;
            }
        }
#pragma unroll 1
        for (int j0 = 0; j0 < kOwn; j0 += kTrip) {
            unsigned key_out[kTrip], phys_out[kTrip];
#pragma unroll
            for (int u = 0; u < kTrip; ++u) { key_out[u] = kWaves == 1 ? own_key[kWaves == 1 ? u : 0] : keys[(wave * kOwn + j0 + u) * 64 + lane]; }
#pragma unroll
            for (int u = 0; u < kTrip; ++u) { phys_out[u] = kWaves == 1 ? pv[kWaves == 1 ? u : 0] : phys[(wave * kOwn + j0 + u) * 64 + lane]; }
#pragma unroll
            for (int u = 0; u < kTrip; ++u) {
                const bool take = key_out[u] > T;
                const unsigned long long taken = __ballot(take);
                if (take) {
                    const int p = pos + static_cast<int>(lanes_below(taken));
                    out[p] = (wave * kOwn + j0 + u) * 64 + lane;
                    if (pout) { pout[p] = static_cast<int32_t>(phys_out[u]); }
                }
                pos += __popcll(taken);
            }
        }
        if (kOutWaves == 1) { count = pos; }
    }
    if (tid == 0) {
        a.count_out[lr] = count;
        if (a.sparse_seq_lens && a.seq_lens) {
            const int len = a.seq_lens[r], rem = len % a.block_size;
            // every block kept: the request keeps its length; otherwise `count` blocks, the last one partial
            a.sparse_seq_lens[lr] = kept_all ? len : (rem == 0 ? count * a.block_size : count * a.block_size - a.block_size + rem);
        }
    }
}

}  // namespace ucm
