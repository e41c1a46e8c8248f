// Block selection of one (layer, request) by one wave or by a workgroup of four: the device
// functions behind ucm_topk_windows / ucm_kvstar_topk (topk.hip) and behind the
// tail of the fused score + select kernel (score.hip).
//
// The request's scores become order-preserving 32-bit keys in a wave's registers (element i
// in lane i%64, register i/64).  Selection is a radix select,
// one bit per step from the top: the threshold T is grown greedily while at
// least so many keys are >= T, each count being a wave ballot + popcount.
// Candidates with key > T are all taken; of those with key == T the first
// `picks - count(key > T)` in index order are taken, which is exactly where a
// stable descending sort leaves equal scores.  Output positions are ballot
// prefix counts in index order, so the result comes out sorted ascending with
// no sort at all, and the logical->physical block-table lookup is applied on
// the way out.
//
// What bounds it is latency: a wave alone issues an instruction in about ten cycles, and a chain of scalar results takes longer.
// select_blocks therefore has all loads stand together without a branch between them (a branch per register had each wait for the
// one before: 4700 of the 11 100 cycles of a request of 512 blocks) and the compares of a step before their counts (42 cycles per
// register and step one after the other, 26 so), and four waves share the loads and the way out.  Alone, 16 requests of 256, 512 and
// 1024 blocks: 4.0, 6.1 and 10.5 us by one wave, 3.2, 3.9 and 5.3 us by four; of integers, many of which tie, 5.1, 7.9 and 13.2 us
// and 4.6, 6.1 and 8.4 us.  With the scores: 16 requests of up to 512 blocks 14.2 -> 12.6 us (fp32 table), one of 1024 14.3 -> 10.5, one of 256 8.0.
// (Halving an interval between the lanes' maxima instead of going bit by bit takes half the steps, each nearly twice as long, and
// 1000 cycles to begin with.)  Two registers and less are faster by one wave, to which the barriers and LDS are only in the way: 64 and
// 128 blocks with their scores 5.6 and 6.7 us, 6.0 and 7.2 as one wave that shared the four waves' code.
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
// Called by all 64 lanes of one wave (select_wave) or by all threads of a workgroup of four (select_blocks) for request r of
// layer l; kEpl * 64 is the longest request the instance holds (longer ones are cut there: host checked).
//
// The request's own descriptors (length, first row, how many to keep) come from the caller, which may have fetched them
// long before.
//
// kCoherent: the scores were written by other workgroups of the SAME launch (device-scope stores that went through
// to memory); they are read with device-scope loads, which do not take a line that an L2 of another part of the
// chip may still hold in an older state - or they are all in this workgroup's LDS (`lds`, not null).
//
// Four waves: every wave makes its share of the keys and leaves them in LDS, the first one holds all of them in registers and finds
// the threshold, with the forced blocks among them as the largest keys there are, and all write out what is above it.
// scratch: select_scratch(kEpl) words of LDS that nothing else uses any more.
constexpr int kSelectWaves = 4;
constexpr int select_scratch(int epl) { return 2 * 64 * epl + 64; }

template <int kEpl, bool kHeapTies, bool kCoherent = false>
__device__ __forceinline__ void select_blocks(const SelectArgs& a, int r, int l, int n, int64_t seg0, int k, unsigned* scratch,
                                              const float* lds = nullptr)
{
    constexpr int kThreads = kSelectWaves * 64;
    static_assert(kEpl % kSelectWaves == 0, "every wave has whole registers of its own");
    constexpr int kOwn = kEpl / kSelectWaves;
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
        {
            float sv[kOwn];
            unsigned pv[kOwn];
            if (kCoherent && lds) {
#pragma unroll
                for (int j = 0; j < kOwn; ++j) { sv[j] = lds[min(j * kThreads + tid, n - 1)]; }
            } else {
#pragma unroll
                for (int j = 0; j < kOwn; ++j) {
                    const float* p = s + min(j * kThreads + tid, n - 1);
                    sv[j] = kCoherent ? __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : *p;
                }
            }
#pragma unroll
            for (int j = 0; j < kOwn; ++j) { pv[j] = static_cast<unsigned>(table[min(j * kThreads + tid, n - 1)]); }
            asm volatile("" ::: "memory");
#pragma unroll
            for (int j = 0; j < kOwn; ++j) {
                const int i = j * kThreads + tid;
                const unsigned forced = i < n ? 0xffffffffu : 0u;        // a forced block's key is above all, a place past the end's below
                keys[i] = i >= start_w && i < hi ? ordered_key(sv[j]) : forced;
                phys[i] = pv[j];
            }
        }
        // The first wave finds the threshold; then all write out what is above it, each from its share of the elements (a register's worth
        // takes a wave 240 cycles, the two barriers 300).
        unsigned* shared = scratch + 2 * 64 * kEpl;      // the threshold, then the waves' counts
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        __syncthreads();
        unsigned T = 0xffffffffu;
        if (wave == 0) {
            const int m = k - start_w - end_w;           // free picks among the candidates
            bool exact = false;
            unsigned key[kEpl];
#pragma unroll
            for (int j = 0; j < kEpl; ++j) { key[j] = keys[j * 64 + lane]; }
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
            }
            if (lane == 0) { shared[0] = T; }
        }
        __syncthreads();
        T = __builtin_amdgcn_readfirstlane(shared[0]);
        // (a trip takes up to four registers' worth of elements, whose LDS reads then stand together)
        constexpr int kTrip = kOwn < 4 ? kOwn : 4;
        int mine = 0, pos = 0;
#pragma unroll 1
        for (int j0 = 0; j0 < kOwn; j0 += kTrip) {
#pragma unroll
            for (int u = 0; u < kTrip; ++u) { mine += __popcll(__ballot(keys[(wave * kOwn + j0 + u) * 64 + lane] > T)); }
        }
        if (lane == 0) { shared[1 + wave] = static_cast<unsigned>(mine); }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < kSelectWaves; ++w) {
            const int c = __builtin_amdgcn_readfirstlane(shared[1 + w]);
            pos += w < wave ? c : 0;
            count += c;
        }
#pragma unroll 1
        for (int j0 = 0; j0 < kOwn; j0 += kTrip) {
            unsigned key_out[kTrip], phys_out[kTrip];
#pragma unroll
            for (int u = 0; u < kTrip; ++u) { key_out[u] = keys[(wave * kOwn + j0 + u) * 64 + lane]; }
#pragma unroll
            for (int u = 0; u < kTrip; ++u) { phys_out[u] = phys[(wave * kOwn + j0 + u) * 64 + lane]; }
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

// One wave.
template <int kEpl, bool kHeapTies, bool kCoherent = false>
__device__ __forceinline__ void select_wave(const SelectArgs& a, int r, int l, int lane, int n, int64_t seg0, int k,
                                            const float* lds = nullptr)
{
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
        for (int i = lane; i < n; i += 64) {
            out[i] = i;
            if (pout) { pout[i] = bt[i]; }
        }
        count = n;
        kept_all = true;
    } else if (k < start_w + end_w) {
        // fewer slots than forced blocks: the first k of [0..start_w) ++ [n-end_w..n)
        for (int j = lane; j < k; j += 64) {
            const int idx = j < start_w ? j : n - end_w + (j - start_w);
            out[j] = idx;
            if (pout) { pout[j] = bt[idx]; }
        }
        count = k;
    } else {
        const int m = k - start_w - end_w;       // free picks among the middle blocks
        const int hi = n - end_w;                // candidates are start_w <= i < hi
        const float* s = a.scores + static_cast<int64_t>(l) * a.scores_layer_stride + seg0;
        unsigned key[kEpl];
        int32_t phys[kEpl];                      // the block table's entries, fetched with the scores: a load per
#pragma unroll                                   // taken element on the way out would cost a memory round trip per register
        for (int j = 0; j < kEpl; ++j) {
            const int i = j * 64 + lane;
            const bool cand = i >= start_w && i < hi;
            const int at = cand ? i : 0;
            float sv;
            if (kCoherent && lds) { sv = lds[at]; }
            else if (kCoherent) { sv = __hip_atomic_load(s + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
            else { sv = s[at]; }
            key[j] = cand ? ordered_key(sv) : 0u;
            phys[j] = bt ? bt[min(i, n - 1)] : 0;
        }
        unsigned T = 0;
        int need = 0;
        int tie_lo = 0, tie_hi = 0;              // kHeapTies: ranks (among the ties) that are kept
        if (m > 0) {
            for (int bit = 31; bit >= 0; --bit) {
                const unsigned c = T | (1u << bit);
                int cnt = 0;
#pragma unroll
                for (int j = 0; j < kEpl; ++j) { cnt += __popcll(__ballot(key[j] >= c)); }
                if (cnt >= m) { T = c; }
                // exactly m keys at or above c: they are the selection, and no lower bit can change that
                if (cnt == m) { T = c - 1u; break; }
            }
            int greater = 0;
#pragma unroll
            for (int j = 0; j < kEpl; ++j) { greater += __popcll(__ballot(key[j] > T)); }
            need = m - greater;
            if (kHeapTies) {
                // walk the list in index order up to the k-th block with key >= T
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
                tie_lo = greater - g_p;          // one tie left per block above T that came after P
                tie_hi = m - g_p;                // ties inside P
            }
        }
        int pos = 0, ties_seen = 0;
#pragma unroll
        for (int j = 0; j < kEpl; ++j) {
            if (j * 64 < n) {
                const int i = j * 64 + lane;
                const bool window = i < n && (i < start_w || i >= hi);
                const bool cand = i >= start_w && i < hi;
                const bool gt = cand && m > 0 && key[j] > T;
                const bool eq = cand && m > 0 && key[j] == T;
                const unsigned long long eq_mask = __ballot(eq);
                const int tie_rank = ties_seen + static_cast<int>(lanes_below(eq_mask));
                const bool take = window || gt || (eq && (kHeapTies ? (tie_rank >= tie_lo && tie_rank < tie_hi) : tie_rank < need));
                ties_seen += __popcll(eq_mask);
                const unsigned long long take_mask = __ballot(take);
                if (take) {
                    const int p = pos + static_cast<int>(lanes_below(take_mask));
                    out[p] = i;
                    if (pout) { pout[p] = phys[j]; }
                }
                pos += __popcll(take_mask);
            }
        }
        count = pos;
    }
    if (lane == 0) {
        a.count_out[lr] = count;
        if (a.sparse_seq_lens && a.seq_lens) {
            const int len = a.seq_lens[r], rem = len % a.block_size;
            // every block kept: the request keeps its length; otherwise `count` blocks, the last one partial
            a.sparse_seq_lens[lr] = kept_all ? len : (rem == 0 ? count * a.block_size : count * a.block_size - a.block_size + rem);
        }
    }
}

}  // namespace ucm
