// Paged-KV block moves: pointer-array batch copy, block-id driven dump/load in
// the stored-block layout, and the gather of selected blocks from a device
// block table.  Pure HBM traffic: every byte is read once and written once, so
// the kernels are 16-byte vector copies with non-temporal hints, a 1024-thread
// workgroup per slice or per 128 KiB of it (a 256 KiB K or V block is two),
// launched with far more workgroups than the 256 CUs.  Of the
// shapes tried on MI355X (8 KiB .. 256 KiB per workgroup, 64 .. 1024 threads,
// 1 .. 16 loads in flight per thread, persistent grids, with and without the
// non-temporal hint) this one was the fastest; all of them sit between 5.2 and
// 6.1 TB/s for a 1:1 read/write mix.  (Short slices take smaller ones.)
#include "common.h"

namespace {

using ucm::u32x4;

constexpr int kThreads = 1024;
constexpr int kUnroll = 8;
constexpr size_t kStep = static_cast<size_t>(kThreads) * 16 * kUnroll;  // 128 KiB per trip

// Gathers, dumps and loads by block list: a workgroup moves a whole slice, or one piece of it (a trip, 128 KiB) and ends with its
// stores on their way: see cut_slices.
// Slices of up to 8 KiB, the blocks of one or two kv heads, take 256 threads: a compute unit has eight of them under way and only
// two of 1024 (32 layers x 1024 blocks out and back, 4 KiB 299 -> 175 us = 6.1 TB/s, 8 KiB 435 -> 377; 16 KiB 730 -> 760, so no more).
constexpr int kShortThreads = 256;
constexpr size_t kShortSlice = 8 * 1024;

// kN x 16 KiB of a slice: every load is issued before the first store goes out.  Stores that start as the
// loads trickle in mix reads and writes on the HBM channels and cost about 6 % of the copy rate (1.64 ms ->
// 1.75 ms for the 5.1 GB gather), hence the wait for ALL of the trip's loads.
// (`meanwhile` runs while the loads are on their way.)
struct Nothing { __device__ __forceinline__ void operator()() const {} };

template <int kN, int kT = kThreads, typename F = Nothing>
__device__ __forceinline__ void copy_trip(uint8_t* __restrict__ dst, const uint8_t* __restrict__ src, size_t base, F meanwhile = F())
{
    u32x4 v[kN];
#pragma unroll
    for (int u = 0; u < kN; ++u) {
        v[u] = ucm::gload16_nt(src + base + static_cast<size_t>(u) * kT * 16);
    }
    asm volatile("" ::: "memory");
    meanwhile();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int u = 0; u < kN; ++u) {
        ucm::gstore16_nt(dst + base + static_cast<size_t>(u) * kT * 16, v[u]);
    }
}

// A workgroup's share of a slice; size is a multiple of 16.  What is left after the 128 KiB trips goes in trips of 64, 32 and 16 KiB (the slices of 64-, 32- and
// 16-token blocks), each with all its loads in flight at once, and a last partial one.  (kT threads: a trip is kT * 128 bytes.)
template <int kT = kThreads>
__device__ __forceinline__ void copy_slice(uint8_t* __restrict__ dst, const uint8_t* __restrict__ src, size_t size, unsigned thread = threadIdx.x)
{
    constexpr size_t kTrip = static_cast<size_t>(kT) * 16 * kUnroll;
    size_t o = 0;
    const size_t mine = thread * 16u;
    for (; o + kTrip <= size; o += kTrip) { copy_trip<kUnroll, kT>(dst, src, o + mine); }
    if (o + kTrip / 2 <= size) { copy_trip<kUnroll / 2, kT>(dst, src, o + mine); o += kTrip / 2; }
    if (o + kTrip / 4 <= size) { copy_trip<kUnroll / 4, kT>(dst, src, o + mine); o += kTrip / 4; }
    if (o + kTrip / 8 <= size) { copy_trip<kUnroll / 8, kT>(dst, src, o + mine); o += kTrip / 8; }
    if (o + mine < size) { ucm::gstore16_nt(dst + o + mine, ucm::gload16_nt(src + o + mine)); }
}

__global__ __launch_bounds__(kThreads) void copy_batch_kernel(void* const* __restrict__ dst,
                                                              const void* const* __restrict__ src,
                                                              size_t size, size_t piece)
{
    // large copies are cut into pieces so that one pointer pair still fills the chip
    const size_t pieces = (size + piece - 1) / piece;
    const size_t i = blockIdx.x / pieces, c = blockIdx.x % pieces;
    const size_t off = c * piece;
    const size_t len = off + piece <= size ? piece : size - off;
    copy_slice(static_cast<uint8_t*>(dst[i]) + off, static_cast<const uint8_t*>(src[i]) + off, len);
}

// Where a cache block's K and V slices of a layer sit inside a stored block: at layer * layer_pitch + slice_base
// (K) and block_bytes later (V).  One rank's blocks: layer_pitch = 2 * block_bytes, slice_base = 0; rank r of tp
// ranks that share the stored block: layer_pitch = 2 * block_bytes * tp, slice_base = 2 * block_bytes * r.
struct StoredLayout {
    size_t layer_pitch, slice_base;
    __host__ __device__ size_t slice(size_t layer, unsigned kv, size_t block_bytes) const
    {
        return layer * layer_pitch + slice_base + kv * block_bytes;
    }
};

// kCut: a workgroup takes one of the slice's `pieces`
// grid: x = index into block_ids (* pieces + piece), y = layer, z = K|V
template <bool kToStaging, bool kCut, int kT>
__global__ __launch_bounds__(kT) void kv_blocks_kernel(void* const* __restrict__ layers,
                                                             size_t kv_stride, size_t block_bytes,
                                                             const int32_t* __restrict__ block_ids,
                                                             unsigned num_blocks,
                                                             uint8_t* __restrict__ staging, unsigned pieces, StoredLayout lay)
{
    const unsigned i = kCut ? blockIdx.x / pieces : blockIdx.x, l = blockIdx.y, kv = blockIdx.z, n_layers = gridDim.y;
    const size_t off = kCut ? (blockIdx.x - i * pieces) * kStep : 0;
    const unsigned id = static_cast<unsigned>(block_ids[i]);
    if (id >= num_blocks) { return; }  // ids outside the cache are skipped, never dereferenced
    uint8_t* cache = static_cast<uint8_t*>(layers[l]) + kv * kv_stride +
                     static_cast<size_t>(id) * block_bytes + off;
    uint8_t* stage = staging + static_cast<size_t>(i) * n_layers * lay.layer_pitch + lay.slice(l, kv, block_bytes) + off;
    const size_t size = kCut ? min(kStep, block_bytes - off) : block_bytes;
    if (kToStaging) { copy_slice<kT>(stage, cache, size); }
    else { copy_slice<kT>(cache, stage, size); }
}

// grid: x = position in the request's selection (* pieces + piece), y = request, z = layer*2 + K|V
template <bool kCut, int kT>
__global__ __launch_bounds__(kT) void kv_gather_selected_kernel(
    const void* const* __restrict__ layers, size_t kv_stride, size_t block_bytes,
    const int32_t* __restrict__ phys, const int32_t* __restrict__ count, unsigned num_blocks,
    unsigned n_req, unsigned phys_stride, const int64_t* __restrict__ dst_off,
    const int32_t* __restrict__ region_k, uint8_t* __restrict__ staging, uint64_t staging_blocks, unsigned pieces)
{
    const unsigned j = kCut ? blockIdx.x / pieces : blockIdx.x, r = blockIdx.y, l = blockIdx.z >> 1, kv = blockIdx.z & 1;
    const size_t lr = static_cast<size_t>(l) * n_req + r;
    if (static_cast<int32_t>(j) >= count[lr]) { return; }
    const unsigned id = static_cast<unsigned>(phys[lr * phys_stride + j]);
    if (id >= num_blocks) { return; }
    const uint8_t* src = static_cast<const uint8_t*>(layers[l]) + kv * kv_stride +
                         static_cast<size_t>(id) * block_bytes;
    const int64_t off = dst_off[r], region = region_k[r];
    if (off < 0 || region < 0) { return; }
    const uint64_t slot = static_cast<uint64_t>(off) + (static_cast<uint64_t>(l) * 2 + kv) * static_cast<uint64_t>(region) + j;
    if (slot >= staging_blocks) { return; }              // never write outside the staging buffer
    const size_t at = kCut ? (blockIdx.x - j * pieces) * kStep : 0;
    copy_slice<kT>(staging + slot * block_bytes + at, src + at, kCut ? min(kStep, block_bytes - at) : block_bytes);
}

// Loads planned on the device: slot j of request row `row` receives logical block load_sel[l][row][j] (or
// nothing, -1) from a pool of stored blocks laid out [block][layer][K|V].
//
// A workgroup of kT threads follows one slot, or one piece of it (kT * 128 bytes, a trip), and nothing else: it ends with its
// stores on their way, and one whose slot loads nothing ends after one read.  The shorter the slice, the fewer threads: what
// limits short slices is how many of them a compute unit has under way, and what limits a plan that loads little is how
// fast it gets through idle workgroups (1024 threads: two a unit; 256: eight).  us, 1024 threads for every 16th (or
// every) slot of a row | a list per row as below, one slice after the other | this:
//   64 requests x 50 slots, 4 KiB, all load          30.0 | 30.7 | 12.0       a tenth  22.4 | 20.5 | 8.4
//   8 layers x 16 x 50, 32 KiB                       159  | 158  | 145                 26.2 | 33.0 | 18.7
//   32 layers x 32 x 153, 32 KiB                     3840 | 4010 | 3810                406  | 403  | 397
//   8 layers x 64 x 48, 32 KiB                       563  | 606  | 588                 85.1 | 66.6 | 62.7
//   4 layers x 32 x 60, 64 KiB                       345  | 343  | 352                 41.5 | 55.0 | 39.5
//   8 layers x 8 x 100, 128 KiB                      594  | 590  | 580                 63.7 | 84.2 | 61.1
// (A loop over further pieces, for grids that stop short of a row, made an idle workgroup 1.8 times as long.)
// grid: x = slot * pieces + piece, y = request of the call, z = layer*2 + K|V
template <int kT>
__global__ __launch_bounds__(kT) void kv_load_slot_kernel(
    void* const* __restrict__ layers, size_t kv_stride, size_t block_bytes, unsigned num_blocks,
    const uint8_t* __restrict__ pool, uint64_t pool_blocks, size_t pool_block_bytes, unsigned store_first_layer,
    const int32_t* __restrict__ load_sel, unsigned n_slots, const int32_t* __restrict__ src_table, unsigned src_stride,
    const int32_t* __restrict__ dst_table, unsigned dst_stride, int64_t dst_layer_stride,
    const int32_t* __restrict__ load_count, const int32_t* __restrict__ rows, unsigned table_rows, unsigned pieces, StoredLayout lay)
{
    constexpr size_t kPiece = static_cast<size_t>(kT) * 16 * kUnroll;
    const unsigned b = blockIdx.y, l = blockIdx.z >> 1, kv = blockIdx.z & 1;
    unsigned row = b;
    if (rows) {
        const int32_t r = rows[b];
        if (r < 0) { return; }
        row = static_cast<unsigned>(r);
    }
    if (row >= table_rows) { return; }
    const unsigned j = blockIdx.x / pieces;
    if (load_count && static_cast<int>(j) >= load_count[static_cast<size_t>(l) * table_rows + row]) { return; }
    const int32_t sel = load_sel[(static_cast<size_t>(l) * table_rows + row) * n_slots + j];
    if (sel < 0 || static_cast<unsigned>(sel) >= src_stride) { return; }          // slot keeps what it holds
    const int32_t src = src_table[static_cast<size_t>(row) * src_stride + sel];
    const unsigned dst = static_cast<unsigned>(dst_table[l * dst_layer_stride + static_cast<int64_t>(row) * dst_stride + j]);
    if (src < 0 || static_cast<uint64_t>(src) >= pool_blocks || dst >= num_blocks) { return; }   // not in the pool, or outside the cache
    const size_t off = (blockIdx.x - j * pieces) * kPiece;
    copy_slice<kT>(static_cast<uint8_t*>(layers[l]) + kv * kv_stride + static_cast<size_t>(dst) * block_bytes + off,
                   pool + static_cast<size_t>(src) * pool_block_bytes + lay.slice(store_first_layer + l, kv, block_bytes) + off,
                   min(kPiece, block_bytes - off));
}

// The same for slices of more than a 128 KiB trip in launches of many pieces, where a workgroup each costs more in idle ones
// than it brings (8 layers x 16 requests x 153 slots of 256 KiB, one in fifty loads: 155 us that way, 87 this way).
// A workgroup looks at all of its row's slots at once, keeps the ones that load something in a list in LDS, and takes its
// share of their pieces: the row's workgroups deal the pieces (one trip each) out between them.  (Stepping from slot to
// slot costs a trip to memory for every slot that has nothing to load, with the copies standing still, and whole
// slices of 256 KiB leave the chip half empty at the end: 2 layers x 16 requests with 779 blocks to load 181 us, 143 this
// way; 8 layers x 16 requests, 1875 blocks, 359 and 353 us = 5.6 TB/s.  Pieces of 64 KiB: 148 and 360 us.)
// grid: x = workgroup of the row, y = request of the call, z = layer*2 + K|V
constexpr size_t kLoadPiece = kStep;

__global__ __launch_bounds__(kThreads) void kv_load_planned_kernel(
    void* const* __restrict__ layers, size_t kv_stride, size_t block_bytes, unsigned num_blocks,
    const uint8_t* __restrict__ pool, uint64_t pool_blocks, size_t pool_block_bytes, unsigned store_first_layer,
    const int32_t* __restrict__ load_sel, unsigned n_slots, const int32_t* __restrict__ src_table, unsigned src_stride,
    const int32_t* __restrict__ dst_table, unsigned dst_stride, int64_t dst_layer_stride,
    const int32_t* __restrict__ load_count, const int32_t* __restrict__ rows, unsigned table_rows, StoredLayout lay)
{
    __shared__ int32_t s_src[kThreads];
    __shared__ unsigned s_dst[kThreads];
    __shared__ unsigned s_cnt[kThreads / 64];
    const unsigned b = blockIdx.y, l = blockIdx.z >> 1, kv = blockIdx.z & 1;
    unsigned row = b;
    if (rows) {
        const int32_t r = rows[b];
        if (r < 0) { return; }
        row = static_cast<unsigned>(r);
    }
    if (row >= table_rows) { return; }
    unsigned limit = n_slots;
    if (load_count) { limit = min(limit, static_cast<unsigned>(max(load_count[static_cast<size_t>(l) * table_rows + row], 0))); }
    const unsigned pieces = static_cast<unsigned>((block_bytes + kLoadPiece - 1) / kLoadPiece);
    uint8_t* cache = static_cast<uint8_t*>(layers[l]) + kv * kv_stride;
    const uint8_t* stored = pool + lay.slice(store_first_layer + l, kv, block_bytes);
    const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (unsigned j0 = 0; j0 < limit; j0 += kThreads) {           // (uniform: one trip for up to 1024 slots)
        const unsigned j = j0 + threadIdx.x;
        int32_t src = -1;
        unsigned dst = 0;
        if (j < limit) {
            const int32_t sel = load_sel[(static_cast<size_t>(l) * table_rows + row) * n_slots + j];
            dst = static_cast<unsigned>(dst_table[l * dst_layer_stride + static_cast<int64_t>(row) * dst_stride + j]);
            if (sel >= 0 && static_cast<unsigned>(sel) < src_stride) { src = src_table[static_cast<size_t>(row) * src_stride + sel]; }
        }
        // a slot without an entry keeps what it holds; a block that is not in the pool, or outside the cache, is skipped
        const bool loads = src >= 0 && static_cast<uint64_t>(src) < pool_blocks && dst < num_blocks;
        const unsigned long long mask = __ballot(loads);
        if (lane == 0) { s_cnt[wave] = static_cast<unsigned>(__popcll(mask)); }
        __syncthreads();
        unsigned at = __builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(mask >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(mask), 0u));
        unsigned total = 0;
        for (unsigned w = 0; w < kThreads / 64; ++w) {
            const unsigned c = s_cnt[w];
            if (w < wave) { at += c; }
            total += c;
        }
        if (loads) { s_src[at] = src; s_dst[at] = dst; }
        __syncthreads();
        for (unsigned u = blockIdx.x; u < total * pieces; u += gridDim.x) {   // (uniform in the workgroup)
            const unsigned i = u / pieces;
            const size_t off = (u - i * pieces) * kLoadPiece;
            // (the waves start a piece together: HBM serves their reads and writes 2 to 4 % faster in turns than mixed)
            __syncthreads();
            copy_slice(cache + static_cast<size_t>(s_dst[i]) * block_bytes + off,
                       stored + static_cast<size_t>(s_src[i]) * pool_block_bytes + off, min(kLoadPiece, block_bytes - off));
        }
        __syncthreads();                                          // (the list is rebuilt in the next trip)
    }
}

// The same loads when every row says how many of its leading entries are loads (load_count): the work is
// known exactly, so it is dealt out evenly.  Every workgroup builds the running total of the (layer, request)
// pairs' counts in LDS (a few hundred integers), and takes the pieces w, w + grid, ... of the 2 * total slices
// (K and V); which pair a slice belongs to is a binary search in the totals.
// (Pieces of one 128 KiB trip, and a running total by wave scans: 47 loads of one layer 21.4 us with whole slices and a scan
// of ten barriers, 15.7 so; 116 loads 29.5 and 27.4; 887 loads of 8 layers 170.7 and 169.8.)
// grid: x = workgroup.
constexpr unsigned kMaxPlannedPairs = 4096;
// Slices of up to kShortSlice go through one wave each, in workgroups that are all resident at once: sixteen are found and copied side
// by side where the whole workgroup took them one after the other.  us, the whole workgroup | a workgroup of 256 threads per slot of
// the plan (idle ones cost 0.4 ns each) | this, 4 KiB: 8 layers x 64 x 24 slots, all load 141 | 35 | 36, a fifth 34 | 16.7 | 9.9;
// 8 x 32 x 800, a tenth 221 | 151 | 60 to 64, one in a hundred 27.7 | 123 | 8.2; 32 x 64 x 1000, one in a hundred 251 | 1110 | 61 to 73.
// 8 KiB: all of 8 x 64 x 24 142 | 64 | 70 to 75, one in a hundred of 32 x 64 x 1000 253 | 1112 | 114 to 118.  Teams of two and four
// waves 0 to 8 and 10 to 110 % slower at up to 4 KiB, alike at 8; twice the workgroups 2 us slower, half of them waiting for the others.
constexpr int kTeamThreads = 64;
constexpr unsigned kTeamGroups = 512;

// kWhole: slices of at most one piece.  kT threads copy one: the whole workgroup, or a team of it.
template <bool kWhole, int kT>
__global__ __launch_bounds__(kThreads) void kv_load_counted_kernel(
    void* const* __restrict__ layers, size_t kv_stride, size_t block_bytes, unsigned num_blocks,
    const uint8_t* __restrict__ pool, uint64_t pool_blocks, size_t pool_block_bytes, unsigned store_first_layer,
    const int32_t* __restrict__ load_sel, unsigned n_slots, const int32_t* __restrict__ src_table, unsigned src_stride,
    const int32_t* __restrict__ dst_table, unsigned dst_stride, int64_t dst_layer_stride,
    const int32_t* __restrict__ load_count, const int32_t* __restrict__ rows, unsigned table_rows, unsigned batch,
    unsigned n_layers, StoredLayout lay)
{
    __shared__ unsigned s_total[kMaxPlannedPairs + 1];   // s_total[p] = loads of the pairs before p
    __shared__ unsigned s_part[kThreads / 64];
    const unsigned pairs = n_layers * batch;             // pair p = layer p / batch, request p % batch
    constexpr unsigned kPer = kMaxPlannedPairs / kThreads;
    // (A thread takes one pair, and four only if there are more pairs than threads; loads of pairs that do not exist read the last
    // one's.  With four in a row each waited for two trips to memory of its own before the first piece was copied.)
    const unsigned per = pairs <= kThreads ? 1u : kPer;
    unsigned mine[kPer], sum = 0;
#pragma unroll
    for (unsigned i = 0; i < kPer; ++i) {
        mine[i] = 0;
        if (i >= per) { break; }                         // (uniform)
        const unsigned p = threadIdx.x * per + i, pc = min(p, pairs - 1);
        const unsigned l = pc / batch, b = pc - l * batch;
        const int32_t r = rows ? rows[b] : static_cast<int32_t>(b);
        const bool live = r >= 0 && static_cast<unsigned>(r) < table_rows;
        const int32_t c = load_count[static_cast<size_t>(l) * table_rows + (live ? r : 0)];
        if (p < pairs && live) { mine[i] = min(n_slots, static_cast<unsigned>(max(c, 0))); }
        sum += mine[i];
    }
    // running total of the threads' sums: inside a wave, then over the waves before it
    unsigned incl = sum;
#pragma unroll
    for (unsigned d = 1; d < 64; d <<= 1) {
        const unsigned v = __shfl_up(incl, d, 64);
        if ((threadIdx.x & 63) >= d) { incl += v; }
    }
    if ((threadIdx.x & 63) == 63) { s_part[threadIdx.x >> 6] = incl; }
    __syncthreads();
    unsigned run = incl - sum;
    for (unsigned w = 0; w < kThreads / 64; ++w) { run += w < threadIdx.x >> 6 ? s_part[w] : 0u; }
#pragma unroll
    for (unsigned i = 0; i < kPer; ++i) {
        if (i >= per) { break; }
        s_total[threadIdx.x * per + i] = run;
        run += mine[i];
    }
    if (threadIdx.x == kThreads - 1) { s_total[kMaxPlannedPairs] = run; }
    __syncthreads();
    // Piece p of slice w, counted on by hand and only where slices have several: a 64-bit division per piece in every wave
    // took longer than a short slice's copy (64 requests x 50 loads of 4 KiB 43.2 us, 38.0 without it (39.7 before there were pieces); 32 layers x 8 x 40 of
    // 16 KiB 151, 139 and 141).
    const unsigned slices = 2u * s_total[kMaxPlannedPairs];
    const unsigned pieces = kWhole ? 1u : static_cast<unsigned>((block_bytes + kLoadPiece - 1) / kLoadPiece);
    const unsigned w_step = gridDim.x / pieces, p_step = gridDim.x % pieces;
    // Pieces of 32 KiB and more: the waves start each one together, so that their reads and writes reach HBM in turns (8 layers x 16
    // x 14 loads of 256 KiB 336 -> 325 us, 8 x 32 x 14 of 64 KiB 178 -> 170; of 8 KiB 35.3 -> 37.4).
    const bool in_step = !kWhole || block_bytes >= 32 * 1024;
    // The cache and pool address of piece p of slice w, and its size; dst null: nothing to copy
    struct Piece {
        const uint8_t* src;
        uint8_t* dst;
        size_t size;
    };
    auto find = [&](unsigned w, unsigned p) -> Piece {
        const unsigned t = w >> 1, kv = w & 1u;
        const size_t off = kWhole ? 0 : static_cast<size_t>(p) * kLoadPiece;
        unsigned lo = 0, hi = pairs;                     // last pair whose running total is <= t
        while (hi - lo > 1) {
            const unsigned mid = (lo + hi) >> 1;
            if (s_total[mid] <= t) { lo = mid; } else { hi = mid; }
        }
        const unsigned l = lo / batch, b = lo - l * batch, j = t - s_total[lo];
        const unsigned row = static_cast<unsigned>(rows ? rows[b] : static_cast<int32_t>(b));
        const int32_t sel = load_sel[(static_cast<size_t>(l) * table_rows + row) * n_slots + j];
        if (sel < 0 || static_cast<unsigned>(sel) >= src_stride) { return {nullptr, nullptr, 0}; }
        const int32_t src = src_table[static_cast<size_t>(row) * src_stride + sel];
        if (src < 0 || static_cast<uint64_t>(src) >= pool_blocks) { return {nullptr, nullptr, 0}; }
        const unsigned dst = static_cast<unsigned>(dst_table[l * dst_layer_stride + static_cast<int64_t>(row) * dst_stride + j]);
        if (dst >= num_blocks) { return {nullptr, nullptr, 0}; }
        return {pool + static_cast<size_t>(src) * pool_block_bytes + lay.slice(store_first_layer + l, kv, block_bytes) + off,
                static_cast<uint8_t*>(layers[l]) + kv * kv_stride + static_cast<size_t>(dst) * block_bytes + off,
                kWhole ? block_bytes : min(kLoadPiece, block_bytes - off)};
    };
    unsigned p = blockIdx.x % pieces, w = blockIdx.x / pieces;
    if constexpr (kT < kThreads) {                       // (the teams meet no barrier)
        constexpr unsigned kTeams = kThreads / kT;
        static_assert(kWhole && kT % 64 == 0, "a team is whole waves and copies whole slices");
        const unsigned team = __builtin_amdgcn_readfirstlane(threadIdx.x / kT);
        for (w = blockIdx.x + team * gridDim.x; w < slices; w += kTeams * gridDim.x) {
            const Piece cur = find(w, 0);
            if (cur.dst) { copy_slice<kT>(cur.dst, cur.src, cur.size, threadIdx.x % kT); }
        }
    } else if constexpr (kWhole) {
        for (; w < slices; w += w_step) {                // (uniform in the workgroup)
            const Piece cur = find(w, 0);
            if (!cur.dst) { continue; }
            if (in_step) { __syncthreads(); }
            copy_slice(cur.dst, cur.src, cur.size);
        }
    } else {
        // Where the next piece lies is found while this one's loads are on their way (8 layers x 16 x 14 loads of 256 KiB 325 -> 307 us;
        // short slices, which are copied in less time than it takes to find the next, only lose by it).
        if (w >= slices) { return; }
        Piece cur = find(w, p), next = {nullptr, nullptr, 0};
        for (;;) {
            w += w_step;
            p += p_step;
            if (p >= pieces) {
                p -= pieces;
                ++w;
            }
            const bool more = w < slices;
            auto look_ahead = [&]() { if (more) { next = find(w, p); } };
            __syncthreads();
            if (cur.dst && cur.size == kStep) {
                copy_trip<kUnroll>(cur.dst, cur.src, threadIdx.x * 16u, look_ahead);
            } else {
                if (cur.dst) { copy_slice(cur.dst, cur.src, cur.size); }
                look_ahead();
            }
            if (!more) { break; }
            cur = next;
        }
    }
}

constexpr size_t kBatchPiece = 2 * kStep;  // 256 KiB

int check_block_args(const void* layers, int n_layers, size_t kv_stride, size_t block_bytes,
                     int num_blocks, const void* ids, int n, const void* staging)
{
    UCM_REQUIRE(num_blocks > 0 && static_cast<size_t>(num_blocks) * block_bytes <= kv_stride,
                "kv move: num_blocks=%d does not fit kv_stride=%zu", num_blocks, kv_stride);
    UCM_REQUIRE(n == 0 || (layers && ids && staging), "kv move: null pointer");
    UCM_REQUIRE(n_layers > 0 && n_layers <= 65535, "kv move: n_layers=%d out of range", n_layers);
    UCM_REQUIRE(n >= 0, "kv move: n=%d", n);
    UCM_REQUIRE(block_bytes > 0 && block_bytes % 16 == 0 && kv_stride % 16 == 0,
                "kv move: block_bytes=%zu / kv_stride=%zu must be multiples of 16", block_bytes, kv_stride);
    UCM_REQUIRE(ucm::aligned16(staging), "kv move: staging not 16-byte aligned");
    return UCM_OK;
}

int stored_layout(const char* name, size_t block_bytes, int rank, int tp_size, StoredLayout* lay)
{
    UCM_REQUIRE(tp_size >= 1 && rank >= 0 && rank < tp_size, "%s: rank=%d tp_size=%d", name, rank, tp_size);
    lay->layer_pitch = 2 * block_bytes * static_cast<size_t>(tp_size);
    lay->slice_base = 2 * block_bytes * static_cast<size_t>(rank);
    return UCM_OK;
}

// Pieces (a 128 KiB trip each) that `slices` slices are cut into between workgroups, or 1: left whole.  A launch takes as long as the
// compute unit with the most to move: of 288 slices of 256 KiB some have two, of their 576 pieces none has more than three.  Where
// that is no less for pieces, whole slices are better balanced still; in launches of more than three slices per unit a workgroup that ends
// with its stores on their way is worth more than that, if no part-trips take places of whole ones.  us, whole | cut: 256 KiB, 128 slices
// 14.9 | 10.0, 192 16.6 | 19.8, 256 21.5 | 21.7 to 24, 288 31 to 33 | 26.8, 352 33 to 37 | 31 to 33, 448 40.2 | 41.8 to 46, 512 45 to 47 | 44 to
// 56, 1000 92 to 108 | 91 to 98, 1296 120 to 130 | 114 to 121, 32 layers x 256 blocks out and back 2845 to 2937 | 2769 to 2856, 5.1 GB
// gathered 1724 to 1821 | 1707 to 1757; 384 KiB, 128 21 | 17, 200 27.0 | 27.5, 288 49 | 39; 512 KiB, 96 25.5 | 17.1, 200 34.2 | 37.8, 352 67.5 |
// 63, 512 88 | 90 to 100, 1296 245 | 230; 160 KiB, 200 12.2 | 15.0, 2048 120 | 129; 192 KiB, 400 27.5 | 30.2.
// (What is never cut has an instance without the division: 16 KiB slices 3.1 us for 200 blocks, 3.4 with it.)
constexpr uint64_t kUnits = 256;         // compute units

unsigned cut_slices(size_t block_bytes, uint64_t grid_x, uint64_t slices)
{
    const uint64_t pieces = (block_bytes + kStep - 1) / kStep;
    const uint64_t most_whole = (slices + kUnits - 1) / kUnits * block_bytes, most_cut = (slices * pieces + kUnits - 1) / kUnits * kStep;
    const bool cut = most_cut < most_whole || (slices > 3 * kUnits && block_bytes >= 2 * kStep);
    return cut && grid_x * pieces <= 0xffffffffu / kThreads ? static_cast<unsigned>(pieces) : 1u;
}

template <bool kToStaging>
int move_blocks(const char* name, const void* const* layers, int n_layers, size_t kv_stride, size_t block_bytes, int num_blocks,
                const int32_t* block_ids, int n, void* staging, const StoredLayout& lay, ucm_stream_t stream)
{
    const unsigned pieces = cut_slices(block_bytes, static_cast<uint64_t>(n), static_cast<uint64_t>(n) * n_layers * 2);
    auto launch = [&](auto kernel, int threads) -> int {
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(n) * pieces, n_layers, 2), dim3(threads), 0, ucm::as_stream(stream),
                           const_cast<void* const*>(layers), kv_stride, block_bytes, block_ids, static_cast<unsigned>(num_blocks),
                           static_cast<uint8_t*>(staging), pieces, lay);
        return ucm::check_hip(hipGetLastError(), name);
    };
    if (block_bytes <= kShortSlice) { return launch(kv_blocks_kernel<kToStaging, false, kShortThreads>, kShortThreads); }
    return pieces > 1 ? launch(kv_blocks_kernel<kToStaging, true, kThreads>, kThreads)
                      : launch(kv_blocks_kernel<kToStaging, false, kThreads>, kThreads);
}

// dst row dst_idx[i] = src row src_idx[i]: one 256-thread workgroup per pair (a step's query rows are a few KiB each,
// so the launch is all latency: every thread has its loads in flight before its first store)
constexpr int kRowThreads = 256;

__global__ __launch_bounds__(kRowThreads) void park_rows_kernel(const uint8_t* __restrict__ src, long long src_rows,
                                                                const int32_t* __restrict__ src_idx, uint8_t* __restrict__ dst,
                                                                long long dst_rows, const int32_t* __restrict__ dst_idx,
                                                                size_t row_bytes)
{
    const long long from = src_idx[blockIdx.x], to = dst_idx ? dst_idx[blockIdx.x] : static_cast<long long>(blockIdx.x);
    if (from < 0 || from >= src_rows || to < 0 || to >= dst_rows) { return; }
    const uint8_t* s = src + static_cast<size_t>(from) * row_bytes;
    uint8_t* d = dst + static_cast<size_t>(to) * row_bytes;
    for (size_t o = threadIdx.x * 16u; o < row_bytes; o += static_cast<size_t>(kRowThreads) * 16 * 4) {
        u32x4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const size_t at = o + static_cast<size_t>(u) * kRowThreads * 16;
            if (at < row_bytes) { v[u] = ucm::gload16(s + at); }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const size_t at = o + static_cast<size_t>(u) * kRowThreads * 16;
            if (at < row_bytes) { ucm::gstore16(d + at, v[u]); }
        }
    }
}

}  // namespace

extern "C" int ucm_copy_batch(void* const* dst, const void* const* src, size_t num, size_t size,
                              ucm_stream_t stream)
{
    UCM_REQUIRE(size % 16 == 0, "ucm_copy_batch: size=%zu must be a multiple of 16", size);
    if (num == 0 || size == 0) { return UCM_OK; }
    UCM_REQUIRE(dst && src, "ucm_copy_batch: null pointer array");
    const size_t pieces = (size + kBatchPiece - 1) / kBatchPiece;
    UCM_REQUIRE(num * pieces <= 0x7fffffffull, "ucm_copy_batch: too many pieces for one launch");
    hipLaunchKernelGGL(copy_batch_kernel, dim3(static_cast<unsigned>(num * pieces)), dim3(kThreads), 0,
                       ucm::as_stream(stream), dst, src, size, kBatchPiece);
    UCM_LAUNCH_CHECK("ucm_copy_batch");
}

extern "C" int ucm_kv_gather_blocks_tp(const void* const* layers, int n_layers, size_t kv_stride,
                                       size_t block_bytes, int num_blocks, const int32_t* block_ids,
                                       int n, void* staging, int rank, int tp_size, ucm_stream_t stream)
{
    if (int rc = check_block_args(layers, n_layers, kv_stride, block_bytes, num_blocks, block_ids, n, staging)) { return rc; }
    StoredLayout lay;
    if (int rc = stored_layout("ucm_kv_gather_blocks", block_bytes, rank, tp_size, &lay)) { return rc; }
    if (n == 0) { return UCM_OK; }
    return move_blocks<true>("ucm_kv_gather_blocks", layers, n_layers, kv_stride, block_bytes, num_blocks, block_ids, n, staging, lay, stream);
}

extern "C" int ucm_kv_gather_blocks(const void* const* layers, int n_layers, size_t kv_stride,
                                    size_t block_bytes, int num_blocks, const int32_t* block_ids,
                                    int n, void* staging, ucm_stream_t stream)
{
    return ucm_kv_gather_blocks_tp(layers, n_layers, kv_stride, block_bytes, num_blocks, block_ids, n, staging, 0, 1, stream);
}

extern "C" int ucm_kv_scatter_blocks_tp(void* const* layers, int n_layers, size_t kv_stride,
                                        size_t block_bytes, int num_blocks, const int32_t* block_ids,
                                        int n, const void* staging, int rank, int tp_size, ucm_stream_t stream)
{
    if (int rc = check_block_args(layers, n_layers, kv_stride, block_bytes, num_blocks, block_ids, n, staging)) { return rc; }
    StoredLayout lay;
    if (int rc = stored_layout("ucm_kv_scatter_blocks", block_bytes, rank, tp_size, &lay)) { return rc; }
    if (n == 0) { return UCM_OK; }
    return move_blocks<false>("ucm_kv_scatter_blocks", layers, n_layers, kv_stride, block_bytes, num_blocks, block_ids, n, const_cast<void*>(staging), lay, stream);
}

extern "C" int ucm_kv_scatter_blocks(void* const* layers, int n_layers, size_t kv_stride,
                                     size_t block_bytes, int num_blocks, const int32_t* block_ids,
                                     int n, const void* staging, ucm_stream_t stream)
{
    return ucm_kv_scatter_blocks_tp(layers, n_layers, kv_stride, block_bytes, num_blocks, block_ids, n, staging, 0, 1, stream);
}

extern "C" int ucm_kv_gather_selected(const void* const* layers, int n_layers, size_t kv_stride,
                                      size_t block_bytes, int num_blocks, const int32_t* phys,
                                      const int32_t* count, int n_req, int phys_stride, const int64_t* dst_off,
                                      const int32_t* region_k, int max_count, void* staging,
                                      int64_t staging_blocks, ucm_stream_t stream)
{
    UCM_REQUIRE(staging_blocks >= 0, "ucm_kv_gather_selected: staging_blocks=%lld", static_cast<long long>(staging_blocks));
    UCM_REQUIRE(n_req == 0 || max_count == 0 || (layers && phys && count && dst_off && region_k && staging),
                "ucm_kv_gather_selected: null pointer");
    UCM_REQUIRE(n_layers > 0 && n_layers * 2 <= 65535, "ucm_kv_gather_selected: n_layers=%d", n_layers);
    UCM_REQUIRE(num_blocks > 0 && static_cast<size_t>(num_blocks) * block_bytes <= kv_stride,
                "ucm_kv_gather_selected: num_blocks=%d does not fit kv_stride=%zu", num_blocks, kv_stride);
    UCM_REQUIRE(n_req >= 0 && n_req <= 65535, "ucm_kv_gather_selected: n_req=%d", n_req);
    UCM_REQUIRE(max_count >= 0 && phys_stride >= max_count,
                "ucm_kv_gather_selected: max_count=%d phys_stride=%d", max_count, phys_stride);
    UCM_REQUIRE(block_bytes > 0 && block_bytes % 16 == 0 && kv_stride % 16 == 0 && ucm::aligned16(staging),
                "ucm_kv_gather_selected: sizes and staging must be multiples of 16");
    if (n_req == 0 || max_count == 0) { return UCM_OK; }
    // What is selected fits the staging area, so slots far beyond its blocks are known to be idle, and pieces would only double them (8
    // layers x 16 requests x 1000 slots of 256 KiB, three in use, 227 us whole, 528 cut; 200 slots, five in use, 130 and 161; 100
    // slots, twenty in use, 462 and 446: level at a tenth).
    const uint64_t slots = static_cast<uint64_t>(max_count) * n_req * n_layers * 2;
    const unsigned pieces = slots / 8 > static_cast<uint64_t>(staging_blocks) ? 1u : cut_slices(block_bytes, static_cast<uint64_t>(max_count), slots);
    auto launch = [&](auto kernel, int threads) -> int {
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(max_count) * pieces, n_req, n_layers * 2), dim3(threads), 0,
                           ucm::as_stream(stream), layers, kv_stride, block_bytes, phys, count, static_cast<unsigned>(num_blocks),
                           static_cast<unsigned>(n_req), static_cast<unsigned>(phys_stride), dst_off, region_k,
                           static_cast<uint8_t*>(staging), static_cast<uint64_t>(staging_blocks), pieces);
        return ucm::check_hip(hipGetLastError(), "ucm_kv_gather_selected");
    };
    if (block_bytes <= kShortSlice) { return launch(kv_gather_selected_kernel<false, kShortThreads>, kShortThreads); }
    return pieces > 1 ? launch(kv_gather_selected_kernel<true, kThreads>, kThreads)
                      : launch(kv_gather_selected_kernel<false, kThreads>, kThreads);
}

extern "C" int ucm_kv_load_planned_tp(void* const* layers, int n_layers, size_t kv_stride, size_t block_bytes,
                                      int num_blocks, const void* pool, int64_t pool_blocks, size_t pool_block_bytes,
                                      int store_first_layer, const int32_t* load_sel, int n_slots,
                                      const int32_t* src_table, int src_stride, const int32_t* dst_table,
                                      int dst_stride, int64_t dst_layer_stride, const int32_t* load_count,
                                      const int32_t* rows, int batch, int table_rows, int rank, int tp_size,
                                      ucm_stream_t stream)
{
    StoredLayout lay;
    if (int rc = stored_layout("ucm_kv_load_planned", block_bytes, rank, tp_size, &lay)) { return rc; }
    UCM_REQUIRE(batch >= 0 && n_slots >= 0 && table_rows > 0, "ucm_kv_load_planned: batch=%d n_slots=%d table_rows=%d", batch,
                n_slots, table_rows);
    if (batch == 0 || n_slots == 0) { return UCM_OK; }
    UCM_REQUIRE(layers && pool && load_sel && src_table && dst_table, "ucm_kv_load_planned: null pointer");
    UCM_REQUIRE(n_layers > 0 && n_layers * 2 <= 65535 && batch <= 65535, "ucm_kv_load_planned: n_layers=%d batch=%d", n_layers, batch);
    UCM_REQUIRE(num_blocks > 0 && static_cast<size_t>(num_blocks) * block_bytes <= kv_stride,
                "ucm_kv_load_planned: num_blocks=%d does not fit kv_stride=%zu", num_blocks, kv_stride);
    UCM_REQUIRE(block_bytes > 0 && block_bytes % 16 == 0 && kv_stride % 16 == 0 && pool_block_bytes % 16 == 0 &&
                    ucm::aligned16(pool),
                "ucm_kv_load_planned: sizes and pool must be multiples of 16");
    UCM_REQUIRE(store_first_layer >= 0 && pool_blocks >= 0 &&
                    static_cast<size_t>(store_first_layer + n_layers) * lay.layer_pitch <= pool_block_bytes,
                "ucm_kv_load_planned: layers %d..%d do not fit a stored block of %zu bytes", store_first_layer,
                store_first_layer + n_layers - 1, pool_block_bytes);
    UCM_REQUIRE(src_stride >= 1 && dst_stride >= n_slots && dst_layer_stride >= 0,
                "ucm_kv_load_planned: src_stride=%d dst_stride=%d n_slots=%d", src_stride, dst_stride, n_slots);
    // A short plan of short slices goes slot by slot: a few idle workgroups cost less than the running total of the counts (1 layer x 8
    // x 20 of 4 KiB 2.6 and 4.4 us, 2 x 16 x 50, all load, 6.9 and 7.0, 8 x 16 x 50 with two loads a row 5.9 and 4.8).
    const bool short_slices = block_bytes <= kShortSlice;
    const bool few_slots = short_slices && static_cast<int64_t>(n_slots) * batch * n_layers * 2 <= 4096;
    if (load_count && !few_slots && static_cast<unsigned>(n_layers) * static_cast<unsigned>(batch) <= kMaxPlannedPairs) {
        // the rows' counts say exactly what there is to copy: persistent workgroups share it evenly
        const auto kernel = short_slices                ? kv_load_counted_kernel<true, kTeamThreads>
                            : block_bytes <= kLoadPiece ? kv_load_counted_kernel<true, kThreads>
                                                        : kv_load_counted_kernel<false, kThreads>;
        hipLaunchKernelGGL(kernel, dim3(short_slices ? kTeamGroups : 1024u), dim3(kThreads), 0, ucm::as_stream(stream), layers, kv_stride,
                           block_bytes, static_cast<unsigned>(num_blocks), static_cast<const uint8_t*>(pool),
                           static_cast<uint64_t>(pool_blocks), pool_block_bytes, static_cast<unsigned>(store_first_layer),
                           load_sel, static_cast<unsigned>(n_slots), src_table, static_cast<unsigned>(src_stride), dst_table,
                           static_cast<unsigned>(dst_stride), dst_layer_stride, load_count, rows,
                           static_cast<unsigned>(table_rows), static_cast<unsigned>(batch), static_cast<unsigned>(n_layers), lay);
    } else {
        // The entries to load are scattered over a row (or there are too many rows for the counted kernel's table).
        const int64_t table = static_cast<int64_t>(batch) * n_layers * 2;
        const auto pieces = [&](size_t piece) { return static_cast<int64_t>((block_bytes + piece - 1) / piece); };
        auto follow_slots = [&](auto kernel, int threads) {
            const unsigned per_slot = static_cast<unsigned>(pieces(static_cast<size_t>(threads) * 16 * kUnroll));
            hipLaunchKernelGGL(kernel, dim3(n_slots * per_slot, batch, n_layers * 2), dim3(threads), 0, ucm::as_stream(stream), layers,
                               kv_stride, block_bytes, static_cast<unsigned>(num_blocks), static_cast<const uint8_t*>(pool),
                               static_cast<uint64_t>(pool_blocks), pool_block_bytes, static_cast<unsigned>(store_first_layer),
                               load_sel, static_cast<unsigned>(n_slots), src_table, static_cast<unsigned>(src_stride), dst_table,
                               static_cast<unsigned>(dst_stride), dst_layer_stride, load_count, rows,
                               static_cast<unsigned>(table_rows), per_slot, lay);
        };
        // (64 KiB slices in small launches: 4 requests x 300 slots 51 us with 1024 threads, 55 with 512; in large ones idle
        // workgroups count: 8 layers x 8 requests x 100 slots of 128 KiB, one in fifty loads, 29 us with 512 and 32 with 1024.
        // A row of more than a million slots does not fit the grid; the list takes any number.)
        const bool fits = n_slots <= 1 << 20;
        if (fits && block_bytes <= kStep / 4) {
            follow_slots(kv_load_slot_kernel<256>, 256);
        } else if (n_slots * pieces(kLoadPiece) * table <= 4096) {
            follow_slots(kv_load_slot_kernel<kThreads>, kThreads);
        } else if (fits && block_bytes <= kStep) {
            follow_slots(kv_load_slot_kernel<512>, 512);
        } else {
            // about 4096 workgroups over all rows, at least four a row, never more than a row has pieces
            const unsigned gx = static_cast<unsigned>(std::min(n_slots * pieces(kLoadPiece), std::max<int64_t>(4, 4096 / table)));
            hipLaunchKernelGGL(kv_load_planned_kernel, dim3(gx, batch, n_layers * 2), dim3(kThreads), 0,
                               ucm::as_stream(stream), layers, kv_stride, block_bytes, static_cast<unsigned>(num_blocks),
                               static_cast<const uint8_t*>(pool), static_cast<uint64_t>(pool_blocks), pool_block_bytes,
                               static_cast<unsigned>(store_first_layer), load_sel, static_cast<unsigned>(n_slots), src_table,
                               static_cast<unsigned>(src_stride), dst_table, static_cast<unsigned>(dst_stride), dst_layer_stride,
                               load_count, rows, static_cast<unsigned>(table_rows), lay);
        }
    }
    UCM_LAUNCH_CHECK("ucm_kv_load_planned");
}

extern "C" int ucm_kv_load_planned(void* const* layers, int n_layers, size_t kv_stride, size_t block_bytes,
                                   int num_blocks, const void* pool, int64_t pool_blocks, size_t pool_block_bytes,
                                   int store_first_layer, const int32_t* load_sel, int n_slots,
                                   const int32_t* src_table, int src_stride, const int32_t* dst_table,
                                   int dst_stride, int64_t dst_layer_stride, const int32_t* load_count,
                                   const int32_t* rows, int batch, int table_rows, ucm_stream_t stream)
{
    return ucm_kv_load_planned_tp(layers, n_layers, kv_stride, block_bytes, num_blocks, pool, pool_blocks, pool_block_bytes,
                                  store_first_layer, load_sel, n_slots, src_table, src_stride, dst_table, dst_stride,
                                  dst_layer_stride, load_count, rows, batch, table_rows, 0, 1, stream);
}

extern "C" int ucm_park_rows(const void* src, int64_t src_rows, const int32_t* src_idx, void* dst, int64_t dst_rows,
                             const int32_t* dst_idx, int n, size_t row_bytes, ucm_stream_t stream)
{
    UCM_REQUIRE(n >= 0 && src_rows >= 0 && dst_rows >= 0, "ucm_park_rows: n=%d src_rows=%lld dst_rows=%lld", n,
                static_cast<long long>(src_rows), static_cast<long long>(dst_rows));
    UCM_REQUIRE(row_bytes > 0 && row_bytes % 16 == 0, "ucm_park_rows: row_bytes=%zu must be a positive multiple of 16", row_bytes);
    if (n == 0) { return UCM_OK; }
    UCM_REQUIRE(src && src_idx && dst, "ucm_park_rows: null pointer");
    UCM_REQUIRE(ucm::aligned16(src) && ucm::aligned16(dst), "ucm_park_rows: src and dst must be 16-byte aligned");
    hipLaunchKernelGGL(park_rows_kernel, dim3(static_cast<unsigned>(n)), dim3(kRowThreads), 0, ucm::as_stream(stream),
                       static_cast<const uint8_t*>(src), static_cast<long long>(src_rows), src_idx, static_cast<uint8_t*>(dst),
                       static_cast<long long>(dst_rows), dst_idx, row_bytes);
    UCM_LAUNCH_CHECK("ucm_park_rows");
}
