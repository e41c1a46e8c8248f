// Block representatives: per (kv head, dim) mean over a cache block's tokens,
// fp32 accumulation in token order (column-independent, so every thread owns
// whole columns and the order inside a column is the reference's).
//
// HBM-bound: block_size*row*2 bytes read per block, row*4 written.  A token
// row of the key cache ([kv_heads][head_dim] bf16, or fp16 for a model that runs in float16) is contiguous, so a thread
// owns 8 adjacent columns (one 16-byte load per token) and a workgroup of 128
// threads covers 1024 columns = one whole Llama-shape row; the token loop is
// unrolled 16 deep so 16 x 2 KiB of loads are in flight per workgroup.
#include <algorithm>

#include "common.h"

namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 128;
constexpr int kCols = 8;      // bf16 columns per thread
constexpr int kUnroll = 16;   // token rows in flight
constexpr unsigned kStreamThreads = 256;                  // of block_mean_stream_kernel,
constexpr unsigned kStreamGroups = 256;                   // one workgroup on each compute unit
constexpr unsigned kFewGroups = 256;                      // see block_mean_kernel
constexpr unsigned kStreamLeast = 192;                    // groups: see block_mean_stream_kernel
constexpr uint64_t kStreamBytes = uint64_t{256} << 20;    // see block_mean_stream_kernel
constexpr unsigned kKeepBytes = 158 * 1024;               // of the 160 KiB of LDS: means on their way out

__device__ __forceinline__ float bf16_lo(unsigned w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(unsigned w) { return __uint_as_float(w & 0xffff0000u); }

__device__ __forceinline__ float round_bf16(float x)
{
    unsigned u = __float_as_uint(x);
    if ((u & 0x7fffffffu) > 0x7f800000u) { return __uint_as_float((u | 0x00400000u) & 0xffff0000u); }
    u += 0x7fffu + ((u >> 16) & 1u);
    return __uint_as_float(u & 0xffff0000u);
}

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// fp32 -> fp16 -> fp32, the fp32 value rounded once more.  The value is made opaque first: handed a product, the
// compiler otherwise folds the multiplication into a mixed-precision instruction that rounds the exact product
// straight to fp16 - one rounding instead of the two the reference's arithmetic has (seen at a tie: 1/5 of a sum).
__device__ __forceinline__ float round_f16(float x)
{
    asm volatile("" : "+v"(x));
    return static_cast<float>(static_cast<_Float16>(x));
}

// kAbs: the absolute values (a pair of 16-bit floats of either kind loses its two sign bits with one AND);
// kF16: the cache holds fp16 keys, not bf16 ones
template <bool kAbs, bool kF16>
__device__ __forceinline__ void widen(u32x4 v, float (&f)[kCols])
{
    if (kAbs) { v.x &= 0x7fff7fffu; v.y &= 0x7fff7fffu; v.z &= 0x7fff7fffu; v.w &= 0x7fff7fffu; }
    if (kF16) {
        const unsigned w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const f16x2 p = __builtin_bit_cast(f16x2, w[j]);
            f[2 * j] = static_cast<float>(p[0]);
            f[2 * j + 1] = static_cast<float>(p[1]);
        }
        return;
    }
    f[0] = bf16_lo(v.x); f[1] = bf16_hi(v.x);
    f[2] = bf16_lo(v.y); f[3] = bf16_hi(v.y);
    f[4] = bf16_lo(v.z); f[5] = bf16_hi(v.z);
    f[6] = bf16_lo(v.w); f[7] = bf16_hi(v.w);
}

// kN rows from row t on; the compiler neither sinks the loads to their use nor moves other work in front of them
template <int kN>
__device__ __forceinline__ void load_rows(u32x4 (&v)[kN], const uint16_t* __restrict__ base, unsigned row, unsigned t)
{
#pragma unroll
    for (int u = 0; u < kN; ++u) { v[u] = ucm::gload16_nt(base + static_cast<size_t>(t + u) * row); }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

template <bool kAbs, bool kF16, int kN>
__device__ __forceinline__ void add_loaded(const u32x4 (&v)[kN], float (&acc)[kCols])
{
#pragma unroll
    for (int u = 0; u < kN; ++u) {
        float f[kCols];
        widen<kAbs, kF16>(v[u], f);
#pragma unroll
        for (int c = 0; c < kCols; ++c) { acc[c] = acc[c] + f[c]; }
    }
}

// acc += token rows t .. t+kN-1, in that order, all kN loads issued before the first add
template <int kN, bool kAbs, bool kF16>
__device__ __forceinline__ void add_rows(const uint16_t* __restrict__ base, unsigned row, unsigned t, float (&acc)[kCols])
{
    u32x4 v[kN];
#pragma unroll
    for (int u = 0; u < kN; ++u) { v[u] = ucm::gload16_nt(base + static_cast<size_t>(t + u) * row); }
    add_loaded<kAbs, kF16>(v, acc);
}

// A thread's eight sums as the table holds them: means, rounded as the mode asks; one 16-byte piece of a bf16 table, two of an
// fp32 one.
template <bool kF16>
__device__ __forceinline__ void pack_means(float (&acc)[kCols], unsigned block_size, int round_to_bf16, u32x4 (&o)[2])
{
    const float inv = 1.0f / static_cast<float>(block_size);
#pragma unroll
    for (int c = 0; c < kCols; ++c) {
        acc[c] = acc[c] * inv;
        if (round_to_bf16) { acc[c] = kF16 ? round_f16(acc[c]) : round_bf16(acc[c]); }
    }
    if (round_to_bf16 == 2) {                            // bf16 table: the rounded means themselves
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            o[0][j] = (__float_as_uint(acc[2 * j]) >> 16) | (__float_as_uint(acc[2 * j + 1]) & 0xffff0000u);
        }
        o[1] = o[0];
        return;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        o[0][j] = __float_as_uint(acc[j]);
        o[1][j] = __float_as_uint(acc[4 + j]);
    }
}

template <bool kHint>
__device__ __forceinline__ void store_means(const u32x4 (&o)[2], float* __restrict__ repre, int64_t repre_layer_stride, unsigned layer,
                                            unsigned slot, unsigned row, unsigned col, int round_to_bf16)
{
    const int64_t at = static_cast<int64_t>(layer) * repre_layer_stride + static_cast<int64_t>(static_cast<size_t>(slot) * row + col);
    auto put = [](void* p, const u32x4& v) {
        if (kHint) { ucm::gstore16_nt(p, v); } else { ucm::gstore16(p, v); }
    };
    if (round_to_bf16 == 2) {
        put(reinterpret_cast<uint16_t*>(repre) + at, o[0]);
        return;
    }
    put(repre + at, o[0]);
    put(repre + at + 4, o[1]);
}

// kFew: no more workgroups than compute units, each of which is then alone with its chain of trips to memory: the next
// 16 tokens are in flight while the current ones are added (128 blocks of 128 tokens 12.1 -> 8.6 us, 256 blocks 14.2 -> 11.9 us, of 32
// tokens 3.9 -> 3.7, of 16 tokens, whose next ones are the same again, 3.2 or, in some processes, 4.2 -> 3.4; with more workgroups
// others fill the gaps, and the registers of a second set cost more: 400 blocks 18.5 -> 19.3 us).
//
// grid: x = block index in the list * col_groups + column group of 1024, y = layer; rows narrower than 1024
// columns whose thread count divides the workgroup (a tensor-parallel rank's 4, 2 or 1 kv heads of 128) share a
// workgroup, items_per_group list entries side by side, so that no lane idles
template <bool kAbs, bool kF16, bool kFew>
__global__ __launch_bounds__(kThreads) void block_mean_kernel(
    const void* const* __restrict__ k_layers, const int32_t* __restrict__ block_ids,
    const int32_t* __restrict__ slots, unsigned num_blocks, unsigned repre_rows, unsigned block_size,
    unsigned row /* kv_heads*head_dim */, float* __restrict__ repre, int64_t repre_layer_stride,
    int round_to_bf16, unsigned col_groups, unsigned items_per_group, unsigned n_items)
{
    unsigned item, col;
    if (items_per_group > 1) {
        const unsigned per_item = kThreads / items_per_group;
        item = blockIdx.x * items_per_group + threadIdx.x / per_item;
        col = (threadIdx.x % per_item) * kCols;
        if (item >= n_items) { return; }
    } else {
        item = blockIdx.x / col_groups;
        col = ((blockIdx.x % col_groups) * kThreads + threadIdx.x) * kCols;
    }
    if (col >= row) { return; }
    const unsigned id = static_cast<unsigned>(block_ids[item]);
    const unsigned slot = static_cast<unsigned>(slots[item]);
    if (id >= num_blocks || slot >= repre_rows) { return; }  // never dereference a bad id

    const uint16_t* base = static_cast<const uint16_t*>(k_layers[blockIdx.y]) +
                           static_cast<size_t>(id) * block_size * row + col;
    float acc[kCols];
    if constexpr (kFew) {
        u32x4 va[kUnroll], vb[kUnroll];
        load_rows(va, base, row, 0);
#pragma unroll
        for (int c = 0; c < kCols; ++c) { acc[c] = -0.0f; }       // -0 + x == x for every x, signed zeros included
        for (unsigned t = 0; t < block_size; t += 2 * kUnroll) {
            load_rows(vb, base, row, min(t + kUnroll, block_size - kUnroll));
            add_loaded<kAbs, kF16>(va, acc);
            load_rows(va, base, row, min(t + 2 * kUnroll, block_size - kUnroll));
            if (t + kUnroll < block_size) { add_loaded<kAbs, kF16>(vb, acc); }
        }
    } else {
        widen<kAbs, kF16>(ucm::gload16(base), acc);  // acc = token 0

        unsigned t = 1;
        // full groups of kUnroll tokens: loads first, then the ordered adds; what is left (all of a 16-token block
        // after its first token) goes in groups of 8, 4, 2 and 1, each with its loads issued together
        for (; t + kUnroll <= block_size; t += kUnroll) { add_rows<kUnroll, kAbs, kF16>(base, row, t, acc); }
        if (t + 8 <= block_size) { add_rows<8, kAbs, kF16>(base, row, t, acc); t += 8; }
        if (t + 4 <= block_size) { add_rows<4, kAbs, kF16>(base, row, t, acc); t += 4; }
        if (t + 2 <= block_size) { add_rows<2, kAbs, kF16>(base, row, t, acc); t += 2; }
        if (t < block_size) { add_rows<1, kAbs, kF16>(base, row, t, acc); }
    }

    u32x4 o[2];
    pack_means<kF16>(acc, block_size, round_to_bf16, o);
    store_means<false>(o, repre, repre_layer_stride, blockIdx.y, slot, row, col, round_to_bf16);
}

// Large launches.  What bounds them is HBM, and it serves a few small writes among a stream of reads badly: 4.3 GB of keys
// (32 layers x 512 blocks of 128 tokens x 8 heads) take 690 us in block_mean_kernel, 604 without its stores (7.1 TB/s), though
// the means are 1/128 of the bytes.  So the workgroups are persistent, one per compute unit: each steps over (layer, list
// entries) groups, with the loads of the next unit - of the same block or the next one - in flight while the current one is
// added, and keeps the means in LDS until that is full or its work is done: 632 us (6.8 TB/s), 655 when they leave eight
// groups at a time, 725 -> 672 us into an fp32 table.  Four workgroups of 128 threads per compute unit: 667 us.  How much that brings depends on
// the memory a process gets: 691 -> 633, 710 -> 662, and on one machine 645 either way.
// For more than 256 MiB of keys, what the memory-side cache holds, a group for three in four of the compute units, and not for blocks of
// 16 tokens into an fp32 table, whose means fill LDS too often (1000 MiB 200 | 224, into a bf16 one 186 | 183).  us, block_mean_kernel | this, 8 heads: 256 MiB in blocks of 16, 64, 128, 256 tokens 47.5 | 46.4, 43.7 | 43.3, 42.2 | 43.2, 41.9 | 43.4; 271
// and 289 MiB 46.7 | 43.7 and 51.2 | 49.1; 384 MiB 72 | 69, 64.3 | 63.0, 61.8 | 61.6, 60.3 | 60.1; 2 GiB 396 | 382, 369 | 342, 355 | 337,
// 340 | 334.  256 groups of 512 tokens 163 | 165, 192 of 512 and of 1024 tokens 61.7 | 59.1 and 125 | 121; 128 of 512 tokens 44 | 51,
// 96 of 1024 tokens 73 | 85, 64 of 2048 tokens 142 | 166.
//
// The block is whole 16-token units.  kT threads take `share` = kT / per_item list entries side by side (per_item = row / 8
// threads), or, of a row too wide for that, one of col_groups column groups.  kWaveEntry: a wave's threads belong to one entry,
// whose id and slot are then scalar loads.  A thread reads back from LDS what it wrote itself, so there is no barrier.
template <bool kAbs, bool kF16, bool kWaveEntry>
__global__ __launch_bounds__(kStreamThreads) void block_mean_stream_kernel(
    const void* const* __restrict__ k_layers, const int32_t* __restrict__ block_ids,
    const int32_t* __restrict__ slots, unsigned num_blocks, unsigned repre_rows, unsigned block_size,
    unsigned row /* kv_heads*head_dim */, float* __restrict__ repre, int64_t repre_layer_stride,
    int round_to_bf16, unsigned col_groups, unsigned share, unsigned n_items, unsigned groups, unsigned total, unsigned keep)
{
    constexpr unsigned kT = kStreamThreads;
    extern __shared__ u32x4 kept_means[];                // [keep][1 or 2][kT] pieces, then [keep][row_slots] rows of the table
    constexpr unsigned kNoRow = 0xffffffffu;
    const unsigned per_item = share > 1 ? row / kCols : kT;
    unsigned sub = threadIdx.x / per_item;
    if (kWaveEntry) { sub = __builtin_amdgcn_readfirstlane(sub); }
    const unsigned col_in = (threadIdx.x - sub * per_item) * kCols;
    const unsigned pieces = round_to_bf16 == 2 ? 1u : 2u;
    // (no two waves share a place for their rows either: one may be writing out while the other still adds)
    const unsigned row_slots = max(share, kT / 64), row_slot = share >= kT / 64 ? sub : threadIdx.x / 64;
    unsigned* kept_rows = reinterpret_cast<unsigned*>(kept_means + keep * pieces * kT);

    struct Unit {
        unsigned g, layer, t, slot, col;                 // slot: kNoRow if the entry does not exist or names no block or row
        const uint16_t* base;
    };
    auto split = [&](unsigned g, unsigned& layer, unsigned& item, unsigned& col) {
        layer = g / groups;
        const unsigned idx = g - layer * groups;
        item = share > 1 ? idx * share + sub : idx / col_groups;
        col = share > 1 ? col_in : (idx % col_groups) * (kT * kCols) + col_in;
    };
    unsigned next_id = 0, next_slot = 0;                 // entries of lanes: fetched one group ahead, or every group would wait for them
    auto fetch_entry = [&](unsigned g) {
        unsigned layer, item, col;
        split(g, layer, item, col);
        item = min(item, n_items - 1);
        next_id = static_cast<unsigned>(block_ids[item]);
        next_slot = static_cast<unsigned>(slots[item]);
    };
    auto open = [&](Unit& u, unsigned g) {
        unsigned item;
        u.g = g;
        u.t = 0;
        split(g, u.layer, item, u.col);
        if (kWaveEntry) { fetch_entry(g); }
        const unsigned id = next_id;
        // loads are unconditional: what does not exist reads the layer's first block (a bad id is never followed)
        u.slot = item < n_items && id < num_blocks && next_slot < repre_rows ? next_slot : kNoRow;
        u.base = static_cast<const uint16_t*>(k_layers[u.layer]) +
                 static_cast<size_t>(id < num_blocks ? id : 0u) * block_size * row + min(u.col, row - kCols);
        if (!kWaveEntry) { fetch_entry(min(g + gridDim.x, total - 1)); }
    };
    auto next_of = [&](const Unit& u, bool& exists) -> Unit {
        Unit n = u;
        n.t = u.t + kUnroll;
        if (n.t >= block_size) {
            exists = u.g + gridDim.x < total;
            if (exists) { open(n, u.g + gridDim.x); }
        }
        return n;
    };
    unsigned kept = 0, first = blockIdx.x;               // groups whose means are in LDS, and the first of them
    auto write_out = [&]() {
        for (unsigned k = 0; k < kept; ++k, first += gridDim.x) {
            unsigned layer, item, col;
            split(first, layer, item, col);
            const unsigned slot = kept_rows[k * row_slots + row_slot];
            u32x4 o[2];
            o[0] = kept_means[k * pieces * kT + threadIdx.x];
            o[1] = pieces == 2 ? kept_means[(k * pieces + 1) * kT + threadIdx.x] : o[0];
            if (slot != kNoRow && col < row) { store_means<true>(o, repre, repre_layer_stride, layer, slot, row, col, round_to_bf16); }
        }
        kept = 0;
    };
    float acc[kCols];
    auto finish = [&](const u32x4 (&v)[kUnroll], const Unit& u, bool exists) {
#pragma unroll
        for (int c = 0; c < kCols; ++c) { acc[c] = u.t == 0 ? -0.0f : acc[c]; }   // -0 + x == x for every x, signed zeros included
        add_loaded<kAbs, kF16>(v, acc);
        if (exists && u.t + kUnroll >= block_size) {     // (the same for all threads)
            if (kept == keep) { write_out(); }
            u32x4 o[2];
            pack_means<kF16>(acc, block_size, round_to_bf16, o);
            kept_means[kept * pieces * kT + threadIdx.x] = o[0];
            if (pieces == 2) { kept_means[(kept * pieces + 1) * kT + threadIdx.x] = o[1]; }
            kept_rows[kept * row_slots + row_slot] = u.slot;      // (threads that share a place write the same number)
            ++kept;
        }
    };
    if (!kWaveEntry) { fetch_entry(blockIdx.x); }
    Unit a;
    open(a, blockIdx.x);
    u32x4 va[kUnroll], vb[kUnroll];
    load_rows(va, a.base, row, a.t);
    // two units per round and one way out, at the end (a second exit between the halves would make the compiler wait at the
    // loop's head for every load it believes may have just been issued)
    for (;;) {
        bool has_b = true, has_c = true;
        const Unit b = next_of(a, has_b);
        load_rows(vb, (has_b ? b : a).base, row, (has_b ? b : a).t);
        finish(va, a, true);
        const Unit c = has_b ? next_of(b, has_c) : b;
        has_c = has_c && has_b;
        load_rows(va, (has_c ? c : a).base, row, (has_c ? c : a).t);
        finish(vb, has_b ? b : a, has_b);
        if (!has_c) { break; }
        a = c;
    }
    write_out();
}

struct MeanArgs {
    const void* const* k_layers;
    const int32_t *block_ids, *slots;
    unsigned num_blocks, repre_rows, block_size, row, n_items, n_layers;
    float* repre;
    int64_t repre_layer_stride;
    int mode;
    bool of_abs, keys_f16;
};

// How a launch's work falls into groups: `share` list entries side by side, or one of an entry's column groups.
struct StreamGroups {
    unsigned share, col_groups, groups, total;           // groups: of a layer
};
StreamGroups stream_groups(const MeanArgs& a)
{
    constexpr unsigned kT = kStreamThreads;
    const unsigned per_item = a.row / kCols, share = per_item < kT && kT % per_item == 0 ? kT / per_item : 1u;
    const unsigned col_groups = share > 1 ? 1u : (per_item + kT - 1) / kT;
    const unsigned groups = share > 1 ? (a.n_items + share - 1) / share : a.n_items * col_groups;
    return {share, col_groups, groups, groups * a.n_layers};
}

int launch_stream(const MeanArgs& a, const StreamGroups& g, hipStream_t s)
{
    constexpr unsigned kT = kStreamThreads;
    const unsigned share = g.share, total = g.total;
    const unsigned each = (total + kStreamGroups - 1) / kStreamGroups, wgs = (total + each - 1) / each;
    const unsigned group_bytes = (a.mode == UCM_MEAN_BF16_STORE ? 16u : 32u) * kT + std::max(share, kT / 64) * 4;
    const unsigned keep = std::min(each, kKeepBytes / group_bytes);
    const unsigned lds = std::max(keep * group_bytes, 82u * 1024u);      // more than half of a compute unit's: never two workgroups on one
    const bool wave_entry = share == 1 || a.row / kCols % 64 == 0;
    auto launch = [&](auto kernel) -> int {
        if (int rc = ucm::allow_lds(kernel, kKeepBytes, "ucm_block_mean")) { return rc; }
        hipLaunchKernelGGL(kernel, dim3(wgs), dim3(kT), lds, s, a.k_layers, a.block_ids, a.slots, a.num_blocks, a.repre_rows, a.block_size,
                           a.row, a.repre, a.repre_layer_stride, a.mode, g.col_groups, share, a.n_items, g.groups, total, keep);
        return ucm::check_hip(hipGetLastError(), "ucm_block_mean");
    };
    if (wave_entry) {
        if (a.keys_f16) { return a.of_abs ? launch(block_mean_stream_kernel<true, true, true>) : launch(block_mean_stream_kernel<false, true, true>); }
        return a.of_abs ? launch(block_mean_stream_kernel<true, false, true>) : launch(block_mean_stream_kernel<false, false, true>);
    }
    if (a.keys_f16) { return a.of_abs ? launch(block_mean_stream_kernel<true, true, false>) : launch(block_mean_stream_kernel<false, true, false>); }
    return a.of_abs ? launch(block_mean_stream_kernel<true, false, false>) : launch(block_mean_stream_kernel<false, false, false>);
}

}  // namespace

extern "C" int ucm_block_mean(const void* const* k_layers, int n_layers, int num_blocks,
                              const int32_t* block_ids, const int32_t* slots, int n, int block_size,
                              int kv_heads, int head_dim, void* repre, int repre_rows,
                              int64_t repre_layer_stride, int mode, ucm_stream_t stream)
{
    UCM_REQUIRE(n >= 0, "ucm_block_mean: n=%d", n);
    if (n == 0) { return UCM_OK; }  // an empty list has no pointers to check
    UCM_REQUIRE(k_layers && block_ids && slots && repre, "ucm_block_mean: null pointer");
    UCM_REQUIRE(n_layers > 0 && n_layers <= 65535, "ucm_block_mean: n_layers=%d", n_layers);
    UCM_REQUIRE(block_size > 0 && kv_heads > 0 && head_dim > 0 && num_blocks > 0 && repre_rows > 0,
                "ucm_block_mean: non-positive shape");
    const bool of_abs = (mode & UCM_MEAN_ABS) != 0, keys_f16 = (mode & UCM_MEAN_KEYS_F16) != 0;
    mode &= ~(UCM_MEAN_ABS | UCM_MEAN_KEYS_F16);
    UCM_REQUIRE(mode == UCM_MEAN_F32 || mode == UCM_MEAN_BF16_ROUND || mode == UCM_MEAN_BF16_STORE,
                "ucm_block_mean: mode=%d", mode);
    UCM_SUPPORTED(!(keys_f16 && mode == UCM_MEAN_BF16_STORE), "ucm_block_mean: no bf16 table from an fp16 key cache "
                  "(UCM_MEAN_F32 or UCM_MEAN_BF16_ROUND, which then rounds to fp16)");
    const unsigned row = static_cast<unsigned>(kv_heads) * static_cast<unsigned>(head_dim);
    UCM_SUPPORTED(row % kCols == 0, "ucm_block_mean: kv_heads*head_dim=%u must be a multiple of %d", row, kCols);
    UCM_REQUIRE(repre_layer_stride >= static_cast<int64_t>(repre_rows) * row || n_layers == 1,
                "ucm_block_mean: repre_layer_stride=%lld smaller than one layer's table",
                static_cast<long long>(repre_layer_stride));
    UCM_REQUIRE(ucm::aligned16(repre) && (repre_layer_stride % (mode == UCM_MEAN_BF16_STORE ? 8 : 4) == 0),
                "ucm_block_mean: repre not 16-byte aligned");
    const unsigned gx = (row / kCols + kThreads - 1) / kThreads;
    UCM_REQUIRE(static_cast<uint64_t>(n) * gx <= 0x7fffffffull, "ucm_block_mean: too many blocks for one launch");
    const unsigned per_item = row / kCols;               // threads a list entry needs
    const unsigned share = (per_item < kThreads && kThreads % per_item == 0) ? kThreads / per_item : 1u;
    const unsigned groups = share > 1 ? (static_cast<unsigned>(n) + share - 1) / share : static_cast<unsigned>(n) * gx;
    const bool whole_units = block_size % kUnroll == 0;
    if (whole_units && static_cast<uint64_t>(n) * n_layers * gx <= 0x7fffffffull) {
        const MeanArgs a = {k_layers, block_ids, slots, static_cast<unsigned>(num_blocks), static_cast<unsigned>(repre_rows),
                            static_cast<unsigned>(block_size), row, static_cast<unsigned>(n), static_cast<unsigned>(n_layers),
                            static_cast<float*>(repre), repre_layer_stride, mode, of_abs, keys_f16};
        const uint64_t bytes = static_cast<uint64_t>(n) * n_layers * block_size * row * 2;
        const StreamGroups g = stream_groups(a);
        const bool few_means = mode == UCM_MEAN_BF16_STORE || block_size >= 2 * kUnroll;      // at most a sixteenth of the keys' bytes
        if (bytes > kStreamBytes && g.total >= kStreamLeast && few_means) { return launch_stream(a, g, ucm::as_stream(stream)); }
    }
#define UCM_BLOCK_MEAN_ARGS dim3(groups, n_layers), dim3(kThreads), 0, ucm::as_stream(stream), k_layers, block_ids, slots, \
        static_cast<unsigned>(num_blocks), static_cast<unsigned>(repre_rows), static_cast<unsigned>(block_size), row,       \
        static_cast<float*>(repre), repre_layer_stride, mode, gx, share, static_cast<unsigned>(n)
#define UCM_BLOCK_MEAN(ABS, F16)                                                                                        \
    do {                                                                                                             \
        if (few) { hipLaunchKernelGGL((block_mean_kernel<ABS, F16, true>), UCM_BLOCK_MEAN_ARGS); }                   \
        else { hipLaunchKernelGGL((block_mean_kernel<ABS, F16, false>), UCM_BLOCK_MEAN_ARGS); }                      \
    } while (0)
    const bool few = whole_units && static_cast<uint64_t>(groups) * n_layers <= kFewGroups;
    if (keys_f16) {
        if (of_abs) { UCM_BLOCK_MEAN(true, true); } else { UCM_BLOCK_MEAN(false, true); }
    } else {
        if (of_abs) { UCM_BLOCK_MEAN(true, false); } else { UCM_BLOCK_MEAN(false, false); }
    }
#undef UCM_BLOCK_MEAN
#undef UCM_BLOCK_MEAN_ARGS
    UCM_LAUNCH_CHECK("ucm_block_mean");
}
