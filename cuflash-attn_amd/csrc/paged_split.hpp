#pragma once

// How a decode's keys are split over workgroups: the equal splits of every decode and the balanced
// split of a paged one. Everything that becomes an address or a loop bound in the balanced kernels
// is formed here, in code that also compiles for the host, where
// tests/cpp/test_paged_split.cpp runs it with every index checked.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

namespace cuflash {
namespace dev {

// Where the keys come from. Contiguous: K, V [B, Hkv, kv_len, D]. Paged: K, V
// [num_pages, page_size, Hkv, D] with block_table [B, max_pages] naming the page of each
// page_size keys of a sequence and seq_lens [B] its length (clamped to [0, kv_len], kv_len =
// max_pages * page_size). A workgroup serves G query heads that share one key/value head:
// query head h reads key/value head h / (H / Hkv).
struct DecodeArgs {
    const int* block_table;
    const int* seq_lens;
    int H, Hkv;
    int kv_len;
    int page_size, max_pages;
    int page_shift;  // log2(page_size) when it is a power of two, else -1
    int chunk, nsplit;
    float c;  // scale * log2(e)
};

// Upper bound of the split count (the combine kernel's split weights stand in LDS).
constexpr int kMaxSplits = 1024;

// Minimum keys per split of the automatic split count (4 blocks of the matrix-core kernels):
// short sequences still spread over the chip (512-key chunks -> 128: plain decode, B = 1, 32
// heads, 1024 keys 13.6 -> 9.0 us; grouped-query, B = 1, 2 key/value heads, 32768 keys 26 ->
// 19 us; config 4's automatic 4 splits are unaffected).
constexpr int kMinChunk = 128;

// Sets a.nsplit and a.chunk: enough (unit, split) workgroups for `target_blocks`, with chunks of at
// least kMinChunk keys; an explicit request is clamped to [1, min(kMaxSplits, ceil(kv_len / 16))].
// whole_blocks: chunks of whole 32-key blocks.
inline void equal_splits(DecodeArgs& a, int requested, int units, int target_blocks,
                         bool whole_blocks) {
    const int max_useful = std::max(1, std::min(kMaxSplits, (a.kv_len + 15) / 16));
    if (requested > 0) {
        a.nsplit = std::min(requested, max_useful);
    } else {
        const int s = std::min((target_blocks + units - 1) / units,
                               std::max(1, a.kv_len / kMinChunk));
        a.nsplit = std::max(1, std::min(s, max_useful));
    }
    a.chunk = (a.kv_len + a.nsplit - 1) / a.nsplit;
    if (whole_blocks) {
        a.chunk = std::max(32, (a.chunk + 31) / 32 * 32);
        a.nsplit = std::max(1, (a.kv_len + a.chunk - 1) / a.chunk);
    }
}

// Balanced split of a paged decode (decode_mma_rows_kernel with automatic splits). The sequences'
// lengths are known on the device only, and equal splits of the cache's capacity leave the
// workgroups past a sequence's end without work: with 16 sequences of 512 to 8191 keys, half of
// them. Instead every (sequence, head group) unit is cut into as many segments as W blocks of 32
// keys go into it, rounded up, with the least W whose segments number at most max_segments: whole
// rounds of workgroups (one per CU). A few workgroups more cost a round: 9 sequences of up to 20045
// keys, 24 heads over 8, took 112 us on 270 segments, 71 on 256, where the 270 equal splits,
// many of them past a sequence's end, take 93. From 7/8 of the capacity on, the equal splits of the
// capacity (chunk) are as good, and the search for W is saved.
// Segment x leaves its partials in entry x, so the entries of a unit follow each other; its first
// workgroup notes them for the combine.
// Bound by the cache's reads where the workgroups have equal work: 32 query heads over 8, 16
// sequences of 8191 keys at most, fp16, head_dim 128, lengths spread evenly 74 -> 53 us (3.9 ->
// 5.4 TB/s), one long sequence and fifteen short ones 71 -> 18 us, all full 86.6 -> 86.7 us; 64
// sequences of 2000 keys, spread 77.3 -> 62.8 us, full 90.6 -> 92.5 us (the combine, one workgroup
// per query head and 32 columns, waits for one more load); 16 of 4096, spread 41.0 -> 32.1 us, full
// 48.1 -> 48.7 us.
struct BalancedArgs : DecodeArgs {
    int B;             // sequences
    int groups;        // units per sequence (head groups that one workgroup serves)
    int unit_heads;    // query heads per unit
    int max_segments;  // at least twice the units
    int entries;       // workgroups and partials: max_segments, or the equal splits of all units
    int min_blocks;    // least 32-key blocks per segment
    int full_blocks;   // blocks from which on the equal splits of the capacity are kept
    int2* units;       // [B * groups]: first entry and number of segments (units with keys only)
};

template <class Args>
constexpr bool is_balanced() {
    return std::is_same<Args, BalancedArgs>::value;
}

// The balanced split of a decode of `units` units whose equal splits are set, for about `wgs`
// workgroups, or false: caches with room for fewer than 16 blocks per workgroup, or for too many to
// count in 32 bits, keep the equal splits. Fills everything but `units` (the array).
inline bool balanced_plan(BalancedArgs& bal, const DecodeArgs& a, int B, long long units, int wgs) {
    const long long cap_blocks = (static_cast<long long>(a.kv_len) + 31) / 32;
    if (units * cap_blocks < 16LL * wgs || units * cap_blocks >= (1LL << 27)) return false;
    static_cast<DecodeArgs&>(bal) = a;
    bal.B = B;
    bal.groups = static_cast<int>(units / B);
    bal.unit_heads = a.H / bal.groups;
    // At least kMinChunk keys per segment, and no more per unit than the combine can hold.
    bal.min_blocks = static_cast<int>(
        std::max<long long>(kMinChunk / 32, (cap_blocks + kMaxSplits - 1) / kMaxSplits));
    bal.max_segments = static_cast<int>((2 * units + wgs - 1) / wgs * wgs);
    bal.entries = static_cast<int>(std::max<long long>(bal.max_segments, units * a.nsplit));
    bal.full_blocks = static_cast<int>(units * cap_blocks * 7 / 8);
    return true;
}

// Keys [kbeg, kend) of sequence b for its head group g: segment `part` of the unit's `parts`
// (parts 0: no such segment). A segment has at least one key.
struct PagedSegment {
    int b, g;
    int kbeg, kend;
    int part, parts;
};
__host__ __device__ __forceinline__ int paged_len(const DecodeArgs& a, int b) {
    const int n = a.seq_lens[b] > 0 ? a.seq_lens[b] : 0;
    return n < a.kv_len ? n : a.kv_len;
}

// Segment x (every wave computes it for itself). W: the 64 lanes of a wave, one value each in
// W::Int.
template <class W>
__host__ __device__ __forceinline__ PagedSegment paged_segment(const BalancedArgs& a, int x) {
    using Int = typename W::Int;
    auto blocks_of = [&](int b0) {
        return W::each([&](int lane) {
            return b0 + lane < a.B ? (paged_len(a, b0 + lane) + 31) >> 5 : 0;
        });
    };
    const Int first64 = blocks_of(0);
    // Sum of f(blocks) over the sequences.
    auto sum = [&](auto f) {
        Int v = W::map(first64, f);
        for (int b0 = 64; b0 < a.B; b0 += 64) v = W::add(v, W::map(blocks_of(b0), f));
        return W::lane(W::scan(v), 63);
    };
    const int total = sum([](int n) { return n; }) * a.groups;
    PagedSegment r{0, 0, 0, 0, 0, 0};
    if (total >= a.full_blocks) {
        const int unit = x / a.nsplit;
        if (unit >= a.B * a.groups) return r;
        r.part = x - unit * a.nsplit;
        r.b = unit / a.groups;
        r.g = unit - r.b * a.groups;
        const int len = paged_len(a, r.b);
        r.kbeg = r.part * a.chunk;
        r.kend = len - r.kbeg < a.chunk ? len : r.kbeg + a.chunk;
        r.parts = r.kend > r.kbeg ? (len + a.chunk - 1) / a.chunk : 0;
        return r;
    }
    // Segments of at most w blocks: at most total / w + units, so the least w that keeps them
    // within max_segments lies in [total / max_segments, total / (max_segments - units)].
    const int room = a.max_segments - a.B * a.groups;
    const int least = (total + a.max_segments - 1) / a.max_segments;
    int lo = least > a.min_blocks ? least : a.min_blocks;
    int hi = (total + room - 1) / room;
    if (hi < lo) hi = lo;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (sum([&](int n) { return (n + mid - 1) / mid; }) * a.groups <= a.max_segments)
            hi = mid;
        else
            lo = mid + 1;
    }
    int before = 0;  // segments of the sequences before b0
    for (int b0 = 0; b0 < a.B; b0 += 64) {
        const Int nb = b0 == 0 ? first64 : blocks_of(b0);
        const Int own = W::map(nb, [&](int n) { return (n + lo - 1) / lo; });
        const Int incl = W::scan(own);
        const int i = W::first(incl, [&](int n) { return before + n * a.groups > x; });
        if (i >= 0) {
            const int n = W::lane(nb, i);
            r.parts = W::lane(own, i);
            const int at = x - before - (W::lane(incl, i) - r.parts) * a.groups;
            // (parts - 1) each <= (parts - 1) lo < n: the last part has a block as well.
            const int each = (n + r.parts - 1) / r.parts;
            r.b = b0 + i;
            r.g = at / r.parts;
            r.part = at - r.g * r.parts;
            r.kbeg = r.part * each * 32;
            const int len = paged_len(a, r.b);
            r.kend = len - r.kbeg < each * 32 ? len : r.kbeg + each * 32;
            break;
        }
        before += W::lane(incl, 63) * a.groups;
    }
    return r;
}

// The partials of query head h of a sequence of `len` keys: `count` of them from `first` on,
// unit_heads apart. An empty sequence's unit was never written and is not used.
struct HeadPartials {
    int count;
    size_t first;
};
__host__ __device__ __forceinline__ HeadPartials head_partials(const BalancedArgs& a, int2 unit,
                                                               int len, int h) {
    return {len > 0 ? unit.y : 0, static_cast<size_t>(unit.x) * a.unit_heads + h % a.unit_heads};
}

}  // namespace dev
}  // namespace cuflash
