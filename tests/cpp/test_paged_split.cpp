// The balanced split of a paged decode (cuflash-attn_amd/csrc/paged_split.hpp) on the host: the
// code that the kernels run, over random launches and lengths, with every index that becomes an
// address checked against the array it goes to. No GPU call is made.
//
// Checked for each launch: every segment lies inside its sequence and has keys; every key of every
// unit belongs to exactly one segment; every partial is written to one of the `entries`;
// the segments of caches that are not nearly full fit whole rounds of workgroups;
// the entries of a unit follow each other from the one its first segment notes; the combine of
// every query head reads just these, at most kMaxSplits; pages stay below max_pages.
//
// Arguments: the number of launches, the seed.

#include <array>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "paged_split.hpp"

namespace {

using namespace cuflash::dev;

struct HostWave {
    using Int = std::array<int, 64>;
    template <class F>
    static Int each(F f) {
        Int v;
        for (int i = 0; i < 64; ++i) v[i] = f(i);
        return v;
    }
    template <class F>
    static Int map(const Int& v, F f) {
        return each([&](int i) { return f(v[i]); });
    }
    static Int add(const Int& a, const Int& b) {
        return each([&](int i) { return a[i] + b[i]; });
    }
    static Int scan(Int v) {
        for (int i = 1; i < 64; ++i) v[i] += v[i - 1];
        return v;
    }
    static int lane(const Int& v, int i) {
        if (i < 0 || i >= 64) std::abort();
        return v[i];
    }
    template <class F>
    static int first(const Int& v, F f) {
        for (int i = 0; i < 64; ++i)
            if (f(v[i])) return i;
        return -1;
    }
};

int g_case = 0;
#define CHECK(cond)                                                            \
    do {                                                                       \
        if (!(cond)) {                                                         \
            std::printf("launch %d, line %d: %s\n", g_case, __LINE__, #cond); \
            std::exit(1);                                                      \
        }                                                                      \
    } while (0)

int spread(std::mt19937& rng, int lo, int hi) {  // over the logarithm
    std::uniform_real_distribution<double> u(std::log(double(lo)), std::log(double(hi) + 1.0));
    return std::min(hi, std::max(lo, int(std::exp(u(rng)))));
}

// One launch; returns 0 if it keeps the equal splits, 1 balanced, 2 balanced with the capacity's
// equal splits (nearly full).
int launch(std::mt19937& rng) {
    auto pick = [&](int n) { return int(rng() % unsigned(n)); };
    const int row_heads = std::array<int, 3>{4, 8, 16}[pick(3)];  // 512 / head_dim
    const int wgs = std::array<int, 4>{256, 256, 304, 64}[pick(4)];
    DecodeArgs a{};
    a.Hkv = row_heads * (1 + pick(4));
    a.H = a.Hkv * (2 + pick(31));
    a.page_size = std::array<int, 6>{1, 6, 16, 32, 64, 256}[pick(6)];
    const int B = spread(rng, 2, 200);
    a.max_pages = spread(rng, 1, std::max(1, 40000 / a.page_size));
    a.kv_len = a.page_size * a.max_pages;
    const long long units = static_cast<long long>(B) * (a.Hkv / row_heads);
    equal_splits(a, 0, int(units), wgs, true);
    CHECK(a.nsplit >= 1 && a.nsplit <= kMaxSplits && a.chunk % 32 == 0 && a.chunk > 0);
    CHECK(static_cast<long long>(a.chunk) * (a.nsplit - 1) < a.kv_len);
    CHECK(static_cast<long long>(a.chunk) * a.nsplit >= a.kv_len);

    // Lengths: all full, all empty, around 7/8 of the capacity, one long among short ones, any;
    // some below 0 and past the capacity, which are clamped.
    std::vector<int> lens(B);
    const int kind = pick(6);
    for (int b = 0; b < B; ++b) {
        switch (kind) {
            case 0: lens[b] = a.kv_len; break;
            case 1: lens[b] = 0; break;
            case 2: lens[b] = int(a.kv_len * (0.86 + 0.03 * (pick(1000) / 1000.0))); break;
            case 3: lens[b] = pick(B) == 0 ? a.kv_len : pick(200); break;
            case 4: lens[b] = pick(4) == 0 ? 0 : spread(rng, 1, a.kv_len); break;
            default: lens[b] = pick(a.kv_len + 1);
        }
        if (pick(20) == 0) lens[b] = -1 - pick(9);
        if (pick(20) == 0) lens[b] = a.kv_len + pick(1000);
        if (pick(20) == 0) lens[b] = 0;
    }
    a.seq_lens = lens.data();
    BalancedArgs bal{};
    if (!balanced_plan(bal, a, B, units, wgs)) return 0;
    CHECK(bal.groups * static_cast<long long>(B) == units);
    CHECK(bal.unit_heads * bal.groups == a.H);
    CHECK(bal.max_segments >= 2 * units && bal.max_segments % wgs == 0);
    CHECK(bal.entries >= bal.max_segments && bal.entries >= units * a.nsplit);

    // The split kernel: one workgroup per entry.
    const int2 unwritten = make_int2(0x7ffffff0, 0x7ffffff0);
    std::vector<int2> table(units, unwritten);
    std::vector<int> owner(bal.entries, -1);  // the unit that wrote entry x
    std::vector<std::vector<std::array<int, 2>>> keys(units);
    long long total = 0;
    for (int b = 0; b < B; ++b) total += (paged_len(a, b) + 31) / 32;
    const bool full = total * bal.groups >= bal.full_blocks;
    for (int x = 0; x < bal.entries; ++x) {
        const PagedSegment s = paged_segment<HostWave>(bal, x);
        if (s.parts == 0) continue;
        CHECK(s.b >= 0 && s.b < B && s.g >= 0 && s.g < bal.groups);
        CHECK(s.part >= 0 && s.part < s.parts && s.parts <= kMaxSplits);
        CHECK(s.kbeg >= 0 && s.kbeg % 32 == 0 && s.kbeg < s.kend && s.kend <= paged_len(a, s.b));
        CHECK((s.kend - 1) / a.page_size < a.max_pages);
        const int unit = s.b * bal.groups + s.g;
        owner[x] = unit;
        if (s.part == 0) {
            CHECK(table[unit].x == unwritten.x);  // noted once
            table[unit] = make_int2(x, s.parts);
        }
        CHECK(table[unit].x != unwritten.x);  // the entries follow the first one
        CHECK(x == table[unit].x + s.part && s.parts == table[unit].y);
        keys[unit].push_back({s.kbeg, s.kend});
    }
    // Below 7/8 of the capacity: at most max_segments, whole rounds of workgroups.
    if (!full) {
        size_t segments = 0;
        for (const auto& k : keys) segments += k.size();
        CHECK(segments <= static_cast<size_t>(bal.max_segments));
    }
    // Every key of a unit once, in order.
    for (int unit = 0; unit < units; ++unit) {
        int at = 0;
        for (const auto& k : keys[unit]) {
            CHECK(k[0] == at);
            at = k[1];
        }
        CHECK(at == paged_len(a, unit / bal.groups));
    }
    // The combine: head bh reads `count` entries from `first` on, unit_heads apart.
    const size_t slots = static_cast<size_t>(bal.entries) * bal.unit_heads;
    for (int b = 0; b < B; ++b) {
        for (int h = 0; h < a.H; ++h) {
            const int unit = b * bal.groups + h / bal.unit_heads;
            const HeadPartials hp = head_partials(bal, table[unit], paged_len(a, b), h);
            CHECK(hp.count == static_cast<int>(keys[unit].size()) && hp.count <= kMaxSplits);
            for (int i = 0; i < hp.count; ++i) {
                const size_t slot = hp.first + static_cast<size_t>(i) * bal.unit_heads;
                CHECK(slot < slots);
                CHECK(owner[slot / bal.unit_heads] == unit);
                CHECK(static_cast<int>(slot % bal.unit_heads) == h % bal.unit_heads);
            }
        }
    }
    return full ? 2 : 1;
}

}  // namespace

int main(int argc, char** argv) {
    const int n = argc > 1 ? std::atoi(argv[1]) : 1000;
    std::mt19937 rng(argc > 2 ? std::atoi(argv[2]) : 1);
    int seen[3] = {0, 0, 0};
    for (g_case = 0; g_case < n; ++g_case) ++seen[launch(rng)];
    std::printf("equal %d, balanced %d, nearly full %d\n", seen[0], seen[1], seen[2]);
    return seen[0] > n / 20 && seen[1] > n / 20 && seen[2] > n / 20 ? 0 : 1;
}
