#pragma once

// Which of two kernels a launch takes: models of both kernels' times, in microseconds, from the
// shape and the number of CUs. Host code without HIP calls; tests/cpp/test_kernel_rules.cpp holds the
// rules to times measured on both sides of their lines.

#include <algorithm>
#include <cmath>

namespace cuflash {
namespace detail {

// Query/key extents of one launch.
struct FwdShape {
    int BH;     // query heads over the batch
    int Nq;     // query rows per head
    int Nk;     // key rows per key/value head
    int group;  // query heads per key/value head
};

// Query/key extents of one launch.
struct BwdShape {
    int BH;     // query heads over the batch
    int Nq;     // query rows per head
    int Nk;     // key rows per key/value head
    int group;  // query heads per key/value head
};

// Waves per workgroup of fwd16_rows_kernel and bwd16_rows_kernel, and the device memory that the
// fused backward's dK / dV shares of grouped heads may take.
template <int D>
constexpr int fwd_rows_waves() {
    return D == 256 ? 4 : 8;  // LDS: 134 KB at head_dim 256, 140 KB at 128 and 96, 75 KB below
}
template <int D>
constexpr int bwd16_rows_waves() {
    return D <= 64 ? 8 : 4;  // two waves per SIMD, or one (registers)
}
constexpr long long kMaxShareBytes = 2LL << 30;

// Chunks over which fwd16_rows_kernel cuts the keys of this launch, or 0 where the general kernels
// are faster. The times are modelled from measurements (causal and not, 4 to 32 heads, 64 to 16384
// keys; event times of one MI355X):
//  * fwd16_rows_kernel: a workgroup walks its longest tile in rounds of one block per wave, tb
//    each, and t0 for its start, merge and store; as many workgroups as the slots run at once.
//    Several chunks add the merge kernel and the partials, written and read at about 4 TB/s. In one
//    chunk every tile reads its head's keys by itself: where they do not stay in the L2s, at about
//    6 TB/s.
//  * the general kernels: g per 64-key block of the longest row while their 128-row workgroups all
//    run at once (more with two workgroups per CU), else 1.5 g per round of them and block of the
//    average row. They do not pack heads: a few tokens of many heads fill their rows badly.
// bf16/fp16, causal, B = 1, before -> after: 8 heads, head_dim 128, N = 129 8.4 -> 6.3, 1024 23.9 ->
// 11.9, 4096 82 -> 64; head_dim 64, N = 256 6.3 -> 5.0, 1024 16.9 -> 8.5, 4096 55.6 -> 34.5;
// head_dim 256, N = 1024 40.1 -> 22.0; 32 heads over 8 against 8253 keys, head_dim 128: 61 queries
// 160 -> 22 (4 chunks), one query 156 -> 11.6 (11 chunks); one query of 64 x 32 heads over 8,
// 1000 keys 206 -> 41. The other side of the line: 32 heads, head_dim 128, N = 1024 25.7 general,
// 32.7 here; head_dim 64, N = 1536 25.8 and 26.9; 224 heads, 62 of 458 keys, head_dim 128 16.4, 22.4.
// Over 2500 random launches of 1 to 8192 keys the choice is on average 0.9% slower than the better
// kernel, and no launch is both 3% and 0.8 us slower than the general kernel.
template <int D>
int forward_rows_chunks(const FwdShape& sh, bool causal, int compute_units) {
    constexpr double tb = D == 32 ? 1.2 : D == 64 ? 1.6 : D == 96 ? 1.1 : D == 128 ? 1.36 : 1.95;
    constexpr double t0 = D <= 64 ? 3.0 : 4.2;
    constexpr double g = D == 32 ? 0.75 : D == 64 ? 0.85 : D == 96 ? 1.15 : D == 128 ? 1.27 : 2.25;
    constexpr int kWaves = fwd_rows_waves<D>();
    constexpr double kL2Bytes = 32e6;
    const double cus = compute_units;
    const double slots = D <= 64 ? 2 * cus : cus;
    const double rows = static_cast<double>(sh.BH) * sh.Nq;
    const double units = static_cast<double>(sh.BH) * ((sh.Nq + 127LL) / 128);
    const double tiles = static_cast<double>(sh.BH / sh.group) *
                         ((static_cast<long long>(sh.group) * sh.Nq + 31) / 32);
    const double longest = (sh.Nk + 31LL) / 32 / static_cast<double>(kWaves);
    const double part = causal ? (2.0 * sh.Nk - sh.Nq) / (2.0 * sh.Nk) : 1.0;
    const double average = longest * part;
    double best = 0.0;
    int chunks = 0;
    for (int n = 1; n == 1 || (n <= 32 && 2 * n <= longest); ++n) {
        const double rounds = std::ceil(tiles * n / slots);
        // Blocks are taken in whole rounds of the waves: half a round more than the average.
        const double whole = std::ceil(longest / n);
        const double walk =
            rounds > 1 ? std::min(whole, average / n + (kWaves - 1) / (2.0 * kWaves)) : whole;
        double t = rounds * (walk * tb + t0) - 2.0;
        const double kv_bytes = 4.0 * D * sh.Nk;
        if (n == 1 && tiles > units && sh.BH / sh.group * kv_bytes > kL2Bytes)
            t = std::max(t, 1.0 + tiles * kv_bytes * part / 6e6);
        if (n > 1) t += 4.0 + 2.0 * n * rows * D * sizeof(float) / 4e6;
        if (chunks == 0 || t < best) {
            best = t;
            chunks = n;
        }
    }
    const double blocks = static_cast<double>((sh.Nk + 63LL) / 64);
    double general;
    if (units > 2 * cus)
        general = 1.5 * g * blocks * part * units / (2 * cus);
    else if (D <= 64)
        general = g * blocks * (1.0 + 0.3 * std::min(1.0, std::max(0.0, units / cus - 1.0)));
    else
        general = g * blocks + 4.0 * units / cus;
    return 1.1 * best < general ? chunks : 0;
}

// The keys of each chunk (whole 32-key blocks) and the number of chunks that have any.
struct KeyChunks {
    int chunk, nsplit;
};
inline KeyChunks key_chunks(int Nk, int chunks) {
    const int chunk = ((Nk + chunks - 1) / chunks + 31) / 32 * 32;
    return {chunk, (Nk + chunk - 1) / chunk};
}

// A backward's items: dq and dkdv items, the average and the longest item of each kind. For the
// kernels of 32-row items in rounds of one 32 x 32 block per wave, for those of 128-row items in
// 32-row blocks of the other side.
struct BwdItems {
    double nq, nk;  // items
    double aq, ak;  // average
    double lq, lk;  // longest
};
inline BwdItems row_items(const BwdShape& sh, bool causal, int waves) {
    const double nqt = (sh.Nq + 31LL) / 32, nkt = (sh.Nk + 31LL) / 32;
    BwdItems it;
    it.nq = sh.BH * nqt;
    it.nk = sh.BH / sh.group * nkt;
    it.lq = std::ceil(nkt / waves);
    it.lk = std::ceil(sh.group * nqt / waves);
    it.aq = it.lq;
    it.ak = it.lk;
    if (causal && nqt > 1) {
        const double half = (waves - 1) / (2.0 * waves);  // what rounding up adds on average
        const double q = nkt - (nqt - 1) / 2.0, k = nqt * (1.0 - (nqt - 1) / (2.0 * nkt));
        it.aq = std::min(std::max(1.0, q / waves + half), it.lq);
        it.ak = std::min(std::max(1.0, sh.group * k / waves + half), it.lk);
    }
    return it;
}
// heads: the query heads that one dkdv item takes (the group, or 1 where they leave shares).
inline BwdItems block_items(const BwdShape& sh, bool causal, int heads) {
    const double nqt = (sh.Nq + 31LL) / 32, nkt = (sh.Nk + 31LL) / 32;
    BwdItems it;
    it.nq = static_cast<double>(sh.BH) * ((sh.Nq + 127LL) / 128);
    it.nk = static_cast<double>(sh.BH / heads) * ((sh.Nk + 127LL) / 128);
    it.lq = nkt;
    it.lk = heads * nqt;
    it.aq = it.lq;
    it.ak = it.lk;
    if (causal) {
        if (nqt > 4) it.aq = nkt - (nqt - 4) / 2.0;
        const double k = nqt * (1.0 - (nqt - 1) / (2.0 * nkt));
        it.ak = heads * std::min(nqt, std::max(k, 1.0) + (nqt > 1 ? 1.5 : 0.0));
    }
    return it;
}

// A kernel's costs: what an item of each kind pays besides its blocks (start, merge, store) and per
// round or block, the share by which blocks cost more once the CUs are full, and the part of the
// longest item by which a launch of many items ends late.
struct BwdCost {
    double iq, ik;
    double cq, ck;
    double full, tail;
};
// Time of `it` where `per_cu` workgroups share a CU: the longest item, or all of them spread over
// the CUs and the tail.
inline double item_time(const BwdItems& it, const BwdCost& c, double cus, double per_cu) {
    const double n = it.nq + it.nk;
    const double per = std::min(per_cu, std::max(1.0, n / cus));
    const double more = 1.0 + c.full * (per_cu > 1 ? per - 1.0 : std::min(1.0, n / cus));
    const double work = (it.nq * (c.iq + it.aq * c.cq * more) + it.nk * (c.ik + it.ak * c.ck * more)) /
                        (cus * per);
    const double longest = std::max(c.iq + it.lq * c.cq, c.ik + it.lk * c.ck);
    return std::max(longest, work + c.tail * longest);
}

// Whether bwd32_kernel (32-row items whose blocks are spread over four waves) beats the kernels of
// 128-row items for an fp32 backward. Those run dq and dkdv one after the other, each in its longest
// item or its total and a tail under a causal mask, in whole rounds of workgroups without; or
// both at once where they fit the CUs. The costs are fitted to 1500 random launches (32 to 8192
// keys), in which the choice is on average 1.2% slower than the better kernel (bwd32_kernel alone
// wins by 2x on average) and 8 take a kernel that is more than 2% slower.
// Measured (128-row kernels, bwd32_kernel, us, whole backward). Taken: causal B=2 H=8 N=1024
// head_dim 64 169, 101, head_dim 32 104, 52; B=2 H=16 N=4096 head_dim 64 2930, 2330; B=1 H=8
// N=4096 head_dim 128 2037, 1343; 32 heads over 8, N=512, head_dim 128 575, 173. Not taken: causal
// B=2 H=16 N=4096 head_dim 128 4726, 5314; 32 heads over 8, N=2000, head_dim 128 3240, 4030; and
// where the short side has few blocks for the waves: 448 heads, 98 of 459 keys, head_dim 64 292, 458.
template <int D>
bool bwd32_faster(const BwdShape& sh, bool causal, int compute_units) {
    constexpr double kPer = D <= 64 ? 2.0 : 1.0;  // workgroups per CU, of either kind
    constexpr BwdCost kRows = D == 32   ? BwdCost{1.61, 1.37, 2.05, 2.94, 0.95, 0.35}
                              : D == 64 ? BwdCost{2.15, 2.67, 3.98, 5.12, 1.34, 0.30}
                              : D == 96 ? BwdCost{3.03, 3.81, 5.87, 7.55, 0.58, 0.09}
                                        : BwdCost{6.70, 4.23, 7.38, 9.85, 0.54, 0.19};
    constexpr BwdCost kBlocks = D == 32   ? BwdCost{2.49, 2.49, 2.29, 3.09, 0.72, 0.18}
                                : D == 64 ? BwdCost{4.45, 4.45, 3.89, 5.16, 0.80, 0.35}
                                : D == 96 ? BwdCost{8.45, 8.45, 5.36, 7.02, 0.80, 0.42}
                                          : BwdCost{10.8, 10.8, 6.86, 9.21, 0.80, 0.48};
    const double cus = compute_units;
    const BwdItems it = block_items(sh, causal, sh.group);
    auto grid = [&](double n, double average, double longest, double c) {
        const double per = std::min(kPer, std::max(1.0, n / cus));
        c *= 1.0 + (kPer > 1 ? kBlocks.full * (per - 1.0) : 0.0);
        if (!causal) return std::ceil(n / (cus * per)) * (kBlocks.iq + average * c);
        longest = kBlocks.iq + longest * c;
        return std::max(longest, n * (kBlocks.iq + average * c) / (cus * per) +
                                     kBlocks.tail * longest);
    };
    const double blocks = it.nq + it.nk <= cus
                              ? kBlocks.iq + std::max(it.lq * kBlocks.cq, it.lk * kBlocks.ck)
                              : grid(it.nq, it.aq, it.lq, kBlocks.cq) +
                                    grid(it.nk, it.ak, it.lk, kBlocks.ck);
    return 1.15 * item_time(row_items(sh, causal, 4), kRows, cus, kPer) < blocks;
}

// Whether bwd16_rows_kernel beats bwd_fused_kernel. The first spreads better, the second moves a
// fourth of the tile bytes per product; grouped heads leave it shares that another launch sums. The
// costs are fitted to 2200 random launches (32 to 8192 keys), in which the choice is on average
// 3% slower than the better kernel (bwd_fused_kernel alone: 37%) and 20 take a kernel that is
// more than 2% slower. Measured (bwd_fused_kernel, bwd16_rows_kernel, us; more at the kernel): taken:
// 8 heads, N=1024, head_dim 64 28.5, 14.4. Not taken: causal 16 heads, N=2048, head_dim 64 61, 69
// and 128 92, 140; 32 heads, N=1024, head_dim 64 38, 52; 8 heads over 1, N=2000, head_dim 128 98,
// 203; no mask, 22 heads, 278 of 943 keys, head_dim 96 29, 53 (and causal 36 heads, 43 of 349
// keys, head_dim 128 19, 26): the short side has too few blocks for the waves.
// Beyond eight items per CU the fused kernel is kept, although with grouped heads and few query rows
// this one measures faster there as well (B=10, 32 heads over 4, 65 of 2197 keys, head_dim 32 524, 144).
template <int D>
bool bwd16_rows_faster(const BwdShape& sh, bool causal, int compute_units) {
    constexpr BwdCost kRows = D == 32   ? BwdCost{3.25, 3.74, 0.80, 1.03, 0.14, 0.47}
                              : D == 64 ? BwdCost{4.97, 6.71, 0.93, 1.19, 0.19, 0.36}
                              : D == 96 ? BwdCost{4.77, 6.48, 1.13, 1.46, 0.31, 0.24}
                                        : BwdCost{5.26, 7.65, 1.35, 1.63, 0.36, 0.19};
    constexpr BwdCost kFused = D == 32   ? BwdCost{10.6, 10.6, 0.44, 0.56, 0.03, 0.62}
                               : D == 64 ? BwdCost{10.7, 10.7, 0.48, 0.68, 0.73, 0.41}
                               : D == 96 ? BwdCost{10.8, 10.8, 0.61, 0.93, 0.81, 0.38}
                                         : BwdCost{12.8, 12.8, 0.65, 1.05, 0.93, 0.54};
    // The sum of the shares: its launch, and the shares at so many bytes per microsecond.
    constexpr double kSum = D == 32 ? 0.2 : D == 64 ? 6.2 : D == 96 ? 8.2 : 5.4;
    constexpr double kRate = (D == 32 ? 0.76 : D == 64 ? 1.90 : D == 96 ? 2.28 : 2.49) * 1e6;
    const double cus = compute_units;
    const double share_bytes = 2.0 * sh.BH * sh.Nk * D * sizeof(float);
    const bool shares = sh.group > 1 && share_bytes <= kMaxShareBytes;
    double fused = item_time(block_items(sh, causal, shares ? 1 : sh.group), kFused, cus, 2.0);
    if (shares) fused += kSum + share_bytes / kRate;
    const BwdItems rows = row_items(sh, causal, bwd16_rows_waves<D>());
    return rows.nq + rows.nk <= 8.0 * cus && 1.2 * item_time(rows, kRows, cus, 1.0) < fused;
}

}  // namespace detail
}  // namespace cuflash
