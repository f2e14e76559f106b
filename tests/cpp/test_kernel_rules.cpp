// The rules that choose between two kernels (cuflash-attn_amd/csrc/kernel_rules.hpp), held to measured
// times: where one kernel was more than 15% faster, the rule takes that one. No GPU call is made.
//
// Times of one MI355X in microseconds of a whole call, fp16 / bf16 or fp32, on 256 CUs.
//
// With arguments (B, heads, key/value heads, queries, keys, head_dim, causal of each launch): prints
// the chunks of a 16-bit forward, 0 for the general kernels, and the keys of a chunk.

#include <cstdio>
#include <cstdlib>

#include "kernel_rules.hpp"

namespace {

using namespace cuflash::detail;
constexpr int kCus = 256;

struct Row {
    int D, B, H, Hkv, Nq, Nk;
    bool causal;
    double before, rows;  // the kernels of 128-row blocks, the kernel of 32-row items
};

// bwd_fused_kernel and bwd16_rows_kernel.
constexpr Row kBackward16[] = {
    {128, 1, 8, 8, 1147, 5009, false, 139.2, 249.3},
    {64, 3, 16, 16, 54, 371, true, 15.2, 26.9},
    {64, 10, 4, 4, 71, 579, true, 19.9, 32.5},
    {128, 14, 1, 1, 393, 2682, false, 82.6, 133.2},
    {96, 5, 8, 8, 74, 575, true, 22.5, 35.6},
    {128, 11, 1, 1, 794, 1944, true, 57.3, 90.3},
    {128, 5, 4, 4, 293, 1527, true, 53.2, 80.0},
    {64, 1, 32, 32, 97, 948, true, 28.3, 42.4},
    {96, 11, 1, 1, 166, 1019, true, 29.6, 22.2},
    {128, 3, 2, 2, 223, 411, true, 20.3, 13.2},
    {32, 1, 8, 8, 513, 5734, true, 97.0, 69.0},
    {64, 6, 1, 1, 47, 4603, true, 81.8, 37.2},
    {96, 4, 12, 2, 295, 295, true, 39.1, 28.1},
    {128, 3, 4, 4, 364, 364, true, 25.8, 15.1},
    {32, 1, 8, 1, 45, 868, true, 40.3, 14.3},
    {64, 3, 1, 1, 1787, 1787, false, 53.9, 28.5},
    {128, 1, 32, 4, 36, 536, false, 37.5, 14.3},
    {128, 1, 32, 8, 87, 89, false, 40.1, 14.4},
    {32, 6, 16, 16, 137, 567, true, 37.0, 49.0},
    {64, 5, 8, 8, 1689, 1689, true, 99.0, 149.7},
    {128, 10, 32, 32, 57, 443, true, 110.0, 219.0},
    {96, 1, 8, 1, 1376, 1376, true, 65.6, 125.4},
    {96, 10, 8, 1, 1083, 1083, true, 137.1, 299.8},
    {64, 15, 4, 4, 61, 428, false, 20.8, 36.4},
};

// dq_kernel and dkdv_kernel, bwd32_kernel.
constexpr Row kBackward32[] = {
    {64, 8, 32, 32, 57, 562, false, 171.7, 281.5},
    {64, 14, 32, 32, 98, 459, false, 291.9, 457.5},
    {96, 7, 32, 32, 68, 206, true, 126.2, 183.9},
    {96, 12, 16, 16, 40, 231, true, 111.6, 159.7},
    {128, 7, 32, 32, 97, 244, true, 190.5, 265.4},
    {64, 8, 32, 32, 77, 214, true, 81.8, 110.2},
    {32, 6, 32, 32, 173, 1775, false, 403.2, 543.2},
    {64, 9, 16, 16, 54, 1242, true, 259.5, 335.1},
    {96, 2, 8, 8, 685, 685, true, 169.0, 96.2},
    {64, 1, 16, 4, 73, 81, false, 68.8, 21.8},
    {64, 1, 16, 4, 464, 464, true, 309.4, 84.1},
    {128, 10, 2, 2, 112, 3011, true, 783.3, 249.4},
    {96, 5, 32, 32, 152, 152, true, 163.2, 101.1},
    {32, 1, 16, 16, 1946, 1946, true, 333.4, 160.7},
    {128, 1, 12, 2, 57, 281, true, 128.0, 38.7},
    {96, 8, 12, 2, 171, 854, true, 415.7, 305.8},
    {64, 1, 1, 1, 283, 415, false, 60.8, 22.1},
    {32, 8, 32, 4, 109, 119, true, 117.0, 30.2},
    {96, 14, 32, 32, 51, 138, true, 183.4, 246.5},
    {96, 3, 32, 32, 164, 1000, true, 367.3, 589.2},
    {128, 15, 16, 16, 50, 608, false, 348.7, 636.9},
    {64, 15, 32, 32, 244, 539, false, 655.0, 893.9},
    {96, 6, 16, 16, 171, 1036, false, 421.9, 639.2},
    {96, 3, 32, 32, 132, 1124, true, 408.5, 615.7},
};

// The general forwards, fwd16_rows_kernel.
constexpr Row kForward[] = {
    {256, 6, 32, 32, 57, 2032, true, 85.3, 120.5},
    {128, 7, 32, 32, 62, 458, true, 16.4, 22.4},
    {256, 3, 16, 16, 294, 294, true, 17.0, 19.9},
    {32, 4, 32, 32, 131, 4092, false, 52.1, 36.2},
    {256, 1, 8, 8, 620, 620, true, 27.7, 15.8},
    {32, 3, 32, 8, 2, 1263, false, 18.1, 10.1},
    {256, 3, 2, 2, 395, 395, true, 20.0, 12.4},
    {64, 1, 8, 8, 146, 3647, false, 48.9, 14.2},
    {256, 1, 8, 1, 1350, 1350, true, 51.1, 25.6},
    {96, 2, 8, 1, 913, 7566, true, 145.0, 71.8},
    {32, 4, 12, 2, 1, 6239, true, 76.8, 13.2},
    {96, 2, 12, 2, 1, 6305, false, 117.0, 13.1},
    {32, 4, 4, 4, 117, 3010, true, 39.0, 13.4},
    {256, 9, 32, 4, 177, 451, false, 70.6, 95.7},
    {96, 5, 12, 2, 762, 762, false, 24.2, 46.5},
    {32, 13, 16, 16, 927, 927, false, 57.2, 83.4},
    {96, 4, 32, 32, 267, 267, true, 11.4, 23.0},
    {64, 3, 32, 8, 930, 930, false, 34.9, 51.7},
    {256, 5, 32, 4, 84, 84, true, 11.3, 16.4},
};

template <class Rule>
int wrong(const char* name, const Row* rows, int n, Rule rule) {
    int bad = 0;
    for (int i = 0; i < n; ++i) {
        const Row& r = rows[i];
        const bool takes_rows = rule(r);
        if (takes_rows == (r.rows < r.before)) continue;
        std::printf("%s: head_dim %d, B=%d, %d heads over %d, %d queries, %d keys, causal %d: %g, "
                    "%g us, takes the %s\n", name, r.D, r.B, r.H, r.Hkv, r.Nq, r.Nk, r.causal,
                    r.before, r.rows, takes_rows ? "second" : "first");
        ++bad;
    }
    return bad;
}
#define COUNT(t) static_cast<int>(sizeof(t) / sizeof(t[0]))

bool backward16(const Row& r) {
    const BwdShape s{r.B * r.H, r.Nq, r.Nk, r.H / r.Hkv};
    switch (r.D) {
        case 32: return bwd16_rows_faster<32>(s, r.causal, kCus);
        case 64: return bwd16_rows_faster<64>(s, r.causal, kCus);
        case 96: return bwd16_rows_faster<96>(s, r.causal, kCus);
        case 128: return bwd16_rows_faster<128>(s, r.causal, kCus);
    }
    return false;
}
bool backward32(const Row& r) {
    const BwdShape s{r.B * r.H, r.Nq, r.Nk, r.H / r.Hkv};
    switch (r.D) {
        case 32: return bwd32_faster<32>(s, r.causal, kCus);
        case 64: return bwd32_faster<64>(s, r.causal, kCus);
        case 96: return bwd32_faster<96>(s, r.causal, kCus);
        case 128: return bwd32_faster<128>(s, r.causal, kCus);
    }
    return false;
}
int chunks(const Row& r) {
    const FwdShape s{r.B * r.H, r.Nq, r.Nk, r.H / r.Hkv};
    switch (r.D) {
        case 32: return forward_rows_chunks<32>(s, r.causal, kCus);
        case 64: return forward_rows_chunks<64>(s, r.causal, kCus);
        case 96: return forward_rows_chunks<96>(s, r.causal, kCus);
        case 128: return forward_rows_chunks<128>(s, r.causal, kCus);
        case 256: return forward_rows_chunks<256>(s, r.causal, kCus);
    }
    return 0;
}
bool forward(const Row& r) { return chunks(r) > 0; }

}  // namespace

int main(int argc, char** argv) {
    if (argc > 1) {
        for (int i = 1; i + 6 < argc; i += 7) {
            int v[7];
            for (int j = 0; j < 7; ++j) v[j] = std::atoi(argv[i + j]);
            const int n = chunks(Row{v[5], v[0], v[1], v[2], v[3], v[4], v[6] != 0, 0.0, 0.0});
            const KeyChunks kc = n > 1 ? key_chunks(v[4], n) : KeyChunks{v[4], n};
            std::printf("%d %d\n", kc.nsplit, kc.chunk);
        }
        return 0;
    }
    int bad = wrong("16-bit backward", kBackward16, COUNT(kBackward16), backward16);
    bad += wrong("fp32 backward", kBackward32, COUNT(kBackward32), backward32);
    bad += wrong("forward", kForward, COUNT(kForward), forward);
    return bad;
}
