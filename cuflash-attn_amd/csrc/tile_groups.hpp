#pragma once

// LDS tile layouts of the LDS-DMA kernels: the forward kernels' layouts, used by the backward's
// work items and by the matrix-core decode.

#include "common.hpp"

namespace cuflash {
namespace dev {

// LDS layout of a 16-bit tile with D-element rows: rows in groups filled by 1 KB load instructions
// (lane i writes the 16-byte slot i of its kilobyte). Every four consecutive lanes load 64
// contiguous bytes of one row: the memory path takes four lanes a clock only where they fall
// into one cache line. Measured on loads alone, L2-resident, four waves on each of 256 CUs: 129
// GB/s per CU, as for wholly linear lanes, against 37 with the rows of a group interleaved by 16
// bytes (consecutive lanes in four rows). The kernels, whose loads hide in part behind their
// MFMAs, gained 0.5 to 4% (bf16 training step, 16 heads over 4, N = 2001: 231.8 -> 222.3 us;
// head_dim 256, N = 2049: 246.1 -> 238.6 us; head_dim 128, N = 16384: 8454 -> 8381 us). The one-head
// decode kernel (decode_mma_kernel) gained 1 to 9% up to some 5000 keys and 1 to 14% on paged caches
// (32 heads over 8, B = 4, 3000 keys, head_dim 128: 15.2 -> 14.1 us); where it runs at the HBM rate it
// is level, or 1% slower (head_dim 128, B = 16, 12000 keys: 119.7 -> 120.9 us).
//   D = 128: 4-row groups, chunk c of row r at 16 (16 (c / 4) + 4 r + c % 4): the rows of a group
//            interleaved by 64 bytes. The padding of kBytes shifts successive groups by an odd
//            number of 16-byte slots modulo 64 bytes, so that 16 rows read at one chunk cover all
//            banks.
//   D = 64:  8-row groups, chunk c of row r at 16 (32 (c / 4) + 4 r + (c % 4 ^ 2 (r / 4))): as
//            above, and the rows r and r + 4 of a group, which share banks, swap chunk pairs.
//   D = 256: 4-row groups, two 1 KB column halves laid out as the D = 128 groups.
// Both serve conflict-free row reads (A operands of 32 rows x 16 k) and transpose reads
// (A operands whose k runs down 16 rows) with per-lane offsets and immediates.
template <int D>
struct TileGroups;
template <>
struct TileGroups<128> {
    static constexpr int kRows = 4;        // rows per group
    static constexpr int kBytes = 1104;    // bytes per group
    static constexpr int kHalves = 1;      // 1 KB load instructions per group
    static constexpr int kTrRows16 = 4 * kBytes;  // transpose reads: 16 rows further
    static constexpr int kTrHigh = 2 * kBytes;    // second read of a transpose operand (+8 rows)
    // Row reads: k-step ks.
    static constexpr int k_off(int ks) { return (ks >> 1) * 256 + (ks & 1) * 32; }
    static constexpr int dtile_off(int dt) { return dt * 256; }  // transpose reads: 32 columns
    __device__ static int ld_row(int lane) { return (lane >> 2) & 3; }
    __device__ static int ld_col(int lane) { return ((lane >> 4) * 4 + (lane & 3)) * 8; }
    // Row reads, k-step ks: this lane's 16 bytes (row lane % 32, chunk 2 ks + lane / 32) sit at
    // row_base(lane, ks & 1) + k_off(ks).
    __device__ static int row_base(int lane, int) {
        return ((lane & 31) >> 2) * kBytes + (lane & 3) * 64 + (lane >> 5) * 16;
    }
    // Transpose reads (see tr_frag_at): lane provides the 8-byte chunk of row 4 (lane / 32) +
    // (lane % 16) / 4, columns 16 ((lane / 16) % 2) + 4 (lane % 4).
    __device__ static int tr_off(int lane) {
        return (lane >> 5) * kBytes + ((lane & 15) >> 2) * 64 + ((lane >> 4) & 1) * 32 +
               (lane & 3) * 8;
    }
};
template <>
struct TileGroups<256> : TileGroups<128> {
    static constexpr int kBytes = 2 * 1024 + 80;
    static constexpr int kHalves = 2;
    static constexpr int kTrRows16 = 4 * kBytes;
    static constexpr int kTrHigh = 2 * kBytes;
    static constexpr int k_off(int ks) {
        return (ks >> 3) * 1024 + TileGroups<128>::k_off(ks & 7);
    }
    static constexpr int dtile_off(int dt) { return (dt >> 2) * 1024 + (dt & 3) * 256; }
    __device__ static int row_base(int lane, int) {
        return ((lane & 31) >> 2) * kBytes + (lane & 3) * 64 + (lane >> 5) * 16;
    }
    __device__ static int tr_off(int lane) {
        return (lane >> 5) * kBytes + ((lane & 15) >> 2) * 64 + ((lane >> 4) & 1) * 32 +
               (lane & 3) * 8;
    }
};
template <>
struct TileGroups<64> {
    static constexpr int kRows = 8;
    static constexpr int kBytes = 1168;
    static constexpr int kHalves = 1;
    static constexpr int kTrRows16 = 2 * kBytes;
    static constexpr int kTrHigh = kBytes;
    static constexpr int k_off(int ks) { return (ks >> 1) * 512; }
    static constexpr int dtile_off(int dt) { return dt * 512; }
    __device__ static int ld_row(int lane) { return (lane >> 2) & 7; }
    __device__ static int ld_col(int lane) {
        return ((lane >> 5) * 4 + ((lane & 3) ^ (2 * ((lane >> 4) & 1)))) * 8;
    }
    __device__ static int row_base(int lane, int odd) {
        return ((lane & 31) >> 3) * kBytes + (lane & 7) * 64 + (lane >> 5) * 16 +
               (odd ^ ((lane >> 2) & 1)) * 32;
    }
    __device__ static int tr_off(int lane) {
        const int g2 = lane >> 5;
        return (4 * g2 + ((lane & 15) >> 2)) * 64 + (((lane >> 4) & 1) ^ g2) * 32 +
               (lane & 3) * 8;
    }
};
// head_dim 32: the head_dim-64 layout with each 64-byte row in the first half of its 128-byte
// slot (operand reads touch chunks 0-3 only); lanes 32-63 of a load read the row's four
// chunks again into the unused slots 4-7.
template <>
struct TileGroups<32> : TileGroups<64> {
    __device__ static int ld_col(int lane) {
        return ((lane & 3) ^ (2 * ((lane >> 4) & 1))) * 8;
    }
};
// head_dim 96: the head_dim-128 layout with each 192-byte row in the first 12 chunks of its
// 256-byte slot (operand reads touch chunks 0-11 only); lanes 48-63 of a load read chunks 0-3
// again into the unused slots 12-15.
template <>
struct TileGroups<96> : TileGroups<128> {
    __device__ static int ld_col(int lane) { return (((lane >> 4) % 3) * 4 + (lane & 3)) * 8; }
};
// The tiles of fwd16_d128_kernel. With four waves at head_dim 96 the rows of a group stay interleaved
// by 16 bytes, chunk c of row r at 16 (4 c + r). Measured, 16 heads, this order -> TileGroups<96>:
// N=1400 29.0 -> 29.9 us (causal 28.9 -> 29.7), N=1700 34.8 -> 35.7; with eight waves
// TileGroups<96> is level or faster.
template <int D, int NW>
struct FwdTileGroups : TileGroups<D> {};
template <>
struct FwdTileGroups<96, 4> {
    static constexpr int kBytes = 1088;
    static constexpr int k_off(int ks) { return ks * 128; }
    static constexpr int dtile_off(int dt) { return dt * 256; }
    __device__ static int ld_row(int lane) { return lane & 3; }
    __device__ static int ld_col(int lane) { return ((lane >> 2) % 12) * 8; }
    __device__ static int row_base(int lane, int) {
        return ((lane & 31) >> 2) * kBytes + (lane >> 5) * 64 + (lane & 3) * 16;
    }
    __device__ static int tr_off(int lane) {
        const int kq = lane & 15;
        return (lane >> 5) * kBytes + (2 * ((lane >> 4) & 1) + ((kq & 3) >> 1)) * 64 +
               (kq >> 2) * 16 + (kq & 1) * 8;
    }
};
// The tiles of fwd16_d64_seq_kernel. Its loads hide behind the vector work of four waves per SIMD,
// so at head_dim 64 the rows of a group stay interleaved by 16 bytes, chunk c of row r at
// 16 (8 c + (r ^ 4 ((c / 2) % 2))), on the same 16 and 32 bank slots (fwd16_d64_kernel has the same
// order). Measured, no mask, this order -> TileGroups<64> on one MI355X: B=4, 16 heads, N=3000
// 162.5 -> 164.7 us; B=12, 16 heads over 4, 183 queries of 2264 keys 45.0 -> 45.7. At head_dim 32
// TileGroups is the faster one (causal, B=2, 32 heads, N=2500 49.5 -> 49.0).
// The row and transpose offsets take the kernel's l32 = lane % 32 and g2 = lane / 32 too: formed
// from the lane, the compiler's address code made the four-wave kernel 1.5% slower (no mask, 32
// heads, N=1024 17.1 -> 17.4 us; from l32 and g2 16.6).
template <int D>
struct SeqTileGroups : TileGroups<D> {
    __device__ static int row_base(int lane, int, int, int odd) {
        return TileGroups<D>::row_base(lane, odd);
    }
    __device__ static int tr_off(int lane, int) { return TileGroups<D>::tr_off(lane); }
};
template <>
struct SeqTileGroups<64> {
    static constexpr int kBytes = 1152;
    static constexpr int k_off(int ks) { return ks * 256; }
    static constexpr int dtile_off(int dt) { return dt * 512; }
    __device__ static int ld_row(int lane) { return (lane & 7) ^ (4 * ((lane >> 4) & 1)); }
    __device__ static int ld_col(int lane) { return ((lane >> 3) % 8) * 8; }
    __device__ static int row_base(int, int l32, int g2, int odd) {
        return (l32 >> 3) * kBytes + g2 * 128 + ((l32 & 7) ^ (4 * odd)) * 16;
    }
    __device__ static int tr_off(int lane, int g2) {
        const int kq = lane & 15;
        const int gl = (lane >> 4) & 1;
        return (2 * gl + ((kq & 3) >> 1)) * 128 + (g2 ^ gl) * 64 + (kq >> 2) * 16 + (kq & 1) * 8;
    }
};

}  // namespace dev
}  // namespace cuflash
