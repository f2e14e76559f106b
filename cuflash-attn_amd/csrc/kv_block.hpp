#pragma once

// The 32-key block of a wave that owns 32 query rows and its own K / V tiles, shared by the
// matrix-core decode kernels and the forward's fwd16_rows_kernel.

#include "common.hpp"
#include "softmax.hpp"

namespace cuflash {
namespace dev {

// One 32-key block for the 32 query rows of a wave (lane l32 = row; in the decode, query head):
// the scores S^T = K Q^T, the mask of keys at or past kend (this lane's; blocks that end at or
// before mask_from need none), the lazily rescaled softmax (m in log2 units, l this lane's share
// of the row sum), and O^T += V^T P^T. kt / vt are the block's K / V tiles; k_base (for even and
// odd k-steps) and v_off are this lane's operand offsets in layout Lay. before_pv() runs once the
// K tile has been read and before the V tile is: a kernel whose K and V tiles land separately
// waits for V and issues its next loads there.
template <typename T, int D, class Lay, class F>
__device__ __forceinline__ void kv_block32(const unsigned char* kt, const unsigned char* vt,
                                           const int (&k_base)[2], int v_off, int key0,
                                           int mask_from, int kend, int g2, float cs,
                                           const typename Elem<T>::frag (&qf)[D / 16],
                                           f32x16 (&o)[D / 32], float& m, float& l,
                                           F&& before_pv) {
    using frag = typename Elem<T>::frag;
    constexpr int KS = D / 16;
    constexpr int NDT = D / 32;
    constexpr int BN = 32;
    constexpr int kAhead = 3;
    f32x16 s = f32x16{};
    {
        frag fk[KS];
#pragma unroll
        for (int k = 0; k < kAhead && k < KS; ++k)
            fk[k] = as_frag<T>(ld16(kt + k_base[k & 1] + Lay::k_off(k)));
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            if (ks + kAhead < KS)
                fk[ks + kAhead] =
                    as_frag<T>(ld16(kt + k_base[(ks + kAhead) & 1] + Lay::k_off(ks + kAhead)));
            s = Elem<T>::mma(fk[ks], qf[ks], s);
        }
    }
    if (key0 + BN > mask_from) {
        const int lim = kend - key0 - 4 * g2;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = (8 * (r >> 2) + (r & 3) < lim) ? s[r] : -INFINITY;
    }
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = __builtin_elementwise_maximum(mx, s[r]);
    const float m_new = fmaxf(m, pair_max(mx) * cs);
    const bool grow = m_new > m + kLazyRescale;
    const float alpha = grow ? fast_exp2(m_new == -INFINITY ? 0.0f : m - m_new) : 1.0f;
    m = grow ? m_new : m;
    l *= alpha;
    if (__ballot(grow) != 0) {
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) o[dt] *= alpha;
    }
    const float m_use = (m == -INFINITY) ? 0.0f : m;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = fast_exp2(fmaf(s[r], cs, -m_use));
    float sum = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; r += 2) sum += s[r] + s[r + 1];
    l += sum;
    frag p[2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
        p[h] = pack_frag<T>(s[8 * h + 0], s[8 * h + 1], s[8 * h + 2], s[8 * h + 3], s[8 * h + 4],
                            s[8 * h + 5], s[8 * h + 6], s[8 * h + 7]);
    before_pv();
    constexpr int kMma = 2 * NDT;
    frag fv[kMma];
    auto v_frag = [&](int i) {
        const unsigned char* a0 =
            vt + v_off + (i / NDT) * Lay::kTrRows16 + Lay::dtile_off(i % NDT);
        return tr_frag_at<T>(a0, a0 + Lay::kTrHigh);
    };
#pragma unroll
    for (int k = 0; k < kAhead && k < kMma; ++k) fv[k] = v_frag(k);
#pragma unroll
    for (int i = 0; i < kMma; ++i) {
        if (i + kAhead < kMma) fv[i + kAhead] = v_frag(i + kAhead);
        o[i % NDT] = Elem<T>::mma(fv[i], p[i / NDT], o[i % NDT]);
    }
}

}  // namespace dev
}  // namespace cuflash
