// fa_mask_rows.h — the pre-pass over a mask tensor: the live interval of each
// mask row (device code shared by the launches that run it).
#pragma once

#include "fa_common.h"

namespace vxfa {

// min / max / sum over the 16 lanes of a DPP row (every lane of the row gets
// the result; row rotates are VALU operand modifiers, no LDS traffic)
__device__ __forceinline__ int row16_min_i(int x) {
    x = min(x, __builtin_amdgcn_update_dpp(0, x, 0x128, 0xF, 0xF, false));
    x = min(x, __builtin_amdgcn_update_dpp(0, x, 0x124, 0xF, 0xF, false));
    x = min(x, __builtin_amdgcn_update_dpp(0, x, 0x122, 0xF, 0xF, false));
    return min(x, __builtin_amdgcn_update_dpp(0, x, 0x121, 0xF, 0xF, false));
}
__device__ __forceinline__ int row16_max_i(int x) {
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x128, 0xF, 0xF, false));
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x124, 0xF, 0xF, false));
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x122, 0xF, 0xF, false));
    return max(x, __builtin_amdgcn_update_dpp(0, x, 0x121, 0xF, 0xF, false));
}
__device__ __forceinline__ int row16_sum_i(int x) {
    x += __builtin_amdgcn_update_dpp(0, x, 0x128, 0xF, 0xF, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x124, 0xF, 0xF, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x122, 0xF, 0xF, false);
    return x + __builtin_amdgcn_update_dpp(0, x, 0x121, 0xF, 0xF, false);
}

// min / max / sum over the 64 lanes: DPP row reductions, then the four rows'
// results read into scalar registers (uniform result, no LDS traffic)
__device__ __forceinline__ int wave_min_dpp(int x) {
    x = row16_min_i(x);
    return min(min(__builtin_amdgcn_readlane(x, 0), __builtin_amdgcn_readlane(x, 16)),
               min(__builtin_amdgcn_readlane(x, 32), __builtin_amdgcn_readlane(x, 48)));
}
__device__ __forceinline__ int wave_max_dpp(int x) {
    x = row16_max_i(x);
    return max(max(__builtin_amdgcn_readlane(x, 0), __builtin_amdgcn_readlane(x, 16)),
               max(__builtin_amdgcn_readlane(x, 32), __builtin_amdgcn_readlane(x, 48)));
}
__device__ __forceinline__ int wave_sum_dpp(int x) {
    x = row16_sum_i(x);
    return (__builtin_amdgcn_readlane(x, 0) + __builtin_amdgcn_readlane(x, 16)) +
           (__builtin_amdgcn_readlane(x, 32) + __builtin_amdgcn_readlane(x, 48));
}

// The pre-pass of a mask tensor: one wavefront per mask row
// w = (batch bm_i, plane p, row q), w = (bm_i * hm + p) * nq + q, four rows
// per 256-thread block (mask_rows_kernel, and the first blocks of the launch
// that also stages F32 K/V, prep_kernel, or of each row of the launch that
// appends new rows, kv_append_kernel); writes out[w] = {lo, hi} when the row's
// entries are 0 (+0 or -0) on [lo, hi] and -inf elsewhere, {n, -1}
// when every entry is -inf, {-2, -2} otherwise. The row is read as the
// 16-byte-aligned chunks that cover it (any row alignment; a chunk holds at
// least one byte of the row, so it lies in the same granule as mask data):
// in rounds of 192 chunks, lane s loading chunks c0 + 64 u + s (u < 3, all
// in flight; a chunk past the row's last reloads the last and counts
// nothing). Branch-free per chunk: bit e of `live` is set when entry e lies
// in the row and is not -inf, of `nz` when it is also non-zero; one pass
// gives the first and last live column, their count and whether one is
// non-zero (the row is an interval iff the count is hi - lo + 1), reduced
// over the wavefront. A whole wavefront per row, not a 16-lane DPP row: the
// pre-pass is bound by its VALU work per lane, which a single wavefront per
// SIMD issues at about half the SIMD's rate (1500 realtime-encoder rows:
// 4.8 us with 16 lanes and 12 chunks per lane).
constexpr int kMaskRowChunks = 3;    // chunks per lane per round
struct MaskRowArgs {
    const uint16_t* mask;
    int64_t nb1, nb2, nb3;
    int n, nq, hm, nrows;
    int2* out;
};
// What thread s of NT sees of mask row w: first and last live column, their
// count, and whether one is not zero.
struct MaskRowPart {
    int lo, hi, cnt;
    uint32_t nz;
};
template <int NT>
__device__ __forceinline__ MaskRowPart mask_row_part(const MaskRowArgs& m, int w, int s) {
    constexpr int kMaskRowRound = NT * kMaskRowChunks;
    const int q = w % m.nq, pb = w / m.nq, p = pb % m.hm, bb = pb / m.hm;
    const char* rowp = (const char*)m.mask + (int64_t)q * m.nb1 + (int64_t)p * m.nb2 + (int64_t)bb * m.nb3;
    const int mis = (int)(reinterpret_cast<uintptr_t>(rowp) & 15);   // even: the mask is 2-byte aligned
    const char* base = rowp - mis;
    const int n = m.n;
    const int nch = (mis + 2 * n + 15) / 16;
    const int nchmax = (14 + 2 * n + 15) / 16;                         // the same loop for every row
    int lo = 0x7fffffff, hi = -1, cnt = 0;
    uint32_t nzall = 0;
    for (int c0 = 0; c0 < nchmax; c0 += kMaskRowRound) {
        u32x4 wv[kMaskRowChunks];
#pragma unroll
        for (int u = 0; u < kMaskRowChunks; ++u) wv[u] = *(const u32x4*)(base + 16 * min(c0 + NT * u + s, nch - 1));
#pragma unroll
        for (int u = 0; u < kMaskRowChunks; ++u) {
            const int col0 = 8 * (c0 + NT * u + s) - mis / 2;      // column of the chunk's first entry
            const int elo = max(-col0, 0), ehi = min(n - col0, 8);  // entries [elo, ehi) lie in the row
            const uint32_t valid = ehi > elo ? ((1u << ehi) - 1u) & ~((1u << elo) - 1u) : 0u;
            uint32_t live = 0, nz = 0;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t v = (wv[u][e >> 1] >> (16 * (e & 1))) & 0xFFFFu;
                const uint32_t l = v != kF16NegInf ? 1u : 0u;
                live |= l << e;
                nz |= (l & ((v & 0x7FFFu) != 0 ? 1u : 0u)) << e;
            }
            live &= valid;
            nzall |= nz & valid;
            const int first = col0 + (int)__builtin_ctz(live | 0x100u);
            const int last = col0 + 31 - (int)__builtin_clz(live | 1u);
            lo = live ? min(lo, first) : lo;
            hi = live ? max(hi, last) : hi;
            cnt += __builtin_popcount(live);
        }
    }
    return MaskRowPart{lo, hi, cnt, nzall};
}
// Mask row w (w < nrows, uniform over the wavefront) by lane s (0..63);
// every lane calls it (waves past the last row pass w = nrows - 1 and store
// nothing).
__device__ __forceinline__ void mask_row_interval(const MaskRowArgs& m, int w, int s, bool store) {
    const MaskRowPart p = mask_row_part<64>(m, w, s);
    const int lo = wave_min_dpp(p.lo);
    const int hi = wave_max_dpp(p.hi);
    const int cnt = wave_sum_dpp(p.cnt);
    const int nonzero = wave_max_dpp(p.nz != 0 ? 1 : 0);
    if (s == 0 && store)
        m.out[w] = hi < lo ? int2{m.n, -1} : ((nonzero || cnt != hi - lo + 1) ? int2{-2, -2} : int2{lo, hi});
}

// mask rows [4 bx, 4 bx + 4), one per wavefront
__device__ __forceinline__ void mask_rows_block(const MaskRowArgs& m, uint32_t bx, int tid) {
    const int w = (int)bx * 4 + __builtin_amdgcn_readfirstlane(tid >> 6);
    mask_row_interval(m, min(w, m.nrows - 1), tid & 63, w < m.nrows);
}

}  // namespace vxfa
