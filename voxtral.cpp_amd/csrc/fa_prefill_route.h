// fa_prefill_route.h — host code: which kernel a prefill call takes beyond the
// short masked one (fa_prefill_pair.hip), and the KV pieces of the grouped
// kernel. The lines look at sizes and at the form of the mask, never at a
// tensor's values, which are on the device.
#pragma once

#include <cmath>

#include "fa_common.h"

namespace vxfa {

// The grouped kernel's query heads per workgroup of nw wavefronts (log2): the
// largest power of two, up to nw, that divides the GQA group
inline uint32_t prefill_group_heads_log2(const AttnArgs& a, int nw) {
    uint32_t l = 0;
    while ((2 << l) <= nw && (a.hq / a.hkv) % (2 << l) == 0) ++l;
    return l;
}

// blocks of 32 positions per piece at most, and pieces per tile in the grid
struct GroupPlan {
    uint32_t lp, np;
};
constexpr int kGroupWaves = 8;                    // hd 128: wavefronts of 32 query rows per workgroup
constexpr int kGroupRecord = 64 * 16 * 4 + 64;    // floats of a wavefront's piece record: O, then (m, l) of 32 rows

// Tiles of the grouped kernel (hd 128): `rows` positions of 2^heads heads each
struct GroupTiles {
    int heads_log2, rows, n;     // n per head group
    int64_t groups;              // head groups of all batches
    explicit GroupTiles(const AttnArgs& a) {
        heads_log2 = (int)prefill_group_heads_log2(a, kGroupWaves);
        rows = 32 * (kGroupWaves >> heads_log2);
        n = (int)(((int64_t)a.nq + rows - 1) / rows);
        groups = (int64_t)(a.hq >> heads_log2) * a.b;
    }
    // tiles for four rounds of the chip's 256 CUs: no pieces
    bool many() const { return groups * n >= 1024; }
};

// Blocks per piece and pieces per tile, for record_bytes of scratch. (Any mask is
// taken for a causal one that ends at n_kv, as voxtral's are; another only
// balances worse. An implicit mask and the tensor that it stands for so get the
// same pieces.) Time in units of a block (~0.9 us): a workgroup costs its blocks
// plus kWg, and 256 run at once; merging costs a launch and the records' traffic.
// Forced counts of 1 to 24 over 12 shapes (1000 rows alone to 1000 on 4000, 10 to
// 600 on 600 to 4000, a shard of two kv heads) were at best 2 % better: 600 on
// 3000 1 piece 96.7 us, 2 62.9, 3 54.4 (taken), 4 96.9 (two rounds); 10 on 4000 1
// 75.7, 8 20.4, 16 18.4 (taken), 24 19.7.
inline GroupPlan group_pieces(const AttnArgs& a, const GroupTiles& g, size_t record_bytes) {
    constexpr double kWg = 4.0, kLaunch = 4.0, kRecord = 0.05;
    const int nblk = (a.nkv + 31) / 32;
    auto len = [&](int t) -> int {
        int64_t hi = a.nkv;
        if ((a.mask || a.im_causal) && a.nkv >= a.nq) {
            const int64_t q1 = (int64_t)(t + 1) * g.rows < a.nq ? (int64_t)(t + 1) * g.rows : a.nq;
            hi = q1 + (a.nkv - a.nq);
        }
        return (int)((hi + 31) / 32);
    };
    GroupPlan plan{(uint32_t)nblk, 1};
    if (g.many()) return plan;
    int longest = 1;
    for (int t = 0; t < g.n; ++t) { const int n = len(t); longest = n > longest ? n : longest; }
    double best = 1e30;
    static const int cand[] = {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32, 48, 64};
    for (int P : cand) {
        if (P > 1 && longest < 2 * P) break;
        const int l = ((longest + P - 1) / P + 1) & ~1;
        // pieces per tile: the kernel's own count for the longest possible tile
        const int pn = P == 1 ? 1 : (nblk + l - 1) / l;
        const size_t need = (size_t)g.groups * g.n * (sizeof(int) + (size_t)pn * kGroupWaves * kGroupRecord * sizeof(float)) + 256;
        if (P > 1 && need > record_bytes) break;
        int64_t total = 0, count = 0, recs = 0;
        for (int t = 0; t < g.n; ++t) {
            const int n = len(t), k = n > l ? (n + l - 1) / l : 1;
            total += n;
            count += k;
            if (k > 1) recs += k;
        }
        total *= g.groups;
        count *= g.groups;
        recs *= g.groups;
        const double rounds = (double)((count + 255) / 256);
        const double mean = (double)total / (double)count;
        double cost = rounds * (mean + kWg);
        if (cost < l + kWg) cost = l + kWg;
        if (recs) cost += kLaunch + kRecord * (double)recs;
        if (cost < best) {
            best = cost;
            plan = GroupPlan{(uint32_t)(P == 1 ? nblk : l), (uint32_t)pn};
        }
    }
    return plan;
}

// Blocks of 32 positions from the first to the last that query rows [q0, q1)
// attend; the rows of a mask tensor are taken for causal ones that end at n_kv.
inline int reach_blocks(const AttnArgs& a, int64_t q0, int64_t q1) {
    constexpr int64_t kFar = (int64_t)1 << 40;
    int64_t lo = 0, hi = a.nkv;
    if (a.im_causal) {
        const int64_t off = a.im_offset < -kFar ? -kFar : (a.im_offset > kFar ? kFar : a.im_offset);
        hi = q1 + off < hi ? q1 + off : hi;
        if (a.im_window > 0 && q0 + off - a.im_window + 1 > 0) lo = q0 + off - a.im_window + 1;
    } else if (a.mask && a.nkv >= a.nq) {
        hi = q1 + (a.nkv - a.nq);
    }
    return hi > lo ? (int)((hi + 31) / 32 - lo / 32) : 0;
}

// Estimates of a layer's time at hd 128, in us, without what both kernels' calls
// need (F32 staging, the append launch). Fitted to 2400 calls of either kernel:
// 2 to 4000 rows on up to 4096 cached ones, 4/1 to 32/8 and 8/8 to 32/32 heads, 1
// to 5 batches, no mask, implicit masks and tensors; nine in ten lie within 12 %.

// The general kernel (fa_prefill.hip): a workgroup takes 64 rows of one head and
// splits its walk over four wavefront groups; 256 run at once. A tensor costs each
// of them the scan of its rows, more with every CU at it; a rotary embedding the
// rotation of its queries (the grouped kernel's are rotated by the append launch:
// 16/4 heads, 700 rows alone 37.6 -> 32.4 us grouped, 1000 42.1 -> 35.4).
inline double general128_us(const AttnArgs& a) {
    const int64_t nt = ((int64_t)a.nq + 63) / 64, per = (int64_t)a.hq * a.b, n = nt * per;
    const double scan = n <= 256 ? 12.0 + 3.0 * (double)n / 256 : 12.8;   // (later rounds start apart)
    const double fix = (a.mask ? scan + 0.107 * ((a.nkv + 31) / 32) : (a.im_causal ? 10.2 : 9.4)) +
                       (a.rope_pos ? 4.0 : 0.0);
    const double blk = a.mask ? 0.513 : (a.im_causal ? 0.495 : 0.347);
    auto wg = [&](int64_t i) {   // of workgroup i, the last rows' first
        const int64_t t = nt - 1 - i / per, q1 = 64 * t + 64 < a.nq ? 64 * t + 64 : a.nq;
        return fix + blk * reach_blocks(a, 64 * t, q1);
    };
    double one = wg(0);
    if (nt > 1 && wg(per) > one) one = wg(per);   // (a last tile of a few rows under a window)
    if (n <= 256) return one;
    if (!a.mask && !a.im_causal) return (double)((n + 255) / 256) * one;
    if (per % 8 == 0 && n <= 512) {
        // the longest first: the second round's workgroup i starts when the first's
        // shortest end
        double t = one;
        for (int64_t i = 0; i < n - 256; i += per > 4 ? per / 4 : 1) {
            const double x = wg(255 - i) + wg(256 + i);
            t = x > t ? x : t;
        }
        return t;
    }
    double total = 0;
    for (int64_t t = 0; t < nt; ++t) total += (double)per * wg(t * per);
    const double x = per % 8 ? one : one + wg(n - 1), y = total / 256 + (per % 8 ? 0.6 * one : 0.5 * wg(n - 1));
    return x > y ? x : y;
}

// The grouped kernel with this plan, and its merge. One workgroup a CU.
inline double grouped128_us(const AttnArgs& a, const GroupTiles& g, const GroupPlan& plan) {
    const bool masked = a.mask || a.im_causal;
    const int lp = (int)plan.lp, np = (int)plan.np;
    auto reach = [&](int t) -> int {
        const int64_t q0 = (int64_t)t * g.rows, q1 = q0 + g.rows < a.nq ? q0 + g.rows : a.nq;
        return reach_blocks(a, q0, q1);
    };
    auto pieces = [&](int n) -> int { return n > lp ? (n + lp - 1) / lp : 1; };
    auto waves = [&](int64_t rows) -> int {   // of a workgroup, with rows
        const int w = (int)((rows + 31) / 32) << g.heads_log2;
        return w < kGroupWaves ? w : kGroupWaves;
    };
    int64_t count = 0, recs = 0, total = 0;   // pieces, wavefronts' records, blocks
    int longest = 0;
    for (int t = 0; t < g.n; ++t) {
        const int64_t left = (int64_t)a.nq - (int64_t)t * g.rows;
        const int n = reach(t), k = pieces(n), len = n < lp ? n : lp;
        count += k;
        if (k > 1) recs += k * waves(left < g.rows ? left : g.rows);
        total += n;
        longest = len > longest ? len : longest;
    }
    double w = (double)(count * g.groups) / 256;   // workgroups per CU
    if (g.groups < 8 && g.groups % 8) {
        // fewer head groups than XCDs: the grid's eighths are unequal, the last
        // holds the longest tiles' pieces
        int64_t left = ((int64_t)g.n * np * g.groups + 7) / 8, c = 0;
        for (int t = g.n - 1; t >= 0 && left > 0; --t) {
            const int64_t take = left < np ? left : np, k = pieces(reach(t)) - (np - take);
            c += k > 0 ? k : 0;
            left -= take;
        }
        if ((double)c / 32 > w) w = (double)c / 32;
    }
    // (a workgroup takes longer with every CU at it: memory, clock and power)
    const double fix = 7.6 + (waves(a.nq < g.rows ? a.nq : g.rows) > 4 ? 2.7 : 0.0) + (masked ? 0.3 : 0.0) +
                       7.7 * (w < 1.0 ? w : 1.0);
    const double blk = 0.77, mean = (double)total / (double)count;
    double t = fix + blk * longest;
    if (w > 1.0) {
        const double x = t + 0.3 * (fix + blk * mean), y = 1.14 * w * (fix + blk * mean);
        t = x > y ? x : y;
    }
    if (recs) t += (np > 4 ? 0.8 : 3.1) + 8.3 * pow((double)(recs * g.groups) / (256 * kGroupWaves), 0.78);
    return t;
}

// Whether the grouped kernel takes an hd 128 call (not the short masked one's),
// and its plan. Never with fewer than half of a workgroup's wavefronts at work.
// The lines come from the estimates: measured, us per layer, general -> grouped,
// 32/8 heads: 600 rows on 3000 implicit 119 -> 53.7, 10 on 4000 33.7 -> 18.4, 8192
// alone 1127 -> 550 here; 200 on 320 18.6 -> 23.5, 512 on 88 21.3 -> 32.0, 400
// unmasked 16.2 -> 22.5 (few rows' work, cut into pieces that have to be merged)
// there. own_prep: a mask tensor's intervals cost a launch, ~4 us, which they do not
// where they ride along with F32 staging or an append. But appending within the
// call and appending before it have to give the same bits, so one kernel: both are
// counted at 2.5 us, or 4.5 where the general kernel has more than a round of
// workgroups (over 424 sizes of four head counts the plain call is then at most 3.8 %
// slower than on the general kernel; 383 rows on 1017 40.6 -> 36.5, appended 44.7 ->
// 36.4). A rotated append is counted without (own_prep false).
inline bool prefill_group128(const AttnArgs& a, size_t record_bytes, bool own_prep, int force, GroupPlan& plan) {
    if (((((int64_t)a.nq + 31) / 32) << prefill_group_heads_log2(a, kGroupWaves)) < 4 || force == 0) return false;
    const GroupTiles g(a);
    plan = group_pieces(a, g, record_bytes);
    if (force > 0 || g.many()) return true;
    const bool one_round = ((int64_t)a.nq + 63) / 64 * a.hq * a.b <= 256;
    return general128_us(a) > 1.04 * (grouped128_us(a, g, plan) + (a.mask && own_prep ? (one_round ? 2.5 : 4.5) : 0.0));
}

// Whether the grouped kernel takes a masked hd 64 call from the pipelined one
// (fa_prefill_pp.hip): 4 wavefronts and no pieces, two workgroups a CU, each walking
// its whole range, against one workgroup of 128 rows and 4 KV groups a CU, ~8 us
// of it outside the loop, in two rounds from 257 workgroups on. From 384
// workgroups of this kernel on, where their walks are short or so many (560, dealt
// to the XCDs longest first; else by the walk) that the longest do not set the
// time; a tensor's reach is not known here, so it is
// taken for one that leaves each row a window (the realtime encoder's), unless few
// rows on a long cache make the walks even. Measured, us per layer, pipelined ->
// grouped, 32 heads unless said: implicit window 750, 1500 frames 26.6 -> 24.9, 4000
// 70.5 -> 57.4; causal 1500 26.9 -> 29.6, 2000 35.7 -> 37.6, 24 heads 2000 31.2 ->
// 36.9, 20 heads 4000 86 -> 98 (there), 24 heads 3000 56.3 ->
// 51.8, 2500 55.1 -> 46.8, 64 heads 1500 47.4 -> 40.8 (here). Tensor:
// window 750, 1500 frames 32.7 -> 29.4, F32 K/V 39.3 -> 35.9; causal 1500 31.8 ->
// 34.1 (here all the same), 2000 46.7 -> 42.9, 24 heads 2048 37.6 -> 43.1 (there); 12
// batches of 2 rows on 4000 127 -> 106, of 128 on 2000 63.9 -> 59.1.
inline bool prefill_group64(const AttnArgs& a) {
    constexpr int kWaves = 4;
    if (!a.mask && !a.im_causal) return false;
    const uint32_t hl = prefill_group_heads_log2(a, kWaves);
    const int64_t rows = 32 * (kWaves >> hl), groups = (int64_t)(a.hq >> hl) * a.b;
    const int64_t n = ((int64_t)a.nq + rows - 1) / rows * groups;
    if (n < 384) return false;
    if (n >= 560 && groups % 8 == 0) return true;
    int64_t reach = a.nkv;
    if (a.im_causal && a.im_window > 0 && a.im_window + rows - 1 < reach) reach = a.im_window + rows - 1;
    const int64_t walk = (reach + 31) / 32;   // blocks of the longest
    if (walk <= 32) return true;
    if (!a.mask) return n >= 11 * walk;
    return n >= 7 * walk || (a.nkv >= a.nq && n * (2 * (int64_t)a.nkv - a.nq) >= 600 * (int64_t)a.nkv);
}

// Whether an hd 64 call with a rotary embedding has its query rows rotated by the
// append launch, for the pipelined or the grouped kernel; else the general kernel
// rotates them in each workgroup, and splits a long walk over more of a
// workgroup. Measured, us per layer, general -> pipelined, causal tensor, 32
// heads: 4 rows on 300 18.2 -> 16.0, on 700 20.1 -> 20.7, on 2000 32.6 -> 37.9; 100 on
// 700 24.2 -> 22.9; 200 on 400 22.0 -> 19.5, on 2000 37.2 -> 41.2; 700 on 700 47.2 -> 34.1, on 2300 1.45 times
// as fast: from more than 256 workgroups on (128 of the unmasked form's 128 rows)
// the general kernel runs in rounds.
inline bool prefill_rope64(const AttnArgs& a) {
    const int64_t rows = a.mask ? 64 : 128, n = ((int64_t)a.nq + rows - 1) / rows * a.hq * a.b;
    return a.nkv <= (a.mask ? 800 : 900) || (a.mask ? n > 256 : n >= 128);
}

}  // namespace vxfa
