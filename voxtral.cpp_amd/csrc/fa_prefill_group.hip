// fa_prefill_group.hip — prefill for gfx950 (hd 128, and masked hd 64 of many
// workgroups): the query heads of one kv head share each K/V block, the KV
// range is cut into pieces when the query rows alone leave the chip idle (hd
// 128).
//
// Replaces the backend kernel of GGML_OP_FLASH_ATTN_EXT for the decoder
// prefill calls of voxtral.cpp (src/voxtral.cpp:1802, GQA 32/8, hd 128, the
// causal mask of :2104-2111) that the short masked kernel does not take (n_kv
// over 512, or no mask), where it is faster than the general one
// (prefill_group128 in fa_prefill_route.h). With head dim 64 also the realtime
// encoder's calls (:2179-2190) of many workgroups (prefill_group64).
// Measured, us per layer, on the general kernel (one head and one wavefront per
// SIMD) and here: 8192 rows causal 1127 -> 546-567 (~980 TFLOP/s), 600 rows on 3000
// cached, implicit mask 119 -> 54, with rope, append and mask tensor 164 -> 61, 10
// rows on 4000 cached 33.7 -> 18.5.
//
// Work decomposition
//   Workgroup = 8 wavefronts (hd 64: 4) of 32 query rows, two per SIMD: HPW
//   query heads of one kv head (the largest power of two dividing the GQA
//   group, up to 8) x 8 / HPW row tiles, so a group of 4 takes 64 positions of 4 heads. All
//   of them walk the same 32-position K/V blocks, read from L2 once for 256
//   query rows and shared in LDS.
//   A tile's live blocks are cut into pieces of at most `lp` blocks, one
//   workgroup each (piece p of a tile with fewer pieces ends at once). A tile
//   of one piece writes its output; otherwise every piece leaves its
//   unnormalised O with the rows' running max and sum in the workspace, and
//   fa_prefill_group_combine merges them in piece order.
// What bounds it: per wavefront and block 16 MFMAs (512 cycles of its SIMD's
//   matrix pipe) against ~130 VALU instructions of softmax, so the two pipes
//   are about even and have to overlap. PV runs one block behind:
//     half t:  MFMA  O += V_{t-1}^T P(t-1)^T, then S(t+1) = K_{t+1} Q^T
//              VALU  softmax of S(t) -> P(t)
//   where no MFMA waits for that half's VALU work (at 8192 rows the matrix pipe
//   is busy 50 % of the cycles at ~1.88 GHz; other orders of the half measured
//   0-4 % slower). K_{t+1} is read at the top
//   of the half and lands under the PV MFMAs, V_t after them and lands under
//   the S MFMAs.
// K/V staging: a ring of 4 steps of 64 positions (32 KiB each), filled by
//   global_load_lds_dwordx4 (hd 64: 16 KiB a step); step u + 3 is issued in iteration u into the slot
//   of step u - 1, one barrier after its last read, and has two iterations to
//   land. One barrier per 64 positions.
// MFMA operand layouts, LDS swizzles and the row-to-KV permutation are those
// of fa_prefill.hip; the softmax without a block max (P against the running
// max; the sum of P tells when a score passed it by more than 2^8) is that of
// fa_prefill_pp.hip.
// Masks: each lane's row has a live interval, from the formula of an implicit
// mask or from the pre-pass over a mask tensor (launch_mask_prep); blocks not
// wholly live for a wavefront's rows get their dead scores set to -inf. A
// workgroup with a row that is no interval (finite values, holes) reads the
// mask per block and skips the blocks that are dead for its rows.
// A block that is dead for all 32 rows of a wavefront (the second of a step at
// the end of an odd walk, a part of the union that only other rows attend)
// takes a block of zeros for V, so an infinity or NaN at positions that the
// mask removes from those rows cannot reach them as 0 x V. (8192 rows causal
// 550 -> 560 us, the realtime encoder's layer 34.5 -> 35.1, with no mask 83.7 ->
// 81.6 at 2000 rows.)
#include "fa_common.h"
#include "fa_prefill_route.h"

#include <type_traits>

namespace vxfa {

template <int HD>
struct PG {
    static constexpr int D = HD;
    static constexpr int KS = D / 16;             // S-MFMA k-steps
    static constexpr int DB = D / 32;             // O^T row blocks
    static constexpr int BK = 32;                 // positions per block
    static constexpr int ROW = D * 2;             // bytes per K/V row
    static constexpr int BLK = BK * ROW;          // bytes of one matrix block
    static constexpr int STEP = 2 * BLK;          // one matrix of a 64-position step
    static constexpr int NS = 4;                  // ring slots
    static constexpr int NW = D / 16;             // wavefronts (8 or 4)
    static constexpr int LOGR = D == 128 ? 8 : 7; // log2 of a workgroup's rows (32 per wavefront)
    static constexpr int NT = 64 * NW;
    static constexpr int RECO = 64 * 16 * DB;     // floats of O in a wavefront's record
    static constexpr int REC = RECO + 64;         // and (m, l) of 32 rows
    // 1/sqrt(hd) in log2 units, as the host computes it from ggml's float scale
    static constexpr float C = (D == 128 ? 0.08838834764831845f : 0.125f) * kLog2e;
};
constexpr float PG_TAU_SUM = 256.0f;              // 2^8
constexpr float PG_TAU = 8.0f;

struct Pieces {
    uint32_t hpw_log2;                 // log2 of the query heads per workgroup
    uint32_t lp;                       // blocks per piece at most
    DivMod np;                         // pieces per tile in the grid
    int32_t nqt;                       // tiles
    int32_t nhg;                       // head groups (hq / heads per workgroup)
    int* count;                        // pieces of each tile [b][nhg][nqt]
    float* rec;                        // records [b][nhg][nqt][np][NW][REC]
};

template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 16, "vmcnt range");
    __builtin_amdgcn_s_waitcnt(N | (7 << 4) | (15 << 8));
}

__device__ __forceinline__ int wave_min32(int x) {
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) x = min(x, __shfl_xor(x, m, 64));
    return __builtin_amdgcn_readfirstlane(x);
}
__device__ __forceinline__ int wave_max32(int x) {
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) x = max(x, __shfl_xor(x, m, 64));
    return __builtin_amdgcn_readfirstlane(x);
}

// MM: 0 no mask, 1 a mask tensor (intervals in a.mask_rows), 2 implicit.
// CL: the scale is exactly 1/sqrt(hd) (c is a literal, see exps below).
// QT: 0 F32 rows, 1 f16 rows, 2 F32 rows to rotate (a call whose rotated rows
// do not fit the scratch; 14 KB of code that the others do not fetch).
template <int HD, int QT, bool CL, int MM>
__global__ __launch_bounds__(PG<HD>::NT, 2) void fa_prefill_group(AttnArgs a, GridMap gm, Pieces pc) {
    using P = PG<HD>;
    constexpr int D = P::D, KS = P::KS, DB = P::DB, BK = P::BK, ROW = P::ROW, BLK = P::BLK, STEP = P::STEP,
                  NS = P::NS, NW = P::NW, REC = P::REC;
    // K steps, V steps, and with 8 wavefronts half of the Q staging (160 KiB, all
    // of a CU's LDS; 68 KiB with 4). The first block past the ring is zeros from
    // iteration 0 on: what a wavefront reads for V of a block dead for its rows.
    constexpr bool QPAST = QT != 2 && NW == 8;            // Q staging past the ring
    constexpr int ZERO = 2 * NS * STEP;
    __shared__ __attribute__((aligned(16))) char smem[ZERO + (QPAST ? 4 : 1) * BLK];

    int idx, hg, b, hk, bkv;
    gm.locate(blockIdx.x, idx, hg, b, hk, bkv);
    const int qt = (int)pc.np.div((uint32_t)idx);
    const int piece = idx - qt * (int)pc.np.d;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nl = lane & 31;
    const int hh = lane >> 5;
    const int hpw = 1 << pc.hpw_log2;
    const int bm = 32 * (NW >> pc.hpw_log2);              // positions per workgroup
    const int h = hg * hpw + (wave & (hpw - 1));
    const int q0 = qt * bm;                               // the workgroup's first row
    const int r0 = q0 + 32 * (wave >> pc.hpw_log2);       // the wavefront's first row
    const int qrow = r0 + nl;
    const bool qvalid = qrow < a.nq;
    const bool active = r0 < a.nq;                        // the wavefront has rows
    const int qld = min(qrow, a.nq - 1);
    const char* kb = (const char*)a.k + (int64_t)hk * a.k_nb2 + (int64_t)bkv * a.k_nb3;
    const char* vb = (const char*)a.v + (int64_t)hk * a.v_nb2 + (int64_t)bkv * a.v_nb3;

    // ---- live interval of the lane's row, union over the workgroup ----------
    // (MM = 1: NW / 2 table entries per lane cover the workgroup's rows; every
    // wavefront reduces them itself, no barrier)
    int rlo = 0, rhi = a.nkv - 1;                         // the lane's row
    int lo = 0, hi = a.nkv;                               // the workgroup
    bool slow = false;
    if constexpr (MM == 1) {
        const int2* tab = a.mask_rows + (int64_t)(b % a.bm) * a.hm * a.nq;
        int2 iv[NW / 2];
#pragma unroll
        for (int u = 0; u < NW / 2; ++u) {
            const int i = 64 * u + lane;                  // head i / bm of the workgroup, row i % bm
            const int hi_ = i >> (P::LOGR - (int)pc.hpw_log2), row = min(q0 + (i & (bm - 1)), a.nq - 1);
            iv[u] = tab[(int64_t)((hg * hpw + hi_) % a.hm) * a.nq + row];
        }
        const int2 mine = tab[(int64_t)(h % a.hm) * a.nq + qld];
        int tlo = 0x7fffffff, thi = -1;
        bool non = false;
#pragma unroll
        for (int u = 0; u < NW / 2; ++u) {
            non = non || iv[u].x == -2;
            if (iv[u].x >= 0 && iv[u].x <= iv[u].y) {
                tlo = min(tlo, iv[u].x);
                thi = max(thi, iv[u].y);
            }
        }
        slow = __any(non);
        lo = wave_min32(tlo);
        hi = wave_max32(thi) + 1;
        rlo = mine.x;
        rhi = mine.y;
        if (slow) { lo = 0; hi = a.nkv; }
    }
    if constexpr (MM == 2) {
        const int64_t q1 = min(q0 + bm, a.nq) - 1;        // the workgroup's last real row
        const int64_t wb = a.im_window > 0 ? a.im_offset - a.im_window + 1 : INT64_MIN / 2;
        auto clampkv = [&](int64_t x) { return (int)(x < -1 ? -1 : (x > a.nkv ? a.nkv : x)); };
        lo = max(clampkv(q0 + wb), 0);
        hi = min(clampkv(q1 + a.im_offset), a.nkv - 1) + 1;
        rlo = clampkv(qld + wb);
        rhi = min(clampkv(qld + a.im_offset), a.nkv - 1);
    }
    const int blo = hi > lo ? lo / BK : 0;
    const int nblk = hi > lo ? (hi + BK - 1) / BK - blo : 0;

    // ---- this piece's blocks [bs, bs + nb) -----------------------------------
    int bs = blo, nb = nblk;
    bool whole = true;
    if (pc.np.d > 1) {
        const int n = max((nblk + (int)pc.lp - 1) / (int)pc.lp, 1);
        if (piece >= n) return;
        whole = n == 1;
        const int len = ((nblk + n - 1) / n + 1) & ~1;    // whole steps
        bs = blo + min(piece * len, nblk);
        nb = min(len, blo + nblk - bs);
        if (piece == 0 && tid == 0) pc.count[((int64_t)b * pc.nhg + hg) * pc.nqt + qt] = n;
    }

    // ---- Q loads -----------------------------------------------------------------
    // Whole rows of the wavefront's 32 (rows past n_q read the last one), turned
    // into the operand layout through LDS below: a load of the operand layout
    // touches 32 rows per instruction, and its 16 instructions of 8 wavefronts
    // kept the CU's address unit busy for ~2 us. QT 2 (rotation) needs a row's
    // pairs together and loads the operand layout.
    constexpr int QL = QT == 1 ? KS : 2 * KS;        // 16-byte loads per lane
    constexpr int QCH = QT == 1 ? D / 8 : D / 4;     // 16-byte chunks per row
    floatx4 qraw[QL];
    int qpos = 0;
    {
        const char* qp = (const char*)a.q + (int64_t)h * a.q_nb2 + (int64_t)b * a.q_nb3;
        if constexpr (QT == 2) {
            const char* p = qp + (int64_t)qld * a.q_nb1 + 32 * hh;
#pragma unroll
            for (int u = 0; u < QL; ++u) qraw[u] = *(const floatx4*)(p + 64 * (u >> 1) + 16 * (u & 1));
            qpos = a.rope_pos[(int64_t)b * a.nq + qld];
        } else {
#pragma unroll
            for (int u = 0; u < QL; ++u) {
                const int row = min(r0 + (64 / QCH) * u + lane / QCH, a.nq - 1);
                qraw[u] = __builtin_nontemporal_load((const floatx4*)(qp + (int64_t)row * a.q_nb1) + lane % QCH);
            }
        }
    }

    // ---- step loads: global -> LDS ring ----------------------------------------
    // Instruction i (0, 1) of wavefront w fills rows [RPI (w + NW i), + RPI) of
    // the step; lane l writes LDS chunk l % CH of row + l / CH, which holds the
    // row's chunk (l % CH) ^ swizzle(row). Rows at or past n_kv read row
    // n_kv - 1.
    constexpr int CH = D / 8, RPI = 64 / CH;
    static_assert(2 * NW * RPI == 2 * BK, "two instructions per matrix and step");
    const int nstep = (nb + 1) >> 1;
    uint32_t ldk[2], ldv[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = RPI * (wave + NW * i) + lane / CH;
        ldk[i] = (uint32_t)r * (uint32_t)a.k_nb1 + ((lane % CH) ^ swz_k<D>(r)) * 16;
        ldv[i] = (uint32_t)r * (uint32_t)a.v_nb1 + ((lane % CH) ^ swz_v<D>(r)) * 16;
    }
    const uint32_t lds0 = lds_offset(smem);
    auto issue = [&](int u) {
        const int kv0 = (bs + 2 * u) * BK;
        const uint32_t kd = lds0 + (u & (NS - 1)) * STEP, vd = kd + NS * STEP;
        const char* kst = kb + (int64_t)kv0 * a.k_nb1;
        const char* vst = vb + (int64_t)kv0 * a.v_nb1;
        if (kv0 + 2 * BK <= a.nkv) {
#pragma unroll
            for (int i = 0; i < 2; ++i) dma16(kst, ldk[i], kd + RPI * (wave + NW * i) * ROW);
#pragma unroll
            for (int i = 0; i < 2; ++i) dma16(vst, ldv[i], vd + RPI * (wave + NW * i) * ROW);
        } else {
            // (recomputed here rather than held across the loop; the empty asm
            // keeps it here)
            int ln = lane;
            asm volatile("" : "+v"(ln));
            const int rmax = a.nkv - 1 - kv0;   // kv0 < n_kv
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int r = RPI * (wave + NW * i) + ln / CH;
                dma16(kst, (uint32_t)min(r, rmax) * (uint32_t)a.k_nb1 + ((ln % CH) ^ swz_k<D>(r)) * 16,
                      kd + RPI * (wave + NW * i) * ROW);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int r = RPI * (wave + NW * i) + ln / CH;
                dma16(vst, (uint32_t)min(r, rmax) * (uint32_t)a.v_nb1 + ((ln % CH) ^ swz_v<D>(r)) * 16,
                      vd + RPI * (wave + NW * i) * ROW);
            }
        }
    };
    for (int u = 0; u < min(nstep, 2); ++u) issue(u);

    // ---- Q operand: row qrow, dims 16 ks + 8 hh .. + 7, rounded to f16; the sign
    // of the scale folded in (0 for scale 0) -----------------------------------------
    const float c = a.scale_log2 != 0.f ? fabsf(a.scale_log2) : 1.0f;
    half8 qb[KS];
    {
        const float sg = a.scale_log2 < 0.f ? -1.0f : (a.scale_log2 > 0.f ? 1.0f : 0.0f);
        if constexpr (QT == 2) {
            // one running product over the row's pairs, as ggml builds its
            // cos / sin cache: pair 8 ks + o belongs to the lanes of half o / 4
            float th = (float)qpos;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = qraw[2 * ks + (e >> 2)][e & 3];
                float ang[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int o = 0; o < 8; ++o) {
                    if (ks > 0 || o > 0) th *= a.rope_ts;
                    if ((o >> 2) == hh) ang[o & 3] = th;
                }
                rope8_ang(x, ang, 16 * ks + 8 * hh, a.rope_dims);
#pragma unroll
                for (int e = 0; e < 8; ++e) qb[ks][e] = (_Float16)(x[e] * sg);
            }
        } else {
            // the wavefront's 32 rows, 16-byte chunk j of row r at j ^ (r % CH);
            // wavefronts 0-3 in ring slot 3 (filled from iteration 0 on), 4-7 past
            // the ring
            char* qs = smem + (wave < 2 ? 3 * STEP + wave * BLK
                                        : (wave < 4 ? (NS + 3) * STEP + (wave - 2) * BLK
                                                    : 2 * NS * STEP + (wave - 4) * BLK));
#pragma unroll
            for (int u = 0; u < QL; ++u) {
                const int r = (64 / QCH) * u + lane / QCH, j = lane % QCH;
                if constexpr (QT == 1) {
                    *(half8*)(qs + r * ROW + ((j ^ (r % CH)) * 16)) = __builtin_bit_cast(half8, qraw[u]) * (_Float16)sg;
                } else {
                    half4 y;
#pragma unroll
                    for (int e = 0; e < 4; ++e) y[e] = (_Float16)(qraw[u][e] * sg);
                    *(half4*)(qs + r * ROW + (((j >> 1) ^ (r % CH)) * 16) + (j & 1) * 8) = y;
                }
            }
            __builtin_amdgcn_wave_barrier();   // (one wavefront's LDS accesses run in order)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                qb[ks] = *(const half8*)(qs + nl * ROW + (((2 * ks + hh) ^ (nl % CH)) * 16));
            __builtin_amdgcn_wave_barrier();
        }
    }
    // the block of zeros (past the ring: by the wavefront whose rows it held)
    if constexpr (QPAST) {
        if (wave == 4) {
#pragma unroll
            for (int i = 0; i < BLK / 1024; ++i) *(half8*)(smem + ZERO + 1024 * i + 16 * lane) = half8{};
        }
    } else {
        static_assert(QPAST || BLK == 16 * P::NT, "one 16-byte store per thread");
        *(half8*)(smem + ZERO + 16 * tid) = half8{};
    }

    // ---- operand reads ------------------------------------------------------------
    // K: A-operand row nl of a block is K row krow, chunk 2 ks + hh; the blocks
    // and rows are 256-byte aligned, so the chunk (with its swizzle) is a field
    // of the address and ks is an XOR of it.
    int kbase;
    {
        const int am = nl >> 3, ahb = (nl >> 2) & 1, ab = nl & 3;
        const int krow = ahb ? 16 + ((am + 2) & 3) * 4 + ab : 4 * am + ab;
        kbase = krow * ROW + (hh ^ swz_k<D>(krow)) * 16;
    }
    // V^T operand (cc, db): rows (hh ? 24 - 8 cc : 8 cc) + vq, chunk 4 db + clo
    // (cc flips bit 3 of the row, db bits 2 and 3 of the chunk)
    int vbase;
    {
        const int vq = (lane & 15) >> 2;
        const int clo = 2 * ((lane & 31) >> 4) + ((lane & 3) >> 1);
        vbase = NS * STEP + ((hh ? 24 : 0) + vq) * ROW + (clo ^ swz_v<D>(vq)) * 16 + (lane & 1) * 8;
    }
    // block t of the piece
    auto read_k = [&](int t, half8 (&kr)[KS]) {
        const int base = kbase + (t & (2 * NS - 1)) * BLK;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) kr[ks] = *(const half8*)(smem + (base ^ (32 * ks)));
    };
    auto v_at = [&](int t) -> int { return (t & (2 * NS - 1)) * BLK; };
    auto read_v = [&](int at, half8 (&vr)[2][DB]) {
        const int base = vbase + at;
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                const char* p = smem + (base ^ (8 * ROW * cc + 64 * db));
                const half4 lo4 = lds_read_tr16(p);
                const half4 hi4 = lds_read_tr16(p + 4 * ROW);
                vr[cc][db] = half8{lo4[0], lo4[1], lo4[2], lo4[3], hi4[0], hi4[1], hi4[2], hi4[3]};
            }
    };
    auto s_mfma = [&](floatx16& s, const half8 (&kr)[KS]) {
        s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kr[0], qb[0], floatx16{}, 0, 0, 0);
#pragma unroll
        for (int ks = 1; ks < KS; ++ks) s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kr[ks], qb[ks], s, 0, 0, 0);
    };
    floatx16 o[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) o[db] = floatx16{};
    auto pv_mfma = [&](const half8 (&p)[2], const half8 (&vr)[2][DB]) {
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
#pragma unroll
            for (int db = 0; db < DB; ++db) o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vr[cc][db], p[cc], o[db], 0, 0, 0);
    };

    // largest lower and smallest upper bound over the wavefront's rows: a
    // block inside both is wholly live
    const int last = min(a.nkv, (bs + nb) * BK) - 1;      // this piece's last position
    rhi = min(rhi, last);
    int hlo = 0, hhi = last;
    if constexpr (MM == 1) {
        hlo = wave_max32(rlo);
        hhi = wave_min32(rhi);
    }
    if constexpr (MM == 2) {
        hlo = __builtin_amdgcn_readlane(rlo, 31);
        hhi = __builtin_amdgcn_readlane(rhi, 0);
    }
    int dlo = 0, dhi = last;                              // MM = 2: the union of its rows' intervals
    if constexpr (MM == 2) {
        dlo = __builtin_amdgcn_readlane(rlo, 0);
        dhi = __builtin_amdgcn_readlane(rhi, 31);
    }
    // (returns where block t's V is read: the zeros when the block is dead for all
    // of the wavefront's rows, as P x V has to be 0 there whatever V holds)
    auto mask_fix = [&](floatx16& sc, int t) -> int {
        const int kv0 = (bs + t) * BK;
        int at = v_at(t);
        if (!(kv0 >= hlo && kv0 + BK - 1 <= hhi)) {
            if constexpr (MM == 0) {
                if (kv0 > last) at = ZERO - NS * STEP;
            } else if constexpr (MM == 1) {
                if (!__any(kv0 <= rhi && kv0 + BK > rlo && rlo <= rhi)) at = ZERO - NS * STEP;
            } else {
                if (kv0 > dhi || kv0 + BK <= dlo) at = ZERO - NS * STEP;
            }
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int kv = kv0 + pf_kv_of(hh, j);
                if constexpr (MM == 0) sc[j] = kv > last ? -INFINITY : sc[j];
                else sc[j] = (kv < rlo || kv > rhi) ? -INFINITY : sc[j];
            }
        }
        return at;
    };

    // ---- softmax ------------------------------------------------------------------
    // P = 2^(c s - m) as two f16 B operands, and the lane's sum of them. With CL
    // c is a literal: v_fmamk_f32 issues at twice the rate of the
    // three-register FMA; -m has to reach it as a plain register.
    const half2 ones = {(_Float16)1.0f, (_Float16)1.0f};
    float m = -INFINITY, l = 0.f;
    auto exps = [&](const floatx16& sc, half8 (&p)[2]) -> float {
        float nm = (m == -INFINITY) ? 0.f : -m;
        asm("" : "+v"(nm));
        float ls[2] = {0.f, 0.f};
#pragma unroll
        for (int cc = 0; cc < 2; ++cc) {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                p[cc][i] = (_Float16)exp2_fast(fmaf(sc[8 * cc + i], CL ? P::C : c, nm));
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const half2 p2 = {p[cc][2 * i], p[cc][2 * i + 1]};
                ls[i & 1] = __builtin_amdgcn_fdot2(p2, ones, ls[i & 1], false);
            }
        }
        return ls[0] + ls[1];
    };
    auto block_max = [&](const floatx16& sc) -> float {
        float r = sc[0];
#pragma unroll
        for (int j = 1; j < 16; ++j) r = fmaxf(r, sc[j]);
        return pair32_max(r) * c;
    };
    auto raise = [&](float mx) {
        const float mnew = fmaxf(m, mx);
        const float ms = (mnew == -INFINITY) ? 0.f : mnew;
        const float alpha = exp2_fast(m - ms);
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int j = 0; j < 16; ++j) o[db][j] *= alpha;
        l *= alpha;
        m = mnew;
    };
    // (a row that has no live score yet takes the exact path; rows past n_q
    // take no part in the choice)
    auto softmax = [&](const floatx16& sc, half8 (&p)[2]) {
        float ls = exps(sc, p);
        bool up = !(ls <= PG_TAU_SUM);
        if constexpr (MM != 0) up = (up || m == -INFINITY) && qvalid;
        if (__any(up)) {
            raise(block_max(sc));
            ls = exps(sc, p);
        }
        l += ls;
    };

    // before iteration 0: steps 0 and 1 (step 2's loads, issued after the wait
    // for Q, may stay in flight)
    if (nstep > 2) {
        issue(2);
        wait_vm<4>();
    } else {
        wait_vm<0>();
    }
    __syncthreads();

    auto walk = [&](auto slow_tag) __attribute__((always_inline)) {
        constexpr bool SLOW = decltype(slow_tag)::value;
        half8 kr[KS], vr[2][DB], pa[2], pb[2];
        floatx16 sa, sb;
        if constexpr (SLOW) {
            // each block on its own, its mask values read per row
            const uint16_t* mr = (const uint16_t*)((const char*)a.mask + (int64_t)(h % a.hm) * a.m_nb2 +
                                                   (int64_t)(b % a.bm) * a.m_nb3 + (int64_t)qld * a.m_nb1);
            const float inv_c = kLog2e / c;
            for (int u = 0; u < nstep; ++u) {
                if (u + NS - 1 < nstep) issue(u + NS - 1);
                for (int t = 2 * u; active && t < min(2 * u + 2, nb); ++t) {
                    const int kv0 = (bs + t) * BK;
                    uint16_t mv[16];
                    if (a.mask_vec && kv0 + BK <= a.nkv) {
                        const uint16_t* p = mr + kv0 + 16 * hh;
                        const u32x4 w0 = *(const u32x4*)(p + 8 * hh), w1 = *(const u32x4*)(p + 8 - 8 * hh);
#pragma unroll
                        for (int w = 0; w < 4; ++w) {
                            mv[2 * w] = (uint16_t)w0[w];
                            mv[2 * w + 1] = (uint16_t)(w0[w] >> 16);
                            mv[8 + 2 * w] = (uint16_t)w1[w];
                            mv[8 + 2 * w + 1] = (uint16_t)(w1[w] >> 16);
                        }
                    } else {
#pragma unroll
                        for (int j = 0; j < 16; ++j) mv[j] = mr[min(kv0 + pf_kv_of(hh, j), a.nkv - 1)];
#pragma unroll
                        for (int j = 0; j < 16; ++j)
                            if (kv0 + pf_kv_of(hh, j) >= a.nkv) mv[j] = kF16NegInf;
                    }
                    bool live = false;
#pragma unroll
                    for (int j = 0; j < 16; ++j) live |= mv[j] != kF16NegInf;
                    if (!__any(live && qvalid)) continue;
                    read_k(t, kr);
                    s_mfma(sa, kr);
                    read_v(v_at(t), vr);
#pragma unroll
                    for (int j = 0; j < 16; ++j)
                        sa[j] = mv[j] == kF16NegInf ? -INFINITY : fmaf(f16_bits_to_f32(mv[j]), inv_c, sa[j]);
                    const float mx = block_max(sa);
                    if (__any(mx > m + PG_TAU && qvalid)) raise(mx);
                    l += exps(sa, pa);
                    pv_mfma(pa, vr);
                }
                wait_vm<0>();
                __syncthreads();
            }
        } else {
            if (nb == 0) return;
            // PV of the block before the first adds zero
#pragma unroll
            for (int cc = 0; cc < 2; ++cc) {
                pb[cc] = half8{};
#pragma unroll
                for (int db = 0; db < DB; ++db) vr[cc][db] = half8{};
            }
            read_k(0, kr);
            s_mfma(sa, kr);
            mask_fix(sa, 0);
            m = block_max(sa);
            // half t: PV(t - 1), S(t + 1) and the softmax of S(t)
            auto half = [&](int t, floatx16& scur, floatx16& snext, half8 (&pcur)[2], half8 (&pprev)[2]) {
                const int va = mask_fix(scur, t);
                read_k(t + 1, kr);
                pv_mfma(pprev, vr);
                __builtin_amdgcn_sched_barrier(0x6);   // VALU and SALU may cross
                read_v(va, vr);
                s_mfma(snext, kr);
                softmax(scur, pcur);
            };
            // (whole steps: a second block past nb has no live score, and the last
            // half's S is not used)
            for (int u = 0; u < nstep; ++u) {
                if (u + NS - 1 < nstep) issue(u + NS - 1);
                if (active) {
                    half(2 * u, sa, sb, pa, pb);
                    half(2 * u + 1, sb, sa, pb, pa);
                }
                // K of step u + 2 and V of step u + 1 have landed: at most the
                // loads of step u + 3 and V of step u + 2 are in flight
                if (u + 3 < nstep) wait_vm<6>();
                else if (u + 2 < nstep) wait_vm<2>();
                else wait_vm<0>();
                __syncthreads();
            }
            pv_mfma(pb, vr);
        }
    };
    if constexpr (MM == 1) {
        if (slow) walk(std::true_type{});
        else walk(std::false_type{});
    } else {
        walk(std::false_type{});
    }

    // ---- output, or this piece's record --------------------------------------------
    const float lt = pair32_sum(l);
    if (whole) {
        const float inv = (lt == 0.f) ? 0.f : 1.0f / lt;
        if (qvalid) {
            float* out = a.dst + (((int64_t)b * a.nq + qrow) * a.hq + h) * D;
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int a4 = 0; a4 < 4; ++a4)
                    *(floatx4*)(out + 32 * db + 8 * a4 + 4 * hh) =
                        floatx4{o[db][4 * a4] * inv, o[db][4 * a4 + 1] * inv, o[db][4 * a4 + 2] * inv,
                                o[db][4 * a4 + 3] * inv};
        }
    } else if (active) {
        const int64_t ri = ((((int64_t)b * pc.nhg + hg) * pc.nqt + qt) * pc.np.d + piece) * NW + wave;
        float* rec = pc.rec + ri * REC;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int a4 = 0; a4 < 4; ++a4)
                *(floatx4*)(rec + (4 * db + a4) * 256 + 4 * lane) =
                    floatx4{o[db][4 * a4], o[db][4 * a4 + 1], o[db][4 * a4 + 2], o[db][4 * a4 + 3]};
        if (hh == 0) *(float2*)(rec + P::RECO + 2 * nl) = float2{m, lt};
    }
}

// Merge of the pieces of a tile; lane layout as in the records. A wavefront
// takes 32 output dims of one wavefront tile (32 rows of a head) and every
// SP-th piece, with UP records' loads in flight; the SP wavefronts of a
// workgroup then merge through LDS (SP = 1: a workgroup is the four dim
// groups of a wavefront tile).
template <int SP, int UP>
__global__ __launch_bounds__(256) void fa_prefill_group_combine(AttnArgs a, Pieces pc) {
    using P = PG<128>;
    constexpr int D = P::D, DB = P::DB, NW = P::NW, REC = P::REC;
    static_assert(SP == 1 || SP == 4, "wavefronts per tile and dims");
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nl = lane & 31, hh = lane >> 5;
    const uint32_t wt = SP == 1 ? blockIdx.x : blockIdx.x / DB;         // wavefront tile
    const int db = SP == 1 ? w : (int)(blockIdx.x % DB);
    const int sp = SP == 1 ? 0 : w;
    const int64_t tile = wt / NW;                         // (b nhg + hg) nqt + qt
    const int wave = wt % NW;
    const int n = pc.count[tile];
    const int qt = (int)(tile % pc.nqt);
    const int hg = (int)(tile / pc.nqt % pc.nhg), b = (int)(tile / pc.nqt / pc.nhg);
    const int hpw = 1 << pc.hpw_log2;
    const int h = hg * hpw + (wave & (hpw - 1));
    const int qrow = qt * 32 * (NW >> pc.hpw_log2) + 32 * (wave >> pc.hpw_log2) + nl;
    if (n <= 1 || qrow - nl >= a.nq) return;
    const float* rec = pc.rec + (tile * pc.np.d * NW + wave) * REC;
    const int64_t stride = (int64_t)NW * REC;
    float M = -INFINITY, L = 0.f;
    floatx4 acc[4];
#pragma unroll
    for (int a4 = 0; a4 < 4; ++a4) acc[a4] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int p0 = sp; p0 < n; p0 += SP * UP) {
        float2 ml[UP];
        floatx4 v[UP][4];
#pragma unroll
        for (int i = 0; i < UP; ++i) {
            const float* r = rec + min(p0 + SP * i, n - 1) * stride;
            ml[i] = *(const float2*)(r + P::RECO + 2 * nl);
#pragma unroll
            for (int a4 = 0; a4 < 4; ++a4) v[i][a4] = *(const floatx4*)(r + (4 * db + a4) * 256 + 4 * lane);
        }
        float mn = M;
#pragma unroll
        for (int i = 0; i < UP; ++i) {
            if (p0 + SP * i >= n) ml[i] = float2{-INFINITY, 0.f};
            mn = fmaxf(mn, ml[i].x);
        }
        const float ms = mn == -INFINITY ? 0.f : mn;
        const float al = exp2_fast(M - ms);
        L *= al;
#pragma unroll
        for (int a4 = 0; a4 < 4; ++a4) acc[a4] *= al;
#pragma unroll
        for (int i = 0; i < UP; ++i) {
            const float wt_ = exp2_fast(ml[i].x - ms);
            L = fmaf(wt_, ml[i].y, L);
            if (p0 + SP * i < n) {
#pragma unroll
                for (int a4 = 0; a4 < 4; ++a4)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[a4][e] = fmaf(wt_, v[i][a4][e], acc[a4][e]);
            }
        }
        M = mn;
    }
    if constexpr (SP > 1) {
        __shared__ floatx4 xo[SP][4][64];
        __shared__ float2 xm[SP][64];
#pragma unroll
        for (int a4 = 0; a4 < 4; ++a4) xo[sp][a4][lane] = acc[a4];
        xm[sp][lane] = float2{M, L};
        __syncthreads();
        // wavefront w merges quarter w of the 16 dims a lane holds
        float mm = -INFINITY;
#pragma unroll
        for (int s = 0; s < SP; ++s) mm = fmaxf(mm, xm[s][lane].x);
        const float ms = mm == -INFINITY ? 0.f : mm;
        L = 0.f;
        floatx4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < SP; ++s) {
            const float f = exp2_fast(xm[s][lane].x - ms);
            L = fmaf(f, xm[s][lane].y, L);
            const floatx4 x = xo[s][w][lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = fmaf(f, x[e], o[e]);
        }
        if (qrow < a.nq) {
            const float inv = (L == 0.f) ? 0.f : 1.0f / L;
            *(floatx4*)(a.dst + (((int64_t)b * a.nq + qrow) * a.hq + h) * D + 32 * db + 8 * w + 4 * hh) = o * inv;
        }
    } else if (qrow < a.nq) {
        const float inv = (L == 0.f) ? 0.f : 1.0f / L;
        float* out = a.dst + (((int64_t)b * a.nq + qrow) * a.hq + h) * D + 32 * db + 4 * hh;
#pragma unroll
        for (int a4 = 0; a4 < 4; ++a4) *(floatx4*)(out + 8 * a4) = acc[a4] * inv;
    }
}

template <int HD, int QT, bool CL>
static void launch_pg(const AttnArgs& a, const GridMap& gm, const Pieces& pc, unsigned nwg, hipStream_t st) {
    const dim3 grid(nwg), block(PG<HD>::NT);
    if (a.mask) hipLaunchKernelGGL((fa_prefill_group<HD, QT, CL, 1>), grid, block, 0, st, a, gm, pc);
    else if (a.im_causal) hipLaunchKernelGGL((fa_prefill_group<HD, QT, CL, 2>), grid, block, 0, st, a, gm, pc);
    else if constexpr (HD == 128) hipLaunchKernelGGL((fa_prefill_group<HD, QT, CL, 0>), grid, block, 0, st, a, gm, pc);
}

template <int HD>
static hipError_t launch_group(const AttnArgs& a, hipStream_t st) {
    using P = PG<HD>;
    if (a.mask && !a.mask_rows) return hipErrorInvalidValue;
    if (a.nkv <= 0 || a.nq <= 0) return hipErrorInvalidValue;
    const bool masked = a.mask || a.im_causal;
    if (HD == 64 && (!masked || a.rope_pos)) return hipErrorInvalidValue;
    Pieces pc;
    pc.hpw_log2 = prefill_group_heads_log2(a, P::NW);
    const int hpw = 1 << pc.hpw_log2, bm = 32 * (P::NW >> pc.hpw_log2);
    const int nqt = (a.nq + bm - 1) / bm, nhg = a.hq / hpw;
    const int64_t groups = (int64_t)nhg * a.b;
    // (the kernel cuts a tile into ceil(blocks / lp) pieces: np has to hold them)
    const int32_t np = a.n_split;
    if (np < 1 || a.dec_chunk < 1 || (np > 1 && HD != 128) || (int64_t)a.dec_chunk * np * P::BK < a.nkv)
        return hipErrorInvalidValue;
    pc.lp = (uint32_t)a.dec_chunk;
    pc.np = DivMod::make((uint32_t)np);
    pc.nqt = nqt;
    pc.nhg = nhg;
    pc.count = reinterpret_cast<int*>(a.ws);
    const size_t counts = ((size_t)groups * nqt + 63) & ~(size_t)63;
    pc.rec = np > 1 ? a.ws + counts : nullptr;
    if (np > 1 && (!a.ws || (counts + (size_t)groups * nqt * np * P::NW * P::REC) * sizeof(float) > a.ws_bytes))
        return hipErrorInvalidValue;
    const int64_t nwg = groups * nqt * np;
    if (nwg <= 0 || nwg > 0x7fffffff) return hipErrorInvalidValue;
    const GridMap gm = masked ? GridMap::make_tiles_desc((int)nwg, nqt * (int)np, nhg, a.hkv, a.b, a.bk)
                              : GridMap::make((int)nwg, nqt * (int)np, nhg, a.hkv, a.b, a.bk);
    const bool cl = fabsf(a.scale_log2) == P::C;
    const unsigned n = (unsigned)nwg;
    if (a.q_f16) {
        if (cl) launch_pg<HD, 1, true>(a, gm, pc, n, st);
        else launch_pg<HD, 1, false>(a, gm, pc, n, st);
    } else if (HD == 128 && a.rope_pos) {
        if (cl) launch_pg<128, 2, true>(a, gm, pc, n, st);
        else launch_pg<128, 2, false>(a, gm, pc, n, st);
    } else {
        if (cl) launch_pg<HD, 0, true>(a, gm, pc, n, st);
        else launch_pg<HD, 0, false>(a, gm, pc, n, st);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || np == 1) return e;
    if constexpr (HD == 128) {
        const unsigned nwt = (unsigned)(groups * nqt * P::NW);
        if (np <= 4) hipLaunchKernelGGL((fa_prefill_group_combine<1, 4>), dim3(nwt), dim3(256), 0, st, a, pc);
        else hipLaunchKernelGGL((fa_prefill_group_combine<4, 4>), dim3(nwt * P::DB), dim3(256), 0, st, a, pc);
    }
    return hipGetLastError();
}

hipError_t launch_prefill_group(const AttnArgs& a, int head_dim, hipStream_t st) {
    static_assert(PG<128>::NW == kGroupWaves && PG<128>::REC == kGroupRecord, "the plan's sizes");
    if (head_dim == 128) return launch_group<128>(a, st);
    if (head_dim == 64) return launch_group<64>(a, st);
    return hipErrorInvalidValue;
}

}  // namespace vxfa
