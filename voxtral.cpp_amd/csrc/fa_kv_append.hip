// fa_kv_append.hip — appends new K and V rows to an f16 KV cache.
//
// Replaces the two ggml_cpy nodes of build_decoder_layer that store the
// layer's new keys and values in the cache (src/voxtral.cpp:1758-1770) when
// the cache is F16: each F32 element is rounded to f16 (round to nearest
// even, overflow to inf, the F16C conversion ggml's CPU copy uses). One
// launch writes K and V: workgroup (t, b) writes token t of kv batch b, each
// thread converts 8 consecutive elements (two 16-byte loads, one 16-byte
// store). The source row is Hkv * D floats, kv head h at h * D (the layout of
// the reshape at :1743); the cache row of head h is the view's (pos, h) row.
// With rope_pos set, K rows are first turned by the rotary embedding of
// their token's position (ggml_rope_ext mode 0, :1748-1749), as the
// reference rotates K before storing it.
//
// A prefill call has more to prepare, and its launch does it along the way:
// with a rotary embedding the query rows of token t are rotated from the same
// cos / sin table and left as f16 for the attention kernel, which otherwise
// forms a table of its own in each of its workgroups; a mask tensor's row
// intervals are found by further workgroups (first in the grid, as they are
// the long ones).
#include "fa_common.h"
#include "fa_mask_rows.h"

namespace vxfa {

// a mask block takes four mask rows
__global__ __launch_bounds__(256) void kv_append_kernel(AppendArgs a, AppendGrid g) {
    int mb, t;
    if (!g.unit(blockIdx.x, blockIdx.y, mb, t)) return;
    if (mb >= 0) {
        const MaskRowArgs m{a.mask, a.m_nb1, a.m_nb2, a.m_nb3, a.m_n, a.m_nq, a.m_hm, a.m_rows, a.m_out};
        mask_rows_block(m, (uint32_t)mb, (int)threadIdx.x);
        return;
    }
    const int b = blockIdx.y;
    const int per = a.hkv * a.d / 8;   // 8-element chunks per matrix row
    const int perq = a.q_out ? a.hq * a.d / 8 : 0;
    // the token's rotary cos / sin per pair, shared by its heads
    __shared__ float2 cs[128];
    if (a.rope_pos) {
        const int p = a.rope_pos[b * a.n_new + t];
        // (pairs below 64: one unrolled running product shared by the lanes)
        for (int j = threadIdx.x; j < a.d / 2; j += 256)
            cs[j] = j < 64 ? rope_cs_chain<64>(p, j, a.rope_ts) : rope_cs(p, j, a.rope_ts);
        __syncthreads();
    }
    for (int c = threadIdx.x; c < 2 * per + perq; c += 256) {
        const int m = c < per ? 0 : (c < 2 * per ? 1 : 2);   // K, V, Q
        const int e = 8 * (c - m * per);
        const int h = e / a.d, d = e - h * a.d;
        const char* src;
        if (m == 2) src = (const char*)a.q + (int64_t)t * a.q_nb1 + (int64_t)h * a.q_nb2 + (int64_t)b * a.q_nb3 + 4 * d;
        else if (m == 1) src = (const char*)a.v_new + (int64_t)t * a.vn_nb1 + (int64_t)b * a.vn_nb3 + 4 * e;
        else src = (const char*)a.k_new + (int64_t)t * a.kn_nb1 + (int64_t)b * a.kn_nb3 + 4 * e;
        const floatx4* sp = (const floatx4*)src;
        const floatx4 x0 = sp[0], x1 = sp[1];
        float x[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
        if (m != 1 && a.rope_pos) rope8_tab(x, d, cs, a.rope_dims);
        half8 y;
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] = (_Float16)x[i];
        const int64_t pos = (int64_t)a.pos0 + t;
        char* dst;
        if (m == 2) dst = (char*)(a.q_out + (((int64_t)b * a.n_new + t) * a.hq + h) * a.d);
        else if (m == 1) dst = (char*)a.v + pos * a.v_nb1 + (int64_t)h * a.v_nb2 + (int64_t)b * a.v_nb3;
        else dst = (char*)a.k + pos * a.k_nb1 + (int64_t)h * a.k_nb2 + (int64_t)b * a.k_nb3;
        *(half8*)(dst + 2 * d) = y;
    }
}

hipError_t launch_kv_append(const AppendArgs& a, hipStream_t st) {
    if (a.n_new <= 0 || a.bk <= 0) return hipSuccess;
    if (a.d % 8 || a.d > 256 || a.bk > 65535) return hipErrorInvalidValue;
    if (a.m_out && a.m_rows <= 0) return hipErrorInvalidValue;
    const AppendGrid g = AppendGrid::make(a.m_out ? ((uint32_t)a.m_rows + 3) / 4 : 0, (uint32_t)a.bk);
    if ((int64_t)a.n_new + g.mx > kMaxGridX) return hipErrorInvalidValue;
    hipLaunchKernelGGL(kv_append_kernel, dim3((unsigned)a.n_new + g.mx, (unsigned)a.bk), dim3(256), 0, st, a, g);
    return hipGetLastError();
}

}  // namespace vxfa
