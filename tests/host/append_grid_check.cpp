// Host check of the append launch (fa_kv_append.hip, linked in; no GPU): the
// launch call is replaced by a stand-in that keeps the grid. For row and batch
// counts up to more than 2^24 new rows in all, the grid stays within what a
// launch takes (fewer than 2^32 threads along x, 65535 along y), and
// AppendGrid::unit gives every new row of every batch and every block of mask
// rows to exactly one workgroup. Built by tests/test_append_grid.py.
#include <cstdio>
#include <cstring>
#include <vector>

#include "../../voxtral.cpp_amd/csrc/fa_common.h"

static dim3 g_grid, g_block;
static int g_launches = 0;
extern "C" {
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t, hipStream_t) {
    g_grid = grid;
    g_block = block;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream) {
    *grid = g_grid;
    *block = g_block;
    *shared = 0;
    *stream = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) {
    ++g_launches;
    return hipSuccess;
}
}
extern "C" hipError_t hipGetLastError(void) { return hipSuccess; }

static int fail(const char* what, long a, long b, long c) {
    printf("FAIL %s: %ld %ld %ld\n", what, a, b, c);
    return 1;
}

int main() {
    const int shapes[][3] = {   // new rows, batches, mask rows (0: none)
        {1, 1, 0}, {3, 1, 0}, {39, 4, 0}, {39, 4, 39}, {1, 7, 1}, {2, 5, 9}, {600, 1, 600}, {5, 3, 4001}, {1, 65535, 5},
        {4096, 4096, 0}, {4100, 4097, 0}, {8192, 2100, 64}, {(1 << 24) - 1, 1, 0}};
    for (const auto& s : shapes) {
        vxfa::AppendArgs a;
        memset(&a, 0, sizeof(a));
        static float word[8];
        static int2 tab[1];
        a.d = 64; a.hkv = 1; a.n_new = s[0]; a.bk = s[1];
        a.k_new = a.v_new = word;
        if (s[2]) { a.m_rows = s[2]; a.m_out = tab; }
        g_launches = 0;
        if (vxfa::launch_kv_append(a, nullptr) != hipSuccess || g_launches != 1) return fail("refused", s[0], s[1], s[2]);
        if ((uint64_t)g_grid.x * g_block.x >= (1ull << 32) || g_grid.y > 65535 || g_grid.z != 1)
            return fail("grid", g_grid.x, g_grid.y, g_grid.z);
        const uint32_t nmb = (uint32_t)(s[2] + 3) / 4;
        const vxfa::AppendGrid g = vxfa::AppendGrid::make(nmb, (uint32_t)s[1]);
        std::vector<uint8_t> rows((size_t)s[0] * s[1], 0), masks(nmb, 0);
        for (uint32_t y = 0; y < g_grid.y; ++y)
            for (uint32_t x = 0; x < g_grid.x; ++x) {
                int mb = 0, t = 0;
                if (!g.unit(x, y, mb, t)) continue;
                if (mb >= 0) {
                    if ((uint32_t)mb >= nmb || masks[mb]++) return fail("mask block", mb, x, y);
                } else if (t < 0 || t >= s[0] || rows[(size_t)y * s[0] + t]++) {
                    return fail("row", t, x, y);
                }
            }
        for (size_t i = 0; i < rows.size(); ++i) if (!rows[i]) return fail("row left out", (long)i, s[0], s[1]);
        for (uint32_t i = 0; i < nmb; ++i) if (!masks[i]) return fail("mask block left out", i, s[0], s[1]);
    }
    printf("ok\n");
    return 0;
}
