// Host check of the routes of vxfa_api.cpp (linked in, no GPU): the HIP calls a
// run makes are stand-ins and the launchers note which one was called, so the
// lines between kernels are held on both sides at sizes where both were timed.
// Built and run by tests/test_routes.py.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>

#include "../../include/vxfa.h"
#include "../../voxtral.cpp_amd/csrc/fa_common.h"

extern "C" {
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { *p = std::malloc(n); return *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) { *s = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { *p = nullptr; return hipErrorInvalidValue; }
}

static std::string g_route;
static void note(const char* s) { g_route += (g_route.empty() ? "" : " ") + std::string(s); }
namespace vxfa {
hipError_t launch_decode(const AttnArgs& a, int, int, hipStream_t) { note(a.mask_rows ? "decode+rows" : "decode"); return hipSuccess; }
hipError_t launch_prefill(const AttnArgs& a, int, int, hipStream_t) {
    note(a.n_split > 1 ? "grouped, cut" : (a.n_split == 1 ? "grouped" : "general"));
    return hipSuccess;
}
hipError_t launch_prefill64_pp(const AttnArgs& a, const StageReq*, hipStream_t) {
    note(a.n_split > 0 ? "grouped" : "pipelined");
    return hipSuccess;
}
hipError_t launch_prefill_pair(const AttnArgs&, hipStream_t) { note("pair"); return hipSuccess; }
bool prefill_pair_fits(const AttnArgs&) { return true; }
hipError_t launch_mask_prep(const AttnArgs&, const StageReq*, hipStream_t) { note("prep"); return hipSuccess; }
hipError_t launch_to_f16_kv(const StageReq&, hipStream_t) { note("stage"); return hipSuccess; }
hipError_t launch_zero(float*, int64_t, hipStream_t) { note("zero"); return hipSuccess; }
hipError_t launch_kv_append(const AppendArgs&, hipStream_t) { note("append"); return hipSuccess; }
}  // namespace vxfa

static vxfa_tensor tensor(int type, int64_t n0, int64_t n1, int64_t n2, int64_t n3, size_t nb1, size_t nb2, size_t nb3) {
    vxfa_tensor t;
    std::memset(&t, 0, sizeof(t));
    t.data = reinterpret_cast<void*>(0x7e0000000000ull);   // (never dereferenced)
    t.type = type;
    t.ne[0] = n0; t.ne[1] = n1; t.ne[2] = n2; t.ne[3] = n3;
    t.nb[0] = type == VXFA_TYPE_F32 ? 4 : 2;
    t.nb[1] = nb1; t.nb[2] = nb2; t.nb[3] = nb3;
    return t;
}

enum Mask { NONE, TENSOR, CAUSAL };
struct Call {
    int hq, hkv, hd;
    int64_t nq, nkv;
    int batch;
    Mask mask;
    int window;
    bool f32, rope, append;
};
static vxfa_ctx* g_ctx;
static std::string route(const Call& c) {
    const size_t e = c.f32 ? 4 : 2, D = c.hd;
    vxfa_tensor q = tensor(VXFA_TYPE_F32, c.hd, c.nq, c.hq, c.batch, c.hq * D * 4, D * 4, c.nq * c.hq * D * 4);
    vxfa_tensor k = tensor(c.f32 ? VXFA_TYPE_F32 : VXFA_TYPE_F16, c.hd, c.nkv, c.hkv, c.batch, c.hkv * D * e, D * e,
                           c.nkv * c.hkv * D * e);
    vxfa_tensor v = k;
    vxfa_tensor dst = tensor(VXFA_TYPE_F32, c.hd, c.hq, c.nq, c.batch, D * 4, c.hq * D * 4, c.nq * c.hq * D * 4);
    const int64_t bm = c.nq == 1 ? c.batch : 1;   // a decode step's streams have a row each
    vxfa_tensor m = tensor(VXFA_TYPE_F16, c.nkv, c.nq, 1, bm, c.nkv * 2, c.nkv * c.nq * 2, c.nkv * c.nq * 2);
    g_route.clear();
    int rc;
    if (c.rope || c.append) {
        vxfa_tensor n = tensor(VXFA_TYPE_F32, c.hkv * c.hd, c.nq, 1, c.batch, c.hkv * D * 4, c.nq * c.hkv * D * 4,
                               c.nq * c.hkv * D * 4);
        vxfa_rope rp{reinterpret_cast<const int32_t*>(0x7e0000000000ull), c.hd, 0, 1e6f, 1.0f};
        const vxfa_tensor* mt = c.mask == TENSOR ? &m : nullptr;
        rc = c.rope ? vxfa_flash_attn_ext_rope(g_ctx, &q, &k, &v, &n, &n, &rp, mt, &dst, 0.125f, 0.f, 0.f, nullptr)
                    : vxfa_flash_attn_ext_append(g_ctx, &q, &k, &v, &n, &n, mt, &dst, 0.125f, 0.f, 0.f, nullptr);
    } else if (c.mask == CAUSAL) {
        vxfa_mask_desc md{VXFA_MASK_CAUSAL, c.window, c.nkv - c.nq};
        rc = vxfa_flash_attn_ext_implicit(g_ctx, &q, &k, &v, &md, &dst, 0.125f, 0.f, 0.f, nullptr);
    } else {
        rc = vxfa_flash_attn_ext(g_ctx, &q, &k, &v, c.mask == TENSOR ? &m : nullptr, &dst, 0.125f, 0.f, 0.f, nullptr);
    }
    return rc == VXFA_OK ? g_route : "status " + std::to_string(rc);
}

int main() {
    g_ctx = vxfa_ctx_create(0);
    if (!g_ctx) return 1;
    struct { Call c; const char* want; } t[] = {
        // batched decode under a mask row per stream: {hq, hkv, hd, nq, n_kv, streams}
        {{32, 8, 128, 1, 300, 2, TENSOR}, "decode"},
        {{32, 8, 128, 1, 8192, 2, TENSOR}, "decode"},
        {{32, 8, 128, 1, 1500, 4, TENSOR}, "decode"},
        {{32, 8, 128, 1, 2048, 4, TENSOR}, "decode+rows"},
        {{32, 8, 128, 1, 500, 8, TENSOR}, "decode"},
        {{32, 8, 128, 1, 1000, 8, TENSOR}, "decode+rows"},
        {{32, 8, 128, 1, 8192, 32, TENSOR}, "decode+rows"},
        {{32, 8, 128, 1, 1000, 3, TENSOR, 0, true}, "decode"},
        {{32, 8, 128, 1, 1500, 3, TENSOR, 0, true}, "decode+rows"},
        {{32, 8, 128, 1, 4096, 3, TENSOR, 0, true}, "decode+rows"},
        {{32, 8, 128, 1, 4097, 3, TENSOR, 0, true}, "decode"},
        {{32, 8, 128, 1, 8192, 4, TENSOR, 0, true}, "decode"},
        {{32, 8, 128, 1, 8192, 5, TENSOR, 0, true}, "decode+rows"},
        {{32, 8, 128, 1, 256, 24, TENSOR, 0, true}, "decode"},
        {{32, 8, 128, 1, 300, 16, TENSOR, 0, true}, "decode+rows"},
        {{8, 2, 128, 1, 8192, 4, TENSOR}, "decode"},
        {{32, 8, 128, 1, 8192, 1, TENSOR}, "decode"},
        // hd 128 prefill: {hq, hkv, hd, nq, n_kv, batch}
        {{32, 8, 128, 8192, 8192, 1, CAUSAL}, "grouped"},
        {{32, 8, 128, 600, 3600, 1, CAUSAL}, "grouped, cut"},
        {{32, 8, 128, 10, 4000, 1, CAUSAL}, "grouped, cut"},
        {{32, 8, 128, 64, 1000, 1, CAUSAL}, "grouped, cut"},
        {{32, 8, 128, 200, 520, 1, CAUSAL}, "general"},
        {{32, 8, 128, 512, 600, 1, CAUSAL}, "general"},
        {{32, 8, 128, 700, 700, 1, CAUSAL}, "general"},
        {{32, 8, 128, 1500, 1700, 1, CAUSAL}, "grouped"},
        {{8, 2, 128, 200, 700, 1, CAUSAL}, "grouped, cut"},
        {{8, 2, 128, 2200, 2200, 1, CAUSAL}, "general"},
        {{8, 8, 128, 1634, 1634, 1, CAUSAL, 373}, "general"},
        {{32, 32, 128, 128, 520, 1, CAUSAL}, "general"},
        {{32, 32, 128, 64, 4000, 1, CAUSAL}, "general"},
        {{32, 8, 128, 200, 720, 1, TENSOR}, "general"},
        {{32, 8, 128, 100, 900, 1, TENSOR}, "prep grouped, cut"},
        {{32, 8, 128, 513, 513, 1, TENSOR}, "general"},
        {{16, 4, 128, 1025, 1025, 1, TENSOR}, "general"},
        {{32, 8, 128, 383, 1400, 1, TENSOR}, "prep grouped, cut"},
        {{32, 8, 128, 700, 1000, 1, TENSOR}, "prep grouped, cut"},
        {{32, 8, 128, 600, 3600, 1, TENSOR, 0, true}, "prep grouped, cut"},
        {{32, 8, 128, 600, 3600, 1, TENSOR, 0, false, true}, "append grouped, cut"},
        {{16, 4, 128, 1000, 1000, 1, TENSOR, 0, false, true}, "append grouped, cut"},
        {{16, 4, 128, 700, 700, 1, TENSOR, 0, false, true}, "append grouped, cut"},
        {{32, 8, 128, 300, 439, 1, CAUSAL}, "pair"},
        {{8, 2, 128, 3000, 3000, 1, TENSOR}, "prep grouped, cut"},
        {{32, 8, 128, 64, 520, 1, CAUSAL}, "grouped, cut"},
        {{32, 8, 128, 512, 2200, 1, CAUSAL}, "general"},
        {{32, 8, 128, 700, 1300, 1, CAUSAL}, "grouped, cut"},
        {{32, 8, 128, 64, 512, 1, NONE}, "general"},
        {{32, 8, 128, 400, 400, 1, NONE}, "general"},
        {{32, 8, 128, 400, 400, 4, NONE}, "grouped"},
        {{32, 8, 128, 2000, 2000, 1, NONE}, "grouped"},
        {{32, 8, 128, 8, 3000, 1, NONE}, "grouped, cut"},
        // hd 64
        {{20, 20, 64, 1500, 1500, 1, NONE}, "pipelined"},
        {{32, 32, 64, 1400, 1400, 1, CAUSAL, 750}, "pipelined"},
        {{32, 32, 64, 1500, 1500, 1, CAUSAL, 750}, "grouped"},
        {{32, 32, 64, 1500, 1500, 1, CAUSAL}, "pipelined"},
        {{32, 32, 64, 4000, 4000, 1, CAUSAL, 750}, "grouped"},
        {{20, 20, 64, 4000, 4000, 1, CAUSAL}, "pipelined"},
        {{64, 64, 64, 1500, 1500, 1, CAUSAL}, "grouped"},
        {{32, 32, 64, 2500, 2500, 1, CAUSAL}, "grouped"},
        {{28, 28, 64, 3000, 3000, 1, CAUSAL}, "pipelined"},
        {{80, 80, 64, 513, 513, 1, CAUSAL}, "grouped"},
        {{32, 32, 64, 1500, 1500, 1, TENSOR, 0, true}, "grouped"},
        {{24, 24, 64, 2048, 2048, 1, TENSOR}, "pipelined"},
        {{32, 32, 64, 2, 4000, 12, TENSOR}, "grouped"},
        {{32, 32, 64, 32, 8192, 12, CAUSAL}, "pipelined"},
        {{32, 8, 64, 1530, 1600, 1, TENSOR}, "grouped"},
        {{32, 32, 64, 4, 400, 1, TENSOR, 0, false, true}, "append pipelined"},
        {{32, 32, 64, 4, 2004, 1, TENSOR, 0, false, true}, "append general"},
        {{32, 32, 64, 200, 2200, 1, NONE, 0, false, true}, "append general"},
        {{32, 32, 64, 700, 2200, 1, TENSOR, 0, false, true}, "append pipelined"},
        {{32, 32, 64, 400, 2200, 1, NONE, 0, false, true}, "append pipelined"},
    };
    int bad = 0;
    for (const auto& x : t) {
        const std::string got = route(x.c);
        if (got != x.want) {
            std::printf("FAIL %d/%d hd %d nq %lld n_kv %lld batch %d mask %d window %d f32 %d rope %d: %s, not %s\n", x.c.hq,
                        x.c.hkv, x.c.hd, (long long)x.c.nq, (long long)x.c.nkv, x.c.batch, x.c.mask, x.c.window, x.c.f32,
                        x.c.rope, got.c_str(), x.want);
            bad = 1;
        }
    }
    // appended rows: the same kernel, and so the same bits, as appending and then
    // attending. (The launches ahead of it are not compared.)
    const int heads[][2] = {{32, 8}, {8, 2}, {16, 4}, {32, 32}, {8, 8}, {12, 2}};
    int64_t calls = 0;
    for (const auto& h : heads)
        for (int hd : {64, 128})
            for (int batch : {1, 3})
                for (int64_t nq : {2, 10, 39, 64, 100, 200, 383, 512, 700, 1000, 1500, 2200})
                    for (int64_t past = 0; past < 4000; past = past * 5 / 4 + 37)
                        for (Mask m : {NONE, TENSOR}) {
                            auto kernel = [](const std::string& r) {
                                const size_t p = r.find("prep ") == 0 ? 5 : r.find("append ") == 0 ? 7 : 0;
                                return r.substr(p);
                            };
                            Call c{h[0], h[1], hd, nq, past + nq, batch, m};
                            const std::string op = route(c);
                            c.append = true;
                            const std::string ap = route(c);
                            ++calls;
                            if (kernel(op) != kernel(ap) && ++bad <= 10)
                                std::printf("FAIL %d/%d hd %d nq %lld n_kv %lld batch %d mask %d: %s, appended %s\n", h[0], h[1],
                                            hd, (long long)nq, (long long)(past + nq), batch, m, op.c_str(), ap.c_str());
                        }
    vxfa_ctx_destroy(g_ctx);
    if (calls < 3000) bad = 1;
    if (!bad) std::printf("ok\n");
    return bad != 0;
}
