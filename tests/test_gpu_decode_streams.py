"""Batched decode with a mask tensor: the rows' live ranges found by a
pre-pass and splits sized to each stream, or by a scan in every workgroup
(fa_decode.hip). Stream lengths at the
edges of tiles, rounds and splits, rows that are no range of zeros, appended
rows, F32 caches and hd 64, against the exact float64 reference.

Bound: as for every decode test, 2e-3 absolute and 2e-3 relative against an
f16 cache (Q, K, V rounded to f16; measured 2e-4 relative), 2e-6 relative
against an F32 cache (F32 products; measured 4e-7)."""
import numpy as np
import pytest

import cases
from oracle import oracle

pytestmark = pytest.mark.gpu


# every test with the pre-pass, and with a scan in each workgroup (what a call
# takes by itself depends on its size)
@pytest.fixture(scope="module", params=[1, 0], ids=["pre-pass", "scan"])
def runner(request):
    import gpu_util
    r = gpu_util.Runner(VXFA_DECODE_ROWS=request.param)
    yield r
    r.close()


def agree(out, c):
    ref = cases.oracle_f64(c)
    assert np.isfinite(out).all()
    d = out.astype(np.float64) - ref
    m, r = np.abs(d).max(), np.linalg.norm(d) / np.linalg.norm(ref)
    print(f"[{c.name}] maxabs {m:.2e} rel {r:.2e}", flush=True)
    f32 = c.views["k"][1] == oracle.F32
    assert m <= 2e-3 and r <= (2e-6 if f32 else 2e-3), (c.name, m, r)


def streams(lens, cap, **kw):
    c = cases.decode_case(cap, batch=len(lens), seed=3000 + len(lens), name=f"streams {cap} {lens[:4]}", **kw)
    m = np.zeros((len(lens), 1, cap), dtype=np.uint16)
    for b, n in enumerate(lens):
        m[b, 0, n:] = cases.NEG_INF_F16
    c.add("mask", "mask", m, oracle.F16, *cases.views.mask(cap, 1, 1, len(lens)))
    return c


def run(runner, c):
    print(f"[case] {c.name}", flush=True)
    rc, out = runner.run(c)
    assert rc == 0
    agree(out, c)


@pytest.mark.parametrize("kv_f32", [False, True])
@pytest.mark.parametrize("cap,lens", [(64, (1, 15, 16, 17, 33, 64)), (700, (700, 1, 63, 65, 128, 129, 640)),
                                      (2051, (2051, 2048, 2049, 5)), (1, (1, 1))])
def test_lengths(runner, cap, lens, kv_f32):
    run(runner, streams(lens, cap, kv_f32=kv_f32))


@pytest.mark.parametrize("hq,hkv,hd", [(8, 8, 64), (8, 4, 128), (4, 1, 128), (8, 2, 64)])
def test_groups(runner, hq, hkv, hd):
    run(runner, streams((300, 31, 1000, 512), 1000, hq=hq, hkv=hkv, hd=hd))


def test_rows_of_every_kind(runner):
    """A range in the middle, a hole, finite values, one entry at each end,
    nothing live (zeros come out), everything live."""
    cap = 900
    c = streams((cap,) * 6, cap)
    m = c.bufs["mask"].reshape(6, cap)
    m[0, :200] = m[0, 700:] = cases.NEG_INF_F16
    m[1, 300:340] = cases.NEG_INF_F16
    m[2, :] = np.random.default_rng(31).normal(0, 1, cap).astype(np.float16).view(np.uint16)
    m[2, 100:] = cases.NEG_INF_F16
    m[3, 1:-1] = cases.NEG_INF_F16
    m[4, :] = cases.NEG_INF_F16
    print(f"[case] {c.name} kinds", flush=True)
    rc, out = runner.run(c)
    assert rc == 0
    assert not out[4].any()
    agree(out, c)


def test_one_mask_row_for_all_streams(runner):
    c = streams((500,) * 4, 800)
    m = c.bufs["mask"].reshape(4, 1, 800)[:1]
    c.bufs.pop("mask"); c.views.pop("mask")
    c.add("mask", "mask", m, oracle.F16, *cases.views.mask(800, 1, 1, 1))
    run(runner, c)


def test_append(runner):
    """The new row of each stream is the cache's last: live for the stream that
    sees all of it, stored for every stream."""
    lens, cap = (600, 100, 599), 600
    c = streams(lens, cap)
    rng = np.random.default_rng(41)
    kn, vn = cases.normal(rng, (3, 1, 1024)), cases.normal(rng, (3, 1, 1024))
    res = runner.run_append(c, kn, vn)
    for t, new in (("k", kn), ("v", vn)):
        c.bufs[t].reshape(3, cap, 1024)[:, -1] = cases.f16_bits(new)[:, 0]
        assert np.array_equal(res[2][t], c.bufs[t].view(np.uint8).reshape(-1)), t
    assert res[0] == 0
    agree(res[1], c)
