"""The hd 128 prefill whose workgroups share K/V blocks among the heads of a
kv group (fa_prefill_group.hip): tile, block and piece edges, GQA groups, mask
forms, types and scratch limits, against the exact float64 reference.

Bound: Q, K, V and P are rounded to f16 (relative 2^-11 each), sums are F32;
outputs are averages of unit-normal V rows, so 2e-3 absolute and 2e-3 relative
(2-norm) leave a factor of about three over the largest error of the f16
rounding (measured 2e-4 to 7e-4)."""
import numpy as np
import pytest

import cases
from oracle import oracle

pytestmark = pytest.mark.gpu

vx = cases.load_package().vxfa


# (hd 128 wherever it can: which kernel a call takes by itself depends on its size)
@pytest.fixture(scope="module")
def runner():
    import gpu_util
    r = gpu_util.Runner(VXFA_PREFILL_GROUP=1)
    yield r
    r.close()


def agree(out, c, atol=2e-3, rel=2e-3):
    ref = cases.oracle_f64(c)
    assert np.isfinite(out).all()
    d = out.astype(np.float64) - ref
    m, r = np.abs(d).max(), np.linalg.norm(d) / max(np.linalg.norm(ref), 1e-30)
    print(f"[{c.name}] maxabs {m:.2e} rel {r:.2e}", flush=True)
    assert m <= atol and r <= rel, (c.name, m, r)


def run(runner, c, **kw):
    print(f"[case] {c.name}", flush=True)
    rc, out = runner.run(c)
    assert rc == 0
    agree(out, c, **kw)
    return out


# rows around a wavefront's 32 and a workgroup's 64 positions, positions around
# a block's 32, a step's 64 and several pieces
@pytest.mark.parametrize("n,n_kv", [(2, 513), (31, 545), (33, 576), (64, 640), (65, 1000), (100, 2047), (7, 4100),
                                    (300, 801), (513, 513)])
def test_causal_edges(runner, n, n_kv):
    c = cases.prefill_case(n, kv_offset=n_kv - n, seed=2000 + n, name=f"causal {n} of {n_kv}")
    out = run(runner, c)
    rc, out2 = runner.run_implicit(c, vx.mask_desc(vx.MASK_CAUSAL, 0, n_kv - n))
    assert rc == 0 and np.array_equal(out, out2)


@pytest.mark.parametrize("hq,hkv,n,n_kv", [(8, 1, 40, 700), (4, 2, 90, 900), (3, 3, 130, 700), (6, 2, 150, 650),
                                           (10, 2, 257, 520), (4, 1, 64, 3000)])
def test_groups(runner, hq, hkv, n, n_kv):
    run(runner, cases.prefill_case(n, hq=hq, hkv=hkv, kv_offset=n_kv - n, seed=2100 + hq, name=f"{hq}/{hkv}"))
    run(runner, cases.prefill_case(n, hq=hq, hkv=hkv, causal=False, kv_offset=n_kv - n, seed=2200 + hq,
                                   name=f"{hq}/{hkv} no mask"))


def test_no_mask_short(runner):
    for n, n_kv in ((40, 1), (40, 31), (33, 33), (64, 65)):
        run(runner, cases.prefill_case(n, causal=False, kv_offset=n_kv - n, seed=2300 + n_kv, name=f"no mask {n_kv}"),
            rel=4e-3)


def _mask_case(kind, n=100, n_kv=901, **kw):
    c = cases.prefill_case(n, kv_offset=n_kv - n, seed=2400, name=kind, hq=8, hkv=2, **kw)
    rng = np.random.default_rng(2401)
    m = cases.implicit_mask(n, n_kv, n_kv - n)
    if kind == "window":
        m = cases.implicit_mask(n, n_kv, n_kv - n, 130)
    elif kind == "finite":
        b = rng.normal(0, 2, m.shape).astype(np.float16).view(np.uint16)
        m = np.where(m == 0, b, m).astype(np.uint16)
    elif kind == "holes":
        m = np.where(rng.random(m.shape) < 0.3, cases.NEG_INF_F16, m).astype(np.uint16)
        m[50, :] = cases.NEG_INF_F16
    elif kind == "lowest":
        m = np.where(m == 0, m, np.uint16(0xFBFF)).astype(np.uint16)
        m[60, :] = 0xFBFF
    elif kind == "dead rows":
        m[10:14, :] = cases.NEG_INF_F16
        m[64:, :] = cases.NEG_INF_F16
    elif kind == "far":   # live entries in blocks far apart
        m[:] = cases.NEG_INF_F16
        m[:, 3] = 0
        m[:, 880] = 0
    return cases.with_mask(c, m)


# (a row whose every entry is the type's lowest value keeps only a few bits of
# its scores: s + m in F32 at |m| log2(e) = 9.4e4 is exact to 2^-8, which as an
# exponent is 0.3 %; its outputs are averages below 0.2)
@pytest.mark.parametrize("kind", ["window", "finite", "holes", "lowest", "dead rows", "far"])
def test_masks(runner, kind):
    run(runner, _mask_case(kind), atol=4e-3 if kind == "lowest" else 2e-3)
    c = _mask_case(kind, n_kv=904)     # 16-byte aligned rows: vector mask loads
    run(runner, c, atol=4e-3 if kind == "lowest" else 2e-3)


def test_mask_planes_and_batches(runner):
    n, n_kv = 70, 600
    c = cases.decode_case(n_kv, hq=8, hkv=2, batch=2, seed=2500, name="planes")
    rng = np.random.default_rng(2501)
    c.bufs.pop("q"); c.views.pop("q")
    ne, nb = cases._batched_q(n, 8, 128, 4, 2)
    c.add("q", "q", cases.normal(rng, (2, n, 8, 128)), oracle.F32, ne, nb)
    m = np.stack([cases.implicit_mask(n, n_kv, n_kv - n, w) for w in (0, 100, 300, 50, 0, 64, 512, 33)])
    c.add("mask", "mask", m.reshape(2, 4, n, n_kv), oracle.F16, *cases.views.mask(n_kv, n, 4, 2))
    run(runner, c)


@pytest.mark.parametrize("scale", [0.0, -0.11, 0.3])
def test_scales(runner, scale):
    c = cases.prefill_case(70, kv_offset=530, hq=8, hkv=2, seed=2600, name=f"scale {scale}")
    c.scale = cases.f32(scale)
    run(runner, c, rel=3e-3)
    rng = np.random.default_rng(2602)
    b = rng.normal(0, 1, (70, 600)).astype(np.float16).view(np.uint16)
    run(runner, cases.with_mask(c, b), rel=3e-3)


def test_f32_kv(runner):
    run(runner, cases.prefill_case(90, kv_offset=700, seed=2700, kv_f32=True, name="f32 K/V"))


def test_scratch_of_a_call_without_context(runner):
    """8 MiB of scratch, and the piece records' own array."""
    for kw in ({}, {"kv_f32": True}):
        c = cases.prefill_case(128, kv_offset=1800, seed=2800, name=f"no-alloc {kw}", **kw)
        print(f"[case] {c.name}", flush=True)
        rc, out = runner.run_noalloc(c)
        assert rc == 0
        agree(out, c)


def test_f16_q_and_rows_that_raise_the_maximum(runner):
    """K grows along the cache, so every block passes the running maximum."""
    n, n_kv = 96, 1500
    c = cases.prefill_case(n, kv_offset=n_kv - n, hq=8, hkv=2, seed=2900, name="ramp")
    k = c.bufs["k"].view(np.float16).astype(np.float32)
    k *= (1.0 + 6.0 * np.arange(n_kv, dtype=np.float32) / n_kv)[:, None, None]
    c.bufs["k"] = cases.f16_bits(k)
    q = cases.f16_bits(c.bufs["q"])
    c.bufs["q"] = q
    b, _, ne, nb, off = c.views["q"]
    c.views["q"] = (b, oracle.F16, ne, tuple(x // 2 for x in nb), off)
    run(runner, c, atol=8e-3, rel=3e-3)


# hd 64 (4 wavefronts, no pieces) takes masked calls of at least 384
# workgroups: 128 rows of a head each, or 32 of a group of four
def _hd64(kind, n, heads, q_f16=False, kv_f32=False):
    c = cases.encoder_case(n, heads, 64, seed=3100 + n, window=750 if kind == "window" else None, q_f16=q_f16,
                           kv_f32=kv_f32, name=f"hd64 {kind} {n}x{heads}")
    if kind == "window":
        return c
    rng = np.random.default_rng(3101)
    m = cases.implicit_mask(n, n, 0)
    if kind == "finite":
        m = np.where(m == 0, rng.normal(0, 2, m.shape).astype(np.float16).view(np.uint16), m).astype(np.uint16)
    elif kind == "dead rows":
        m[:130] = cases.NEG_INF_F16
        m[300] = cases.NEG_INF_F16
    return cases.with_mask(c, m)


@pytest.mark.parametrize("kind,n,heads,kw", [("window", 1057, 44, {}), ("causal", 513, 80, {}), ("finite", 481, 96, {}),
                                             ("dead rows", 500, 96, {"q_f16": True}),
                                             ("window", 1100, 43, {"kv_f32": True})])
def test_hd64(runner, kind, n, heads, kw):
    c = _hd64(kind, n, heads, **kw)
    out = run(runner, c)
    if kind == "dead rows":
        assert not out[0, :130].any() and not out[0, 300].any()
    if kind in ("window", "causal"):
        rc, out2 = runner.run_implicit(c, vx.mask_desc(vx.MASK_CAUSAL, 750 if kind == "window" else 0, 0))
        assert rc == 0 and np.array_equal(out, out2)


def test_hd64_group_and_scale(runner):
    c = cases.prefill_case(1530, hq=32, hkv=8, hd=64, kv_offset=70, seed=3200, name="hd64 32/8")
    run(runner, c)
    c.scale = cases.f32(-0.2)
    run(runner, c, rel=3e-3)


@pytest.mark.parametrize("kind", ["holes", "planes", "batch"])
def test_hd64_mask_forms(runner, kind):
    """A third of the entries removed; a plane for each of two heads; two
    batches with masks of their own."""
    n, rng = 500, np.random.default_rng(3300)
    m = cases.implicit_mask(n, n, 0, 130)
    if kind == "batch":
        c = cases.decode_case(n, hq=48, hkv=48, hd=64, batch=2, seed=3301, name="hd64 batch")
        c.bufs.pop("q"); c.views.pop("q")
        c.add("q", "q", cases.normal(rng, (2, n, 48, 64)), oracle.F32, *cases._batched_q(n, 48, 64, 4, 2))
        c.add("mask", "mask", np.stack([m, cases.implicit_mask(n, n, 0)]), oracle.F16, *cases.views.mask(n, n, 1, 2))
    else:
        c = cases.encoder_case(n, 96, 64, seed=3302, name=f"hd64 {kind}")
        if kind == "planes":
            bias = rng.normal(0, 2, m.shape).astype(np.float16).view(np.uint16)
            planes = np.stack([m, np.where(m == 0, bias, m).astype(np.uint16)])
            c.add("mask", "mask", planes, oracle.F16, *cases.views.mask(n, n, 2, 1))
        else:
            cases.with_mask(c, np.where(rng.random(m.shape) < 0.3, cases.NEG_INF_F16, m).astype(np.uint16))
    run(runner, c)
