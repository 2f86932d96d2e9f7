"""Positions that the mask removes from every query row, holding infinities
and NaN in K and V: the grouped prefill kernel's workgroups walk the union of
their rows' live blocks in pairs, so they meet blocks that are dead for a
wavefront's 32 rows, or past the last live one; none may reach an output."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu

vx = cases.load_package().vxfa


@pytest.fixture(scope="module")
def runner():
    import gpu_util
    r = gpu_util.Runner(VXFA_PREFILL_GROUP=1)
    yield r
    r.close()


def check(c, ref, out):
    assert np.isfinite(out).all(), c.name
    d = out.astype(np.float64) - ref
    m, r = np.abs(d).max(), np.linalg.norm(d) / np.linalg.norm(ref)
    print(f"[{c.name}] maxabs {m:.2e} rel {r:.2e}", flush=True)
    # (Q, K, V and P rounded to f16; measured 2e-4 to 7e-4)
    assert m <= 2e-3 and r <= 2e-3, (c.name, m, r)


def poisoned(c, positions):
    """The exact answer, then K and V of the positions made inf, -inf and NaN in turn."""
    ref = cases.oracle_f64(c)
    bad = np.array([0x7C00, 0xFC00, 0x7E00], dtype=np.uint16)
    for role in ("k", "v"):
        x = c.bufs[c.views[role][0]]
        for i, p in enumerate(positions):
            x[p] = bad[i % 3]
    return ref


def rows_mask(n, n_kv, spans):
    """Group of 32 rows g attends spans[g % len(spans)]."""
    m = np.full((n, n_kv), cases.NEG_INF_F16, np.uint16)
    for g in range(0, n, 32):
        lo, hi = spans[(g // 32) % len(spans)]
        m[g:g + 32, lo:hi] = 0
    return m


HD128 = [(8, 2), (2, 2), (8, 1)]


@pytest.mark.parametrize("hq,hkv", HD128)
def test_block_past_an_odd_walk(runner, hq, hkv):
    """Live positions end in the first block of a pair (and of a KV piece)."""
    n, n_kv = 130, 901
    c = cases.with_mask(cases.prefill_case(n, hq=hq, hkv=hkv, kv_offset=n_kv - n, seed=4000 + hq,
                                           name=f"odd walk {hq}/{hkv}"), rows_mask(n, n_kv, [(100, 700)]))
    ref = poisoned(c, [*range(0, 96), *range(704, n_kv)])
    rc, out = runner.run(c)
    assert rc == 0
    check(c, ref, out)
    c = cases.prefill_case(n, hq=hq, hkv=hkv, kv_offset=n_kv - n, seed=4010 + hq, name=f"implicit {hq}/{hkv}")
    cases.with_mask(c, cases.implicit_mask(n, n_kv, 530))     # rows up to 529: positions to 659
    ref = poisoned(c, range(672, n_kv))
    rc, out = runner.run_implicit(c, vx.mask_desc(vx.MASK_CAUSAL, 0, 530))
    assert rc == 0
    check(c, ref, out)


@pytest.mark.parametrize("hq,hkv", HD128)
def test_blocks_between_the_rows_of_a_workgroup(runner, hq, hkv):
    n, n_kv = 130, 900
    c = cases.with_mask(cases.prefill_case(n, hq=hq, hkv=hkv, kv_offset=n_kv - n, seed=4100 + hq,
                                           name=f"between {hq}/{hkv}"), rows_mask(n, n_kv, [(0, 200), (600, 800)]))
    ref = poisoned(c, range(256, 576))
    rc, out = runner.run(c)
    assert rc == 0
    check(c, ref, out)


def test_hd64(runner):
    """96 heads x 4 tiles of 128 rows: the size from which hd 64 goes to this kernel."""
    n = 500
    for name, spans, bad in (("odd walk", [(100, 300)], [*range(0, 96), *range(320, n)]),
                             ("between", [(0, 90), (400, 480)], range(96, 384))):
        c = cases.with_mask(cases.encoder_case(n, 96, 64, seed=4200, name=f"hd64 {name}"), rows_mask(n, n, spans))
        ref = poisoned(c, bad)
        rc, out = runner.run(c)
        assert rc == 0
        check(c, ref, out)
