"""Appended rows and rotary embedding on every route of a prefill or batched
decode call: query rows rotated ahead by the append launch or by the kernel
that reads them, mask intervals found in the append launch, with each of the
prefill kernels; a decode step's new row as a tile of its own, under ranges
found by a pre-pass or a scan. Outputs against the exact float64 reference
(and, rotated, against the host-rotated call), caches byte for byte, as in
test_gpu_parity.py, whose helpers and bars these are: 2e-3 absolute, 1e-2
relative."""
import numpy as np
import pytest

import cases
from oracle import oracle
from test_gpu_parity import _append_rows, _check_append, _rope_check

pytestmark = pytest.mark.gpu

# which kernel takes hd 128 beyond n_kv 512, and who rotates
ROUTES = {"grouped": dict(VXFA_PREFILL_GROUP=1), "grouped, rotating": dict(VXFA_PREFILL_GROUP=1, VXFA_ROPE_Q=0),
          "general": dict(VXFA_PREFILL_GROUP=0), "general, rotating": dict(VXFA_PREFILL_GROUP=0, VXFA_ROPE_Q=0)}


@pytest.fixture(scope="module", params=ROUTES, ids=[r.replace(", ", "-") for r in ROUTES])
def runner(request):
    import gpu_util
    r = gpu_util.Runner(**ROUTES[request.param])
    yield r
    r.close()


def prefill(n, n_kv, kind="causal", batch=1, hq=8, hkv=2, hd=128, seed=6000):
    """n new rows at the end of n_kv, in `batch` sequences with a mask batch each."""
    c = cases.decode_case(n_kv, hq=hq, hkv=hkv, hd=hd, batch=batch, seed=seed + n + n_kv,
                          name=f"{kind} {n} of {n_kv} x{batch} {hq}/{hkv} hd{hd}")
    rng = np.random.default_rng(seed + 1)
    c.bufs.pop("q"); c.views.pop("q")
    c.add("q", "q", cases.normal(rng, (batch, n, hq, hd)), oracle.F32, *cases._batched_q(n, hq, hd, 4, batch))
    if kind != "none":
        ms = []
        for b in range(batch):
            m = cases.implicit_mask(n, n_kv, n_kv - n, 100 if kind == "window" else 0)
            if kind == "holes":
                m = np.where(rng.random(m.shape) < 0.3, cases.NEG_INF_F16, m).astype(np.uint16)
                m[:, -1] = 0
            if b == 1:
                m[:, :50] = cases.NEG_INF_F16
            ms.append(m)
        c.add("mask", "mask", np.stack(ms), oracle.F16, *cases.views.mask(n_kv, n, 1, batch))
    return c


def new_rows(c, n, seed):
    b, _, ne, _, _ = c.views["k"]
    return _append_rows(np.random.default_rng(seed), ne[3], n, ne[2] * ne[0])


# n_kv 513 and up: grouped or general; 300: the short masked kernel; hd 64: the
# pipelined kernel, or the general one
PREFILL = [("causal", 70, 600, 1, 8, 2, 128), ("window", 70, 600, 2, 8, 2, 128), ("holes", 40, 577, 2, 8, 2, 128),
           ("none", 65, 530, 1, 4, 4, 128), ("causal", 2, 1000, 1, 32, 8, 128), ("causal", 40, 300, 2, 8, 2, 128),
           ("causal", 40, 150, 2, 4, 2, 64), ("holes", 33, 200, 1, 4, 4, 64)]


@pytest.mark.parametrize("kind,n,n_kv,batch,hq,hkv,hd", PREFILL)
def test_prefill_rope(runner, kind, n, n_kv, batch, hq, hkv, hd):
    c = prefill(n, n_kv, kind, batch, hq, hkv, hd)
    k, v = new_rows(c, n, 6100 + n)
    pos = [n_kv - n + i + 7 * b for b in range(batch) for i in range(n)]
    _rope_check(runner, c, k, v, pos, hd if kind != "window" else 96, 1.0e6)


@pytest.mark.parametrize("kind,n,n_kv,batch,hq,hkv,hd", PREFILL)
def test_prefill_append(runner, kind, n, n_kv, batch, hq, hkv, hd):
    c = prefill(n, n_kv, kind, batch, hq, hkv, hd)
    k, v = new_rows(c, n, 6200 + n)
    a = _check_append(runner, c, k, v, fused=True)
    b = _check_append(runner, c, k, v, fused=False)
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("kind,n,n_kv,batch,hq,hkv", [("causal", 100, 654, 1, 32, 8), ("causal", 200, 929, 1, 32, 8),
                                                      ("window", 39, 593, 3, 32, 8), ("none", 383, 1112, 1, 32, 8)])
def test_prefill_append_own_route(kind, n, n_kv, batch, hq, hkv):
    """Near the line between the general and the grouped kernel, as called by
    default: appending within the call gives the bits of appending before it."""
    import gpu_util
    r = gpu_util.Runner()
    try:
        c = prefill(n, n_kv, kind, batch, hq, hkv)
        k, v = new_rows(c, n, 6300 + n)
        a = _check_append(r, c, k, v, fused=True)
        b = _check_append(r, c, k, v, fused=False)
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    finally:
        r.close()


def test_prefill_rope_hd64_long_cache():
    """Few rows on a long cache go to the general kernel, the host-rotated append
    call that they are compared with to the pipelined one, whose roundings of P
    differ by more than the helper's bar (2.8e-4): both on the general one here."""
    import gpu_util
    r = gpu_util.Runner(VXFA_PREFILL_PP=0)
    try:
        c = prefill(5, 1100, "causal", 1, 4, 4, 64)
        k, v = new_rows(c, 5, 6105)
        _rope_check(r, c, k, v, list(range(1095, 1100)), 64, 1.0e6)
    finally:
        r.close()


def test_fewer_new_rows_than_queries(runner):
    c = prefill(70, 600)
    k, v = new_rows(c, 3, 6300)
    _check_append(runner, c, k, v)


def streams(lens, cap, hq=32, hkv=8, hd=128):
    """Decode streams of these lengths (0: nothing live); the second row is a bias."""
    c = cases.decode_case(cap, hq=hq, hkv=hkv, hd=hd, batch=len(lens), seed=6400 + cap, name=f"streams {lens} hd{hd}")
    m = np.zeros((len(lens), 1, cap), dtype=np.uint16)
    m[1] = np.random.default_rng(64).normal(0, 1, cap).astype(np.float16).view(np.uint16)
    for b, n in enumerate(lens):
        m[b, 0, n:] = cases.NEG_INF_F16
    c.add("mask", "mask", m, oracle.F16, *cases.views.mask(cap, 1, 1, len(lens)))
    return c


@pytest.fixture(scope="module", params=[1, 0], ids=["pre-pass", "scan"])
def decoder(request):
    import gpu_util
    r = gpu_util.Runner(VXFA_DECODE_ROWS=request.param)
    yield r
    r.close()


LENS = [((600, 600, 0, 599, 100), 600), ((1, 17, 0, 16), 17), ((700, 64, 0, 65, 129, 1), 700)]


@pytest.mark.parametrize("hq,hkv,hd", [(32, 8, 128), (8, 8, 64), (4, 2, 128)])
@pytest.mark.parametrize("lens,cap", LENS)
def test_decode_streams_append(decoder, lens, cap, hq, hkv, hd):
    c = streams(lens, cap, hq, hkv, hd)
    out = _check_append(decoder, c, *new_rows(c, 1, 6500))
    assert not out[lens.index(0)].any()


@pytest.mark.parametrize("hq,hkv,hd", [(32, 8, 128), (8, 4, 64)])
@pytest.mark.parametrize("lens,cap", LENS)
def test_decode_streams_rope(decoder, lens, cap, hq, hkv, hd):
    c = streams(lens, cap, hq, hkv, hd)
    _rope_check(decoder, c, *new_rows(c, 1, 6600), [cap - 1 + b for b in range(len(lens))], hd, 1.0e6)


# spans of 16-position tiles, whose new row is loaded ahead of the loop: its turn
# falls to every wavefront, to a split of its own, alone
@pytest.mark.parametrize("n_kv", [2, 16, 17, 49, 65, 97, 113, 129, 435, 1025])
def test_decode_rope_turns(decoder, n_kv):
    c = cases.decode_case(n_kv, seed=6700 + n_kv)
    _rope_check(decoder, c, *new_rows(c, 1, 6700), [n_kv - 1], 128, 1.0e6)
