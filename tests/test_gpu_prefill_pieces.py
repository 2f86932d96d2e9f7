"""KV pieces of the grouped hd 128 prefill at the workspace's limit: the
number of pieces depends on the call's sizes alone, so calls that stand for
each other give the same bits."""
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


@pytest.mark.parametrize("hq,hkv,n,n_kv", [(4, 1, 2177, 2689), (4, 1, 1000, 3000), (8, 2, 300, 4000)])
def test_tensor_and_implicit_mask_are_cut_alike(runner, hq, hkv, n, n_kv):
    """At 2177 rows on 2689 the records of nine pieces fill the workspace to the
    bytes that a table of mask rows takes."""
    c = cases.prefill_case(n, hq=hq, hkv=hkv, kv_offset=n_kv - n, seed=5000 + n)
    rc, out = runner.run(c)
    assert rc == 0
    rc, out2 = runner.run_implicit(c, vx.mask_desc(vx.MASK_CAUSAL, 0, n_kv - n))
    assert rc == 0
    assert np.array_equal(out.view(np.uint32), out2.view(np.uint32)), float(np.abs(out - out2).max())
