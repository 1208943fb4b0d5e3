"""The on-demand layer's slot uploads by a kernel: every number of missed
records from none to n_used, 1 and 16 of them, a last use of the slots on
another stream, and a refused upload; bit-identical to the resident handle."""
import ctypes

import numpy as np
import pytest

import hoard_amd as H
from hoard_amd import workloads as W

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

Q4, Q6 = H.TYPE_Q4_K, H.TYPE_Q6_K


@pytest.mark.parametrize("k,K", [(1, 2), (3, 5), (16, 20)])
def test_on_demand_uploads_match_resident(k, K):
    from hoard_amd.runtime import MoEStage
    shape = W.Shape(f"fill_k{k}", 40 + k, 512, 24, k, 256, 1, Q4, Q4, Q6, 1)
    hl = W.make_layer(shape, 0, 0)
    full = MoEStage(shape, n_layer=1, layers={0: hl})
    pool = MoEStage(shape, n_layer=1, layers={0: hl}, pool_k=K)
    other = torch.cuda.Stream()
    seen = set()
    try:
        order = [0, 0, 1, 2, 1, 3, 4, 5, 4, 6, 7, 8]
        for i, t in enumerate(order):
            print(f"slot fill k={k} call {i}", flush=True)
            fx, res = W.make_hidden(shape, 0, 0, t)
            ref, sel, _ = full.layer(0, fx, res)
            before = pool.stats().misses
            if i % 3 == 2:  # the slots' last use on another stream
                with torch.cuda.stream(other):
                    out, sel_p, _ = pool.layer(0, fx, res)
            else:
                out, sel_p, _ = pool.layer(0, fx, res)
            seen.add(pool.stats().misses - before)
            assert np.array_equal(sel, sel_p)
            assert np.array_equal(ref.view(np.uint32), out.view(np.uint32))
        assert 0 in seen and k in seen, seen
        pool.set_option(H.OPT_FAIL_UPLOAD, 1)
        fx, res = W.make_hidden(shape, 0, 0, 20)
        fx_d, res_d, out_d = pool.dev(fx), pool.dev(res), pool.dev(res)
        p = lambda a: ctypes.c_void_p(a.data_ptr())  # noqa: E731
        rc = pool.lib.hoard_moe_layer(pool.h, 0, p(fx_d), p(res_d), p(out_d), None, None, pool.stream())
        refused = rc == H.ERR_HIP
        pool.set_option(H.OPT_FAIL_UPLOAD, 0)
        before = pool.stats().misses
        out, _, _ = pool.layer(0, fx, res)
        assert not refused or pool.stats().misses - before == k  # a refused upload forgets the layer's residency
        assert np.array_equal(out.view(np.uint32), full.layer(0, fx, res)[0].view(np.uint32))
    finally:
        full.close()
        pool.close()
