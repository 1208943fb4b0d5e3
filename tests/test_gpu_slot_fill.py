"""The on-demand layer's slot uploads by a kernel: every number of missed
records from none to n_used, 1 and 16 of them, calls on another stream, a last
use of the slots that is still to come on another stream, and a refused upload;
bit-identical to the resident handle."""
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


def _layer(st, fx, res, out):
    p = lambda a: ctypes.c_void_p(a.data_ptr())  # noqa: E731
    return st.lib.hoard_moe_layer(st.h, 0, p(fx), p(res), p(out), None, None, st.stream())


def _counts(st):
    s = st.stats()
    return s.reqs, s.hits, s.misses, s.bytes_h2d


@pytest.mark.parametrize("k,K,refused", [(1, 2, 1), (3, 5, 2), (16, 20, 16)])
def test_refused_upload_leaves_nothing_behind(k, K, refused):
    """The refused-th of a call's missed records is refused: the call returns the error, takes the hook, counts no
    request, hit, miss or byte (nothing was issued), and forgets the layer's residency, so that the next call
    uploads every expert again."""
    from hoard_amd.runtime import MoEStage
    shape = W.Shape(f"refuse_k{k}", 40 + k, 512, 40, k, 256, 1, Q4, Q4, Q6, 1)
    hl = W.make_layer(shape, 0, 0)
    full = MoEStage(shape, n_layer=1, layers={0: hl})
    pool = MoEStage(shape, n_layer=1, layers={0: hl}, pool_k=K)
    try:
        toks = [W.make_hidden(shape, 0, 0, t) for t in range(40)]
        sels = [set(full.route(0, fx)[0].tolist()) for fx, _ in toks]
        for first in (None, 0):  # an empty pool, and one that holds another token's experts
            if first is not None:
                pool.set_layer(0, hl)  # empties the pool
                pool.layer(0, *toks[first])
            held = sels[first] if first is not None else set()
            t = next(i for i in range(1, 40) if len(sels[i] - held) >= min(refused, 3))
            missed = len(sels[t] - held)
            print(f"refused upload k={k}: token {t}, {missed} missed", flush=True)
            fx, res = (pool.dev(v) for v in toks[t])
            out = torch.empty_like(res)
            before = _counts(pool)
            pool.set_option(H.OPT_FAIL_UPLOAD, min(refused, missed))
            assert _layer(pool, fx, res, out) == H.ERR_HIP
            assert pool.get_option(H.OPT_FAIL_UPLOAD) == 0
            assert _counts(pool) == before
            got, _, _ = pool.layer(0, *toks[t])
            after = _counts(pool)
            assert after[0] - before[0] == k and after[1] == before[1] and after[2] - before[2] == k
            assert (after[3] - before[3]) % k == 0 and after[3] > before[3]
            assert np.array_equal(got.view(np.uint32), full.layer(0, *toks[t])[0].view(np.uint32))
    finally:
        full.close()
        pool.close()


def test_uploads_wait_for_a_last_use_on_another_stream():
    """Slots ensured for one token, whose FFN on stream A is queued behind tens of milliseconds of other work; a layer
    call on stream B then evicts them.  Its uploads wait for A's FFN: both outputs are the resident handle's."""
    from hoard_amd.runtime import MoEStage
    k = 4
    shape = W.Shape("fill_streams", 60, 512, 24, k, 256, 1, Q4, Q4, Q6, 1)
    hl = W.make_layer(shape, 0, 0)
    full = MoEStage(shape, n_layer=1, layers={0: hl})
    pool = MoEStage(shape, n_layer=1, layers={0: hl}, pool_k=k)  # every miss evicts
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    try:
        toks = [W.make_hidden(shape, 0, 0, t) for t in range(12)]
        routed = [full.route(0, fx) for fx, _ in toks]
        second = next(i for i in range(1, 12) if not set(routed[i][0]) & set(routed[0][0]))
        want = [full.layer(0, *toks[i])[0] for i in (0, second)]
        (fx0, res0), (fx1, res1) = ([pool.dev(v) for v in toks[i]] for i in (0, second))
        w0 = pool.dev(routed[0][1])
        out0, out1 = torch.empty_like(res0), torch.empty_like(res1)
        busy = torch.randn(8192, 8192, device="cuda")
        torch.mm(busy, busy)  # the library's own set-up
        for rnd in range(2):
            torch.cuda.synchronize()
            print(f"last use on another stream, round {rnd}", flush=True)
            with torch.cuda.stream(a):
                _, slots = pool.pool_ensure(0, routed[0][0])
                for _ in range(4):
                    busy2 = torch.mm(busy, busy)
                pool.ffn_combine_dev(0, fx0, slots, w0, res0, out0)
                used = torch.cuda.Event()
                used.record()
            with torch.cuda.stream(b):
                H.check(_layer(pool, fx1, res1, out1))
            late = not used.query()  # A's FFN was still to come when B's call returned
            torch.cuda.synchronize()
            del busy2
            for got, ref in zip((out0, out1), want):
                assert np.array_equal(got.cpu().numpy().view(np.uint32), ref.view(np.uint32))
            assert late, "stream A was idle before the call on stream B: nothing was tested"
    finally:
        full.close()
        pool.close()
