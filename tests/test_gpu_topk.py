"""Router selections around the ranked top-k's bounds, against the oracle: the
most experts that tie at one probability (its candidates overflow, the
round-by-round form runs), zero probabilities, E not a multiple of 64, E of one
lane pair, k of 1 and 16, NaN; the per-layer router, the one-launch layer and the batched
tails."""
import numpy as np
import pytest

import hoard_amd as H
from hoard_amd import workloads as W

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

CASES = [(1, 1), (2, 2), (17, 16), (63, 8), (64, 16), (65, 1), (100, 10), (129, 8), (300, 16), (512, 10), (1000, 16)]


def _routers(E, n, rng):
    base = rng.standard_normal((E, n), dtype=np.float32) * 0.02
    yield "random", base
    same = base.copy()
    same[:] = base[0]
    yield "all tie", same
    half = base.copy()
    half[E // 2:] = base[E - 1]
    yield "half tie", half
    # a few logits so far up that the others' probabilities are zero
    spread = base * 1.0
    spread[rng.permutation(E)[: max(1, E // 8)]] *= 400.0
    yield "zeros", spread


@pytest.mark.parametrize("E,k", CASES, ids=lambda v: str(v))
def test_selection_matches_oracle(orc, E, k):
    from hoard_amd.runtime import MoEStage
    rng = np.random.default_rng(1000 * E + k)
    shape = W.Shape(f"topk{E}_{k}", 60, 2048, E, k, 512, 1, H.TYPE_Q4_K, H.TYPE_Q4_K, H.TYPE_Q6_K, 1)
    hl = W.make_layer(shape, 0, 0, experts=[])
    M = 34 if E % 2 else 6
    toks = np.stack([W.make_hidden(shape, 0, 0, t)[0] for t in range(M)])
    for what, router in _routers(E, shape.n_embd, rng):
        print(f"top-k E={E} k={k} {what}", flush=True)
        hl.router = np.ascontiguousarray(router, dtype=np.float32)
        st = MoEStage(shape, n_layer=1, layers={0: hl}, max_tokens=M)
        try:
            want = [orc.route(hl.router, x, E, k, 1) for x in toks]
            for t in range(3):
                sel, w = st.route(0, toks[t])
                assert np.array_equal(sel, want[t][0]), (what, t)
                assert np.allclose(w, want[t][1], rtol=1e-6, atol=1e-30)
                _, sel_l, w_l = st.layer(0, toks[t], toks[t])
                assert np.array_equal(sel_l, sel) and np.array_equal(w_l.view(np.uint32), w.view(np.uint32))
            _, sel, w = st.forward_batched(0, toks, toks)
            assert np.array_equal(sel, np.stack([v[0] for v in want])), what
            if what == "random":  # a NaN selects no expert, for its token alone
                bad = toks.copy()
                bad[1, 5] = np.nan
                assert (st.route(0, bad[1])[0] >= E).all()
                assert np.isnan(st.layer(0, bad[1], toks[1])[0]).all()
                out, sel, _ = st.forward_batched(0, bad, toks)
                assert (sel[1] >= E).all()
                assert np.isfinite(np.delete(out, 1, 0)).all()
        finally:
            st.close()
