"""Work units of 4 (per-token dots), 16, 32 and 64 pairs: caller ids whose expert groups end just
before, at and after a unit's and an MFMA chunk's edge, at batches that take
each unit size (and verify-sized ones that run as units), and hiddens whose
Q8_K quants and sums are the largest there are.  The folded operands and the
fp16 sums are exact, so every token equals the single-token path bit for bit."""
import numpy as np
import pytest

from hoard_amd import workloads as W

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

EDGES = [1, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65, 129]
# tokens of units of 4 (10, 16), 16 (31, 32: as verify-sized batches), 32 and 64 pairs over 64 experts
CASES = [(s, m) for s in (W.OLMOE_Q3, W.OLMOE) for m in (10, 16, 31, 32, 66, 140, 200)]
# a shared expert's group of every token beside Q5_K routed rows; Q4_K / Q6_K rows
# (Qwen3.5 at 33 and 64 and Qwen3-Next at 102: prefill-sized on units of 4)
CASES += [(W.QWEN35, 8), (W.QWEN35, 33), (W.QWEN35, 64), (W.QWEN35, 66), (W.QWEN3_NEXT, 102), (W.QWEN35, 400), (W.QWEN3_30B, 32), (W.QWEN3_30B, 66), (W.QWEN3_30B, 200),
          (W.QWEN3_30B, 400)]


def _ids(shape, M, rng):
    """[M][k] distinct ids per token; experts 0, 1, ... have EDGES tokens each (at most M)."""
    left = [min(n, M) for n in EDGES]
    ids = np.empty((M, shape.n_used), np.int32)
    for t in range(M):
        # the edge experts with most tokens left go first, at most k of them
        want = sorted((e for e in range(len(left)) if left[e] > 0), key=lambda e: -left[e])[: shape.n_used]
        want = [e for e in want if left[e] >= M - t or rng.random() < 0.7]
        for e in want:
            left[e] -= 1
        rest = rng.permutation(np.arange(len(left), shape.n_expert))[: shape.n_used - len(want)]
        ids[t] = rng.permutation(np.concatenate([np.array(want, np.int32), rest]))
    return ids


@pytest.mark.parametrize("shape,M", CASES, ids=lambda v: v.name if hasattr(v, "name") else str(v))
def test_unit_edges_match_single_token(shape, M):
    from hoard_amd.runtime import MoEStage
    rng = np.random.default_rng(M)
    st = MoEStage(shape, n_layer=1, layers={0: W.make_layer(shape, 8, 0)}, max_tokens=M)
    try:
        fx, res = (np.stack(v) for v in zip(*(W.make_hidden(shape, 8, 0, 100 + t) for t in range(M))))
        fx[0] = 1.0  # every quant -127, every 32-element sum -4064
        fx[1] = np.where(np.arange(shape.n_embd) % 64 == 0, 3.0, -3.0)
        ids = _ids(shape, M, rng)
        w = rng.random((M, shape.n_used), dtype=np.float32) + 0.1
        print(f"units {shape.name} M={M}", flush=True)
        out = st.ffn_combine_batched(0, fx, ids, w, res)
        for t in range(M):
            o1 = st.ffn_combine(0, fx[t], ids[t], w[t], res[t])
            assert np.array_equal(o1.view(np.uint32), out[t].view(np.uint32)), t
    finally:
        st.close()
