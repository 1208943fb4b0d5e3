"""Work units of 4 (per-token dots), 16, 32 and 64 pairs: caller ids whose expert groups end just
before, at and after a unit's and an MFMA chunk's edge, at batches that take
each cut (dots beside units of 16, dots in gate/up alone beside units of 16 and
32, units of 16 beside 32, units of 64), and
hiddens whose Q8_K quants and sums are the largest there are.  The folded
operands and the fp16 sums are exact, so every token equals the single-token
path bit for bit.  Batches whose tokens share experts cost no more than larger
ones of the kind."""
import ctypes

import numpy as np
import pytest

import hoard_amd as H
from hoard_amd import workloads as W

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

EDGES = [1, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65, 129]
# around the dots' line of 8 pairs and the units of 16 beside them
DOT_EDGES = [1, 4, 5, 7, 8, 9, 15, 16, 17, 24, 25, 32]
# over 64 experts: dots beside units of 16 (10, 16), units of 16 and 32 (31, 32: as verify-sized
# batches; 66, 140), of 64 (200)
CASES = [(s, m) for s in (W.OLMOE_Q3, W.OLMOE) for m in (10, 16, 31, 32, 66, 140, 200)]
# a shared expert's group of every token beside Q5_K routed rows; Q4_K / Q6_K rows
# (Qwen3.5 at 33 and 64 and Qwen3-Next at 102: dots in gate/up alone)
CASES += [(W.QWEN35, 8), (W.QWEN35, 33), (W.QWEN35, 64), (W.QWEN35, 66), (W.QWEN3_NEXT, 102), (W.QWEN35, 400),
          (W.QWEN3_30B, 32), (W.QWEN3_30B, 66), (W.QWEN3_30B, 200), (W.QWEN3_30B, 400)]
DOT_CASES = [(W.OLMOE_Q3, 9), (W.OLMOE_Q3, 16), (W.OLMOE, 16), (W.QWEN3_30B, 17), (W.QWEN3_30B, 32), (W.QWEN35, 25),
             (W.QWEN35, 32), (W.QWEN35, 40), (W.QWEN3_NEXT, 8), (W.QWEN3_NEXT, 32), (W.QWEN3_NEXT, 40)]


def _ids(shape, M, rng, edges):
    """[M][k] distinct ids per token; experts 0, 1, ... have `edges` tokens each (at most M)."""
    left = [min(n, M) for n in edges]
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


def _name(v):
    return v.name if hasattr(v, "name") else str(v)


@pytest.mark.parametrize("shape,M", CASES, ids=_name)
def test_unit_edges_match_single_token(shape, M):
    _check(shape, M, EDGES)


@pytest.mark.parametrize("shape,M", DOT_CASES, ids=_name)
def test_dot_unit_edges_match_single_token(shape, M):
    _check(shape, M, DOT_EDGES)


def _check(shape, M, edges):
    from hoard_amd.runtime import MoEStage
    rng = np.random.default_rng(M)
    st = MoEStage(shape, n_layer=1, layers={0: W.make_layer(shape, 8, 0)}, max_tokens=M)
    try:
        fx, res = (np.stack(v) for v in zip(*(W.make_hidden(shape, 8, 0, 100 + t) for t in range(M))))
        fx[0] = 1.0  # every quant -127, every 32-element sum -4064
        fx[1] = np.where(np.arange(shape.n_embd) % 64 == 0, 3.0, -3.0)
        ids = _ids(shape, M, rng, edges)
        w = rng.random((M, shape.n_used), dtype=np.float32) + 0.1
        print(f"units {shape.name} M={M}", flush=True)
        out = st.ffn_combine_batched(0, fx, ids, w, res)
        for t in range(M):
            o1 = st.ffn_combine(0, fx[t], ids[t], w[t], res[t])
            assert np.array_equal(o1.view(np.uint32), out[t].view(np.uint32)), t
    finally:
        st.close()


@pytest.mark.parametrize("shape,M,more", [(W.QWEN3_NEXT, 102, 128), (W.QWEN3_NEXT, 64, 128), (W.QWEN35, 64, 80)],
                         ids=_name)
def test_shared_experts_cost_no_more_than_in_a_larger_batch(shape, M, more):
    """Every token on the same experts: M tokens take at most 1.4 times what a larger batch of them takes (a cut
    chosen by the batch's mean pairs an expert took 2 to 3 times)."""
    from hoard_amd.runtime import MoEStage
    st = MoEStage(shape, n_layer=1, layers={0: W.make_layer(shape, 8, 0)}, max_tokens=more)
    try:
        ids = torch.randperm(shape.n_expert)[: shape.n_used].to(torch.int32).repeat(more, 1).cuda()
        fx, res, out = (torch.randn(more, shape.n_embd, device="cuda") for _ in range(3))
        w = torch.rand(more, shape.n_used, device="cuda")
        p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731

        def us(m):
            times = []
            for _ in range(9):
                a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                a.record()
                for _ in range(20):
                    H.check(st.lib.hoard_moe_ffn_combine_batched(st.h, 0, m, p(fx), p(ids), p(w), p(res), p(out),
                                                                 st.stream()))
                b.record()
                torch.cuda.synchronize()
                times.append(a.elapsed_time(b) / 20 * 1000)
            return sorted(times)[4]

        print(f"shared experts {shape.name} M={M} and {more}", flush=True)
        us(more)
        few, many = us(M), us(more)
        print(f"   {few:.1f} and {many:.1f} us", flush=True)
        assert few <= 1.4 * many, (few, many)
    finally:
        st.close()
