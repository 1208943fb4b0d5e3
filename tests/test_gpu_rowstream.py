"""The single-token kernels of any shape (router, gate/up, down + combine) at
block counts around the streams' depth of 4 and the router's 4096-element
chunk, every quant type and mixtures of them, units past the waves of a
workgroup, activations that are only 4-byte aligned; against the oracle,
whose integer sums and fp32 order they keep."""
import ctypes

import numpy as np
import pytest

import hoard_amd as H
import parity
from hoard_amd import workloads as W

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

Q3, Q4, Q5, Q6 = H.TYPE_Q3_K, H.TYPE_Q4_K, H.TYPE_Q5_K, H.TYPE_Q6_K


def _shape(name, n, E, k, ff, gate, up, down, ff_sh=0, sh=(Q4, Q4, Q6)):
    return W.Shape(name, 20, n, E, k, ff, 1, gate, up, down, 1, n_ff_shexp=ff_sh, sh_gate_type=sh[0],
                   sh_up_type=sh[1], sh_down_type=sh[2])


CASES = [
    _shape("one_block_q3", 256, 5, 3, 256, Q3, Q3, Q3),
    _shape("n3_ff5_q4_q5", 768, 6, 2, 1280, Q4, Q4, Q5),
    _shape("n5_ff3_q5_q6", 1280, 9, 4, 768, Q5, Q5, Q6),
    _shape("n7_ff9_q6", 1792, 7, 5, 2304, Q6, Q6, Q6),
    _shape("n17_past_the_router_chunk", 4352, 11, 3, 256, Q4, Q4, Q4),
    _shape("mixed_types_shared", 512, 8, 2, 512, Q4, Q6, Q3, 1024, (Q5, Q3, Q4)),
    _shape("sixteen_experts_and_a_shared_one", 1024, 33, 16, 256, Q4, Q4, Q6, 768),
    # enough rows for the wider gate/up workgroups and two or four down waves a unit
    _shape("wide_k8", 4096, 9, 8, 1024, Q3, Q3, Q5),
    _shape("wide_k4", 8192, 5, 4, 512, Q4, Q4, Q6),
]


@pytest.mark.parametrize("shape", CASES, ids=lambda s: s.name)
def test_any_shape_matches_oracle(orc, shape):
    from hoard_amd.runtime import MoEStage
    hl = W.make_layer(shape, 0, 0)
    st = MoEStage(shape, n_layer=1, layers={0: hl})
    try:
        st.set_option(H.OPT_LAYER_KERNELS, 0)
        for t in range(2):
            print(f"row streams {shape.name} token {t}", flush=True)
            fx, res = W.make_hidden(shape, 0, 0, t)
            ref, sel_o, w_o = orc.moe_layer(hl, fx, res)
            out, sel, w = st.layer(0, fx, res)
            assert np.array_equal(sel, sel_o)
            assert np.allclose(w, w_o, rtol=1e-6, atol=0)
            m = parity.assert_parity(out, ref, f"{shape.name} token {t}")
            # fp32 sums in the oracle's order: what differs is expf's last bit
            assert m["max_rel"] < 1e-5, m
        # activations on 4-byte boundaries give the same bits
        n = shape.n_embd
        buf = torch.zeros(3, n + 4, device="cuda")
        fx_d, res_d, out_d = buf[0, 1:n + 1], buf[1, 3:n + 3], buf[2, 1:n + 1]
        fx_d.copy_(torch.from_numpy(fx))
        res_d.copy_(torch.from_numpy(res))
        p = lambda a: ctypes.c_void_p(a.data_ptr())  # noqa: E731
        H.check(st.lib.hoard_moe_layer(st.h, 0, p(fx_d), p(res_d), p(out_d), None, None, st.stream()))
        torch.cuda.synchronize()
        assert np.array_equal(out_d.cpu().numpy().view(np.uint32), out.view(np.uint32))
        # the residual's rms_norm formed by the router kernel
        y = st.decode(res, 0, 1, W.RMS_EPS)
        ref, _, _ = orc.moe_layer(hl, orc.rms_norm(res, W.RMS_EPS), res)
        parity.assert_parity(y, ref, f"{shape.name} decode")
        # an id out of range poisons the token
        ids = sel.copy()
        ids[-1] = shape.n_expert
        assert np.isnan(st.ffn_combine(0, fx, ids, w, res)).all()
    finally:
        st.close()
