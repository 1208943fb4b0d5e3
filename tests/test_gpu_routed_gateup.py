"""A small router formed by the gate/up launch: the separate router launch's
selection, weights and output bit for bit, around the LDS bound of the rule
(the last expert count inside it and the first outside), with odd expert
counts, more experts than half-waves, a shared expert, ties, NaN and an
activation that is only 4-byte aligned."""
import ctypes

import numpy as np
import pytest

import hoard_amd as H
from hoard_amd import workloads as W

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

Q3, Q4, Q5, Q6 = H.TYPE_Q3_K, H.TYPE_Q4_K, H.TYPE_Q5_K, H.TYPE_Q6_K


def _shape(n, E, k, ff=256, gate=Q4, up=Q4, down=Q6, sh=0):
    return W.Shape(f"rg{n}_{E}_{k}", 70, n, E, k, ff, 1, gate, up, down, 1, n_ff_shexp=sh, sh_gate_type=gate,
                   sh_up_type=up, sh_down_type=down)


# Inside and outside each line of the rule: 32 experts, 4096 rows of gate over
# the units, 61440 bytes for (E + 1) n + E floats and n / 256 blocks of 304 bytes
CASES = [_shape(256, 32, 16), _shape(256, 33, 16), _shape(256, 19, 3), _shape(512, 27, 9), _shape(512, 29, 9),
         _shape(1024, 8, 2, 512, Q4, Q4, Q4), _shape(1024, 13, 1, 512, Q3, Q3, Q5), _shape(1024, 14, 4),
         _shape(2304, 4, 4, 512, Q5, Q6, Q6, sh=768), _shape(2304, 4, 3, 1024, Q5, Q5, Q6, sh=1024),
         _shape(2304, 4, 4, 1024, Q5, Q6, Q6, sh=256), _shape(4096, 2, 2, 2048, Q6, Q6, Q6), _shape(6912, 1, 1)]


@pytest.mark.parametrize("shape", CASES, ids=lambda s: s.name)
def test_routed_gateup_matches_router_launch(orc, shape):
    from hoard_amd.runtime import MoEStage
    hl = W.make_layer(shape, 0, 0)
    if shape.n_expert > 4:
        hl.router[shape.n_embd:2 * shape.n_embd] = hl.router[:shape.n_embd]  # two experts tie
    st = MoEStage(shape, n_layer=1, layers={0: hl})
    n, k = shape.n_embd, shape.n_used
    bits = lambda a: np.asarray(a).view(np.uint32)  # noqa: E731
    try:
        for t in range(3):
            print(f"routed gate/up {shape.name} token {t}", flush=True)
            fx, res = W.make_hidden(shape, 0, 0, t)
            if t == 2:
                fx[n // 2] = np.nan
            out, sel, w = st.layer(0, fx, res)
            sel_r, w_r = st.route(0, fx)
            assert np.array_equal(sel, sel_r) and np.array_equal(bits(w), bits(w_r))
            if t == 2:
                assert np.isnan(out).all()
                continue
            assert np.array_equal(bits(out), bits(st.ffn_combine(0, fx, sel_r, w_r, res)))
            sel_o, _, _ = orc.route(hl.router, fx, shape.n_expert, k, 1)
            assert np.array_equal(sel, sel_o)
            buf = torch.zeros(3, n + 4, device="cuda")
            x, r, y = buf[0, 1:n + 1], buf[1, 2:n + 2], buf[2, 3:n + 3]
            x.copy_(torch.from_numpy(fx))
            r.copy_(torch.from_numpy(res))
            p = lambda a: ctypes.c_void_p(a.data_ptr())  # noqa: E731
            H.check(st.lib.hoard_moe_layer(st.h, 0, p(x), p(r), p(y), None, None, st.stream()))
            torch.cuda.synchronize()
            assert np.array_equal(bits(y.cpu().numpy()), bits(out))
    finally:
        st.close()
