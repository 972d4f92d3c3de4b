"""The routed FFN of a single-token pass on both sides of the shapes that its fused kernels take, against the CPU oracle: what they do
not take is issued op by op."""
import numpy as np
import pytest

from test_gpu_fused_fast import Both, bufs
from util import close, q8_0_weights, rng, worst

pytestmark = pytest.mark.gpu
NE = 16


@pytest.mark.parametrize("exact,nd,ff,sff,nu,fused", [
    (False, 512, 256, 256, 4, True),       # both fast kernels
    (False, 512, 768, 512, 4, True),       # the down product by the kernel that keeps the CPU path's order
    (False, 768, 256, 256, 4, False),      # no fast gate / up kernel, which makes the picks
    (False, 2560, 64, 64, 4, False),
    (False, 512, 256, 2112, 4, False),     # a row of the shared down product is more than a wave takes at once
    (True, 512, 256, 2048, 4, True),
    (True, 512, 256, 2112, 4, False),
    (True, 512, 1024, 1024, 10, True),     # 11,264 intermediates: staged in LDS
    (True, 512, 3840, 1024, 8, True),      # 31,744: all of it
    (True, 512, 4096, 512, 8, False),
    (True, 8192, 64, 64, 4, True),         # a gate / up row is 256 units
    (True, 8224, 64, 64, 4, False),
])
def test_ffn_block(exact, nd, ff, sff, nu, fused):
    import inferred_hip as ih
    from oracle import binding as ob
    hip = ih.Hip(exact=exact)
    pair = Both(hip, ob.Oracle(threads=8))
    orc = pair.orc
    r = rng(nd + ff + sff)
    router, sh_inp = pair.q8(r, NE, nd, 3.0), pair.q8(r, 1, nd, 1.0)
    ones = np.ones(NE, np.float32)
    ew = lambda n_out, n_in: pair.e(q8_0_weights(orc, r, NE * n_out, n_in, std=2.0 / np.sqrt(n_in)), ih.Q8_0, n_in, n_out, NE, ones)
    gate, up, down = ew(ff, nd), ew(ff, nd), ew(nd, ff)
    sg, su, sd = pair.q8(r, sff, nd, 1.5), pair.q8(r, sff, nd, 1.5), pair.q8(r, nd, sff, 2.0)
    norm_w = (0.5 + r.random(nd)).astype(np.float32)
    B = bufs(x=nd, normed=nd, e_in=nd, router=NE, logit=1, g_all=nu * ff, u_all=nu * ff, o_all=nu * nd, e_gate=sff, e_up=sff,
             e_out=nd, ffn_out=nd)

    def block(ops, i, b):
        W = lambda t: t[i]
        ops.rms_norm(b["x"], norm_w, 1e-6, b["normed"])
        ops.gather_chunks(b["normed"], nd, nd, 0, b["e_in"])
        ops.matmul_pair(W(router), W(sh_inp), b["e_in"], b["router"], b["logit"])
        ops.softmax(b["router"], NE)
        route = ops.route(b["router"], NE, nu)
        picks = (route,) if i == 0 else (route[0], nu)
        ops.moe_glu(W(gate), W(up), *picks, b["e_in"], b["g_all"], b["u_all"])
        ops.matmul_experts(W(down), *picks, b["g_all"], b["o_all"])
        ops.matmul(W(sg), b["e_in"], b["e_gate"]); ops.matmul(W(su), b["e_in"], b["e_up"])
        ops.silu_mul(b["e_gate"], b["e_up"])
        ops.matmul(W(sd), b["e_gate"], b["e_out"])
        ops.moe_finish(b["ffn_out"], 0, nd, b["o_all"], *((route,) if i == 0 else (route[1], nu)), b["e_out"], b["logit"], 0)
        ops.add_assign(b["x"], b["ffn_out"])

    try:
        for p in range(5):                  # two op by op, one recorded, two replayed; other picks in each
            x0 = rng(900 + p).standard_normal(nd).astype(np.float32)
            for b in B:
                b["x"][:] = x0
            hip.begin_pass(1); hip.host_wrote(B[0]["x"]); block(hip, 0, B[0]); hip.end_pass()
            hip.host_needs(B[0]["x"]); hip.raise_if_error()
            block(orc, 1, B[1])
            got, want = B[0]["x"], B[1]["x"]
            if exact:
                assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), p
            else:   # (a last bit of an intermediate can move a step of its Q8_0 form, 1e-3 of the sum)
                assert close(got - x0, want - x0, 1e-2), (p, worst(got - x0, want - x0))
        g = hip.graph_stats()
        assert g["captures"] == 1 and g["replays"] == 3 and (g["graph_kernels"] == 3) == fused, g
    finally:
        hip.take_error()
        hip.close()
