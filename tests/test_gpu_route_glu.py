"""Exact mode's routed FFN: with few experts the norm, the router and the shared gate formed by every block of the expert
gate / up launch, on both sides of the sizes that takes, else the picks by a whole block, against the CPU oracle bit for bit."""
import numpy as np
import pytest

from test_gpu_fused_fast import Both, bufs
from util import q8_0_weights, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nd,ne,ff,sff,nu,kernels", [
    (512, 16, 256, 256, 4, 2),
    (32, 1, 32, 32, 1, 2),          # the smallest: a unit a row, one expert
    (1024, 31, 64, 96, 16, 2),      # 32 rows of 32 units: four a thread; the most picks
    (1024, 32, 64, 96, 8, 3),       # one row more
    (96, 63, 160, 32, 3, 2),        # 64 rows: all lanes of the wave that folds them
    (96, 64, 160, 32, 3, 3),
    (992, 8, 1008 + 16, 32, 3, 2),  # 64 x 4 blocks: one a CU; threads without a quad
    (992, 8, 1024 + 32, 32, 3, 3),
    (1056, 8, 64, 64, 2, 3),        # more than a quad a thread
    (544, 512, 32, 32, 10, 3),      # the picks by the router's last block, an expert a thread
    (544, 513, 32, 32, 16, 3),      # and more
    (1056, 1040, 32, 32, 10, 3),    # (the last pass: equal keys, all of them candidates)
])
def test_routed_block(nd, ne, ff, sff, nu, kernels):
    import inferred_hip as ih
    from oracle import binding as ob
    hip = ih.Hip(exact=True)
    pair = Both(hip, ob.Oracle(threads=8))
    orc = pair.orc
    r = rng(nd + ne + ff)
    router, sh_inp = pair.q8(r, ne, nd, 3.0), pair.q8(r, 1, nd, 1.0)
    ones = np.ones(ne, np.float32)
    ew = lambda n_out, n_in: pair.e(q8_0_weights(orc, r, ne * n_out, n_in, std=2.0 / np.sqrt(n_in)), ih.Q8_0, n_in, n_out, ne, ones)
    gate, up, down = ew(ff, nd), ew(ff, nd), ew(nd, ff)
    sg, su, sd = pair.q8(r, sff, nd, 1.5), pair.q8(r, sff, nd, 1.5), pair.q8(r, nd, sff, 2.0)
    norm_w = (0.5 + r.random(nd)).astype(np.float32)
    B = bufs(x=nd, normed=nd, e_in=nd, router=ne, logit=1, g_all=nu * ff, u_all=nu * ff, o_all=nu * nd, e_gate=sff, e_up=sff,
             e_out=nd, ffn_out=nd)

    def block(ops, i, b):
        W = lambda t: t[i]
        ops.rms_norm(b["x"], norm_w, 1e-6, b["normed"])
        ops.gather_chunks(b["normed"], nd, nd, 0, b["e_in"])
        ops.matmul_pair(W(router), W(sh_inp), b["e_in"], b["router"], b["logit"])
        ops.softmax(b["router"], ne)
        route = ops.route(b["router"], ne, nu)
        picks = (route,) if i == 0 else (route[0], nu)
        ops.moe_glu(W(gate), W(up), *picks, b["e_in"], b["g_all"], b["u_all"])
        ops.matmul_experts(W(down), *picks, b["g_all"], b["o_all"])
        ops.matmul(W(sg), b["e_in"], b["e_gate"]); ops.matmul(W(su), b["e_in"], b["e_up"])
        ops.silu_mul(b["e_gate"], b["e_up"])
        ops.matmul(W(sd), b["e_gate"], b["e_out"])
        ops.moe_finish(b["ffn_out"], 0, nd, b["o_all"], *((route,) if i == 0 else (route[1], nu)), b["e_out"], b["logit"], 0)
        ops.add_assign(b["x"], b["ffn_out"])

    try:
        for p in range(6):                  # two op by op, one recorded, three replayed; other picks in each
            x0 = rng(700 + p).standard_normal(nd).astype(np.float32) * np.float32(0.0 if p == 5 else 1.0)   # (the last: equal logits)
            for b in B:
                b["x"][:] = x0
            hip.begin_pass(1); hip.host_wrote(B[0]["x"]); block(hip, 0, B[0]); hip.end_pass()
            for name in ("x", "normed", "e_in", "logit"):
                hip.host_needs(B[0][name])
            hip.raise_if_error()
            block(orc, 1, B[1])
            for name in ("x", "normed", "e_in", "logit"):
                assert np.array_equal(B[0][name].view(np.uint32), B[1][name].view(np.uint32)), (p, name)
        g = hip.graph_stats()
        assert g["captures"] == 1 and g["replays"] == 4 and g["graph_kernels"] == kernels, g
    finally:
        hip.take_error()
        hip.close()
