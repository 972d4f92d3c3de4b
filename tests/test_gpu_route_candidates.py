"""The ten largest of 512 router logits where the selection has to look twice: ties within and across half waves, every logit the
same, all the large ones in one half wave, probabilities that are zero but for three.  The layer chain (a token) and the two-launch
FFN of a short batch against the oracle's picks, exactly: equal rows of the router give equal logits, and equal logits go to the
lower expert."""
import numpy as np
import pytest

from test_gpu_chain import Layers, make_pair, hip_pass, ND, NE, NU
from test_gpu_small_ffn import buffers, ffn_batch
from util import rng

pytestmark = pytest.mark.gpu


def router_rows(kind):
    r = rng(5)
    w = r.standard_normal((NE, ND)).astype(np.float32) * np.float32(3.0 / np.sqrt(ND))
    if kind == "zeros":
        w[:] = 0.0
    elif kind == "eightfold":
        w[:] = w[np.arange(NE) % 64]
    elif kind == "neighbours":
        w[:] = w[np.arange(NE) // 16]
    elif kind == "one half wave":
        w[:96] = 0.0
        w[128:] = 0.0
    elif kind == "three":          # one logit of the three, another of all the others, thousands apart
        w[:] = w[0] * 1e5
        w[[7, 300, 511]] = -w[0]
    return w


@pytest.mark.parametrize("kind", ["zeros", "eightfold", "neighbours", "one half wave", "three"])
def test_ties_and_zero_probabilities(kind):
    import inferred_hip as ih
    pair = make_pair()
    hip, orc = pair.hip, pair.orc
    try:
        layers = Layers(pair, 1, "nvfp4_scaled", small_f32=True)
        d = layers.L[0]
        w = router_rows(kind)
        d["router"] = pair.w(w.reshape(-1).view(np.uint8), ih.F32, ND, NE)
        before = np.zeros(NE, np.int64)

        def same_picks(picked, what):
            nonlocal before
            counts = hip.expert_counts(layers.gate_raw, NE).astype(np.int64)
            want = np.zeros(NE, np.int64)
            np.add.at(want, np.asarray(picked).astype(np.int64).reshape(-1), 1)
            assert np.array_equal(counts - before, want), (kind, what, np.flatnonzero(counts - before != want))
            before = counts

        B = layers.buffers()
        for p in range(5):            # the first passes op by op, the others the chain
            x0 = rng(900 + p).standard_normal(ND).astype(np.float32)
            hip_pass(hip, layers, B[0], x0)
            B[1]["x"][:] = x0
            picked = layers.run(orc, 1, B[1], False)
            same_picks(picked, p)
            for name in ("ssm", "conv_state"):
                B[1]["layers"][0][name][:] = B[0]["layers"][0][name]
        assert hip.chain_stats()["chains"] == 1
        for n in (2, 9, 32):
            S = buffers(n)
            for rep in range(2):      # the first pass of a size sizes the mirrors
                x0 = rng(40 * n + rep).standard_normal(n * ND).astype(np.float32)
                S[0]["x"][:] = x0
                hip.begin_pass(n); hip.host_wrote(S[0]["x"])
                ffn_batch(layers, hip, 0, d, S[0], S[0]["x"], n, True)
                hip.end_pass(); hip.host_needs(S[0]["x"]); hip.raise_if_error()
                S[1]["x"][:] = x0
                same_picks(ffn_batch(layers, orc, 1, d, S[1], S[1]["x"], n, False), (n, rep))
    finally:
        err = hip.take_error()
        hip.close()
    assert err is None, err
