"""Q8_0 quants of a single-token product's activation at the edges of the short arithmetic that forms them: against the CPU
oracle's, one quant a row (the weights are a unit matrix), bit for bit."""
import numpy as np
import pytest

from util import rng

pytestmark = pytest.mark.gpu

N = 1024


def unit_rows():
    rows = np.zeros((N, N // 32, 34), np.uint8)
    rows[:, :, :2] = np.frombuffer(np.float16(1).tobytes(), np.uint8)
    i = np.arange(N)
    rows[i, i // 32, 2 + i % 32] = 1
    return rows.reshape(-1)


def blocks():
    r = rng(9)
    x = r.standard_normal((N // 32, 32)).astype(np.float32)
    x[0] = np.arange(32) * 4 - 62.5                   # a step of 1: halves round away from zero
    x[0, 0] = 127
    x[1] = np.nextafter(x[0], np.float32(0))          # ... and just below them
    x[1, 0] = 127
    x[2] = 0
    x[3, 5] = np.nan                                  # counts for nothing in the largest value, becomes 0
    x[4] *= 1e-30                                     # steps that are 0, subnormal and smallest in f16
    x[5] *= 127 * 2.0 ** -24
    x[6] *= 127 * 2.0 ** -14
    x[7] *= 2.0 ** -120                               # below the range of the short reciprocal
    x[8] *= 127 * 60000 / np.abs(x[8]).max()          # the largest finite steps
    x[9] = 1e-45
    x[10, 1:] = 0
    x[11:16] *= np.float32(2.0) ** np.arange(-10, 15, 5)[:, None]
    return x.reshape(-1)


def test_quants_of_a_single_token():
    import inferred_hip as ih
    from oracle import binding as ob
    orc, hip = ob.Oracle(threads=4), ih.Hip(exact=False)
    data = unit_rows()
    W = [m.weights(data, ih.Q8_0, N, N) for m in (ih, ob)]
    B = [dict(x=blocks(), y=np.zeros(N, np.float32), res=np.zeros(N, np.float32)) for _ in range(2)]

    def block(ops, w, b):
        ops.matmul(w, b["x"], b["y"])
        ops.add_assign(b["res"], b["y"])

    try:
        for _ in range(4):
            for b in B:
                b["res"][:] = 0
            hip.begin_pass(1); hip.host_wrote(B[0]["x"]); hip.host_wrote(B[0]["res"])
            block(hip, W[0], B[0])
            hip.end_pass(); hip.host_needs(B[0]["res"]); hip.raise_if_error()
        block(orc, W[1], B[1])
        got, want = B[0]["res"], B[1]["res"]
        assert hip.graph_stats()["graph_kernels"] == 1                    # the fused product, which quantizes by itself
        assert np.array_equal(got, want), np.flatnonzero(got != want)
        assert np.count_nonzero(got) > 700
    finally:
        hip.take_error()
        hip.close()
