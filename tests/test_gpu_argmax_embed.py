"""The arg-max of logits on the device and the embedding row of its result, on both sides of the vocabulary that one launch
takes: the first of equal maxima (/root/reference src/profile.rs:192-213), its row as the host reads it."""
import ctypes as C

import numpy as np
import pytest

import inferred_hip as ih

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_in", [8, 100, 16392])          # (a block's threads take 8,192 elements of the row at once)
@pytest.mark.parametrize("n", [1, 63, 1024, 1025, 8191, 8192, 8193])
def test_first_maximum_and_its_row(n, n_in):
    r = np.random.default_rng(n + n_in)
    rows = r.standard_normal((n, n_in)).astype(np.float16)
    logits, x, ids = np.zeros(n, np.float32), np.zeros(n_in, np.float32), np.zeros(1, np.uint32)
    be = ih.Hip()
    try:
        w = ih.weights(rows, ih.F16, n_in, n)
        for p, at in enumerate(sorted({0, 1, n // 2, n - 1023, n - 1, n - 2} & set(range(n)))):
            logits[:] = -np.abs(r.standard_normal(n)) - 1
            logits[at] = logits[n - 1] = logits[(at + n) // 2] = -0.25       # equal ones behind it
            if p == 1:
                logits[:] = -np.inf                                          # all of them
            want = int(np.argmax(logits))
            be.begin_pass(1); be.host_wrote(logits); be.scale(logits, 1.0); be.end_pass()
            be.begin_pass(1)
            assert be.L.it_hip_embed_argmax(be.h, C.addressof(w), logits.ctypes.data, n, x.ctypes.data, n_in, 5 + p) == 1
            be.end_pass(); be.host_needs(x)
            be.L.it_hip_read_tokens(be.h, 5 + p, 1, ids.ctypes.data)
            be.raise_if_error()
            assert ids[0] == want and np.array_equal(x, rows[want].astype(np.float32)), (p, at)
    finally:
        be.close()
