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


def serial(logits):
    """src/profile.rs:192-213: the first value stands until one is larger, which nothing is than a NaN"""
    best = 0
    for i, v in enumerate(logits.tolist()):
        if v > logits[best]:
            best = i
    return best


@pytest.mark.parametrize("n", [70, 1030, 5000, 8192, 8193, 20000])
def test_logits_that_are_not_numbers(n):
    """As the serial scan, the same id in every element of the row: NaN beside, before and behind the maximum, in its thread and its
    wave, at the front, everywhere; infinities beside them."""
    n_in = 16400
    r = np.random.default_rng(n)
    rows = (np.arange(n) % 2048).astype(np.float16)[:, None] * np.ones((1, n_in), np.float16)
    logits, x, ids = np.zeros(n, np.float32), np.zeros(n_in, np.float32), np.zeros(1, np.uint32)
    be = ih.Hip()
    try:
        w = ih.weights(rows, ih.F16, n_in, n)
        for p in range(12):
            at = int(r.integers(n))
            logits[:] = r.standard_normal(n)
            logits[at] = np.inf if p == 3 else 9.0
            bad = {0: [0], 1: [at % 1024], 2: [at ^ 1], 3: [1, 2, n - 1], 4: r.permutation(n)[:n // 2],
                   5: np.arange(n), 6: np.arange(1, n), 7: [i for i in range(at % 64, n, 64) if i != at], 8: np.arange(0, n, 64),
                   9: [i for i in range(at % 1024, n, 1024) if i != at]}.get(p, r.permutation(n)[:1 + p])
            logits[np.asarray(bad, int) % n] = np.nan
            want = serial(logits)
            be.begin_pass(1); be.host_wrote(logits); be.scale(logits, 1.0); be.end_pass()
            be.begin_pass(1)
            assert be.L.it_hip_embed_argmax(be.h, C.addressof(w), logits.ctypes.data, n, x.ctypes.data, n_in, 5 + p) == 1
            be.end_pass(); be.host_needs(x)
            be.L.it_hip_read_tokens(be.h, 5 + p, 1, ids.ctypes.data)
            be.raise_if_error()
            assert ids[0] == want and np.array_equal(x, rows[want].astype(np.float32)), (p, at, want, ids[0])
            assert be.argmax(logits) == want
    finally:
        be.close()
