"""Reads of device values by the host: lengths around a block's share, the cells, four floats and the length that is copied instead,
into pageable memory and into page-locked memory at an address of 16 bytes and off one; every float, read after read."""
import numpy as np
import pytest
import torch

from util import rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("where", ["pageable", "locked", "locked, off 16 bytes"])
def test_every_float_arrives(where):
    import inferred_hip as ih
    be = ih.Hip(exact=True)
    try:
        for n in (1, 3, 4, 5, 1023, 1024, 1025, 2049, 8192, 65535, 65536, 65537, 262143, 262144, 262145):
            r = rng(n)
            if where == "pageable":
                x = np.zeros(n, np.float32)
            else:
                x = torch.zeros(n + 4, pin_memory=True).numpy()[1 if "off" in where else 0:][:n]
            add = np.zeros(n, np.float32)
            for turn in range(3):
                first = r.integers(-1000, 1000, n).astype(np.float32)
                x[:] = first
                add[:] = r.integers(-1000, 1000, n)
                be.drop_mirrors()
                be.begin_pass(2)
                be.add_assign(x, add)
                be.end_pass()
                be.host_needs(x)
                be.raise_if_error()
                assert np.array_equal(x, first + add), (n, turn)
    finally:
        be.take_error()
        be.close()
