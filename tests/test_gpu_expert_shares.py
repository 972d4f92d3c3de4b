"""The 16-pair expert tiles whose blocks share all tiles' row batches evenly (k_gemm_f16s.hip, rows of 256, 512, 1,024 or 2,048),
against the CPU oracle: a share that begins and ends inside a tile, several tiles in one share, whole tiles and a rest, fewer batches than blocks, row
groups that do not fill the last batch, row sets without any row, tiles of one pair and full ones.

Products of weights exact in f16 with activations split into f16 hi and lo: 2^-22 of a factor and the f32 order of at most 2,048
terms are left, 2e-5 of a row's largest output; 1e-4 through the hardware exponential of silu."""
import numpy as np
import pytest

from util import nvfp4_weights, rng

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    import inferred_hip as ih
    be = ih.Hip(exact=False)
    yield be
    err = be.take_error()
    be.close()
    assert err is None, err


@pytest.fixture(scope="module")
def orc():
    from oracle import binding as ob
    return ob.Oracle(threads=8)


def worst(a, b, n_rows):
    a, b = a.reshape(n_rows, -1), b.reshape(n_rows, -1)
    assert np.isfinite(a).all()
    return float((np.abs(a - b).max(axis=1) / (np.abs(b).max(axis=1) + 1e-30)).max())


@pytest.mark.parametrize("n_in", [256, 512, 1024, 2048])
@pytest.mark.parametrize("n_tok,n_expert,n_used,n_out", [
    (32, 4, 1, 16),         # one row group: fewer batches than blocks, row sets with nothing to do
    (40, 16, 4, 48),        # three: the last batch is not full
    (33, 33, 2, 16 * 33),   # an odd number of groups over a few dozen tiles
    (300, 96, 8, 256),      # more batches than blocks: shares of a few batches, cut anywhere
    (17, 3, 3, 2048),       # two tiles an expert, the second of one pair
    (768, 16, 16, 16),      # one batch a tile, 768 tiles for 512 blocks: whole tiles and a rest
    (2049, 128, 8, 16),     # 1,100: two rounds of whole tiles, of which an expert has several
])
def test_shares_of_the_tiles(hip, orc, n_tok, n_expert, n_used, n_out, n_in):
    import inferred_hip as ih
    from oracle import binding as ob
    r = rng(n_in + n_out)
    scale = [r.random(n_expert).astype(np.float32) * 0.01 + 0.002 for _ in range(2)]
    gate, up = nvfp4_weights(r, n_expert * n_out, n_in), nvfp4_weights(r, n_expert * n_out, n_in)
    x = (r.standard_normal(n_tok * n_in) * np.repeat(10.0 ** r.uniform(-2.0, 1.0, n_tok), n_in)).astype(np.float32)
    ids = np.stack([r.choice(n_expert, n_used, replace=False) for _ in range(n_tok)]).astype(np.uint32).reshape(-1)
    pairs = ids.size
    hip.drop_mirrors(); hip.begin_pass(n_tok)
    route = ih.Hip.host_route(ids, r.random(pairs).astype(np.float32), n_used)
    got, want, tmp, tmp2 = (np.zeros(pairs * n_out, np.float32) for _ in range(4))
    hip.moe_glu(ih.experts(gate, ih.NVFP4, n_in, n_out, n_expert, scale[0]), ih.experts(up, ih.NVFP4, n_in, n_out, n_expert, scale[1]), route, x, got, tmp)
    orc.moe_glu(ob.experts(gate, ih.NVFP4, n_in, n_out, n_expert, scale[0]), ob.experts(up, ih.NVFP4, n_in, n_out, n_expert, scale[1]), ids, n_used, x, want, tmp2)
    hip.host_needs(got); hip.raise_if_error()
    assert worst(got, want, pairs) <= 1e-4
    xp = r.standard_normal(pairs * n_in).astype(np.float32)           # one activation row per token, then one per pair
    for rows in (x, xp):
        hip.matmul_experts(ih.experts(gate, ih.NVFP4, n_in, n_out, n_expert, scale[0]), route, rows, got)
        orc.matmul_experts(ob.experts(gate, ih.NVFP4, n_in, n_out, n_expert, scale[0]), ids, n_used, rows, want)
        hip.host_needs(got); hip.raise_if_error()
        assert worst(got, want, pairs) <= 2e-5
    hip.end_pass()
