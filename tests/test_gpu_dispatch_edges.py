"""Where the dispatch changes kernels: the NVFP4 tiles' token and pair counts, copies to the host by size, bit-exact paths
that take a short cut and fall back, and a chain of two layers against its stages by vocabulary."""
import numpy as np
import pytest

import test_gpu_ops_fast as fast
from util import assert_bits_equal, f16_bits, nvfp4_weights, rng

pytestmark = pytest.mark.gpu


def backend(exact):
    import inferred_hip as ih
    be = ih.Hip(exact=exact)
    yield be
    err = be.take_error()
    be.close()
    assert err is None, err


@pytest.fixture(scope="module")
def hip():
    yield from backend(False)


@pytest.fixture(scope="module")
def exact():
    yield from backend(True)


@pytest.fixture(scope="module")
def orc():
    from oracle import binding as ob
    return ob.Oracle(threads=8)


def fresh(be, n=1):
    be.drop_mirrors()
    be.begin_pass(n)


@pytest.mark.parametrize("n_tok,n_expert,n_used", [(7, 16, 4), (8, 16, 4), (191, 16, 4), (192, 16, 4), (575, 64, 4), (576, 64, 4), (33, 512, 1), (63, 512, 10)])
def test_expert_tiles_by_pairs(hip, orc, n_tok, n_expert, n_used):
    fast.test_moe_stage_fast_nvfp4(hip, orc, n_tok, n_expert, n_used, 512, 256)


@pytest.mark.parametrize("n_in,n_out,n", [(512, 256, 32), (512, 256, 33), (256, 68, 63), (512, 260, 64), (2048, 512, 1023), (2048, 512, 1024)])
def test_dense_nvfp4_by_tokens(hip, orc, n_in, n_out, n):
    fast.test_matmul_nvfp4_batched_fast(hip, orc, n_in, n_out, n)


@pytest.mark.parametrize("n", [1, 3, 4, 5, 4097, 262144, 262145, 600001])
def test_copies_home_by_size(hip, n):
    fresh(hip)
    x = rng(n).standard_normal(n).astype(np.float32)
    for _ in range(3):
        a = x.copy()
        hip.host_wrote(a); hip.scale(a, 2.0); hip.host_needs(a)
        assert np.array_equal(a, 2 * x)
        hip.release(a)


@pytest.mark.parametrize("at,n", [(0, 4096), (4, 4092), (1, 4095), (0, 5), (4080, 16)])
def test_copies_home_into_page_locked_memory(hip, at, n):
    """Aligned ranges of a page-locked allocation, up to its end, are written by the device itself, others through the
    backend's own; the same addresses in turn with pageable ones, on one backend."""
    import ctypes as C
    fresh(hip)
    rt = C.CDLL("libamdhip64.so")
    p = C.c_void_p()
    assert rt.hipHostMalloc(C.byref(p), C.c_size_t(4096 * 4), 0) == 0
    try:
        locked = np.frombuffer((C.c_float * 4096).from_address(p.value), np.float32)
        locked[:] = -1.0
        a, x = locked[at:at + n], rng(n).standard_normal(n).astype(np.float32)
        for k in range(3):
            pageable = x.copy()
            a[:] = x
            for buf in (a, pageable):
                hip.host_wrote(buf); hip.scale(buf, 2.0 + k); hip.host_needs(buf)
                assert np.array_equal(buf, np.float32(2.0 + k) * x)
                hip.release(buf)
        assert (locked[:at] == -1.0).all() and (locked[at + n:] == -1.0).all()
        hip.raise_if_error()
    finally:
        rt.hipHostFree(p)


@pytest.mark.parametrize("n_in,n_out,n", [(512, 70, 63), (512, 70, 64), (512, 68, 65), (256, 36, 200)])
def test_exact_dense_nvfp4_batches(exact, orc, n_in, n_out, n):
    import inferred_hip as ih
    from oracle import binding as ob
    fresh(exact, n)
    r = rng(n)
    wb = nvfp4_weights(r, n_out, n_in)
    x = r.standard_normal(n * n_in).astype(np.float32)
    a = np.zeros(n * n_out, np.float32); b = np.zeros_like(a)
    exact.matmul(ih.weights(wb, ih.NVFP4, n_in, n_out), x, a); exact.host_needs(a)
    orc.matmul(ob.weights(wb, ob.NVFP4, n_in, n_out), x, b)
    exact.raise_if_error()
    assert_bits_equal(a, b, "matmul nvfp4")


@pytest.mark.parametrize("n_q,n_pos,hd,nh,nkv", [(1, 4096, 64, 8, 2), (1, 4097, 64, 8, 2), (2, 5003, 256, 16, 2), (33, 70, 128, 4, 2)])
def test_exact_attention_over_long_contexts(exact, orc, n_q, n_pos, hd, nh, nkv):
    fresh(exact)
    r = rng(n_pos)
    kv_dim = nkv * hd
    q = r.standard_normal(n_q * nh * hd).astype(np.float32)
    k = f16_bits(r.standard_normal(n_pos * kv_dim)); v = f16_bits(r.standard_normal(n_pos * kv_dim))
    a, b = np.zeros(n_q * nh * hd, np.float32), np.zeros(n_q * nh * hd, np.float32)
    sc = 1.0 / np.sqrt(np.float32(hd))
    exact.attend(q, k, v, kv_dim, n_pos, hd, nh, nkv, sc, a); exact.host_needs(a)
    orc.attend(q, k, v, kv_dim, n_pos, hd, nh, nkv, sc, b)
    exact.raise_if_error()
    assert_bits_equal(a, b, "attend")


@pytest.mark.parametrize("n,nd", [(1, 512), (3, 512), (1, 2048), (40, 2048)])
def test_exact_mean_square_at_a_rounding_tie(exact, orc, n, nd):
    """nd / 2 ones and one 2^-k: the mean of squares lies half way between two f32, so the order of the sum decides it."""
    fresh(exact, n)
    x = np.zeros((n, nd), np.float32)
    half = nd // 2
    for t in range(n):
        at = rng(t).permutation(nd)
        x[t, at[:half]] = 1.0
        x[t, at[half]] = np.sqrt(half * 2.0 ** -24) if half in (256, 1024) else 0.0
    w = np.ones(nd, np.float32)
    a, b = np.zeros(n * nd, np.float32), np.zeros(n * nd, np.float32)
    exact.rms_norm(x.reshape(-1), w, 1e-6, a); exact.host_needs(a)
    orc.rms_norm(x.reshape(-1), w, 1e-6, b)
    exact.raise_if_error()
    assert_bits_equal(a, b, "rms_norm at a tie")


@pytest.mark.parametrize("n_vocab", [8195, 16384, 16385])
def test_short_chain_by_vocabulary(tmp_path, n_vocab):
    """Decode steps of a two-layer model, its layers as one chain, against the same steps on a backend that launches every
    stage by itself; turn by turn, so that the later ones replay.  The stages' sums are in another order, which moves Q8_0
    steps of 1/127 of a block and now and then exchanges an expert: fast and exact mode differ by 5e-3 to 1.4e-2 of the logits'
    2-norm on such models, so 2e-2 bounds two orders of sums, where a lost layer or a stale row gives about 1."""
    import inferred_hip as ih
    path = str(tmp_path / "short.gguf")
    ih.synth_write_gguf(path, ih.big_config(n_layer=2, full_attention_interval=2, n_vocab=n_vocab))
    got = []
    for chain in (True, False):
        be, m = ih.Hip(exact=False, chain=chain), ih.Model(path)
        e = ih.Engine(m, be, 64)
        turns = []
        for turn in range(3):
            e.reset()
            turns.append(np.stack([np.array(e.forward([(37 * t + 5) % n_vocab])) for t in range(6)]))
        be.raise_if_error()
        assert (be.chain_stats()["chains"] > 0) == chain
        assert np.array_equal(turns[1], turns[2])
        got.append(turns[2])
        e.close(); m.close(); be.close()
    err = np.linalg.norm(got[0] - got[1]) / np.linalg.norm(got[1])
    print(n_vocab, err, flush=True)
    assert err <= 2e-2, err
