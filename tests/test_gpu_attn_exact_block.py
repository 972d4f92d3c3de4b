"""A single-token attention block of exact mode, recorded and replayed with the new position's norms, rotation and cache rows formed
by the attention kernel itself, against the CPU oracle bit for bit: contexts across its loops' edges, the scores' place in LDS, one
to eight query heads a KV head."""
import numpy as np
import pytest

from test_gpu_fused_fast import Both, bufs
from util import Hiprt, f16_bits, rng

pytestmark = pytest.mark.gpu
ND, EPS, THETA, PASSES = 256, 1e-6, 1e7, 9


@pytest.mark.parametrize("nh,nkv,hd,n_rot,n_ctx,pos0,kernels", [
    (8, 1, 64, 32, 512, 0, 3),          # the first positions: nothing in the slabs
    (8, 1, 64, 64, 512, 251, 3),        # 256 values' rows brought at a time
    (8, 4, 256, 64, 300, 58, 3),        # 64 keys a wave
    (2, 2, 128, 128, 1200, 508, 3),     # 512 a block; the last thread has a position of its own beside the new one
    (2, 1, 256, 256, 1200, 1021, 3),
    (4, 4, 64, 16, 4200, 4092, 3),      # scores past LDS
    (2, 1, 256, 64, 300, 125, 3),       # 128 rows at a time
    (8, 2, 128, 64, 300, 251, 3),       # 256
    (6, 2, 96, 48, 256, 247, 4),        # other heads: norms, rotation and cache write by themselves
    (4, 4, 8, 4, 200, 30, 4),
    (2, 1, 320, 64, 64, 31, 4),
])
def test_block(nh, nkv, hd, n_rot, n_ctx, pos0, kernels):
    recorded_block(nh, nkv, hd, n_rot, n_ctx, pos0, kernels)


@pytest.mark.parametrize("over,kernels", [("q", 4), ("k", 4), ("v", 4), ("qg", 0)])
@pytest.mark.parametrize("nh,nkv,hd", [(8, 8, 64), (4, 4, 256)])
def test_result_over_an_input(nh, nkv, hd, over, kernels):
    """What one block reads another must not have written: the rows by themselves, or the ops one by one."""
    recorded_block(nh, nkv, hd, 64, 300, 125, kernels, attn=over)


def recorded_block(nh, nkv, hd, n_rot, n_ctx, pos0, kernels, attn="attn"):
    import inferred_hip as ih
    from oracle import binding as ob
    hip = ih.Hip(exact=True)
    pair = Both(hip, ob.Oracle(threads=8))
    orc = pair.orc
    qd, kd = nh * hd, nkv * hd
    r = rng(hd + pos0)
    wq, wk, wv, wo = pair.q8(r, 2 * qd, ND, 2.0), pair.q8(r, kd, ND, 2.0), pair.q8(r, kd, ND, 2.0), pair.q8(r, ND, qd, 8.0)
    norm_w, qn, kn = [(0.5 + r.random(n)).astype(np.float32) for n in (ND, hd, hd)]
    B = bufs(x=ND, normed=ND, qg=2 * qd, q=qd, g=qd, k=kd, v=kd, attn=qd, mixed=ND)
    small = np.where(np.arange(n_ctx) % 5 == 3, 2.0 ** -18, 1.0)[:, None]        # (some rows subnormal in f16)
    k0, v0 = (f16_bits((r.standard_normal((n_ctx, kd)) * small).reshape(-1)) for _ in range(2))
    k0[pos0 * kd:] = 0
    v0[pos0 * kd:] = 0
    slabs = [dict(k=k0.copy(), v=v0.copy()) for _ in range(2)]
    sc = float(1.0 / np.sqrt(np.float32(hd)))
    res = lambda b: b[attn][:qd]   # noqa: E731
    read = ("x",) if attn != "attn" else ("x", "attn", "q")

    def block(ops, i, b, s, pos):
        W = lambda t: t[i]
        ops.rms_norm(b["x"], norm_w, EPS, b["normed"])
        ops.matmul(W(wq), b["normed"], b["qg"])
        ops.gather_chunks(b["qg"], hd, 2 * hd, 0, b["q"]); ops.gather_chunks(b["qg"], hd, 2 * hd, hd, b["g"])
        ops.matmul(W(wk), b["normed"], b["k"]); ops.matmul(W(wv), b["normed"], b["v"])
        ops.rms_norm_heads(b["q"], qn, hd, EPS); ops.rms_norm_heads(b["k"], kn, hd, EPS)
        ops.rope_neox(b["q"], pos, hd, n_rot, nh, THETA); ops.rope_neox(b["k"], pos, hd, n_rot, nkv, THETA)
        ops.kv_write(s["k"], pos * kd, b["k"]); ops.kv_write(s["v"], pos * kd, b["v"])
        ops.attend(b["q"], s["k"], s["v"], kd, pos + 1, hd, nh, nkv, sc, res(b))
        ops.sigmoid_mul(res(b), b["g"])
        ops.matmul(W(wo), res(b), b["mixed"])
        ops.add_assign(b["x"], b["mixed"])

    try:
        for p in range(PASSES):              # two op by op, one recorded (again, where the scratch has grown), the rest replayed
            pos = pos0 + p
            x0 = rng(500 + p).standard_normal(ND).astype(np.float32)
            for b in B:
                b["x"][:] = x0
            hip.begin_pass(1); hip.host_wrote(B[0]["x"]); block(hip, 0, B[0], slabs[0], pos); hip.end_pass()
            for name in read:
                hip.host_needs(B[0][name])
            hip.read_kv(slabs[0]["k"]); hip.read_kv(slabs[0]["v"])
            hip.raise_if_error()
            block(orc, 1, B[1], slabs[1], pos)
            for name in read:
                assert np.array_equal(B[0][name].view(np.uint32), B[1][name].view(np.uint32)), (p, name)
            for t in "kv":
                assert np.array_equal(slabs[0][t], slabs[1][t]), (p, t)
        g = hip.graph_stats()
        assert g["captures"] == 1 and g["replays"] >= 1 and (not kernels or g["graph_kernels"] == kernels), g
    finally:
        hip.take_error()
        hip.close()


@pytest.mark.parametrize("exact,nh,hd", [(False, 64, 320), (True, 64, 256), (True, 128, 1024)])
def test_scratch_of_an_unrecorded_call(exact, nh, hd):
    """A row of scores a head: only the recorded form of exact mode leaves more.  (Measured as what the call takes from the device:
    its mirrors and slabs, and 4 bytes a score and an eighth to a quarter more; 8 MB for what the allocator rounds up to.)"""
    import inferred_hip as ih
    n_pos, rt = 40000, Hiprt()
    hip = ih.Hip(exact=exact)
    try:
        q, out = (np.zeros(nh * hd, np.float32) for _ in range(2))
        k, v = (np.zeros(n_pos * hd, np.uint16) for _ in range(2))
        hip.attend(q, k, v, hd, 8, hd, nh, 1, 1.0, out)           # mirrors and slabs
        hip.sync()
        before = rt.mem_free()
        hip.attend(q, k, v, hd, n_pos, hd, nh, 1, 1.0, out)
        hip.sync()
        hip.raise_if_error()
        assert before - rt.mem_free() <= nh * n_pos * 4 * 1.25 + (8 << 20)
    finally:
        hip.close()
