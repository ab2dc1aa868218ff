"""Kernels at the edges of their dispatch rules and tiles, through the C ABI,
against the oracle's dequantised weights in float64."""
import numpy as np
import pytest

import kanjoos_amd as K
import oracle as O
from conftest import rel_rmse

pytestmark = pytest.mark.gpu

SEED = 11
U = 2.0 ** -24  # unit roundoff of float32


@pytest.mark.parametrize("n_in,n_out", [(256, 1), (256, 4097), (512, 127), (768, 33), (1280, 1000), (2304, 97),
                                        (4096, 13), (4096, 3203), (4352, 66)])
@pytest.mark.parametrize("fused", [False, True])
def test_gemv_q6k_edges(device, n_in, n_out, fused):
    """Every lanes-per-row instance, rows over one grid step, ragged row
    counts, both sides of the n_in = 4096 line; with and without the fused
    norm and residual."""
    print(f"gemv q6_k {n_in}x{n_out} fused={fused}", flush=True)
    w = O.synth_tensor(O.tensor_key(SEED, 0, "q", -1), K.TYPE_Q6_K, n_in, n_out)
    x = O.synth_f32(O.tensor_key(SEED, 0, "input"), n_in)
    nw = (1.0 + 0.1 * O.synth_f32(O.tensor_key(SEED, 0, "input", 7), n_in)).astype(np.float32)
    r = O.synth_f32(O.tensor_key(SEED, 0, "input", 8), n_out)
    x64 = x.astype(np.float64)
    if fused:
        x64 = x64 / np.sqrt(np.mean(x64 * x64) + 1e-6) * nw
    wd = O.dequant(K.TYPE_Q6_K, w, n_in * n_out).astype(np.float64).reshape(n_out, n_in)
    want = wd @ x64 + (r if fused else 0.0)
    # Weights are exact in the sums' terms and no chain of additions is over 32
    # long on any route; with the norm the roundings of x's mean square, its
    # root and the two products come on top.
    bound = (32 + 32 * fused) * U * (np.abs(wd) @ np.abs(x64) + (np.abs(r) if fused else 0.0))
    kw = dict(norm_w=K.DeviceBuffer.from_array(nw), eps=1e-6, resid=K.DeviceBuffer.from_array(r)) if fused else {}
    dy = K.DeviceBuffer(4 * n_out)
    K.gemv(K.TYPE_Q6_K, K.DeviceBuffer.from_array(w), n_in, n_out, K.DeviceBuffer.from_array(x), dy, **kw)
    got = dy.download(np.float32).astype(np.float64)
    assert np.all(np.abs(got - want) <= bound)
    assert rel_rmse(got, want) <= 1e-5


@pytest.mark.parametrize("n_in", [256, 768, 2048, 2304, 4096, 4352])
def test_gemv_q6k_lone_weights(device, n_in):
    """Rows with one nonzero weight each, at every position of a super-block in
    turn: the output is that weight's product alone, with nothing of the other
    inputs' size in its error (codes are stored with an offset of 32, and an
    offset subtracted only from the finished sums leaves their rounding)."""
    print(f"gemv q6_k lone weights {n_in}", flush=True)
    n_out, nb = 1024, n_in // 256
    rng = np.random.default_rng(n_in)
    w = O.synth_tensor(O.tensor_key(SEED, 0, "q", -1), K.TYPE_Q6_K, n_in, n_out)
    blocks = np.ascontiguousarray(w).view(np.uint8).reshape(n_out, nb, 210).copy()
    ql, qh = blocks[:, :, :128].copy(), blocks[:, :, 128:192].copy()
    blocks[:, :, :128], blocks[:, :, 128:192] = 0x00, 0xAA  # code 32: weight 0
    for j in range(n_out):
        # weight i of block b: half h, quarter t, byte l of the quarter
        b, i = int(rng.integers(nb)), (j * 7 + j // 256) % 256
        h, t, l = i // 128, i % 128 // 32, i % 32
        at, low = 64 * h + l + 32 * (t & 1), 0xF << (4 * (t >> 1))
        blocks[j, b, at] = ql[j, b, at] & low
        at, high = 32 * h + l, 3 << (2 * t)
        blocks[j, b, 128 + at] = (0xAA & ~high & 0xFF) | (qh[j, b, at] & high)
    w = blocks.reshape(-1)
    wd = O.dequant(K.TYPE_Q6_K, w, n_in * n_out).astype(np.float64).reshape(n_out, n_in)
    assert np.all(np.count_nonzero(wd, axis=1) <= 1) and np.count_nonzero(wd) > 0.9 * n_out
    x = rng.standard_normal(n_in).astype(np.float32)
    dy = K.DeviceBuffer(4 * n_out)
    K.gemv(K.TYPE_Q6_K, K.DeviceBuffer.from_array(w), n_in, n_out, K.DeviceBuffer.from_array(x), dy)
    got, want = dy.download(np.float32).astype(np.float64), wd @ x.astype(np.float64)
    assert np.all(np.abs(got - want) <= 4 * U * np.abs(want))  # the code's, the scale's and d's product


@pytest.mark.parametrize("n_embd,n_vocab,B", [(256, 65, 1), (512, 2049, 3), (1280, 4127, 33), (2048, 2048, 5)])
def test_batch_bf16_head_edges(device, n_embd, n_vocab, B):
    """The batched bf16 head and its argmax at ragged row counts (64-row
    workgroups, 2048-entry argmax chunks), at one tile of sequences and more,
    and at one to eight steps of 64 weights per wave (the model's widths are
    multiples of 256, so the four waves' shares are equal): logits against the
    oracle's within the parity bar (1e-5), the greedy token exactly the batch's
    own first maximum."""
    print(f"batch head {n_embd}x{n_vocab} B={B}", flush=True)
    cfg = dict(n_layer=1, n_embd=n_embd, n_head=8, n_head_kv=2, head_dim=64, n_ff=256, n_expert=16,
               n_expert_used=4, n_vocab=n_vocab, n_ctx=64)
    gm = K.Model.synthetic(K.qwen3_30b_a3b(**cfg), seed=SEED)
    toks = (np.arange(B, dtype=np.int32) * 7 + 1) % n_vocab
    img = gm.download_image()
    batch = K.Batch(gm, B, 64)
    lg = batch.forward(toks)
    om = O.OracleModel(O.make_config(**cfg), seed=SEED, image=img)
    for s in range(B):
        om.reset()
        om.set_kv_source(*batch.kv_download(s))  # the cache's f16 roundings are the device's
        assert rel_rmse(lg[s], om.forward([int(toks[s])])) <= 1e-5, s
    om.close()
    batch.close()
    batch = K.Batch(gm, B, 64)
    first = batch.decode_greedy(toks, 1)
    batch.close()
    assert np.array_equal(np.asarray(first).reshape(-1), lg.argmax(axis=1))
    gm.close()


@pytest.mark.parametrize("n_embd,n_ff,n_expert,m", [
    (256, 256, 8, 1), (768, 512, 8, 9), (2304, 768, 8, 5), (4096, 256, 8, 12), (1024, 1280, 8, 3),
    (2048, 256, 8, 2), (1280, 256, 80, 120), (2304, 512, 32, 20), (1280, 1024, 32, 40)])
def test_moe_few_pairs_edges(device, n_embd, n_ff, n_expert, m):
    """The few-pair expert products (fewer than ten pairs per expert) at one
    super-block, at counts of super-blocks that the waves of a workgroup share
    unevenly, at the widest row, in each form of gate/up (32 rows at once for
    narrow rows and short lists; six units with a last workgroup of four or two,
    one and two super-blocks per wave; four units) and with items of one to
    eight pairs: against the oracle within the parity bar (1e-5)."""
    k = 4
    print(f"few pairs {n_embd}x{n_ff} of {n_expert} m={m}", flush=True)
    syn = lambda kind, t, a, b, e=-1: O.synth_tensor(O.tensor_key(SEED, 1, kind, e), t, a, b)
    router = syn("router", K.TYPE_F32, n_embd, n_expert)
    gate, up = (np.concatenate([syn(n, K.TYPE_Q4_K, n_embd, n_ff, e) for e in range(n_expert)]) for n in ("gate", "up"))
    down = np.concatenate([syn("down", K.TYPE_Q4_K, n_ff, n_embd, e) for e in range(n_expert)])
    rng = np.random.default_rng(n_embd + m)
    x = rng.standard_normal((m, n_embd)).astype(np.float32)
    if m >= 12:  # ten equal tokens: two work items for each of their experts
        x[-9:] = x[0]
    resid = rng.standard_normal((m, n_embd)).astype(np.float32)
    want, _, ti_w, _ = O.moe(x, router, gate, up, down, n_embd, n_ff, n_expert, k, type_down=K.TYPE_Q4_K)
    assert m < 12 or np.bincount(ti_w.ravel()).max() > 8
    d = [K.DeviceBuffer.from_array(a) for a in (x, router, gate, up, down)]
    out, logits = K.DeviceBuffer(4 * m * n_embd), K.DeviceBuffer(4 * m * n_expert)
    ti, tw = K.DeviceBuffer(4 * m * k), K.DeviceBuffer(4 * m * k)
    K.moe_batch_layer(*d, m, n_embd, n_ff, n_expert, k, out, logits, ti, tw, resid=K.DeviceBuffer.from_array(resid))
    assert np.array_equal(ti.download(np.int32).reshape(m, k), ti_w)
    got = out.download(np.float32).reshape(m, n_embd) - resid
    for t in range(m):
        assert rel_rmse(got[t], want[t]) <= 1e-5, t


@pytest.mark.parametrize("n_head,n_kv,D", [(32, 4, 128), (16, 2, 64)])
def test_decode_attention_long_cache(device, n_head, n_kv, D):
    """The decode step's attention, which takes its position from the device and
    so splits the whole cache's slots: one sequence and two in lockstep over
    40,000 slots, seven and three chunks of 64 per workgroup, at positions that
    leave the first split part-way, most splits past the position, one split
    part-way far into the cache, and none.  The layer's output and the logits
    against the oracle's over the same cache within the parity bar (1e-5)."""
    n_ctx = 40000
    print(f"decode attention {n_head}/{n_kv} x {D} over {n_ctx} slots", flush=True)
    cfg = dict(n_layer=1, n_embd=512, n_head=n_head, n_head_kv=n_kv, head_dim=D, n_ff=256, n_expert=16,
               n_expert_used=4, n_vocab=1024, n_ctx=n_ctx)
    gm = K.Model.synthetic(K.qwen3_30b_a3b(**cfg), seed=SEED)
    om = O.OracleModel(O.make_config(**cfg), seed=SEED, image=gm.download_image())
    batch = K.Batch(gm, 2, n_ctx)
    rng = np.random.default_rng(D)
    shape = (1, n_kv, n_ctx, D)
    kc = (0.7 * rng.standard_normal(shape, dtype=np.float32)).astype(np.float16).view(np.uint16)
    vc = rng.standard_normal(shape, dtype=np.float32).astype(np.float16).view(np.uint16)
    ok, ov = om.kv()

    def same_as_oracle(tok, pos, cache, hidden, logits):
        """The oracle's step over a cache that holds what the device appended."""
        ok[...], ov[...] = kc, vc
        om.set_kv_source(*cache)
        om.set_pos(pos)
        want = om.forward([tok])
        assert om.kv_stats()["max_mid_dist"] <= 1e-5
        assert rel_rmse(hidden, om.hidden(0)) <= 1e-5, pos
        assert rel_rmse(logits, want) <= 1e-5, pos

    for pos in (40, 160, 30100, n_ctx - 1):
        print(f"position {pos}", flush=True)
        gm.kv_upload(kc, vc)
        gm.set_pos(pos)
        lg = gm.forward([7])
        same_as_oracle(7, pos, gm.kv_download(), gm.hidden(0), lg)
        for s in range(2):
            batch.kv_upload(s, kc, vc)
        batch.set_pos(pos)
        lg = batch.forward(np.array([7, 300], np.int32))
        for s, tok in enumerate((7, 300)):
            same_as_oracle(tok, pos, batch.kv_download(s), batch.hidden(0, s), lg[s])
    batch.close()
    om.close()
    gm.close()
