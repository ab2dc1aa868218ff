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
    blocks = np.ascontiguousarray(w).view(np.uint8).reshape(n_out, n_in // 256, 210)
    d = np.ascontiguousarray(blocks[:, :, 208:210]).view(np.float16).astype(np.float64)
    step = np.abs(np.ascontiguousarray(blocks[:, :, 192:208]).view(np.int8) * d)  # |d sc| per 16 weights
    # The dot is d sc (sum q x - 32 sum x): terms up to |w| + 64 |d sc| in
    # size, no chain of additions over 64 long on any route, a product each,
    # and with the norm a few roundings more on x (its mean square's too).
    size = (np.abs(wd) + 64.0 * np.repeat(step.reshape(n_out, -1), 16, axis=1)) @ np.abs(x64)
    bound = 80 * U * (size + (np.abs(r) if fused else 0.0))
    kw = dict(norm_w=K.DeviceBuffer.from_array(nw), eps=1e-6, resid=K.DeviceBuffer.from_array(r)) if fused else {}
    dy = K.DeviceBuffer(4 * n_out)
    K.gemv(K.TYPE_Q6_K, K.DeviceBuffer.from_array(w), n_in, n_out, K.DeviceBuffer.from_array(x), dy, **kw)
    got = dy.download(np.float32).astype(np.float64)
    assert np.all(np.abs(got - want) <= bound)
    assert rel_rmse(got, want) <= 1e-5


@pytest.mark.parametrize("n_embd,n_vocab,B", [(256, 65, 1), (512, 2049, 3), (1280, 4127, 33), (2048, 2048, 5)])
def test_batch_bf16_head_edges(device, n_embd, n_vocab, B):
    """The batched bf16 head and its argmax at ragged row counts (64-row
    workgroups, 2048-entry argmax chunks), at one tile of sequences and more,
    and at widths that leave the four K-splits uneven: logits against the
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
