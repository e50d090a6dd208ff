"""The attention of the prompt chunks that predict and predict_batch run, against the steps they stand for: as many bits of q.

A two-layer model in which everything but the first layer's softmax is exact in fp32, whatever order it is summed in: every
projection row has one weight, the norm's mean square is 1 and its epsilon 0, and the rotated dims carry nothing. K holds
+- 2^15 r (r = 1, 1/2, 1/4, 1/8) in two dims, q two numbers of 24 bits there that differ by about 2^-12: scores of about 1 in
which the last bit of q counts 2^-23 x 2^15 / 8 = 4.9e-4. Two fp16 terms of q drop that bit in about every other head; the
second layer's fp16 cache rows then round elsewhere for a share of about 4.9e-4 / 2^-11 (2^-10) of the values. In full fp32
the paths differ by a few 2^-24 around each probability: a share below 1e-3; the bar is 5e-3.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
D, HD, HEADS, KVH, V, N = 256, 64, 4, 2, 64, 60
ONE, TWO, Q1, Q2 = 0, 4, 8, 16  # first columns: the one-hot r, the 2, a pair of q columns per head


def _model(batch, w):
    from simplellminference_amd.model import LlamaModel, LlamaModelConfig
    from simplellminference_amd.tp import KINDS
    cfg = LlamaModelConfig(V, HD, D, KVH * HD, 128, N + 4, 2, HEADS, KVH, 0.0, 1e30)
    m = LlamaModel(config=cfg, w_dtype=w, kv_dtype="f16", seed=0, batch=batch).init()
    r = np.random.default_rng(5)
    emb = r.choice([-1.0, 1.0], (V, D))
    emb[:, ONE:ONE + 4] = 0
    emb[np.arange(V), ONE + np.arange(V) % 4] = 1
    emb[:, TWO] = 2
    emb[:, Q2:Q2 + HEADS] = emb[:, Q1:Q1 + HEADS]
    assert ((emb * emb).mean(1) == 1).all()
    n1 = np.ones(D)
    n1[Q1:Q1 + HEADS] = 1 + r.integers(1 << 18, 1 << 20, HEADS) * 2.0 ** -22
    n1[Q2:Q2 + HEADS] = n1[Q1:Q1 + HEADS] + r.choice([-1, 1], HEADS) * r.integers(700, 1365, HEADS) * 2.0 ** -22
    n1[32:] = r.integers(512, 1024, D - 32) / 512  # (v: exact in fp16)
    z = lambda rows, cols: np.zeros((rows, cols), np.float32)
    wq, wk, wv, wo = z(D, D), z(KVH * HD, D), z(KVH * HD, D), z(D, D)
    for h in range(HEADS):
        wq[h * HD + 20, Q1 + h] = wq[h * HD + 21, Q2 + h] = 1.5
    for g in range(KVH):
        for i in range(4):
            wk[g * HD + 20, ONE + i] = 2.0 ** (15 - i)
            wk[g * HD + 21, ONE + i] = -2.0 ** (15 - i)
    wv[np.arange(KVH * HD), 32 + r.permutation(D - 32)[:KVH * HD]] = 1
    wo[np.arange(D), r.permutation(D)] = 8
    for i in range(5):
        m.set_weight(KINDS["norm"], i, n1 if i == 0 else np.ones(D))
    for l in range(2):
        m.set_weight(KINDS["wq"], l, wq)
        m.set_weight(KINDS["wo"], l, wo)
        m.set_weight(KINDS["up"], l, z(128, D))
        m.set_weight(KINDS["gate"], l, z(128, D))
        m.set_weight(KINDS["down"], l, z(D, 128))
        if l == 1:
            wk, wv = z(KVH * HD, D), z(KVH * HD, D)
            for t in (wk, wv):
                t[np.arange(KVH * HD), r.permutation(D)[:KVH * HD]] = 1
        m.set_weight(KINDS["wk"], l, wk)
        m.set_weight(KINDS["wv"], l, wv)
    m.set_weight(KINDS["emb"], 0, emb)
    return m


@pytest.mark.parametrize("batch,w", [(1, "f32"), (2, "f16")])
def test_chunk_keeps_the_bits_of_the_steps(gpu, batch, w):
    m = _model(batch, w)
    r = np.random.default_rng(batch)
    prompts = [r.integers(0, V, N).tolist() for _ in range(batch)]
    run = (lambda **k: m.predict_batch(prompts, N, **k)) if batch > 1 else (lambda **k: m.predict(prompts[0], N, **k))
    rows = lambda layer: np.stack([m.kv(layer, which, N - 1, seq=b) for b in range(batch) for which in (0, 1)])
    run(want_logits=True)  # steps
    first, want = rows(0), rows(1)
    m.reset()
    run()  # a chunk, then the last position's step
    assert np.array_equal(rows(0), first), "the first layer's rows are exact"
    got = rows(1)
    share = (got != want).mean()
    print("share of the second layer's rows that differ", share)
    assert share <= 5e-3
    m.close()


def test_batch_chunk_of_wide_waves(gpu):
    """head_dim 64 and enough rows: 32 positions per wave with three terms. 1e-3 and one fp16 rounding of values up to 8, as in
    the other batch tests."""
    from simplellminference_amd.model import LlamaModel, LlamaModelConfig
    n, B = 401, 8
    m = LlamaModel(config=LlamaModelConfig(500, 64, 1024, 1024, 512, n + 3, 2, 16, 16, 1e-5, 1e4), w_dtype="f16", kv_dtype="f16",
                   seed=9, batch=B).init()
    r = np.random.default_rng(9)
    prompts = [r.integers(0, 500, n).tolist() for _ in range(B)]
    want, wl = m.predict_batch(prompts, n + 1, want_logits=True)
    kv = [m.kv(1, which, n, seq=b) for b in range(B) for which in (0, 1)]
    m.reset()
    assert np.array_equal(m.predict_batch(prompts, n + 1), want)
    assert np.abs(m.logits()[0] - wl[:, -1]).max() <= 1e-3
    for a, b in zip(kv, [m.kv(1, which, n, seq=b) for b in range(B) for which in (0, 1)]):
        assert np.abs(a - b).max() <= 2 ** -7
    m.close()
