"""Batched decode (B sequences decoding in lockstep, projections on MFMA in
bgemm.h) against the C oracle run once per sequence on identical synthetic weights and prompts.

Bar: per-sequence greedy token ids bit-exact; logits within the north_star tolerance 1e-3 (fp16 weights:
the oracle computes in fp32 on the identically rounded weights and the same fp16 K/V rounding). The
batched projection itself is held to 1e-4 (relative + absolute) against a float64 product of the same
fp16 weights, and is bit-exact on small-integer data (exact in fp16 and fp32).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PROMPTS = [[1, 17, 42, 99], [5, 6], [300, 2, 77, 8, 9], [11]]  # ragged prompts, one per sequence


def _t(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _ocfg(oracle, cfg):
    return oracle.Config(cfg.vocab_size, cfg.hidden_size, cfg.num_attention_heads, cfg.num_key_value_heads,
                         cfg.head_dim, cfg.intermediate_size, cfg.num_hidden_layers, cfg.max_length,
                         cfg.rms_norm_eps, cfg.rope_theta)


@pytest.mark.parametrize("rows,cols,batch", [(4096, 4096, 8), (768, 4096, 8), (4096, 14336, 8), (4096, 512, 8),
                                             (16032, 4096, 8), (100, 256, 3), (4000, 4096, 5), (16, 32, 1),
                                             (6144, 4096, 2)])
def test_matmul_batch_f16(gpu, rows, cols, batch):
    torch = gpu
    from simplellminference_amd import ops
    r = np.random.default_rng(rows + cols + batch)
    x = r.standard_normal((batch, cols)).astype(np.float32)
    w16 = (r.standard_normal((rows, cols)) / np.sqrt(cols)).astype(np.float16)
    want = x.astype(np.float64) @ w16.astype(np.float64).T
    got = ops.matmul_batch(_t(torch, x), _t(torch, w16)).cpu().numpy()
    err = np.abs(got - want)
    assert np.all(err <= 1e-4 + 1e-4 * np.abs(want)), err.max()


@pytest.mark.parametrize("rows,cols,batch", [(64, 128, 8), (48, 4096, 7), (4096, 1024, 8)])
def test_matmul_batch_exact_integers(gpu, rows, cols, batch):
    """Small integers are exact in fp16 (weights, hi part; lo = 0) and their sums exact in fp32, so any
    fragment-layout, tile-map or split-merge error shows as a mismatch."""
    torch = gpu
    from simplellminference_amd import ops
    r = np.random.default_rng(7 + rows)
    x = r.integers(-3, 4, (batch, cols)).astype(np.float32)
    w = r.integers(-3, 4, (rows, cols)).astype(np.float16)
    want = (x.astype(np.int64) @ w.astype(np.int64).T).astype(np.float32)
    got = ops.matmul_batch(_t(torch, x), _t(torch, w)).cpu().numpy()
    assert np.array_equal(got, want)


# (rows, cols, batch) -> blocks of a step: waves with 5 k-blocks of a tile (or 4 and 5, unevenly), 6, 7 and 4
STEP_SHAPES = {(2048, 10240, 1): 5, (2048, 10240, 6): 5, (2048, 10240, 8): 5, (2048, 8224, 3): 5, (2048, 8416, 8): 5,
               (2048, 10272, 8): 7, (2048, 14336, 1): 7, (2048, 8192, 6): 4}


@pytest.mark.parametrize("rows,cols,batch", [(8200, 2080, 8), (8200, 2560, 5), (8200, 2592, 3),
                                             (16, 16384, 8), (48, 9216, 6), (64, 4640, 1)] + list(STEP_SHAPES))
def test_matmul_batch_steps_of_five_and_many_splits(gpu, rows, cols, batch):
    """A wave's 5, 6 or 7 k-blocks of a tile as one step (STEP_SHAPES; test_host_runtime.py looks that they run), and merges of 3
    and 4 splits and of 9 and 16, more than one round of loads holds. Small integers: sums are exact in any order."""
    test_matmul_batch_exact_integers(gpu, rows, cols, batch)


@pytest.mark.parametrize("name", ["tiny", "tiny-gqa"])
@pytest.mark.parametrize("kv", ["f16", "f32"])
def test_batch_predict_parity(gpu, oracle, name, kv):
    from simplellminference_amd.model import LlamaModel, preset
    cfg = preset(name)
    gm = LlamaModel(config=cfg, w_dtype="f16", kv_dtype=kv, seed=0, batch=len(PROMPTS)).init()
    steps = 36  # prompt + greedy, 36 positions
    toks, logits = gm.predict_batch(PROMPTS, steps, want_logits=True)
    gm.close()
    for b, p in enumerate(PROMPTS):
        om = oracle.Model(_ocfg(oracle, cfg), seed=0, wmode=oracle.W_F16, kv_f16=(kv == "f16"))
        otok, olog = om.predict(p, steps)
        om.close()
        assert np.array_equal(toks[b], otok), (b, toks[b], otok)
        assert np.abs(logits[b] - olog).max() <= 1e-3, (b, np.abs(logits[b] - olog).max())


def test_batch_state_and_history(gpu, oracle):
    """Per-sequence state after a batched predict: positions advance together, last_argmax is each
    sequence's own greedy choice, history is the fed tokens, KV rows match the oracle's."""
    from simplellminference_amd.model import LlamaModel, preset
    cfg = preset("tiny-gqa")
    gm = LlamaModel(config=cfg, w_dtype="f16", kv_dtype="f16", seed=0, batch=len(PROMPTS)).init()
    toks, logits = gm.predict_batch(PROMPTS, 12, want_logits=True)
    for b, p in enumerate(PROMPTS):
        st = gm.state(b)
        assert st["pos"] == 12 and st["error"] == 0
        assert st["last_argmax"] == int(np.argmax(logits[b, -1]))
        assert np.array_equal(gm.history(b, 12), toks[b])
        om = oracle.Model(_ocfg(oracle, cfg), seed=0, wmode=oracle.W_F16, kv_f16=True)
        om.predict(p, 12)
        ok, ov = om.kv_cache()
        for layer in range(cfg.num_hidden_layers):
            np.testing.assert_allclose(gm.kv(layer, 0, 12, seq=b), ok[layer, :12], rtol=0, atol=2e-3)
            np.testing.assert_allclose(gm.kv(layer, 1, 12, seq=b), ov[layer, :12], rtol=0, atol=2e-3)
        om.close()
    gm.close()


def test_batch_tp_step_on_one_rank_communicator(gpu, oracle, monkeypatch):
    """SLI_DEBUG_FORCE_COMM with a batch: partials, the [B][D] RCCL sum all-reduces and the [B] uint64 MAX
    argmax all-reduce, all captured in the step graph."""
    from simplellminference_amd.model import LlamaModel, preset
    monkeypatch.setenv("SLI_DEBUG_FORCE_COMM", "1")
    cfg = preset("tiny-gqa")
    prompts = PROMPTS[:2]
    gm = LlamaModel(config=cfg, w_dtype="f16", kv_dtype="f16", seed=0, batch=2).init()
    toks, logits = gm.predict_batch(prompts, 24, want_logits=True)
    gm.close()
    for b, p in enumerate(prompts):
        om = oracle.Model(_ocfg(oracle, cfg), seed=0, wmode=oracle.W_F16, kv_f16=True)
        otok, olog = om.predict(p, 24)
        om.close()
        assert np.array_equal(toks[b], otok)
        assert np.abs(logits[b] - olog).max() <= 1e-3


def test_llama3_8b_shape_two_layers_batch8(gpu, oracle):
    """Llama-3-8B layer shapes (D 4096, GQA 32/8, I 14336, vocab 128256, theta 5e5) at ctx 4096, batch 8,
    two layers; sequence b's KV filled with seed 7 + b to its own (ragged) position, one step each."""
    from simplellminference_amd.model import LlamaModel, preset
    cfg = preset("llama3-8b", num_hidden_layers=2)
    gm = LlamaModel(config=cfg, w_dtype="f16", kv_dtype="f16", seed=1, batch=8).init()
    gm.fill_kv_synthetic(7, 4095)
    tokens = [1234 + 9001 * b for b in range(8)]
    positions = [4095, 4095, 100, 2047, 4000, 1, 3333, 4095]
    got = gm.forward_batch(tokens, positions)
    gm.close()
    om = oracle.Model(_ocfg(oracle, cfg), seed=1, wmode=oracle.W_F16, kv_f16=True)
    for b in range(8):
        om.fill_kv_synthetic(7 + b, 4095)
        want = om.forward(tokens[b], positions[b])
        assert np.abs(got[b] - want).max() <= 1e-3, (b, np.abs(got[b] - want).max())
        assert int(np.argmax(got[b])) == int(np.argmax(want))
    om.close()


def test_llama3_8b_full_batch8_properties(gpu):
    """The C4 workload at TP 1 (32 layers, batch 8, ctx 4096): deterministic idempotent step, finite
    logits, per-sequence argmax state, algorithmic bytes = SURVEY.md §8(d) (15.009 GB weights, 4.295 GB
    KV)."""
    from simplellminference_amd.model import LlamaModel, preset
    gm = LlamaModel(config=preset("llama3-8b"), w_dtype="f16", kv_dtype="f16", seed=1, batch=8).init()
    gm.fill_kv_synthetic(7, 4095)
    tokens = [100 + 17 * b for b in range(8)]
    a = gm.forward_batch(tokens, [4095] * 8)
    b = gm.forward_batch(tokens, [4095] * 8)
    assert np.isfinite(a).all()
    assert np.array_equal(a, b)
    for s in range(8):
        st = gm.state(s)
        assert st["last_argmax"] == int(np.argmax(a[s])) and st["error"] == 0
    wb, kb = gm.step_bytes()
    assert abs(wb - 15.009e9) / 15.009e9 < 0.01 and abs(kb - 4.295e9) / 4.295e9 < 0.01
    gm.close()


@pytest.mark.timeout(900)
def test_llama3_8b_full_batch8_matches_oracle(gpu, oracle):
    """The whole C4 workload at TP 1 (Llama-3-8B, 32 layers, vocab 128256, batch 8, ctx 4096) against the
    oracle's full forward per sequence (the lazy oracle: each layer's weights regenerated in turn), ragged
    positions. Bar: the same argmax for every sequence and logits within 1e-3 absolute (north star: "1e-3 fp16
    tolerance"). Sequence 5 sits at position 1. A float64 restatement of that step (tests/golden/make_f64_c4.py,
    committed as c4_f64_seq5.npz) puts the ORACLE 1.33e-3 from float64, six further fp32 restatements that differ
    only in their dot-product summation order 1.04e-3 .. 1.34e-3 (fp32_spread), and the GPU 1.36e-3 (round 4):
    every fp32 path sits that far from float64, so the 1.4e-3 is the step's own conditioning at a two-position
    context (each layer's new K/V row, half of the attention's input, is rounded to fp16 from an fp32 value;
    32 layers amplify which side of a rounding boundary it lands on), not an error of either side. That
    sequence is therefore bounded by the fp32 paths' own float64 distance: GPU vs float64 within 1.1x of the
    largest of them, and GPU vs oracle within 1e-3 plus the oracle's."""
    import os
    from simplellminference_amd.model import LlamaModel, preset
    f64 = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "c4_f64_seq5.npz"))
    cfg = preset("llama3-8b")
    gm = LlamaModel(config=cfg, w_dtype="f16", kv_dtype="f16", seed=1, batch=8).init()
    gm.fill_kv_synthetic(7, 4095)
    tokens = [1234 + 9001 * b for b in range(8)]
    positions = [4095, 4095, 100, 2047, 4000, 1, 3333, 4095]
    assert (tokens[5], positions[5], 7 + 5) == (int(f64["token"]), int(f64["pos"]), int(f64["kv_seed"]))
    got = gm.forward_batch(tokens, positions)
    gm.close()
    err64 = float(np.abs(got[5] - f64["logits"]).max())
    print(f"C4 sequence 5 (pos 1): GPU vs float64 max|d| {err64:.2e}; oracle vs float64 {float(f64['oracle_err']):.2e}")
    fp32_worst = max(float(f64["oracle_err"]), float(np.max(f64["fp32_spread"])))
    assert err64 <= 1.1 * fp32_worst, (err64, fp32_worst)
    assert int(np.argmax(got[5])) == int(f64["argmax"])
    om = oracle.Model(_ocfg(oracle, cfg), seed=1, wmode=oracle.W_F16, kv_f16=True, lazy=True)
    errs = []
    for b in range(8):
        om.fill_kv_synthetic(7 + b, 4095)
        want = om.forward(tokens[b], positions[b])
        errs.append(float(np.abs(got[b] - want).max()))
        assert int(np.argmax(got[b])) == int(np.argmax(want)), b
    om.close()
    print(f"C4 full model, per-sequence max|dlogit| vs the oracle: {['%.2e' % e for e in errs]}")
    bound = [1e-3] * 8
    bound[5] = 1e-3 + float(f64["oracle_err"])
    assert all(e <= b for e, b in zip(errs, bound)), errs


@pytest.mark.timeout(900)
def test_llama3_8b_short_context_band_vs_float64(gpu, oracle):
    """The C4 model (Llama-3-8B, 32 layers, batch 8) at the short contexts where 32 layers amplify the fp16 rounding
    of every layer's new K/V row: sequence b at position b + 1 (b = 0..7), against the float64 restatement of the
    same eight steps (tests/golden/make_f64_c4_band.py -> c4_f64_band.npz). At each position the bar is the fp32
    conditioning measured there: GPU vs float64 within 1.1x the largest float64 distance of seven fp32 paths (the
    oracle's sequential sums, BLAS, and five column-block orders), argmax equal. The fixture's distances of those
    orders to the oracle itself (fp32_vs_oracle) show where the north star's 1e-3 against the reference cannot hold
    for ANY fp32 order: the GPU is also held to the oracle run here (the reference's own order), within
    the north star's 1e-3, or 1.1x the largest fp32 order's distance to it at that position where that is larger, so
    a drift away from the reference is caught and not only one away from float64. Past position 8 the full test above holds every sequence to 1e-3 absolute against the
    oracle; position 1 is the documented exception to the north star's 1e-3."""
    import os
    from simplellminference_amd.model import LlamaModel, preset
    f64 = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "c4_f64_band.npz"))
    tokens, positions = [int(t) for t in f64["tokens"]], [int(p) for p in f64["positions"]]
    assert [int(s) for s in f64["kv_seeds"]] == [7 + b for b in range(8)] and positions == list(range(1, 9))
    gm = LlamaModel(config=preset("llama3-8b"), w_dtype="f16", kv_dtype="f16", seed=1, batch=8).init()
    gm.fill_kv_synthetic(7, 9)  # sequence b: seed 7 + b, rows 0..8
    got = gm.forward_batch(tokens, positions)
    gm.close()
    rows = []
    for b in range(8):
        err = float(np.abs(got[b] - f64["logits"][b]).max())
        worst = max(float(f64["oracle_err"][b]), float(np.max(f64["fp32_spread"][b])))
        rows.append((positions[b], err, worst))
        assert int(np.argmax(got[b])) == int(f64["argmax"][b]), b
    print("C4 band (pos, GPU vs float64, worst fp32 order vs float64): "
          + ", ".join(f"({p}, {e:.2e}, {w:.2e})" for p, e, w in rows))
    assert all(e <= 1.1 * w for _, e, w in rows), rows
    om = oracle.Model(_ocfg(oracle, preset("llama3-8b")), seed=1, wmode=oracle.W_F16, kv_f16=True, lazy=True)
    orows = []
    for b in range(8):
        om.fill_kv_synthetic(7 + b, 9)
        want = om.forward(tokens[b], positions[b])
        assert int(np.argmax(want)) == int(f64["oracle_argmax"][b]), b  # the fixture's oracle, reproduced
        orows.append((positions[b], float(np.abs(got[b] - want).max()), float(np.max(f64["fp32_vs_oracle"][b]))))
    om.close()
    print("C4 band (pos, GPU vs oracle, worst fp32 order vs oracle): "
          + ", ".join(f"({p}, {e:.2e}, {w:.2e})" for p, e, w in orows))
    # the north star's 1e-3 against the reference, widened only where the fp32 orders themselves exceed it (the
    # documented exception: positions 1-2)
    assert all(e <= max(1e-3, 1.1 * w) for _, e, w in orows), orows


@pytest.mark.parametrize("world", [2, 8])
def test_batch_tp_shard_step_nocomm(gpu, monkeypatch, world):
    """One rank of a C4-shaped tensor-parallel batch (Llama-3-8B shapes, 2 layers, batch 8): the rank's
    shard geometry (1 kv head per rank at TP 8, FFN 1792, vocab shard 16032) plans, allocates and steps
    without a communicator (SLI_DEBUG_NOCOMM: placement and kernel shapes only; values are not a model)."""
    from simplellminference_amd.model import LlamaModel, preset
    monkeypatch.setenv("SLI_DEBUG_NOCOMM", "1")
    cfg = preset("llama3-8b", num_hidden_layers=2)
    m = LlamaModel(config=cfg, w_dtype="f16", kv_dtype="f16", seed=1, batch=8, tp_rank=world - 1,
                   tp_size=world).init()
    m.fill_kv_synthetic(7, 4095)
    a = m.forward_batch([5 + b for b in range(8)], [4095, 17, 4000, 1, 2048, 3000, 4095, 9])
    b = m.forward_batch([5 + b for b in range(8)], [4095, 17, 4000, 1, 2048, 3000, 4095, 9])
    assert a.shape == (8, m.local_vocab) and np.isfinite(a).all() and np.array_equal(a, b)
    m.close()


@pytest.mark.parametrize("kv", ["f16", "f32"])
@pytest.mark.parametrize("name,batch,short,long,length", [
    ("tiny-gqa", 2, 9, 9, 30), ("tiny", 3, 8, 12, 20), ("tiny-gqa", 8, 10, 17, 17), ("small-h128-gqa", 8, 40, 49, 60),
    ("small-h128", 5, 200, 210, 214), ("small-h128-gqa", 8, 500, 508, 511)])
def test_predict_batch_prompt_chunks_match_steps(gpu, kv, name, batch, short, long, length):
    """Without wanted logits predict_batch runs what every prompt has as packed chunks (9 shared positions and more; 8:
    steps; 8 sequences of 499: two chunks), with them as steps: the same tokens, states, last logits (1e-3, the bar of these
    files) and K/V rows (one fp16 rounding of values up to 8)."""
    from simplellminference_amd.model import LlamaModel, preset
    m = LlamaModel(config=preset(name), w_dtype="f16", kv_dtype=kv, seed=6, batch=batch).init()
    r = np.random.default_rng(batch)
    lens = [short + (long - short) * b // (batch - 1) for b in range(batch)]
    prompts = [r.integers(0, m.config.vocab_size, n).tolist() for n in lens]
    want, wl = m.predict_batch(prompts, length, want_logits=True)
    states = [m.state(b) for b in range(batch)]
    kv0 = [m.kv(1, w, length, seq=b) for w in (0, 1) for b in range(batch)]
    m.reset()
    got = m.predict_batch(prompts, length)
    lg = m.logits()[0]
    assert np.array_equal(got, want)
    assert [m.state(b) for b in range(batch)] == states
    assert np.abs(lg - wl[:, -1]).max() <= 1e-3
    for a, b in zip(kv0, [m.kv(1, w, length, seq=b) for w in (0, 1) for b in range(batch)]):
        assert np.abs(a - b).max() <= 2 ** -7
    m.close()


@pytest.mark.parametrize("w,batch,layers", [("f16", 3, 2), ("f16", 3, 1), ("f32", 1, 2), ("f32", 1, 1)])
@pytest.mark.parametrize("short,length", [(9, 9), (12, 12), (33, 34), (499, 501)])
def test_first_step_of_a_prompt_chunk(gpu, w, batch, layers, short, length):
    """Calls whose first step (the last one too, where the shortest prompt is as long as the call) runs as a chunk's last position up to
    its last layer: tokens, state, logits and K/V rows of the steps (bars of test_predict_batch_prompt_chunks_match_steps; fp32: sums in
    another order). 1024 wide: no small model's launch; one layer: the step runs whole; 500 positions of 3 sequences: past one attention
    block of rows."""
    from simplellminference_amd.model import LlamaModel, preset
    m = LlamaModel(config=preset("small-h128-gqa", num_hidden_layers=layers), w_dtype=w, kv_dtype=w, seed=6, batch=batch).init()
    r = np.random.default_rng(short)
    prompts = [r.integers(0, m.config.vocab_size, short + b).tolist() for b in range(batch)]
    want, wl = m.predict_batch(prompts, length, want_logits=True)
    states = [m.state(b) for b in range(batch)]
    kv0 = [m.kv(layers - 1, which, length, seq=b) for which in (0, 1) for b in range(batch)]
    m.reset()
    for _ in range(2):
        assert np.array_equal(m.predict_batch(prompts, length), want)
        assert np.abs(m.logits()[0].reshape(batch, -1) - wl[:, -1]).max() <= (1e-3 if w == "f16" else 2e-5)
        assert [m.state(b) for b in range(batch)] == states
        for a, b in zip(kv0, [m.kv(layers - 1, which, length, seq=b) for which in (0, 1) for b in range(batch)]):
            assert np.abs(a - b).max() <= (2 ** -7 if w == "f16" else 2e-5)
    m.close()
