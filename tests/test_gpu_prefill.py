"""Prompt prefill (sli_model_prefill): the prompt's positions 0..n-2 run through the
layers in chunks of up to 4096 positions — every projection one MFMA GEMM over the chunk, attention
block-causal over the cache — then decoding continues from the last prompt token. The reference
teacher-forces the prompt one token per forward (model.cpp:157-165); the oracle's predict does the same, so
the bar is the oracle's predict: greedy token ids bit-exact, logits of every computed position within 1e-3,
and the K/V rows the prefill writes within the fp16 cache rounding.

The row-wise launches of a chunk run a multiple of 32 rows, and each GEMM pads them to its own tiles (32, 64, 96 or 128
chunk rows): the prompt lengths below cover padding rows, GEMMs whose last round of tiles is cut over the depth, every
tiling, and a second chunk.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ocfg(oracle, cfg):
    return oracle.Config(cfg.vocab_size, cfg.hidden_size, cfg.num_attention_heads, cfg.num_key_value_heads,
                         cfg.head_dim, cfg.intermediate_size, cfg.num_hidden_layers, cfg.max_length,
                         cfg.rms_norm_eps, cfg.rope_theta)


def _wmode(oracle, w):
    return {"f32": oracle.W_F32, "f16": oracle.W_F16, "i8": oracle.W_I8}[w]


def _pair(oracle, name, w="f16", kv="f16", seed=0, **over):
    from simplellminference_amd.model import LlamaModel, preset
    cfg = preset(name, **over)
    om = oracle.Model(_ocfg(oracle, cfg), seed=seed, wmode=_wmode(oracle, w), kv_f16=(kv == "f16"))
    gm = LlamaModel(config=cfg, w_dtype=w, kv_dtype=kv, seed=seed).init()
    return cfg, om, gm


def _prompt(n, vocab, seed=3):
    return [int(t) for t in np.random.default_rng(seed + n).integers(0, vocab, n)]


def _check(gtok, glog, otok, olog, n, tol=1e-3):
    assert np.array_equal(gtok, otok), (gtok, otok)
    assert np.isnan(glog[:n - 1]).all()
    err = np.abs(glog[n - 1:] - olog[n - 1:]).max()
    assert err <= tol, err


@pytest.mark.parametrize("name", ["tiny", "tiny-gqa"])
@pytest.mark.parametrize("n", [1, 2, 9, 33, 63])
def test_prefill_predict_matches_oracle(gpu, oracle, name, n):
    """Short prompts (n - 1 prefilled positions = 0, 1, 8, 32, 62: 32 and 64 rows, padding rows),
    then greedy up to the context end."""
    cfg, om, gm = _pair(oracle, name)
    prompt = _prompt(n, cfg.vocab_size)
    steps = 64
    otok, olog = om.predict(prompt, steps)
    gtok, glog = gm.predict_prefill(prompt, steps, want_logits=True)
    gm.close()
    om.close()
    _check(gtok, glog, otok, olog, n)


@pytest.mark.parametrize("n", [129, 200, 257, 300])
def test_prefill_long_prompts(gpu, oracle, n):
    """Prompts of 129..300 tokens: 128, 224, 256 and 320 rows, GQA."""
    cfg, om, gm = _pair(oracle, "tiny-gqa", max_length=320)
    prompt = _prompt(n, cfg.vocab_size)
    steps = n + 12
    otok, olog = om.predict(prompt, steps)
    gtok, glog = gm.predict_prefill(prompt, steps, want_logits=True)
    gm.close()
    om.close()
    _check(gtok, glog, otok, olog, n)


@pytest.mark.parametrize("n", [21, 150])
def test_prefill_kv_rows_match_oracle(gpu, oracle, n):
    cfg, om, gm = _pair(oracle, "tiny-gqa", max_length=160)
    prompt = _prompt(n, cfg.vocab_size)
    om.predict(prompt, n)
    gm.prefill(prompt)
    st = gm.state()
    assert st["pos"] == n - 1 and st["token"] == prompt[-1]
    assert np.array_equal(gm.history(0, n), prompt)
    ok, ov = om.kv_cache()
    for layer in range(cfg.num_hidden_layers):  # rows 0..n-2 come from the prefill (row n-1 from the step)
        np.testing.assert_allclose(gm.kv(layer, 0, n - 1), ok[layer, :n - 1], rtol=0, atol=2e-3)
        np.testing.assert_allclose(gm.kv(layer, 1, n - 1), ov[layer, :n - 1], rtol=0, atol=2e-3)
    gm.close()
    om.close()


def test_prefill_llama7b_shape(gpu, oracle):
    """Llama-2-7B layer shapes (2 layers, full vocab): a 40-token prompt prefilled on MFMA, then 4 greedy
    steps, against the oracle's token-by-token predict."""
    cfg, om, gm = _pair(oracle, "llama2-7b", seed=1, num_hidden_layers=2, max_length=64)
    prompt = _prompt(40, cfg.vocab_size)
    otok, olog = om.predict(prompt, 44)
    gtok, glog = gm.predict_prefill(prompt, 44, want_logits=True)
    gm.close()
    om.close()
    _check(gtok, glog, otok, olog, 40)


@pytest.mark.timeout(400)
def test_prefill_llama7b_shape_long(gpu, oracle):
    """Llama-2-7B layer shapes (2 layers; vocab cut to 512 so the CPU oracle stays in budget), a 140-token
    prompt: 139 rows, padded to 160 and to the GEMMs' tiles, hd 128, 4096 x 11008 projections."""
    cfg, om, gm = _pair(oracle, "llama2-7b", seed=1, num_hidden_layers=2, max_length=160, vocab_size=512)
    prompt = _prompt(140, cfg.vocab_size)
    otok, olog = om.predict(prompt, 144)
    gtok, glog = gm.predict_prefill(prompt, 144, want_logits=True)
    gm.close()
    om.close()
    _check(gtok, glog, otok, olog, 140)


@pytest.mark.parametrize("kv", ["f16", "f32"])
@pytest.mark.parametrize("n", [13, 150])
def test_prefill_int8(gpu, oracle, kv, n):
    """int8 weights: the GEMM converts each int8 weight image to fp16 in registers (exact) and applies the
    per-row scales in the epilogue."""
    cfg, om, gm = _pair(oracle, "tiny-gqa", w="i8", kv=kv, max_length=160)
    prompt = _prompt(n, cfg.vocab_size)
    otok, olog = om.predict(prompt, n + 10)
    gtok, glog = gm.predict_prefill(prompt, n + 10, want_logits=True)
    gm.close()
    om.close()
    _check(gtok, glog, otok, olog, n)


@pytest.mark.parametrize("over", [dict(intermediate_size=704), dict(hidden_size=320, num_attention_heads=5,
                                                                      num_key_value_heads=5, kv_hidden_size=320)])
def test_prefill_int8_half_last_stage(gpu, oracle, over):
    """int8 GEMM depths that are 64 mod 128 (the int8 pgemm stage is 128 deep): the last stage is a half stage
    (prefill.h). Llama-2-7B int8 at TP 4 has such a down projection (2752 = 21.5 x 128); here the FFN width
    704 (down) and a hidden size of 320 (q/k/v, gate/up and wo)."""
    cfg, om, gm = _pair(oracle, "tiny", w="i8", kv="f16", max_length=160, **over)
    assert gm.prefill_path() == "mfma"
    prompt = _prompt(150, cfg.vocab_size)
    otok, olog = om.predict(prompt, 160)
    gtok, glog = gm.predict_prefill(prompt, 160, want_logits=True)
    gm.close()
    om.close()
    _check(gtok, glog, otok, olog, 150)


def test_prefill_f32_weights_teacher_forces(gpu, oracle):
    """fp32 weights have no MFMA projection: the prompt runs through the decode step (same tokens)."""
    cfg, om, gm = _pair(oracle, "tiny-gqa", w="f32", kv="f32")
    assert gm.prefill_path() == "decode"
    prompt = _prompt(13, cfg.vocab_size)
    otok, olog = om.predict(prompt, 30)
    gtok, glog = gm.predict_prefill(prompt, 30, want_logits=True)
    gm.close()
    om.close()
    _check(gtok, glog, otok, olog, 13, tol=1e-4)


def test_prefill_twice_reuses_graphs(gpu, oracle):
    """A second and a third prompt on the same model, of other row counts, give the oracle's tokens too: over the first one's
    cache rows and scratch, and with the same decode graph."""
    cfg, om, gm = _pair(oracle, "tiny-gqa", max_length=320)
    for n in (70, 260, 5):
        prompt = _prompt(n, cfg.vocab_size, seed=11)
        otok, olog = om.predict(prompt, n + 6)
        gtok, glog = gm.predict_prefill(prompt, n + 6, want_logits=True)
        _check(gtok, glog, otok, olog, n)
    gm.close()
    om.close()


@pytest.mark.parametrize("name,tp,w,over", [("tiny-h8", 2, "f16", {}), ("tiny-h8", 8, "f16", {}),
                                            ("tiny-gqa-h16", 4, "i8", {}),
                                            ("tiny-gqa-h16", 4, "i8", dict(intermediate_size=2816))])
def test_prefill_tp_group(gpu, oracle, name, tp, w, over):
    """The sharded prefill (sli_tp_group_prefill): every rank's chunk GEMMs on its shard, the residual rows
    summed over the ranks after every wo and down GEMM; against the unsharded oracle. FFN 2816 at TP 4: each
    rank's int8 down projection is 704 deep, a half last stage (the Llama-2-7B int8 TP-4 case)."""
    from simplellminference_amd.model import TPGroup, preset
    cfg = preset(name, max_length=160, **over)
    g = TPGroup(cfg, tp, w_dtype=w, kv_dtype="f16", seed=2).init()
    om = oracle.Model(_ocfg(oracle, cfg), seed=2, wmode=_wmode(oracle, w), kv_f16=True)
    prompt = _prompt(140, cfg.vocab_size)
    otok, olog = om.predict(prompt, 150)
    gtok, glog = g.predict_prefill(prompt, 150, want_logits=True)
    states = [m.state() for m in g.ranks]
    g.close()
    om.close()
    assert all(s == states[0] for s in states), states
    _check(gtok, glog, otok, olog, 140)


@pytest.mark.parametrize("w", ["f16", "i8"])
@pytest.mark.parametrize("n", [34, 65, 66, 129, 130, 258, 514, 770, 1026])
def test_prefill_splits_match_decode(gpu, w, n):
    """Every row count's tilings with their last round cut over the depth (small outputs: the whole launch), a wave's and a
    workgroup's worth of padding rows, and (int8) a depth that ends in a half stage (2752 = 21.5 x 128), against the
    engine's own decode step over the same prompt. 1e-3: this file's bar; the two paths differ by where fp32 sums fall
    around the fp16 rounding of K and V."""
    from simplellminference_amd.model import LlamaModel, preset
    cfg = preset("small-h128-gqa", max_length=1088, intermediate_size=2752)
    m = LlamaModel(config=cfg, w_dtype=w, kv_dtype="f16", seed=4).init()
    prompt = _prompt(n, cfg.vocab_size)
    ref = m.predict(prompt, n + 3, want_logits=True)
    k0 = m.kv(1, 0, n), m.kv(1, 1, n)
    m.reset()
    tok, log = m.predict_prefill(prompt, n + 3, want_logits=True)
    k1 = m.kv(1, 0, n), m.kv(1, 1, n)
    m.close()
    assert np.array_equal(tok, ref[0])
    assert np.abs(log[n - 1:] - ref[1][n - 1:]).max() <= 1e-3
    for a, b in zip(k0, k1):  # one fp16 rounding of values up to 8
        assert np.abs(a - b).max() <= 2 ** -7


@pytest.mark.parametrize("n", [20, 66, 131, 200, 290])
def test_prefill_int8_half_last_stage_of_split_rings(gpu, n):
    """int8 depths that end in a half stage (1088 = 8.5 x 128, 11072 = 86.5 x 128) in the tilings whose weights have a ring of
    their own, against the decode steps; test_prefill_splits_match_decode's bounds."""
    from simplellminference_amd.model import LlamaModel, preset
    cfg = preset("tiny", max_length=320, hidden_size=1088, num_attention_heads=17, num_key_value_heads=17, kv_hidden_size=1088,
                 intermediate_size=11072)
    m = LlamaModel(config=cfg, w_dtype="i8", kv_dtype="f16", seed=6).init()
    prompt = _prompt(n, cfg.vocab_size)
    ref = m.predict(prompt, n + 3, want_logits=True)
    m.reset()
    tok, log = m.predict_prefill(prompt, n + 3, want_logits=True)
    m.close()
    assert np.array_equal(tok, ref[0])
    assert np.abs(log[n - 1:] - ref[1][n - 1:]).max() <= 1e-3


@pytest.mark.parametrize("n", [97, 98, 161, 193, 194, 290])
def test_prefill_rows_of_each_tiling(gpu, n):
    """Row counts around multiples of 96: every GEMM of a chunk pads to its own tile (96 rows where that is cheaper than 64
    or 128), so the rows that one writes and the next reads differ. A wide MLP, so that its two GEMMs take other tiles
    than the attention's; the same bounds as above."""
    from simplellminference_amd.model import LlamaModel, preset
    cfg = preset("small-h128-gqa", max_length=320, intermediate_size=14336)
    m = LlamaModel(config=cfg, w_dtype="f16", kv_dtype="f16", seed=5).init()
    prompt = _prompt(n, cfg.vocab_size)
    ref = m.predict(prompt, n + 3, want_logits=True)
    k0 = m.kv(1, 0, n), m.kv(1, 1, n)
    m.reset()
    tok, log = m.predict_prefill(prompt, n + 3, want_logits=True)
    k1 = m.kv(1, 0, n), m.kv(1, 1, n)
    m.close()
    assert np.array_equal(tok, ref[0])
    assert np.abs(log[n - 1:] - ref[1][n - 1:]).max() <= 1e-3
    for a, b in zip(k0, k1):  # one fp16 rounding of values up to 8
        assert np.abs(a - b).max() <= 2 ** -7


@pytest.mark.parametrize("hd,heads,kvh,n", [(128, 8, 1, 65), (128, 8, 2, 130), (64, 8, 4, 17), (64, 8, 8, 300), (128, 8, 2, 64),
                                            (64, 32, 32, 2050), (128, 16, 4, 2100)])
def test_prefill_attention_groups(gpu, hd, heads, kvh, n):
    """The prompt attention's heads per workgroup (1, 2, 4 of a kv head, 8 as two workgroups), 16 and (the long prompts)
    32 positions per wave, last tiles and position blocks of 1, 16 and 64 rows, against the engine's decode step. Two layers: the
    first one's attention shows in the second's cache rows, and through them in the logits. 1e-3 as above; cache rows within one
    fp16 rounding of the largest, in norm below 2^-12 (2^-11 / sqrt 3 would be every value rounded the other way)."""
    from simplellminference_amd.model import LlamaModel, LlamaModelConfig
    cfg = LlamaModelConfig(vocab_size=600, head_dim=hd, hidden_size=hd * heads, kv_hidden_size=hd * kvh,
                           intermediate_size=512, max_length=n + 8, num_hidden_layers=2, num_attention_heads=heads,
                           num_key_value_heads=kvh, rms_norm_eps=1e-5, rope_theta=1e4)
    m = LlamaModel(config=cfg, w_dtype="f16", kv_dtype="f16", seed=2).init()
    prompt = _prompt(n, cfg.vocab_size)
    ref = m.predict(prompt, n + 2)
    lref, kv = m.logits()[0], [m.kv(1, which, n - 1) for which in (0, 1)]
    m.reset()
    tok = m.predict_prefill(prompt, n + 2)
    log = m.logits()[0]
    for a, b in zip([m.kv(1, which, n - 1) for which in (0, 1)], kv):
        assert np.abs(a - b).max() <= 2.0 ** -10 * np.abs(b).max()
        assert np.linalg.norm(a - b) <= 2.0 ** -12 * np.linalg.norm(b)
    m.close()
    assert np.array_equal(tok, ref)
    assert np.abs(log - lref).max() <= 1e-3


@pytest.mark.parametrize("width,ff,n", [(4096, 192, 20), (4096, 11008, 66), (4096, 2048, 97), (4096, 11008, 128), (4096, 11008, 129),
                                        (8192, 1024, 33), (4160, 2048, 97), (2048, 8192, 66)])
def test_prefill_rotated_walk(gpu, width, ff, n):
    """Chunks of one position block at 4096 and 8192 columns, whose row blocks start apart in the depth: fewer and more of them
    than stages (64, 128), whole tiles and two splits, a last row block of a few rows; 129 positions and widths that keep the
    order. Against the decode steps: the cache rows of one layer, bounds of test_prefill_every_tiling."""
    from simplellminference_amd.model import LlamaModel, preset
    cfg = preset("tiny", max_length=160, hidden_size=width, num_attention_heads=width // 64, num_key_value_heads=width // 64,
                 kv_hidden_size=width, intermediate_size=ff)
    m = LlamaModel(config=cfg, w_dtype="f16", kv_dtype="f16", seed=8).init()
    prompt = _prompt(n, cfg.vocab_size)
    want = m.predict(prompt, n + 1)
    lw, kv = m.logits()[0], [m.kv(1, which, n) for which in (0, 1)]
    m.reset()
    got = m.predict_prefill(prompt, n + 1)
    log = m.logits()[0]
    assert np.array_equal(got, want)
    assert np.linalg.norm(log - lw) <= 8e-4 * np.linalg.norm(lw)
    for a, b in zip([m.kv(1, which, n) for which in (0, 1)], kv):
        assert np.abs(a - b).max() <= 2.0 ** -10 * np.abs(b).max()
        assert np.linalg.norm(a - b) <= 2.0 ** -12 * np.linalg.norm(b)
    m.close()


# (weights, shape, batch, prompt): between them every tiling of the prompt GEMMs runs (test_host_runtime.py looks)
TILING_SHAPES = [("f16", "llama2-7b", 1, 10), ("f16", "llama2-7b", 1, 74), ("f16", "llama2-7b", 1, 200),
                 ("f16", "llama3-8b", 1, 104), ("f16", "llama3-8b", 1, 200), ("f16", "llama2-7b", 2, 400),
                 ("i8", "llama2-7b", 1, 10), ("i8", "llama2-7b", 1, 50), ("i8", "llama2-7b", 1, 74), ("i8", "llama2-7b", 1, 130),
                 ("i8", "llama3-8b", 1, 120), ("i8", "llama3-8b", 1, 130), ("i8", "llama3-8b", 1, 200), ("f32", "llama2-7b", 1, 18),
                 ("f32", "llama2-7b", 1, 50), ("f32", "llama2-7b", 1, 74), ("f32", "llama3-8b", 1, 20), ("f32", "llama3-8b", 1, 104),
                 ("i8", "llama3-8b", 1, 10), ("i8", "small-h128", 1, 10), ("f16", "llama2-7b", 1, 800)]


def tiling_model(w, name, batch, n=400):
    from simplellminference_amd.model import LlamaModel, preset
    return LlamaModel(config=preset(name, num_hidden_layers=2, vocab_size=500, max_length=max(400, n) + 16), w_dtype=w,
                      kv_dtype="f32" if w == "f32" else "f16", seed=12, batch=batch).init()


def tiling_run(m, prompts, length, steps):
    """Prompts through the chunks, or (steps) through the decode step."""
    if m.batch > 1:
        return m.predict_batch(prompts, length, want_logits=steps)
    if steps or m.w_dtype == 0:  # (fp32: predict's chunk)
        return m.predict(prompts[0], length, want_logits=steps)
    return m.predict_prefill(prompts[0], length)


@pytest.mark.parametrize("w,name,batch,n", TILING_SHAPES)
def test_prefill_every_tiling(gpu, w, name, batch, n):
    """Two layers of real width against the decode steps: fp16 and int8 logits within the 8e-4 of their norm that an fp16
    cache's roundings either way make, fp32 within 2e-6 (sums of up to 14336 products in another order). The second layer's
    cache rows follow from the first's, whose values round either way: within one fp16 rounding of the largest, and in norm
    below 2^-12 (2^-11 / sqrt 3 would be every value rounded the other way). fp32 rows: 2^-14."""
    m = tiling_model(w, name, batch, n)
    prompts = [_prompt(n + b, m.config.vocab_size)[b:] for b in range(batch)]
    want, wl = tiling_run(m, prompts, n + 1, True)
    rows = lambda: [m.kv(1, which, n, seq=b) for b in range(batch) for which in (0, 1)]
    kv = rows()
    wl = (wl if batch == 1 else wl.swapaxes(0, 1))[-1]
    m.reset()
    got = tiling_run(m, prompts, n + 1, False)
    log = m.logits()[0]
    assert np.array_equal(got, want)
    assert np.linalg.norm(log - wl) <= (2e-6 if w == "f32" else 8e-4) * np.linalg.norm(wl)
    for a, b in zip(rows(), kv):
        d = np.abs(a - b).max()
        assert d <= (2.0 ** -14 if w == "f32" else 2.0 ** -10 * np.abs(b).max())
        assert np.linalg.norm(a - b) <= 2.0 ** -12 * np.linalg.norm(b)
    m.close()


@pytest.mark.parametrize("w", ["f16", "i8", "f32"])
def test_prefill_sums_left_to_the_norm(gpu, w):
    """wo and down of chunks up to 128 rows leave cut sums (int8: unscaled) to the next norm, of 129 rows they merge them: three
    layers, so that both hand over, in chunks on both sides. Bars as above; a third layer's cache rows follow from two."""
    from simplellminference_amd.model import LlamaModel, preset
    m = LlamaModel(config=preset("llama2-7b", num_hidden_layers=3, vocab_size=500, max_length=140), w_dtype=w,
                   kv_dtype="f32" if w == "f32" else "f16", seed=4).init()
    for n in (10, 47, 129, 130):
        prompt = _prompt(n, 500)
        want, wl = tiling_run(m, [prompt], n + 1, True)
        kv = [m.kv(2, which, n) for which in (0, 1)]
        m.reset()
        got = tiling_run(m, [prompt], n + 1, False)
        assert np.array_equal(got, want), n
        assert np.linalg.norm(m.logits()[0] - wl[-1]) <= (2e-6 if w == "f32" else 8e-4) * np.linalg.norm(wl[-1]), n
        for which in (0, 1):
            a, b = m.kv(2, which, n), kv[which]
            assert np.linalg.norm(a - b) <= 2.0 ** -11 * np.linalg.norm(b), n
        m.reset()
    m.close()


@pytest.mark.parametrize("w,kv", [("f16", "f16"), ("i8", "f16"), ("f16", "f32"), ("f32", "f32"), ("f32", "f16")])
@pytest.mark.parametrize("n", [4098, 4130])
def test_prompt_past_one_chunk(gpu, w, kv, n):
    """Prompts of 4097 and 4129 positions: a second chunk of 1 and of 33 rows, whose queries see the first one's cache rows.
    The bars of this file (fp32: 1e-4)."""
    from simplellminference_amd.model import LlamaModel, preset
    m = LlamaModel(config=preset("tiny-gqa", max_length=4200), w_dtype=w, kv_dtype=kv, seed=3).init()
    prompt = _prompt(n, m.config.vocab_size)
    want = m.predict_prefill(prompt, n + 6) if w == "f32" else m.predict(prompt, n + 6)  # the decode steps
    log, rows = m.logits()[0], [m.kv(1, which, n)[4090:] for which in (0, 1)]
    m.reset()
    got = m.predict(prompt, n + 6) if w == "f32" else m.predict_prefill(prompt, n + 6)
    assert np.array_equal(got, want)
    assert np.abs(m.logits()[0] - log).max() <= (1e-4 if (w, kv) == ("f32", "f32") else 1e-3)
    for a, b in zip([m.kv(1, which, n)[4090:] for which in (0, 1)], rows):
        assert np.abs(a - b).max() <= (1e-4 if kv == "f32" and w == "f32" else 2 ** -7)
    m.close()


def test_prompt_past_one_chunk_tp_group(gpu):
    """The same of an in-process group of two ranks, against one rank."""
    from simplellminference_amd.model import LlamaModel, TPGroup, preset
    cfg, n = preset("tiny-gqa", max_length=4200), 4130
    prompt = _prompt(n, cfg.vocab_size)
    m = LlamaModel(config=cfg, w_dtype="f16", kv_dtype="f16", seed=3).init()
    want = m.predict_prefill(prompt, n + 6)
    m.close()
    g = TPGroup(cfg, 2, w_dtype="f16", kv_dtype="f16", seed=3).init()
    got = g.predict_prefill(prompt, n + 6)
    g.close()
    assert np.array_equal(np.asarray(got).reshape(-1)[:n + 6], want)
