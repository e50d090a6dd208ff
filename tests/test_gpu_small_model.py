"""The greedy loop of a small model as one launch (csrc/small_model.h) against the same model's steps, launch by launch, which
test_gpu_model.py holds to the oracle. Both compute in fp32 and differ in the order of their sums only."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _model(w, kv, **over):
    from simplellminference_amd.model import LlamaModel, preset
    return LlamaModel(config=preset("tiny-gqa", **over), w_dtype=w, kv_dtype=kv, seed=5).init()


# heads of 64 and 128, one to eight queries a kv head, widths whose rows are no whole pieces, an FFN wider than the width, heads
# that do not divide 64, a vocabulary of many more rows than a wave asks for ahead
SHAPES = {"tiny": {}, "h128": dict(head_dim=128, hidden_size=512, kv_hidden_size=256, num_attention_heads=4, num_key_value_heads=2,
                                   intermediate_size=1032, vocab_size=700),
          "h8": dict(hidden_size=512, kv_hidden_size=64, num_attention_heads=8, num_key_value_heads=1, intermediate_size=2048),
          "h6": dict(hidden_size=384, kv_hidden_size=192, num_attention_heads=6, num_key_value_heads=3, intermediate_size=520,
                     num_hidden_layers=3, vocab_size=333),
          "v20k": dict(vocab_size=20000),
          "h1": dict(hidden_size=64, kv_hidden_size=64, num_attention_heads=1, num_key_value_heads=1, intermediate_size=72,
                     num_hidden_layers=1, vocab_size=50)}


def _place(shape, w):
    """Where the loop runs: rows past 1 KiB, heavy layers and large vocabularies over all XCDs."""
    return "all" if shape in ("v20k", "h8", "w2k") or w == "f32" and shape in ("h128", "h6") else "one"


@pytest.mark.parametrize("w,kv", [("f32", "f32"), ("f16", "f16"), ("f16", "f32"), ("f32", "f16")])
@pytest.mark.parametrize("shape", SHAPES)
def test_loop_matches_steps(gpu, shape, w, kv, place=None):
    m = _model(w, kv, max_length=150, **SHAPES[shape])
    V = m.config.vocab_size
    # one step; a prompt alone; past the keys of one pass (16 to 64) and of several; up to the last position
    for n, length in ((1, 1), (3, 3), (2, 18), (7, 34), (5, 66), (4, 131), (1, 150)):
        ids = [(13 * i + n) % V for i in range(n)]
        want, wl = m.predict(ids, length, want_logits=True)
        kv_want = [m.kv(m.config.num_hidden_layers - 1, which, length) for which in (0, 1)]
        m.reset()
        for _ in range(2):
            assert np.array_equal(m.predict(ids, length), want), (n, length)
            assert m.predict_path() == (place or _place(shape, w)), (n, length)
            log = m.logits()[0]
            # fp32 sums in another order (1e-6 of the norm); an fp16 cache rounds K and V either way (2^-11 of a value)
            assert np.linalg.norm(log - wl[-1]) <= (5e-6 if kv == "f32" else 5e-4) * np.linalg.norm(wl[-1]), (n, length)
            for which in (0, 1):
                d = np.abs(m.kv(m.config.num_hidden_layers - 1, which, length) - kv_want[which]).max()
                assert d <= (2e-5 if kv == "f32" else 1e-2), (n, length, which)
        assert m.state()["pos"] == min(length, 149) and m.state()["error"] == 0
    m.close()


@pytest.mark.parametrize("w", ["f32", "f16"])
@pytest.mark.parametrize("shape", ["tiny", "h6"])
def test_wait_that_gives_up(gpu, monkeypatch, shape, w):
    """A launch whose waits give up at their first miss ends, and the call, like those after it, gives what the steps give."""
    m = _model(w, w, max_length=150, **SHAPES[shape])
    calls = [([(7 * i + n) % 300 for i in range(n)], length) for n, length in ((3, 40), (20, 150), (1, 1))]
    want = []
    for ids, length in calls:
        tok, log = m.predict(ids, length, want_logits=True)
        want.append((tok, log[-1], [m.kv(1, which, length) for which in (0, 1)]))
    m.close()
    monkeypatch.setenv("SLI_DEBUG_SMALL_SPIN", "0")
    m = _model(w, w, max_length=150, **SHAPES[shape])
    for (ids, length), (tok, log, kv) in zip(calls, want):
        assert np.array_equal(m.predict(ids, length), tok) and m.predict_path() == "steps", length
        # fp32: prompts of 9 and more run as chunks, their sums in another order
        assert np.linalg.norm(m.logits()[0] - log) <= (5e-6 if w == "f32" else 0) * np.linalg.norm(log), length
        for which in (0, 1):
            assert np.abs(m.kv(1, which, length) - kv[which]).max() <= (2e-5 if w == "f32" else 0), (length, which)
        assert m.state() == dict(m.state(), pos=min(length, 149), error=0)
    m.close()


def test_tags_that_wrap(gpu, monkeypatch):
    """Launches on both sides of the wrap of the granules' tags (36 of them a launch of 3 steps)."""
    m = _model("f32", "f32", max_length=60)
    want = [m.predict([5, 6], n, want_logits=True)[0] for n in (3, 3, 40)]
    m.close()
    monkeypatch.setenv("SLI_DEBUG_SMALL_TAG", str(2 ** 32 - 50))
    m = _model("f32", "f32", max_length=60)
    for w, n in zip(want, (3, 3, 40)):
        assert np.array_equal(m.predict([5, 6], n), w), n
        assert m.state()["error"] == 0
    m.close()


def test_context_beyond_the_loop(gpu):
    """Contexts on both sides of the rule (512 KiB of a head's keys) give the same tokens."""
    m = _model("f32", "f32", max_length=2100)
    want = m.predict([3, 1, 4], 2100, want_logits=True)[0]
    assert np.array_equal(m.predict([3, 1, 4], 2048), want[:2048])
    assert np.array_equal(m.predict([3, 1, 4], 2049), want[:2049])
    m.close()


@pytest.mark.parametrize("w", ["f32", "f16"])
@pytest.mark.parametrize("shape", SHAPES)
def test_loop_over_all_xcds(gpu, monkeypatch, shape, w):
    """As test_loop_matches_steps, where that ran on one XCD."""
    monkeypatch.setenv("SLI_DEBUG_SMALL_ALL", "1")
    test_loop_matches_steps(gpu, shape, w, w, "all")


def test_loop_of_many_units(gpu, monkeypatch):
    """An fp32 layer past what one XCD reads beside its edges."""
    monkeypatch.setitem(SHAPES, "w2k", dict(intermediate_size=2048))
    test_loop_matches_steps(gpu, "w2k", "f32", "f32")


def test_loops_side_by_side(gpu):
    """Models of both places (one XCD; all of them, fp32 wider than 256) called from threads at the same time: each gets its own
    tokens in its own place, and no launch's workgroups keep another's from running (a wait that gave up would change the place)."""
    import threading
    models, want = [], []
    for i in range(8):
        w = "f32" if i % 2 else "f16"
        m = _model(w, w, max_length=100, **(SHAPES["h6"] if i in (1, 5) else {}))
        models.append(m)
        want.append(m.predict([i + 1, 7, 300 - i], 90))
    got = [[] for _ in models]

    def calls(i):
        for _ in range(6):
            got[i].append((models[i].predict([i + 1, 7, 300 - i], 90), models[i].predict_path()))
    threads = [threading.Thread(target=calls, args=(i,)) for i in range(len(models))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i, (m, g, w) in enumerate(zip(models, got, want)):
        assert len(g) == 6 and all(np.array_equal(x, w) for x, _ in g)
        assert {p for _, p in g} == {"all" if i in (1, 5) else "one"}, i
        assert m.state()["error"] == 0
        m.close()


def test_short_calls_beside_a_long_one(gpu):
    """A loop of many steps leaves room for others: calls of 36 steps end while one of 2048 runs. (Of three models, as streams may
    share a hardware queue.)"""
    import threading
    long = _model("f16", "f16", max_length=2048, num_hidden_layers=6)
    short = [_model("f32", "f32") for _ in range(3)]
    want = [long.predict([1, 2, 3], 2048), *(m.predict([1, 2, 3], 36) for m in short)]
    got, ends = [], []
    for m, w in zip(short, want[1:]):
        t = threading.Thread(target=lambda: got.append(long.predict([1, 2, 3], 2048)))
        t.start()
        n = 0
        while t.is_alive() and n < 1000:
            assert np.array_equal(m.predict([1, 2, 3], 36), w)
            n += 1
        t.join()
        ends.append(n)
    assert max(ends) >= 20, ends
    assert len(got) == 3 and all(np.array_equal(g, want[0]) for g in got)
    assert {m.predict_path() for m in (long, *short)} == {"one"}
    for m in (long, *short):
        m.close()
