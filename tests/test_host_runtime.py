"""The engine's host side on a HIP runtime of host memory (cpp/host_hip.cpp): kernels do nothing, so results mean nothing;
what is checked is which device is current, what is allocated, launched and replayed, and what a call leaves behind.

Each case runs in a process of its own (the runtime replaces HIP for the whole process): ``python test_host_runtime.py CASE``.
"""
import ctypes
import os
import re
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB = os.path.join(HERE, "cpp", "_build", "libhost_hip.so")


def _llama(**kw):
    from simplellminference_amd.model import LlamaModel, preset
    return LlamaModel(config=preset(kw.pop("preset", "tiny-gqa"), **kw.pop("over", {})), seed=1, **kw).init()


def _prompts(m, n):
    return [[(7 * b + i) % m.config.vocab_size for i in range(n)] for b in range(m.batch)]


# ---------------------------------------------------------------- cases (in the child)
def device_of_predict(H):
    """predict and predict_batch of a model on device 1 from a thread whose device is 0: what they allocate is on device 1,
    what they launch is launched there, and the thread's device is what it was."""
    for kw in (dict(w_dtype="f32", kv_dtype="f32"), dict(w_dtype="f16", batch=2)):
        m = _llama(device=1, **kw)
        H.hipSetDevice(0)
        before = H.hh_mallocs_on(0), H.hh_attributes_on(0), H.hh_mallocs_on(1)
        m.predict_batch(_prompts(m, 20), 24)
        assert H.hh_mallocs_on(1) > before[2], "the call allocates its scratch"
        assert (H.hh_mallocs_on(0), H.hh_attributes_on(0)) == before[:2], "memory or attributes of the other device"
        d = ctypes.c_int(-1)
        H.hipGetDevice(ctypes.byref(d))
        assert d.value == 0, "the caller's device"
        H.hipSetDevice(0)
        m.set_state_seq(0, 1, 0)
        m.step()
        m.close()
    assert H.hh_wrong_device() == 0, "launches on a stream of another device"


CHUNK_CALLS = [(dict(w_dtype="f32", kv_dtype="f32"), lambda m: m.predict_batch(_prompts(m, 20), 24)),
               (dict(w_dtype="f16", batch=2), lambda m: m.predict_batch(_prompts(m, 20), 24)),
               (dict(w_dtype="f16"), lambda m: m.prefill(_prompts(m, 20)[0])),
               (dict(w_dtype="i8"), lambda m: m.predict_prefill(_prompts(m, 20)[0], 24))]


def scratch_that_does_not_fit(H):
    """Every allocation of the chunks' scratch in turn fails: the call runs (through the steps, which need none), nothing of
    the scratch is left, and the next call allocates all of it."""
    for kw, call in CHUNK_CALLS:
        m = _llama(**kw)
        had = H.hh_mallocs()
        call(m)
        n = H.hh_mallocs() - had
        assert n >= 5
        m.close()
        for k in range(n):
            m = _llama(**kw)
            live = H.hh_live()
            H.hh_fail_at(k)
            steps = H.hh_graph_launches()
            call(m)
            assert H.hh_live() == live and H.hh_graph_launches() - steps >= 19
            had = H.hh_mallocs()
            call(m)
            assert (H.hh_mallocs() - had, H.hh_live() - live) == (n, n)
            m.close()
    assert H.hh_live() == 0


def scratch_of_smaller_chunks(H):
    """Scratch for 4096 positions does not fit, for 1024 it does: chunks of 1024. Ranks in one process agree on the chunks."""
    from simplellminference_amd.model import TPGroup, preset
    over = dict(max_length=4500)
    for kw, call in CHUNK_CALLS:
        launches = []
        for room in (0, 80 << 20):  # (64 MB of it for the partial sums)
            m = _llama(over=over, **kw)
            H.hh_room(room)
            ids = _prompts(m, 4200)
            had, steps = H.hh_launches(), H.hh_graph_launches()
            if "f32" in kw.values() or m.batch > 1:
                m.predict_batch(ids, 4201)
            else:
                m.prefill(ids[0])
            launches.append(H.hh_launches() - had)
            assert H.hh_graph_launches() - steps <= 2, "the prompt ran as steps"
            H.hh_room(0)
            m.close()
        assert launches[1] > 2 * launches[0], launches
    g = TPGroup(preset("tiny-gqa", **over), 2, w_dtype="f16", seed=1).init()
    had, steps = H.hh_launches(), H.hh_graph_launches()
    H.hh_room(160 << 20)  # the second rank's are the smaller ones
    g.prefill([1] * 4200)
    H.hh_room(0)
    assert H.hh_graph_launches() == steps and H.hh_launches() - had > 4 * 2 * 2 * 2 * 5, "five chunks of both ranks"
    g.close()
    assert H.hh_live() == 0


def callers_arrays_are_read(H):
    """When a call that takes prompts returns, nothing is still to be copied out of the caller's arrays."""
    from simplellminference_amd.model import TPGroup, preset
    from simplellminference_amd.stack import BlockSpec, StackModel, StackSpec
    for kw in (dict(w_dtype="f32", kv_dtype="f32"), dict(w_dtype="f16")):
        m = _llama(**kw)
        for n in (1, 2, 20):
            m.prefill(_prompts(m, n)[0])
            assert H.hh_pending_host_reads() == 0, (kw, n)
            m.set_prompt(_prompts(m, n)[0])
            assert H.hh_pending_host_reads() == 0, (kw, n)
        m.close()
        g = TPGroup(preset("tiny-gqa"), 2, seed=1, **kw).init()
        for n in (1, 20):
            g.prefill([1] * n)
            assert H.hh_pending_host_reads() == 0, ("group", kw, n)
        g.close()
    b = BlockSpec("attention", 2, 64, 64, kv_heads=1, scale=0.125, ff=128, ff_limit=7.0)
    m = StackModel(StackSpec(64, 128, (b,) * 2, max_length=64), batch=2, seed=1).init()
    for lens in ((1, 1), (1, 5), (3, 4)):
        P = (ctypes.c_int32 * 10)(*range(10))
        from simplellminference_amd._lib import call
        call("sli_model_prefill_batch", m._h, P, (ctypes.c_int32 * 2)(*lens), 5)
        assert H.hh_pending_host_reads() == 0, ("stack", lens)
    m.close()


def small_stacks_replay_their_prompts(H):
    """A prompt pass of a small block stack launches the first time its row count comes and is a graph from then on; a large one
    always launches."""
    from simplellminference_amd.stack import BlockSpec, StackModel, StackSpec

    def spec(D, arrangement):
        b = dict(parallel=BlockSpec("attention", D // 64, 64, 64, kv_heads=D // 128, scale=0.125, ff=D, ff_limit=7.0),
                 sequential=BlockSpec("latent", D // 64, 64, 64, scale=0.125, kv_rank=64, window=32, ff=D, experts=4, top=2))
        return StackSpec(64, D, (b[arrangement],) * 2, max_length=300, arrangement=arrangement,
                         positions=300 if arrangement == "sequential" else 0)
    for arrangement, D, small in (("parallel", 256, True), ("sequential", 256, True), ("parallel", 3072, False)):
        m = StackModel(spec(D, arrangement), batch=2, seed=1).init()
        for n in (20, 100, 200):
            counts = []
            for _ in range(3):
                had = H.hh_launches(), H.hh_graph_launches()
                m.feed([0], [0], [[1] * n])
                counts.append((H.hh_launches() - had[0], H.hh_graph_launches() - had[1]))
            assert counts[0][0] > 10 and counts[0][1] == 0
            assert counts[1:] == ([(0, 1)] * 2 if small else [counts[0]] * 2), (arrangement, D, n, counts)
        m.close()


def small_models_predict_in_one_launch(H):
    """predict of a narrow model without logits is one launch; a wider one, a long context and int8 weights take the steps, and so
    does one whose vocabulary or feed-forward is too wide for what its layers save."""
    wide = dict(hidden_size=512, num_attention_heads=8, num_key_value_heads=8, kv_hidden_size=512, intermediate_size=1024)
    odd = dict(hidden_size=320, num_attention_heads=5, num_key_value_heads=5, kv_hidden_size=320, intermediate_size=2048, num_hidden_layers=3)
    for kw, n, steps in ((dict(w_dtype="f32", kv_dtype="f32"), 30, 0), (dict(w_dtype="f16"), 30, 0), (dict(w_dtype="i8"), 30, 30),
                         (dict(w_dtype="f16", preset="tiny-h8"), 30, 0), (dict(w_dtype="f16", preset="small-h128"), 30, 30),
                         (dict(w_dtype="f32", kv_dtype="f32", over=dict(max_length=2100)), 2049, 2049),
                         (dict(w_dtype="f32", kv_dtype="f32", over=dict(vocab_size=20000)), 30, 0),
                         (dict(w_dtype="f32", kv_dtype="f32", over=dict(vocab_size=32000)), 30, 30),
                         (dict(w_dtype="f32", kv_dtype="f32", over=dict(vocab_size=32000, num_hidden_layers=8)), 30, 0),
                         (dict(w_dtype="f32", kv_dtype="f32", over=dict(vocab_size=20000, max_length=2048)), 2048, 2048),
                         (dict(w_dtype="f32", kv_dtype="f32", over=dict(wide, vocab_size=8192)), 30, 0),
                         (dict(w_dtype="f32", kv_dtype="f32", over=dict(wide, vocab_size=32000)), 30, 30),
                         (dict(w_dtype="f16", over=dict(wide, vocab_size=128256, num_hidden_layers=8)), 30, 30),
                         (dict(w_dtype="f32", kv_dtype="f32", over=odd), 30, 30)):
        m = _llama(**kw)
        had = H.hh_graph_launches()
        m.predict([1, 2, 3], n)
        assert H.hh_graph_launches() - had == steps, (kw, n)
        m.close()


def small_models_on_one_xcd(H):
    """The loop's place by the model's sizes; a launch that did nothing (all of these, as kernels do nothing here) is not taken for its
    result but goes over all XCDs, and one that failed leaves no tickets to the next."""
    from simplellminference_amd import _lib
    H.hh_xcds(1)
    loops = lambda: set(re.findall(r"small_predict_kernelI\w+?Li(?:64|128)ELi(\d+)ELb([01])E", H.hh_launched().decode()))
    one, over_all = ("16", "1"), ("8", "0")
    wide = dict(hidden_size=512, num_attention_heads=8, num_key_value_heads=4, kv_hidden_size=256, intermediate_size=1536)
    for w, over, place in (("f32", {}, one), ("f16", {}, one), ("f32", dict(vocab_size=4096), one), ("f32", dict(vocab_size=20000), over_all),
                           ("f16", dict(vocab_size=20000), over_all), ("f32", dict(vocab_size=20000, num_hidden_layers=12), one),
                           ("f32", dict(intermediate_size=2048), over_all), ("f32", wide, over_all), ("f16", wide, one),
                           ("f16", dict(wide, vocab_size=4096), over_all)):
        m = _llama(w_dtype=w, kv_dtype=w, over=over)
        H.hh_launched()
        for again in range(2):
            steps = H.hh_graph_launches()
            m.predict([1, 2, 3], 30)
            # (a launch over all XCDs is not asked whether it ran)
            assert loops() == ({one, over_all} if place == one and not again else {over_all}), (w, over, again)
            assert m.predict_path() == "all" and H.hh_graph_launches() == steps, (w, over, again)
        m.close()
    m = _llama(w_dtype="f32", kv_dtype="f32")
    had = H.hh_memsets()
    H.hh_fail_launch(b"small_predict_kernel")
    try:
        m.predict([1, 2, 3], 30)
        assert False, "the launch's error"
    except _lib.SliError:
        pass
    assert H.hh_memsets() == had
    m.predict([1, 2, 3], 30)
    assert H.hh_memsets() == had + 1, "the tickets"
    m.close()
    assert H.hh_live() == 0


def batched_inputs_share_a_launch(H):
    """A decode pass of a block with a feed-forward projects both of its inputs in one launch; without one there is one input."""
    from simplellminference_amd.stack import BlockSpec, StackModel, StackSpec
    for ff, want in ((300, "BgPair2"), (0, "BgPair")):
        b = BlockSpec("attention", 5, 64, 64, kv_heads=1, scale=0.1, ff=ff, ff_limit=7.0)
        m = StackModel(StackSpec(64, 256, (b,) * 2, taps=4, max_length=32), batch=3, seed=1).init()
        H.hh_launched()
        m.feed(range(3), [0] * 3, [[1]] * 3, [[0]] * 3)
        ran = set(re.findall(r"bgemm_kernelINS_\d+(BgPair2?)INS_4HyIn", H.hh_launched().decode()))
        assert ran == {want}, (ff, ran)
        m.close()


def weight_copies_where_they_are_read(H):
    """Stacks allocate the batched projections' copies of their weights (the blocks' and the head's, an allocation each) in the first
    pass that reads them: not at creation, not for prompts, single rows and steps of more than 8 sequences, and not where they are
    more than a quarter of the free memory or the allocation fails."""
    from simplellminference_amd.stack import BlockSpec, StackModel, StackSpec
    b = BlockSpec("attention", 4, 64, 64, kv_heads=2, scale=0.1, ff=300, ff_limit=7.0)

    def copies(m, call):
        had = H.hh_mallocs()
        H.hh_launched()
        call()
        return H.hh_mallocs() - had, len(re.findall("bg_tile_kernel", H.hh_launched().decode()))  # (each instance once)

    def rows(m, n, pos, wanted=True):
        return lambda: m.feed(range(n), [pos] * n, [[1]] * n, [[0]] * n if wanted else None)

    def model(batch, width=256):
        return StackModel(StackSpec(64, width, (b,) * 2, taps=4, max_length=64), batch=batch, seed=1).init()
    m = model(3)
    assert copies(m, lambda: m.feed([0, 1], [0, 0], [[1] * 20] * 2)) == (0, 0)
    assert copies(m, rows(m, 1, 20)) == (0, 0)
    assert copies(m, lambda: m.feed([0, 1], [0, 0], [[1] * 20] * 2, [[0, 5], [1]])) == (1, 1), "the head of three rows"
    assert copies(m, rows(m, 2, 20)) == (1, 2), "the blocks' two matrices"
    assert copies(m, rows(m, 3, 21)) == (0, 0)
    m.set_tensor("l0.mix.o", np.zeros((256, 256), np.float32))
    assert copies(m, rows(m, 2, 22)) == (0, 3)
    m.close()
    for batch, want in ((1, (0, 0)), (2, (2, 3)), (8, (2, 3)), (9, (0, 0))):
        m = model(batch)
        assert copies(m, m.step) == want, batch
        m.close()
    m = model(2)
    H.hh_fail_at(0)
    assert copies(m, rows(m, 2, 0)) == (2, 1), "the blocks' failed, the head's did not"
    H.hh_fail_at(-1)
    assert copies(m, rows(m, 2, 1)) == (0, 0)
    m.close()
    m = model(2)
    H.hh_free(2 << 20)  # (more than the blocks' 1.7 MB, of which it is not four times as much)
    assert copies(m, rows(m, 2, 0)) == (1, 1)
    H.hh_free(0)
    m.close()
    assert H.hh_live() == 0


def attention_forms_of_a_prompt_pass(H):
    """Prompt attention of a block stack: passes of few rows by 16 of them, others the flash form, wide where it fills the chip; one
    graph a form."""
    from simplellminference_amd.stack import BlockSpec, StackModel, StackSpec

    def forms(m, slots, start, n):
        H.hh_launched()
        m.feed(range(slots), [start] * slots, [[1] * n] * slots)
        return set(re.findall(r"(pf_flash_kernelILi\d+ELi\dELi2ELb1E|pf_attn_mfma_kernelILi\d+ELb0E)", H.hh_launched().decode()))
    for hd, heads, kv, cases in ((64, 32, 8, ((2, 9, 0, "16"), (1, 512, 0, "16"), (1, 512, 1500, "16"), (1, 513, 0, "1"), (1, 1920, 0, "1"),
                                              (1, 1921, 0, "2"), (3, 170, 0, "1"))),
                                 (128, 32, 32, ((8, 32, 1000, "16"), (1, 256, 0, "16"), (1, 257, 0, "1"), (1, 2048, 0, "2"))),
                                 (128, 8, 1, ((1, 1024, 0, "16"), (1, 1025, 0, "1")))):
        b = BlockSpec("attention", heads, hd, hd, kv_heads=kv, scale=0.1)
        m = StackModel(StackSpec(64, 3072, (b,) * 2, taps=4, max_length=2080), batch=8, seed=1).init()
        for slots, n, start, form in cases:
            want = f"pf_attn_mfma_kernelILi{hd}ELb0E" if form == "16" else f"pf_flash_kernelILi{hd}ELi{form}ELi2ELb1E"
            assert forms(m, slots, start, n) == {want}, (hd, heads, kv, slots, n, start)
        m.close()
    b = BlockSpec("attention", 48, 128, 16, kv_heads=48, scale=0.1)
    m = StackModel(StackSpec(64, 64, (b,), taps=4, max_length=300), batch=8, seed=1).init()
    for again in range(2):  # 256 rows both: each form launches once, then is a graph
        for slots, n in ((8, 2), (1, 250)):
            had = H.hh_graph_launches()
            ran = forms(m, slots, 0, n)
            assert len(ran) == 1 and H.hh_graph_launches() - had == again, (slots, n, again, ran)
    m.close()


def _tilings(names, epilogue=""):
    """(weight type, tiling) of the prompt GEMM instances among kernel names, of one epilogue or all."""
    out = set()
    for n in names.decode().split():
        if epilogue not in n:
            continue
        g = re.search(r"pgemm_kernel.*PgCfgI((?:L[ib]\d+E)+)E+(a|f|6__half|DF16_|S\d*_)EE", n)
        if g:
            cfg = tuple(int(v) for v in re.findall(r"L[ib](\d+)E", g[1]))
            if not cfg[6]:  # (not the grouped ones: the expert rows' and the latent expansion's)
                out.add((g[2] if g[2] in "af" else "half", cfg))
    return out


def every_tiling_is_tested(H):
    """The shapes that the GPU tests name run every tiling that the library holds."""
    from tests import test_gpu_prefill as P, test_gpu_stack as S
    H.hh_launched()
    run = set()
    for w, name, batch, n in P.TILING_SHAPES:
        m = P.tiling_model(w, name, batch, n)
        H.hh_launched()
        P.tiling_run(m, [[1] * n] * batch, n + 1, False)
        run |= _tilings(H.hh_launched())
        m.close()
    for model, rows in ((S.wide_model, S.TILING_ROWS), (S.middle_model, [700])):
        m = model()
        for n in rows:
            H.hh_launched()
            m.feed([0], [0], [[1] * n])
            run |= _tilings(H.hh_launched())
        m.close()
    held = _tilings(H.hh_kernels())
    assert len(held) > 20 and run == held, sorted(held - run)


# Output GEMMs of block stacks (width, heads of 128, feed-forward) at prompts of n rows, padded to 128: the (BM, WR, AT) of the
# tilings within 3 % of the fastest, each at its best split. us: 3072 x 11264 at 768 rows 75.8, others 86 and more; at 896 rows
# 79.4 and 91.
STACK_TILES = {((3072, 24, 8192), 700): {(128, 4, 2)}, ((3072, 24, 8192), 800): {(128, 4, 2)}}


def stack_prompts_take_the_fast_tilings(H):
    """The plan of a stack's output GEMM takes a tiling that was within 3 % of the fastest."""
    from simplellminference_amd.stack import BlockSpec, StackModel, StackSpec
    for ((D, heads, ff), n), fast in STACK_TILES.items():
        b = BlockSpec("attention", heads, 128, 128, kv_heads=heads, scale=0.1, ff=ff, ff_limit=7.0)
        m = StackModel(StackSpec(64, D, (b,), taps=4, max_length=1500), batch=1, seed=1).init()
        H.hh_launched()
        m.feed([0], [0], [[1] * n])
        ran = _tilings(H.hh_launched(), "HyOut")
        assert len(ran) == 1 and {(c[0], c[1], c[3]) for _, c in ran} <= fast, (D, n, ran)
        m.close()


# Input GEMMs of 2048-wide blocks with 8192 units: (block, prompt) -> (BM, WR, AT). A tiling and its cuts set the order of the sums,
# so they are part of what a prompt's rows are; each of these would be another one at half the price of the looped epilogue, or with
# rows to spare.
STACK_IN_TILES = {("attention", 20): (32, 2, 2), ("attention", 120): (128, 4, 2), ("attention", 500): (128, 4, 2),
                  ("attention", 620): (128, 4, 2), ("retention", 380): (128, 4, 2), ("retention", 1100): (128, 4, 4)}


def stack_inputs_keep_their_sums(H):
    """The input GEMM of a stack's prompt runs the tiling, and so the order of sums, that its price gives."""
    from simplellminference_amd.stack import BlockSpec, StackModel, StackSpec
    blocks = dict(attention=BlockSpec("attention", 32, 64, 64, kv_heads=8, scale=0.125, ff=8192, ff_limit=7.0),
                  retention=BlockSpec("retention", 8, 128, 256, decay=(0.9,) * 8, rot_dims=128, rot_base=1e4, ff=8192, ff_limit=7.0))
    for kind, b in blocks.items():
        m = StackModel(StackSpec(64, 2048, (b,), taps=4, max_length=1200), batch=1, seed=1).init()
        for (k, n), tiling in STACK_IN_TILES.items():
            if k == kind:
                H.hh_launched()
                m.feed([0], [0], [[1] * n])
                ran = {(c[0], c[1], c[3]) for _, c in _tilings(H.hh_launched(), "HyIn")}
                assert ran == {tiling}, (kind, n, ran)
        m.close()


# Prompts of Llama-2-7B: (weights, positions through the chunk, epilogue) -> (BM, WR, AT) of the tilings, each within 4 % of the
# fastest at its best split. us of that tiling | of the one that stale stage times took: fp16 512 rows wo 39 | 43, down 79 | 103;
# 64 rows down 28 | 33; int8 96 rows gate/up 45 | 54; fp32 512 rows gate/up 1024 | 1350, 96 rows gate/up 238 | 294
PROMPT_TILES = {("f16", 512, "PgEpiResid"): {(128, 4, 2), (128, 4, 4)}, ("f16", 64, "PgEpiResid"): {(32, 2, 2), (64, 4, 2)},
                ("i8", 96, "PgEpiSwiGLU"): {(96, 4, 3)}, ("f32", 512, "PgEpiSwiGLU"): {(128, 4, 2)},
                ("f32", 96, "PgEpiSwiGLU"): {(32, 2, 4)}}


def prompts_take_the_fast_tilings(H):
    """The plans of a prompt's GEMMs take tilings that were within 4 % of the fastest."""
    from tests import test_gpu_prefill as P
    from simplellminference_amd.model import LlamaModel, preset
    for (w, n, epi), fast in PROMPT_TILES.items():
        m = LlamaModel(config=preset("llama2-7b", num_hidden_layers=1, vocab_size=500, max_length=600), w_dtype=w,
                       kv_dtype="f32" if w == "f32" else "f16", seed=1).init()
        H.hh_launched()
        P.tiling_run(m, [[1] * (n + 1)], n + 1, False)
        ran = {(c[0], c[1], c[3]) for _, c in _tilings(H.hh_launched(), epi)}
        assert ran == fast, (w, n, epi, ran)
        m.close()


# Prompts -> whether predict runs their first step as one more row of the chunk: (preset, weights, cache, batch) -> (taken, left). ms of a
# call with the row | with the step: fp32 65 tokens 29.2 | 26.7, 129 40.5 | 36.3, 193 50.4 | 46.8, 257 62.6 | 55.3, 33 22.1 | 22.7, 64 22.3 |
# 26.7; eight of 8B 33 tokens 18.5 | 18.3, 81 28.2 | 27.7, 129 37.2 | 35.6, 49 21.0 | 21.7, 121 32.7 | 35.6; with a fp32 cache 65 tokens
# 34.2 | 25.4, 129 49.3 | 38.0, 66 34.2 | 37.8; three of 8B 33 tokens 14.1 | 15.1, 129 20.0 | 21.1
FIRST_STEPS = {("llama2-7b", "f32", "f32", 1): ((9, 32, 33, 64, 66, 75, 97, 128, 130), (65, 129, 193, 257, 385)),
               ("llama3-8b", "f16", "f16", 8): ((16, 17, 32, 34, 49, 64, 97, 121, 128), (33, 81, 129, 257)),
               ("llama3-8b", "f16", "f32", 8): ((33, 64, 66, 128), (65, 129, 257)),
               ("llama3-8b", "f16", "f16", 3): ((16, 33, 65, 129), ())}


def first_steps_join_the_chunk_where_they_pay(H):
    """predict runs its first step in the prompt's chunk, but not where the row opens a tile that costs more than the step."""
    from simplellminference_amd.model import LlamaModel, preset
    for (name, w, kv, batch), (taken, left) in FIRST_STEPS.items():
        m = LlamaModel(config=preset(name, num_hidden_layers=2, vocab_size=500, max_length=400), w_dtype=w, kv_dtype=kv, seed=1,
                       batch=batch).init()
        for n in taken + left:
            H.hh_launched()
            had = H.hh_graph_launches()
            m.predict_batch(_prompts(m, n), n + 2)
            joined = b"pf_last_rows_kernel" in H.hh_launched()
            assert joined == (n in taken) and H.hh_graph_launches() - had == 3 - joined, (name, w, kv, batch, n, joined)
        m.close()


def short_prompts_sum_in_short_chains(H):
    """GEMMs that sum in one chain over the depth: none up to 769 tokens, gate/up alone up to 1537, then down too."""
    from simplellminference_amd.model import LlamaModel, preset
    m = LlamaModel(config=preset("llama2-7b", num_hidden_layers=1, vocab_size=500, max_length=2100), seed=1).init()
    chain = lambda names, epi: any(c[3] == 4 and c[5] == 2 and not c[7] for _, c in _tilings(names, epi))
    for n, gate_up, down in ((513, False, False), (701, False, False), (769, False, False), (1025, True, False),
                             (1537, True, False), (2049, True, True)):
        H.hh_launched()
        m.prefill([1] * n)
        names = H.hh_launched()
        assert (chain(names, "PgEpiSwiGLU"), chain(names, "PgEpiResid"), chain(names, "PgEpiQKV")) == (gate_up, down, False), n
    m.close()


def fp32_output_projection_steps(H):
    """A fp32 output projection reads 8 vectors a lane and step only where a wave has two whole such steps (of 2048 columns):
    one rank of 4096 columns, not the ranks of 512 to 2048 of a group, nor a width that they do not divide."""
    from simplellminference_amd.model import LlamaModel, TPGroup, preset
    kw = dict(w_dtype="f32", kv_dtype="f32", seed=1)
    steps = lambda: set(re.findall(r"gemv_kernelIfLi1ELi(\d)ELb1ENS_8EpiStore", H.hh_launched().decode()))
    for heads, tp, want in ((32, 1, 8), (32, 2, 2), (32, 8, 2), (24, 1, 2), (64, 4, 8), (64, 8, 2)):
        cfg = preset("tiny", max_length=2048, vocab_size=64, head_dim=128, hidden_size=128 * heads, num_attention_heads=heads,
                     num_key_value_heads=heads, kv_hidden_size=128 * heads, num_hidden_layers=1, intermediate_size=256)
        H.hh_launched()
        if tp == 1:
            m = LlamaModel(config=cfg, **kw).init()
            m.step()
        else:
            m = TPGroup(cfg, tp, **kw).init()
            m.step()
        # (a down projection's steps are 6)
        assert {int(v) for v in steps()} - {6, 1} == {want}, (heads, tp, want)
        m.close()


def steps_of_the_batched_projection(H):
    """The shapes that the GPU tests name run the steps that they name."""
    from simplellminference_amd import _lib
    from tests import test_gpu_batch as B, test_gpu_stack as S
    ran = lambda tag: {int(v) for v in re.findall(r"bgemm_kernel\w*" + tag + r"\w*?ELb0ELi(\d)E", H.hh_launched().decode())}
    H.hh_launched()
    for (rows, cols, batch), step in B.STEP_SHAPES.items():
        n = _lib.load().sli_matmul_batch_workspace_bytes(rows, cols, batch)
        buf = [ctypes.c_void_p() for _ in range(4)]
        for p, size in zip(buf, (4 * batch * cols, 2 * rows * cols, 4 * batch * rows, n)):
            assert H.hipMalloc(ctypes.byref(p), ctypes.c_size_t(size)) == 0
        x, w, y, ws = buf
        _lib.call("sli_matmul_batch", x, w, _lib.DT_F16, y, rows, cols, batch, ws, n, None)
        assert ran("BgEpiStore") == {step}, (rows, cols, batch)
        for p in buf:
            H.hipFree(p)
    for batch in (2, 6, 8):
        m = S.narrow_model(batch)
        H.hh_launched()
        m.feed(range(batch), [0] * batch, [[1]] * batch, [[0]] * batch)
        assert ran("HyOut") == {5}, batch
        m.close()


# ---------------------------------------------------------------- the tests
CASES = ["device_of_predict", "scratch_that_does_not_fit", "scratch_of_smaller_chunks",
         "callers_arrays_are_read", "small_stacks_replay_their_prompts", "small_models_predict_in_one_launch", "small_models_on_one_xcd",
         "batched_inputs_share_a_launch", "attention_forms_of_a_prompt_pass", "weight_copies_where_they_are_read",
         "every_tiling_is_tested", "stack_prompts_take_the_fast_tilings", "stack_inputs_keep_their_sums", "prompts_take_the_fast_tilings",
         "first_steps_join_the_chunk_where_they_pay", "short_prompts_sum_in_short_chains",
         "fp32_output_projection_steps", "steps_of_the_batched_projection"]


@pytest.fixture(scope="module")
def host_hip():
    from simplellminference_amd import build
    build.ensure()
    os.makedirs(os.path.dirname(LIB), exist_ok=True)
    src = os.path.join(HERE, "cpp", "host_hip.cpp")
    part = f"{LIB}.{os.getpid()}"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", src, "-o", part], check=True)
    os.replace(part, LIB)
    return LIB


@pytest.mark.parametrize("case", CASES)
def test_host(host_hip, case):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), case], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


if __name__ == "__main__":
    sys.path.insert(0, ROOT)
    H = ctypes.CDLL(LIB, mode=ctypes.RTLD_GLOBAL)  # before libsli.so: its references to HIP end here
    H.hh_room.argtypes = H.hh_free.argtypes = [ctypes.c_size_t]
    H.hh_launched.restype = H.hh_kernels.restype = ctypes.c_char_p
    globals()[sys.argv[1]](H)
    print("ok", sys.argv[1])
