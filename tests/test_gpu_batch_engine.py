"""Batched decode (zh_engine_generate_batch): several sequences over one copy
of the weights step in lockstep, the projections as batched DMMV launches.

Each sequence must decode exactly as it does alone (generate() on its own
engine: the single-sequence path that test_gpu_engine.py pins token-exact to
the oracle), and its last logits must agree with that run's within the DMMV
tolerance (the batched path stages the SwiGLU output from f32 where the
single path copies its XQ image, so the last bits may differ)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# Q4_K_M-style mix: attn_v / ffn_down Q6_K on the use_more_bits layers, so
# the Q/K/V launches split into runs of equal types; K = 1024 / 2048 keep the
# Q6_K rows 16-byte multiples (the Q6_K tile kernels)
CFG = dict(n_layers=4, hidden=1024, n_heads=8, n_kv_heads=2, head_dim=128, ffn=2048, vocab=4096,
           n_experts=0, n_experts_used=0, expert_ffn=0, max_ctx=512, type_attn=12, type_ffn_gate_up=12,
           type_ffn_down=12, type_lm_head=14, type_embd=12, type_router=8, type_more_bits=14,
           rope_base=1e6, eps=1e-6, seed=57)


@pytest.fixture(scope="module")
def ctx():
    import zinc_amd
    c = zinc_amd.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n_seq", [3, 4, 6])
def test_batch_matches_single_sequences(ctx, n_seq):
    import zinc_amd
    print(f"batch engine n_seq={n_seq}", flush=True)
    base = zinc_amd.InferenceEngine(ctx, CFG)
    engines = [base] + [base.share(ctx) for _ in range(n_seq - 1)]
    rng = np.random.default_rng(n_seq)
    prompts = rng.integers(0, CFG["vocab"], (n_seq, 5)).astype(np.uint32)
    prefill, steps = 40, 12
    solo, solo_logits = [], []
    for v, e in enumerate(engines):
        e.prefill_kv_random(prefill, 100 + v)
        solo.append(e.generate(prompts[v].tolist(), steps, start_pos=prefill))
        solo_logits.append(e.logits())
    for v, e in enumerate(engines):
        e.prefill_kv_random(prefill, 100 + v)
    got = zinc_amd.InferenceEngine.generate_batch(engines, prompts, steps, start_pos=prefill)
    for v, e in enumerate(engines):
        assert got[v] == solo[v], (v, got[v], solo[v])
        lg = e.logits()
        ref = solo_logits[v]
        assert np.allclose(lg, ref, rtol=1e-3, atol=1e-4 + 1e-3 * np.abs(ref).max()), (v, np.abs(lg - ref).max())
    assert len({tuple(t) for t in got}) == n_seq  # the sequences really differ
    # a second batched run of the same engine set, after other work on the
    # same stream (a single-sequence decode), repeats the first
    base.prefill_kv_random(prefill, 100)
    assert base.generate(prompts[0].tolist(), steps, start_pos=prefill) == solo[0]
    for v, e in enumerate(engines):
        e.prefill_kv_random(prefill, 100 + v)
    assert zinc_amd.InferenceEngine.generate_batch(engines, prompts, steps, start_pos=prefill) == got
    for e in engines[1:]:
        e.deinit()
    base.deinit()


@pytest.mark.parametrize("n_seq,prefill,heads,paged", [(2, 1, 8, False), (5, 255, 16, True), (16, 130, 8, True),
                                                       (3, 1000, 2, False), (17, 63, 4, False)])
def test_batch_attention_edges(ctx, n_seq, prefill, heads, paged):
    """Chunks per sequence from 64 (2 sequences) to 1 (17: two launches), the
    new token at a page's and a chunk's first row, 1 to 8 q heads per kv head,
    each sequence's own shuffled page table: tokens and logits as alone."""
    import zinc_amd
    print(f"batch attention n={n_seq} at {prefill} heads {heads} paged {paged}", flush=True)
    cfg = dict(CFG, n_layers=2, hidden=1024, n_heads=heads, max_ctx=1024, vocab=1024)
    base = zinc_amd.InferenceEngine(ctx, cfg)
    engines = [base] + [base.share(ctx) for _ in range(n_seq - 1)]
    rng = np.random.default_rng(n_seq)
    prompts = rng.integers(0, cfg["vocab"], (n_seq, 2)).astype(np.uint32)
    solo, logits = [], []
    for v, e in enumerate(engines):
        if paged:
            e.set_pages(rng.permutation(cfg["max_ctx"] // 16))
        e.prefill_kv_random(prefill, 300 + v)
        solo.append(e.generate(prompts[v].tolist(), 6, start_pos=prefill))
        logits.append(e.logits())
        e.prefill_kv_random(prefill, 300 + v)
    assert zinc_amd.InferenceEngine.generate_batch(engines, prompts, 6, start_pos=prefill) == solo
    for v, e in enumerate(engines):
        lg = e.logits()
        assert np.allclose(lg, logits[v], rtol=1e-3, atol=1e-4 + 1e-3 * np.abs(logits[v]).max()), v
    for e in engines[1:]:
        e.deinit()
    base.deinit()


@pytest.mark.parametrize("n_seq,vocab", [(2, 1000), (5, 1023), (16, 257), (17, 1026)])
def test_batch_tail(ctx, n_seq, vocab):
    """Embedding rows, argmax and step advance of up to 16 sequences a launch:
    vocabularies off the 4 logits of a load and the workgroups of a launch (few
    and many sequences), a prompt of three tokens, a second run from another
    position; then logits that are all NaN, whose greedy token is 0, as alone."""
    import ctypes as C
    import zinc_amd
    from zinc_amd.hip import lib
    print(f"batch tail n={n_seq} vocab {vocab}", flush=True)
    cfg = dict(CFG, n_layers=1, vocab=vocab, max_ctx=128)
    base = zinc_amd.InferenceEngine(ctx, cfg)
    engines = [base] + [base.share(ctx) for _ in range(n_seq - 1)]
    rng = np.random.default_rng(vocab)
    for start in (20, 33):
        prompts = rng.integers(0, vocab, (n_seq, 3)).astype(np.uint32)
        prompts[0] = [0, vocab - 1, vocab - 1]
        solo = []
        for v, e in enumerate(engines):
            e.prefill_kv_random(start, 500 + v)
            solo.append(e.generate(prompts[v].tolist(), 5, start_pos=start))
            e.prefill_kv_random(start, 500 + v)
        assert zinc_amd.InferenceEngine.generate_batch(engines, prompts, 5, start_pos=start) == solo
    nan = np.full(cfg["hidden"], np.nan, np.float32)
    b, off, n = C.c_void_p(), C.c_uint64(), C.c_uint64()
    ctx.check(lib().zh_engine_tensor(base.h, 2, C.byref(b), C.byref(off), C.byref(n)))  # output_norm
    assert n.value == nan.nbytes
    ctx.check(lib().zh_buf_upload(ctx.h, b, off.value, C.c_void_p(nan.ctypes.data), nan.nbytes))
    got = zinc_amd.InferenceEngine.generate_batch(engines, prompts, 3, start_pos=33)
    assert got == [[0, 0, 0]] * n_seq
    assert base.generate(prompts[0].tolist(), 3, start_pos=33) == [0, 0, 0]
    for e in engines[1:]:
        e.deinit()
    base.deinit()


@pytest.mark.parametrize("heads", [2, 8, 16])  # 1, 4 and 8 per kv head
def test_batch_attention_q_past_f16(ctx, heads):
    """Query norm weights of 2^15 put q's components far past f16's 65504:
    tokens and logits as alone on the attention kernel that multiplies in
    f32."""
    import ctypes as C
    import zinc_amd
    from zinc_amd.hip import lib
    print(f"batch attention, q past f16, heads {heads}", flush=True)
    cfg = dict(CFG, n_layers=2, n_heads=heads, vocab=1024)
    base = zinc_amd.InferenceEngine(ctx, cfg)
    w = np.full(128, 2.0 ** 15, np.float32)
    for layer in range(2):
        b, off, n = C.c_void_p(), C.c_uint64(), C.c_uint64()
        ctx.check(lib().zh_engine_tensor(base.h, (layer + 1) << 8 | 6, C.byref(b), C.byref(off), C.byref(n)))
        assert n.value == w.nbytes
        ctx.check(lib().zh_buf_upload(ctx.h, b, off.value, C.c_void_p(w.ctypes.data), w.nbytes))
    engines = [base] + [base.share(ctx) for _ in range(2)]
    prompts = np.array([[5], [600], [71]], np.uint32)
    solo, logits = [], []
    for v, e in enumerate(engines):
        e.set_fused_attn(False)
        e.prefill_kv_random(200, 400 + v)
        solo.append(e.generate(prompts[v].tolist(), 4, start_pos=200))
        logits.append(e.logits())
        e.prefill_kv_random(200, 400 + v)
    assert zinc_amd.InferenceEngine.generate_batch(engines, prompts, 4, start_pos=200) == solo
    for v, e in enumerate(engines):
        lg = e.logits()
        assert np.isfinite(lg).all()
        assert np.allclose(lg, logits[v], rtol=1e-3, atol=1e-4 + 1e-3 * np.abs(logits[v]).max()), v
    for e in engines[1:]:
        e.deinit()
    base.deinit()


def test_batch_rejects_foreign_engines(ctx):
    import zinc_amd
    a = zinc_amd.InferenceEngine(ctx, dict(CFG, n_layers=2))
    b = zinc_amd.InferenceEngine(ctx, dict(CFG, n_layers=2, seed=58))  # other weights
    with pytest.raises(zinc_amd.ZincError) as e:
        zinc_amd.InferenceEngine.generate_batch([a, b], [[1, 2], [3, 4]], 2, start_pos=0)
    assert e.value.name == "InvalidArgument"
    with pytest.raises(zinc_amd.ZincError) as e:
        zinc_amd.InferenceEngine.generate_batch([a, a], [[1, 2], [3, 4]], 2, start_pos=0)
    assert e.value.name == "InvalidArgument"
    a.deinit()
    b.deinit()
    # Q8_0 attention: no tile kernel for the batched projections
    q8 = zinc_amd.InferenceEngine(ctx, dict(CFG, n_layers=2, type_attn=8))
    q8b = q8.share(ctx)
    with pytest.raises(zinc_amd.ZincError) as e:
        zinc_amd.InferenceEngine.generate_batch([q8, q8b], [[1, 2], [3, 4]], 2, start_pos=0)
    assert e.value.name == "UnsupportedQuantType"
    q8b.deinit()
    q8.deinit()


def test_batch_groups_on_two_streams(ctx):
    """Two batches of 2 sequences, each on its own context (HIP stream) and
    host thread, decode at once; every sequence as it decodes alone."""
    import threading
    import zinc_amd
    ctx2 = zinc_amd.Context(0)
    cfg = dict(CFG, n_layers=2)
    base = zinc_amd.InferenceEngine(ctx, cfg)
    groups = [[base, base.share(ctx)], [base.share(ctx2), base.share(ctx2)]]
    rng = np.random.default_rng(9)
    prompts = [rng.integers(0, cfg["vocab"], (2, 3)).astype(np.uint32) for _ in range(2)]
    prefill, steps = 30, 10
    solo = []
    for g in range(2):
        for v, e in enumerate(groups[g]):
            e.prefill_kv_random(prefill, 200 + 2 * g + v)
            solo.append(e.generate(prompts[g][v].tolist(), steps, start_pos=prefill))
            e.prefill_kv_random(prefill, 200 + 2 * g + v)
    ctx.sync()
    ctx2.sync()
    got = [None, None]

    def run(g):
        got[g] = zinc_amd.InferenceEngine.generate_batch(groups[g], prompts[g], steps, start_pos=prefill)
    th = [threading.Thread(target=run, args=(g,)) for g in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert got[0] + got[1] == solo
    for e in groups[1] + groups[0][1:]:
        e.deinit()
    base.deinit()
    ctx2.close()
