"""End-to-end parity of the token loop on the MI355X against the CPU oracle, on seeded synthetic
models of the configs' families (Qwen3 with q/k-norm, Qwen2 with q/k/v biases, Llama).

Invariants mirror the reference's model tests (Tests/MLXEngineTests/ModelTests.swift):
prefill vs token-by-token decode (argmax equal, max |d logit| < 0.1, :50-93), sparse attention with a
budget covering the context is bit-identical to dense (:155-182), prefix reuse (:235-255). Against the
oracle: final logits within 2e-2 max-abs (north star) and greedy tokens identical, checked teacher-forced
(the oracle is fed the GPU's tokens; a step whose oracle top-2 margin is below 2e-2 cannot decide
the argmax at this tolerance and is counted, not failed).
"""
import os
import tempfile

import numpy as np
import pytest

import configs
import mlxr
import oracle

pytestmark = pytest.mark.gpu

LOGIT_TOL = 2e-2
GREEDY = mlxr.SamplingParameters.greedy()


@pytest.fixture(scope="module")
def models():
    tmp = tempfile.mkdtemp(prefix="mlxr_models_")
    out = {}
    for name, cfg in {
        "qwen3": configs.tiny("qwen3"),
        "qwen2": configs.tiny("qwen2", tie=False),
        "llama": configs.tiny("llama", tie=False, theta=500000.0),
        "qwen3_g128_8bit": configs.tiny("qwen3", bits=8, gs=128, layers=1),
        "qwen3_3bit": configs.tiny("qwen3", bits=3, gs=32, layers=1),
        # hidden 1024 at gs 32: wider rows (two scale groups per 16-row tile)
        "qwen3_h1024": configs.tiny("qwen3", hidden=1024, inter=1024, gs=32),
        # RoPE variants: interleaved pairs, and half the head dims rotated
        "qwen3_rope_trad": dict(configs.tiny("qwen3"), rope_traditional=True),
        "qwen3_rope_half": dict(configs.tiny("qwen3"), partial_rotary_factor=0.5),
    }.items():
        d = os.path.join(tmp, name)
        mlxr.synth_write(cfg, seed=1234, directory=d)
        out[name] = d
    return out


def prompt(n, vocab, seed=5):
    return np.random.default_rng(seed).integers(0, vocab, n).astype(np.int32)


@pytest.mark.parametrize("name", ["qwen3", "qwen2", "llama", "qwen3_g128_8bit", "qwen3_3bit"])
def test_prefill_logits_match_oracle(gpu, models, name):
    d = models[name]
    with mlxr.Transformer(d, context_length=1024) as m:
        ref = oracle.Model(d, m.max_seq)
        for n in (1, 5, 40):
            toks = prompt(n, m.vocab_size, seed=n)
            got = m.forward(toks, 0)
            exp = ref.forward(toks, 0)
            assert np.max(np.abs(got - exp)) < LOGIT_TOL, (name, n, np.max(np.abs(got - exp)))
            assert m.written_high >= n


def greedy_check(m, ref, toks, gen):
    """Teacher-forced greedy parity: the oracle recomputes each step from the GPU's tokens."""
    ambiguous = 0
    logits = ref.forward(toks, 0)
    pos = len(toks)
    for t in gen:
        order = np.argsort(-logits.astype(np.float64), kind="stable")
        if t != order[0]:
            margin = logits[order[0]] - logits[t]
            assert margin < LOGIT_TOL, (t, int(order[0]), float(margin))
            ambiguous += 1
        logits = ref.forward(np.array([t], np.int32), pos)
        pos += 1
    return ambiguous


@pytest.mark.parametrize("name", ["qwen3", "qwen2", "llama"])
def test_greedy_generation_matches_oracle(gpu, models, name):
    d = models[name]
    with mlxr.Transformer(d, context_length=1024) as m:
        ref = oracle.Model(d, m.max_seq)
        toks = prompt(32, m.vocab_size)
        gen = m.generate(toks, 24, GREEDY)
        assert len(gen) == 24
        amb = greedy_check(m, ref, toks, gen)
        assert amb <= 2, amb


def test_graph_and_eager_decode_agree(gpu, models):
    d = models["qwen3"]
    toks = prompt(16, 1000)
    with mlxr.Transformer(d, context_length=512) as m:
        a = m.generate(toks, 20, GREEDY)
        m.set_graphs(False)
        b = m.generate(toks, 20, GREEDY)
    assert a == b


@pytest.mark.parametrize("name", ["qwen3", "qwen2", "llama", "qwen3_h1024"])
def test_persistent_decode_matches_kernel_per_op(gpu, models, name):
    """The persistent decode step (one launch per token) against the kernel-per-op step: same greedy
    tokens (teacher-forced against the oracle where they part), logits within the 2e-2 gate."""
    d = models[name]
    toks = prompt(20, 1000, seed=12)
    with mlxr.Transformer(d, context_length=512) as m:
        assert m.persistent_decode, "the tiny model must take the persistent path"
        a = m.generate(toks, 24, GREEDY)
        m.set_decode_mode(False)
        assert not m.persistent_decode
        b = m.generate(toks, 24, GREEDY)
        ref = oracle.Model(d, m.max_seq)
        assert greedy_check(m, ref, toks, a) <= 2
        if a != b:
            i = next(k for k in range(len(a)) if a[k] != b[k])
            logits = ref.forward(np.concatenate([toks, np.array(a[:i], np.int32)]), 0)
            assert abs(logits[a[i]] - logits[b[i]]) < LOGIT_TOL


@pytest.mark.parametrize("name", ["qwen3_rope_trad", "qwen3_rope_half"])
def test_persistent_decode_rope_variants(gpu, models, name):
    """Interleaved (traditional) RoPE and partial rotation (rot_dim 64) in the persistent step, whose
    q/k norm + RoPE takes a different path for each, against the kernel-per-op step's qkv_post
    (checked against the oracle's RoPE in test_qkv_post): same greedy tokens, or, where they part,
    the two tokens' logits (full prefill of the shared prefix) within the 2e-2 gate."""
    d = models[name]
    toks = prompt(40, 1000, seed=21)
    with mlxr.Transformer(d, context_length=512) as m:
        assert m.persistent_decode
        a = m.generate(toks, 16, GREEDY)
        m.set_decode_mode(0)
        b = m.generate(toks, 16, GREEDY)
        if a != b:
            i = next(k for k in range(len(a)) if a[k] != b[k])
            logits = m.forward(np.concatenate([toks, np.array(a[:i], np.int32)]), 0)
            assert abs(logits[a[i]] - logits[b[i]]) < LOGIT_TOL, (name, i)


def test_persistent_decode_long_ranges(gpu, models):
    """Key ranges longer than one and two 128-key chunks per workgroup (the tiny model's two KV
    heads give 128 ranges each: ~156 keys at 20000 tokens, ~265 at 34000): the persistent step's
    greedy tokens against the kernel-per-op step's; where they part, the two tokens' logits (full
    prefill of the shared prefix) are within the 2e-2 gate."""
    d = models["qwen3"]
    with mlxr.Transformer(d, context_length=34100) as m:
        assert m.persistent_decode
        for n in (20000, 34000):
            toks = prompt(n, 1000, seed=n % 97)
            m.set_decode_mode(1)
            a = m.generate(toks, 6, GREEDY)
            m.set_decode_mode(0)
            b = m.generate(toks, 6, GREEDY)
            if a != b:
                i = next(k for k in range(len(a)) if a[k] != b[k])
                logits = m.forward(np.concatenate([toks, np.array(a[:i], np.int32)]), 0)
                assert abs(logits[a[i]] - logits[b[i]]) < LOGIT_TOL, (n, i)


@pytest.mark.parametrize("name", ["qwen3", "qwen2", "llama"])
def test_decode_tiles_match_mlx_layout(gpu, models, name):
    """Single-token steps of the kernel-per-op path: the matvecs over the repacked tiles (decode mode
    0) against the MLX-layout matvecs (mode 2) and the oracle, logits within the 2e-2 gate."""
    d = models[name]
    toks = prompt(12, 1000, seed=21)
    with mlxr.Transformer(d, context_length=512) as m:
        ref = oracle.Model(d, m.max_seq)
        want = ref.forward(toks, 0)
        got = {}
        for mode in (0, 2):
            m.set_decode_mode(mode)
            for i, t in enumerate(toks):
                got[mode] = m.forward(np.array([t], np.int32), i)
        assert np.max(np.abs(got[0] - got[2])) < LOGIT_TOL
        assert np.max(np.abs(got[0] - want)) < LOGIT_TOL
        assert np.argmax(got[0]) == np.argmax(want)


def test_prefill_vs_incremental_decode(gpu, models):
    """ModelTests.swift:50-69: same argmax and max |d logit| < 0.1 (here: the 2e-2 gate)."""
    d = models["qwen3"]
    with mlxr.Transformer(d, context_length=1024) as m:
        toks = prompt(40, m.vocab_size, seed=9)
        full = m.forward(toks, 0)
        for i, t in enumerate(toks):
            last = m.forward(np.array([t], np.int32), i)
        assert np.argmax(full) == np.argmax(last)
        assert np.max(np.abs(full - last)) < LOGIT_TOL


def test_long_prefill_chunks(gpu, models):
    """Prompts longer than one prefill chunk (ModelTests.swift:73-93; this build's chunk is 2048)."""
    d = models["qwen3"]
    with mlxr.Transformer(d, context_length=4096) as m:
        ref = oracle.Model(d, m.max_seq)
        toks = prompt(2300, m.vocab_size, seed=4)
        got = m.forward(toks, 0)
        assert np.max(np.abs(got - ref.forward(toks, 0))) < LOGIT_TOL


@pytest.mark.parametrize("name", ["qwen2", "qwen3_rope_half"])
@pytest.mark.parametrize("n", [9, 16, 17, 33, 65, 129, 300])
def test_short_prefills_match_oracle(gpu, tmp_path, name, n):
    """Short and ragged prompts through the prefill tile GEMM (biases; half RoPE: the q|k|v reader of one
    workgroup per head). Logits at the gate against the oracle, or, for the half RoPE that the oracle's
    model does not have, against the same tokens decoded one by one."""
    cfg = configs.tiny("qwen2" if name == "qwen2" else "qwen3", tie=False, hidden=1024, inter=2048)
    if name != "qwen2":
        cfg = dict(cfg, partial_rotary_factor=0.5)
    mlxr.synth_write(cfg, seed=n, directory=str(tmp_path))
    with mlxr.Transformer(str(tmp_path), context_length=1024) as m:
        toks = prompt(n, m.vocab_size, seed=n)
        if name == "qwen2":
            exp = oracle.Model(str(tmp_path), m.max_seq).forward(toks, 0)
        else:
            for i in range(n):
                exp = m.forward(toks[i:i + 1], i)
        got = m.forward(toks, 0)
        assert np.max(np.abs(got - exp)) < LOGIT_TOL


@pytest.mark.parametrize("family,bits,gs", [("qwen2", 4, 64), ("qwen3", 4, 32), ("qwen3", 3, 32)])
def test_prefill_is_chunk_invariant(gpu, tmp_path, family, bits, gs):
    """A prompt leaves the same K/V bits and the same last logits whether it comes in one prefill or in
    pieces of any length past 8 tokens (repacked tiles at 4 bits, MLX layout at 3): a second turn after a
    reused prefix repeats the one-shot prompt."""
    cfg = configs.tiny(family, bits=bits, gs=gs, tie=False, hidden=1024, inter=2048)
    mlxr.synth_write(cfg, seed=bits, directory=str(tmp_path))
    n, nkv, L = 700, cfg["num_key_value_heads"], cfg["num_hidden_layers"]
    with mlxr.Transformer(str(tmp_path), context_length=1024) as m:
        toks = prompt(n, m.vocab_size, seed=bits)
        whole = m.forward(toks, 0).copy()
        kv = [m.read_kv(i, n, nkv, 128) for i in range(L)]
        for cuts in ((0, 9, 26, 59, 124, 253, 700), (0, 640, 700), (0, 300, 316, 700)):
            for a, b in zip(cuts, cuts[1:]):
                got = m.forward(toks[a:b], a)
            for i in range(L):
                for want, have in zip(kv[i], m.read_kv(i, n, nkv, 128)):
                    assert np.array_equal(want.view(np.uint32), have.view(np.uint32)), (cuts, i)
            assert np.array_equal(got.view(np.uint32), whole.view(np.uint32)), cuts


def test_sparse_full_budget_is_bit_identical(gpu, models):
    """sparseDecodeWithFullBudgetIsBitIdentical (ModelTests.swift:155-182)."""
    d = models["qwen3"]
    sp = mlxr.SparseAttention(top_k=1 << 20, window=4, sink=4, min_context=8)
    with mlxr.Transformer(d, context_length=1024, sparse=sp) as m:
        assert m.sparse_available
        toks = prompt(300, m.vocab_size, seed=2)
        m.forward(toks, 0)
        nxt = np.array([17], np.int32)
        dense = m.forward(nxt, 300, dense=True)
        sparse = m.forward(nxt, 300)
        assert np.array_equal(dense.view(np.uint32), sparse.view(np.uint32))


def test_sparse_decode_matches_oracle(gpu, models):
    """A budget smaller than the context: the GPU's selection and attention vs the oracle's."""
    d = models["qwen3"]
    sp = mlxr.SparseAttention(top_k=64, window=32, sink=4, min_context=128)
    with mlxr.Transformer(d, context_length=1024, sparse=sp) as m:
        ref = oracle.Model(d, m.max_seq)
        ref.set_sparse(True, top_k=64, window=32, sink=4, min_context=128)
        toks = prompt(400, m.vocab_size, seed=8)
        m.forward(toks, 0)
        # the oracle decodes over the GPU's cache (the prefill itself is checked against the oracle
        # elsewhere): the block selection is discrete, so it must see the same keys
        for layer in range(2):
            ref.set_kv(layer, *m.read_kv(layer, 400, 2, 128))
        for i, t in enumerate([3, 99, 500]):
            got = m.forward(np.array([t], np.int32), 400 + i)
            exp = ref.forward(np.array([t], np.int32), 400 + i)
            assert np.max(np.abs(got - exp)) < LOGIT_TOL
        # sparse changes outputs relative to dense
        dense = m.forward(np.array([7], np.int32), 403, dense=True)
        spl = m.forward(np.array([7], np.int32), 403)
        assert not np.array_equal(dense, spl)


def test_prefix_reuse_second_turn(gpu, models):
    """prefix-cache reuse (ModelTests.swift:235-255; Engine.swift:558-564): a second turn sharing the
    first turn's tokens reuses the cache and gives the logits of a full re-prefill."""
    d = models["qwen3"]
    with mlxr.Transformer(d, context_length=1024) as m:
        turn1 = prompt(100, m.vocab_size, seed=1)
        m.forward(turn1, 0)
        turn2 = np.concatenate([turn1, prompt(30, m.vocab_size, seed=2)])
        common = m.reusable_prefix(100, 100)
        assert common == 100
        reused = m.forward(turn2[common:], common)
        m.reset_write_tracking()
        fresh = m.forward(turn2, 0)
        assert np.max(np.abs(reused - fresh)) < LOGIT_TOL
        assert np.argmax(reused) == np.argmax(fresh)


def test_errors(gpu, models):
    d = models["qwen3"]
    with mlxr.Transformer(d, context_length=256) as m:
        with pytest.raises(mlxr.EngineError) as e:
            m.forward(np.array([m.vocab_size], np.int32), 0)
        assert e.value.case == "invalidFile"
        with pytest.raises(mlxr.EngineError) as e:
            m.forward(np.zeros(10, np.int32), m.max_seq - 5)
        assert e.value.case == "contextFull"
        with pytest.raises(mlxr.EngineError) as e:
            m.prefill(np.zeros(4, np.int32), m.max_seq - 4, GREEDY)
        assert e.value.case == "contextFull"


def test_sampled_generation_is_seeded(gpu, models):
    d = models["qwen3"]
    sp = mlxr.SamplingParameters(temperature=0.8, top_k=40, top_p=0.95, repetition_penalty=1.05)
    toks = prompt(12, 1000, seed=3)
    with mlxr.Transformer(d, context_length=512) as m:
        m.seed_sampler(42)
        a = m.generate(toks, 16, sp)
        m.seed_sampler(42)
        b = m.generate(toks, 16, sp)
        m.seed_sampler(43)
        c = m.generate(toks, 16, sp)
    assert a == b
    assert all(0 <= t < 1000 for t in a)
    assert a != c or len(set(a)) == 1


def test_persistent_abort_fails_both_steps_in_flight(gpu, models):
    """Failure path of the persistent step, forced from the host: the first step's first wait asks for
    a tag no launch writes with a short bound, so it expires and raises the abort flag; every kernel
    still runs to its end. Both steps in flight then report a GPU error, the model falls back to the
    kernel-per-op step, and a fresh turn decodes the same tokens as a healthy model."""
    d = models["qwen3"]
    toks = prompt(20, 1000, seed=12)
    with mlxr.Transformer(d, context_length=512) as m:
        assert m.persistent_decode
        want = m.generate(toks, 8, GREEDY)
        first = m.prefill(toks, 0, GREEDY)
        m.debug_stall_next_step()
        s1 = m.begin_decode_step(len(toks), GREEDY)
        s2 = m.begin_decode_step(len(toks) + 1, GREEDY)
        for s in (s1, s2):
            with pytest.raises(mlxr.EngineError) as e:
                m.finish(s)
            assert e.value.case == "gpuFailure"
        assert not m.persistent_decode
        assert first == want[0]
        assert m.generate(toks, 8, GREEDY) == want


@pytest.mark.parametrize("name", ["qwen3", "llama", "qwen3_3bit", "qwen3_g128_8bit"])
def test_verify_batch_matches_incremental_decode(gpu, models, name):
    """verifyBatchMatchesIncrementalDecode (ModelTests.swift:201-230): each row of a T = 2..8 batch
    (all_logits) gives the next-token logits of decoding the tokens one at a time: same argmax, max
    difference < 0.1; and the batch rows against the oracle within the 2e-2 gate."""
    d = models[name]
    ids = prompt(40, 1000, seed=21)
    o = 24
    with mlxr.Transformer(d, context_length=512) as m:
        ref = oracle.Model(d, m.max_seq)
        for T in (2, 3, 5, 8):
            m.forward(ids[:o], 0)
            batch = ids[o:o + T]
            rows = m.forward(batch, o, all_logits=True)
            assert rows.shape == (T, m.vocab_size)
            for i, t in enumerate(batch):
                inc = m.forward(np.array([t], np.int32), o + i)
                assert int(np.argmax(rows[i])) == int(np.argmax(inc)), (T, i)
                assert np.max(np.abs(rows[i] - inc)) < 0.1, (T, i)
            want = ref.forward(ids[:o + T], 0)
            assert np.max(np.abs(rows[-1] - want)) < LOGIT_TOL, T


def test_cancel_between_prefill_chunks(gpu, models):
    """isCancelled is polled between chunks (Transformer.swift:1127,1233): a cancel after the first
    2048-token chunk returns `cancelled`; the chunk's rows stay cached, so prefilling the rest at
    offset 2048 gives the token of an uncancelled prefill."""
    d = models["qwen3"]
    ids = prompt(2100, 1000, seed=8)
    with mlxr.Transformer(d, context_length=4096) as m:
        want = m.prefill(ids, 0, GREEDY)
        calls = []
        with pytest.raises(mlxr.EngineError) as e:
            m.prefill(ids, 0, GREEDY, is_cancelled=lambda: calls.append(1) or True)
        assert e.value.case == "cancelled" and len(calls) == 1
        assert m.prefill(ids[2048:], 2048, GREEDY) == want
        with pytest.raises(mlxr.EngineError) as e:
            m.forward(ids, 0, is_cancelled=lambda: True)
        assert e.value.case == "cancelled"
        assert np.argmax(m.forward(ids, 0, is_cancelled=lambda: False)) == want
        assert m.prefill(ids[:100], 0, GREEDY, is_cancelled=lambda: True) == m.prefill(ids[:100], 0, GREEDY)   # one chunk: never polled


def test_engine_speculative_greedy_is_identical(gpu, models):
    """speculativeGreedyOutputIsIdentical (ModelTests.swift:411-434) on token ids: a prompt that
    repeats itself, decoded plainly (GPU sampling, pipelined steps) and speculatively (prompt-lookup
    drafts verified in batched passes): same tokens; drafts are accepted; a second turn reuses the
    prompt cache and still matches a fresh engine."""
    import engine
    d = models["qwen3"]
    base = list(prompt(24, 1000, seed=30))
    ids = base * 3
    with mlxr.Transformer(d, context_length=1024) as m:
        eng = engine.InferenceEngine(m)
        p = engine.GenerationParameters(temperature=0.0, repetition_penalty=1.0, max_tokens=48)
        plain = eng.generate(ids, p)
        spec = eng.generate(ids, engine.GenerationParameters(temperature=0.0, repetition_penalty=1.0, max_tokens=48, speculative=True))
        tp = [e[1] for e in plain if e[0] == "token"]
        ts = [e[1] for e in spec if e[0] == "token"]
        st = spec[-1][1]
        assert len(tp) == 48
        amb = greedy_check(m, oracle.Model(d, m.max_seq), np.array(ids, np.int32), tp)
        assert amb <= 2
        if tp != ts:   # only where the oracle's top-2 margin cannot decide at the 2e-2 gate
            i = next(k for k in range(len(tp)) if tp[k] != ts[k])
            ref = oracle.Model(d, m.max_seq).forward(np.array(ids + tp[:i], np.int32), 0)
            assert abs(ref[tp[i]] - ref[ts[i]]) < LOGIT_TOL
        assert st.draft_tokens and st.accepted_draft_tokens > 0
        follow = ids + tp + base[:5]
        again = eng.generate(follow, p)
        assert again[-1][1].cached_prompt_tokens > len(ids)
        fresh = engine.InferenceEngine(m)
        m.reset_write_tracking()
        ref_turn = fresh.generate(follow, p)
        assert [e[1] for e in again if e[0] == "token"] == [e[1] for e in ref_turn if e[0] == "token"]


def test_checkpoint_layouts_load_identically(gpu, models, tmp_path):
    """Loader parity across the checkpoint layouts MLX-community repositories use (GPU.swift:330-357,
    Transformer.swift:48-111): the same tensors re-written by an independent writer as two shards
    with model.safetensors.index.json, in another tensor order, with a multimodal
    `language_model.` prefix, extra config fields and an unused extra tensor, give bit-identical
    logits to the single-file model. (No real checkpoint is available offline: the layouts are built
    from the synthetic model's own tensors.)"""
    import json
    from qfix import read_safetensors, write_safetensors
    d = models["qwen2"]
    src = read_safetensors(os.path.join(d, "model.safetensors"))
    cfg = json.load(open(os.path.join(d, "config.json")))
    dt_of = {np.uint32: "U32", np.uint16: "BF16", np.float16: "F16", np.float32: "F32"}
    dtypes = {k: dt_of[v.dtype.type] for k, v in src.items()}
    out = str(tmp_path / "sharded")
    os.makedirs(out)
    names = sorted(src, reverse=True)
    renamed = {("language_model." + k if not k.startswith("lm_head") else "language_model." + k): k for k in names}
    half = len(names) // 2
    shards = {"model-00001-of-00002.safetensors": names[:half], "model-00002-of-00002.safetensors": names[half:]}
    weight_map = {}
    for fn, ks in shards.items():
        tens = {[r for r, o in renamed.items() if o == k][0]: src[k] for k in ks}
        dts = {[r for r, o in renamed.items() if o == k][0]: dtypes[k] for k in ks}
        if fn.startswith("model-00002"):
            tens["language_model.model.rotary_emb.inv_freq"] = np.ones(64, np.float32)
            dts["language_model.model.rotary_emb.inv_freq"] = "F32"
        write_safetensors(os.path.join(out, fn), tens, dts)
        weight_map.update({k: fn for k in tens})
    json.dump({"metadata": {"total_size": 0}, "weight_map": weight_map}, open(os.path.join(out, "model.safetensors.index.json"), "w"))
    cfg2 = dict(cfg, architectures=["Qwen2ForCausalLM"], torch_dtype="bfloat16", transformers_version="4.51.0")
    json.dump(cfg2, open(os.path.join(out, "config.json"), "w"))
    toks = prompt(33, 1000, seed=44)
    with mlxr.Transformer(d, context_length=256) as a, mlxr.Transformer(out, context_length=256) as b:
        la, lb = a.forward(toks, 0), b.forward(toks, 0)
        assert np.array_equal(la.view(np.uint32), lb.view(np.uint32))
        assert a.generate(toks, 8, GREEDY) == b.generate(toks, 8, GREEDY)


def test_misaligned_tensors_load_identically(gpu, models, tmp_path):
    """loadsTensorsZeroCopyAndRealignsMisalignedOnes (EngineTests.swift:125-150): a 6-byte F16
    tensor first leaves the later tensors (codes, scales, norm weights) off their natural alignment
    in the file; the model loads them realigned and its logits are bit-identical to the aligned
    file's."""
    import json
    import shutil
    from qfix import read_safetensors, write_safetensors
    d = models["llama"]
    src = read_safetensors(os.path.join(d, "model.safetensors"))
    dt_of = {np.uint32: "U32", np.uint16: "BF16", np.float16: "F16", np.float32: "F32"}
    out = str(tmp_path / "misaligned")
    shutil.copytree(d, out)
    tens = {"a_pad": np.array([1, 2, 3], np.float16)}
    tens.update(src)
    hdr, off, blobs = {}, 0, []
    for k, a in tens.items():
        b = np.ascontiguousarray(a).tobytes()
        hdr[k] = {"dtype": dt_of[a.dtype.type], "shape": list(a.shape), "data_offsets": [off, off + len(b)]}
        off += len(b)
        blobs.append(b)
    h = json.dumps(hdr)
    h += " " * (-(8 + len(h)) % 16)           # data starts 16-byte aligned, as the reference test's does
    with open(os.path.join(out, "model.safetensors"), "wb") as f:
        f.write(len(h).to_bytes(8, "little") + h.encode() + b"".join(blobs))
    starts = [8 + len(h) + v["data_offsets"][0] for k, v in hdr.items() if k != "a_pad"]
    assert all(s % 4 == 2 for s in starts)   # every tensor after the F16 one starts 2 bytes off
    toks = prompt(21, 1000, seed=45)
    with mlxr.Transformer(d, context_length=256) as a, mlxr.Transformer(out, context_length=256) as b:
        assert np.array_equal(a.forward(toks, 0).view(np.uint32), b.forward(toks, 0).view(np.uint32))


def test_begin_steps_matches_prefill(gpu, models):
    """beginSteps (Transformer.swift:1265-1296): n tokens written at offset and one step over them
    whose token the GPU selects, not waited for. begin_steps(tokens) then begin_decode gives the
    same tokens as prefill of the same tokens then begin_decode, for a single token, a few (the
    small-batch pass) and more than eight (the prefill GEMMs); a step in flight is refused."""
    d = models["qwen3"]
    toks = prompt(60, 1000, seed=41)
    P = 30
    with mlxr.Transformer(d, context_length=512) as a, mlxr.Transformer(d, context_length=512) as b:
        for n in (1, 3, 8, 12):
            a.reset_write_tracking(); b.reset_write_tracking()
            want = [b.prefill(toks[:P + n], 0, GREEDY)]
            for i in range(4):
                want.append(b.finish(b.begin_decode_step(P + n + i, GREEDY)))
            a.prefill(toks[:P], 0, GREEDY)
            st = a.begin_steps(toks[P:P + n], P, GREEDY)
            assert st.offset == P + n - 1
            nxt = a.begin_decode_step(P + n, GREEDY)        # queued behind it: two in flight
            got = [a.finish(st), a.finish(nxt)]
            for i in range(3):
                got.append(a.finish(a.begin_decode_step(P + n + 1 + i, GREEDY)))
            assert got == want, n
        st = a.begin_decode_step(P, GREEDY)
        with pytest.raises(mlxr.EngineError):
            a.begin_steps(toks[:2], P + 1, GREEDY)
        a.finish(st)


def test_engine_draft_model_greedy_is_identical(gpu, models):
    """Draft-model speculation (Engine.swift:619-669): a draft model catches up through
    begin_steps and proposes greedy tokens in pipelined steps, the target verifies them in batched
    passes. With the target's own weights as the draft, the tokens equal plain decoding's and the
    drafts are accepted."""
    import engine
    d = models["qwen3"]
    ids = list(prompt(40, 1000, seed=44))
    with mlxr.Transformer(d, context_length=1024) as m, mlxr.Transformer(d, context_length=1024) as dm:
        p = engine.GenerationParameters(temperature=0.0, repetition_penalty=1.0, max_tokens=40)
        plain = [e[1] for e in engine.InferenceEngine(m).generate(ids, p) if e[0] == "token"]
        m.reset_write_tracking()
        eng = engine.InferenceEngine(m, draft_model=dm)
        ev = eng.generate(ids, p)
        spec = [e[1] for e in ev if e[0] == "token"]
        st = ev[-1][1]
        assert st.model_draft_tokens and st.accepted_model_draft_tokens > 0, st
        if spec != plain:   # only where the oracle's top-2 margin cannot decide at the 2e-2 gate
            i = next(k for k in range(len(plain)) if plain[k] != spec[k])
            ref = oracle.Model(d, m.max_seq).forward(np.array(ids + plain[:i], np.int32), 0)
            assert abs(ref[plain[i]] - ref[spec[i]]) < LOGIT_TOL


def test_config_getters(gpu, models, tmp_path):
    """The config members InferenceEngine reads (Engine.swift:322-355): model type, end-of-sequence
    ids from config.json (a number or a list) and generation_config.json, deduplicated; no hybrid
    model loads; every loadable model verifies in batches (supportsBatchedVerify)."""
    import json
    import shutil
    d = str(tmp_path / "m")
    shutil.copytree(models["qwen2"], d)
    with open(os.path.join(d, "config.json")) as f:
        cfg = json.load(f)
    cfg["eos_token_id"] = [7, 5, 7]
    with open(os.path.join(d, "config.json"), "w") as f:
        json.dump(cfg, f)
    with open(os.path.join(d, "generation_config.json"), "w") as f:
        json.dump({"eos_token_id": 9, "do_sample": True}, f)
    with mlxr.Transformer(d, context_length=256) as m:
        assert m.model_type == "qwen2"
        assert m.eos_token_ids == [5, 7, 9]
        assert not m.is_hybrid and m.supports_batched_verify
    with mlxr.Transformer(models["llama"], context_length=256) as m:
        assert m.model_type == "llama" and m.eos_token_ids == []
        assert m.sparse_layer_count == 0 and m.sparse_off_reason == ""
    sp = mlxr.SparseAttention(min_context=1024)
    with mlxr.Transformer(models["llama"], context_length=256, sparse=sp) as m:   # below where it starts
        assert not m.sparse_available and m.sparse_layer_count == 0 and "below 1024" in m.sparse_off_reason
    with mlxr.Transformer(models["llama"], context_length=2048, sparse=sp) as m:
        assert m.sparse_available and m.sparse_layer_count == 2 and m.sparse_off_reason == ""
