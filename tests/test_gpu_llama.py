"""The device decoder against the reference's golden logits and against the
oracle's Llama forward, on a real MI355X: the tiny fixture models (Q8_0, F16,
BF16, F32, Q4_K and Q6_K weights), and a random-init Q4_0 / Q8_0 model at
reduced size with 8B-like proportions."""
import base64
import json
import os

import numpy as np
import pytest
import torch

import oracle as O
from mimir_amd import capi
from mimir_amd.llama import Llama, load_mim
from mimir_amd.mimfile import MimFile
from oracle import llama as OL
from tests import gpu
from tests import test_gpu_decode_ops as ops
from tests.helpers import bits_equal
from tests.test_oracle_llama import compare_logits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,tol", [("spm", 0.02), ("bpe", 0.04)])
def test_fixture_models_match_golden_logits_and_oracle(golden_dir, name, tol):
    gpu.lib()
    path = os.path.join(golden_dir, f"{name}.mim")
    ref = MimFile(os.path.join(golden_dir, f"{name}.logits.mim"))
    tokens, want = ref["tokens"].data.tolist(), ref["logits"].data
    gpu.say(f"llama fixture {name}: batched pass")
    m = load_mim(path, max_tokens=len(tokens), context=len(tokens))
    v = m.config.vocab
    batched = m.logits(tokens, all=True)[0]
    compare_logits(batched, want, v, tol)  # examples/llama/llama_test.go:177: quantized weights, 2% / 4%
    # the oracle computes the same int8-activation products: far closer than that
    om = OL.Model.from_mim(MimFile(path))
    ow = om.logits(tokens, om.new_caches(len(tokens)), all=True)
    compare_logits(batched, ow, v, 1e-4)
    gpu.say(f"llama fixture {name}: one token at a time")
    m.reset()
    stepped = np.stack([m.logits([t])[0] for t in tokens])
    compare_logits(stepped, batched, v, 1e-4)  # llama_test.go:216
    assert m.cache_len == len(tokens)


def test_tiny_q4km_known_answers_with_f16_cache(golden_dir):
    """io/mim/mim_test.go:184-262: prompt logits, 8 greedy tokens and each
    step's logits, with a binary16 cache; int8 activations ("a8": within 1.5x
    of llama.cpp's own distance from the float64 oracle)."""
    e = json.load(open(os.path.join(golden_dir, "expected.json")))
    dec = lambda s: np.frombuffer(base64.b64decode(s), "<f4")
    gpu.lib()
    gpu.say("tiny-q4km a8")
    m = load_mim(os.path.join(golden_dir, "tiny-q4km-exact.mim"), max_tokens=16, context=64, cache_dtype=capi.F16)
    lim = 1.5 * e["llama_cpp_max_diff"]
    all_ = m.logits(e["prompt_ids"], all=True)[0]
    assert np.abs(all_.reshape(-1) - dec(e["prompt_logits"])).max() <= lim
    logits = all_[-1]
    om = OL.Model.from_mim(MimFile(os.path.join(golden_dir, "tiny-q4km-exact.mim")))
    caches = om.new_caches(64, O.F16)
    ologits = om.logits(e["prompt_ids"], caches, all=True)[-1]
    for i, tok in enumerate(e["greedy"]):
        assert np.abs(logits - dec(e["greedy_logits"][i])).max() <= lim
        assert np.abs(logits - ologits).max() <= 1e-4 * np.abs(ologits).max()  # the same arithmetic as the CPU path
        logits = m.logits([tok])[0]
        ologits = om.logits([tok], caches)
    # greedy generation picks what the oracle picks
    m.reset()
    got, _ = m.generate(e["prompt_ids"], 8)
    want, margins = om.generate(e["prompt_ids"], 8, capacity=64, cache_dtype=O.F16)
    for i, (a, b) in enumerate(zip(got[0].tolist(), want)):
        assert a == b, f"token {i}: device {a}, oracle {b}, the oracle's margin there {margins[i]:.4g}"


@pytest.mark.parametrize("cache", [capi.F32, capi.F16])
def test_qwen2_biases_on_queries_keys_and_values(golden_dir, cache):
    """The reference's qwen2 fixture (llm/llm_test.go:36-39): biases on q, k and v added behind the products and
    before the rotation (llm/model.go:251-258, nn/layers.go:49-55), rotation over halves. Every position of the
    prompt at once, then token by token through the caches, then greedy tokens: against the oracle's model, which
    multiplies with int8 activations as the device does."""
    path = os.path.join(golden_dir, "qwen2-exact.mim")
    prompt = [1, 79, 110, 99, 101, 363, 264, 315, 307, 280]
    gpu.lib()
    gpu.say(f"qwen2, cache dtype {cache}")
    m = load_mim(path, max_tokens=16, context=64, cache_dtype=cache)
    om = OL.Model.from_mim(MimFile(path))
    ocache = O.F32 if cache == capi.F32 else O.F16
    want = om.logits(prompt, om.new_caches(64, ocache), all=True)
    got = m.logits(prompt, all=True)[0]
    scale = np.abs(want).max()
    assert np.abs(got - want).max() <= 1e-4 * scale
    m.reset()
    caches = om.new_caches(64, ocache)
    for t in prompt:
        assert np.abs(m.logits([t])[0] - om.logits([t], caches)).max() <= 1e-4 * scale
    owant, margins = om.generate(prompt, 12, capacity=64, cache_dtype=ocache)
    # the decoding step three ways: launched operator by operator with the position from the host (2), its device-resident
    # form, where one launch adds the biases, rotates and writes the caches (1), and that form replayed from a graph (0, twice)
    lib = gpu.lib()
    try:
        for mode in (2, 1, 0, 0):
            gpu.say(f"qwen2, cache dtype {cache}: step mode {mode}")
            capi.check(lib.mi355x_tune(b"llama.step", mode))
            m.reset()
            toks, _ = m.generate(prompt, 12)
            assert toks[0].tolist() == owant, (mode, toks[0].tolist(), owant, min(margins))
    finally:
        capi.check(lib.mi355x_tune(b"llama.step", 0))


def test_some_but_not_all_biases_is_an_error(golden_dir):
    gpu.lib()
    path = os.path.join(golden_dir, "qwen2-exact.mim")
    f = MimFile(path)
    from mimir_amd.llama import config_from_metadata, _MIM_TO_ABI
    m = Llama(config_from_metadata(f.metadata, f["token_embd.weight"].shape[0], context=16))
    for name, t in f.tensors.items():
        if name.endswith(".weight"):
            m.set_tensor(name, _MIM_TO_ABI[t.dtype_name], t.data, int(np.prod(t.shape)))
    m.set_tensor("blk.0.attn_q.bias", capi.F32, f["blk.0.attn_q.bias"].data, int(np.prod(f["blk.0.attn_q.bias"].shape)))
    with pytest.raises(capi.Mi355xError) as ei:
        m.finalize(8)
    assert ei.value.status == capi.ERR_SHAPE


def test_q4_0_tensors_from_a_file_under_the_callers_code(tmp_path):
    """A .mim file whose Q4_0 tensors carry a container code that the caller names (the reference's fixtures
    hold none): load_mim uploads them as Q4_0 and the model decodes as the oracle's copy of it does."""
    from oracle.llama import Config, synthetic
    from tests.helpers import synthetic_llama_mim
    gpu.lib()
    oc = Config(embed=512, hidden=1024, layers=2, heads=4, kv_heads=2, head_dim=128, rope_dim=128, vocab=320, context=32, rope_base=500000.0)
    om = synthetic(oc, seed=5)
    path = str(tmp_path / "q4_0.mim")
    synthetic_llama_mim(path, om, q4_0_code=65)
    gpu.say("a .mim file with Q4_0 tensors")
    m = load_mim(path, max_tokens=8, q4_0_code=65, cache_dtype=capi.F16)
    prompt = [3, 200, 41, 7, 19]
    want = om.logits(prompt, om.new_caches(32, O.F16))
    got = m.logits(prompt)[0]
    assert np.abs(got - want).max() <= 1e-4 * np.abs(want).max()
    m.reset()
    toks, _ = m.generate(prompt, 8)
    owant, margins = om.generate(prompt, 8, capacity=32, cache_dtype=O.F16)
    assert toks[0].tolist() == owant, (toks[0].tolist(), owant, min(margins))


def test_errors_before_anything_is_queued(golden_dir):
    gpu.lib()
    m = load_mim(os.path.join(golden_dir, "spm.mim"), max_tokens=8, context=8)
    with pytest.raises(capi.Mi355xError) as ei:
        m.logits([1, 2, 400])  # llm/model.go:396-400
    assert ei.value.status == capi.ERR_INDEX
    with pytest.raises(capi.Mi355xError) as ei:
        m.logits(list(range(9)))
    assert ei.value.status == capi.ERR_SHAPE
    m.logits([1, 2, 3, 4, 5, 6, 7])
    with pytest.raises(capi.Mi355xError) as ei:  # a full cache (nn/transformer.go:408-411)
        m.logits([1, 2])
    assert ei.value.status == capi.ERR_SHAPE
    assert m.cache_len == 7


def _small_q4_config(batch, cache):
    c = capi.LlamaConfig()
    c.embed, c.hidden, c.layers, c.heads, c.kv_heads, c.head_dim, c.rope_dim, c.vocab = 512, 1792, 3, 4, 1, 128, 128, 1003
    c.context, c.interleaved, c.cache_dtype, c.batch = 96, 1, cache, batch
    c.rope_base, c.rope_scale, c.eps = 500000.0, 1.0, 1e-5
    return c


def _upload_synthetic(m: Llama, om: OL.Model):
    dt = {O.Q4_0: capi.Q4_0, O.Q8_0: capi.Q8_0, O.Q4_K: capi.Q4_K, O.Q6_K: capi.Q6_K}
    m.set_tensor("token_embd.weight", dt[om.embed.dtype], om.embed.data, om.embed.n * om.embed.k)
    m.set_tensor("output.weight", dt[om.output.dtype], om.output.data, om.output.n * om.output.k)
    m.set_tensor("output_norm.weight", capi.F32, om.norm, om.norm.size)
    for i, b in enumerate(om.blocks):
        p = f"blk.{i}."
        m.set_tensor(p + "attn_norm.weight", capi.F32, b.attn_norm, b.attn_norm.size)
        m.set_tensor(p + "ffn_norm.weight", capi.F32, b.ffn_norm, b.ffn_norm.size)
        for leaf, w in (("attn_q", b.q), ("attn_k", b.k), ("attn_v", b.v), ("attn_output", b.o), ("ffn_gate", b.gate), ("ffn_up", b.up), ("ffn_down", b.down)):
            m.set_tensor(p + leaf + ".weight", dt[w.dtype], w.data, w.n * w.k)


def _oracle_config(c):
    return OL.Config(arch="llama", embed=c.embed, hidden=c.hidden, layers=c.layers, heads=c.heads, kv_heads=c.kv_heads, head_dim=c.head_dim,
                     rope_dim=c.rope_dim, rope_base=c.rope_base, rope_scale=1.0, eps=c.eps, vocab=c.vocab, context=c.context)


def test_random_init_model_without_rounding_steps_is_close_everywhere():
    """Q4_0 linears, a Q4_0 output projection and a float32 cache: nothing on
    the way rounds to int8 or binary16, so the device and the CPU reference
    differ by float32 rounding alone: about 2e-7 of the largest logit at almost
    every position, which is also how far the float32 reference itself is from
    a float64 forward. One position of this prompt is ill-conditioned (the
    reference is 3e-5 from float64 there); it stays within 1e-3."""
    gpu.lib()
    c = _small_q4_config(1, capi.F32)
    om = OL.synthetic(_oracle_config(c), seed=0, output_dt=O.Q4_0)
    gpu.say("random-init q4_0 model, q4_0 output, f32 cache")
    m = Llama(c)
    _upload_synthetic(m, om)
    m.finalize(40)
    prompt = np.random.default_rng(0).integers(0, c.vocab, (1, 33))
    got = m.logits(prompt, all=True)[0]
    want = om.logits(prompt[0].tolist(), om.new_caches(c.context, O.F32), all=True)
    err = np.abs(got - want).max(1) / np.abs(want).max()
    assert err.max() <= 1e-3 and np.quantile(err, 0.9) <= 2e-6, err


@pytest.mark.parametrize("batch", [1, 3])
def test_random_init_q4_0_model_matches_oracle_and_greedy_tokens(batch):
    """A random-init decoder in the 8B model's proportions (heads of 128, four
    query heads a key head, SwiGLU 3.5x, theta 500000, Q4_0 linears, Q8_0
    embeddings and output), binary16 cache. The Q8_0 output projection rounds
    its input to int8 on both sides (backend/cpu/qmatmul.go:208-254), a step
    function: where a value sits on a rounding boundary, the last bit of the
    hidden state decides a quant, so single logits move by about 1e-3 of the
    largest. The bound is the reference's own for quantized weights, 2%
    (examples/llama/llama_test.go:177), with most positions far inside it; the
    greedy tokens are the same except where the reference's own top two logits
    are that close."""
    gpu.lib()
    c = _small_q4_config(batch, capi.F16)
    om = OL.synthetic(_oracle_config(c), seed=0)
    gpu.say(f"random-init q4_0 model batch={batch}")
    m = Llama(c)
    _upload_synthetic(m, om)
    m.finalize(40)
    rng = np.random.default_rng(0)
    prompts = rng.integers(0, c.vocab, (batch, 33))
    got = m.logits(prompts, all=True)
    for b in range(batch):
        want = om.logits(prompts[b].tolist(), om.new_caches(c.context, O.F16), all=True)
        scale = np.abs(want).max()
        err = np.abs(got[b] - want).max(1) / scale
        assert err.max() <= 0.02 and np.median(np.abs(got[b] - want)) <= 1e-5 * scale, (float(err.max()), err)
    m.reset()
    toks, _ = m.generate(prompts, 24)
    for b in range(batch):
        want, margins = om.generate(prompts[b].tolist(), 24, capacity=c.context, cache_dtype=O.F16)
        scale = 170.0
        for i, (a, w) in enumerate(zip(toks[b].tolist(), want)):
            assert a == w, f"token {i}: device {a}, oracle {w}, oracle's margin there {margins[i]:.4g}"


@pytest.mark.parametrize("batch,cache", [(1, capi.F32), (2, capi.F16)])
def test_fused_and_graph_replayed_steps_choose_the_per_operator_tokens(batch, cache):
    """The decoding step exists three times: per operator (what the logits tests
    above pin against the oracle), fused launches (norm with conversion, q|k|v
    in one product, rotation with the cache write, SwiGLU and residual
    epilogues), and those launches replayed as a graph that reads position and
    tokens from device memory. All three must choose the same tokens, replay
    after replay, and again on a second call that starts from another cache
    length with the graph the first call built."""
    lib = gpu.lib()
    c = _small_q4_config(batch, cache)
    om = OL.synthetic(_oracle_config(c), seed=1, output_dt=O.Q4_0)
    m = Llama(c)
    _upload_synthetic(m, om)
    m.finalize(40)
    rng = np.random.default_rng(5)
    runs = {}
    try:
        for mode in (2, 1, 0, 0):
            gpu.say(f"generate, step mode {mode}, batch {batch}")
            capi.check(lib.mi355x_tune(b"llama.step", mode))
            m.reset()
            prompts = np.random.default_rng(5).integers(0, c.vocab, (batch, 9))
            first, _ = m.generate(prompts, 30)
            assert m.cache_len == 9 + 29
            # a second call continues the same caches from where the first stopped
            more, _ = m.generate(first[:, -1:], 12)
            assert m.cache_len == 9 + 29 + 1 + 11
            runs.setdefault(mode, []).append(np.concatenate([first, more], 1))
    finally:
        capi.check(lib.mi355x_tune(b"llama.step", 0))
    # the per-operator steps against the oracle, then the others against them
    want, margins = om.generate(prompts[0].tolist(), 30, capacity=c.context, cache_dtype=O.F32 if cache == capi.F32 else O.F16)
    got = runs[2][0][0, :30].tolist()
    for i, (a, w) in enumerate(zip(got, want)):
        assert a == w, f"token {i}: device {a}, oracle {w}, oracle's margin there {margins[i]:.4g}"
    # attention splits the keys differently when the position comes from the
    # device (a fixed plan for the whole context), so a sum may round another
    # way; tokens differ only if two logits tie to that precision
    same = [np.array_equal(runs[2][0], r) for r in (runs[1][0], runs[0][0], runs[0][1])]
    assert np.array_equal(runs[0][0], runs[0][1])
    assert np.array_equal(runs[1][0], runs[0][0])
    assert all(same), (runs[2][0], runs[0][0])


@pytest.mark.parametrize("batch,output_dt", [(1, O.Q4_0), (2, O.Q4_0), (5, O.Q4_0), (16, O.Q8_0), (17, O.Q4_0)])
def test_logits_of_one_token_as_a_decoding_step(batch, output_dt):
    """One token a sequence goes through the decoding step's launches (of one and two sequences; of more through the operators'), one by one before a generation
    has recorded them and replayed after it, from an empty cache too, and leaves cache and logits as the per-operator pass does. A product is
    within 2e-7 of the float32 one either way and a model has some tens: 1e-5 of the largest logit; a Q8_0 head rounds x to a 127th of a block's largest (0.02)."""
    lib = gpu.lib()
    c = _small_q4_config(batch, capi.F16)
    om = OL.synthetic(_oracle_config(c), seed=3, output_dt=output_dt)
    m = Llama(c)
    _upload_synthetic(m, om)
    m.finalize(40)
    rng = np.random.default_rng(batch)
    prompts, one, two = rng.integers(0, c.vocab, (batch, 9)), rng.integers(0, c.vocab, (batch, 1)), rng.integers(0, c.vocab, (batch, 1))
    want = [batch - 1, 0]
    runs = {}
    try:
        for name, mode, recorded in (("operators", 2, False), ("launches", 0, False), ("replayed", 0, True), ("one by one", 1, True)):
            gpu.say(f"one token as a step: {name}, batch {batch}")
            capi.check(lib.mi355x_tune(b"llama.step", mode))
            if recorded:
                m.generate(prompts, 3)
            m.reset()
            first = m.logits(one)  # on empty caches
            m.reset()
            m.logits(prompts)
            runs[name] = [first, m.logits(one), m.logits_at(two, want), m.logits_at(one, [0, 0]), m.logits(prompts)]
            assert m.cache_len == 9 + 3 + 9
    finally:
        capi.check(lib.mi355x_tune(b"llama.step", 0))
    tol = 0.02 if output_dt == O.Q8_0 else 1e-5
    for name, got in runs.items():
        for i, (g, w) in enumerate(zip(got, runs["operators"])):
            assert g.shape == w.shape and np.abs(g - w).max() <= tol * np.abs(w).max(), (name, i, float(np.abs(g - w).max() / np.abs(w).max()))
    assert all(np.array_equal(a, b) for a, b in zip(runs["launches"], runs["replayed"]))
    with pytest.raises(RuntimeError):
        m.logits_at(one, [batch])


@pytest.mark.parametrize("batch,output_dt", [(3, O.Q8_0), (8, O.Q8_0), (16, O.Q4_0)])
def test_logits_of_one_token_of_several_sequences_are_the_operators(batch, output_dt):
    """Bit for bit: a Q8_0 head's rounding of x makes a step of any difference before it. With a recorded step at hand and without."""
    lib = gpu.lib()
    c = _small_q4_config(batch, capi.F16)
    om = OL.synthetic(_oracle_config(c), seed=4, output_dt=output_dt)
    m = Llama(c)
    _upload_synthetic(m, om)
    m.finalize(16)
    rng = np.random.default_rng(batch)
    prompts, one = rng.integers(0, c.vocab, (batch, 9)), rng.integers(0, c.vocab, (batch, 1))
    runs = []
    try:
        for mode, recorded in ((2, False), (0, False), (0, True)):
            gpu.say(f"one token of {batch} sequences, step mode {mode}")
            capi.check(lib.mi355x_tune(b"llama.step", mode))
            if recorded:
                m.generate(prompts, 3)
            m.reset()
            m.logits(prompts)
            runs.append([m.logits(one), m.logits(one)])
    finally:
        capi.check(lib.mi355x_tune(b"llama.step", 0))
    for got in runs[1:]:
        assert all(np.array_equal(g.view(np.uint32), w.view(np.uint32)) for g, w in zip(got, runs[0]))


@pytest.mark.parametrize("embed,batch", [(4160, 1), (8192, 1), (8192, 2)])
def test_rows_longer_than_one_step_through_the_fused_rotation(embed, batch):
    """A llama-layout model whose rows of x are longer than 4096: the q|k|v product with the rotation and the cache
    writes as its tail then runs on the whole-chip kernel with every row cut into chunks over wavefronts (4160: two
    unequal chunks), the chunks' sums meeting in LDS before the rotation, and the norm in front of it as a launch of
    its own. Logits against the oracle, then the three step modes and the finer-grained launch ("q4_0.stream" = 1)
    must choose the oracle's tokens."""
    lib = gpu.lib()
    c = capi.LlamaConfig()
    c.embed, c.hidden, c.layers, c.heads, c.kv_heads, c.head_dim, c.rope_dim, c.vocab = embed, 1792, 2, 4, 1, 128, 128, 1003
    c.context, c.interleaved, c.cache_dtype, c.batch = 64, 1, capi.F16, batch
    c.rope_base, c.rope_scale, c.eps = 500000.0, 1.0, 1e-5
    om = OL.synthetic(_oracle_config(c), seed=3, output_dt=O.Q4_0, centered=True)
    m = Llama(c)
    _upload_synthetic(m, om)
    m.finalize(16)
    prompts = np.random.default_rng(6).integers(0, c.vocab, (batch, 9))
    gpu.say(f"long rows: embed {embed}, batch {batch}: logits")
    got = m.logits(prompts, all=True)
    for b in range(batch):
        want = om.logits(prompts[b].tolist(), om.new_caches(c.context, O.F16), all=True)
        assert np.abs(got[b] - want).max() <= 1e-3 * np.abs(want).max()
    wants = [om.generate(prompts[b].tolist(), 24, capacity=c.context, cache_dtype=O.F16) for b in range(batch)]
    try:
        for mode, stream in ((2, 0), (1, 0), (0, 0), (0, 1)):
            gpu.say(f"long rows: embed {embed}, batch {batch}: step mode {mode}, q4_0.stream {stream}")
            capi.check(lib.mi355x_tune(b"llama.step", mode))
            capi.check(lib.mi355x_tune(b"q4_0.stream", stream))
            m.reset()
            toks, _ = m.generate(prompts, 24)
            for b in range(batch):
                want, margins = wants[b]
                gotb = toks[b].tolist()
                first = next((i for i in range(24) if gotb[i] != want[i]), None)
                assert first is None, f"mode {mode} stream {stream} sequence {b} token {first}: device {gotb[first]}, oracle {want[first]}, margin {margins[first]:.4g}"
    finally:
        capi.check(lib.mi355x_tune(b"llama.step", 0))
        capi.check(lib.mi355x_tune(b"q4_0.stream", 0))


@pytest.mark.parametrize("batch", [2, 5, 8, 11, 16])
def test_batch_step_that_reads_weights_once_chooses_the_same_tokens(batch):
    """Two to sixty-four sequences decode with products that read each weight once per eight of them (int8 matrix
    cores, the output and down projections cut into two shares of K that the next norm adds; the rotation
    with the cache writes and SiLU * up with its conversion ride on the products, or run as launches of
    their own). Their integers are those of the one-sequence kernels, only float32 sums are ordered differently, so the tokens
    must be those of the one-sequence kernels run per sequence (llama.rows = 1), of the per-operator path,
    and, up to near-ties, the oracle's."""
    lib = gpu.lib()
    c = _small_q4_config(batch, capi.F16)
    om = OL.synthetic(_oracle_config(c), seed=2, output_dt=O.Q4_0)
    m = Llama(c)
    _upload_synthetic(m, om)
    m.finalize(40)
    prompts = np.random.default_rng(17).integers(0, c.vocab, (batch, 11))
    runs = {}
    try:
        for name, key, v in (("rows graph", b"llama.rows", 0), ("rows launches", b"llama.step", 1), ("rows without riders", b"llama.rows", 2),
                             ("per sequence", b"llama.rows", 1), ("per operator", b"llama.step", 2)):
            capi.check(lib.mi355x_tune(b"llama.rows", 0))
            capi.check(lib.mi355x_tune(b"llama.step", 0))
            capi.check(lib.mi355x_tune(key, v))
            gpu.say(f"generate batch {batch}: {name}")
            m.reset()
            first, _ = m.generate(prompts, 30)
            more, _ = m.generate(first[:, -1:], 10)  # the graph of the first call, from another cache length
            runs[name] = np.concatenate([first, more], 1)
    finally:
        capi.check(lib.mi355x_tune(b"llama.rows", 0))
        capi.check(lib.mi355x_tune(b"llama.step", 0))
    for name in ("rows launches", "rows without riders", "per sequence", "per operator"):
        assert np.array_equal(runs["rows graph"], runs[name]), (name, runs["rows graph"], runs[name])
    for b in range(batch):
        want, margins = om.generate(prompts[b].tolist(), 30, capacity=c.context, cache_dtype=O.F16)
        for i, (a, w) in enumerate(zip(runs["rows graph"][b, :30].tolist(), want)):
            assert a == w, f"token {i}: device {a}, oracle {w}, oracle's margin there {margins[i]:.4g}"


@pytest.mark.parametrize("linear_dt,batch,cache", [(O.Q4_0, 1, capi.F32), (O.Q4_0, 8, capi.F16), (O.Q4_K, 3, capi.F16), (O.Q6_K, 1, capi.F32)])
def test_steps_of_a_context_of_96_share_its_keys_between_two_workgroups(linear_dt, batch, cache):
    """65 to 128 positions are two shares of the keys ("attention.share": 64), whose hand-over leaves the result in each form that a step
    reads. The caches that ten steps from position 70 on fill give the logits of a model held to two shares bit for bit; held to one, which adds in another
    order, those of a difference of some 1e-7 (K-quants: 2 %, the bound of quantized weights, since their int8 rounding is a step)."""
    lib = gpu.lib()
    c = _small_q4_config(batch, cache)
    om = OL.synthetic(_oracle_config(c), seed=4, linear_dt=linear_dt, output_dt=O.Q4_0)
    prompts = np.random.default_rng(29).integers(0, c.vocab, (batch, 70))
    got = {}
    try:
        capi.check(lib.mi355x_tune(b"llama.step", 1))
        for shares in (0, 2, 1):
            gpu.say(f"context of 96, dtype {linear_dt}, batch {batch}, shares {shares}")
            capi.check(lib.mi355x_tune(b"attention.splits", shares))  # before the model sizes its workspaces
            m = Llama(c)
            _upload_synthetic(m, om)
            m.finalize(80)
            m.generate(prompts, 11)
            capi.check(lib.mi355x_tune(b"attention.splits", 0))
            got[shares] = m.logits(np.full((batch, 1), 7))
            m.close()
    finally:
        capi.check(lib.mi355x_tune(b"attention.splits", 0))
        capi.check(lib.mi355x_tune(b"llama.step", 0))
    assert np.array_equal(got[0], got[2])
    if linear_dt == O.Q4_0:  # (int8 rounding may swallow the difference)
        assert not np.array_equal(got[0], got[1])
    scale = np.abs(got[1]).max()
    assert np.abs(got[0] - got[1]).max() <= (1e-3 if linear_dt == O.Q4_0 else 0.02) * scale


@pytest.mark.parametrize("heads,kv_heads,head_dim,cache,batch", [(2, 1, 128, capi.F16, 1), (4, 1, 128, capi.F32, 3), (3, 3, 64, capi.F16, 1), (8, 1, 64, capi.F32, 2)])
def test_shares_of_the_keys_are_put_together_for_every_number_of_them(heads, kv_heads, head_dim, cache, batch):
    """A step's attention in up to 40 shares, handed over by flagged pairs (requests of 4, 8, 12 and 16 shares, and several of 16) or by tickets, of
    heads that do not fill a workgroup's four: the logits of a model held to one share, to 1e-5 of the largest (float32 sums in another order, some 1e-7
    each, of three blocks). Shares past the last key are empty; a second step finds the slots clear."""
    lib = gpu.lib()
    c = _small_q4_config(batch, cache)
    c.heads, c.kv_heads, c.head_dim, c.rope_dim, c.context = heads, kv_heads, head_dim, head_dim, 200
    om = OL.synthetic(_oracle_config(c), seed=6, output_dt=O.Q4_0)
    prompts = np.random.default_rng(31).integers(0, c.vocab, (batch, 70))
    want = None
    try:
        for handover in (0, 1):
            capi.check(lib.mi355x_tune(b"attention.handover", handover))
            for shares in (1, 2, 4, 5, 6, 9, 10, 13, 14, 17, 18, 33, 34, 40):
                gpu.say(f"{heads} heads of {head_dim}, batch {batch}, {shares} shares, handover {handover}")
                capi.check(lib.mi355x_tune(b"attention.splits", shares))  # before the model sizes its workspaces
                m = Llama(c)
                _upload_synthetic(m, om)
                m.finalize(70)
                m.logits(prompts)
                got = [m.logits(np.full((batch, 1), 7)) for _ in range(3)]
                m.close()
                want = want or got
                for g, w in zip(got, want):
                    assert np.abs(g - w).max() <= 1e-5 * np.abs(w).max(), (shares, handover, float(np.abs(g - w).max() / np.abs(w).max()))
    finally:
        capi.check(lib.mi355x_tune(b"attention.splits", 0))
        capi.check(lib.mi355x_tune(b"attention.handover", 0))


@pytest.mark.parametrize("embed,batch,rows", [(512, 1, 3), (512, 3, 2), (4160, 2, 5), (8192, 1, 9)])
def test_the_heads_norm_and_conversion_in_one_launch_are_the_two_launches(embed, batch, rows):
    """A block of zeros leaves a token's embedding as it is: the logits of a Q8_0 head are, bit for bit, those of rmsnorm, conversion and product one by one, for all rows of a
    call (a row's length apart) and for the last of each sequence (further apart)."""
    lib = gpu.lib()
    c = _small_q4_config(batch, capi.F16)
    c.embed, c.hidden, c.layers, c.heads, c.kv_heads, c.head_dim, c.rope_dim, c.vocab, c.interleaved = embed, 64, 1, 1, 1, 64, 64, 515, 0
    om = OL.synthetic(OL.Config(embed=embed, hidden=64, layers=1, heads=1, kv_heads=1, head_dim=64, rope_dim=64, rope_base=c.rope_base, rope_scale=1.0, eps=c.eps,
                                vocab=c.vocab, context=c.context), seed=9, output_dt=O.Q8_0)
    b = om.blocks[0]
    for w in (b.o, b.down):
        w.data[:] = 0
    m = Llama(c)
    _upload_synthetic(m, om)
    m.finalize(batch * rows)
    tokens = np.random.default_rng(31).integers(0, c.vocab, (batch, rows))
    gpu.say(f"head embed={embed} batch={batch} rows={rows}")
    every = m.logits(tokens, all=True)
    m.reset()
    last = m.logits(tokens)
    x = gpu.dev(np.ascontiguousarray(O.dequantize(O.Q8_0, om.embed.data).reshape(c.vocab, embed)[tokens.reshape(-1)]))
    normed, norm = torch.empty_like(x), gpu.dev(om.norm.reshape(-1).astype(np.float32))
    capi.check(lib.mi355x_rmsnorm(x.data_ptr(), norm.data_ptr(), normed.data_ptr(), batch * rows, embed, c.eps, gpu.stream()))
    buf, ptr = gpu.dev_bytes_at(om.output.data, 4)
    want = gpu.qgemv_act(O.Q8_0, ptr, normed, c.vocab, embed).reshape(batch, rows, c.vocab)
    assert np.array_equal(np.asarray(every).reshape(want.shape).view(np.uint32), want.view(np.uint32))
    assert np.array_equal(np.asarray(last).reshape(batch, c.vocab).view(np.uint32), np.ascontiguousarray(want[:, -1]).view(np.uint32))


@pytest.mark.parametrize("embed,vocab,batch", [(512, 8192, 1), (512, 8195, 3), (4160, 8195, 2), (512, 70001, 9)])
def test_the_choice_brings_in_the_next_embedding(embed, vocab, batch):
    """From 8192 tokens on, the launch that chooses a step's tokens also records them, moves the position on and looks the next step's
    embeddings up: tokens of the graph and of its launches equal to the per-operator path's, over three calls with one of logits between."""
    lib = gpu.lib()
    c = _small_q4_config(batch, capi.F16)
    c.embed, c.hidden, c.layers, c.vocab, c.context = embed, 320, 1, vocab, 32
    if embed > 512:
        c.heads, c.kv_heads, c.head_dim, c.rope_dim, c.interleaved = 2, 1, 64, 64, 0
    om = OL.synthetic(_oracle_config(c) if embed == 512 else OL.Config(
        embed=c.embed, hidden=c.hidden, layers=c.layers, heads=c.heads, kv_heads=c.kv_heads, head_dim=c.head_dim, rope_dim=c.rope_dim,
        rope_base=c.rope_base, rope_scale=1.0, eps=c.eps, vocab=c.vocab, context=c.context), seed=3, output_dt=O.Q8_0)
    m = Llama(c)
    _upload_synthetic(m, om)
    m.finalize(16)
    prompts = np.random.default_rng(23).integers(0, c.vocab, (batch, 5))
    runs = []
    try:
        for mode in (0, 1, 2):
            capi.check(lib.mi355x_tune(b"llama.step", mode))
            m.reset()
            first, _ = m.generate(prompts, 8)
            more, _ = m.generate(first[:, -1:], 6)
            last = m.logits(more[:, -1:])
            again, _ = m.generate(last.argmax(-1).reshape(batch, 1).astype(np.int32), 3)
            runs.append(np.concatenate([first, more, again], 1))
    finally:
        capi.check(lib.mi355x_tune(b"llama.step", 0))
    assert np.array_equal(runs[0], runs[1]) and np.array_equal(runs[0], runs[2])


@pytest.mark.parametrize("batch", [1, 3])
def test_a_generation_whose_choices_give_up_on_their_candidates(batch):
    """With no polls, recorded so, and with as many as ever on the same workspace: the same tokens."""
    lib = gpu.lib()
    c = _small_q4_config(batch, capi.F16)
    c.vocab, c.context = 9000, 32
    om = OL.synthetic(_oracle_config(c), seed=3, output_dt=O.Q8_0)
    prompts = np.random.default_rng(23).integers(0, c.vocab, (batch, 5))
    runs = []
    try:
        for spins in ((-1,), (0, -1)):
            m = Llama(c)
            _upload_synthetic(m, om)
            m.finalize(16)
            for n in spins:
                capi.check(lib.mi355x_tune(b"argmax.spins", n))
                capi.check(lib.mi355x_tune(b"llama.step", 1 if n < 0 else 0))
                gpu.say(f"generation of {batch}, argmax.spins {n}")
                m.reset()
                runs.append(m.generate(prompts, 12)[0])
            m.close()
    finally:
        capi.check(lib.mi355x_tune(b"argmax.spins", -1))
        capi.check(lib.mi355x_tune(b"llama.step", 0))
    assert np.array_equal(runs[0], runs[1]) and np.array_equal(runs[0], runs[2])


@pytest.mark.parametrize("linear_dt,batch", [(O.Q4_K, 1), (O.Q6_K, 1), (O.Q4_K, 2), (O.Q6_K, 3)])
def test_kquant_steps_with_norms_and_swiglu_in_the_products_have_the_bits_of_those_without(linear_dt, batch):
    """One to three sequences: the norms and SwiGLU as parts of the products (rows of three super-blocks, 1280 results) against launches of their own."""
    lib = gpu.lib()
    c = _small_q4_config(batch, capi.F16)
    c.embed, c.hidden, c.layers, c.heads, c.kv_heads, c.head_dim, c.rope_dim, c.vocab, c.context = 768, 1280, 2, 6, 2, 128, 128, 301, 32
    om = OL.synthetic(_oracle_config(c), seed=5, linear_dt=linear_dt)
    m = Llama(c)
    _upload_synthetic(m, om)
    m.finalize(8 * batch)
    prompts = np.random.default_rng(7).integers(0, c.vocab, (batch, 5))
    runs = []
    try:
        for stream in (0, 1):
            capi.check(lib.mi355x_tune(b"kquant.stream", stream))
            capi.check(lib.mi355x_tune(b"llama.step", 1))  # launches, which a graph of the other choice would stand in for
            gpu.say(f"steps dt={linear_dt} batch={batch} stream={stream}")
            m.reset()
            tokens, _ = m.generate(prompts, 12)
            runs.append((tokens, np.asarray(m.logits(tokens[:, -1:]))))
    finally:
        capi.check(lib.mi355x_tune(b"kquant.stream", 0))
        capi.check(lib.mi355x_tune(b"llama.step", 0))
    assert np.array_equal(runs[0][0], runs[1][0]) and np.array_equal(runs[0][1].view(np.uint32), runs[1][1].view(np.uint32))


@pytest.mark.parametrize("embed", [2304, 3072, 4096])
@pytest.mark.parametrize("linear_dt", [O.Q4_K, O.Q6_K])
def test_kquant_norms_in_the_products_of_several_tasks(linear_dt, embed):
    """Rows of nine, twelve and sixteen super-blocks, a norm's three tasks (of which two wavefronts share one) and four, two turns of them for three sequences, rows of Q6_K cut over two
    wavefronts behind a norm: caches and logits of one to three sequences bit for bit those of launches of their own."""
    lib = gpu.lib()
    c = _small_q4_config(1, capi.F16)
    c.embed, c.hidden, c.layers, c.heads, c.kv_heads, c.vocab, c.context = embed, 1280, 2, 6, 2, 301, 32
    om = OL.synthetic(_oracle_config(c), seed=5, linear_dt=linear_dt)
    for batch in (1, 2, 3):
        c.batch = batch
        m = Llama(c)
        _upload_synthetic(m, om)
        m.finalize(8 * batch)
        prompts = np.random.default_rng(7).integers(0, c.vocab, (batch, 5))
        runs = []
        try:
            capi.check(lib.mi355x_tune(b"llama.step", 1))
            for stream in (8, 1):
                capi.check(lib.mi355x_tune(b"kquant.stream", stream))
                gpu.say(f"steps dt={linear_dt} embed={embed} batch={batch} stream={stream}")
                m.reset()
                tokens, _ = m.generate(prompts, 8)
                capi.check(lib.mi355x_tune(b"kquant.stream", 1))
                runs.append((tokens, np.asarray(m.logits(tokens[:, -1:]))))
        finally:
            capi.check(lib.mi355x_tune(b"kquant.stream", 0))
            capi.check(lib.mi355x_tune(b"llama.step", 0))
        m.close()
        assert np.array_equal(runs[0][0], runs[1][0]) and np.array_equal(runs[0][1].view(np.uint32), runs[1][1].view(np.uint32))


@pytest.mark.parametrize("embed,hidden,heads", [(4096, 4608, 36), (2304, 14336, 4), (256, 768, 4)])
def test_steps_of_two_q4_0_sequences_by_the_kernel_for_few_rows(embed, hidden, heads):
    """Two sequences: rows of a wavefront's 64 pairs of blocks and of more (72 and 224, cut over two and four wavefronts), of converted rows with the residual, of two norm items a
    thread; and rows of four pairs. Tokens of the steps by the kernel for eight rows, logits of the next token within 1e-5 of the largest (a product is within 2e-7, and a model has some tens)."""
    lib = gpu.lib()
    c = _small_q4_config(2, capi.F16)
    c.embed, c.hidden, c.layers, c.heads, c.vocab, c.context = embed, hidden, 2, heads, 515, 40
    om = OL.synthetic(_oracle_config(c), seed=9, output_dt=O.Q4_0)
    m = Llama(c)
    _upload_synthetic(m, om)
    m.finalize(16)
    prompts = np.random.default_rng(8).integers(0, c.vocab, (2, 7))
    runs = []
    try:
        for few, step in ((1, 1), (0, 1), (0, 0)):
            capi.check(lib.mi355x_tune(b"q4_0.few", few))
            capi.check(lib.mi355x_tune(b"llama.step", step))
            gpu.say(f"two sequences of {embed} features, few={few}, step={step}")
            m.reset()
            tokens, _ = m.generate(prompts, 9)
            runs.append((tokens, m.logits(tokens[:, -1:])))
    finally:
        capi.check(lib.mi355x_tune(b"q4_0.few", 0))
        capi.check(lib.mi355x_tune(b"llama.step", 0))
    for tokens, logits in runs[1:]:
        assert np.array_equal(tokens, runs[0][0]) and np.abs(logits - runs[0][1]).max() <= 1e-5 * np.abs(runs[0][1]).max()
    assert np.array_equal(runs[1][1], runs[2][1]) and not np.array_equal(runs[0][1], runs[1][1])


def test_fused_steps_without_their_riders_choose_the_per_operator_tokens():
    """The fused step lets the rotation, the norms and the conversion of SwiGLU's results ride on the products
    only where their shapes allow: interleaved pairs, rows of x one step of a wavefront long. A model with
    half-split pairs (qwen2's layout) and 4160 features takes the separate launches instead, and must choose the
    same tokens as the per-operator path."""
    lib = gpu.lib()
    c = capi.LlamaConfig()
    c.embed, c.hidden, c.layers, c.heads, c.kv_heads, c.head_dim, c.rope_dim, c.vocab = 4160, 320, 2, 2, 1, 64, 64, 301
    c.context, c.interleaved, c.cache_dtype, c.batch = 48, 0, capi.F16, 2
    c.rope_base, c.rope_scale, c.eps = 10000.0, 1.0, 1e-5
    oc = OL.Config(arch="qwen2", embed=c.embed, hidden=c.hidden, layers=c.layers, heads=c.heads, kv_heads=c.kv_heads, head_dim=c.head_dim,
                   rope_dim=c.rope_dim, rope_base=c.rope_base, rope_scale=1.0, eps=c.eps, vocab=c.vocab, context=c.context)
    om = OL.synthetic(oc, seed=3, output_dt=O.Q4_0)
    m = Llama(c)
    _upload_synthetic(m, om)
    m.finalize(16)
    prompts = np.random.default_rng(9).integers(0, c.vocab, (2, 7))
    runs = {}
    try:
        for mode in (2, 1, 0):
            gpu.say(f"generate without riders, step mode {mode}")
            capi.check(lib.mi355x_tune(b"llama.step", mode))
            m.reset()
            runs[mode], _ = m.generate(prompts, 20)
    finally:
        capi.check(lib.mi355x_tune(b"llama.step", 0))
    want, margins = om.generate(prompts[0].tolist(), 20, capacity=c.context, cache_dtype=O.F16)
    for i, (a, w) in enumerate(zip(runs[2][0].tolist(), want)):
        assert a == w, f"token {i}: device {a}, oracle {w}, oracle's margin there {margins[i]:.4g}"
    assert np.array_equal(runs[1], runs[2]) and np.array_equal(runs[0], runs[2])


@pytest.mark.parametrize("linear_dt,batch,heads,head_dim", [(O.Q4_K, 1, 4, 64), (O.Q6_K, 2, 4, 64), (O.Q8_0, 1, 4, 64), (O.Q4_K, 5, 4, 64),
                                                            (O.Q4_K, 11, 4, 64), (O.Q6_K, 9, 4, 64), (O.Q4_K, 1, 4, 128), (O.Q6_K, 3, 8, 64),
                                                            (O.Q4_K, 9, 16, 128)])
def test_k_quant_and_q8_0_models_decode_from_a_graph(linear_dt, batch, heads, head_dim):
    """Models whose linears are not Q4_0 take the generic decoding step: q|k|v and gate|up as one product
    each over weights kept together, norm and SwiGLU with the int8 conversion in the same launch (K-quants),
    residuals in the products' epilogues, the position on the device, the whole step replayed as a graph. It
    must choose the tokens of the per-operator path (position from the host) and of the oracle. Where the query
    heads of a key-value head are whole super-blocks of 256 (the last three shapes), attention leaves its result
    in the int8 form the K-quant output projection reads."""
    lib = gpu.lib()
    c = capi.LlamaConfig()
    c.embed, c.hidden, c.layers, c.heads, c.kv_heads, c.head_dim, c.rope_dim, c.vocab = 512, 1024, 2, heads, 2, head_dim, head_dim, 301
    c.context, c.interleaved, c.cache_dtype, c.batch = 64, 1, capi.F16, batch
    c.rope_base, c.rope_scale, c.eps = 10000.0, 1.0, 1e-5
    om = OL.synthetic(_oracle_config(c), seed=7, linear_dt=linear_dt)
    m = Llama(c)
    _upload_synthetic(m, om)
    m.finalize(16)
    prompts = np.random.default_rng(11).integers(0, c.vocab, (batch, 6))
    runs = {}
    try:
        for mode in (2, 1, 0, 0):
            gpu.say(f"generate dtype {linear_dt}, step mode {mode}, batch {batch}")
            capi.check(lib.mi355x_tune(b"llama.step", mode))
            m.reset()
            first, _ = m.generate(prompts, 20)
            more, _ = m.generate(first[:, -1:], 9)  # a second call continues the caches (and replays the graph)
            runs.setdefault(mode, []).append(np.concatenate([first, more], 1))
    finally:
        capi.check(lib.mi355x_tune(b"llama.step", 0))
    want, margins = om.generate(prompts[0].tolist(), 20, capacity=c.context, cache_dtype=O.F16)
    for i, (a, w) in enumerate(zip(runs[2][0][0, :20].tolist(), want)):
        assert a == w, f"token {i}: device {a}, oracle {w}, oracle's margin there {margins[i]:.4g}"
    assert np.array_equal(runs[1][0], runs[2][0]) and np.array_equal(runs[0][0], runs[2][0]) and np.array_equal(runs[0][1], runs[2][0])


@pytest.mark.parametrize("arch,heads,head_dim,rope_dim,cache", [
    ("llama", 4, 128, 64, capi.F32),   # neighbouring features turn, the upper half passes
    ("qwen2", 4, 128, 128, capi.F32),  # halves turn against each other
    ("qwen2", 8, 64, 48, capi.F16),    # of a head in part, a binary16 cache
    ("llama", 8, 36, 36, capi.F32),    # heads that are no whole eights of features: the launches apart
])
def test_a_prompts_rotation_and_cache_writes(arch, heads, head_dim, rope_dim, cache):
    """Two sequences, two calls, the second behind the first's positions: logits of every position against the oracle (binary16 rounds the cache on
    both sides, so a value on a boundary moves a logit by 2^-11 of a key: the bound there is the one of the other binary16 tests)."""
    gpu.lib()
    c = _small_q4_config(2, cache)
    c.heads, c.kv_heads, c.head_dim, c.rope_dim, c.interleaved = heads, heads // 4, head_dim, rope_dim, int(arch == "llama")
    cfg = _oracle_config(c)
    cfg.arch = arch
    om = OL.synthetic(cfg, seed=3, output_dt=O.Q4_0)
    gpu.say(f"prompt rotation {arch} {heads} x {head_dim}, {rope_dim} turn")
    m = Llama(c)
    _upload_synthetic(m, om)
    m.finalize(40)
    prompts = np.random.default_rng(3).integers(0, c.vocab, (2, 38))
    got = np.concatenate([m.logits(prompts[:, :33], all=True), m.logits(prompts[:, 33:], all=True)], 1)
    odt = O.F32 if cache == capi.F32 else O.F16
    for b in range(2):
        caches = om.new_caches(c.context, odt)
        want = np.concatenate([om.logits(prompts[b, :33].tolist(), caches, all=True), om.logits(prompts[b, 33:].tolist(), caches, all=True)])
        err = np.abs(got[b] - want).max(1) / np.abs(want).max()
        assert err.max() <= (1e-3 if cache == capi.F32 else 0.02) and np.median(err) <= 1e-5, err


@pytest.mark.parametrize("linear_dt,batch,tokens", [(O.Q4_K, 1, 5), (O.Q4_K, 2, 10), (O.Q6_K, 1, 90), (O.Q4_K, 2, 150), (O.Q6_K, 3, 95)])
def test_a_prompt_by_k_quants_takes_matrices_of_one_x_together(linear_dt, batch, tokens):
    """q, k and v, gate and up as one product each, residuals added as products are stored, x converted by the norms and SwiGLU: by the kernels for a row,
    for a few (up to 8, 20, 90 rows) and the tiled one (90 to 300). Against the oracle, whose int8 rounding of x is the same: a value on a
    boundary moves a quant, a 127th of its super-block's largest, which three layers and 8 products of them carry to some 1e-3 of a logit; 5 % holds any few."""
    gpu.lib()
    c = _small_q4_config(batch, capi.F32)
    c.context = 160
    om = OL.synthetic(_oracle_config(c), seed=4, linear_dt=linear_dt)
    gpu.say(f"k-quant prompt dt={linear_dt} {batch} x {tokens}")
    m = Llama(c)
    _upload_synthetic(m, om)
    m.finalize(tokens)
    prompts = np.random.default_rng(tokens).integers(0, c.vocab, (batch, tokens))
    got = m.logits(prompts, all=True)
    for b in range(batch):
        want = om.logits(prompts[b].tolist(), om.new_caches(c.context, O.F32), all=True)
        err = np.abs(got[b] - want).max(1) / np.abs(want).max()
        assert err.max() <= 0.05 and np.median(err) <= 0.01, err


@pytest.mark.parametrize("linear_dt,batch,tokens", [(O.Q4_K, 11, 3), (O.Q6_K, 9, 5), (O.Q4_K, 2, 33), (O.Q6_K, 1, 77)])
def test_k_quant_products_of_some_rows_in_a_decoder(linear_dt, batch, tokens):
    """Prompts and steps whose products take W once for up to 64 rows, x left in the order of their lanes by the norms, SwiGLU and the conversion, the
    residual added as they store: the same integers and the same sums in the same order, so the same bits as by the other kernels."""
    lib = gpu.lib()
    c = _small_q4_config(batch, capi.F32)
    c.context = 100
    m = Llama(c)
    _upload_synthetic(m, OL.synthetic(_oracle_config(c), seed=4, linear_dt=linear_dt, output_dt=linear_dt))
    m.finalize(tokens)
    prompts = np.random.default_rng(tokens).integers(0, c.vocab, (batch, tokens))
    runs = []
    try:
        for mode in (1, 2, 0):
            gpu.say(f"k-quant rows in a decoder, dtype {linear_dt} {batch} x {tokens}, mode {mode}")
            capi.check(lib.mi355x_tune(b"kquant.shared", mode))
            capi.check(lib.mi355x_tune(b"llama.step", 1))  # launches, which a graph of the first mode would stand in for
            m.reset()
            logits = m.logits(prompts, all=True)
            m.reset()
            chosen = m.generate(prompts, 6)[0]
            capi.check(lib.mi355x_tune(b"kquant.shared", 1))
            runs.append((logits, chosen, m.logits(chosen[:, -1:])))  # by the same kernels from what the steps have left in the caches
    finally:
        capi.check(lib.mi355x_tune(b"kquant.shared", 0))
        capi.check(lib.mi355x_tune(b"llama.step", 0))
    for logits, chosen, after in runs[1:]:
        assert np.array_equal(logits.view(np.uint32), runs[0][0].view(np.uint32)) and np.array_equal(chosen, runs[0][1])
        assert np.array_equal(after.view(np.uint32), runs[0][2].view(np.uint32))


@pytest.mark.parametrize("linear_dt", [O.Q4_K, O.Q6_K, O.Q8_0, O.Q4_0])
def test_a_prompt_whose_products_round_to_int8_keeps_the_order_of_attentions_sums(linear_dt):
    """Rounding to int8 makes a step of a difference in the last place: a decoder of such products takes attention of a prompt over a binary16 cache on float32
    operands, bit for bit as the setting that has every call there does. One of Q4_0 products does not."""
    lib = gpu.lib()
    c = _small_q4_config(2, capi.F16)
    om = OL.synthetic(_oracle_config(c), seed=6, linear_dt=linear_dt, output_dt=O.Q4_0)
    gpu.say(f"prompt attention of a decoder by dtype {linear_dt}")
    m = Llama(c)
    _upload_synthetic(m, om)
    m.finalize(90)
    prompts = np.random.default_rng(6).integers(0, c.vocab, (2, 90))
    got = m.logits(prompts, all=True)
    try:
        capi.check(lib.mi355x_tune(b"attention.prompt", 2))
        m.reset()
        assert np.array_equal(m.logits(prompts, all=True), got) == (linear_dt != O.Q4_0)
    finally:
        capi.check(lib.mi355x_tune(b"attention.prompt", 1))


@pytest.mark.parametrize("linear_dt,batch,first,arch,biased,rope_dim,cache", [
    (O.Q4_K, 2, 70, "qwen2", True, 128, capi.F16),   # halves turn against each other behind a bias, on rows as far apart as q, k and v are wide
    (O.Q6_K, 1, 3, "qwen2", True, 64, capi.F32),     # a few rows, half of a head turning
    (O.Q6_K, 3, 67, "llama", False, 128, capi.F16),  # neighbours turn
])
def test_k_quant_prompts_together_are_their_products_apart_bit_for_bit(linear_dt, batch, first, arch, biased, rope_dim, cache):
    """A K-quant prompt's launches (q, k and v as one product, gate and up as another, biases, rotation and cache writes in one launch, norms and SwiGLU that round to
    int8, residuals added as products are stored) against the library's operators one by one, whose products have the CPU's bits as these have: every logit of two
    calls, the second behind the first's positions, is the same."""
    lib = gpu.lib()
    c = _small_q4_config(batch, cache)
    c.interleaved, c.rope_dim = int(arch == "llama"), rope_dim
    om = OL.synthetic(_oracle_config(c), seed=8, linear_dt=linear_dt, output_dt=O.Q6_K)
    rng = np.random.default_rng(first)
    biases = [[rng.normal(size=w.n).astype(np.float32) for w in (b.q, b.k, b.v)] if biased else None for b in om.blocks]
    gpu.say(f"k-quant prompt together and apart, dt={linear_dt} {batch} x {first} {arch}")
    m = Llama(c)
    _upload_synthetic(m, om)
    for i, three in enumerate(biases):
        for leaf, v in zip(("attn_q", "attn_k", "attn_v"), three or ()):
            m.set_tensor(f"blk.{i}.{leaf}.bias", capi.F32, v, v.size)
    m.finalize(max(first, 5))
    weights = [{leaf: gpu.dev_bytes_at(w.data, 0) + (w,) for leaf, w in (("q", b.q), ("k", b.k), ("v", b.v), ("o", b.o), ("gate", b.gate), ("up", b.up), ("down", b.down))}
               for b in om.blocks]
    output = gpu.dev_bytes_at(om.output.data, 0) + (om.output,)
    D, H, HK = c.head_dim, c.heads, c.kv_heads
    cos, sin = O.rope_angles(rope_dim, c.rope_base, 0, c.context)
    kept = [[np.zeros((batch, HK, c.context, D), np.uint16 if cache == capi.F16 else np.float32) for _ in range(2)] for _ in om.blocks]

    def times(x, weight):
        _, ptr, w = weight
        return gpu.qgemv(linear_dt if w is not om.output else O.Q6_K, ptr, gpu.dev(x), w.n, w.k)

    def swiglu(gate, up):
        gd, ud = gpu.dev(gate), gpu.dev(up)
        out = torch.empty_like(gd)
        capi.check(lib.mi355x_swiglu(gd.data_ptr(), ud.data_ptr(), out.data_ptr(), gate.shape[0], gate.shape[1], gate.shape[1], gpu.stream()))
        gpu.sync()
        return out.cpu().numpy()

    def apart(tokens, past):
        s = tokens.shape[1]
        x = O.dequantize(om.embed.dtype, om.embed.data).reshape(c.vocab, c.embed)[tokens.reshape(-1)].copy()
        for b, w, three, caches in zip(om.blocks, weights, biases, kept):
            h = ops.rmsnorm(x, b.attn_norm, c.eps)
            parts = [times(h, w[leaf]) for leaf in "qkv"]
            if three:
                parts = [p + v for p, v in zip(parts, three)]
            q, k, v = (np.ascontiguousarray(p.reshape(batch, s, -1, D).transpose(0, 2, 1, 3)) for p in parts)
            q, k = (ops.rope(t, cos, sin, rope_dim, arch == "llama", past) for t in (q, k))
            for kept_rows, new in zip(caches, (k, v)):
                kept_rows[:, :, past:past + s] = O.f32_to_f16(new) if cache == capi.F16 else new
            o, _ = ops.attention(q, *caches, 1 / np.sqrt(D), causal=True, offset=past, kv_dt=cache, k_len=past + s)
            x = x + times(np.ascontiguousarray(o.transpose(0, 2, 1, 3)).reshape(batch * s, H * D), w["o"])
            h = ops.rmsnorm(x, b.ffn_norm, c.eps)
            x = x + times(swiglu(times(h, w["gate"]), times(h, w["up"])), w["down"])
        return times(ops.rmsnorm(x, om.norm, c.eps), output).reshape(batch, s, c.vocab)

    prompts = rng.integers(0, c.vocab, (batch, first + 5))
    try:
        capi.check(lib.mi355x_tune(b"attention.prompt", 2))  # the order of sums that a decoder of such products keeps
        for tokens, past in ((prompts[:, :first], 0), (prompts[:, first:], first)):
            assert bits_equal(m.logits(tokens, all=True), apart(tokens, past))
    finally:
        capi.check(lib.mi355x_tune(b"attention.prompt", 1))
