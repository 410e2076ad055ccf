"""The Q4_0 product of many rows of float32 x on the binary16 matrix cores, x as pairs of binary16 (qgemm_q4_0_fx16.hip,
qgemm_q4_0_direct.hip, qgemm_q4_0_parts.hip), against the product in 64 bits. Bound: a pair holds an element to 2^-23 of its block's largest magnitude (kernel's comment), beside
float32 sums' 2e-6 sum |x||w|; what the fixed-point forms of this product are held to."""
import ctypes

import numpy as np
import pytest
import torch

import oracle as O
from mimir_amd import capi
from mimir_amd.llama import Llama
from oracle import llama as OL
from tests import gpu
from tests.helpers import bench_blocks, random_blocks
from tests.test_gpu_llama import _oracle_config, _upload_synthetic

pytestmark = pytest.mark.gpu


def last_kernel():
    buf = ctypes.create_string_buffer(200)
    capi.check(gpu.lib().mi355x_last_kernel(buf, 200))
    return buf.value.decode()


def tuned(rows, pairs):
    capi.check(gpu.lib().mi355x_tune(b"q4_0.fx_rows", rows))
    capi.check(gpu.lib().mi355x_tune(b"q4_0.fx_pairs", pairs))


PANEL, DIRECT, PARTS = "qgemm_q4_0_fx16_kernel: ", "qgemm_q4_0_direct_kernel", "qgemm_q4_0_parts_kernel"
IN_PLACE = (DIRECT, PARTS)  # W read where it lies


@pytest.mark.parametrize("m,n,k,kernel", [
    (1, 5, 128, PANEL + "1 x 1 tiles of 128 x 256"), (40, 100, 256, PANEL + "1 x 1 tiles of 128 x 256"), (129, 257, 384, PANEL + "2 x 2 tiles of 128 x 256"),
    (300, 520, 6272, PANEL + "3 x 3 tiles of 128 x 256, 2 shares of K"), (257, 129, 14336, PANEL + "3 x 1 tiles of 128 x 256, 5 shares of K"),
    (1000, 16500, 128, PANEL + "4 x 64 tiles of 256 x 256, 8 x 1 tiles of 128 x 256"), (2047, 8192, 128, PANEL + "8 x 32 tiles of 256 x 256"),
    (33, 60, 16512, PANEL + "1 x 1 tiles of 128 x 256, 5 shares of K"),
    # W read where it lies: one to four strips of x and two tiles, columns that fill no group, shares that are not of one length
    (16, 5, 64, DIRECT + "<1>: 1 x 1 tiles, 1 shares of K"), (33, 129, 192, DIRECT + "<2>: 1 x 2 tiles, 1 shares of K"),
    (77, 515, 2048, DIRECT + "<3>: 1 x 5 tiles, 8 shares of K"), (96, 97, 1984, DIRECT + "<3>: 1 x 1 tiles, 8 shares of K"),
    (100, 200, 2048, DIRECT + "<4>: 1 x 2 tiles, 8 shares of K"), (128, 515, 1984, DIRECT + "<4>: 1 x 5 tiles, 8 shares of K"),
    (130, 200, 320, DIRECT + "<4>: 2 x 2 tiles, 1 shares of K"),
    # and by a wavefront a part of K
    (77, 515, 5120, PARTS + "<5>: 1 x 9 tiles of 80 x 64, 10 shares of K"), (128, 4096, 4160, PARTS + "<4>: 2 x 64 tiles of 64 x 64, 2 shares of K"),
    (256, 70, 16448, PARTS + "<4>: 4 x 2 tiles of 64 x 64, 17 shares of K")])
@pytest.mark.parametrize("rows", ["even", "wide", "special"])
def test_pairs_of_halves(m, n, k, kernel, rows):
    """Every cut of the product, tiles and strips that rows and columns do not fill. Rows of x: of very different magnitude; some whose
    blocks differ by up to 2^60 (those take an exponent a block, and a tile with one of them its slower loop); blocks and
    rows of zeros, the smallest and largest magnitudes, a NaN and an infinity (a row of NaNs each, and of no other)."""
    rng = np.random.default_rng(m + n + k)
    raw = random_blocks(rng, O.Q4_0, n * k)
    x = (rng.normal(size=(m, k)) * np.exp(rng.normal(size=(m, 1)) * 3)).astype(np.float32)
    bad = []
    if rows == "wide":
        x[m // 3, :32] *= 2.0 ** 30
        x[m - 1, 32:64] *= 2.0 ** -40
        x[m - 1, 5] *= 2.0 ** 20
    if rows == "special" and m >= 12:
        x[m // 2, :32] = 0
        x[1] = 0
        x[2, 3], x[5, k - 1] = np.nan, np.inf
        x[7] *= np.float32(1e-36)
        x[8] *= np.float32(1e30)
        x[9] = np.float32(1e-42)
        bad = [2, 5]
    wide = torch.zeros((m, k + 8), device="cuda:0")  # rows further apart than K
    wide[:, :k] = gpu.dev(x)
    buf, ptr = gpu.dev_bytes_at(raw, 4)
    gpu.say(f"q4_0 halves M={m} N={n} K={k} {rows}")
    try:
        tuned(1 if kernel.startswith(PANEL) else 0, 3)
        got = gpu.qgemv(O.Q4_0, ptr, wide[:, :k], n, k)
        assert last_kernel() == kernel
    finally:
        tuned(0, 1)
    x64 = gpu.dev(x).double()
    w = gpu.dev(O.dequantize(O.Q4_0, raw).reshape(n, k)).double()
    want, bound = x64 @ w.T, 2e-6 * (x64.abs() @ w.abs().T)
    bound += 2.0 ** -23 * (x64.abs().reshape(m, -1, 32).amax(2) @ w.abs().reshape(n, -1, 32).sum(2).T) + 1e-30
    good = [i for i in range(m) if i not in bad]
    got = gpu.dev(got).double()
    assert torch.isnan(got[bad]).all()
    assert ((got - want).abs() <= bound)[good].all()


@pytest.mark.parametrize("k", [384, 640])
def test_tiles_of_256_by_256_over_groups_of_scales(k):
    """Twelve and twenty blocks: a stage's refill from the fourth on, the scales' second and third group of eight, fragments read past the last block's stage."""
    test_pairs_of_halves(1000, 16500, k, PANEL + "4 x 64 tiles of 256 x 256, 8 x 1 tiles of 128 x 256", "even")


@pytest.mark.parametrize("m,kernel", [(20, DIRECT + "<1>"), (64, PARTS + "<4>"), (77, PARTS + "<5>"), (128, PARTS + "<4>"), (200, DIRECT + "<4>")])
def test_rows_held_by_block_among_others(m, kernel):
    """One row with a block 2^17 above its others, which is held with an exponent a block, beside ordinary rows, a row of zeros and one with
    a NaN, by W read where it lies: results as above, and no more than half as long again as without it (such a row is rare, but takes the
    tile's other rows with it; twice as long and more where a tile then went through W once for each 32 rows of x)."""
    n, k, l = 14336, 4096, gpu.lib()
    rng = np.random.default_rng(m)
    raw = bench_blocks(rng, O.Q4_0, n * k)
    x = rng.normal(size=(m, k)).astype(np.float32)
    wide = x.copy()
    wide[m // 2, 96:128] *= 2.0 ** 17
    odd = wide.copy()
    odd[1], odd[m - 1, 40] = 0, np.nan
    w, xs = gpu.dev(raw), [gpu.dev(v) for v in (x, wide, odd)]
    y = torch.empty((m, n), device="cuda:0")

    def call(i, times=1):
        for _ in range(times):
            capi.check(l.mi355x_qgemv(capi.Q4_0, w.data_ptr(), xs[i].data_ptr(), y.data_ptr(), m, n, k, k, gpu.stream()))
    gpu.say(f"q4_0 halves, a row held by block, M={m}")
    took = [[], []]
    try:
        tuned(0, 3)
        call(2)
        assert last_kernel().startswith(kernel)
        w64, x64, got = gpu.dev(O.dequantize(O.Q4_0, raw).reshape(n, k)).double(), xs[2].double(), y.double()
        for _ in range(5):
            for i in (0, 1):
                start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                call(i, 3)
                start.record()
                call(i, 20)
                stop.record()
                stop.synchronize()
                took[i].append(start.elapsed_time(stop))
    finally:
        tuned(0, 1)
    bound = 2e-6 * (x64.abs() @ w64.abs().T) + 2.0 ** -23 * (x64.abs().reshape(m, -1, 32).amax(2) @ w64.abs().reshape(n, -1, 32).sum(2).T) + 1e-30
    assert torch.isnan(got[m - 1]).all() and ((got - x64 @ w64.T).abs() <= bound)[:m - 1].all()
    assert min(took[1]) <= 1.5 * min(took[0]), (min(took[1]), min(took[0]))


@pytest.mark.parametrize("m", [25, 32, 33, 48, 49, 80, 81, 112, 128, 129, 160, 161, 256])
@pytest.mark.parametrize("n,k", [(97, 2112), (513, 4224), (64, 9280)])
@pytest.mark.parametrize("rows", ["even", "wide"])
def test_a_wavefront_a_part_of_k(m, n, k, rows):
    """Rows of W of more than 2048: every number of sixteens of rows, a sixteen and a tile begun and filled, columns that fill no strip; 66, 132 and
    290 blocks, which leave some parts less than a chunk of eight blocks or none at all (161 x 97 x 2112: a last share of two blocks for eight of
    them), and a last chunk that reaches back. Bound as in test_pairs_of_halves."""
    rng = np.random.default_rng(m + n + k)
    raw = random_blocks(rng, O.Q4_0, n * k)
    x = (rng.normal(size=(m, k)) * np.exp(rng.normal(size=(m, 1)) * 3)).astype(np.float32)
    if rows == "wide":
        x[m // 3, :32] *= 2.0 ** 30
        x[m - 1, k - 32:] *= 2.0 ** -40
    buf, ptr = gpu.dev_bytes_at(raw, 4)
    gpu.say(f"q4_0 parts M={m} N={n} K={k} {rows}")
    try:
        tuned(0, 3)
        got = gpu.dev(gpu.qgemv(O.Q4_0, ptr, gpu.dev(x), n, k)).double()
        assert last_kernel().startswith(PARTS)
    finally:
        tuned(0, 1)
    x64, w = gpu.dev(x).double(), gpu.dev(O.dequantize(O.Q4_0, raw).reshape(n, k)).double()
    bound = 2e-6 * (x64.abs() @ w.abs().T) + 2.0 ** -23 * (x64.abs().reshape(m, -1, 32).amax(2) @ w.abs().reshape(n, -1, 32).sum(2).T) + 1e-30
    assert ((got - x64 @ w.T).abs() <= bound).all()


def prompt_model(batch, prompt, embed, hidden, heads, kv_heads, head_dim, layers):
    c = capi.LlamaConfig()
    c.embed, c.hidden, c.layers, c.heads, c.kv_heads, c.head_dim, c.rope_dim, c.vocab = embed, hidden, layers, heads, kv_heads, head_dim, head_dim, 515
    c.context, c.interleaved, c.cache_dtype, c.batch = prompt + 8, 1, capi.F32, batch
    c.rope_base, c.rope_scale, c.eps = 10000.0, 1.0, 1e-5
    return c


@pytest.mark.parametrize("batch,prompt,embed,hidden,heads,kv_heads,head_dim", [
    (1, 150, 320, 1088, 5, 1, 64), (2, 24, 320, 1024, 5, 1, 64), (3, 100, 320, 992, 5, 1, 64),  # a down projection whose K (992) this form does not take
    (1, 45, 320, 1088, 4, 1, 80),      # k and v of 80 rows: their last strips are half of the next one's place
    (1, 37, 1024, 4096, 8, 2, 128),    # shares of K, W read where it lies
    (2, 150, 1024, 4096, 8, 2, 128)])  # and by the panel
def test_a_prompt_pass_with_products_taken_together(batch, prompt, embed, hidden, heads, kv_heads, head_dim):
    """A model whose q, k, v and whose gate and up (with SwiGLU) are one product each: column strips that no tile is filled by, K of 320 and of 1088, shares of K.
    Nothing on the way rounds to int8 or binary16, so that the passes as pairs and in fixed point, and the oracle's, differ by float32 rounding and by what
    x is held to (2^-23 of a block's largest) alone: some 1e-6 of the largest logit after two layers; every logit of every sequence within 1e-5."""
    c = prompt_model(batch, prompt, embed, hidden, heads, kv_heads, head_dim, 2)
    om = OL.synthetic(_oracle_config(c), seed=3, output_dt=O.Q4_0, centered=True)
    m = Llama(c)
    _upload_synthetic(m, om)
    m.finalize(prompt)
    tokens = np.random.default_rng(1).integers(0, c.vocab, (batch, prompt))
    out = {}
    try:
        for pairs in (3, 0):
            gpu.say(f"prompt pass batch={batch} prompt={prompt} embed={embed} hidden={hidden} pairs={pairs}")
            tuned(0, pairs)
            m.reset()
            out[pairs] = m.logits(tokens, all=True)
    finally:
        tuned(0, 1)
    assert not np.array_equal(out[3], out[0])
    scale = np.abs(out[0]).max()
    assert np.abs(out[3] - out[0]).max() <= 1e-5 * scale, np.abs(out[3] - out[0]).max() / scale
    for b in range(batch):
        want = om.logits(tokens[b].tolist(), om.new_caches(c.context, O.F32), all=True)
        assert np.abs(out[3][b] - want).max() <= 1e-5 * scale, np.abs(out[3][b] - want).max() / scale


@pytest.mark.parametrize("rows,embed,hidden,kernel", [
    (37, 1024, 4096, DIRECT + "<2>: 1 x 64 tiles, 4 shares of K"), (77, 2048, 8192, DIRECT + "<3>: 1 x 128 tiles, 2 shares of K"),
    (100, 320, 992, DIRECT + "<4>: 1 x 16 tiles, 1 shares of K"), (300, 1024, 4096, PANEL + "3 x 32 tiles of 128 x 256, 2 shares of K"),
    (300, 320, 992, PANEL + "3 x 8 tiles of 128 x 256")])
def test_gate_and_up_are_one_product(rows, embed, hidden, kernel):
    """Where the down projection and the output are of Q8_0, whose kernels leave no name, the name of the pass is gate's and up's: one product of both
    matrices' strips (twice `hidden`), cut as asked. SwiGLU in the tile where K is whole, with the shares' sums where it is not; results against the oracle, whose
    int8 roundings may fall on the other side here and there (test_gpu_llama.py)."""
    c = prompt_model(1, rows, embed, hidden, 5 if embed == 320 else embed // 128, 1, 64 if embed == 320 else 128, 1)
    om = OL.synthetic(_oracle_config(c), seed=6, centered=True)
    om.blocks[0].down = OL._q_blocks(np.random.default_rng(8), O.Q8_0, embed, hidden)
    m = Llama(c)
    _upload_synthetic(m, om)
    m.finalize(rows)
    tokens = np.random.default_rng(1).integers(0, c.vocab, (1, rows))
    try:
        gpu.say(f"gate and up rows={rows} embed={embed} hidden={hidden}")
        tuned(0, 3)
        got = m.logits(tokens, all=True)[0]
        ran = last_kernel()
    finally:
        tuned(0, 1)
    assert ran == kernel
    want = om.logits(tokens[0].tolist(), om.new_caches(c.context, O.F32), all=True)
    scale = np.abs(want).max()
    assert np.abs(got - want).max() <= 0.02 * scale and np.median(np.abs(got - want)) <= 1e-5 * scale


@pytest.mark.parametrize("rows,hidden,shares", [(40, 96, 5), (130, 2080, 1)])
def test_gate_and_up_by_parts_of_k(rows, hidden, shares):
    """The same by rows of W of 2112, SwiGLU in the tile and with the shares' sums; hidden that fills no group of strips."""
    c = prompt_model(1, rows, 2112, hidden, 33, 1, 64, 1)
    om = OL.synthetic(_oracle_config(c), seed=6, centered=True)
    om.blocks[0].down = OL._q_blocks(np.random.default_rng(8), O.Q8_0, 2112, hidden)
    m = Llama(c)
    _upload_synthetic(m, om)
    m.finalize(rows)
    tokens = np.random.default_rng(1).integers(0, c.vocab, (1, rows))
    try:
        gpu.say(f"gate and up by parts, rows={rows} hidden={hidden}")
        tuned(0, 3)
        got = m.logits(tokens, all=True)[0]
        ran = last_kernel()
    finally:
        tuned(0, 1)
    assert ran.startswith(PARTS) and ran.endswith(f", {shares} shares of K")
    want = om.logits(tokens[0].tolist(), om.new_caches(c.context, O.F32), all=True)
    scale = np.abs(want).max()
    assert np.abs(got - want).max() <= 0.02 * scale and np.median(np.abs(got - want)) <= 1e-5 * scale


@pytest.mark.parametrize("m,n,k,in_place", [(24, 8192, 14336, False), (20, 14336, 11008, False), (17, 8192, 11008, False), (24, 14336, 8192, False),
                                            (32, 14336, 4096, True), (77, 5120, 5120, True), (24, 14336, 14336, True)])
def test_the_row_kernel_keeps_up_to_24_rows_that_it_multiplies_faster(m, n, k, in_place):
    raw = bench_blocks(np.random.default_rng(m), O.Q4_0, 16 * k)
    w = gpu.dev(raw).repeat(n // 16)
    x = torch.ones((m, k), device="cuda:0")
    gpu.say(f"q4_0 choice M={m} N={n} K={k}")
    gpu.qgemv(O.Q4_0, w.data_ptr(), x[:1], n, k)  # another kernel's name
    before = last_kernel()
    gpu.qgemv(O.Q4_0, w.data_ptr(), x, n, k)
    assert before and last_kernel().startswith(IN_PLACE) == in_place


def test_digits_on_request_in_a_prompt_pass():
    """"q4_0.fx_pairs" = 2 sends the decoder's products of many rows to the binary16 matrix cores as digits too: the int8 form's bits."""
    c = capi.LlamaConfig()
    c.embed, c.hidden, c.layers, c.heads, c.kv_heads, c.head_dim, c.rope_dim, c.vocab = 384, 1024, 2, 6, 2, 64, 64, 2048
    c.context, c.interleaved, c.cache_dtype, c.batch = 520, 1, capi.F32, 1
    c.rope_base, c.rope_scale, c.eps = 10000.0, 1.0, 1e-5
    m = Llama(c)
    _upload_synthetic(m, OL.synthetic(_oracle_config(c), seed=4, output_dt=O.Q4_0))
    m.finalize(512)
    tokens = np.random.default_rng(2).integers(0, c.vocab, (1, 512))
    out, ran = {}, {}
    try:
        for pairs in (2, 0):
            gpu.say(f"prompt pass, digits, pairs={pairs}")
            tuned(0, pairs)
            m.reset()
            out[pairs] = m.logits(tokens, all=True)
            ran[pairs] = last_kernel()  # the output matrix's product
    finally:
        tuned(0, 1)
    assert ran[2].startswith(PANEL) and ran[0] == "qgemm_q4_0_fx_kernel"
    assert np.array_equal(out[2].view(np.uint32), out[0].view(np.uint32))


@pytest.mark.parametrize("prompt", [100, 40])
def test_a_model_of_few_rows_holds_no_panel(prompt):
    """Prompts of up to 256 rows are multiplied with W read where it lies: finalize allocates a workspace for shares' sums alone, not the 67 MB that gate's
    and up's integers would be and 96 MiB of sums. 100 rows hold 10 + 6 MB of float32 and 12 MB of converted rows, sums of one round of
    workgroups are 17 MB, and some twenty allocations may each end up to 2 MB further on: 64 MiB for 100 rows, 48 for 40."""
    most_mib = 64 if prompt == 100 else 48
    c = capi.LlamaConfig()
    c.embed, c.hidden, c.layers, c.heads, c.kv_heads, c.head_dim, c.rope_dim, c.vocab = 2048, 8192, 1, 16, 4, 128, 128, 256
    c.context, c.interleaved, c.cache_dtype, c.batch = prompt + 8, 1, capi.F16, 1
    c.rope_base, c.rope_scale, c.eps = 10000.0, 1.0, 1e-5
    m = Llama(c)
    _upload_synthetic(m, OL.synthetic(_oracle_config(c), seed=5, output_dt=O.Q4_0))
    held = []
    for rows in (8, prompt):
        gpu.say(f"finalize for {rows} rows")
        m.finalize(rows)
        gpu.sync()
        held.append(torch.cuda.mem_get_info()[0])
    assert held[0] - held[1] <= most_mib << 20, (held[0] - held[1]) / 2.0 ** 20
    tokens = np.random.default_rng(2).integers(0, c.vocab, (1, prompt))
    out = {}
    try:
        for pairs in (1, 0):
            tuned(0, pairs)
            m.reset()
            out[pairs] = m.logits(tokens, all=True)
            if pairs:
                m.reset()
                m.generate(tokens, 1)
    finally:
        tuned(0, 1)
    scale = np.abs(out[0]).max()
    assert np.median(np.abs(out[1] - out[0])) <= 1e-5 * scale and not np.array_equal(out[1], out[0])
