"""Workloads of this framework as its users meet them, through its public entry points: block-quantized
products (mi355x_qgemv, mi355x_qgemm_bf16), greedy generation by a Llama-shaped decoder (prompt pass and
decoding steps), and generation by the two mixer-stack designs. Weights are random, of the
configurations' shapes; a model has fewer layers than a real one, since its layers are alike."""
import numpy as np
import torch

from mimir_amd import capi, stack
from mimir_amd.llama import Llama

DEV = "cuda:0"
DTYPE = {"q8_0": capi.Q8_0, "q4_0": capi.Q4_0, "q4_K": capi.Q4_K, "q6_K": capi.Q6_K}
#: dtype -> (weights of a block, bytes of a block)
BLOCK = {"q8_0": (32, 34), "q4_0": (32, 18), "q4_K": (256, 144), "q6_K": (256, 210)}


def listed():
    product = dict(kind="product")
    llama = dict(kind="llama", embed=4096, hidden=14336, vocab=32768, layers=4)
    return [
        # products of one row of x by several matrices in turn, as a program's decoding loop makes them: out of memory, not cache
        dict(product, name="q8_0 1x4096x4096", dtype="q8_0", x="f32", m=1, n=4096, k=4096, mats=8),
        dict(product, name="q4_0 1x14336x4096", dtype="q4_0", x="f32", m=1, n=14336, k=4096, mats=8),
        # eight sequences' rows by the long-rowed matrix of a feed-forward
        dict(product, name="q6_K 8x4096x14336", dtype="q6_K", x="f32", m=8, n=4096, k=14336, mats=4),
        # a short prompt's rows, a number of rows that fills no tile
        dict(product, name="q4_0 77x5120x5120", dtype="q4_0", x="f32", m=77, n=5120, k=5120, mats=4),
        # half-precision activations by a prompt's rows
        dict(product, name="q4_0 bf16 512x14336x4096", dtype="q4_0", x="bf16", m=512, n=14336, k=4096, mats=2),
        # one user's chat turn: a prompt, then an answer
        dict(llama, name="llama q4_0 1x512+64", dtype="q4_0", batch=1, prompt=512, new=64),
        # a short question to a K-quant model
        dict(llama, name="llama q4_K 1x37+64", dtype="q4_K", batch=1, prompt=37, new=64),
        # a long document, then a short answer against its cache
        dict(llama, name="llama q4_0 1x2048+32", dtype="q4_0", batch=1, prompt=2048, new=32),
        # a server's batch
        dict(llama, name="llama q4_0 8x512+32", dtype="q4_0", batch=8, prompt=512, new=32),
        # a batch of an odd number of short prompts by a K-quant model
        dict(llama, name="llama q4_K 5x131+32", dtype="q4_K", batch=5, prompt=131, new=32),
        # the mixer-stack designs: a long prompt and a short answer, and a few sequences in lockstep
        dict(kind="genetar", name="genetar 1x2048+32", width=4096, ff=14336, vocab=32768, layers=2, batch=1, prompt=2048, new=32),
        dict(kind="fuvolix", name="fuvolix 4x301+32", width=2048, ff=8192, vocab=32768, layers=3, batch=4, prompt=301, new=32),
    ]


def _log(rng, low, high):
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    kind = rng.choice(["product", "product", "product", "llama", "llama", "genetar", "fuvolix"])
    if kind == "product":
        dtype = rng.choice(sorted(BLOCK))
        x = rng.choice(["f32", "f32", "bf16"])
        m = _log(rng, 1, 512) if x == "f32" else _log(rng, 16, 1024)
        n = _log(rng, 512, 14336)
        k = _log(rng, 1024, 14336)
        step = 32 if dtype in ("q4_0", "q8_0") and rng.random() < 0.3 else 256
        k = max(step, k // step * step)
        if rng.random() < 0.6:
            n = max(64, n // 64 * 64)
        if x == "bf16" and dtype == "q8_0":
            m = min(m, 64)
        return dict(kind=kind, dtype=dtype, x=x, m=m, n=n, k=k, mats=rng.choice([2, 4, 8]))
    if kind == "llama":
        embed = rng.choice([1024, 2048, 4096])
        batch = rng.choice([1, 1, 2, 4, 8, 11, 16])
        prompt = min(_log(rng, 16, 2048), 4096 // batch)
        return dict(kind=kind, embed=embed, hidden={1024: 4096, 2048: 8192, 4096: 14336}[embed], vocab=32768, layers=rng.choice([2, 3, 4]),
                    dtype=rng.choice(["q4_0", "q4_0", "q4_K", "q6_K"]), batch=batch, prompt=prompt, new=_log(rng, 4, 32))
    width = rng.choice([1024, 2048, 4096])
    batch = rng.choice([1, 1, 2, 4, 8])
    return dict(kind=kind, width=width, ff={1024: 4096, 2048: 8192, 4096: 14336}[width], vocab=32768, layers=rng.choice([1, 2, 3]), batch=batch,
                prompt=min(_log(rng, 16, 2048), 2048 // batch), new=_log(rng, 4, 32))


# ---- inputs ------------------------------------------------------------------------------------


def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 1000003 + 17)
    return g


def _half_scales(g, nb, scale):
    return (torch.randn(nb, generator=g, device=DEV) * scale).abs().to(torch.float16).view(torch.uint8).reshape(nb, 2)


def _blocks(g, dtype, n, k, scale=None):
    """[n, bytes of a row]: quants uniform over their range and binary16 scales |N(0, scale)|; `scale` None: such that a
    product keeps its input's size."""
    size, nbytes = BLOCK[dtype]
    nb = n * k // size
    if scale is None:
        scale = k ** -0.5 / {"q4_0": 4.6, "q8_0": 73.0, "q4_K": 250.0, "q6_K": 1366.0}[dtype]
    raw = torch.randint(0, 256, (nb, nbytes), dtype=torch.uint8, generator=g, device=DEV)
    if dtype == "q6_K":
        raw[:, 208:210] = _half_scales(g, nb, scale)
    else:
        raw[:, 0:2] = _half_scales(g, nb, scale)
    if dtype == "q4_K":
        raw[:, 2:4] = (raw[:, 0:2].contiguous().view(torch.float16).float() * 7.5).to(torch.float16).view(torch.uint8).reshape(nb, 2)
    if dtype == "q8_0":
        raw[:, 2:][raw[:, 2:] == 128] = 0  # -128 is no value of the format
    return raw.reshape(n, -1)


def _product_inputs(case, seed):
    g = _generator(seed)
    ws = [_blocks(g, case["dtype"], case["n"], case["k"], 0.02) for _ in range(case["mats"])]
    x = torch.randn(case["m"], case["k"], generator=g, device=DEV)
    return ws, x.to(torch.bfloat16) if case["x"] == "bf16" else x


def _llama_tensors(case, seed):
    """name -> (dtype, blocks or float32 values on the device, rows, columns)."""
    g = _generator(seed)
    e, h = case["embed"], case["hidden"]
    kv = e // 4
    out = {"token_embd.weight": ("q8_0", _blocks(g, "q8_0", case["vocab"], e, 1 / 73), case["vocab"], e),
           "output_norm.weight": ("f32", 1 + 0.02 * torch.randn(e, generator=g, device=DEV), 1, e)}
    for i in range(case["layers"]):
        for leaf in ("attn_norm", "ffn_norm"):
            out[f"blk.{i}.{leaf}.weight"] = ("f32", 1 + 0.02 * torch.randn(e, generator=g, device=DEV), 1, e)
        for leaf, n, k in (("attn_q", e, e), ("attn_k", kv, e), ("attn_v", kv, e), ("attn_output", e, e), ("ffn_gate", h, e), ("ffn_up", h, e), ("ffn_down", e, h)):
            out[f"blk.{i}.{leaf}.weight"] = (case["dtype"], _blocks(g, case["dtype"], n, k), n, k)
    return out


def _tokens(case, seed):
    return np.random.default_rng(seed).integers(0, case["vocab"], (case["batch"], case["prompt"])).astype(np.int32)


def _stack_config(case):
    width, ff, heads = case["width"], case["ff"], case["width"] // 128
    mixers = [("attention", dict(heads=heads, kv_heads=max(1, heads // 4), dim=128, vdim=128, scale=128 ** -0.5, softcap=30.0, v_mix=True)),
              ("attention_2", dict(heads=heads, kv_heads=max(1, heads // 4), dim=128, vdim=128, scale=128 ** -0.5, softcap=30.0, v_mix=True,
                                   rot=dict(base=500000.0, dims=128, scaling=dict(factor=8.0, low=1.0, high=4.0, original=8192))))]
    if case["kind"] == "fuvolix":
        mixers = [("latent_attention", dict(heads=heads, dim=128, rot_dim=64, vdim=128, kv_rank=512, scale=192 ** -0.5, rot=dict(base=10000.0, dims=64))),
                  ("mlstm", dict(heads=heads, dim=128, vdim=128, gate_cap=15.0)),
                  ("lightning", dict(heads=heads, dim=128, vdim=128, decay=[float(np.exp(-2.0 ** (-8 * (h + 1) / heads))) for h in range(heads)]))]
    layers = [dict(type=mixers[i % len(mixers)][0], mixer=mixers[i % len(mixers)][1], mlp=dict(kind="dense", ff=ff)) for i in range(case["layers"])]
    return dict(width=width, vocab=case["vocab"], canon=dict(taps=4), norm=dict(groups=2, eps=1e-6), layers=layers,
                embedding=dict(bigram=dict(buckets=case["vocab"], mul_prev=31, mul_cur=7)), logit_scale=1.0)


def _stack_model(case):
    context = case["prompt"] + case["new"]
    design = {"genetar": "Genetar", "fuvolix": "Fuvolix"}[case["kind"]]
    return stack.Stack(*stack.CONFIGS[design](_stack_config(case), context, case["batch"]))


def _stack_tensors(case, names, seed):
    """name -> bfloat16 tensor [n, k]. The output matrix is the embedding's, scaled, as where the two are tied."""
    g = _generator(seed)
    out = {}
    for name, n, k in names:
        leaf = name.rsplit(".", 1)[-1]
        scale, at = (k ** -0.5 if n > 1 else 0.5), 0.0
        if leaf in ("embed", "bigram"):
            scale = 1.0 if leaf == "embed" else 0.3
        elif leaf == "dwa":
            scale, at = 0.02, 1.0 / k
        elif leaf in ("norm1b", "norm2b"):
            scale, at = 0.02, 0.3
        elif "norm" in leaf or leaf in ("ls1", "ls2"):
            scale, at = 0.02, 1.0
        if leaf == "head":
            out[name] = (out["embed"].float() * k ** -0.5).to(torch.bfloat16)
        else:
            out[name] = (torch.randn(n, k, generator=g, device=DEV) * scale + at).to(torch.bfloat16)
    return out


def prepare(case, seed):
    if case["kind"] == "product":
        lib = capi.load()
        capi.check(lib.mi355x_init(0))
        ws, x = _product_inputs(case, seed)
        y = [torch.empty(case["m"], case["n"], dtype=x.dtype, device=DEV) for _ in ws]
        return dict(case=case, lib=lib, ws=ws, x=x, y=y)
    context = case["prompt"] + case["new"]
    if case["kind"] == "llama":
        c = capi.LlamaConfig()
        c.embed, c.hidden, c.layers, c.vocab, c.batch, c.context = case["embed"], case["hidden"], case["layers"], case["vocab"], case["batch"], context
        c.head_dim = c.rope_dim = 128
        c.heads, c.kv_heads = case["embed"] // 128, case["embed"] // 512
        c.interleaved, c.cache_dtype, c.rope_base, c.rope_scale, c.eps = 1, capi.F16, 500000.0, 1.0, 1e-5
        m = Llama(c)
        for name, (dtype, data, n, k) in _llama_tensors(case, seed).items():
            m.set_tensor(name, capi.F32 if dtype == "f32" else DTYPE[dtype], data.cpu().numpy(), n * k)
    else:
        m = _stack_model(case)
        for name, data in _stack_tensors(case, m.tensors(), seed).items():
            m.set_tensor(name, capi.BF16, data.view(torch.int16).cpu().numpy().view(np.uint16), data.numel())
    m.finalize(case["prompt"])
    return dict(case=case, model=m, tokens=_tokens(case, seed))


def run(state):
    case = state["case"]
    if case["kind"] == "product":
        lib, x, dt, stream = state["lib"], state["x"], DTYPE[case["dtype"]], torch.cuda.current_stream().cuda_stream
        for w, y in zip(state["ws"], state["y"]):
            if case["x"] == "bf16":
                capi.check(lib.mi355x_qgemm_bf16(dt, w.data_ptr(), x.data_ptr(), y.data_ptr(), case["m"], case["n"], case["k"], case["k"], capi.BF16, stream))
            else:
                capi.check(lib.mi355x_qgemv(dt, w.data_ptr(), x.data_ptr(), y.data_ptr(), case["m"], case["n"], case["k"], case["k"], stream))
        return state["y"]
    m = state["model"]
    m.reset()
    tokens, _ = m.generate(state["tokens"], case["new"])
    return dict(tokens=tokens, logits=m.logits(tokens[:, -1:]))  # the distribution that the next token would come from


def _layer_sizes(case):
    """(weights of a layer, cached values a position and layer) of a model."""
    if case["kind"] == "llama":
        return case["embed"] * (case["embed"] * 5 // 2 + 3 * case["hidden"]), case["embed"] // 2
    w = case["width"]
    if case["kind"] == "genetar":
        return w * (w * 5 // 2 + 3 * case["ff"]), w // 2
    return w * 5 * w + 2 * w * case["ff"], 0


def work(case):
    if case["kind"] == "product":
        size, nbytes = BLOCK[case["dtype"]]
        weights = case["n"] * case["k"]
        one = 2 if case["x"] == "bf16" else 4
        return {"bytes": case["mats"] * (weights * nbytes // size + one * case["m"] * case["n"]) + one * case["m"] * case["k"], "flops": 2 * case["mats"] * case["m"] * weights}
    weights, cached = _layer_sizes(case)
    size, nbytes = BLOCK[case["dtype"]] if case["kind"] == "llama" else (1, 2)
    width = case.get("embed") or case["width"]
    head = case["vocab"] * width
    b, s, new, layers = case["batch"], case["prompt"], case["new"], case["layers"]
    passes = 1 + new  # the prompt's, the new tokens' but the last one's, and the logits'
    positions = sum(s + i for i in range(new + 1))  # read from the cache by all passes
    read = passes * (layers * weights * nbytes // size + head * (17 if case["kind"] == "llama" else 32) // 16) + b * layers * 2 * cached * positions
    attend = 4 * width * layers * b * (s * (s + 1) // 2 + positions - s) if cached else 0
    return {"bytes": read, "flops": 2 * b * (layers * weights * (s + new) + head * passes) + attend}


def tolerance(case):
    """About four times the error against 64 bits that was measured, over all sizes: for float32 products the sums' order; for
    K-quants and the Q8_0 output matrix the steps of x's rounding to int8, which a difference of 1e-7 before them can move."""
    if case["kind"] == "product":
        return {"rel": 7e-3} if case["x"] == "bf16" else {"rel": 1e-6}
    if case["kind"] == "genetar":
        return {"rel": 2e-3, "max": 0.01}
    if case["kind"] == "fuvolix":
        return {"rel": 6e-3, "max": 0.04}
    return {"rel": 3e-4, "max": 4e-3} if case["dtype"] == "q4_0" else {"rel": 3e-2, "max": 0.4}


# ---- the same in 64 bits -----------------------------------------------------------------------


def _dequantize(raw, dtype):
    """Blocks [n, bytes] -> weights [n, k] float64."""
    n = raw.shape[0]
    b = raw.reshape(-1, BLOCK[dtype][1])

    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).double()
    if dtype == "q8_0":
        v = b[:, 2:].contiguous().view(torch.int8).double() * half(0)
    elif dtype == "q4_0":
        v = (torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8) * half(0)
    elif dtype == "q4_K":
        s = b[:, 4:16].int()
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6 << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6 << 4)], 1).double()
        q = b[:, 16:].reshape(-1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
        v = q * (sc * half(0))[:, :, None] - (mn * half(2))[:, :, None]
    else:
        low, high = b[:, :128].reshape(-1, 2, 2, 32).int(), b[:, 128:192].reshape(-1, 2, 1, 32).int()
        q = torch.stack([low[:, :, k % 2] >> (4 * (k // 2)) & 15 | (high[:, :, 0] >> (2 * k) & 3) << 4 for k in range(4)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double() * half(208)
        v = (q.reshape(-1, 16, 16).double() - 32) * sc[:, :, None]
    return v.reshape(n, -1)


def _round_activations(x, dtype):
    """What the integer dot products of a dtype read: x as int8 and a scale per block (Q4_0: x itself)."""
    if dtype == "q4_0":
        return x
    b = x.reshape(-1, BLOCK[dtype][0]).float()
    amax = b.abs().amax(1, keepdim=True)
    q = torch.round(b * torch.where(amax > 0, 127 / amax, amax)).clamp(-127, 127)
    return (q.double() * (amax / 127).double()).reshape(x.shape)


def _times(x, w, dtype):
    return _round_activations(x, dtype) @ w.T


def _rms(x, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _attend(q, k, v, scale, past, cap=0.0):
    """q [H, s, d] against k, v [G, past + s, d], causal."""
    group = q.shape[0] // k.shape[0]
    hidden = torch.ones(q.shape[1], k.shape[1], dtype=torch.bool, device=DEV).triu(past + 1)
    out = []
    for a in range(q.shape[0]):
        s = q[a] @ k[a // group].T.contiguous() * scale
        s = cap * torch.tanh(s / cap) if cap else s
        out.append(torch.softmax(s.masked_fill(hidden, -torch.inf), 1) @ v[a // group])
    return torch.stack(out)


def _exact_llama(case, seed):
    t = {name: v.double() if d == "f32" else (_dequantize(v, d), v) for name, (d, v, _, _) in _llama_tensors(case, seed).items()}
    heads, kv_heads, dt = case["embed"] // 128, case["embed"] // 512, case["dtype"]
    freq = 500000.0 ** (-2 * torch.arange(64, dtype=torch.float64, device=DEV) / 128)
    b = case["batch"]
    caches = [[[None, None] for _ in range(b)] for _ in range(case["layers"])]

    def rotate(x, past):  # [s, heads, 128], neighbouring features are pairs
        ang = (past + torch.arange(x.shape[0], dtype=torch.float64, device=DEV))[:, None, None] * freq
        u, v = x[..., 0::2], x[..., 1::2]
        return torch.stack([u * ang.cos() - v * ang.sin(), v * ang.cos() + u * ang.sin()], -1).reshape(x.shape)

    def forward(tokens, past):  # [b, s] -> logits of the last position
        s = tokens.shape[1]
        x = t["token_embd.weight"][0][tokens].reshape(b * s, -1)
        for i in range(case["layers"]):
            p = f"blk.{i}."
            h = _rms(x, 1e-5) * t[p + "attn_norm.weight"]
            q, k, v = (_times(h, t[p + f"attn_{c}.weight"][0], dt).reshape(b, s, -1, 128) for c in "qkv")
            rows = []
            for j in range(b):
                cache = caches[i][j]
                for at, new in ((0, rotate(k[j], past)), (1, v[j])):
                    new = new.transpose(0, 1).half().double()  # the cache is binary16
                    cache[at] = new if cache[at] is None else torch.cat([cache[at], new], 1)
                o = _attend(rotate(q[j], past).transpose(0, 1).contiguous(), cache[0], cache[1], 128 ** -0.5, past)
                rows.append(o.transpose(0, 1).reshape(s, heads * 128))
            x = x + _times(torch.cat(rows), t[p + "attn_output.weight"][0], dt)
            h = _rms(x, 1e-5) * t[p + "ffn_norm.weight"]
            gate, up = (_times(h, t[p + f"ffn_{c}.weight"][0], dt) for c in ("gate", "up"))
            x = x + _times(torch.nn.functional.silu(gate) * up, t[p + "ffn_down.weight"][0], dt)
        last = x.reshape(b, s, -1)[:, -1]
        return _times(_rms(last, 1e-5) * t["output_norm.weight"], t["token_embd.weight"][0], "q8_0")

    tokens, chosen = torch.from_numpy(_tokens(case, seed)).long().to(DEV), []
    past = 0
    for _ in range(case["new"] + 1):
        logits = forward(tokens, past)
        past += tokens.shape[1]
        tokens = logits.argmax(1, keepdim=True)
        chosen.append(tokens)
    return dict(tokens=torch.cat(chosen[:-1], 1).int().cpu().numpy(), logits=logits.cpu().numpy())


def _rotate_by(x, angles, halves):
    u, v = (x[..., :x.shape[-1] // 2], x[..., x.shape[-1] // 2:]) if halves else (x[..., 0::2], x[..., 1::2])
    a, b = u * angles.cos() - v * angles.sin(), v * angles.cos() + u * angles.sin()
    return torch.cat([a, b], -1) if halves else torch.stack([a, b], -1).reshape(x.shape)


def _genetar_mixer(h, t, p, layer, first):
    mx, n = layer["mixer"], h.shape[0]
    q, k, v = ((h @ t[p + c].T).reshape(n, -1, 128) for c in "qkv")
    own = v
    if layer["type"] == "attention":
        q, k = _rms(q, 1e-6), _rms(k, 1e-6)
    else:
        rot = mx["rot"]
        f = rot["base"] ** (-2 * torch.arange(64, dtype=torch.float64, device=DEV) / 128)
        length, sc = 2 * np.pi / f, rot["scaling"]
        mix = ((sc["original"] / length - sc["low"]) / (sc["high"] - sc["low"])).clamp(0, 1)
        f = (1 - mix) * f / sc["factor"] + mix * f
        ang = torch.arange(n, dtype=torch.float64, device=DEV)[:, None, None] * f
        q, k = _rotate_by(q, ang, True), _rotate_by(k, ang, True)
    if first is not None:
        v = (1 - t[p + "vmix"].reshape(-1, 1, 1)[:1]) * v + t[p + "vmix"].reshape(-1, 1, 1)[:1] * first
    o = _attend(q.transpose(0, 1).contiguous(), k.transpose(0, 1).contiguous(), v.transpose(0, 1).contiguous(), mx["scale"], 0, mx["softcap"]).transpose(0, 1)
    if layer["type"] == "attention_2":
        o = o * torch.sigmoid(h @ t[p + "g"].T)[:, :, None]
    return o.reshape(n, -1) @ t[p + "o"].T, own if first is None else first


def _genetar_logits(cfg, t, tokens):
    big = cfg["embedding"]["bigram"]
    before = torch.cat([tokens[:1], tokens[:-1]])
    rows = (before * big["mul_prev"] + tokens * big["mul_cur"]) % big["buckets"]
    rows[0] = big["buckets"]
    x, first = t["embed"][tokens] + t["bigram"][rows], None
    for i, layer in enumerate(cfg["layers"]):
        p = f"l{i}."
        h = _rms(x, 1e-6) * t[p + "norm1"]
        o, first = _genetar_mixer(h, t, p + "mix.", layer, first)
        ff = (torch.nn.functional.silu(h @ t[p + "mlp.gate"].T) * (h @ t[p + "mlp.up"].T)) @ t[p + "mlp.down"].T
        x = x + o * t[p + "ls1"] + ff * t[p + "ls2"]
    return (_rms(x[-1:], 1e-6) * t["final.norm"]) @ t["head"].T


def _matrix_memory(h, t, p, layer):
    """mLSTM and lightning attention as the sum over earlier positions that their recurrences are."""
    mx, n, lightning = layer["mixer"], h.shape[0], layer["type"] == "lightning"
    act = torch.nn.functional.silu if lightning else (lambda z: z)
    q, k, v = (act(h @ t[p + c].T).reshape(n, -1, 128).transpose(0, 1).contiguous() for c in "qkv")
    at = torch.arange(n, dtype=torch.float64, device=DEV)
    if lightning:
        decay = torch.tensor(mx["decay"], dtype=torch.float64, device=DEV)
        weight = torch.exp((at[:, None] - at).clamp(min=0) * decay.log()[:, None, None]).tril()
        o = (q @ k.transpose(1, 2).contiguous() * weight) @ v
    else:
        cap = mx["gate_cap"]
        gi = cap * torch.tanh((h @ t[p + "i"].T + t[p + "i.b"]) / cap)
        gf = torch.nn.functional.logsigmoid(cap * torch.tanh((h @ t[p + "f"].T + t[p + "f.b"]) / cap))
        total = gf.cumsum(0)
        a = gi - total
        top = a.cummax(0).values.clamp(min=0)
        weight = torch.exp((a.T[:, None, :] - top.T[:, :, None]).clamp(max=0)).tril()
        s = q @ k.transpose(1, 2).contiguous() * 128 ** -0.5 * weight
        o = s @ v / (torch.maximum(s.sum(2).abs(), torch.exp(-(total + top).T)) + 1e-6)[:, :, None]
    o = o.transpose(0, 1)
    o = _rms(o.reshape(n, -1) if lightning else o, 1e-6).reshape(n, -1) * t[p + "norm"] * torch.sigmoid(h @ t[p + "g"].T)
    return o @ t[p + "o"].T


def _latent_attention(h, t, p, layer):
    mx, n = layer["mixer"], h.shape[0]
    ang = torch.arange(n, dtype=torch.float64, device=DEV)[:, None] * mx["rot"]["base"] ** (-2 * torch.arange(32, dtype=torch.float64, device=DEV) / 64)
    q, low = (h @ t[p + "q"].T).reshape(n, -1, 192), h @ t[p + "dkv"].T
    q = torch.cat([q[..., :128], _rotate_by(q[..., 128:], ang[:, None], False)], -1)
    c = _rms(low[:, :512], 1e-6) * t[p + "dkv.norm"]
    ku, v = (c @ t[p + "uk"].T).reshape(n, -1, 128), (c @ t[p + "uv"].T).reshape(n, -1, 128)
    k = torch.cat([ku, _rotate_by(low[:, 512:], ang, False)[:, None].expand(-1, ku.shape[1], -1)], -1)
    o = _attend(q.transpose(0, 1).contiguous(), k.transpose(0, 1).contiguous(), v.transpose(0, 1).contiguous(), mx["scale"], 0)
    return o.transpose(0, 1).reshape(n, -1) @ t[p + "o"].T


def _fuvolix_logits(cfg, t, tokens):
    def norm(x, name):
        return _rms(x.reshape(*x.shape[:-1], 2, -1), 1e-6).reshape(x.shape) * t[name]
    x = norm(t["embed"][tokens], "embed.norm")
    past = [x]
    for i, layer in enumerate(cfg["layers"]):
        p = f"l{i}."
        h = norm(x, p + "norm1")
        padded = torch.cat([h.new_zeros(3, h.shape[1]), h])
        h = h + sum(padded[j:j + h.shape[0]] * t[p + "canon1"].reshape(-1, 4)[:, j] for j in range(4))
        mix = _latent_attention if layer["type"] == "latent_attention" else _matrix_memory
        x = x + norm(mix(h, t, p + "mix.", layer), p + "norm1b")
        x = x + norm(torch.relu(norm(x, p + "norm2") @ t[p + "mlp.up"].T).square() @ t[p + "mlp.down"].T, p + "norm2b")
        past.append(x)
        x = sum(w * y for w, y in zip(t[p + "dwa"].reshape(-1), past))
    return norm(x[-1:], "final.norm") @ t["embed"].T


def _exact_stack(case, seed):
    m = _stack_model(case)
    t = {name: v.double() if v.shape[0] > 1 else v[0].double() for name, v in _stack_tensors(case, m.tensors(), seed).items()}
    m.close()
    cfg, logits_of = _stack_config(case), _genetar_logits if case["kind"] == "genetar" else _fuvolix_logits
    chosen, logits = [], []
    for row in torch.from_numpy(_tokens(case, seed)).long().to(DEV):
        for _ in range(case["new"] + 1):
            out = logits_of(cfg, t, row)
            row = torch.cat([row, out.argmax(1)])
        chosen.append(row[case["prompt"]:-1])
        logits.append(out[0])
    return dict(tokens=torch.stack(chosen).int().cpu().numpy(), logits=torch.stack(logits).cpu().numpy())


def exact(case, seed):
    if case["kind"] == "product":
        ws, x = _product_inputs(case, seed)
        x = _round_activations(x.double(), case["dtype"])
        return [x @ _dequantize(w, case["dtype"]).T for w in ws]
    return _exact_llama(case, seed) if case["kind"] == "llama" else _exact_stack(case, seed)
