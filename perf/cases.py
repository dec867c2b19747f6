"""The work a program has this framework do, as cases that can be timed and compared.

Every case goes through the entry points a user's program calls: the patched
NF4 linear and transformer block, the prompt attention, the prompt prefill and
the frame decode of the Dual-AR model, weight quantisation and the sampler.
Widths are those of the repository's own model (slow transformer 2560 wide, 32
query and 8 KV heads, FFN 9728; fast transformer 1024 wide; codebooks of 4096)
with a few odd ones; row counts, positions and prompt lengths cover what the
model's 2304-position cache allows.

Each case is a dict with a "kind":

* "linear": one NF4 layer on `rows` activation rows, with the epilogue `epi`
  (none: the patched module call; residual / gate: `nf4gemv.matmul`).
* "block": one transformer block on `rows` positions after `start` cached ones
  (one position: the decode step; several: a prompt).
* "attention": `rows` new positions over `start` cached ones, with the boolean
  mask of the module's forward or with the positions of a causal prompt span.
* "prompt": a prompt of `tokens` after `start` cached positions through the
  Dual-AR model's bucket graphs. Twelve of the benchmark model's 36 layers:
  the layers are alike, and past a dozen the 16-bit roundings of one layer,
  carried through all the others, hide what is compared.
* "frame": `frames` greedy frames of the benchmark model (all 36 + 4 layers)
  from its 2048-position cache.
* "quantize": a dense layer's weight into the NF4 layout, as a model is loaded.
* "sample": one top-k / top-p draw from a logit row.
"""

import dataclasses
import math

import torch

from ttspipe_amd import dualar, fastpath, fusedlayer, fusedops, fusedsample, nf4gemv, quant
from ttspipe_amd.llama import BaseModelArgs, KVCache, TransformerBlock, precompute_freqs_cis

DEV = "cuda"
HD = 128
MAX_LEN = 2304
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
EPIS = {"none": nf4gemv.EPI_NONE, "residual": nf4gemv.EPI_RESIDUAL, "gate": nf4gemv.EPI_SILU_GATE}
MODELS = {
    "slow": dict(dim=2560, n_head=32, n_local_heads=8, intermediate_size=9728, max_len=MAX_LEN),
    "fast": dict(dim=1024, n_head=8, n_local_heads=2, intermediate_size=3072, max_len=16),
}
#: [out, in] of the model's linears (wqkv, wo, w1 / w3, w2 and heads, slow and fast), and two odd ones.
SHAPES = [(6144, 2560), (2560, 4096), (9728, 2560), (2560, 9728), (4096, 2560), (1536, 1024), (1024, 1024),
          (3072, 1024), (1024, 3072), (4096, 1024), (1540, 2560), (9730, 2560)]
PROMPT_LAYERS = 12


def listed():
    return [
        # a decode step's largest linear: the smallest call, one row
        dict(name="linear_1row", kind="linear", out=9728, inp=2560, rows=1, dtype="bf16", nested=True, bs=64, epi="none"),
        # a short prompt tail or a few streams: few rows, the residual folded into the store
        dict(name="linear_6rows", kind="linear", out=2560, inp=9728, rows=6, dtype="bf16", nested=True, bs=64,
             epi="residual"),
        # a sentence-long prompt, fp16 and plain scales
        dict(name="linear_100rows", kind="linear", out=9728, inp=2560, rows=100, dtype="fp16", nested=False, bs=64,
             epi="none"),
        # a whole reference-voice prompt in one call
        dict(name="linear_2048rows", kind="linear", out=9728, inp=2560, rows=2048, dtype="bf16", nested=True, bs=64,
             epi="none"),
        # one decode position through a block, as the patched model's forward runs it without a graph
        dict(name="block_decode", kind="block", model="slow", rows=1, start=1187, dtype="bf16", nested=True, qk_norm=True),
        # a ragged prompt through a block in one call
        dict(name="block_prompt", kind="block", model="slow", rows=700, start=0, dtype="bf16", nested=True, qk_norm=True),
        # a ragged prompt span attending over a cached prefix, as the module's forward calls it
        dict(name="attention_390", kind="attention", n_head=32, n_kv=8, rows=390, start=1610, dtype="bf16", causal=False),
        # what is left of a prompt after a prefix-cache hit
        dict(name="prompt_tail", kind="prompt", tokens=24, start=700),
        # a long prompt from an empty cache: the largest call
        dict(name="prompt_long", kind="prompt", tokens=1900, start=0),
        # the next frame of a stream
        dict(name="frame", kind="frame", frames=1),
        # loading a dense checkpoint
        dict(name="quantize", kind="quantize", out=9728, inp=2560, dtype="bf16", nested=True, bs=64),
        # a codebook's draw
        dict(name="sample", kind="sample", vocab=4096, top_k=30, top_p=0.8, temperature=0.7, dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5))))))


def draw(rng):
    kind = rng.choice(["linear"] * 4 + ["block"] * 2 + ["attention", "prompt", "prompt", "frame", "quantize", "sample"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    nested = rng.random() < 0.7
    if kind == "linear":
        out, inp = rng.choice(SHAPES)
        bs = rng.choice([64, 64, 128])
        return dict(kind=kind, out=out, inp=inp, rows=_log_int(rng, 1, 2048), dtype=dtype, nested=nested, bs=bs,
                    epi=rng.choice(["none", "none", "residual", "gate"]))
    if kind == "block":
        model = rng.choice(["slow", "slow", "fast"])
        if model == "fast":
            return dict(kind=kind, model=model, rows=1, start=rng.randint(0, 9), dtype=dtype, nested=nested,
                        qk_norm=rng.random() < 0.7)
        rows = rng.choice([1, _log_int(rng, 2, 1500)])
        return dict(kind=kind, model=model, rows=rows, start=rng.randint(0, MAX_LEN - rows), dtype=dtype, nested=nested,
                    qk_norm=rng.random() < 0.7)
    if kind == "attention":
        n_head, n_kv = rng.choice([(32, 8), (32, 8), (8, 2), (16, 8)])
        rows = _log_int(rng, 2, 1024)
        return dict(kind=kind, n_head=n_head, n_kv=n_kv, rows=rows,
                    start=rng.choice([0, rng.randint(0, MAX_LEN - rows)]), dtype=dtype, causal=rng.random() < 0.5)
    if kind == "prompt":
        tokens = _log_int(rng, 1, 1700)
        return dict(kind=kind, tokens=tokens, start=rng.choice([0, rng.randint(0, MAX_LEN - 512 * (-(-tokens // 512)))]))
    if kind == "frame":
        return dict(kind=kind, frames=rng.randint(2, 4))
    if kind == "quantize":
        out, inp = rng.choice(SHAPES)
        return dict(kind=kind, out=out + rng.choice([0, 0, 2 * rng.randint(1, 50)]), inp=inp, dtype=dtype, nested=nested,
                    bs=rng.choice([64, 64, 128]))
    return dict(kind=kind, vocab=_log_int(rng, 512, 32768), top_k=rng.randint(1, 64), top_p=round(rng.uniform(0.3, 0.99), 3),
                temperature=round(rng.uniform(0.3, 1.2), 3), dtype=dtype)


# ------------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, dtype, scale=1.0):
    return torch.randn(*shape, generator=g, device=DEV).mul_(scale).to(dtype)


def _linear(g, out, inp, dtype, nested, bs=64):
    """A quantised layer: uniform codes (a normal weight's NF4 codes are close to that), scales around 0.02."""
    packed = torch.randint(0, 256, (out * inp // 2, 1), generator=g, device=DEV, dtype=torch.uint8)
    code = torch.tensor(quant.NF4_CODE, dtype=torch.float32, device=DEV)
    nblk = out * inp // bs
    if nested:
        a8 = torch.randint(0, 256, (nblk,), generator=g, device=DEV, dtype=torch.uint8)
        amax2 = torch.rand(-(-nblk // 256), generator=g, device=DEV).mul_(0.004).add_(0.004)
        state2 = quant.QuantState(absmax=amax2, shape=(nblk,), code=quant.create_dynamic_map().to(DEV), blocksize=256,
                                  quant_type="dynamic", dtype=torch.float32)
        state = quant.QuantState(absmax=a8, shape=(out, inp), code=code, blocksize=bs, dtype=dtype,
                                 offset=torch.tensor(0.02, device=DEV), state2=state2)
    else:
        absmax = torch.rand(nblk, generator=g, device=DEV).mul_(0.02).add_(0.01)
        state = quant.QuantState(absmax=absmax, shape=(out, inp), code=code, blocksize=bs, dtype=dtype)
    lin = quant.Linear4bit(inp, out, bias=False, compute_dtype=dtype, compress_statistics=nested, blocksize=bs)
    lin.set_quantized(packed, state)
    nf4gemv.prepare(lin)
    return lin


def _install():
    if not (nf4gemv.install() and fusedops.install() and fusedlayer.install()):
        raise RuntimeError("the kernels are not available: no GPU, or the library is not built")


def _prepare_linear(c, g):
    dtype = DTYPES[c["dtype"]]
    lin = _linear(g, c["out"], c["inp"], dtype, c["nested"], c["bs"])
    x = _randn(g, 1, c["rows"], c["inp"], dtype=dtype)
    operand = None if c["epi"] == "none" else _randn(g, 1, c["rows"], c["out"], dtype=dtype)
    return dict(lin=lin, x=x, operand=operand, epi=EPIS[c["epi"]])


def _prepare_block(c, g):
    m, dtype = MODELS[c["model"]], DTYPES[c["dtype"]]
    dim, nh, nkv, inter, max_len = (m[k] for k in ("dim", "n_head", "n_local_heads", "intermediate_size", "max_len"))
    args = BaseModelArgs(dim=dim, n_head=nh, n_local_heads=nkv, head_dim=HD, intermediate_size=inter,
                         attention_qk_norm=c["qk_norm"], max_seq_len=max_len)
    with torch.device("meta"):
        block = TransformerBlock(args, dtype=dtype)
    a, ff = block.attention, block.feed_forward
    a.wqkv = _linear(g, (nh + 2 * nkv) * HD, dim, dtype, c["nested"])
    a.wo = _linear(g, dim, nh * HD, dtype, c["nested"])
    ff.w1, ff.w3 = (_linear(g, inter, dim, dtype, c["nested"]) for _ in range(2))
    ff.w2 = _linear(g, dim, inter, dtype, c["nested"])
    norms = [block.attention_norm, block.ffn_norm] + ([a.q_norm, a.k_norm] if c["qk_norm"] else [])
    for norm in norms:
        w = torch.rand(norm.weight.shape, generator=g, device=DEV).mul_(0.2).add_(0.9).to(dtype)
        norm.weight = torch.nn.Parameter(w, requires_grad=False)
    cache = KVCache(1, max_len, nkv, HD, dtype=dtype, device=DEV)
    start, rows = c["start"], c["rows"]
    cache.k_cache[:, :, :start] = _randn(g, 1, nkv, start, HD, dtype=dtype)
    cache.v_cache[:, :, :start] = _randn(g, 1, nkv, start, HD, dtype=dtype)
    a.kv_cache = cache
    pos = torch.arange(start, start + rows, device=DEV)
    freqs = precompute_freqs_cis(max_len, HD, 1e6).to(DEV)[pos].contiguous()
    mask = torch.tril(torch.ones(max_len, max_len, dtype=torch.bool, device=DEV))[pos][None, None]
    return dict(block=block, x=_randn(g, 1, rows, dim, dtype=dtype), freqs=freqs, mask=mask, pos=pos)


def _prepare_attention(c, g):
    dtype, rows, start = DTYPES[c["dtype"]], c["rows"], c["start"]
    nh, nkv = c["n_head"], c["n_kv"]
    q = _randn(g, 1, rows, nh, HD, dtype=dtype).transpose(1, 2)
    k, v = (_randn(g, 1, nkv, MAX_LEN, HD, dtype=dtype)[:, :, : start + rows] for _ in range(2))
    pos = torch.arange(start, start + rows, device=DEV)
    mask = torch.tril(torch.ones(MAX_LEN, MAX_LEN, dtype=torch.bool, device=DEV))[pos][None, None, :, : start + rows]
    return dict(q=q, k=k, v=v, mask=mask, pos=pos if c["causal"] else None, n_head=nh, n_kv=nkv)


def _prepare_prompt(c, g, seed):
    cfg = dataclasses.replace(dualar.DualARConfig(), n_layer=PROMPT_LAYERS, seed=seed)
    model = dualar.SyntheticDualAR(cfg, device=DEV)
    tokens = torch.randint(0, cfg.codebook_size, (cfg.n_tokens, c["tokens"]), generator=g, device=DEV, dtype=torch.int32)
    if not model.prefill(tokens, c["start"]):  # captures the bucket graphs a serving program keeps
        raise RuntimeError("the prompt does not fit the cache")
    return dict(model=model, tokens=tokens, start=c["start"], end=c["start"] + c["tokens"])


def _prepare_frame(c, seed):
    model = dualar.SyntheticDualAR(dataclasses.replace(dualar.DualARConfig(), seed=seed), device=DEV)
    model.decode(c["frames"])  # captures the frame's graph
    return dict(model=model, frames=c["frames"])


def prepare(case, seed):
    c, kind = case, case["kind"]
    _install()
    g = _gen(seed)
    if kind == "linear":
        return dict(kind=kind, **_prepare_linear(c, g))
    if kind == "block":
        return dict(kind=kind, **_prepare_block(c, g))
    if kind == "attention":
        return dict(kind=kind, **_prepare_attention(c, g))
    if kind == "prompt":
        return dict(kind=kind, **_prepare_prompt(c, g, seed))
    if kind == "frame":
        return dict(kind=kind, **_prepare_frame(c, seed))
    if kind == "quantize":
        return dict(kind=kind, dense=_randn(g, c["out"], c["inp"], dtype=DTYPES[c["dtype"]], scale=0.02),
                    nested=c["nested"], bs=c["bs"])
    dtype = DTYPES[c["dtype"]]
    return dict(kind=kind, logits=_randn(g, 1, c["vocab"], dtype=dtype, scale=3.0),
                uniform=torch.rand(c["vocab"], generator=g, device=DEV),
                temperature=torch.tensor([c["temperature"]], device=DEV, dtype=dtype),
                top_p=torch.tensor([c["top_p"]], device=DEV, dtype=dtype), top_k=torch.tensor([c["top_k"]], device=DEV))


# --------------------------------------------------------------------- work


def _prompt_outputs(s):
    """What a prompt leaves: the last position's logits and the cache up to the
    prompt's end (the padding's rows past it are overwritten before they are
    read) of the first, a middle and the last layer. Every position of every
    layer reaches these through the layers above it."""
    layers = s["model"].layers
    out = {"logits": s["model"].logits}
    for i in (0, len(layers) // 2, len(layers) - 1):
        cache = layers[i].attention.kv_cache
        out[f"k{i}"], out[f"v{i}"] = cache.k_cache[:, :, : s["end"]], cache.v_cache[:, :, : s["end"]]
    return out


def run(s):
    kind = s["kind"]
    if kind == "linear":
        if s["operand"] is None:
            return s["lin"](s["x"])
        return nf4gemv.matmul(s["lin"], s["x"], epi=s["epi"], operand=s["operand"])
    if kind == "block":
        y = s["block"](s["x"], s["freqs"], s["mask"], s["pos"])
        cache = s["block"].attention.kv_cache
        return {"y": y, "k": cache.k_cache, "v": cache.v_cache}
    if kind == "attention":
        return fastpath.prefill_attention(s["q"], s["k"], s["v"], s["mask"], s["n_head"], s["n_kv"], HD, positions=s["pos"])
    if kind == "prompt":
        s["model"].prefill(s["tokens"], s["start"])
        return _prompt_outputs(s)
    if kind == "frame":
        tokens = s["model"].decode(s["frames"])
        cache = s["model"].layers[-1].attention.kv_cache  # every layer's new rows reach the logits
        return {"tokens": tokens, "logits": s["model"].logits, "fast_logits": s["model"].fast_logits,
                "k": cache.k_cache, "v": cache.v_cache}
    if kind == "quantize":
        dense = s["dense"]
        lin = quant.Linear4bit(dense.shape[1], dense.shape[0], bias=False, compute_dtype=dense.dtype,
                               compress_statistics=s["nested"], blocksize=s["bs"])
        lin.load_weight(dense)
        state = lin.weight.quant_state
        out = {"packed": lin.weight.data, "absmax": state.absmax}
        if s["nested"]:
            out["absmax2"], out["offset"] = state.state2.absmax, state.offset
        return out
    return fusedsample.sample(s["logits"], s["temperature"], s["top_p"], s["top_k"], uniform=s["uniform"])


# ------------------------------------------------------------ what is needed


def _weight_bytes(out, inp, nested, bs=64):
    nblk = out * inp // bs
    return out * inp // 2 + (nblk + 4 * -(-nblk // 256) + 1028 if nested else 4 * nblk)


def _block_work(m, rows, start, nested):
    dim, nh, nkv, inter = m["dim"], m["n_head"], m["n_local_heads"], m["intermediate_size"]
    shapes = [((nh + 2 * nkv) * HD, dim), (dim, nh * HD), (inter, dim), (inter, dim), (dim, inter)]
    keys = rows * start + rows * (rows + 1) // 2  # (query, key) pairs of the causal mask
    nbytes = (sum(_weight_bytes(o, i, nested) for o, i in shapes) + 2 * nkv * HD * 2 * (start + rows) + 4 * rows * dim)
    return nbytes, 2 * rows * sum(o * i for o, i in shapes) + 4 * keys * nh * HD


def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        y = 2 * c["rows"] * c["out"]
        return {"bytes": _weight_bytes(c["out"], c["inp"], c["nested"], c["bs"]) + 2 * c["rows"] * c["inp"]
                + y * (1 if c["epi"] == "none" else 2), "flops": 2 * c["rows"] * c["out"] * c["inp"]}
    if kind == "block":
        nbytes, flops = _block_work(MODELS[c["model"]], c["rows"], c["start"], c["nested"])
        return {"bytes": nbytes, "flops": flops}
    if kind == "attention":
        keys = c["rows"] * c["start"] + c["rows"] * (c["rows"] + 1) // 2
        return {"bytes": 4 * c["rows"] * c["n_head"] * HD + 4 * c["n_kv"] * HD * (c["start"] + c["rows"]),
                "flops": 4 * keys * c["n_head"] * HD}
    if kind == "prompt":
        cfg, n = dualar.DualARConfig(), c["tokens"]
        nbytes, flops = _block_work(MODELS["slow"], n, c["start"], True)
        head = _weight_bytes(cfg.vocab_size, cfg.dim, True) + 2 * (cfg.dim + cfg.vocab_size)
        return {"bytes": PROMPT_LAYERS * (nbytes - 4 * n * cfg.dim) + 2 * cfg.n_tokens * n * cfg.dim + head,
                "flops": PROMPT_LAYERS * flops + 2 * cfg.vocab_size * cfg.dim}
    if kind == "frame":
        cfg = dualar.DualARConfig()
        nbytes = sum(dualar.step_bytes(cfg, cfg.prefill_len + i) for i in range(c["frames"]))
        return {"bytes": nbytes, "flops": 4 * nbytes}  # two codes a byte, a multiply and an add each
    if kind == "quantize":
        n = c["out"] * c["inp"]
        return {"bytes": 2 * n + _weight_bytes(c["out"], c["inp"], c["nested"], c["bs"]), "flops": 4 * n}
    return {"bytes": 6 * c["vocab"] + 4, "flops": 8 * c["vocab"]}


def tolerance(case):
    """Two correct implementations differ by their roundings to the activation
    type (bf16 keeps 8 bits, fp16 11) and by which the sums' order turns over."""
    kind = case["kind"]
    if kind in ("quantize", "sample"):
        return "exact"
    if kind == "prompt":
        return {"rel": 0.03, "max": 0.9}
    if kind == "frame":
        return {"rel": 0.02, "max": 0.5}
    bf16 = case["dtype"] == "bf16"
    if kind == "block":
        return {"rel": 0.012, "max": 0.12} if bf16 else {"rel": 0.002, "max": 0.02}
    return {"rel": 0.008, "max": 0.05} if bf16 else {"rel": 0.0012, "max": 0.008}


# ------------------------------------------------------------ in 64 bits


def _dense64(packed, state):
    flat = packed.reshape(-1)
    codes = torch.stack([flat >> 4, flat & 15], dim=1).reshape(-1).long()
    values = state.code.double()[codes].view(-1, state.blocksize)
    if state.nested:
        s = state.state2.code.double()[state.absmax.long()].view(-1)
        group = torch.arange(s.numel(), device=s.device) // state.state2.blocksize
        s = s * state.state2.absmax.double()[group] + float(state.offset)
    else:
        s = state.absmax.double()
    return (values * s[:, None]).view(state.shape)


def _mm64(lin, x):
    return x @ _dense64(lin.weight.data, lin.weight.quant_state).t()


def _rms64(x, weight, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * weight.double()


def _rope64(x, freqs):  # x (rows, heads, 128), freqs (rows, 64, 2)
    f = freqs.double()[:, None]
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * f[..., 0] - b * f[..., 1], b * f[..., 0] + a * f[..., 1]], dim=-1).flatten(-2)


def _attend64(q, k, v, pos):
    """q (heads, rows, 128), k / v (kv heads, keys, 128), row i sees keys 0 .. pos[i]."""
    groups = q.shape[0] // k.shape[0]
    seen = torch.arange(k.shape[1], device=q.device)[None] <= pos[:, None]
    out = []
    for h in range(q.shape[0]):
        p = (q[h] @ k[h // groups].t() * HD**-0.5).masked_fill(~seen, float("-inf")).softmax(-1)
        out.append(p @ v[h // groups])
    return torch.stack(out)


def _block64(block, x, freqs, pos, kc, vc):
    """x (rows, dim) at positions pos; kc / vc (kv heads, max_len, 128) get the new rows."""
    a, ff = block.attention, block.feed_forward
    nh, nkv, rows = a.n_head, a.n_local_heads, x.shape[0]
    qkv = _mm64(a.wqkv, _rms64(x, block.attention_norm.weight, block.attention_norm.eps))
    q, k, v = (t.view(rows, -1, HD) for t in qkv.split([nh * HD, nkv * HD, nkv * HD], dim=-1))
    if a.attention_qk_norm:
        q, k = _rms64(q, a.q_norm.weight, a.q_norm.eps), _rms64(k, a.k_norm.weight, a.k_norm.eps)
    q, k = _rope64(q, freqs), _rope64(k, freqs)
    kc[:, pos], vc[:, pos] = k.transpose(0, 1), v.transpose(0, 1)
    end = int(pos[-1]) + 1
    y = _attend64(q.transpose(0, 1), kc[:, :end], vc[:, :end], pos)
    h = x + _mm64(a.wo, y.transpose(0, 1).reshape(rows, nh * HD))
    n = _rms64(h, block.ffn_norm.weight, block.ffn_norm.eps)
    return h + _mm64(ff.w2, torch.nn.functional.silu(_mm64(ff.w1, n)) * _mm64(ff.w3, n))


def _caches64(block):
    cache = block.attention.kv_cache
    return cache.k_cache[0].double(), cache.v_cache[0].double()


def _model64(model, tokens, pos, keep):
    """The slow transformer's (logits of the last position, {layer: caches}) for tokens (n_tokens, n)."""
    cfg = model.cfg
    table = model.tensors["embeddings"].view(cfg.n_tokens, cfg.vocab_size, cfg.dim)
    x = sum(table[c][tokens[c].long()].double() for c in range(cfg.n_tokens))
    freqs, kept = model.freqs[pos], {}
    for i, block in enumerate(model.layers):
        kc, vc = _caches64(block)
        x = _block64(block, x, freqs, pos, kc, vc)
        if i in keep:
            kept[i] = (kc[None], vc[None])
    return _mm64(model.output, _rms64(x[-1:], model.tensors["norm"], cfg.norm_eps)), kept


def _exact_quantize(s):
    """The scales in 64 bits; the codes are whole numbers."""
    blocks = s["dense"].double().reshape(-1)
    pad = -blocks.numel() % s["bs"]
    absmax = torch.nn.functional.pad(blocks, (0, pad)).view(-1, s["bs"]).abs().amax(1)
    if not s["nested"]:
        return {"packed": None, "absmax": absmax}
    offset = absmax.mean()
    centred = torch.nn.functional.pad(absmax - offset, (0, -absmax.numel() % 256)).view(-1, 256)
    return {"packed": None, "absmax": None, "absmax2": centred.abs().amax(1), "offset": offset}


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "sample" or (kind == "frame" and c["frames"] > 1):
        return None  # whole numbers; frames that follow the tokens of the first
    s = prepare(case, seed)
    if kind == "linear":
        y = _mm64(s["lin"], s["x"].double())
        if c["epi"] == "residual":
            y = s["operand"].double() + y
        elif c["epi"] == "gate":
            y = torch.nn.functional.silu(s["operand"].double()) * y
        return y
    if kind == "block":
        kc, vc = _caches64(s["block"])
        y = _block64(s["block"], s["x"][0].double(), s["freqs"], s["pos"], kc, vc)
        return {"y": y[None], "k": kc[None], "v": vc[None]}
    if kind == "attention":
        pos = torch.arange(c["start"], c["start"] + c["rows"], device=DEV)
        return _attend64(s["q"][0].double(), s["k"][0].double(), s["v"][0].double(), pos)[None]
    if kind == "quantize":
        return _exact_quantize(s)
    model = s["model"]
    last = len(model.layers) - 1
    if kind == "prompt":
        pos = torch.arange(s["start"], s["end"], device=DEV)
        keep = (0, len(model.layers) // 2, last)
        logits, kept = _model64(model, s["tokens"], pos, keep)
        out = {"logits": logits}
        for i in keep:
            out[f"k{i}"], out[f"v{i}"] = kept[i][0][:, :, : s["end"]], kept[i][1][:, :, : s["end"]]
        return out
    first = torch.tensor(dualar.first_tokens(model.cfg), device=DEV)[:, None]
    pos = torch.tensor([model.cfg.prefill_len], device=DEV)
    logits, kept = _model64(model, first, pos, (last,))
    return {"tokens": None, "logits": logits, "fast_logits": None, "k": kept[last][0], "v": kept[last][1]}
