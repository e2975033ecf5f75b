"""Workloads of this framework, as its users run them: AWQ linears and their offline tools, the Qwen3 module forward, decode
steps of the engines and prompt passes of the hybrid decoders.

Sizes are those of the Qwen3 models and of the hybrid layer sizes this repository configures, tests and benchmarks.  Weights are
random with the distributions of real ones: AWQ words come from quantised normal weights, linears keep the scale of their
input."""
from __future__ import annotations

import math

import torch

GROUP = 128
VOCAB = 32768
EPS = 1e-6
BLOCK = 64
F64 = torch.float64
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
# layer sizes: width, query heads, kv heads, feed-forward width (heads of 128)
SIZES = {"0.6b": (1024, 16, 8, 3072), "1.7b": (2048, 16, 8, 6144), "4b": (2560, 32, 8, 9728), "8b": (4096, 32, 8, 12288)}
# the linears of the Qwen3 models, [in, out]
LINEARS = [(1024, 2048), (1024, 1024), (2048, 1024), (1024, 3072), (3072, 1024), (1024, 6144), (2048, 6144), (6144, 2048),
           (2560, 9728), (9728, 2560), (4096, 4096), (4096, 12288), (12288, 4096), (4096, 24576), (5120, 10240), (8192, 5120),
           (5120, 17408), (17408, 5120), (5120, 25600), (25600, 5120)]
MOST_LINEAR = 8192 * 4096 * 12288
EXPERTS, TOP = 8, 2
TAPS, STATES, RANK, ROT = 4, 16, 512, 64


def _linear(name, rows, k, n, dtype, group=GROUP, bias=False):
    return {"name": name, "kind": "linear", "rows": rows, "k": k, "n": n, "dtype": dtype, "group": group, "bias": bias}


def listed():
    return [
        # one projection of a small model for a batch of 16 decoding sequences: launch and host latency
        _linear("linear_16x1024x3072_f16", 16, 1024, 3072, "f16"),
        # an MLP projection of the largest model, one sequence decoding: the packed weight streams from memory
        _linear("linear_1x5120x25600_f16", 1, 5120, 25600, "f16"),
        # the same MLP's other projection for a full batch of 64 sequences
        _linear("linear_64x25600x5120_bf16", 64, 25600, 5120, "bf16"),
        # a short ragged prompt through a linear with bias, finer groups and an odd output width
        _linear("linear_333x2816x9720_f16_g64_bias", 333, 2816, 9720, "f16", 64, True),
        # a batch of prompts through an MLP projection
        _linear("linear_8192x4096x12288_bf16", 8192, 4096, 12288, "bf16"),
        # unpacking a weight for a caller that wants it dense
        {"name": "dequantize_4096x12288_bf16", "kind": "dequantize", "k": 4096, "n": 12288, "dtype": "bf16", "group": GROUP},
        # quantising one linear of a checkpoint, which is done once for every weight of a model
        {"name": "quantize_4096x12288_bf16", "kind": "quantize", "k": 4096, "n": 12288, "dtype": "bf16", "group": GROUP},
        # the module forward with logits of every position: scoring and perplexity
        {"name": "qwen3_forward_0.6b_4x2048", "kind": "qwen3_forward", "size": "0.6b", "layers": 6, "batch": 4, "tokens": 2048},
        # one decode step of the whole Qwen3-0.6B architecture for 32 sequences
        {"name": "qwen3_decode_0.6b_32x640", "kind": "qwen3_decode", "size": "0.6b", "layers": 28, "batch": 32, "context": 640},
        # four prompts of unequal lengths through attention, gated linear attention and experts
        {"name": "gafulix_prompt_8b_4x8192", "kind": "hybrid_prompt", "model": "gafulix", "size": "8b", "prompts": 4,
         "tokens": 8192},
        # one decode step of the same layers for 16 sequences
        {"name": "gafulix_decode_8b_16x2048", "kind": "hybrid_decode", "model": "gafulix", "size": "8b", "batch": 16,
         "context": 2048},
        # sixteen prompts through attention, selective scan and latent attention
        {"name": "roletar_prompt_0.6b_16x8192", "kind": "hybrid_prompt", "model": "roletar", "size": "0.6b", "prompts": 16,
         "tokens": 8192},
    ]


def _spread(rng, low, high):
    """A whole number, spread over the logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def draw(rng):
    kind = rng.choice(["linear"] * 5 + ["dequantize", "quantize", "qwen3_forward", "qwen3_decode", "hybrid_prompt",
                                        "hybrid_prompt", "hybrid_decode", "hybrid_decode"])
    if kind in ("linear", "dequantize", "quantize"):
        k, n = rng.choice(LINEARS)
        group = rng.choice([128, 128, 128, 64, 32])
        if rng.random() < 0.4:                       # widths of no particular model
            step = max(group, 64)
            k, n = step * _spread(rng, 512 // step, 16384 // step), 8 * _spread(rng, 64, 2048)
        case = {"kind": kind, "k": k, "n": n, "dtype": rng.choice(["f16", "bf16"]), "group": group}
        if kind == "linear":
            case["rows"] = _spread(rng, 1, max(1, min(8192, MOST_LINEAR // (k * n))))
            case["bias"] = rng.random() < 0.25
        return case
    if kind == "qwen3_forward":
        size, batch = rng.choice(["0.6b", "1.7b"]), _spread(rng, 1, 8)
        return {"kind": kind, "size": size, "layers": rng.randint(1, 3 if size == "1.7b" else 6), "batch": batch,
                "tokens": _spread(rng, 64, 8192 // batch)}
    if kind == "qwen3_decode":
        batch = _spread(rng, 1, 64)
        return {"kind": kind, "size": rng.choice(list(SIZES)), "layers": rng.randint(2, 6), "batch": batch,
                "context": _spread(rng, 64, min(8192, 65536 // batch))}
    case = {"kind": kind, "model": rng.choice(["gafulix", "roletar"]), "size": rng.choice(["0.6b", "1.7b", "8b"])}
    if kind == "hybrid_prompt":
        case["prompts"] = _spread(rng, 1, 16)
        case["tokens"] = _spread(rng, 40 * case["prompts"], 8192 if case["size"] != "8b" else 4096)
    else:
        case["batch"] = _spread(rng, 1, 64)
        case["context"] = _spread(rng, 64, min(8192, 65536 // case["batch"]))
    return case


# ---- inputs, from the seed alone ----------------------------------------------------------------------------------------
def _generator(seed, salt=0):
    return torch.Generator(device="cuda").manual_seed(seed * 1009 + salt)


def _normal(gen, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=gen, device="cuda") * std).to(dtype)


def _pack(q):
    """[R, C] whole numbers 0..15 -> int32 words, nibble j = column 8 i + (0, 2, 4, 6, 1, 3, 5, 7)[j]."""
    q = q.to(torch.int32).view(q.shape[0], -1, 8)
    words = torch.zeros_like(q[:, :, 0])
    for j, c in enumerate((0, 2, 4, 6, 1, 3, 5, 7)):
        words |= q[:, :, c] << (4 * j)
    return words


def _awq(gen, k, n, group, dtype, std=0.02):
    """A normal weight [k, n] quantised per group: (words, scales, zero words), (q, z)."""
    w = _normal(gen, k // group, group, n, std=std)
    low, high = w.amin(dim=1, keepdim=True), w.amax(dim=1, keepdim=True)
    s = (high - low).clamp(min=1e-5) / 15.0
    z = (-torch.round(low / s)).clamp(0, 15)
    q = (torch.round(w / s) + z).clamp(0, 15)
    return (_pack(q.view(k, n)), s[:, 0].to(dtype), _pack(z[:, 0])), (q, z)


def _dense(packed, whole, k, n):
    return ((whole[0] - whole[1]).to(F64) * packed[1].to(F64).unsqueeze(1)).view(k, n)


def _linear_inputs(c, seed):
    gen = _generator(seed)
    dtype = DTYPES[c["dtype"]]
    packed, whole = _awq(gen, c["k"], c["n"], c["group"], dtype)
    x = _normal(gen, c["rows"], c["k"], dtype=dtype)
    # the module's bias buffer is bfloat16 whatever the other types are
    bias = _normal(gen, c["n"], std=0.5, dtype=torch.bfloat16) if c["bias"] else None
    return packed, whole, x, bias


def _qwen3_config(c):
    width, heads, kv, inter = SIZES[c["size"]]
    full = c["layers"] == 28           # the whole architecture has its own vocabulary
    return dict(num_hidden_layers=c["layers"], vocab_size=151936 if full else VOCAB, hidden_size=width, total_num_heads=heads,
                total_num_kv_heads=kv, max_position_embeddings=16384, intermediate_size=inter, head_dim=128,
                tie_word_embeddings=full, rope_theta=1000000.0, rms_norm_eps=EPS)


def _qwen3_weights(c, seed):
    """Dense tensors by name, and (packed, whole numbers) of the linears."""
    cfg, gen, bf = _qwen3_config(c), _generator(seed, 1), torch.bfloat16
    width, heads, kv, inter = SIZES[c["size"]]
    dense = {"model.embed_tokens.weight": _normal(gen, cfg["vocab_size"], width, std=0.02, dtype=bf),
             "model.norm.weight": 1 + _normal(gen, width, std=0.1, dtype=bf)}
    dense["lm_head.weight"] = (dense["model.embed_tokens.weight"] if cfg["tie_word_embeddings"]
                               else _normal(gen, cfg["vocab_size"], width, std=0.02, dtype=bf))
    dense["lm_head.bias"] = torch.zeros(cfg["vocab_size"], dtype=bf, device="cuda")
    packed = {}
    for i in range(c["layers"]):
        p = f"model.layers.{i}."
        for name, size in (("input_layernorm", width), ("post_attention_layernorm", width), ("self_attn.q_norm", 128),
                           ("self_attn.k_norm", 128)):
            dense[f"{p}{name}.weight"] = 1 + _normal(gen, size, std=0.1, dtype=bf)
        for name, k, n in (("self_attn.q_proj", width, heads * 128), ("self_attn.k_proj", width, kv * 128),
                           ("self_attn.v_proj", width, kv * 128), ("self_attn.o_proj", heads * 128, width),
                           ("mlp.up_proj", width, inter), ("mlp.gate_proj", width, inter), ("mlp.down_proj", inter, width)):
            packed[p + name] = _awq(gen, k, n, GROUP, bf, std=k ** -0.5)
    return cfg, dense, packed


def _qwen3_model(c, seed):
    from nanoquantization_amd.models.qwen3_quantized import Qwen3QuantizedForCausalLM
    cfg, dense, packed = _qwen3_weights(c, seed)
    with torch.device("cuda"):
        model = Qwen3QuantizedForCausalLM(**cfg).to(torch.bfloat16).cuda()
    for name, t in dense.items():
        model.get_parameter(name).data = t
    for name, ((qw, qs, qz), _) in packed.items():
        m = model.get_submodule(name)
        m.qweight, m.qscales, m.qzeros = qw, qs, qz
    return model.eval()


def _hybrid_config(c):
    """Three layers, one or two of each mixer; chunks and windows longer than the contexts."""
    width, heads, kv, inter = SIZES[c["size"]]
    attention = {"heads": heads, "kv_heads": kv, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "mask": {"size": 16384}}
    if c["model"] == "gafulix":
        mlp = {"kind": "moe", "expert": {"ff": inter // TOP}, "router": {"experts": EXPERTS, "top": TOP}}
        attention["rot"] = {"base": 1e6, "dims": 128}
        gla = {"heads": heads // 2, "dim": 128, "vdim": 128, "tau": 16.0}
        layers = [{"type": "attention", "mixer": attention, "mlp": mlp}] * 2 + [{"type": "gla", "mixer": gla, "mlp": mlp}]
        return {"architecture": "Gafulix", "layers": layers, "loop": None, "norm": {"eps": EPS}, "vocab": VOCAB, "width": width}
    mlp = {"kind": "dense", "ff": 3 * inter // 2}
    scan = {"inner": 2 * width, "state": STATES, "dt_rank": width // 16, "conv": TAPS}
    latent = {"heads": heads, "dim": 128, "rot_dim": ROT, "vdim": 128, "kv_rank": RANK, "scale": (128 + ROT) ** -0.5,
              "rot": {"base": 10000.0, "dims": ROT}}
    layers = [{"type": t, "mixer": m, "mlp": mlp}
              for t, m in (("attention", attention), ("mamba1", scan), ("latent_attention", latent))]
    return {"architecture": "Roletar", "layers": layers, "loop": None, "norm": {"eps": EPS}, "vocab": VOCAB, "width": width,
            "streams": 2, "logit_softcap": 30.0}


def _hybrid_shapes(cfg):
    """Checkpoint tensor name -> shape."""
    w = cfg["width"]
    shapes = {"embed": (cfg["vocab"], w), "final.norm": (w,), "head": (cfg["vocab"], w)}
    for i, layer in enumerate(cfg["layers"]):
        p, m, f, t = f"l{i}.", layer["mixer"], layer["mlp"], {}
        if layer["type"] in ("attention", "gla"):
            nq, nk, nv = m["heads"] * m["dim"], m.get("kv_heads", m["heads"]) * m["dim"], m.get("kv_heads", m["heads"]) * m["vdim"]
            t.update({"mix.q": (nq, w), "mix.k": (nk, w), "mix.v": (nv, w), "mix.o": (w, m["heads"] * m["vdim"])})
        if layer["type"] == "gla":
            t.update({"mix.g": (nv, w), "mix.a1": (16, w), "mix.a2": (nq, 16), "mix.a2.b": (nq,), "mix.norm": (m["vdim"],)})
        elif layer["type"] == "latent_attention":
            h, rank = m["heads"], m["kv_rank"]
            t.update({"mix.q": (h * (m["dim"] + m["rot_dim"]), w), "mix.dkv": (rank + m["rot_dim"], w), "mix.dkv.norm": (rank,),
                      "mix.uk": (h * m["dim"], rank), "mix.uv": (h * m["vdim"], rank), "mix.o": (w, h * m["vdim"])})
        elif layer["type"] == "mamba1":
            ch, n, r = m["inner"], m["state"], m["dt_rank"]
            t.update({"mix.in": (2 * ch, w), "mix.conv": (ch, m["conv"]), "mix.conv.b": (ch,), "mix.x": (r + 2 * n, ch),
                      "mix.dt": (ch, r), "mix.dt.b": (ch,), "mix.A_log": (ch, n), "mix.D": (ch,), "mix.o": (w, ch)})
        t.update({"norm1": (w,), "norm2": (w,)})
        if cfg["architecture"] == "Gafulix":
            if layer["type"] == "attention":
                t.update({"mix.q.b": (nq,), "mix.k.b": (nk,), "mix.v.b": (nv,), "mix.q.norm": (nq,), "mix.k.norm": (nk,)})
            t.update({"norm1b": (w,), "norm2b": (w,), "mlp.router": (f["router"]["experts"], w)})
            for e in range(f["router"]["experts"]):
                t.update({f"mlp.e{e}.gate": (f["expert"]["ff"], w), f"mlp.e{e}.up": (f["expert"]["ff"], w),
                          f"mlp.e{e}.down": (w, f["expert"]["ff"])})
        else:
            s = cfg["streams"]
            if layer["type"] == "attention":
                t["mix.sink"] = (m["heads"],)
            t.update({"mlp.up": (f["ff"], w), "mlp.down": (w, f["ff"])})
            t.update({f"hc{n}.{x}": (s, s) if x == "mix" else (s,) for n in (1, 2) for x in ("in", "out", "mix")})
        shapes.update({p + n: s for n, s in t.items()})
    return shapes


def _hybrid_weights(cfg, seed):
    """Every checkpoint tensor in turn.  Linears keep the scale of their input; decays are slow and scan steps small, as trained
    ones are.  A token's experts are decided by a ladder of scores in the first dimensions of its embedding, which no sublayer
    writes: like a trained router's, the choices do not hang on rounding."""
    gen, bf = _generator(seed, 2), torch.bfloat16
    ladder = 0.5 * (torch.arange(EXPERTS, device="cuda", dtype=torch.float32) - 0.5 * (EXPERTS - 1))
    moe = cfg["architecture"] == "Gafulix"
    for name, shape in _hybrid_shapes(cfg).items():
        last = name.split(".")[-1]
        if "norm" in last or last in ("norm1b", "norm2b"):
            t = 1 + _normal(gen, *shape, std=0.1)
        elif name.endswith("a2.b"):
            t = 2 + _normal(gen, *shape, std=0.5)
        elif name.endswith("dt.b"):
            t = -3 + _normal(gen, *shape, std=0.5)
        elif last == "A_log":
            t = torch.arange(1, shape[1] + 1, device="cuda").float().log().expand(shape)
        elif last == "mix":
            t = 0.8 * torch.eye(shape[0], device="cuda") + 0.2 / shape[0]
        elif last in ("in", "out") and len(shape) == 1:
            t = torch.full(shape, 1.0 / shape[0] if last == "in" else 1.0, device="cuda")
        elif last in ("b", "D", "sink"):
            t = _normal(gen, *shape, std=0.3)
        elif last == "router":
            t = torch.zeros(shape, device="cuda")
            t[:, :shape[0]] = torch.eye(shape[0], device="cuda")
        else:
            t = _normal(gen, *shape, std=1.0 if name == "embed" else shape[-1] ** -0.5)
            if moe and name == "embed":
                t[:, :EXPERTS] = ladder[torch.rand(shape[0], EXPERTS, generator=gen, device="cuda").argsort(dim=1)]
            elif moe and (name.endswith("mix.o") or last == "down"):
                t[:EXPERTS] = 0
        yield name, t.to(bf)


def _hybrid_model(cfg, seed):
    from nanoquantization_amd.models import gafulix, roletar
    module, cls = {"Gafulix": (gafulix, "GafulixForCausalLM"), "Roletar": (roletar, "RoletarForCausalLM")}[cfg["architecture"]]
    with torch.device("cuda"):
        model = getattr(module, cls)(module.spec_from_config(cfg)).to(torch.bfloat16)
    views = model.checkpoint_views()
    for name, t in _hybrid_weights(cfg, seed):
        views[name].data.copy_(t)
    return model.eval()


def _lengths(prompts, tokens):
    """Unequal lengths that add up to `tokens`: from about half the mean to one and a half times it."""
    part = [1 + (2 * i + 1 - prompts) / (2 * prompts) for i in range(prompts)]
    out = [max(1, int(tokens * p / prompts)) for p in part]
    out[-1] += tokens - sum(out)
    return out


def _token_ids(gen, vocab, n):
    return torch.randint(0, vocab, (n,), generator=gen, device="cuda")


def _context(c):
    """Tokens in the cache of every sequence of a decode batch: up to an eighth fewer than the case names."""
    return [c["context"] - i * c["context"] // (8 * c["batch"]) for i in range(c["batch"])]


def _decode_inputs(c, seed, vocab):
    return _token_ids(_generator(seed, 3), vocab, c["batch"]).tolist()


def _cached(c, seed, run, shape):
    """What layer run `run` has cached: [batch, tokens, *shape], scale one as behind norms and scale-keeping projections."""
    tokens = -(-(c["context"] + 1) // BLOCK) * BLOCK
    return _normal(_generator(seed, 100 + run), c["batch"], tokens, *shape, dtype=torch.bfloat16)


def _state(c, seed, run, shape):
    return _normal(_generator(seed, 500 + run), c["batch"], *shape)


def _paged(pages, leases, content):
    """Sequence contents [batch, tokens, heads, row] into the sequences' blocks."""
    batch, tokens = content.shape[:2]
    blocks = torch.tensor([l.blocks[:tokens // BLOCK] for l in leases], device="cuda").reshape(-1)
    pages[blocks] = content.view(batch * tokens // BLOCK, BLOCK, *content.shape[2:]).transpose(1, 2)


def _hybrid_runs(cfg):
    """Per layer: the shapes of its cached keys and values, or of its state and of the inputs its convolution keeps."""
    for layer in cfg["layers"]:
        m = layer["mixer"]
        if layer["type"] == "attention":
            yield "kv", (m["kv_heads"], 128), (m["kv_heads"], 128)
        elif layer["type"] == "latent_attention":
            yield "kv", (1, m["kv_rank"] + m["rot_dim"]), None
        elif layer["type"] == "gla":
            yield "state", (m["heads"], m["dim"], m["vdim"]), None
        else:
            yield "state", (m["state"], m["inner"]), (m["conv"] - 1, m["inner"])


# ---- what a program has in hand, and one pass -----------------------------------------------------------------------------
@torch.no_grad()
def prepare(case, seed):
    import nanoquantization_amd as nq
    from nanoquantization_amd.engine import HybridEngine, LLMEngine, Portion
    c, kind = case, case["kind"]
    if kind == "linear":
        packed, _, x, bias = _linear_inputs(c, seed)
        m = nq.WQLinear_GEMM(4, c["group"], c["k"], c["n"], "cuda", bias is not None, DTYPES[c["dtype"]])
        m.qweight, m.qscales, m.qzeros = packed
        if bias is not None:
            m.bias = bias
        return {"kind": kind, "module": m, "x": x}
    if kind == "dequantize":
        return {"kind": kind, "packed": _awq(_generator(seed), c["k"], c["n"], c["group"], DTYPES[c["dtype"]])[0]}
    if kind == "quantize":
        return {"kind": kind, "weight": _normal(_generator(seed), c["n"], c["k"], std=0.02), "group": c["group"],
                "dtype": DTYPES[c["dtype"]]}
    if kind == "qwen3_forward":
        ids = _token_ids(_generator(seed, 3), VOCAB, c["batch"] * c["tokens"]).view(c["batch"], c["tokens"])
        return {"kind": kind, "model": _qwen3_model(c, seed), "ids": ids,
                "positions": torch.arange(c["tokens"], device="cuda").unsqueeze(0)}
    if kind == "hybrid_prompt":
        cfg, lengths = _hybrid_config(c), _lengths(c["prompts"], c["tokens"])
        engine = HybridEngine(_hybrid_model(cfg, seed), max_batch=c["prompts"], max_seq_len=max(lengths) + BLOCK, block_size=BLOCK)
        ids, portions = _token_ids(_generator(seed, 3), VOCAB, c["tokens"]).tolist(), []
        for n in lengths:
            lease = engine.acquire(-(-n // BLOCK))
            portions.append(Portion(lease, 0, ids[:n], [n - 1]))
            ids = ids[n:]
        return {"kind": kind, "engine": engine, "portions": portions}
    # a decode step: sequences with filled caches and states, the step's graph captured
    if kind == "qwen3_decode":
        engine = LLMEngine(_qwen3_model(c, seed), max_batch=c["batch"], max_seq_len=c["context"] + BLOCK, block_size=BLOCK)
        vocab, runs = _qwen3_config(c)["vocab_size"], [("kv", (SIZES[c["size"]][2], 128), (SIZES[c["size"]][2], 128))] * c["layers"]
    else:
        cfg = _hybrid_config(c)
        engine = HybridEngine(_hybrid_model(cfg, seed), max_batch=c["batch"], max_seq_len=c["context"] + BLOCK, block_size=BLOCK)
        vocab, runs = VOCAB, list(_hybrid_runs(cfg))
    leases = [engine.acquire(-(-(n + 1) // BLOCK)) for n in [c["context"]] * c["batch"]]
    rows = list(zip(leases, _context(c), _decode_inputs(c, seed, vocab)))
    engine.decode(rows)
    slots = torch.tensor([max(0, l.slot) for l in leases], device="cuda")
    for i, (what, a, b) in enumerate(runs):
        if what == "kv":
            _paged(engine.cache.k[i], leases, _cached(c, seed, 2 * i, a))
            if b is not None:
                _paged(engine.cache.v[i], leases, _cached(c, seed, 2 * i + 1, b))
        else:
            engine.states.state[i][slots] = _state(c, seed, 2 * i, a)
            if b is not None:
                engine.states.tail[i][slots] = _state(c, seed, 2 * i + 1, b)
    return {"kind": kind, "engine": engine, "rows": rows}


def run(state):
    import nanoquantization_amd as nq
    kind = state["kind"]
    if kind == "linear":
        return state["module"](state["x"])
    if kind == "dequantize":
        return nq.awq_dequantize(*state["packed"])
    if kind == "quantize":
        return dict(zip(("words", "scales", "zeros"), nq.quantize_pack(state["weight"], state["group"], state["dtype"])))
    if kind == "qwen3_forward":
        with torch.no_grad():
            return state["model"].logits(state["model"](state["ids"], state["positions"]))
    engine = state["engine"]
    if kind == "hybrid_prompt":
        out = {"logits": engine.extend(state["portions"])}
        out["keys"], out["values"] = engine.cache.k, [None if v is None or v.numel() == 0 else v for v in engine.cache.v]
    else:
        out = {"logits": engine.decode(state["rows"])}
    if kind != "qwen3_decode" and engine.states is not None:
        out["states"] = engine.states.state
    return out


# ---- what a pass cannot do without ------------------------------------------------------------------------------------------
def _packed_bytes(k, n, group=GROUP):
    return k * n // 2 + (k // group) * n // 2 + 2 * (k // group) * n


def _pairs(lengths):
    return sum(n * (n + 1) // 2 for n in lengths)


def work(case):
    c, kind = case, case["kind"]
    if kind in ("linear", "dequantize", "quantize"):
        k, n = c["k"], c["n"]
        packed = _packed_bytes(k, n, c["group"])
        if kind == "linear":
            return {"bytes": packed + 2 * c["rows"] * (k + n), "flops": 2 * c["rows"] * k * n}
        return {"bytes": packed + (2 if kind == "dequantize" else 4) * k * n, "flops": (2 if kind == "dequantize" else 6) * k * n}
    width, heads, kv, inter = SIZES[c["size"]]
    if kind.startswith("qwen3"):
        vocab = _qwen3_config(c)["vocab_size"]
        weights = [(width, (heads + 2 * kv) * 128), (heads * 128, width), (width, 2 * inter), (inter, width)]
        per_row = sum(k * n for k, n in weights) * c["layers"] + width * vocab
        stored = sum(_packed_bytes(k, n) for k, n in weights) * c["layers"] + 2 * width * vocab
        if kind == "qwen3_forward":
            rows, pairs = c["batch"] * c["tokens"], c["batch"] * _pairs([c["tokens"]])
            return {"bytes": stored + rows * (8 + 2 * vocab),
                    "flops": 2 * rows * per_row + 4 * 128 * heads * pairs * c["layers"]}
        cached = sum(n + 1 for n in _context(c))
        return {"bytes": stored + c["layers"] * cached * kv * 128 * 4 + 2 * c["batch"] * vocab,
                "flops": 2 * c["batch"] * per_row + 4 * 128 * heads * cached * c["layers"]}
    cfg = _hybrid_config(c)
    prompt = kind == "hybrid_prompt"
    lengths = _lengths(c["prompts"], c["tokens"]) if prompt else [1] * c["batch"]
    rows, seqs = sum(lengths), len(lengths)
    pairs = _pairs(lengths) if prompt else sum(n + 1 for n in _context(c))
    nbytes, flops = 2 * width * VOCAB + seqs * VOCAB * 4, 2 * seqs * width * VOCAB
    for layer in cfg["layers"]:
        m, f, kept = layer["mixer"], layer["mlp"], rows if prompt else pairs
        if layer["type"] == "attention":
            dense = width * (heads + 2 * kv) * 128 + heads * 128 * width
            nbytes += 4 * kept * kv * 128
            flops += 4 * 128 * heads * pairs
        elif layer["type"] == "latent_attention":
            dense = width * (heads * (128 + ROT) + RANK + ROT) + 2 * heads * 128 * RANK + heads * 128 * width
            nbytes += 2 * kept * (RANK + ROT)
            flops += 2 * heads * pairs * ((256 + ROT) if prompt else (2 * RANK + ROT))
        elif layer["type"] == "gla":
            h = m["heads"]
            dense = width * (4 * h * 128 + 16) + 16 * h * 128 + h * 128 * width
            nbytes += 8 * seqs * h * 128 * 128
            flops += 5 * rows * h * 128 * 128
        else:
            ch = m["inner"]
            dense = 2 * width * ch + ch * (2 * m["dt_rank"] + 2 * STATES) + ch * width
            nbytes += 8 * seqs * ch * (STATES + TAPS - 1)
            flops += rows * ch * (7 * STATES + 2 * TAPS)
        flops += 2 * rows * dense
        if c["model"] == "gafulix":
            ff = f["expert"]["ff"]
            nbytes += 2 * (dense + min(EXPERTS, TOP * rows) * 3 * width * ff)
            flops += 2 * rows * TOP * 3 * width * ff
        else:
            nbytes += 2 * (dense + 2 * width * f["ff"])
            flops += 4 * rows * width * f["ff"]
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind in ("dequantize", "quantize"):
        return "exact"
    # about four times the distance of the path from the same in 64 bits: 3e-4 and 2.2e-3 for a linear, 7e-3 for three hybrid
    # layers (fp32 residual), up to 4.6e-2 for the 16-bit residual of a Qwen3 model
    if kind == "linear":
        return {"rel": 1.2e-3} if case["dtype"] == "f16" else {"rel": 9e-3}
    return {"rel": 3e-2} if kind.startswith("hybrid") else {"rel": 1e-1}


# ---- the same in 64 bits -----------------------------------------------------------------------------------------------------
def _rms(x, weight):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + EPS) * weight.to(F64)


def _mm(x, w):
    """x w^T."""
    return x @ w.to(F64).t()


def _attend(q, k, v, scale, sink=None):
    """The last len(q) of len(k) tokens: q [T, H, d], k [S, G, d], v [S, G, dv] -> [T, H * dv]."""
    (T, H, d), (S, G, dv) = q.shape, v.shape
    k, v, out = k.to(F64).permute(1, 2, 0), v.to(F64).transpose(0, 1), torch.empty(T, H, dv, dtype=F64, device=q.device)
    step = max(1, (1 << 27) // (H * S))
    for a in range(0, T, step):
        n = min(step, T - a)
        s = (q[a:a + n].view(n, G, H // G, d).permute(1, 2, 0, 3).reshape(G, -1, d) @ k * scale).view(G, H // G, n, S)
        at = torch.arange(S - T + a, S - T + a + n, device=q.device)
        s = s.masked_fill(torch.arange(S, device=q.device) > at.unsqueeze(1), -math.inf)
        top = s.amax(dim=-1, keepdim=True)
        if sink is not None:
            z = sink.to(F64).view(G, H // G, 1, 1)
            top = torch.maximum(top, z)
        p = torch.exp(s - top)
        total = p.sum(dim=-1, keepdim=True)
        if sink is not None:
            total = total + torch.exp(z - top)
        o = (p / total).view(G, -1, S) @ v
        out[a:a + n] = o.view(G, H // G, n, dv).permute(2, 0, 1, 3).reshape(n, H, dv)
    return out.view(T, H * dv)


def _angles(positions, dims, base):
    f = base ** (-2.0 * torch.arange(dims // 2, dtype=F64, device=positions.device) / dims)
    a = positions.to(F64).unsqueeze(1) * f
    return a.cos().unsqueeze(1), a.sin().unsqueeze(1)


def _half_split(x, cs):
    a, b = x.chunk(2, dim=-1)
    return torch.cat([a * cs[0] - b * cs[1], a * cs[1] + b * cs[0]], dim=-1)


def _interleaved(x, cs):
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * cs[0] - b * cs[1], a * cs[1] + b * cs[0]], dim=-1).flatten(-2)


def _exact_qwen3(c, seed):
    cfg, dense, packed = _qwen3_weights(c, seed)
    width, heads, kv, inter = SIZES[c["size"]]
    decode = c["kind"] == "qwen3_decode"
    if decode:
        contexts = _context(c)
        segments, positions = [(i, i + 1) for i in range(c["batch"])], torch.tensor(contexts, device="cuda")
        ids = torch.tensor(_decode_inputs(c, seed, cfg["vocab_size"]), device="cuda")
    else:
        T = c["tokens"]
        segments = [(i * T, i * T + T) for i in range(c["batch"])]
        positions = torch.arange(T, device="cuda").repeat(c["batch"])
        ids = _token_ids(_generator(seed, 3), VOCAB, c["batch"] * T)
    w = lambda name: dense[name + ".weight"]
    lin = lambda x, name: x @ _dense(*packed[name], x.shape[1], packed[name][0][1].shape[1])
    x, cs = w("model.embed_tokens")[ids].to(F64), _angles(positions, 128, cfg["rope_theta"])
    for i in range(c["layers"]):
        p = f"model.layers.{i}."
        h = _rms(x, w(p + "input_layernorm"))
        q = _half_split(_rms(lin(h, p + "self_attn.q_proj").view(-1, heads, 128), w(p + "self_attn.q_norm")), cs)
        k = _half_split(_rms(lin(h, p + "self_attn.k_proj").view(-1, kv, 128), w(p + "self_attn.k_norm")), cs)
        v = lin(h, p + "self_attn.v_proj").view(-1, kv, 128)
        if decode:
            ck, cv = _cached(c, seed, 2 * i, (kv, 128)), _cached(c, seed, 2 * i + 1, (kv, 128))
        o = []
        for s, (a, b) in enumerate(segments):
            ks, vs = k[a:b], v[a:b]
            if decode:
                ks, vs = (torch.cat([t[s, :contexts[s]].to(F64), new]) for t, new in ((ck, ks), (cv, vs)))
            o.append(_attend(q[a:b], ks, vs, 128 ** -0.5))
        x = x + lin(torch.cat(o), p + "self_attn.o_proj")
        h = _rms(x, w(p + "post_attention_layernorm"))
        gate = lin(h, p + "mlp.gate_proj")
        x = x + lin(gate * torch.sigmoid(gate) * lin(h, p + "mlp.up_proj"), p + "mlp.down_proj")
    logits = _mm(_rms(x, w("model.norm")), w("lm_head"))
    return {"logits": logits} if decode else logits.view(c["batch"], c["tokens"], -1)


def _exact_mixer(c, seed, i, kind, m, t, h, segments, positions, contexts):
    """What the output projection of layer i takes."""
    silu = lambda z: z * torch.sigmoid(z)
    decode, T, H = contexts is not None, h.shape[0], m.get("heads")

    def with_cache(new, which, s, shape):
        if not decode:
            return new
        return torch.cat([_cached(c, seed, 2 * i + which, shape)[s, :contexts[s]].to(F64), new])

    out = []
    if kind == "attention":
        G = m["kv_heads"]
        q, k, v = (_mm(h, t[n]) + (t[n + ".b"].to(F64) if n + ".b" in t else 0) for n in "qkv")
        if "q.norm" in t:
            q, k = _rms(q, t["q.norm"]), _rms(k, t["k.norm"])
        q, k, v = q.view(T, H, 128), k.view(T, G, 128), v.view(T, G, 128)
        if "rot" in m:
            cs = _angles(positions, 128, m["rot"]["base"])
            q, k = _interleaved(q, cs), _interleaved(k, cs)
        for s, (a, b) in enumerate(segments):
            out.append(_attend(q[a:b], with_cache(k[a:b], 0, s, (G, 128)), with_cache(v[a:b], 1, s, (G, 128)), m["scale"],
                               t.get("sink")))
        return torch.cat(out)
    if kind == "latent_attention":
        q, down = _mm(h, t["q"]).view(T, H, 128 + ROT), _mm(h, t["dkv"])
        cs = _angles(positions, ROT, m["rot"]["base"])
        q = torch.cat([q[..., :128], _interleaved(q[..., 128:], cs)], dim=-1)
        new = torch.cat([_rms(down[:, :RANK], t["dkv.norm"]), _interleaved(down[:, None, RANK:], cs)[:, 0]], dim=1)
        for s, (a, b) in enumerate(segments):
            rows = with_cache(new[a:b].unsqueeze(1), 0, s, (1, RANK + ROT))[:, 0]
            k = torch.cat([_mm(rows[:, :RANK], t["uk"]).view(-1, H, 128), rows[:, None, RANK:].expand(-1, H, ROT)], dim=-1)
            out.append(_attend(q[a:b], k, _mm(rows[:, :RANK], t["uv"]).view(-1, H, 128), m["scale"]))
        return torch.cat(out)
    if kind == "gla":
        q, k, v = (_mm(h, t[n]).view(T, H, 128) for n in "qkv")
        decay = torch.sigmoid(_mm(_mm(h, t["a1"]), t["a2"]) + t["a2.b"].to(F64)).pow(1.0 / m["tau"]).view(T, H, 128)
        o = torch.empty(T, H, 128, dtype=F64, device="cuda")
        first = _state(c, seed, 2 * i, (H, 128, 128)).to(F64) if decode else None
        for s, (a, b) in enumerate(segments):
            S = first[s] if decode else torch.zeros(H, 128, 128, dtype=F64, device="cuda")
            for r in range(a, b):
                S = torch.addcmul(k[r].unsqueeze(-1) * v[r].unsqueeze(-2), S, decay[r].unsqueeze(-1))
                o[r] = (q[r].unsqueeze(-2) @ S)[:, 0]
        return _rms(o * 128 ** -0.5, t["norm"]).reshape(T, -1) * silu(_mm(h, t["g"]))
    ch = m["inner"]
    x_in, z = _mm(h, t["in"]).split([ch, ch], dim=1)
    before = _state(c, seed, 2 * i + 1, (TAPS - 1, ch)).to(F64) if decode else None
    first = _state(c, seed, 2 * i, (STATES, ch)).to(F64) if decode else None
    conv = torch.empty_like(x_in)
    for s, (a, b) in enumerate(segments):
        padded = torch.cat([before[s] if decode else x_in.new_zeros(TAPS - 1, ch), x_in[a:b]])
        conv[a:b] = silu(t["conv.b"].to(F64) + sum(t["conv"][:, k].to(F64) * padded[k:k + b - a] for k in range(TAPS)))
    low, B, C = _mm(conv, t["x"]).split([m["dt_rank"], STATES, STATES], dim=1)
    dt, A = torch.nn.functional.softplus(_mm(low, t["dt"]) + t["dt.b"].to(F64)), -torch.exp(t["A_log"].to(F64)).t()
    y = torch.empty_like(conv)
    for s, (a, b) in enumerate(segments):
        S = first[s] if decode else torch.zeros(STATES, ch, dtype=F64, device="cuda")
        for r in range(a, b):
            S = torch.addcmul((dt[r] * conv[r]) * B[r].unsqueeze(1), S, torch.exp(dt[r] * A))
            y[r] = C[r] @ S
    return (y + t["D"].to(F64) * conv) * silu(z)


def _exact_hybrid(c, seed):
    cfg = _hybrid_config(c)
    t = dict(_hybrid_weights(cfg, seed))
    contexts = None
    if c["kind"] == "hybrid_prompt":
        lengths = _lengths(c["prompts"], c["tokens"])
        ids, first = _token_ids(_generator(seed, 3), VOCAB, c["tokens"]), [0]
        for n in lengths:
            first.append(first[-1] + n)
        positions = torch.cat([torch.arange(n, device="cuda") for n in lengths])
    else:
        contexts = _context(c)
        ids, first = torch.tensor(_decode_inputs(c, seed, VOCAB), device="cuda"), list(range(c["batch"] + 1))
        positions = torch.tensor(contexts, device="cuda")
    segments = list(zip(first, first[1:]))
    x = t["embed"][ids].to(F64)
    xs = [x, x]
    for i, layer in enumerate(cfg["layers"]):
        p = f"l{i}."
        mix = {n[len(p) + 4:]: w for n, w in t.items() if n.startswith(p + "mix.")}

        def mixer(h):
            return _mm(_exact_mixer(c, seed, i, layer["type"], layer["mixer"], mix, h, segments, positions, contexts), mix["o"])

        def experts(h):
            score = torch.sigmoid(_mm(h, t[p + "mlp.router"]))
            best, pick = score.topk(TOP, dim=1)
            y = torch.zeros_like(h)
            for e in range(EXPERTS):
                row, choice = (pick == e).nonzero(as_tuple=True)
                u = h[row] * best[row, choice].unsqueeze(1)
                gate = _mm(u, t[f"{p}mlp.e{e}.gate"])
                y.index_add_(0, row, _mm(gate * torch.sigmoid(gate) * _mm(u, t[f"{p}mlp.e{e}.up"]), t[f"{p}mlp.e{e}.down"]))
            return y

        if c["model"] == "gafulix":
            x = x + _rms(mixer(_rms(x, t[p + "norm1"])), t[p + "norm1b"])
            x = x + _rms(experts(_rms(x, t[p + "norm2"])), t[p + "norm2b"])
            continue
        for n, f in ((1, mixer), (2, lambda h: _mm(_mm(h, t[p + "mlp.up"]).clamp(min=0) ** 2, t[p + "mlp.down"]))):
            hc = {k: t[f"{p}hc{n}.{k}"].to(F64) for k in ("in", "out", "mix")}
            y = f(_rms(sum(a * s for a, s in zip(hc["in"], xs)), t[f"{p}norm{n}"]))
            xs = [sum(hc["mix"][s, d] * xs[s] for s in range(2)) + hc["out"][d] * y for d in range(2)]
    last = x if c["model"] == "gafulix" else xs[0] + xs[1]
    rows = torch.tensor([b - 1 for b in first[1:]], device="cuda")
    logits = _mm(_rms(last[rows], t["final.norm"]), t["head"])
    if c["model"] == "roletar":
        logits = 30.0 * torch.tanh(logits / 30.0)
    out = {"logits": logits, "states": None}
    if c["kind"] == "hybrid_prompt":
        out.update(keys=None, values=None)
    return out


@torch.no_grad()
def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "linear":
        packed, whole, x, bias = _linear_inputs(c, seed)
        y = x.to(F64) @ _dense(packed, whole, c["k"], c["n"])
        return y if bias is None else y + bias.to(F64)
    if kind == "dequantize":
        return _dense(*_awq(_generator(seed), c["k"], c["n"], c["group"], DTYPES[c["dtype"]]), c["k"], c["n"])
    if kind == "quantize":
        w = _normal(_generator(seed), c["n"], c["k"], std=0.02).view(c["n"], -1, c["group"]).to(F64)
        return {"words": None, "scales": ((w.amax(dim=2) - w.amin(dim=2)).clamp(min=1e-5) / 15.0).t().contiguous(), "zeros": None}
    return _exact_qwen3(c, seed) if kind.startswith("qwen3") else _exact_hybrid(c, seed)
