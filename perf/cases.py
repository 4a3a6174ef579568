"""The work a user of this package has it do, as cases that can be timed and checked.

Two kinds of work:

* ``decoder``: one whole step of the dense Qwen2 / Qwen3 decoder, from token ids to logits, with the geometries, weight
  formats and batches that bench.py names.  Decode steps run the way the engine runs them, as a captured hipGraph over a
  resident paged KV cache; prefill steps are launched eagerly.
* one mixer or feed-forward of the other registered families, as one step of a layer: ``experts`` (mixture of gated units),
  ``window`` (sliding-window attention beside kept first tokens), ``latent`` (latent attention), ``gla`` (gated linear
  attention), ``mlstm`` (matrix memory with exponential gates), ``ssm`` (Mamba-2).  Sizes are those of bench.py
  --arch-compare.  Prompts are launched eagerly, single-token steps are a captured hipGraph, as in the engine.

Weights, inputs, caches and states are drawn from the seed; ``exact`` computes the same step in float64."""

import math
import random
import zlib

import torch

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
BLOCK = 256                                     # tokens per cache page, the engine's default
FORMATS = {"dense": None, "int8": "w8a16", "int4": "w4a16"}


def listed():
    return [
        # one user, one token at a time: latency and launch count are everything
        dict(name="decoder_b1", kind="decoder", model="qwen2-0.5b", weights="dense", dtype="fp16", phase="decode",
             requests=1, tokens=128, ragged=False, layers=24),
        # the headline: a serving batch of a small model with 4-bit weights at 1k context
        dict(name="decoder_int4_b128", kind="decoder", model="qwen2-0.5b", weights="int4", dtype="bf16", phase="decode",
             requests=128, tokens=1024, ragged=False, layers=24),
        # the same batch on a model whose weights and cache do not fit any on-chip memory
        dict(name="decoder_7b_int4_b128", kind="decoder", model="qwen2-7b", weights="int4", dtype="bf16", phase="decode",
             requests=128, tokens=1024, ragged=True, layers=28),
        # the prompts of the reference's own benchmark: 128 requests of about a hundred tokens in one step
        dict(name="decoder_prefill", kind="decoder", model="qwen3-0.6b", weights="dense", dtype="bf16", phase="prefill",
             requests=128, tokens=128, ragged=True, layers=28),
        # a mixture layer over a prefill step, and over a decode batch of 64
        dict(name="experts_prefill", kind="experts", dtype="bf16", phase="prefill", requests=8, tokens=2048, ragged=False,
             width=2048, experts=16, top=2, ff=3072),
        dict(name="experts_decode", kind="experts", dtype="bf16", phase="decode", requests=64, tokens=256, ragged=False,
             width=1024, experts=16, top=2, ff=1536),
        # windowed attention over long prompts
        dict(name="window_prefill", kind="window", dtype="bf16", phase="prefill", requests=8, tokens=2048, ragged=False,
             width=2048, dim=128, group=2, window=512, keep=16),
        # latent attention over long prompts, and for one new token of each of a few requests with 2k of context
        dict(name="latent_prefill", kind="latent", dtype="bf16", phase="prefill", requests=8, tokens=2048, ragged=True,
             width=2048, window=0),
        dict(name="latent_decode", kind="latent", dtype="bf16", phase="decode", requests=8, tokens=2048, ragged=True,
             width=2048, window=0),
        # the recurrent mixers over prompts: long ones, many short ones, and one in true fp32
        dict(name="gla_prefill", kind="gla", dtype="bf16", phase="prefill", requests=8, tokens=2048, ragged=False,
             width=2048, dim=64, vdim=128),
        dict(name="mlstm_prefill", kind="mlstm", dtype="bf16", phase="prefill", requests=64, tokens=256, ragged=True,
             width=1024, dim=64, vdim=128),
        dict(name="ssm_prefill_fp32", kind="ssm", dtype="fp32", phase="prefill", requests=4, tokens=1024, ragged=True,
             width=1024, dim=64, state=128),
    ]


def draw(rng):
    """One more case: any kind, decode or prefill, batches and lengths over their logarithm, ragged more often than not."""
    def log(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))
    phase = rng.choice(("prefill", "prefill", "decode"))
    kind = rng.choice(("decoder", "experts", "window", "latent", "gla", "mlstm", "ssm"))
    ragged = rng.random() < 0.7
    if kind == "decoder":
        phase = rng.choice(("prefill", "decode"))
        model = rng.choice(("qwen2-0.5b", "qwen3-0.6b"))
        weights = rng.choice(("dense", "int8", "int4"))
        case = dict(kind=kind, model=model, weights=weights, dtype=rng.choice(("bf16", "bf16", "fp16")), phase=phase)
        if phase == "decode":
            return dict(case, requests=log(1, 256), tokens=log(64, 2048), ragged=ragged, layers=24)
        tokens = log(32, 2048)
        return dict(case, requests=max(1, log(256, 8192) // tokens), tokens=tokens, ragged=ragged, layers=24)
    dtype = rng.choice(("bf16", "bf16", "bf16", "fp32"))
    width = rng.choice((512, 1024, 1024, 1536, 2048) if dtype == "bf16" else (512, 1024))
    case = dict(kind=kind, dtype=dtype, phase=phase, ragged=ragged, width=width)
    if phase == "decode":
        case.update(requests=log(1, 128), tokens=log(64, 4096))
    else:
        tokens = log(64, 4096 if dtype == "bf16" else 1024)
        case.update(requests=max(1, log(512, 16384 if dtype == "bf16" else 4096) // tokens), tokens=tokens)
    if kind == "experts":
        case.update(experts=rng.choice((8, 16, 32)), top=rng.choice((1, 2, 3)), ff=width * rng.choice((2, 3)) // 2)
    elif kind == "window":
        case.update(dim=rng.choice((64, 128)), group=rng.choice((1, 2, 4)), window=rng.choice((0, 128, 512, 700)),
                    keep=rng.choice((0, 4, 16)))
    elif kind == "latent":
        case.update(window=rng.choice((0, 512)))
    elif kind in ("gla", "mlstm"):
        case.update(dim=rng.choice((64, 128)) if kind == "mlstm" else rng.choice((32, 64)), vdim=rng.choice((64, 128)))
    else:
        case.update(dim=64, state=rng.choice((64, 128)))
    return case


# ------------------------------------------------------------------------------------------------ shared parts
def normal(seed, name, shape, std=1.0, dtype=torch.float32):
    """N(0, std^2) on the GPU from a stream of its own per (seed, name)."""
    gen = torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + zlib.crc32(name.encode())) % (1 << 62))
    return (torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * std).to(dtype)


def lengths(case):
    """Per request the tokens it has in the end: all alike, or between a half and all of ``tokens``."""
    if not case["ragged"]:
        return [case["tokens"]] * case["requests"]
    rng = random.Random(case["requests"] * 7919 + case["tokens"])
    low = 100 if case["kind"] == "decoder" and case["tokens"] == 128 else max(1, case["tokens"] // 2)
    return [rng.randint(low, case["tokens"]) for _ in range(case["requests"])]


def int32(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


class Step:
    """The integers of one step: every request's pages (dealt in random order), the tokens it brings and where they go."""

    def __init__(self, case, seed):
        self.lens = lengths(case)
        decode = case["phase"] == "decode"
        self.new = [1] * len(self.lens) if decode else self.lens
        self.past = [n - m for n, m in zip(self.lens, self.new)]
        pages = [-(-n // BLOCK) for n in self.lens]
        self.pages = sum(pages) + 1
        order = list(range(self.pages))
        random.Random(seed).shuffle(order)
        self.tables = []
        for n in pages:
            self.tables.append([order.pop() for _ in range(n)])
        width = max(pages)
        self.cu = [0]
        for m in self.new:
            self.cu.append(self.cu[-1] + m)
        self.total = self.cu[-1]
        self.positions = [p + i for p, m in zip(self.past, self.new) for i in range(m)]
        self.slots = [t[(p + i) // BLOCK] * BLOCK + (p + i) % BLOCK
                      for t, p, m in zip(self.tables, self.past, self.new) for i in range(m)]
        self.context = [0]
        for n in self.lens:
            self.context.append(self.context[-1] + -(-n // BLOCK) * BLOCK)
        self.t_positions = torch.tensor(self.positions, dtype=torch.int64, device="cuda")
        self.t_slots, self.t_cu = int32(self.slots), int32(self.cu)
        self.t_tables = int32([t + [0] * (width - len(t)) for t in self.tables])
        self.t_past, self.t_lens = int32(self.past), int32(self.lens)
        self.t_states = int32(list(range(len(self.lens))))
        self.t_owner = int32([i for i, m in enumerate(self.new) for _ in range(m)])
        self.t_context = int32(self.context)

    def publish(self, decode):
        from byox_vllm_amd.utils.context import set_context
        extra = {} if decode else dict(cu_context=self.t_context, context_rows=self.context[-1])
        set_context(True, cu_seqlens_q=self.t_cu, max_seqlen_q=max(self.new), slot_mapping=self.t_slots,
                    block_tables=self.t_tables, past_lens=self.t_past, state_slots=self.t_states,
                    seq_of_token=self.t_owner, **extra)


def captured(launch):
    """``launch`` once eagerly (it sizes its workspaces), then as a graph -> (graph, its outputs)."""
    launch()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = launch()
    return graph, out


def prepare(case, seed):
    with torch.no_grad():
        state = (prepare_decoder if case["kind"] == "decoder" else prepare_layer)(case, seed)
        if case["phase"] == "decode":
            with torch.inference_mode():
                state["graph"], state["out"] = captured(state["launch"])
            for buffer, start in state["fresh"]:         # the pass that sized the workspaces must not count as a step
                buffer.copy_(start)
        state["fresh"] = None
    return state


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    with torch.inference_mode():
        return state["launch"]()


# ------------------------------------------------------------------------------------------------ dense decoder
def geometry(case):
    from byox_vllm_amd.config import qwen2_config
    return qwen2_config(case["model"], dtype=DTYPES[case["dtype"]], num_hidden_layers=case["layers"],
                        max_position_embeddings=8192)


# hidden, intermediate, heads, kv heads, head size, vocabulary, tied head, Qwen2's biases (else Qwen3's head norms)
SHAPES = {"qwen2-0.5b": (896, 4864, 14, 2, 64, 151936, True, True),
          "qwen2-7b": (3584, 18944, 28, 4, 128, 152064, False, True),
          "qwen3-0.6b": (1024, 3072, 16, 8, 128, 151936, True, False)}


def decoder_weights(case, seed, layer):
    """The tensors of one decoder layer under their packed checkpoint names (without the prefix)."""
    hidden, inter, h, hkv, d, _, _, biased = SHAPES[case["model"]]
    dt, at = DTYPES[case["dtype"]], f"{layer}."

    def mat(name, n, k, factor=1.0):
        return normal(seed, at + name, (n, k), 0.6 * factor * k ** -0.5, dt)
    into = (2 * case["layers"]) ** -0.5                 # what a layer adds to the residual is small beside it
    w = {"self_attn.qkv_proj.weight": mat("qkv", (h + 2 * hkv) * d, hidden),
         "self_attn.o_proj.weight": mat("o", hidden, h * d, into),
         "mlp.gate_up_proj.weight": mat("gu", 2 * inter, hidden), "mlp.down_proj.weight": mat("down", hidden, inter, into),
         "input_layernorm.weight": 1 + normal(seed, at + "n1", hidden, 0.1, dt),
         "post_attention_layernorm.weight": 1 + normal(seed, at + "n2", hidden, 0.1, dt)}
    if biased:
        w["self_attn.qkv_proj.bias"] = normal(seed, at + "b", (h + 2 * hkv) * d, 0.02, dt)
    else:
        w["self_attn.q_norm.weight"] = 1 + normal(seed, at + "qn", d, 0.1, dt)
        w["self_attn.k_norm.weight"] = 1 + normal(seed, at + "kn", d, 0.1, dt)
    return w


def decoder_ends(case, seed):
    hidden, _, _, _, _, vocab, tied, _ = SHAPES[case["model"]]
    dt = DTYPES[case["dtype"]]
    ends = {"model.embed_tokens.weight": normal(seed, "embed", (vocab, hidden), 0.25, dt),
            "model.norm.weight": 1 + normal(seed, "norm", hidden, 0.1, dt)}
    if not tied:
        ends["lm_head.weight"] = normal(seed, "head", (vocab, hidden), 0.02, dt)
    return ends


def decoder_ids(case, seed, total):
    gen = torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 62))
    return torch.randint(0, 10000, (total,), generator=gen, device="cuda")


def decoder_cache(case, seed, step):
    """[2, layers, pages, block, kv heads, head size]: what earlier steps left there, or nothing yet."""
    _, _, _, hkv, d, _, _, _ = SHAPES[case["model"]]
    kv = torch.zeros(2, case["layers"], step.pages, BLOCK, hkv, d, dtype=DTYPES[case["dtype"]], device="cuda")
    if case["phase"] == "decode":
        for i in range(case["layers"]):
            kv[:, i] = normal(seed, f"kv{i}", kv[:, i].shape, 1.0, kv.dtype)
    return kv


def prepare_decoder(case, seed):
    from byox_vllm_amd import kernels
    from byox_vllm_amd.models.registry import model_class
    from byox_vllm_amd.utils.context import reset_context, set_context
    from byox_vllm_amd.utils.loader import load_state_dict_packed
    cfg, step = geometry(case), Step(case, seed)
    default = torch.get_default_dtype()
    torch.set_default_dtype(cfg.dtype)
    try:
        with torch.device("cuda"):
            model = model_class(cfg)(cfg)
    finally:
        torch.set_default_dtype(default)
    load_state_dict_packed(model, decoder_ends(case, seed), cfg)
    for i in range(case["layers"]):
        load_state_dict_packed(model, {f"model.layers.{i}.{k}": w for k, w in decoder_weights(case, seed, i).items()}, cfg)
    model.finalize(FORMATS[case["weights"]])
    kv = decoder_cache(case, seed, step)
    rows, decode = len(step.lens), case["phase"] == "decode"
    for i, layer in enumerate(model.model.layers):
        layer.self_attn.attn.k_cache, layer.self_attn.attn.v_cache = kv[0, i], kv[1, i]
        layer.self_attn.attn.decode_splits = kernels.pick_decode_splits(rows, cfg.num_key_value_heads, max(step.lens))
    ids = decoder_ids(case, seed, step.total)
    policy = int(decode and 64 <= rows <= 256)       # the engine's own choice for the stores between launches

    def launch():
        with kernels.result_policy(policy):
            if decode:
                set_context(False, slot_mapping=step.t_slots, context_lens=step.t_lens, block_tables=step.t_tables)
            else:
                set_context(True, step.t_cu, step.t_cu, max(step.new), max(step.new), step.t_slots)
            logits = model.compute_logits(model(ids, step.t_positions))
            reset_context()
        return {"logits": logits, "cache": kv}
    return {"launch": launch, "fresh": []}


def quantised(w, weights):
    """The numbers that 8- or 4-bit weights stand for: groups of 128 along a row share a scale in the model dtype."""
    if weights == "dense":
        return w.double()
    top = 127 if weights == "int8" else 7
    low = -127 if weights == "int8" else -8
    g = w.float().view(w.size(0), -1, 128)
    s = (g.abs().amax(-1) / top).clamp_min(1e-8).to(w.dtype).float().unsqueeze(-1)
    return (torch.clamp(torch.round(g / s), low, top).double() * s.double()).view(w.shape)


def rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def rotated(x, positions, freq):
    """x [T, heads, >= 2 len(freq)]: number i of the first 2 len(freq) turns with number i + len(freq)."""
    n = freq.numel()
    angle = (positions.double()[:, None] * freq.double())[:, None]
    a, b = x[..., :n], x[..., n:2 * n]
    return torch.cat([a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin(), x[..., 2 * n:]], -1)


def frequencies(dims, base):
    return (1.0 / (base ** (torch.arange(0, dims, 2, dtype=torch.float32, device="cuda") / dims)))


def attend(q, k, v, scale, past, window=0, keep=0):
    """q [m, H, d] of the last m of n tokens; k, v [n, G, *] -> [m, H, dv]; in slices of heads to bound memory."""
    m, heads, _ = q.shape
    n, groups = k.shape[:2]
    i, j = torch.arange(past, past + m, device="cuda")[:, None], torch.arange(n, device="cuda")[None]
    seen = j <= i
    if window:
        seen &= (i - j < window) | (j < keep)
    out = torch.empty(m, heads, v.size(-1), dtype=q.dtype, device="cuda")
    for h in range(heads):
        g = h * groups // heads
        s = (q[:, h] @ k[:, g].t().contiguous()) * scale
        out[:, h] = torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ v[:, g]
    return out


def exact_decoder(case, seed):
    hidden, inter, h, hkv, d, _, tied, biased = SHAPES[case["model"]]
    step = Step(case, seed)
    ends, fmt, eps = decoder_ends(case, seed), case["weights"], 1e-6
    kv = decoder_cache(case, seed, step).double()
    freq = frequencies(d, 1000000.0)
    x = ends["model.embed_tokens.weight"][decoder_ids(case, seed, step.total)].double()
    slots = step.t_slots.long()
    rows = [torch.tensor([t[p // BLOCK] * BLOCK + p % BLOCK for p in range(n)], device="cuda")
            for t, n in zip(step.tables, step.lens)]
    width = max(step.lens)
    padded = torch.stack([torch.cat([r, r.new_zeros(width - r.numel())]) for r in rows])
    hidden_keys = (torch.arange(width, device="cuda")[None] >= step.t_lens[:, None])[:, None, None]
    for layer in range(case["layers"]):
        w = decoder_weights(case, seed, layer)
        y = rms(x, eps) * w["input_layernorm.weight"].double()
        qkv = y @ quantised(w["self_attn.qkv_proj.weight"], fmt).t()
        if biased:
            qkv = qkv + w["self_attn.qkv_proj.bias"].double()
        q, k, v = (t.view(step.total, -1, d) for t in qkv.split([h * d, hkv * d, hkv * d], -1))
        if not biased:
            q, k = (rms(t, eps) * w[f"self_attn.{n}_norm.weight"].double() for t, n in ((q, "q"), (k, "k")))
        q, k = rotated(q, step.t_positions, freq), rotated(k, step.t_positions, freq)
        keys, values = kv[0, layer].view(-1, hkv, d), kv[1, layer].view(-1, hkv, d)
        keys[slots], values[slots] = k, v
        if case["phase"] == "decode":
            kk = keys[padded].permute(0, 2, 3, 1).contiguous()          # [B, kv heads, d, n]
            vv = values[padded].transpose(1, 2).contiguous()
            s = torch.matmul(q.view(-1, hkv, h // hkv, d).contiguous(), kk) * d ** -0.5
            o = torch.matmul(torch.softmax(s.masked_fill(hidden_keys, -math.inf), -1), vv).reshape(step.total, -1)
        else:
            o = torch.cat([attend(q[a:b], k[a:b], v[a:b], d ** -0.5, 0) for a, b in zip(step.cu, step.cu[1:])])
        x = x + o.reshape(step.total, -1) @ quantised(w["self_attn.o_proj.weight"], fmt).t()
        y = rms(x, eps) * w["post_attention_layernorm.weight"].double()
        gate, up = (y @ quantised(w["mlp.gate_up_proj.weight"], fmt).t()).chunk(2, -1)
        x = x + (torch.nn.functional.silu(gate) * up) @ quantised(w["mlp.down_proj.weight"], fmt).t()
    x = x[step.t_cu[1:].long() - 1]
    head = ends["model.embed_tokens.weight" if tied else "lm_head.weight"]
    return {"logits": (rms(x, eps) * ends["model.norm.weight"].double()) @ head.double().t(), "cache": kv}


def work_decoder(case):
    hidden, inter, h, hkv, d, vocab, _, _ = SHAPES[case["model"]]
    lens, item = lengths(case), 2
    new = len(lens) if case["phase"] == "decode" else sum(lens)
    matrices = case["layers"] * hidden * ((h + 2 * hkv) * d + h * d + 3 * inter)
    per_weight = {"dense": 2, "int8": 1 + 2 / 128, "int4": 0.5 + 2 / 128}[case["weights"]]
    kv = case["layers"] * 2 * hkv * d * item
    read = sum(lens) if case["phase"] == "decode" else 0
    pairs = sum(lens) if case["phase"] == "decode" else sum(n * (n + 1) // 2 for n in lens)
    return {"bytes": matrices * per_weight + vocab * hidden * item + kv * (read + new) + len(lens) * vocab * item,
            "flops": 2 * matrices * new + 2 * len(lens) * vocab * hidden + case["layers"] * 4 * h * d * pairs}


# ------------------------------------------------------------------------------------------------ single layers
LATENT = dict(dim=96, rot=32, vdim=128)          # numbers per head of latent attention: plain, rotated, values


def sizes(case):
    """Heads and ranks that follow from a layer's width."""
    w = case["width"]
    heads = w // 128
    if case["kind"] == "ssm":
        heads = 2 * w // case["dim"]
    elif case["kind"] == "window":
        heads = w // case["dim"]
    return dict(heads=heads, kv_heads=max(1, heads // case["group"]) if case["kind"] == "window" else heads,
                kv_rank=w // 4, q_rank=w // 2, decay_rank=32)


def layer_weights(case, seed):
    """Parameter name -> tensor; matrices keep the scale of their input, gates and decays lie where trained ones do."""
    z, w, kind, dt = sizes(case), case["width"], case["kind"], DTYPES[case["dtype"]]
    H = z["heads"]

    def mat(name, *shape):
        return normal(seed, name, shape, shape[-1] ** -0.5, dt)

    def vec(name, n, std, mean=0.0, dtype=dt):
        return (mean + normal(seed, name, n, std)).to(dtype)
    if kind == "experts":
        return {"router.weight": mat("r", case["experts"], w), "gate_up": mat("gu", case["experts"], 2 * case["ff"], w),
                "down": mat("d", case["experts"], w, case["ff"])}
    if kind == "window":
        d, G = case["dim"], z["kv_heads"]
        return {"inp.weight": mat("i", (H + 2 * G) * d + H, w), "o.weight": mat("o", w, H * d)}
    if kind == "latent":
        R, r, d, dv = z["kv_rank"], LATENT["rot"], LATENT["dim"], LATENT["vdim"]
        return {"down.weight": mat("dn", z["q_rank"] + R + r + H, w), "uq.weight": mat("uq", H * (d + r), z["q_rank"]),
                "uk_t": normal(seed, "uk", (H, R, d), R ** -0.5, dt), "uv.weight": mat("uv", H * dv, R),
                "dq_norm": vec("dqn", z["q_rank"], 0.1, 1.0), "dkv_norm": vec("dkn", R, 0.1, 1.0),
                "o.weight": mat("o", w, H * dv)}
    if kind == "gla":
        d, dv = case["dim"], case["vdim"]
        return {"qkvg.weight": mat("p", 2 * H * (d + dv), w), "a1.weight": mat("a1", z["decay_rank"], w),
                "a2.weight": mat("a2", H * d, z["decay_rank"]), "a2.bias": vec("a2b", H * d, 1.0),
                "norm": vec("n", dv, 0.1, 1.0), "o.weight": mat("o", w, H * dv)}
    if kind == "mlstm":
        d, dv = case["dim"], case["vdim"]
        bias = torch.zeros(2 * H * (d + dv) + 2 * H, dtype=dt, device="cuda")
        bias[-2 * H:-H] = vec("bi", H, 0.5, -1.0)
        bias[-H:] = vec("bf", H, 1.0, 4.0)
        return {"inp.weight": mat("p", bias.numel(), w), "inp.bias": bias, "norm": vec("n", H * dv, 0.1, 1.0),
                "o.weight": mat("o", w, H * dv)}
    d, n = case["dim"], case["state"]
    dt_at = torch.exp(normal(seed, "dt", H, 1.0) - 4.0)             # steps around 0.02
    return {"inp.weight": mat("p", 2 * H * d + 2 * n + H, w), "conv.weight": normal(seed, "cw", (H * d + 2 * n, 4), 0.5, dt),
            "conv.bias": vec("cb", H * d + 2 * n, 0.1), "dt_bias": torch.log(torch.expm1(dt_at)).to(dt),
            "A_log": vec("A", H, 0.7, 1.0), "D": vec("D", H, 0.1, 1.0), "norm": vec("n", H * d, 0.1, 1.0),
            "o.weight": mat("o", w, H * d)}


def layer_module(case):
    z, w, kind = sizes(case), case["width"], case["kind"]
    if kind == "experts":
        from byox_vllm_amd.layers.moe import MixtureOfExperts
        return MixtureOfExperts(w, case["experts"], case["top"], case["ff"])
    if kind == "window":
        from byox_vllm_amd.layers.sliding_attention import SlidingAttention
        return SlidingAttention(w, z["heads"], z["kv_heads"], case["dim"], case["dim"], case["dim"] ** -0.5, case["window"],
                                case["keep"], rot_dims=32, rot_base=10000.0)
    if kind == "latent":
        from byox_vllm_amd.layers.latent_attention import LatentAttention
        return LatentAttention(w, z["heads"], LATENT["dim"], LATENT["rot"], LATENT["vdim"], z["q_rank"], z["kv_rank"],
                               128 ** -0.5, case["window"], LATENT["rot"], 10000.0, None, 1e-5)
    if kind == "gla":
        from byox_vllm_amd.layers.gla import GatedLinearAttention
        return GatedLinearAttention(w, z["heads"], case["dim"], case["vdim"], z["decay_rank"], 16.0, 1e-5)
    if kind == "mlstm":
        from byox_vllm_amd.layers.matrix_memory import MLSTM
        return MLSTM(w, z["heads"], case["dim"], case["vdim"], 15.0, 1e-5)
    from byox_vllm_amd.layers.mamba2 import Mamba2Mixer
    return Mamba2Mixer(w, z["heads"], case["dim"], case["state"], 1, 4, 1, 1e-5)


def cache_width(case):
    z = sizes(case)
    if case["kind"] == "window":
        return z["kv_heads"] * 2 * case["dim"]
    return z["kv_rank"] + LATENT["rot"] if case["kind"] == "latent" else 0


def layer_cache(case, seed, step):
    shape = (step.pages * BLOCK, cache_width(case))
    if case["phase"] == "decode":
        return normal(seed, "cache", shape, 1.0, DTYPES[case["dtype"]])
    return torch.zeros(shape, dtype=DTYPES[case["dtype"]], device="cuda")


def layer_memory(case, seed):
    """What the requests' earlier tokens left in the recurrent state: matrix [B, H, dim, vdim], and by kind the normaliser
    [B, H, dim] and running maximum [B, H], or the convolution's last inputs [B, 3, channels]."""
    z, B, kind = sizes(case), case["requests"], case["kind"]
    H = z["heads"]
    if kind == "ssm":
        return {"S": normal(seed, "S", (B, H, case["state"], case["dim"]), 0.3),
                "conv": normal(seed, "C", (B, 3, H * case["dim"] + 2 * case["state"]))}
    S = {"S": normal(seed, "S", (B, H, case["dim"], case["vdim"]), 0.5)}
    if kind == "mlstm":
        S.update(n=normal(seed, "n", (B, H, case["dim"]), 0.5), m=normal(seed, "m", (B, H), 0.5).abs())
    return S


def packed_memory(case, memory):
    """The mLSTM's slot: the matrix, then normaliser and maximum once per 64 value columns."""
    S, n, m = memory["S"], memory["n"], memory["m"]
    slices = -(-case["vdim"] // 64)
    parts = [S.reshape(*S.shape[:2], -1)] + [n, m[..., None]] * slices
    return torch.cat(parts, -1).contiguous()


def prepare_layer(case, seed):
    from byox_vllm_amd.utils.context import reset_context
    kind, decode, dt = case["kind"], case["phase"] == "decode", DTYPES[case["dtype"]]
    step = Step(case, seed)
    default = torch.get_default_dtype()
    torch.set_default_dtype(dt)
    try:
        with torch.device("cuda"):
            layer = layer_module(case)
    finally:
        torch.set_default_dtype(default)
    for name, tensor in layer_weights(case, seed).items():
        layer.get_parameter(name).data.copy_(tensor)
    h = normal(seed, "h", (step.total, case["width"]), 1.0, dt)
    state, arguments = [], (h,)
    if kind in ("window", "latent"):
        arguments = (h, step.t_positions)
        holder = layer
        if kind == "window":
            holder = layer.runs[layer.add_run()]
        holder.cache, holder.block_size = layer_cache(case, seed, step), BLOCK
        state = [holder.cache]
    elif kind in ("gla", "mlstm", "ssm"):
        holders = [layer.runs[0]] if kind == "mlstm" else [layer]
        if kind == "ssm":
            holders.append(layer.conv)
        for holder in holders:
            holder.state = torch.zeros(case["requests"], *holder.state_spec()["shape"], device="cuda")
        if decode:
            memory = layer_memory(case, seed)
            if kind == "mlstm":
                holders[0].state.copy_(packed_memory(case, memory))
            else:
                holders[0].state.copy_(memory["S"])
            if kind == "ssm":
                holders[1].state.copy_(memory["conv"])
        state = [holder.state for holder in holders]

    def launch():
        step.publish(decode)
        y = layer(*arguments)
        reset_context()
        return {"y": y, "state": state}
    return {"launch": launch, "fresh": [(s, s.clone()) for s in state] if decode else []}


# -- the same layers in float64
def exact_experts(case, w, h, step, seed):
    logits = h @ w["router.weight"].t()
    best, chosen = logits.topk(case["top"], -1)
    weight, y = torch.softmax(best, -1), torch.zeros_like(h)
    for e in range(case["experts"]):
        token, choice = (chosen == e).nonzero(as_tuple=True)
        if token.numel():
            gate, up = (h[token] @ w["gate_up"][e].double().t()).chunk(2, -1)
            y.index_add_(0, token, (torch.nn.functional.silu(gate) * up) @ w["down"][e].double().t()
                         * weight[token, choice][:, None])
    return {"y": y, "state": []}


def cached_rows(step, cache, b):
    """The cache rows of request b in order of position."""
    return torch.cat([cache[t * BLOCK:(t + 1) * BLOCK] for t in step.tables[b]])[:step.lens[b]]


def exact_window(case, w, h, step, seed):
    z, d = sizes(case), case["dim"]
    H, G = z["heads"], z["kv_heads"]
    q, k, v, g = (h @ w["inp.weight"].t()).split([H * d, G * d, G * d, H], -1)
    freq = frequencies(32, 10000.0)
    q, k = (rotated(t.view(step.total, -1, d), step.t_positions, freq) for t in (q, k))
    cache = layer_cache(case, seed, step).double()
    cache[step.t_slots.long()] = torch.cat([k.reshape(step.total, -1), v], -1)
    out = []
    for b, (lo, hi) in enumerate(zip(step.cu, step.cu[1:])):
        kk, vv = cached_rows(step, cache, b).split(G * d, -1)
        out.append(attend(q[lo:hi], kk.reshape(-1, G, d), vv.reshape(-1, G, d), d ** -0.5, step.past[b], case["window"],
                          case["keep"]))
    y = torch.cat(out) * torch.sigmoid(g)[..., None]
    return {"y": y.reshape(step.total, -1) @ w["o.weight"].t(), "state": [cache]}


def exact_latent(case, w, h, step, seed):
    z, H = sizes(case), sizes(case)["heads"]
    R, r, d, dv = z["kv_rank"], LATENT["rot"], LATENT["dim"], LATENT["vdim"]
    dq, dc, dr, g = (h @ w["down.weight"].t()).split([z["q_rank"], R, r, H], -1)
    freq = frequencies(r, 10000.0)
    q = ((rms(dq, 1e-5) * w["dq_norm"]) @ w["uq.weight"].t()).view(step.total, H, d + r)
    q = torch.cat([q[..., :d], rotated(q[..., d:], step.t_positions, freq)], -1)
    cache = layer_cache(case, seed, step).double()
    cache[step.t_slots.long()] = torch.cat([rms(dc, 1e-5) * w["dkv_norm"],
                                            rotated(dr[:, None], step.t_positions, freq)[:, 0]], -1)
    out = []
    for b, (lo, hi) in enumerate(zip(step.cu, step.cu[1:])):
        c, turned = cached_rows(step, cache, b).split([R, r], -1)
        k = torch.cat([torch.matmul(c[None], w["uk_t"]), turned[None].expand(H, -1, -1)], -1).transpose(0, 1)
        v = (c @ w["uv.weight"].t()).view(-1, H, dv)
        out.append(attend(q[lo:hi], k, v, 128 ** -0.5, step.past[b], case["window"]))
    y = torch.cat(out) * torch.sigmoid(g)[..., None]
    return {"y": y.reshape(step.total, -1) @ w["o.weight"].t(), "state": [cache]}


def walk(step, width, advance):
    """``advance(live, rows)`` -> results [live, *] for the next token of every request that still has one; the requests
    are taken longest first, so the live ones are always the first."""
    order = sorted(range(len(step.new)), key=lambda b: -step.new[b])
    out = torch.zeros(step.total, width, dtype=torch.float64, device="cuda")
    for t in range(max(step.new)):
        live = [b for b in order if step.new[b] > t]
        rows = torch.tensor([step.cu[b] + t for b in live], device="cuda")
        out[rows] = advance(len(live), rows)
    return out, torch.tensor(order, device="cuda")


def start_memory(case, seed, step):
    """The requests' states in the order of ``walk``; zeros where the step starts them."""
    order = torch.tensor(sorted(range(len(step.new)), key=lambda b: -step.new[b]), device="cuda")
    return {k: (v.double() if case["phase"] == "decode" else torch.zeros_like(v, dtype=torch.float64))[order]
            for k, v in layer_memory(case, seed).items()}


def back(v, order):
    """From the order of ``walk`` to the requests' own."""
    out = torch.empty_like(v)
    out[order] = v
    return out


def exact_gla(case, w, h, step, seed):
    H, d, dv = sizes(case)["heads"], case["dim"], case["vdim"]
    q, k, v, g = (h @ w["qkvg.weight"].t()).split([H * d, H * d, H * dv, H * dv], -1)
    decay = torch.sigmoid((h @ w["a1.weight"].t()) @ w["a2.weight"].t() + w["a2.bias"]) ** (1 / 16.0)
    q, k, decay, v = (q.view(-1, H, d) * d ** -0.5, k.view(-1, H, d), decay.view(-1, H, d), v.view(-1, H, dv))
    S = start_memory(case, seed, step)["S"]

    def advance(live, rows):
        S[:live] = S[:live] * decay[rows][..., None] + k[rows][..., None] * v[rows][:, :, None]
        return torch.matmul(q[rows][:, :, None], S[:live]).reshape(live, -1)
    o, order = walk(step, H * dv, advance)
    y = (rms(o.view(-1, H, dv), 1e-5) * w["norm"]).reshape(step.total, -1) * torch.nn.functional.silu(g)
    return {"y": y @ w["o.weight"].t(), "state": [back(S, order)]}


def exact_mlstm(case, w, h, step, seed):
    H, d, dv = sizes(case)["heads"], case["dim"], case["vdim"]
    proj = h @ w["inp.weight"].t() + w["inp.bias"]
    q, k, v, g, i, f = proj.split([H * d, H * d, H * dv, H * dv, H, H], -1)
    i, f = 15.0 * torch.tanh(i / 15.0), torch.nn.functional.logsigmoid(15.0 * torch.tanh(f / 15.0))
    q, k, v = q.view(-1, H, d) * d ** -0.5, k.view(-1, H, d), v.view(-1, H, dv)
    M = start_memory(case, seed, step)
    S, n, m = M["S"], M["n"], M["m"]

    def advance(live, rows):
        top = torch.maximum(f[rows] + m[:live], i[rows])
        keep, take = torch.exp(f[rows] + m[:live] - top), torch.exp(i[rows] - top)
        m[:live] = top
        S[:live] = S[:live] * keep[..., None, None] + (take[..., None] * k[rows])[..., None] * v[rows][:, :, None]
        n[:live] = n[:live] * keep[..., None] + take[..., None] * k[rows]
        below = torch.maximum((n[:live] * q[rows]).sum(-1).abs(), torch.exp(-top)) + 1e-6
        return (torch.matmul(q[rows][:, :, None], S[:live])[:, :, 0] / below[..., None]).reshape(live, -1)
    o, order = walk(step, H * dv, advance)
    y = rms(o.view(-1, H, dv), 1e-5).reshape(step.total, -1) * w["norm"] * torch.sigmoid(g)
    state = packed_memory(case, {"S": back(S, order), "n": back(n, order), "m": back(m, order)})
    return {"y": y @ w["o.weight"].t(), "state": [state]}


def exact_ssm(case, w, h, step, seed):
    H, d, n = sizes(case)["heads"], case["dim"], case["state"]
    z, x, dt = (h @ w["inp.weight"].t()).split([H * d, H * d + 2 * n, H], -1)
    start = start_memory(case, seed, step)
    S, order = start["S"], sorted(range(len(step.new)), key=lambda b: -step.new[b])
    mixed, last = torch.empty_like(x), torch.empty_like(start["conv"])
    for at, b in enumerate(order):
        lo, hi = step.cu[b], step.cu[b + 1]
        rows = torch.cat([start["conv"][at], x[lo:hi]])
        mixed[lo:hi] = sum(rows[j:j + hi - lo] * w["conv.weight"][:, j] for j in range(4)) + w["conv.bias"]
        last[at] = rows[-3:]
    xs, B, C = torch.nn.functional.silu(mixed).split([H * d, n, n], -1)
    xs, dt = xs.view(-1, H, d), torch.nn.functional.softplus(dt + w["dt_bias"])
    keep = torch.exp(-torch.exp(w["A_log"]) * dt)

    def advance(live, rows):
        S[:live] = S[:live] * keep[rows][..., None, None] + B[rows][:, None, :, None] * (dt[rows][..., None] * xs[rows])[:, :, None]
        return torch.matmul(C[rows][:, None, None], S[:live]).reshape(live, -1)
    y, by = walk(step, H * d, advance)
    y = (y.view(-1, H, d) + w["D"][:, None] * xs).reshape(step.total, -1) * torch.nn.functional.silu(z)
    return {"y": (rms(y, 1e-5) * w["norm"]) @ w["o.weight"].t(), "state": [back(S, by), back(last, by)]}


def exact(case, seed):
    if case["kind"] == "decoder":
        return exact_decoder(case, seed)
    step = Step(case, seed)
    w = layer_weights(case, seed)
    if case["kind"] != "experts":
        w = {k: t.double() for k, t in w.items()}
    else:
        w["router.weight"] = w["router.weight"].double()
    h = normal(seed, "h", (step.total, case["width"]), 1.0, DTYPES[case["dtype"]]).double()
    of = {"experts": exact_experts, "window": exact_window, "latent": exact_latent, "gla": exact_gla, "mlstm": exact_mlstm,
          "ssm": exact_ssm}[case["kind"]]
    return of(case, w, h, step, seed)


def work(case):
    """Inputs, weights, states and the cache rows that are seen, each once; results and new rows once; the products and the
    recurrence's own arithmetic."""
    if case["kind"] == "decoder":
        return work_decoder(case)
    lens, z, wd, kind = lengths(case), sizes(case), case["width"], case["kind"]
    decode, item = case["phase"] == "decode", DTYPES[case["dtype"]].itemsize
    T = len(lens) if decode else sum(lens)
    H = z["heads"]
    nbytes = T * wd * (item + 4)                                # input rows, fp32 results
    if kind == "experts":
        unit = 3 * case["ff"] * wd
        hit = case["experts"] * (1 - (1 - case["top"] / case["experts"]) ** T)
        return {"bytes": nbytes + hit * unit * item + case["experts"] * wd * item,
                "flops": 2 * T * (case["top"] * unit + case["experts"] * wd)}
    window = case.get("window", 0)

    def seen(i):                                               # keys that the token at place i sees
        return min(i + 1, window + min(case.get("keep", 0), max(0, i + 1 - window))) if window else i + 1
    if decode:
        pairs = sum(seen(n - 1) for n in lens)
    else:
        pairs = sum(sum(seen(i) for i in range(n)) for n in lens) if window else sum(n * (n + 1) // 2 for n in lens)
    if kind == "window":
        d, G = case["dim"], z["kv_heads"]
        weights = wd * ((H + 2 * G) * d + H) + wd * H * d
        row = cache_width(case) * item
        return {"bytes": nbytes + weights * item + T * row + (pairs * row if decode else 0),
                "flops": 2 * T * weights + 4 * pairs * H * d}
    if kind == "latent":
        R, r, d, dv = z["kv_rank"], LATENT["rot"], LATENT["dim"], LATENT["vdim"]
        weights = wd * (z["q_rank"] + R + r + H) + z["q_rank"] * H * (d + r) + R * H * (d + dv) + wd * H * dv
        row = cache_width(case) * item
        # a decoded token meets the cached latents themselves, a prompt's tokens meet keys and values
        per_pair = 2 * H * (2 * R + r) if decode else 2 * H * (d + r + dv)
        return {"bytes": nbytes + weights * item + T * row + (pairs * row if decode else 0),
                "flops": 2 * T * weights + pairs * per_pair}
    dv, n = (case["dim"], case["state"]) if kind == "ssm" else (case["vdim"], case["dim"])
    inp = {"gla": 2 * H * (n + dv) + z["decay_rank"], "mlstm": 2 * H * (n + dv) + 2 * H, "ssm": 2 * H * dv + 2 * n + H}[kind]
    weights = wd * inp + wd * H * dv + (H * n * z["decay_rank"] if kind == "gla" else 0)
    states = len(lens) * H * n * dv * 4 * (2 if decode else 1)
    return {"bytes": nbytes + weights * item + states, "flops": 2 * T * weights + 4 * T * H * n * dv}


def tolerance(case):
    """A layer rounds its inputs' products to 16 bits once or twice on the way (measured against float64: 2e-3 to 4e-3), a
    whole decoder the result of every launch (1e-2 in bf16, 2e-3 in fp16); fp32 layers differ in the order of their sums
    (up to 3e-6)."""
    if case["kind"] == "decoder":
        return {"rel": 0.03 if case["dtype"] == "bf16" else 6e-3}
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-5}
