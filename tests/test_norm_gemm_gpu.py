"""nv_norm_gemm_* (csrc/norm_gemm.hip): a few rows' residual add and RMSNorm inside the product that reads them, against the same
steps in launches of their own (which have tests against the oracle)."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(autouse=True)
def one_rank(monkeypatch):
    """Layers of one rank and rotation tables of their own, whatever ran before."""
    from byox_vllm_amd.layers import linear
    from byox_vllm_amd.layers.rotary_embedding import get_rope
    monkeypatch.setattr(linear, "_TP_STATE", (0, 1, None))
    monkeypatch.setattr(linear, "_COMM", None)
    get_rope.cache_clear()
    yield
    get_rope.cache_clear()


DT = {"bf16": torch.bfloat16, "fp16": torch.float16}


def inputs(M, K, dt, form):
    """form: the rows alone, rows and residual, or split-K slabs and residual -> (x for the fused call, x as rows, residual)"""
    from byox_vllm_amd import kernels
    res = None if form == "first" else torch.randn(M, K, device=DEV).to(dt)
    if not form.startswith("slabs"):
        x = torch.randn(M, K, device=DEV).to(dt)
        return x, x, res
    n = int(form[5:])
    slabs = torch.randn(n, M, K, device=DEV) * n ** -0.5
    total = slabs[0].clone()
    for z in range(1, n):
        total += slabs[z]
    return kernels.Partials(slabs, n, M, K, None, dt), total.to(dt), res


def normed(rows, res, w):
    from byox_vllm_amd import kernels
    if res is None:
        return kernels.rms_norm(rows, w, 1e-6), rows
    return kernels.add_rms_norm(rows, res, w, 1e-6)


def close(got, want, dt, what):
    # the norms' sums in another order move a normed number over a rounding now and then; products of K of them, rounded
    scale = want.double().pow(2).mean().sqrt()
    off = ((got.double() - want.double()).abs() / torch.maximum(want.double().abs(), scale)).max()
    assert torch.isfinite(got).all() and off < 4 * torch.finfo(dt).eps, f"{what}: off by {off:.3g}"


@pytest.mark.parametrize("name", ["bf16", "fp16"])
@pytest.mark.parametrize("form", ["first", "rows", "slabs1", "slabs3", "slabs11"])
@pytest.mark.parametrize("M,K,inter", [(1, 896, 4864), (1, 128, 8), (3, 1024, 3072), (7, 256, 24), (8, 2048, 520), (16, 1024, 40)])
def test_silu(M, K, inter, form, name):
    from byox_vllm_amd import kernels
    from byox_vllm_amd.layers.quant import LinearWeight, interleave_gate_up
    torch.manual_seed(M + K)
    dt = DT[name]
    x, rows, res = inputs(M, K, dt, form)
    nw = (torch.rand(K, device=DEV) + 0.5).to(dt)
    w = LinearWeight.dense_tiled(interleave_gate_up((torch.randn(2 * inter, K, device=DEV) * K ** -0.5).to(dt)))
    if inter % 16 == 0:
        h, new = normed(rows, res, nw)
        want = kernels.gemm(h, w, silu_mul=True)
    else:
        h, new = normed(rows, res, nw)
        want = kernels.gemm_stream(h, w, silu_mul=True) if w.out_features % 32 == 0 else None
    before = None if res is None else res.clone()
    got, kept = kernels.norm_gemm_silu(x, res, nw, 1e-6, w)
    assert torch.equal(kept, new) and (res is None or torch.equal(res, before))
    if want is None:
        y = (h.double() @ w.logical_dense().double().t()).to(dt).double().view(M, -1, 4)
        want = (torch.nn.functional.silu(y[..., :2]).to(dt).double() * y[..., 2:]).reshape(M, -1).to(dt)
    close(got, want, dt, "silu")


@pytest.mark.parametrize("name", ["bf16", "fp16"])
@pytest.mark.parametrize("form", ["first", "rows", "slabs5"])
@pytest.mark.parametrize("M,K,H,Hkv,D,norms", [(1, 896, 14, 2, 64, False), (1, 1024, 16, 8, 128, True), (5, 896, 14, 2, 64, False),
                                               (8, 256, 3, 1, 64, True), (7, 2048, 2, 1, 128, False), (16, 1024, 1, 1, 128, True)])
def test_rope_kv_store(M, K, H, Hkv, D, norms, form, name):
    from byox_vllm_amd import kernels
    from byox_vllm_amd.layers.quant import LinearWeight
    torch.manual_seed(M + K + H)
    dt, N = DT[name], (H + 2 * Hkv) * D
    x, rows, res = inputs(M, K, dt, form)
    nw = (torch.rand(K, device=DEV) + 0.5).to(dt)
    w = LinearWeight.dense_tiled((torch.randn(N, K, device=DEV) * K ** -0.5).to(dt))
    bias = None if norms else torch.randn(N, device=DEV).to(dt)
    qn, kn = ((torch.rand(D, device=DEV) + 0.5).to(dt) if norms else None for _ in range(2))
    pos = torch.randint(0, 100, (M,), device=DEV)
    angle = torch.rand(100, D // 2, device=DEV) * 6.28
    cos_sin = torch.cat([angle.cos(), angle.sin()], -1).contiguous()
    slots = torch.randperm(3 * 16, device=DEV)[:M].int()
    if M > 1:
        slots[M // 2] = -1
    caches = [torch.zeros(3, 16, Hkv, D, dtype=dt, device=DEV) for _ in range(4)]
    args = dict(slot_mapping=slots, q_norm_w=qn, k_norm_w=kn, eps=1e-6)
    got, kept = kernels.norm_gemm_rope_kv_store(x, res, nw, 1e-6, w, bias, pos, cos_sin, H, Hkv, D, k_cache=caches[0], v_cache=caches[1],
                                                **args)
    h, new = normed(rows, res, nw)
    want = kernels.rope_kv_store(kernels.gemm(h, w, bias), pos, cos_sin, H, Hkv, D, k_cache=caches[2], v_cache=caches[3], **args)
    assert torch.equal(kept, new)
    for a, b, what in ((got, want, "q/k/v"), (caches[0], caches[2], "keys"), (caches[1], caches[3], "values")):
        close(a, b, dt, what)


def norm64(x, res, w, eps, dt):
    """RMSNorm of x + residual in float64 with the roundings the storage type makes: the sum, the normed row, its product with the weight."""
    total = x.double() if res is None else (x.double() + res.double()).to(dt).double()
    normed = (total * torch.rsqrt((total * total).mean(-1, keepdim=True) + eps)).to(dt).double()
    return (normed * w.double()).to(dt).double()


@pytest.mark.parametrize("name", ["bf16", "fp16"])
@pytest.mark.parametrize("form", ["first", "rows", "slabs3"])
@pytest.mark.parametrize("M,K,H,Hkv,D,inter", [(1, 896, 14, 2, 64, 4864), (4, 1024, 3, 1, 128, 520), (2, 2048, 2, 1, 64, 24),
                                               (3, 256, 1, 1, 128, 136)])
def test_against_float64(M, K, H, Hkv, D, inter, form, name):
    """Both products of normed rows, SiLU's and the rotation's ends, from the sums to the last rounding in float64."""
    from byox_vllm_amd import kernels
    from byox_vllm_amd.layers.quant import LinearWeight, interleave_gate_up
    torch.manual_seed(M + K)
    dt, N, u = DT[name], (H + 2 * Hkv) * D, torch.finfo(DT[name]).eps / 2
    x, rows, res = inputs(M, K, dt, form)
    nw = (torch.rand(K, device=DEV) + 0.5).to(dt)
    h = norm64(rows, res, nw, 1e-6, dt)
    # a row's normed numbers may lie on the other side of a rounding: sums of K products of N(0, 1) by N(0, 1 / K) with some of their
    # terms off by two roundings stay within two of a unit number; each result then has its own roundings
    gu = (torch.randn(2 * inter, K, device=DEV) * K ** -0.5).to(dt)
    got, _ = kernels.norm_gemm_silu(x, res, nw, 1e-6, LinearWeight.dense_tiled(interleave_gate_up(gu)))
    gate, up = (h @ gu.double().t()).chunk(2, -1)
    assert ((got.double() - torch.nn.functional.silu(gate) * up).abs() <= 5 * u * (1 + gate.abs()) * (1 + up.abs())).all()

    w, bias = (torch.randn(N, K, device=DEV) * K ** -0.5).to(dt), torch.randn(N, device=DEV).to(dt)
    pos, angle = torch.randint(0, 100, (M,), device=DEV), torch.rand(100, D // 2, device=DEV) * 6.28
    cos_sin = torch.cat([angle.cos(), angle.sin()], -1).contiguous()
    qkv, _ = kernels.norm_gemm_rope_kv_store(x, res, nw, 1e-6, LinearWeight.dense_tiled(w), bias, pos, cos_sin, H, Hkv, D)
    y = (h @ w.double().t() + bias.double()).view(M, -1, D)
    a, b = y[:, :H + Hkv].chunk(2, -1)
    c, s = cos_sin[pos].double().view(M, 1, D).chunk(2, -1)
    want = torch.cat([torch.cat([a * c - b * s, b * c + a * s], -1), y[:, H + Hkv:]], 1)
    size = 1 + torch.maximum(want.abs(), y.abs().amax(-1, keepdim=True))
    assert ((qkv.view(M, -1, D).double() - want).abs() <= 5 * u * size).all()


def test_refuses_what_it_cannot_hold():
    from byox_vllm_amd import kernels
    from byox_vllm_amd.layers.quant import LinearWeight
    w = LinearWeight.dense_tiled(torch.zeros(32, 2048, dtype=torch.bfloat16, device=DEV))
    x, nw = torch.zeros(12, 2048, dtype=torch.bfloat16, device=DEV), torch.ones(2048, dtype=torch.bfloat16, device=DEV)
    assert kernels.takes_norm(x[:4], None, w, nw) and not kernels.takes_norm(x[:5], None, w, nw)
    assert not kernels.takes_norm(x, None, w, nw)
    with pytest.raises(RuntimeError):
        kernels.norm_gemm_silu(x, None, nw, 1e-6, w)


def test_refuses_operands_before_any_launch(monkeypatch):
    """Rows or a residual in host memory, weights of another size or type: an error of the wrapper, no launch."""
    from byox_vllm_amd import kernels
    from byox_vllm_amd.layers.quant import LinearWeight

    def launched():
        raise SystemError("reached the library")
    w = LinearWeight.dense_tiled(torch.zeros(32, 896, dtype=torch.bfloat16, device=DEV))
    x, nw = torch.zeros(2, 896, dtype=torch.bfloat16, device=DEV), torch.ones(896, dtype=torch.bfloat16, device=DEV)
    slabs = torch.zeros(2, 2, 896, device=DEV)
    assert kernels.takes_norm(x, x, w, nw)
    parts = lambda s: kernels.Partials(s, 2, 2, 896, None, torch.bfloat16)  # noqa: E731
    monkeypatch.setattr(kernels, "lib", launched)
    for rows, res, weight in ((x.cpu(), None, nw), (x, x.cpu(), nw), (x, x, nw[:64]), (x, x[:1], nw), (x.half(), None, nw),
                              (x, x.half(), nw), (x, x, nw.half()), (x[:, :512], None, nw[:512]), (x, None, nw.cpu()),
                              (parts(slabs.cpu()), x, nw), (parts(slabs), x, nw[:64])):
        # (a weight or slabs in host memory: no other path has a check for them, so it is the wrapper that raises)
        assert weight.is_cpu or getattr(rows, "slabs", nw).is_cpu or not kernels.takes_norm(rows, res, w, weight)
        with pytest.raises((RuntimeError, AssertionError)):
            kernels.norm_gemm_silu(rows, res, weight, 1e-6, w)
    for rows, bias in ((x.cpu(), None), (x.half(), None), (x[:, :512], None), (x.t().contiguous().t(), None), (x, nw[:31]), (x, nw[:32].half())):
        with pytest.raises((RuntimeError, AssertionError)):
            kernels.gemm_stream(rows, w, bias)


@pytest.fixture()
def layer():
    """A decoder layer with a KV cache, ready for a step of two tokens -> (the layer, its call)"""
    from types import SimpleNamespace

    from byox_vllm_amd.models.qwen3 import Qwen3DecoderLayer
    from byox_vllm_amd.utils.context import reset_context, set_context
    cfg = SimpleNamespace(hidden_size=256, num_attention_heads=4, num_key_value_heads=2, max_position_embeddings=64, rms_norm_eps=1e-6,
                          attention_bias=False, head_dim=64, intermediate_size=512, hidden_act="silu")
    torch.manual_seed(11)
    torch.set_default_dtype(torch.bfloat16)
    try:
        with torch.device(DEV):
            made = Qwen3DecoderLayer(cfg)
    finally:
        torch.set_default_dtype(torch.float32)
    for name, p in made.named_parameters():
        p.data.copy_(torch.rand_like(p) + 0.5 if "norm" in name else torch.randn_like(p) * 0.06)
    made.mlp.gate_up_proj.finalize(None, fuse_silu=True)
    cache = torch.zeros(2, 1, 16, 2, 64, dtype=torch.bfloat16, device=DEV)
    made.self_attn.attn.k_cache, made.self_attn.attn.v_cache = cache[0], cache[1]
    ints = lambda *v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731

    def call(first):
        x = torch.randn(2, 256, generator=torch.Generator(device=DEV).manual_seed(2), device=DEV).bfloat16()
        res = None if first else torch.randn(2, 256, generator=torch.Generator(device=DEV).manual_seed(3), device=DEV).bfloat16()
        set_context(True, ints(0, 2), ints(0, 2), 2, 2, ints(0, 1))
        try:
            out, res = made(torch.arange(2, device=DEV), x, res)
        finally:
            reset_context()
        if not torch.is_tensor(out):                  # split-K slabs, for the next layer's norm to sum
            out = out.slabs.view(torch.float32)[:out.n * 512].view(out.n, 2, 256).sum(0).bfloat16()
        return out, res
    return made, call


def count(monkeypatch, *names):
    """How often each of the library's functions is launched from here on."""
    from byox_vllm_amd import kernels
    real, calls = kernels.lib(), dict.fromkeys(names, 0)

    class Counting:
        def __getattr__(self, name):
            if name in calls:
                calls[name] += 1
            return getattr(real, name)
    monkeypatch.setattr(kernels, "lib", Counting)
    return calls


@pytest.mark.parametrize("first", [True, False])
@pytest.mark.parametrize("where", ["input_layernorm", "post_attention_layernorm", "self_attn", "mlp"])
def test_hooks_on_a_layers_modules_are_called(layer, where, first, monkeypatch):
    """A module with a hook is called as a module: its hook sees a tensor, or slabs, as from five rows on, and not a pair."""
    made, call = layer
    want = call(first)
    calls = count(monkeypatch, "nv_norm_gemm_silu", "nv_norm_gemm_rope_kv_store")
    call(first)
    assert calls == dict(nv_norm_gemm_silu=1, nv_norm_gemm_rope_kv_store=1)
    seen = []
    handle = getattr(made, where).register_forward_hook(lambda m, args, out: seen.append(out))
    got = call(first)
    handle.remove()
    assert len(seen) == 1 and calls["nv_norm_gemm_silu"] + calls["nv_norm_gemm_rope_kv_store"] == 3
    assert isinstance(seen[0], tuple) == (where.endswith("norm") and not (first and where == "input_layernorm"))
    for a, b, what in zip(got, want, ("result", "residual")):
        close(a, b, torch.bfloat16, what)
    every = []
    handle = torch.nn.modules.module.register_module_forward_hook(lambda m, args, out: every.append(m))
    call(first)
    handle.remove()
    assert getattr(made, where) in every
    getattr(made, where).forward = lambda *a, **k: type(getattr(made, where)).forward(getattr(made, where), *a, **k)
    call(first)
    assert calls["nv_norm_gemm_silu"] + calls["nv_norm_gemm_rope_kv_store"] == 4


@pytest.mark.parametrize("force", [False, True])
def test_forced_rotation_behind_the_product(layer, force, monkeypatch):
    """NV_FUSE_QKV_ROPE=2 (read when the layer is made) sends every row count to nv_gemm_rope_kv_store."""
    made, call = layer
    made.self_attn.force_fuse_qkv_rope = force
    calls = count(monkeypatch, "nv_gemm_rope_kv_store", "nv_norm_gemm_rope_kv_store")
    call(False)
    assert calls == dict(nv_gemm_rope_kv_store=int(force), nv_norm_gemm_rope_kv_store=int(not force))
