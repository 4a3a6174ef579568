"""Which launch a call of prefill or decode size takes, on both sides of each line that was drawn from measurements, and that the result
is the same kind of number there: within roundings of float64 on either route."""

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




@pytest.fixture()
def launched(monkeypatch):
    """The library's functions that are called, in their order, without the questions asked of it."""
    from byox_vllm_amd import kernels
    real, names = kernels.lib(), []

    class Listening:
        def __getattr__(self, name):
            got = getattr(real, name)
            if not name.endswith(("_available", "_bytes", "_is_faster", "_pick_split_k", "_policy", "_error")):
                names.append(name)
            return got
    monkeypatch.setattr(kernels, "lib", Listening)
    return names


def close(got, want, K, out_dtype):
    # fp32 sums of K exact products and an element-wise function, then a rounding to the storage type
    tol = 4 * K * 2.0 ** -24 + (2.0 ** -8 if out_dtype == torch.bfloat16 else 2.0 ** -20)
    off = ((got.double() - want).abs() / torch.maximum(want.pow(2).mean().sqrt(), want.abs())).max()
    assert torch.isfinite(got).all() and off < tol, f"off by {off:.3g}, {tol:.3g} allowed"


LIBRARY = ["nv_gemm_lt_f32out"]


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,K,n,epilogue,want", [
    (4100, 1024, 1024, "ACT", LIBRARY + ["nv_bias_act_f32"]), (4096, 1024, 4096, "ACT", ["nv_linear_rows"]),
    (6000, 1024, 1024, "GLU", LIBRARY + ["nv_bias_act_mul_f32"]), (8192, 1024, 1024, "GLU", ["nv_linear_rows"]),
    (6000, 512, 1024, "GLU", ["nv_linear_rows"]), (4095, 1024, 1024, "ACT", ["nv_linear_rows"]),
    (4100, 1024, 1008, "NONE", None), (5500, 256, 3088, "NONE", None), (4096, 256, 3088, "NONE", ["nv_linear_rows"]),
    (4096, 1152, 3088, "NONE", None)])
def test_linear_of_many_rows(M, K, n, epilogue, want, out_dtype, launched):
    """Epilogues are formed on the way where the results fill the rounds of tiles, else in a pass over the library's result."""
    from byox_vllm_amd import kernels
    torch.manual_seed(M + n)
    x = torch.randn(M, K, device=DEV).bfloat16()
    w = (torch.randn(n * (2 if epilogue == "GLU" else 1), K, device=DEV) * 0.05).bfloat16()
    got = kernels.linear(x, w, epilogue=getattr(kernels, "EPI_" + epilogue), out_dtype=out_dtype)
    assert launched == (want or ["nv_gemm_lt" if out_dtype == torch.bfloat16 else "nv_gemm_lt_f32out"])
    y = x.double() @ w.double().t()
    if epilogue == "GLU":
        y = torch.nn.functional.silu(y[:, :n]) * y[:, n:]
    elif epilogue == "ACT":
        y = torch.nn.functional.silu(y)
    close(got, y, K, out_dtype)


OWN, OTHER, LT = ["nv_gemm_stream"], ["nv_gemm"], ["nv_weight_expand", "nv_gemm_lt", "nv_silu_mul"]


@pytest.mark.parametrize("M,K,inter,fmt,want", [
    (2047, 512, 5120, None, OTHER), (2048, 512, 5120, None, OWN), (2048, 512, 2432, None, OTHER), (2048, 512, 2560, None, OWN),
    (2048, 512, 5120, "w4a16", OTHER), (4095, 256, 512, None, OTHER), (4096, 256, 512, None, OWN),
    (4096, 256, 512, "w8a16", ["nv_weight_expand"] + OWN),
    (4096, 3968, 256, None, OWN), (4096, 4096, 256, None, LT), (4096, 1920, 256, "w4a16", ["nv_weight_expand"] + OWN),
    (4096, 2048, 256, "w4a16", LT)])
def test_gate_up_of_many_rows(M, K, inter, fmt, want, launched):
    from byox_vllm_amd import kernels
    from byox_vllm_amd.layers.quant import LinearWeight, interleave_gate_up
    torch.manual_seed(M + K)
    dt = torch.bfloat16
    x = torch.randn(M, K, device=DEV).to(dt)
    lw = LinearWeight.make(interleave_gate_up((torch.randn(2 * inter, K, device=DEV) * K ** -0.5).to(dt)), fmt)
    got = kernels.gemm(x, lw, silu_mul=True)
    assert launched == want
    gate, up = (x.double() @ kernels.expand_weight(lw, gate_up_rows=True).double().t()).to(dt).double().chunk(2, -1)
    # the product, SiLU's and the last number rounded to 16 bits; a gate on the other side of a rounding moves two more
    want = torch.nn.functional.silu(gate).to(dt).double() * up
    off = (got.double() - want).abs() - 3.0 * torch.finfo(dt).eps * want.abs()
    assert torch.isfinite(got).all() and (off <= 8.0 * K ** 0.5 * 2.0 ** -24).all()


@pytest.mark.parametrize("M,K,N,fmt,bias,want", [
    (16384, 896, 896, None, False, OWN), (16384, 896, 896, "w4a16", False, ["nv_weight_expand"] + OWN),
    (16384, 896, 896, None, True, ["nv_weight_expand", "nv_gemm_lt"]), (11000, 896, 640, None, False, ["nv_weight_expand", "nv_gemm_lt"]),
    (14600, 896, 896, None, False, OWN), (14600, 896, 896, "w8a16", False, ["nv_weight_expand", "nv_gemm_lt"]),
    (16384, 896, 1024, None, False, ["nv_weight_expand", "nv_gemm_lt"]), (16384, 384, 896, None, False, ["nv_weight_expand", "nv_gemm_lt"]),
    (16384, 1024, 896, None, False, ["nv_weight_expand", "nv_gemm_lt"])])
def test_products_of_many_rows(M, K, N, fmt, bias, want, launched):
    from byox_vllm_amd import kernels
    from byox_vllm_amd.layers.quant import LinearWeight
    torch.manual_seed(M + K)
    dt = torch.bfloat16
    x = torch.randn(M, K, device=DEV).to(dt)
    lw = LinearWeight.make((torch.randn(N, K, device=DEV) * 0.05).to(dt), fmt)
    b = torch.randn(N, device=DEV).to(dt) if bias else None
    got = kernels.gemm(x, lw, b)
    assert launched == want
    close(got, x.double() @ kernels.expand_weight(lw).double().t() + (b.double() if bias else 0.0), K, dt)


def attention(K, H, Hkv, D, fmt, norms):
    from byox_vllm_amd.models.qwen3 import Qwen3Attention
    torch.set_default_dtype(torch.bfloat16)
    try:
        with torch.device(DEV):
            made = Qwen3Attention(K, H, Hkv, max_position=32768, head_dim=D, qkv_bias=not norms)
    finally:
        torch.set_default_dtype(torch.float32)
    for name, p in made.named_parameters():
        p.data.copy_(torch.rand_like(p) + 0.5 if "norm" in name else torch.randn_like(p) * 0.05)
    made.qkv_proj.finalize(fmt)
    return made


@pytest.mark.parametrize("M,K,H,Hkv,D,fmt,own", [
    (8192, 1024, 16, 8, 128, None, True), (4100, 1024, 16, 8, 128, None, False), (8192, 1024, 16, 8, 128, "w4a16", True),
    (14600, 896, 14, 2, 64, None, True), (14600, 896, 14, 2, 64, "w4a16", False), (5000, 896, 14, 2, 64, None, False),
    (11000, 896, 14, 2, 64, "w8a16", True), (8192, 2048, 16, 8, 128, None, True), (8192, 2048, 16, 8, 128, "w4a16", False),
    (8192, 2176, 8, 4, 128, None, False)])
def test_rotation_behind_the_product(M, K, H, Hkv, D, fmt, own, launched, monkeypatch):
    """q/k/v of many rows: one launch or two by the share of its rounds; rotated rows and the cache against float64."""
    from byox_vllm_amd import kernels
    from byox_vllm_amd.utils.context import reset_context, set_context
    torch.manual_seed(M + K)
    dt = torch.bfloat16
    made = attention(K, H, Hkv, D, fmt, norms=D == 128)
    x = torch.randn(M, K, device=DEV).to(dt)
    cache = torch.zeros(2, -(-M // 16), 16, Hkv, D, dtype=dt, device=DEV)
    made.attn.k_cache, made.attn.v_cache = cache[0], cache[1]
    pos, slots = torch.arange(M, device=DEV), torch.arange(M, device=DEV, dtype=torch.int32)
    monkeypatch.setattr(made, "_attend", lambda qkv: qkv)
    set_context(True, slot_mapping=slots)
    try:
        got = made(pos, x)
    finally:
        reset_context()
    assert ("nv_gemm_stream_rope_kv_store" in launched) == own and ("nv_rope_kv_store" in launched) != own
    y = x.double() @ kernels.expand_weight(made.qkv_proj.packed).double().t()
    if made.qkv_proj.bias is not None:
        y += made.qkv_proj.bias.data.double()
    y = y.view(M, H + 2 * Hkv, D)
    turned = y[:, :H + Hkv]
    if D == 128:
        turned = turned * torch.rsqrt((turned * turned).mean(-1, keepdim=True) + 1e-6)
        turned = torch.cat([turned[:, :H] * made.q_norm.weight.data.double(), turned[:, H:] * made.k_norm.weight.data.double()], 1)
    cos, sin = made.rotary_emb.cos_sin_cache[:M].view(M, 1, D).double().chunk(2, -1)
    a, b = turned.chunk(2, -1)
    want = torch.cat([torch.cat([a * cos - b * sin, b * cos + a * sin], -1), y[:, H + Hkv:]], 1)
    # roundings to eight bits, each up to 2^-8: the product's, with head norms two more ahead of the turn, and the last.  A turn adds two
    # numbers' errors: of a head's largest number, where the turned ones cancel.
    size = torch.maximum(want.abs(), torch.cat([turned, y[:, H + Hkv:]], 1).abs().amax(-1, keepdim=True))
    assert ((got.view(M, -1, D).double() - want).abs() <= 2.0 ** -8 * (1 + 2 ** 0.5 * (3 if D == 128 else 1)) * size + 1e-4).all()
    kv = got.view(M, -1, D)[:, H:].reshape(M, 2, Hkv, D)
    assert torch.equal(cache.view(2, -1, Hkv, D)[:, :M], kv.transpose(0, 1))


def decoder_layer(K, H, Hkv, D, inter):
    from types import SimpleNamespace

    from byox_vllm_amd.models.qwen3 import Qwen3DecoderLayer
    cfg = SimpleNamespace(hidden_size=K, num_attention_heads=H, num_key_value_heads=Hkv, max_position_embeddings=64, rms_norm_eps=1e-6,
                          attention_bias=D == 64, head_dim=D, intermediate_size=inter, hidden_act="silu")
    torch.set_default_dtype(torch.bfloat16)
    try:
        with torch.device(DEV):
            made = Qwen3DecoderLayer(cfg)
    finally:
        torch.set_default_dtype(torch.float32)
    for name, p in made.named_parameters():
        p.data.copy_(torch.rand_like(p) + 0.5 if "norm" in name else torch.randn_like(p) * 0.02)
    made.mlp.gate_up_proj.finalize(None, fuse_silu=True)
    return made


@pytest.mark.parametrize("rows,K,H,Hkv,D,inter,attn,mlp", [
    (1, 896, 14, 2, 64, 4864, True, True), (2, 896, 14, 2, 64, 4864, True, True), (4, 896, 14, 2, 64, 4864, True, False),
    (5, 896, 14, 2, 64, 1024, False, False), (2, 1024, 16, 8, 128, 3072, True, True), (3, 1024, 16, 8, 128, 3072, False, True),
    (1, 1536, 12, 2, 128, 8960, False, True), (2, 1536, 12, 2, 128, 8960, False, False), (1, 2048, 32, 8, 64, 6144, True, True),
    (3, 2048, 32, 8, 64, 3072, False, True), (4, 2048, 32, 8, 64, 3072, False, False), (1, 256, 4, 2, 64, 8960, True, False),
    (4, 512, 8, 2, 64, 1024, True, True), (1, 2176, 4, 2, 128, 1024, False, False)])
def test_norms_of_a_few_rows(rows, K, H, Hkv, D, inter, attn, mlp, launched):
    """A decoder layer's two norms, each inside the product behind it or in a launch of its own."""
    from byox_vllm_amd.utils.context import reset_context, set_context
    torch.manual_seed(K + rows)
    made = decoder_layer(K, H, Hkv, D, inter)
    cache = torch.zeros(2, 1, 16, Hkv, D, dtype=torch.bfloat16, device=DEV)
    made.self_attn.attn.k_cache, made.self_attn.attn.v_cache = cache[0], cache[1]
    ints = lambda *v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    x, res = (torch.randn(rows, K, device=DEV).bfloat16() for _ in range(2))
    set_context(True, ints(0, rows), ints(0, rows), rows, rows, ints(*range(rows)))
    try:
        made(torch.arange(rows, device=DEV), x, res)
    finally:
        reset_context()
    assert ("nv_norm_gemm_rope_kv_store" in launched, "nv_norm_gemm_silu" in launched) == (attn, mlp), launched
    assert sum(n.startswith("nv_add_rmsnorm") for n in launched) == 2 - attn - mlp


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,n", [(1, 4), (37, 516), (3, 7)])
def test_passes_over_a_products_rows(rows, n, dtype):
    """The passes behind the library's products, with a bias and in the forms without one (which only C callers use)."""
    from byox_vllm_amd._C import check, dtype_code, lib, ptr, stream
    torch.manual_seed(rows + n)
    y, b = torch.randn(rows, 2 * n, device=DEV), torch.randn(2 * n, device=DEV).to(dtype)
    code = dtype_code(dtype, allow_f32=True)
    for bias in (None, b):
        x = y.double() + (0.0 if bias is None else bias.double())
        out, half = torch.empty(rows, 2 * n, dtype=dtype, device=DEV), torch.empty(rows, n, dtype=dtype, device=DEV)
        if bias is None:
            check(lib().nv_act_f32(ptr(y), ptr(out), rows * 2 * n, 1, None, 0.0, code, stream()), "nv_act_f32")
            check(lib().nv_act_mul_f32(ptr(y), ptr(half), rows, n, 0, 0.0, code, stream()), "nv_act_mul_f32")
        else:
            check(lib().nv_bias_act_f32(ptr(y), ptr(bias), 2 * n, ptr(out), rows * 2 * n, 1, None, 0.0, code, stream()), "nv_bias_act_f32")
            check(lib().nv_bias_act_mul_f32(ptr(y), ptr(bias), ptr(half), rows, n, 0, 0.0, code, stream()), "nv_bias_act_mul_f32")
        close(out, torch.nn.functional.gelu(x, approximate="tanh"), 4, dtype)
        close(half, torch.nn.functional.silu(x[:, :n]) * x[:, n:], 4, dtype)
