"""nv_gemm_stream and its rotating form (csrc/gemm_stream.hip) at the edges of their 256 x 256 tiles: ragged row tiles, last
rounds dealt in halves, columns that end inside a tile, both 16-bit weight layouts, both head sizes."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
DT = {"bf16": torch.bfloat16, "fp16": torch.float16}


def weight(w, tiled):
    from byox_vllm_amd.layers.quant import LinearWeight
    return LinearWeight.dense_tiled(w) if tiled else LinearWeight.dense(w)


def close(got, want, dt, K, ulps=1.0):
    # `ulps` roundings to 16 bits, and K roundings of fp32 partial sums of a few units where the products cancel
    eps = torch.finfo(dt).eps
    got, want = got.double(), want.double()
    bad = (got - want).abs() > ulps * eps * want.abs() + 8.0 * K ** 0.5 * 2.0 ** -24
    assert torch.isfinite(got).all() and not bad.any(), f"{int(bad.sum())} of {bad.numel()} off, max {(got - want).abs().max()}"


SHAPES = [(1, 16, 128), (255, 272, 128), (257, 640, 256), (4100, 528, 384), (256 * 66 + 3, 1024, 128), (2300, 4096, 256)]


@pytest.mark.parametrize("name", ["bf16", "fp16"])
@pytest.mark.parametrize("tiled", [True, False])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_plain(M, N, K, tiled, name):
    from byox_vllm_amd import kernels
    torch.manual_seed(M + N)
    dt = DT[name]
    x, w, b = torch.randn(M, K, device=DEV).to(dt), (torch.randn(N, K, device=DEV) * 0.05).to(dt), torch.randn(N, device=DEV).to(dt)
    want = x.double() @ w.double().t()
    out = torch.zeros(M, N + 8, dtype=dt, device=DEV)
    got = kernels.gemm_stream(x, weight(w, tiled), b, out=out[:, :N])
    close(got, want + b.double(), dt, K)
    assert not out[:, N:].any()
    close(kernels.gemm_stream(x, weight(w, tiled)), want, dt, K)


@pytest.mark.parametrize("name", ["bf16", "fp16"])
@pytest.mark.parametrize("tiled", [True, False])
@pytest.mark.parametrize("M,inter,K", [(1, 16, 128), (255, 272, 128), (300, 1536, 256), (2100, 1040, 384), (256 * 66 + 3, 512, 128),
                                       (1, 8, 128), (700, 24, 256), (300, 1000, 128)])
def test_silu_mul(M, inter, K, tiled, name):
    """Gate and up rows as the kernels store them, against the product's, SiLU's and the last rounding taken one by one."""
    from byox_vllm_amd import kernels
    from byox_vllm_amd.layers.quant import interleave_gate_up
    torch.manual_seed(M + inter)
    dt = DT[name]
    x, w = torch.randn(M, K, device=DEV).to(dt), (torch.randn(2 * inter, K, device=DEV) * 0.05).to(dt)
    got = kernels.gemm_stream(x, weight(interleave_gate_up(w), tiled), silu_mul=True)
    gate, up = (x.double() @ w.double().t()).to(dt).double().chunk(2, -1)
    want = torch.nn.functional.silu(gate).to(dt).double() * up
    close(got, want, dt, K, ulps=3.0)      # a gate on the other side of a rounding moves two more


@pytest.mark.parametrize("name", ["bf16", "fp16"])
def test_silu_mul_has_the_bits_of_the_pass_over_rows(name):
    """Gates and ups that the products give exactly, down to where exp(-gate) nearly overflows: nv_silu_mul's bits."""
    from byox_vllm_amd import kernels
    from byox_vllm_amd.layers.quant import interleave_gate_up
    torch.manual_seed(7)
    M, inter, K, dt = 300, 1024, 128, DT[name]
    x, w = torch.zeros(M, K), torch.zeros(2 * inter, K)
    x[:, 0], x[:, 1] = 1.0, 1.0 + torch.rand(M)
    w[:inter, 0], w[inter:, 1] = torch.linspace(-88.5, 20.0, inter), 1.0 + torch.rand(inter)
    x, w = x.to(dt).to(DEV), w.to(dt).to(DEV)
    rows = (x.double() @ w.double().t()).to(dt)
    got = kernels.gemm_stream(x, weight(interleave_gate_up(w), True), silu_mul=True)
    assert torch.equal(got, kernels.silu_mul(rows))


@pytest.mark.parametrize("name", ["bf16", "fp16"])
@pytest.mark.parametrize("tiled", [True, False])
@pytest.mark.parametrize("T,H,Hkv,D,norms", [(1, 1, 1, 64, False), (257, 14, 2, 64, False), (300, 3, 1, 64, True), (513, 16, 8, 128, True),
                                             (4100, 5, 1, 128, False), (256 * 34 + 5, 4, 2, 128, True)])
def test_rope_kv_store(T, H, Hkv, D, norms, tiled, name):
    """The launch against the product and nv_rope_kv_store in two: the same roundings, so equal up to the order of the norm's sum."""
    from byox_vllm_amd import kernels
    torch.manual_seed(T + H)
    dt, K, N = DT[name], 256, (H + 2 * Hkv) * D
    x, w = torch.randn(T, K, device=DEV).to(dt), (torch.randn(N, K, device=DEV) * 0.1).to(dt)
    bias = None if norms else torch.randn(N, device=DEV).to(dt)
    qn, kn = ((torch.rand(D, device=DEV) + 0.5).to(dt) if norms else None for _ in range(2))
    pos = torch.randint(0, 500, (T,), device=DEV)
    cos_sin = torch.randn(500, D, device=DEV)
    pages = -(-T // 16) + 1
    slots = torch.randperm(pages * 16, device=DEV)[:T].int()
    slots[T // 2] = -1 if T > 1 else slots[0]                 # a token that is not kept
    caches = [torch.zeros(pages, 16, Hkv, D, dtype=dt, device=DEV) for _ in range(4)]
    args = dict(slot_mapping=slots, q_norm_w=qn, k_norm_w=kn, eps=1e-6)
    got = kernels.gemm_stream_rope_kv_store(x, weight(w, tiled), bias, pos, cos_sin, H, Hkv, D, k_cache=caches[0], v_cache=caches[1], **args)
    qkv = kernels.gemm_stream(x, weight(w, tiled), bias)
    close(qkv, x.double() @ w.double().t() + (0 if bias is None else bias.double()), dt, K)
    want = kernels.rope_kv_store(qkv, pos, cos_sin, H, Hkv, D, k_cache=caches[2], v_cache=caches[3], **args)
    for a, b in ((got, want), (caches[0], caches[2]), (caches[1], caches[3])):
        if norms:
            # one rounding of the normed number, another of its product with the weight, turned by |(cos, sin)| up to 6, and its own
            scale = torch.finfo(dt).eps * 8.0 * 6.0
            assert ((a.double() - b.double()).abs() <= scale * (1 + b.double().abs())).all()
            assert (a != b).float().mean() < 1e-3
        else:
            # the same fp32 numbers (a compiler may contract a product of up to 32 into the sum: 2^-19) rounded once
            assert ((a.double() - b.double()).abs() <= torch.finfo(dt).eps * b.double().abs() + 2.0 ** -19).all()
            assert (a != b).float().mean() < 1e-3
    bare = kernels.gemm_stream_rope_kv_store(x, weight(w, tiled), bias, pos, cos_sin, H, Hkv, D, q_norm_w=qn, k_norm_w=kn)
    assert torch.equal(bare, got)


@pytest.mark.parametrize("tiled", [True, False])
@pytest.mark.parametrize("K", [128, 192, 256])
@pytest.mark.parametrize("H,Hkv,D,norms", [(25, 4, 64, False), (9, 4, 128, True), (30, 2, 64, True)])
def test_rope_kv_store_of_three_tiles_to_a_workgroup(H, Hkv, D, norms, K, tiled):
    """Positions, cache rows and norm weights of one tile while others are fetched: with one pair of K blocks to a tile (K = 128) the
    wavefronts without columns (33 heads of 64, 17 of 128) or with values alone are two tiles' fetches ahead of those that still read."""
    from byox_vllm_amd import kernels
    if tiled and K % 128:
        pytest.skip("weights in tiles have K in 128s")
    torch.manual_seed(K + H)
    T, N, dt = 256 * 64 + 70, (H + 2 * Hkv) * D, torch.bfloat16
    assert -(-T // 256) * -(-N // 256) > 512
    x, w = torch.randn(T, K, device=DEV).to(dt), (torch.randn(N, K, device=DEV) * 0.1).to(dt)
    bias = None if norms else torch.randn(N, device=DEV).to(dt)
    qn, kn = ((torch.rand(D, device=DEV) + 0.5).to(dt) if norms else None for _ in range(2))
    pos = torch.randint(0, 500, (T,), device=DEV)
    cos_sin = torch.randn(500, D, device=DEV)
    pages = -(-T // 16) + 1
    slots = torch.randperm(pages * 16, device=DEV)[:T].int()
    caches = [torch.zeros(pages, 16, Hkv, D, dtype=dt, device=DEV) for _ in range(4)]
    args = dict(slot_mapping=slots, q_norm_w=qn, k_norm_w=kn, eps=1e-6)
    qkv = kernels.gemm_stream(x, weight(w, tiled), bias)
    want = kernels.rope_kv_store(qkv, pos, cos_sin, H, Hkv, D, k_cache=caches[2], v_cache=caches[3], **args)
    for _ in range(3):
        got = kernels.gemm_stream_rope_kv_store(x, weight(w, tiled), bias, pos, cos_sin, H, Hkv, D, k_cache=caches[0], v_cache=caches[1], **args)
        for a, b in ((got, want), (caches[0], caches[2]), (caches[1], caches[3])):
            # as in test_rope_kv_store: the norm's sum in another order, or the same numbers rounded once
            scale = torch.finfo(dt).eps * 8.0 * 6.0 if norms else torch.finfo(dt).eps
            assert ((a.double() - b.double()).abs() <= scale * (1 + b.double().abs())).all()
            assert (a != b).float().mean() < 1e-3


@pytest.mark.parametrize("M", [300, 2100, 4100])
@pytest.mark.parametrize("inter", [24, 40])
@pytest.mark.parametrize("fmt", [None, "w4a16"])
def test_gate_up_of_any_width_at_every_row_count(M, inter, fmt):
    """Gate/up products whose 2 * inter columns are a multiple of 16 but not of 32: from 2048 and 4096 rows on too."""
    from byox_vllm_amd import kernels
    from byox_vllm_amd.layers.quant import LinearWeight, interleave_gate_up
    torch.manual_seed(M + inter)
    K, dt = 256, torch.bfloat16
    x, w = torch.randn(M, K, device=DEV).to(dt), (torch.randn(2 * inter, K, device=DEV) * 0.05).to(dt)
    lw = LinearWeight.make(interleave_gate_up(w), fmt)
    assert (2 * inter) % 32
    gate, up = (x.double() @ kernels.expand_weight(lw, gate_up_rows=True).double().t()).to(dt).double().chunk(2, -1)
    close(kernels.gemm(x, lw, silu_mul=True), torch.nn.functional.silu(gate).to(dt).double() * up, dt, K, ulps=3.0)


@pytest.mark.parametrize("stride", [0, 64])
def test_rows_that_overlap_stay_with_nv_gemm(stride):
    """One row expanded over all, and windows of one buffer that overlap: as at 2047 rows, so at 2048."""
    from byox_vllm_amd import kernels
    from byox_vllm_amd.layers.quant import interleave_gate_up
    torch.manual_seed(3)
    M, K, inter, dt = 2048, 256, 64, torch.bfloat16
    x = torch.randn(K + M * 64, device=DEV).to(dt).as_strided((M, K), (stride, 1))
    lw = weight(interleave_gate_up((torch.randn(2 * inter, K, device=DEV) * 0.05).to(dt)), True)
    gate, up = (x.double() @ kernels.expand_weight(lw, gate_up_rows=True).double().t()).to(dt).double().chunk(2, -1)
    want = torch.nn.functional.silu(gate).to(dt).double() * up
    for rows in (2047, 2048):
        close(kernels.gemm(x[:rows], lw, silu_mul=True), want[:rows], dt, K, ulps=3.0)


def test_outputs_with_spare_rows_stay_with_nv_gemm():
    """A result buffer of more rows than the product has: its first rows are written from 2048 rows on too, the others left."""
    from byox_vllm_amd import kernels
    from byox_vllm_amd.layers.quant import interleave_gate_up
    torch.manual_seed(4)
    K, inter, dt = 256, 64, torch.bfloat16
    x = torch.randn(2100, K, device=DEV).to(dt)
    lw = weight(interleave_gate_up((torch.randn(2 * inter, K, device=DEV) * 0.05).to(dt)), True)
    gate, up = (x.double() @ kernels.expand_weight(lw, gate_up_rows=True).double().t()).to(dt).double().chunk(2, -1)
    out = torch.zeros(2200, inter, dtype=dt, device=DEV)
    kernels.gemm(x, lw, out=out, silu_mul=True)
    close(out[:2100], torch.nn.functional.silu(gate).to(dt).double() * up, dt, K, ulps=3.0)
    assert not out[2100:].any()
