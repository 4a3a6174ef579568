"""16-bit products on the tiles of csrc/stream_deep.h where they can go wrong: an odd number of K blocks, one pair of blocks to a tile, halves
of tiles in a last round, short tiles, a third tile to a workgroup; and SiLU as it is formed behind them, for every gate."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def close(got, want, K, out_dtype):
    tol = K * 2.0 ** -24 + (2.0 ** -8 if out_dtype == torch.bfloat16 else 2.0 ** -22)       # fp32 sums of K exact products, one rounding
    off = ((got.double() - want).abs() / torch.maximum(want.pow(2).mean().sqrt(), want.abs())).max()
    assert torch.isfinite(got).all() and off < tol, f"off by {off:.3g}, {tol:.3g} allowed"


@pytest.mark.parametrize("K", [128, 192, 256, 320, 832])
@pytest.mark.parametrize("M,N", [(65, 300), (128, 64), (129, 512), (256 * 33 + 5, 2000), (256 * 17 + 130, 4100), (256 * 70 + 1, 1000),
                                 (256 * 64 + 70, 2104)])
def test_blocks_and_tiles(M, N, K, monkeypatch):
    """The last of the sizes: 585 tiles, three to some workgroups, one column of wavefronts empty in every ninth.  One row alone in a tile:
    256 * 70 + 1 here, and a group of one below."""
    from byox_vllm_amd import kernels
    monkeypatch.setenv("NV_LINEAR_TILE", "2")
    kernels.block_many_rows(True)
    try:
        torch.manual_seed(M + N + K)
        x, w = torch.randn(M, K, device=DEV).bfloat16(), (torch.randn(N, K, device=DEV) * 0.1).bfloat16()
        bias, scale = torch.randn(N, device=DEV).bfloat16(), torch.rand(M, device=DEV)
        want = x.double() @ w.double().t()
        for out_dtype in (torch.bfloat16, torch.float32):
            close(kernels.linear(x, w, out_dtype=out_dtype), want, K, out_dtype)
            close(kernels.linear(x, w, bias, out_dtype=out_dtype, row_scale=scale), want * scale.double()[:, None] + bias.double(), 2 * K, out_dtype)
    finally:
        kernels.block_many_rows(False)


@pytest.mark.parametrize("gated", [False, True])
def test_weights_of_4_gib(gated, monkeypatch):
    """Rows of W that lie 4 GiB and more from its first, and a gated product's ups as far from their gates."""
    from byox_vllm_amd import kernels
    monkeypatch.setenv("NV_LINEAR_TILE", "2")
    torch.manual_seed(4)
    M, K, n = 300, 4096, 2 ** 32 // 8192 + 696
    x = torch.randn(M, K, device=DEV).bfloat16()
    w = torch.empty((1 + gated) * n, K, device=DEV, dtype=torch.bfloat16).normal_(0.0, 0.1)
    got = kernels.linear(x, w, epilogue=kernels.EPI_GLU if gated else kernels.EPI_NONE)
    for at in (0, n // 2, n - 1000, n - 296):
        c = slice(at, at + 296)
        want = x.double() @ w[:n][c].double().t()
        if gated:
            want = torch.nn.functional.silu(want) * (x.double() @ w[n:][c].double().t())
        close(got[:, c], want, 4 * K, torch.bfloat16)


@pytest.mark.parametrize("tile", ["2", "4"])
def test_weight_rows_far_apart(tile, monkeypatch):
    """Rows of W 16 MiB apart: 256 of them span 4 GiB, which the tiles of eight wavefronts take."""
    from byox_vllm_amd import kernels
    monkeypatch.setenv("NV_LINEAR_TILE", tile)
    torch.manual_seed(6)
    x, w = torch.randn(300, 320, device=DEV).bfloat16(), torch.empty(300, 2 ** 23, device=DEV, dtype=torch.bfloat16)[:, :320]
    w.normal_(0.0, 0.1)
    close(kernels.linear(x, w), x.double() @ w.double().t(), 320, torch.bfloat16)


@pytest.mark.parametrize("tops", [[0, 0, 1000], [300, 1, 0, 129, 128, 257], [513] * 3])
def test_gathered_groups(tops, monkeypatch):
    """Groups that end anywhere in a tile, empty ones, rows from anywhere, gated."""
    from byox_vllm_amd import kernels
    monkeypatch.setenv("NV_LINEAR_TILE", "2")
    torch.manual_seed(sum(tops))
    T, K, n, E = 700, 320, 200, len(tops)
    x, w = torch.randn(T, K, device=DEV).bfloat16(), (torch.randn(E, 2 * n, K, device=DEV) * 0.1).bfloat16()
    rows = torch.randint(0, T, (sum(tops),), device=DEV, dtype=torch.int32)
    off = torch.tensor([sum(tops[:i]) for i in range(E + 1)], dtype=torch.int32, device=DEV)
    got = kernels.linear(x, w, rows=sum(tops), a_rows=rows, batch=E, w_batch_stride=2 * n * K, group_offsets=off, max_group_rows=max(max(tops), 65),
                         epilogue=kernels.EPI_GLU, n=n)
    at = 0
    for e, m in enumerate(tops):
        y = x[rows[at:at + m].long()].double() @ w[e].double().t()
        if m:
            close(got[at:at + m], torch.nn.functional.silu(y[:, :n]) * y[:, n:], 4 * K, torch.bfloat16)
        at += m


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("act", [-1, 3, 7])
def test_gated_products_without_an_activation_of_their_own(act, out_dtype, monkeypatch):
    """What is neither GELU nor the clamped unit is SiLU, on these tiles as on the others."""
    from byox_vllm_amd import kernels
    torch.manual_seed(5)
    K, n = 320, 300
    x, w = torch.randn(700, K, device=DEV).bfloat16(), (torch.randn(2 * n, K, device=DEV) * 0.1).bfloat16()
    y = x.double() @ w.double().t()
    want = torch.nn.functional.silu(y[:, :n]) * y[:, n:]
    for tile in ("0", "1", "2"):
        monkeypatch.setenv("NV_LINEAR_TILE", tile)
        got = kernels.linear(x, w, epilogue=kernels.EPI_GLU, act=act, out_dtype=out_dtype)
        close(got, want, 4 * K, out_dtype)
        assert torch.equal(got, kernels.linear(x, w, epilogue=kernels.EPI_GLU, out_dtype=out_dtype))


@pytest.mark.parametrize("tile", ["3", "4", "2"])      # eight wavefronts, four, by the rule
@pytest.mark.parametrize("n", [304, 300, 301])
@pytest.mark.parametrize("biased", [False, True])
def test_results_by_four_and_eight_wavefronts(tile, n, biased, monkeypatch):
    """Every epilogue, whole pieces of 16 bytes and numbers one by one, over tiles with and without a neighbour."""
    from byox_vllm_amd import kernels as k
    F = torch.nn.functional
    monkeypatch.setenv("NV_LINEAR_TILE", tile)
    torch.manual_seed(n)
    M, K = 700, 192
    x, w = torch.randn(M, K, device=DEV).bfloat16(), (torch.randn(2 * n, K, device=DEV) * 0.1).bfloat16()
    bias = torch.randn(2 * n, device=DEV).bfloat16() if biased else None
    rows, gate, prm = torch.rand(M, device=DEV), torch.randn(M, n, device=DEV), torch.tensor([0.7, 0.4], device=DEV)
    y = x.double() @ w.double().t() * rows.double()[:, None] + (bias.double() if biased else 0.0)
    v, u, g = y[:, :n], y[:, n:], torch.sigmoid(gate.double())
    xielu = torch.where(v > 0, prm[0].double() * v * v, prm[1].double() * (torch.expm1(v) - v)) + 0.5 * v
    clamped = torch.clamp(v, max=2.0)
    cases = [(dict(), v), (dict(epilogue=k.EPI_SOFTCAP, cap=3.0), 3.0 * torch.tanh(v / 3.0)),
             (dict(epilogue=k.EPI_ROW_GATE, gate=gate[:, :1].contiguous(), gate_stride=1), v * g[:, :1]),
             (dict(epilogue=k.EPI_ROW_GATE, act=k.GATE_PER_NUMBER, gate=gate, gate_stride=n), v * g),
             (dict(epilogue=k.EPI_ACT, act=k.ACT_SILU), F.silu(v)), (dict(epilogue=k.EPI_ACT, act=k.ACT_GELU_TANH), F.gelu(v, approximate="tanh")),
             (dict(epilogue=k.EPI_ACT, act=k.ACT_XIELU, gate=prm), xielu), (dict(epilogue=k.EPI_ACT, act=k.ACT_SCALE, cap=0.3), 0.3 * v),
             (dict(epilogue=k.EPI_ACT, act=k.ACT_GELU_ERF), F.gelu(v)), (dict(epilogue=k.EPI_GLU, act=k.ACT_SILU), F.silu(v) * u),
             (dict(epilogue=k.EPI_GLU, act=k.ACT_GELU_TANH), F.gelu(v, approximate="tanh") * u),
             (dict(epilogue=k.EPI_GLU, act=k.GLU_CLAMPED, cap=2.0), clamped * torch.sigmoid(1.702 * clamped) * (torch.clamp(u, -2.0, 2.0) + 1.0))]
    for args, want in cases:
        gated = args.get("epilogue") == k.EPI_GLU
        for out_dtype in (torch.bfloat16, torch.float32):
            got = k.linear(x, w if gated else w[:n], bias if gated or not biased else bias[:n], out_dtype=out_dtype, row_scale=rows, **args)
            close(got, want, 16 * K, out_dtype)      # as a product's, and a function that grows by 2 and more where its gate does


@pytest.mark.parametrize("M,n,K", [(2100, 1000, 320), (700, 304, 128)])
def test_silu_is_the_same_in_16_and_32_bits(M, n, K, monkeypatch):
    """Results in 16 bits are those in 32 bits, rounded: SiLU by exp and quotient in both."""
    from byox_vllm_amd import kernels
    monkeypatch.setenv("NV_LINEAR_TILE", "2")
    torch.manual_seed(K)
    x, w = torch.randn(M, K, device=DEV).bfloat16(), (torch.randn(2 * n, K, device=DEV) * 0.1).bfloat16()
    got = [kernels.linear(x, w, epilogue=kernels.EPI_GLU, out_dtype=dt, rows=M) for dt in (torch.bfloat16, torch.float32)]
    assert torch.equal(got[0], got[1].bfloat16())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_silu_of_every_gate(dt):
    """Gates of all 16-bit values: the numbers of nv_silu_mul (exp and an IEEE quotient), which are within 3 units of fp32 ahead of their
    rounding: half a unit of 16 bits, and a tie decided the other way now and then."""
    from byox_vllm_amd import kernels
    from byox_vllm_amd.layers.quant import LinearWeight, interleave_gate_up
    gates = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(dt).to(DEV)
    x = torch.zeros(65536, 128, device=DEV, dtype=dt)
    x[:, 0], x[:, 1] = gates, 1.0
    w = torch.zeros(512, 128, device=DEV, dtype=dt)
    w[:256, 0] = 1.0          # every gate column is the gate, every up column 1
    w[256:, 1] = 1.0
    finite = torch.isfinite(gates)
    x[~finite] = 0.0
    got = kernels.gemm_stream(x, LinearWeight.make(interleave_gate_up(w), None), None, None, True)
    assert torch.equal(got, got[:, :1].expand_as(got))
    alone = kernels.silu_mul(torch.cat([x[:, :1].expand(-1, 8), torch.ones_like(x[:, :8])], 1))[:, 0][finite]
    got, g = got[:, 0][finite], gates[finite].double()
    want = torch.where(g < -700, -0.0, g / (1.0 + torch.exp(-g)))
    tiny = 2.0 ** -126 if dt == torch.bfloat16 else 2.0 ** -24
    normal = (g.abs() >= tiny) & (want.abs() >= tiny)          # the matrix cores may take numbers below as 0
    assert torch.equal(got[normal], alone[normal])
    half = torch.ldexp(torch.ones_like(want), torch.frexp(want)[1] - (9 if dt == torch.bfloat16 else 12))          # of the last place
    deep = g < -88.7                # exp overflows fp32: 0
    assert (got[deep].abs().double() <= 2.0 ** -119).all()
    err = (got.double() - want).abs()[~deep]
    assert (err <= (half + 3 * 2.0 ** -23 * want.abs())[~deep] + tiny).all()
    x[1, 0] = float("nan")          # what is not finite stays in its row
    y = kernels.gemm_stream(x[:300], LinearWeight.make(interleave_gate_up(w), None), None, None, True)
    assert torch.isnan(y[1]).all() and torch.isfinite(y[0]).all() and torch.isfinite(y[2:]).all()
