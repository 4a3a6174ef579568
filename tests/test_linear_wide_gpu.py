"""nv_linear's wide tiles (csrc/linear_wide.h) at the edges of their row, column and K tiles, in every tile size, against
float64; groups that are empty, end on a tile and end inside one; and K sizes the tiles leave to the other kernels."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def close(got, want, K, dtype, out_dtype):
    # fp32 accumulation of K products that are exact (16-bit operands) or rounded once (fp32), then one rounding
    tol = K * 2.0 ** -24 + (2.0 ** -8 if out_dtype == torch.bfloat16 else 2.0 ** -22)
    got, want = got.double().cpu(), want.double().cpu()
    scale = want.pow(2).mean().sqrt()
    off = ((got - want).abs() / torch.maximum(scale, want.abs())).max()
    assert torch.isfinite(got).all() and off < tol, f"off by {off:.3g}, {tol:.3g} allowed"


@pytest.mark.parametrize("tile", ["0", "1", "2", None])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,K", [(65, 4, 64), (129, 127, 128), (255, 130, 192), (256, 256, 64), (300, 513, 320), (200, 96, 96),
                                   (90, 61, 40)])
def test_edges(M, N, K, dtype, tile, monkeypatch):
    from byox_vllm_amd import kernels
    if tile is not None:
        monkeypatch.setenv("NV_LINEAR_TILE", tile)
    torch.manual_seed(M + N + K)
    x, w = torch.randn(M, K + 8).to(dtype)[:, :K], torch.randn(N, K).to(dtype) * 0.1
    b = torch.randn(N).to(dtype)
    want = x.double() @ w.double().t() + b.double()
    for out_dtype in (dtype, torch.float32):
        got = kernels.linear(x.to(DEV), w.to(DEV), b.to(DEV), out_dtype=out_dtype)
        close(got, want, K, dtype, out_dtype)
    wide = torch.zeros(M, N + 3, dtype=torch.float32, device=DEV)         # rows that do not split into 16-byte pieces
    kernels.linear(x.to(DEV), w.to(DEV), b.to(DEV), out=wide[:, :N], out_dtype=torch.float32)
    close(wide[:, :N], want, K, dtype, torch.float32)
    assert not wide[:, N:].any()


@pytest.mark.parametrize("tile", ["0", "1", "2", None])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("sizes,N,K", [([0, 128, 1, 0, 257, 64, 0], 68, 64), ([300], 256, 128), ([5] * 70, 36, 64),
                                       ([0, 0, 256, 256, 3], 130, 192)])
def test_groups(sizes, N, K, dtype, tile, monkeypatch):
    from byox_vllm_amd import kernels
    if tile is not None:
        monkeypatch.setenv("NV_LINEAR_TILE", tile)
    torch.manual_seed(sum(sizes) + N)
    E, rows, T = len(sizes), sum(sizes), 90
    off = torch.tensor([0] + list(torch.tensor(sizes).cumsum(0)), dtype=torch.int32)
    x = torch.randn(T, K).to(dtype)
    token = torch.randint(0, T, (rows,), dtype=torch.int32)
    gu, scale = torch.randn(E, 2 * N, K).to(dtype) * 0.1, torch.rand(rows) + 0.5
    d = lambda t: t.to(DEV)  # noqa: E731
    args = dict(rows=rows, a_rows=d(token), batch=E, group_offsets=d(off), max_group_rows=max(65, max(sizes)))
    hidden = kernels.linear(d(x), d(gu), w_batch_stride=2 * N * K, epilogue=kernels.EPI_GLU, row_scale=d(scale),
                            out_dtype=torch.float32, **args)
    plain = kernels.linear(d(x), d(gu), w_batch_stride=2 * N * K, out_dtype=torch.float32, n=2 * N, **args)
    want_h, want_p = torch.zeros(rows, N, dtype=torch.float64), torch.zeros(rows, 2 * N, dtype=torch.float64)
    for e in range(E):
        a, b = off[e], off[e + 1]
        y = x[token[a:b].long()].double() @ gu[e].double().t()
        want_p[a:b] = y
        g, u = (y * scale[a:b, None].double()).chunk(2, -1)
        want_h[a:b] = torch.nn.functional.silu(g) * u
    close(plain, want_p, K, dtype, torch.float32)
    close(hidden, want_h, 2 * K, dtype, torch.float32)


@pytest.mark.parametrize("M,N,K,act", [(256 * 70 + 12, 1000, 128, None), (256 * 72, 1024, 192, 0), (256 * 33, 2048, 128, 1),
                                       (256 * 140 + 130, 512, 128, 4), (256 * 128 + 1, 515, 256, 2)])
def test_streams_of_tiles(M, N, K, act, monkeypatch):
    """More 256 x 256 tiles than workgroups: whole rounds, a last round dealt in halves of tiles, remainders of rows."""
    from byox_vllm_amd import kernels
    monkeypatch.setenv("NV_LINEAR_TILE", "2")
    kernels.block_many_rows(True)
    try:
        torch.manual_seed(M + N)
        x, w = torch.randn(M, K, device=DEV).bfloat16(), (torch.randn(N, K, device=DEV) * 0.1).bfloat16()
        coefficients = torch.tensor([0.8, 0.4], device=DEV)
        for out_dtype in (torch.bfloat16, torch.float32):
            args = {} if act is None else dict(epilogue=kernels.EPI_ACT, act=act, gate=coefficients if act == 2 else None)
            got = kernels.linear(x, w, out_dtype=out_dtype, **args)
            for lo in range(0, M, 8192):
                want = x[lo:lo + 8192].double() @ w.double().t()
                if act == 2:
                    want = torch.where(want > 0, 0.8 * want * want + 0.5 * want,
                                       0.4 * (torch.special.expm1(want) - want) + 0.5 * want)
                elif act is not None:
                    want = {0: torch.nn.functional.silu, 1: lambda v: torch.nn.functional.gelu(v, approximate="tanh"),
                            4: torch.nn.functional.gelu}[act](want)
                close(got[lo:lo + 8192], want, 4 * K, torch.bfloat16, out_dtype)
    finally:
        kernels.block_many_rows(False)


@pytest.mark.parametrize("M,N,K", [(256 * 70 + 12, 1000, 64), (256 * 33, 2048, 96), (256 * 40 + 130, 515, 160), (300, 260, 64)])
def test_streams_of_fp32_tiles(M, N, K, monkeypatch):
    from byox_vllm_amd import kernels
    monkeypatch.setenv("NV_LINEAR_TILE", "2")
    torch.manual_seed(M + N)
    x, w, b = torch.randn(M, K, device=DEV), torch.randn(N, K, device=DEV) * 0.1, torch.randn(N, device=DEV)
    for out_dtype in (torch.bfloat16, torch.float32):
        got = kernels.linear(x, w, b, out_dtype=out_dtype)
        for lo in range(0, M, 8192):
            close(got[lo:lo + 8192], x[lo:lo + 8192].double() @ w.double().t() + b.double(), K, torch.float32, out_dtype)


def gated(y, act, cap=0.0):
    """[.., gate | up] -> act(gate) * up, the clamped form for act 2."""
    g, u = y.chunk(2, -1)
    if act == 2:
        g, u = g.clamp(max=cap), u.clamp(-cap, cap)
        return g * torch.sigmoid(1.702 * g) * (u + 1)
    return (torch.nn.functional.silu(g) if act == 0 else torch.nn.functional.gelu(g, approximate="tanh")) * u


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,K,act,biased", [(256 * 70 + 12, 520, 128, 0, True), (256 * 66, 512, 192, 1, False),
                                              (256 * 33 + 130, 1027, 128, 2, True),
                                              (256 * 140 + 1, 256, 256, 0, False), (300, 136, 128, 1, True)])
def test_streams_of_gated_tiles(M, N, K, act, biased, out_dtype, monkeypatch):
    """Gate and up rows side by side in a wavefront: 16-byte pieces of 16- and 32-bit results and columns that do not split into them, several
    whole tiles per workgroup, last rounds in halves, remainders of rows and columns."""
    from byox_vllm_amd import kernels
    monkeypatch.setenv("NV_LINEAR_TILE", "2")
    kernels.block_many_rows(True)
    try:
        torch.manual_seed(M + N)
        x, w = torch.randn(M, K, device=DEV).bfloat16(), (torch.randn(2 * N, K, device=DEV) * 0.1).bfloat16()
        b = torch.randn(2 * N, device=DEV).bfloat16() if biased else None
        got = kernels.linear(x, w, b, out_dtype=out_dtype, epilogue=kernels.EPI_GLU, act=act, cap=1.5)
        for lo in range(0, M, 8192):
            want = gated(x[lo:lo + 8192].double() @ w.double().t() + (b.double() if biased else 0.0), act, 1.5)
            close(got[lo:lo + 8192], want, 4 * K, torch.bfloat16, out_dtype)
    finally:
        kernels.block_many_rows(False)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("sizes,N,K", [([4096, 0, 5000, 255, 300, 8192, 1, 1023], 1032, 128), ([700] * 40, 640, 192),
                                       ([33000, 0, 0, 129], 499, 128), ([256, 512] * 70, 264, 128)])
def test_streams_of_grouped_tiles(sizes, N, K, dtype, monkeypatch):
    """Experts' products whose workgroups walk several whole tiles, over gathered rows with a factor per row: gated into 16 and 32 bits, and
    plain."""
    from byox_vllm_amd import kernels
    monkeypatch.setenv("NV_LINEAR_TILE", "2")
    torch.manual_seed(sum(sizes) + N)
    E, rows, T = len(sizes), sum(sizes), 3000
    off = torch.tensor([0] + list(torch.tensor(sizes).cumsum(0)), dtype=torch.int32)
    tiles = sum(-(-n // 256) for n in sizes) * -(-2 * N // 256)
    assert tiles > 512
    x, token = torch.randn(T, K, device=DEV).to(dtype), torch.randint(0, T, (rows,), dtype=torch.int32, device=DEV)
    gu, scale = (torch.randn(E, 2 * N, K, device=DEV) * 0.1).to(dtype), torch.rand(rows, device=DEV) + 0.5
    args = dict(rows=rows, a_rows=token, batch=E, group_offsets=off.to(DEV), max_group_rows=max(sizes), row_scale=scale,
                w_batch_stride=2 * N * K)
    outs = [(o, kernels.linear(x, gu, epilogue=kernels.EPI_GLU, out_dtype=o, **args)) for o in (torch.bfloat16, torch.float32)]
    plain = kernels.linear(x, gu, out_dtype=torch.float32, n=2 * N, **args)
    for e in range(E):
        for lo in range(off[e], off[e + 1], 8192):
            hi = min(lo + 8192, int(off[e + 1]))
            y = (x[token[lo:hi].long()].double() @ gu[e].double().t()) * scale[lo:hi, None].double()
            close(plain[lo:hi], y, 2 * K, dtype, torch.float32)
            for o, got in outs:
                close(got[lo:hi], gated(y, 0), 4 * K, dtype, o)


@pytest.mark.parametrize("M,N,K", [(2500, 6144, 256), (2500, 6144, 224), (2500, 2048, 256), (2500, 2048, 224), (8000, 2048, 256),
                                   (4000, 4096, 256), (1500, 2048, 512), (16384, 64, 256)])
@pytest.mark.parametrize("glu", [False, True])
def test_fp32_on_both_sides_of_each_line(M, N, K, glu):
    """Sizes where fp32 products take 256 x 256, 64 x 128 and 128 x 128 tiles, and just below the K from which they do."""
    from byox_vllm_amd import kernels
    torch.manual_seed(M + N)
    x, w = torch.randn(M, K, device=DEV), torch.randn(N, K, device=DEV) * 0.1
    got = kernels.linear(x, w, epilogue=kernels.EPI_GLU if glu else kernels.EPI_NONE)
    want = x.double() @ w.double().t()
    if glu:
        gate, up = want.chunk(2, -1)
        want = torch.nn.functional.silu(gate) * up
    close(got, want, 2 * K, torch.float32, torch.float32)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_batches_and_gates(dtype):
    """One product per head side by side, with the row gate, the soft cap and the element-wise epilogues."""
    from byox_vllm_amd import kernels
    torch.manual_seed(3)
    M, H, K, n = 150, 3, 128, 72
    x, w, gate = torch.randn(M, H * K).to(dtype), torch.randn(H, n, K).to(dtype) * 0.1, torch.randn(M, H)
    want = torch.einsum("mhk,hnk->mhn", x.double().view(M, H, K), w.double())
    args = dict(batch=H, a_batch_stride=K, w_batch_stride=n * K, out_batch_stride=n, n=n, out_dtype=torch.float32)
    run = lambda **kw: kernels.linear(x.to(DEV), w.to(DEV), **args, **kw).view(M, H, n)  # noqa: E731
    close(run(), want, K, dtype, torch.float32)
    close(run(epilogue=kernels.EPI_ROW_GATE, gate=gate.to(DEV), gate_stride=H), want * torch.sigmoid(gate.double())[..., None], K,
          dtype, torch.float32)
    close(run(epilogue=kernels.EPI_SOFTCAP, cap=2.0), 2.0 * torch.tanh(want / 2.0), K, dtype, torch.float32)
    close(run(epilogue=kernels.EPI_ACT, act=kernels.ACT_SILU), torch.nn.functional.silu(want), K, dtype, torch.float32)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,K", [(150, 128), (150, 32), (40, 256)])          # the wide tiles, the short products, the few rows
@pytest.mark.parametrize("per_number", [False, True])
def test_gates_of_rows_and_of_numbers(dtype, M, K, per_number):
    from byox_vllm_amd import kernels
    torch.manual_seed(M + K)
    H, n = 3, 70
    x, w = torch.randn(M, H * K).to(dtype), torch.randn(H, n, K).to(dtype) * 0.1
    gate = torch.randn(M, H * n if per_number else H)
    got = kernels.linear(x.to(DEV), w.to(DEV), batch=H, a_batch_stride=K, w_batch_stride=n * K, out_batch_stride=n, n=n,
                         out_dtype=torch.float32, epilogue=kernels.EPI_ROW_GATE, act=kernels.GATE_PER_NUMBER if per_number else 0,
                         gate=gate.to(DEV), gate_stride=gate.size(1)).view(M, H, n)
    want = torch.matmul(x.double().view(M, H, K).transpose(0, 1), w.double().transpose(1, 2)).transpose(0, 1)
    close(got, want * torch.sigmoid(gate.double()).view(M, H, -1), K, dtype, torch.float32)


@pytest.mark.parametrize("M,N,K,H,softcap", [(1100, 32, 128, 32, False), (1000, 32, 128, 32, False), (1100, 33, 96, 8, False),
                                             (1300, 5, 64, 30, True), (130, 200, 64, 1, True), (200, 3100, 64, 1, True)])
def test_fp32_products_on_both_sides_of_the_rule(M, N, K, H, softcap):
    """Narrow and short fp32 products that stay with the kernel for any shape, and their neighbours in wide tiles."""
    from byox_vllm_amd import kernels
    torch.manual_seed(M + N)
    x, w = torch.randn(M, H * K), torch.randn(H, N, K) * 0.1
    args = dict(batch=H, a_batch_stride=K, w_batch_stride=N * K, out_batch_stride=N, n=N) if H > 1 else {}
    got = kernels.linear(x.to(DEV), (w if H > 1 else w[0]).to(DEV), out_dtype=torch.float32, cap=2.0,
                         epilogue=kernels.EPI_SOFTCAP if softcap else kernels.EPI_NONE, **args).view(M, H, N)
    want = torch.matmul(x.double().view(M, H, K).transpose(0, 1), w.double().transpose(1, 2)).transpose(0, 1)
    close(got, 2.0 * torch.tanh(want / 2.0) if softcap else want, K, torch.float32, torch.float32)


def correctly_rounded(got, want, dtype, ulps):
    """|got - want| within half a unit of the 16-bit type and ``ulps`` units of fp32 (of the numbers before that rounding)."""
    bits = 8 if dtype == torch.bfloat16 else 11
    spacing = torch.exp2(torch.floor(torch.log2(want.abs().clamp_min(2.0 ** -126))) + 1 - bits)
    bad = (got.double().cpu() - want).abs() > 0.5 * spacing + ulps * 2.0 ** -23 * want.abs()
    assert not bad.any(), f"{int(bad.sum())} of {bad.numel()} off, the first at {want[bad][0]:.6g}: {got.double().cpu()[bad][0]:.6g}"


@pytest.mark.parametrize("tile", ["0", "1", "2"])
def test_gated_unit_is_exact_in_fp32(tile, monkeypatch):
    """SiLU(gate) * up of gates and ups that the products give exactly, down to where exp(-gate) nearly overflows: the exponential
    within 1 unit of fp32, a sum, a quotient and a product within half of one each, then bf16's rounding - in every tile size."""
    from byox_vllm_amd import kernels
    monkeypatch.setenv("NV_LINEAR_TILE", tile)
    torch.manual_seed(7)
    M, N, K = 300, 1024, 128
    x, w = torch.zeros(M, K), torch.zeros(2 * N, K)
    x[:, 0], x[:, 1] = 1.0, 1.0 + torch.rand(M)
    w[:N, 0], w[N:, 1] = torch.linspace(-88.5, 20.0, N), 1.0 + torch.rand(N)
    x, w = x.bfloat16(), w.bfloat16()
    gate, up = (x.double() @ w.double().t()).chunk(2, -1)
    got = kernels.linear(x.to(DEV), w.to(DEV), epilogue=kernels.EPI_GLU)
    assert got.dtype == torch.bfloat16
    correctly_rounded(got, gate / (1.0 + torch.exp(-gate)) * up, torch.bfloat16, 3.0)


@pytest.mark.parametrize("epilogue,n", [("GLU", 16), ("ACT", 16), ("NONE", 1040)])
def test_more_rows_than_one_launch_holds(epilogue, n):
    """65535 * 64 rows and some: gated and element-wise epilogues in pieces of rows, plain products through the library."""
    from byox_vllm_amd import kernels
    torch.manual_seed(5)
    M, K = kernels.LINEAR_ROWS + 300, 128
    x = torch.randn(8192, K, device=DEV).bfloat16().repeat(-(-M // 8192), 1)[:M]
    w = (torch.randn(n * (2 if epilogue == "GLU" else 1), K, device=DEV) * 0.1).bfloat16()
    got = kernels.linear(x, w, epilogue=getattr(kernels, "EPI_" + epilogue))
    assert got.shape == (M, n) and got.dtype == torch.bfloat16
    for lo, hi in ((0, 500), (kernels.LINEAR_ROWS - 300, kernels.LINEAR_ROWS + 300)):
        want = x[lo:hi].double() @ w.double().t()
        if epilogue == "GLU":
            gate, up = want.chunk(2, -1)
            want = torch.nn.functional.silu(gate) * up
        elif epilogue == "ACT":
            want = torch.nn.functional.silu(want)
        close(got[lo:hi], want, 2 * K, torch.bfloat16, torch.bfloat16)
