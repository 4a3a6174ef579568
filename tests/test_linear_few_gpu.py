"""Products of at most 64 rows (csrc/linear_few.h) and of many rows by a short K (csrc/linear_short.h) against float64: rows and
columns around the sixteen of a tile, K around the pieces, rounds and wavefronts that share it, rows that are not aligned, groups
that are empty and full, the epilogues."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def check(got, x, w, bias, epilogue, K):
    from byox_vllm_amd import kernels
    want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    if bias is not None:
        want, size = want + bias.double(), size + bias.double().abs()
    # fp32 sums of K products: K / 16 additions deep at most, and the stored result's own rounding
    err = (K / 16 + 8) * 2.0 ** -24 * size
    if epilogue == kernels.EPI_GLU:
        (g, u), (eg, eu) = want.chunk(2, -1), err.chunk(2, -1)
        want = torch.nn.functional.silu(g) * u
        err = 1.1 * eg * u.abs() + (g.abs() + eg) * eu + 2.0 ** -20 * want.abs()
    elif epilogue == kernels.EPI_SOFTCAP:
        want = 3.0 * torch.tanh(want / 3.0)
        err = err + 2.0 ** -21 * 3.0
    if got.dtype == torch.bfloat16:
        err = err + 2.0 ** -8 * (want.abs() + err)
    assert ((got.double() - want).abs() <= err).all(), float(((got.double() - want).abs() / err).max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M", [1, 16, 17, 48, 64])
@pytest.mark.parametrize("N,K", [(1, 256), (15, 264), (33, 1000), (1000, 520), (256, 2048), (8208, 256), (40, 4104), (17, 777)])
@pytest.mark.parametrize("epilogue", [0, 1, 2])
def test_plain(dtype, M, N, K, epilogue):
    from byox_vllm_amd import kernels
    torch.manual_seed(M + N + K)
    n = 2 * N if epilogue == 1 else N
    x = torch.randn(M, K + 8, device=DEV).to(dtype)[:, :K]
    w = (torch.randn(n, K, device=DEV) * K ** -0.5).to(dtype)
    bias = torch.randn(n, device=DEV).to(dtype) if M % 2 else None
    got = kernels.linear(x, w, bias, out_dtype=torch.float32 if M < 40 else dtype, epilogue=epilogue, cap=3.0, n=N)
    check(got, x, w, bias, epilogue, K)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,K", [(48, 512), (1040, 264)])
@pytest.mark.parametrize("sizes", [[3, 0, 16, 17], [0, 64, 33, 1], [0, 0, 0, 2]])
@pytest.mark.parametrize("epilogue", [0, 1])
def test_groups(dtype, N, K, sizes, epilogue):
    from byox_vllm_amd import kernels
    torch.manual_seed(N + K)
    n, T, rows = 2 * N if epilogue else N, 64, sum(sizes)
    x = torch.randn(T, K, device=DEV).to(dtype)
    w = (torch.randn(4, n, K, device=DEV) * K ** -0.5).to(dtype)
    at = torch.randint(0, T, (rows,), dtype=torch.int32, device=DEV)
    off = torch.tensor([0] + torch.tensor(sizes).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    got = kernels.linear(x, w, out_dtype=torch.float32, rows=rows, a_rows=at, batch=4, w_batch_stride=n * K, group_offsets=off,
                         max_group_rows=T, epilogue=epilogue, act=kernels.ACT_SILU)
    for e in range(4):
        a, b = int(off[e]), int(off[e + 1])
        if a < b:
            check(got[a:b], x[at[a:b].long()], w[e], None, epilogue, K)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,K", [(48, 512), (1040, 264), (40, 1160), (1040, 3080)])
@pytest.mark.parametrize("sizes", [[1, 0, 0, 0], [0, 1, 5, 2], [3, 0, 5, 1]])          # eight rows and the nine beyond the rule
@pytest.mark.parametrize("epilogue", [0, 1])
def test_groups_of_a_few_rows_in_all(dtype, N, K, sizes, epilogue):
    from byox_vllm_amd import kernels
    torch.manual_seed(N + K)
    n, T, rows = 2 * N if epilogue else N, 6, sum(sizes)
    x = torch.randn(T, K, device=DEV).to(dtype)
    w = (torch.randn(4, n, K, device=DEV) * K ** -0.5).to(dtype)
    at = torch.randint(0, T, (rows,), dtype=torch.int32, device=DEV)
    off = torch.tensor([0] + torch.tensor(sizes).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    got = kernels.linear(x, w, out_dtype=torch.float32, rows=rows, a_rows=at, batch=4, w_batch_stride=n * K, group_offsets=off,
                         max_group_rows=T, epilogue=epilogue, act=kernels.ACT_SILU)
    for e in range(4):
        a, b = int(off[e]), int(off[e + 1])
        if a < b:
            check(got[a:b], x[at[a:b].long()], w[e], None, epilogue, K)


@pytest.mark.parametrize("dtype,K", [(torch.bfloat16, 8), (torch.bfloat16, 24), (torch.bfloat16, 32), (torch.bfloat16, 40),
                                     (torch.bfloat16, 64), (torch.float32, 4), (torch.float32, 16), (torch.float32, 20),
                                     (torch.float32, 32)])
@pytest.mark.parametrize("M", [65, 128, 2100])
@pytest.mark.parametrize("N", [1, 63, 256, 1000])
@pytest.mark.parametrize("epilogue", [0, 2])
def test_short_k(dtype, M, N, K, epilogue):
    from byox_vllm_amd import kernels
    torch.manual_seed(M + N + K)
    x = torch.randn(M, K + 8, device=DEV).to(dtype)[:, :K]
    w = torch.randn(N, K, device=DEV).to(dtype)
    bias = torch.randn(N, device=DEV).to(dtype) if N % 2 else None
    got = kernels.linear(x, w, bias, out_dtype=torch.float32 if M % 2 else dtype, epilogue=epilogue, cap=3.0)
    check(got, x, w, bias, epilogue, K)


def test_short_k_batched_gated_rows():
    from byox_vllm_amd import kernels
    torch.manual_seed(0)
    M, N, K, H = 130, 96, 32, 5
    x, w = torch.randn(M, H * K, device=DEV).bfloat16(), torch.randn(H, N, K, device=DEV).bfloat16()
    at, gate = torch.randperm(M, device=DEV).int(), torch.randn(M, H, device=DEV)
    out = torch.empty(M, H * N, device=DEV)
    kernels.linear(x, w, out=out, out_dtype=torch.float32, rows=M, a_rows=at, batch=H, a_batch_stride=K, w_batch_stride=N * K, out_batch_stride=N,
                   epilogue=kernels.EPI_ROW_GATE, act=0, gate=gate, gate_stride=H, n=N)
    rows = x[at.long()].view(M, H, K).double()
    want = torch.stack([rows[:, h] @ w[h].double().t() for h in range(H)], 1) * torch.sigmoid(gate.double())[..., None]
    size = torch.stack([rows[:, h].abs() @ w[h].double().abs().t() for h in range(H)], 1)
    assert ((out.view(M, H, N).double() - want).abs() <= (K / 16 + 24) * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("dtype,K", [(torch.bfloat16, 40), (torch.bfloat16, 64), (torch.float32, 20), (torch.float32, 32)])
@pytest.mark.parametrize("M,N", [(4170, 1000), (8200, 257), (66, 257)])          # 256 columns per workgroup; one workgroup short of it
@pytest.mark.parametrize("epilogue", [0, 3])
def test_short_k_four_tiles_per_wavefront(dtype, K, M, N, epilogue):
    from byox_vllm_amd import kernels
    torch.manual_seed(M + N + K)
    x, w = torch.randn(M, K, device=DEV).to(dtype), torch.randn(N, K, device=DEV).to(dtype)
    gate = torch.randn(M, 1, device=DEV) if epilogue else None
    got = kernels.linear(x, w, out_dtype=torch.float32, epilogue=epilogue, gate=gate, gate_stride=1)
    want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    if epilogue:
        want = want * torch.sigmoid(gate.double())
    assert ((got.double() - want).abs() <= (K / 16 + 24) * 2.0 ** -24 * size).all()
