"""nv_linear's fp32 products in three 16-bit parts (csrc/linear_split.hip): what the parts must not lose.  Edges of tiles, groups and
epilogues in fp32: test_linear_wide_gpu.py."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
TILES = ["0", "1", "2"]


def error(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K", [(65, 100, 32 * 3), (300, 260, 1024), (130, 130, 2048)])
@pytest.mark.parametrize("values", ["normal", "positive", "range", "subnormal parts"])
def test_as_close_as_fp32(M, N, K, values, tile, monkeypatch):
    """Six additions to sixteen products, each rounding a sum of at most the result's size (and the parts' own rounding, 2^-24): their
    errors add up as a random walk."""
    from byox_vllm_amd import kernels
    monkeypatch.setenv("NV_LINEAR_TILE", tile)
    torch.manual_seed(M + K)
    x, w = torch.randn(M, K, device=DEV), torch.randn(N, K, device=DEV)
    if values == "positive":
        x, w = x.abs(), w.abs()
    elif values == "range":
        x, w = x * torch.exp(5 * torch.randn_like(x)), w * torch.exp(5 * torch.randn_like(w))
    elif values == "subnormal parts":      # the lower parts of numbers around 1e-37 lie below the normal range
        x, w = x * 1e-37, w * 1e30
    got, want = kernels.linear(x, w), x.double() @ w.double().t()
    assert error(got, want) < (6 * K / 16) ** 0.5 * 2.0 ** -24 + 2.0 ** -23


@pytest.mark.parametrize("tile", TILES)
def test_values_without_parts(tile, monkeypatch):
    """Infinities, NaNs and numbers too large to be scaled: where they reach, the products are those of fp32; nowhere else
    do they show."""
    from byox_vllm_amd import kernels
    monkeypatch.setenv("NV_LINEAR_TILE", tile)
    torch.manual_seed(3)
    x, w = torch.randn(300, 256, device=DEV), torch.randn(270, 256, device=DEV)
    x[5, 7], x[100, 3], x[299, 255], w[17, 30] = float("inf"), float("nan"), float("-inf"), float("inf")
    w[:, 9], x[:, 9] = 2.0 ** -126, 0.0
    x[200, 9] = 3.4e38          # times 2^-126: about 4
    x[250], x[251, 1:] = 0.0, 0.0
    w[269, 0], x[251, 0] = 3.39e38, 1.0
    got, want = kernels.linear(x, w).double().cpu(), x.double().cpu() @ w.double().cpu().t()
    want = want.float().double()      # infinite where fp32 ends
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[got.isinf()], want[want.isinf()])
    assert abs(got[251, 269] / 3.39e38 - 1) < 1e-6
    finite = want.isfinite()
    finite[:, 269] = False      # 1e38 times normal values: its own scale
    assert (got - want)[finite].abs().max() < 256 * 2.0 ** -24 * 16


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("value", [float("inf"), float("nan"), 1e30, 2.0 ** 60])
def test_results_without_parts_leave_the_others_alone(tile, value, monkeypatch):
    """A row of x and a column of results that are formed again: every other result is the same to the last bit."""
    from byox_vllm_amd import kernels
    monkeypatch.setenv("NV_LINEAR_TILE", tile)
    torch.manual_seed(4)
    x, w = torch.randn(300, 256, device=DEV), torch.randn(270, 256, device=DEV)
    clean = kernels.linear(x, w)
    x[77, 9], w[130, 200] = value, value
    got, rows, columns = kernels.linear(x, w), torch.arange(300) != 77, torch.arange(270) != 130
    assert torch.equal(got[rows][:, columns], clean[rows][:, columns])
    want = (x.double() @ w.double().t()).float()
    for a, b in ((got[77], want[77]), (got[:, 130], want[:, 130])):
        assert torch.equal(a.isfinite(), b.isfinite())
        a, b = (torch.where(b.isfinite(), c, 0.0) for c in (a, b))
        assert (a - b).abs().max() <= 256 * 2.0 ** -24 * b.abs().max()      # 256 additions, one of them next to all of the sum
