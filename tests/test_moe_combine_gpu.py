"""The weighted sum over a token's experts: rows that split into sixteen bytes and that do not, choices held elsewhere."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("width", [1, 6, 8, 1026, 2052])
@pytest.mark.parametrize("top", [1, 2, 4, 5, 9])
@pytest.mark.parametrize("shared", [None, "plain", "gated"])
def test_against_float64(width, top, shared):
    from byox_vllm_amd import kernels
    torch.manual_seed(width + top)
    T = 13
    y, wt = torch.randn(T * top, width, device=DEV), torch.rand(T, top, device=DEV)
    slots = torch.randperm(T * top, device=DEV).view(T, top).int()
    slots[torch.rand(T, top, device=DEV) < 0.3] = -1
    wt[slots < 0] = float("nan")                    # nobody reads them
    extra = torch.randn(T, width, device=DEV) if shared else None
    logits = torch.randn(T, 3, device=DEV)[:, 1:] if shared == "gated" else None
    got = kernels.moe_combine(y, slots, wt, extra, logits).double()
    held = (slots >= 0).double()[..., None]
    terms = wt.double().nan_to_num()[..., None] * held * y.double()[slots.clamp_min(0).long()]
    want, size = terms.sum(1), terms.abs().sum(1)
    if shared:
        add = extra.double() * (torch.sigmoid(logits[:, :1].double()) if logits is not None else 1.0)
        want, size = want + add, size + add.abs()
    assert ((got - want).abs() <= (top + 6) * 2.0 ** -24 * size + 1e-30).all()
