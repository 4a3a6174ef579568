"""Causal convolutions of prompts (csrc/scan.hip, causal_conv_rows_kernel): at the edges of its tiles of eight tokens, for every number of taps,
requests shorter than the taps among them, and channels that leave the last workgroup partly empty."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def i32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


# the last three: no more tokens than requests, not all of which have one
@pytest.mark.parametrize("lens", [[2], [8, 1, 7], [1, 2, 3, 0, 9, 16, 31], [1] * 5 + [65], [0, 0, 0, 0, 0, 6], [0, 2], [0, 9, 0, 1] + [0] * 9])
@pytest.mark.parametrize("taps", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("C,dtype", [(4, torch.float32), (260, torch.bfloat16), (1028, torch.float32), (1540, torch.bfloat16)])
@pytest.mark.parametrize("act", [0, 1, 2])
def test_rows_and_slots(lens, taps, C, dtype, act):
    from byox_vllm_amd import kernels
    torch.manual_seed(taps + C)
    T, keep, B = sum(lens), taps - 1, len(lens)
    cu = [sum(lens[:i]) for i in range(B + 1)]
    past = [3 * (i % 2) for i in range(B)]
    x = torch.randn(T, C + 4)[:, 4:]
    w, bias, x_bias = torch.randn(C, taps).to(dtype), torch.randn(C).to(dtype), torch.randn(C).to(dtype)
    state = torch.randn(B, keep, C)
    want, ends = torch.zeros(T, C, dtype=torch.float64), state.double()
    for b, n in enumerate(lens):
        if n == 0:
            continue
        rows = torch.cat([state[B - 1 - b].double() * (past[b] > 0), (x[cu[b]:cu[b + 1]] + x_bias.float()).double()])
        for k in range(n):
            want[cu[b] + k] = bias.double() + (rows[k:k + taps] * w.double().t()).sum(0)
            if act == 2:
                want[cu[b] + k] += rows[keep + k]
        ends[B - 1 - b] = rows[n:n + keep]
    if act == 1:
        want = torch.nn.functional.silu(want)
    d = state.to(DEV)
    x_d = torch.empty(T, C + 4, device=DEV)
    x_d[:, 4:] = x.to(DEV)
    f32, own = kernels.causal_conv(x_d[:, 4:], w.to(DEV), bias.to(DEV), d, i32(cu), i32(past), i32([B - 1 - b for b in range(B)]),
                                   i32([b for b, n in enumerate(lens) for _ in range(n)]), act=act, want_t=True, x_bias=x_bias.to(DEV))
    assert torch.equal(d.cpu().double(), ends)      # copies of fp32 sums
    # up to ten additions of terms of a few units each, and SiLU's exponential and quotient
    assert ((f32.double().cpu() - want).abs() <= 12 * 2.0 ** -24 * (want.abs() + 8 * taps)).all()
    assert torch.equal(own, f32.to(dtype))
