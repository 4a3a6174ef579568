"""Whole query rows of latent attention (csrc/latent_attn.hip, latent_q_rows_kernel) against float64: one, two and four tokens to a workgroup, last
workgroups with fewer, rows shorter and longer than a workgroup's lanes, rotations that end inside the rotated part."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("T", [1, 5, 2048, 2049, 2051])
@pytest.mark.parametrize("H,d,r,rot", [(1, 4, 8, 8), (3, 32, 16, 8), (4, 96, 32, 32), (5, 96, 32, 32), (9, 100, 28, 24), (2, 64, 0, 0)])
@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("dtype,out_dtype", [(torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32), (torch.float32, torch.float32)])
def test_rows(T, H, d, r, rot, interleaved, dtype, out_dtype):
    from byox_vllm_amd import kernels
    torch.manual_seed(T + H)
    q, positions = torch.randn(T, H * (d + r)).to(dtype), torch.randint(0, 100, (T,))
    freq = 10000.0 ** (-torch.arange(0, max(rot, 2), 2).float() / max(rot, 2))
    want = q.double().view(T, H, d + r).clone()
    if rot:
        part, half = want[..., d:d + rot].clone(), rot // 2
        angle = (positions.float()[:, None] * freq).double()[:, None]      # the product is the kernel's, in fp32
        a, b = (part[..., 0::2], part[..., 1::2]) if interleaved else (part[..., :half], part[..., half:])
        x, y = (a * angle.cos() - b * angle.sin()) * 1.25, (b * angle.cos() + a * angle.sin()) * 1.25
        want[..., d:d + rot] = torch.stack([x, y], -1).flatten(-2) if interleaved else torch.cat([x, y], -1)
    want = (want * 0.125).view(T, -1)
    got = kernels.latent_q_rows(q.to(DEV), positions.to(DEV), freq.to(DEV), 1.25, H, d, r, rot, 0.125, interleaved, out_dtype)
    assert got.dtype == out_dtype
    # cosines within 2 units of 2^-24, two products and their sum of numbers below 6; then one rounding of the result
    assert ((got.double().cpu() - want).abs() <= 2.0 ** -20 + (2.0 ** -8 * want.abs() if out_dtype == torch.bfloat16 else 0.0)).all()
