"""Which products of many rows nv_gemm_stream forms in place of the vendor library, and its results at the new lines."""

import types

import pytest
import torch

from byox_vllm_amd import _C, kernels

TILED, INT4 = _C.W_DENSE_TILED, _C.W_INT4


@pytest.mark.parametrize("M,N,K,fmt,silu,own", [
    (4096, 24576, 3968, TILED, True, True), (8192, 16384, 7296, TILED, True, True), (8192, 16384, 7424, TILED, True, False),
    (5402, 4096, 7040, TILED, True, False), (5402, 4096, 3968, TILED, True, True), (16384, 6144, 1920, INT4, True, True),
    (8192, 37888, 3584, INT4, True, True), (8192, 37888, 7296, INT4, True, True), (8192, 37888, 7424, INT4, True, False),
    (7872, 3072, 6144, INT4, True, False), (4096, 3584, 4608, INT4, True, False),
    (16384, 1024, 384, TILED, False, False), (16384, 2048, 3584, TILED, False, True), (16384, 2048, 3712, TILED, False, False),
    (14600, 1024, 3072, TILED, False, False), (16384, 1024, 1024, TILED, False, False), (16384, 896, 896, INT4, False, True),
    (16384, 2048, 1024, INT4, False, False)])
def test_lines(M, N, K, fmt, silu, own):
    w = types.SimpleNamespace(out_features=N, in_features=K, fmt=fmt)
    assert kernels.gemm_many_rows_streams(M, w, silu) is own


@pytest.mark.parametrize("M,n,K,dt,own", [
    (16384, 4112, 4096, torch.bfloat16, True), (16384, 4112, 4224, torch.bfloat16, False), (16384, 4112, 4096, torch.float32, True),
    (16384, 4112, 12288, torch.float32, False), (16384, 2048, 3584, torch.float32, True), (16384, 2048, 3712, torch.float32, False),
    (16384, 2048, 2048, torch.bfloat16, False), (8192, 6144, 512, torch.float32, True), (8192, 8192, 512, torch.float32, False)])
def test_plain_lines(M, n, K, dt, own):
    assert kernels.linear_streams(M, n, K, dt) is own


def test_rotation_lines():
    says = [kernels.rotation_streams(16384, types.SimpleNamespace(out_features=N, in_features=K, fmt=f))
            for N, K, f in ((2048, 2048, TILED), (2048, 2176, TILED), (4096, 6144, TILED), (4096, 6272, TILED), (4096, 1024, INT4), (4096, 1152, INT4))]
    assert says == [True, False, True, False, True, False]


@pytest.mark.gpu
@pytest.mark.parametrize("N,K,quant,silu", [(4096, 512, None, False), (4160, 1536, None, False), (4096, 3584, None, False),
                                            (8192, 4480, None, True), (8192, 2048, "int4", True)])
@pytest.mark.parametrize("M", [4096, 4099])
def test_results(M, N, K, quant, silu):
    from byox_vllm_amd.layers.quant import LinearWeight, interleave_gate_up
    torch.manual_seed(M + N + K)
    dev = "cuda"
    x = torch.randn(M, K, device=dev).bfloat16()
    rows = (torch.randn(N, K, device=dev) * K ** -0.5).bfloat16()
    w = LinearWeight.make(interleave_gate_up(rows) if silu else rows, quant)
    y = x.double() @ (kernels.expand_weight(w, gate_up_rows=silu) if quant else rows).double().t()
    got = kernels.gemm_stream(x, w, None, None, silu).double()
    assert torch.equal(got, kernels.gemm_stream(x, w, None, None, silu).double())
    if kernels.gemm_many_rows_streams(M, w, silu):
        assert torch.equal(got, kernels.gemm(x, w, silu_mul=silu).double())
    if silu:      # gate, up, SiLU and the product are each rounded to bf16; SiLU grows by at most 1.1 times its gate
        g, u = y[:, :N // 2], y[:, N // 2:]
        want = torch.nn.functional.silu(g) * u
        bound = 2.0 ** -8 * (1.1 * g.abs() * u.abs() + 3 * want.abs())
    else:
        want, bound = y, 2.0 ** -8 * y.abs()
    # fp32 sums of K products of unit size and K ** -0.5
    assert ((got - want).abs() <= bound * 1.02 + K * 2.0 ** -22 * (1 + y.abs().max() if silu else 1)).all()
