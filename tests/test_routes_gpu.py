"""Which launch a call of prefill or decode size takes, on both sides of each line that was drawn from measurements, and that the result
is the same kind of number there: within roundings of float64 on either route."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


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
