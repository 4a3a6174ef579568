"""The machine code of the kernels of csrc/stream_deep.h, whose accumulators are accumulation registers by number: byox_vllm_amd/build_check.py,
through which the build refuses an object, on the objects at hand and on listings with a mistake in them."""

import os

import pytest

from byox_vllm_amd import build_check

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "byox_vllm_amd", "csrc")
TOOLS = [os.path.join(build_check.LLVM, t) for t in ("llvm-objcopy", "clang-offload-bundler", "llvm-objdump")]


@pytest.mark.parametrize("source", ["gemm_stream", "linear_deep", "qk_stream"])
def test_accumulators_are_left_alone(source):
    obj = os.path.join(CSRC, source + ".o")
    if not os.path.exists(obj) or not all(os.path.exists(t) for t in TOOLS):
        pytest.skip("no object file or no tools to read it")
    assert build_check.has_deep_tiles(obj)
    build_check.check_object(obj)


GOOD = """0000000000001000 <_Z18stream_deep_kernelI7RowsJob>:
\tv_accvgpr_read_b32 v9, a7                                  // 000000001000: D3D84009
\tds_read_b128 v[16:19], v3 offset:2048
\tv_add_u32_e32 v40, v2, v3
\ts_nop 0
\tv_mfma_f32_16x16x32_bf16 a[0:3], v[16:19], v[20:23], 0
\tv_mfma_f32_16x16x32_f16 a[252:255], v[16:19], v[20:23], a[252:255]
\ts_nop 15
\ts_nop 7
\tv_accvgpr_read_b32 v12, a252
\ts_cbranch_scc0 65500
"""


@pytest.mark.parametrize("line,says", [
    ("", None), ("v_accvgpr_write_b32 a3, v1", "names"), ("v_accvgpr_mov_b32 a3, a4", "names"), ("ds_read_b128 a[4:7], v1", "names"),
    ("global_load_dwordx4 a[8:11], v[2:3], off", "names"), ("global_load_dword a8, v1, s[2:3]", "names"),
    ("global_store_dwordx4 v[2:3], a[0:3], off", "names"), ("v_mfma_f32_16x16x4_f32 a[0:3], v1, v2, a[0:3]", "not a product"),
    ("v_mfma_f32_16x16x32_bf16 a[0:3], v[4:7], v[8:11], a[4:7]", "not a product"),
    ("v_mfma_f32_16x16x32_bf16 a[2:5], v[4:7], v[8:11], a[2:5]", "not a product"),
    ("v_mfma_f32_16x16x32_bf16 a[0:3], a[4:7], v[8:11], a[0:3]", "not a product"),
    ("v_mfma_f32_16x16x32_bf16 v[0:3], v[4:7], v[8:11], 0", "not a product"),
    ("scratch_store_dwordx4 off, v[0:3], s32", "spilled"), ("scratch_load_dword a1, off, s32", "names"),
    ("v_add_f32_e32 v20, v1, v2", "too close"), ("s_nop 0\n\tv_mov_b32_e32 v5, 0xa5", None), ("s_mov_b32 s5, 0xa12", None)])
def test_what_is_refused(line, says):
    """``line`` ahead of the second product."""
    text = GOOD.replace("\tv_mfma_f32_16x16x32_f16", (f"\t{line}\n" if line else "") + "\tv_mfma_f32_16x16x32_f16")
    kernels, products, faults = build_check.accumulator_faults(text)
    assert len(kernels) == 1 and products >= 2
    assert any(says in f for f in faults) if says else not faults, faults
    other = text.replace("stream_deep_kernel", "stream_tiles_kernel")
    assert build_check.accumulator_faults(other) == (set(), 0, [])


def test_results_read_too_early():
    _, _, faults = build_check.accumulator_faults(GOOD.replace("\ts_nop 7\n", ""))
    assert len(faults) == 1 and "16 wait states" in faults[0]


def test_a_refused_object_is_not_linked(tmp_path, monkeypatch):
    from byox_vllm_amd import build
    src = tmp_path / "x.hip"
    src.write_text("// nothing")

    class Compiler:
        returncode = 0

        def __init__(self, cmd, **_):
            open(cmd[-1], "wb").write(build_check.KERNEL.encode())

        def communicate(self):
            return b"", b""
    monkeypatch.setattr(build.subprocess, "Popen", Compiler)
    monkeypatch.setattr(build_check, "listing", lambda obj: GOOD.replace("a252", "a252\n\tv_accvgpr_write_b32 a3, v1"))
    with pytest.raises(RuntimeError, match="names an accumulator"):
        build.compile_sources([str(src)])
    assert not (tmp_path / "x.o").exists()
