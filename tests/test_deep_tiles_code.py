"""The machine code of the kernels of csrc/stream_deep.h, whose accumulators are accumulation registers by number: the compiler, which does
not know what is in them, must not use them, and the wait states between its instructions and the matrix cores' must be there."""

import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "byox_vllm_amd", "csrc")
LLVM = "/opt/rocm/llvm/bin"


def registers(text):
    out = set()
    for lo, hi, one in re.findall(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b", text):
        out |= set(range(int(lo), int(hi) + 1)) if lo else {int(one)}
    return out


@pytest.mark.parametrize("source", ["gemm_stream", "linear_deep", "qk_stream"])
def test_accumulators_are_left_alone(source, tmp_path):
    obj = os.path.join(CSRC, source + ".o")
    tools = [os.path.join(LLVM, t) for t in ("llvm-objcopy", "clang-offload-bundler", "llvm-objdump")]
    if not os.path.exists(obj) or not all(os.path.exists(t) for t in tools):
        pytest.skip("no object file or no tools to read it")
    fat, code = str(tmp_path / "fat"), str(tmp_path / "code")
    subprocess.check_call([tools[0], "--dump-section", f".hip_fatbin={fat}", obj, str(tmp_path / "copy")])
    subprocess.check_call([tools[1], "--unbundle", "--type=o", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--input={fat}", f"--output={code}"])
    kernels, products, name, since, before = set(), 0, "", 99, []
    for line in subprocess.run([tools[2], "-d", "--no-show-raw-insn", code], capture_output=True, text=True, check=True).stdout.splitlines():
        if head := re.match(r"^[0-9a-f]+ <(\S+)>:", line):
            name, since, before = head.group(1), 99, []
            continue
        text = line.split("//")[0].strip()
        if "stream_deep_kernel" not in name or not text:
            continue
        kernels.add(name)
        assert not text.startswith(("v_accvgpr_write", "v_accvgpr_mov")), (name, text)
        if text.startswith("v_mfma"):
            products += 1
            since = 0
            use = registers(text.split(",", 1)[1])
            for earlier in before[-2:]:
                if earlier.startswith("v_") and not earlier.startswith("v_mfma"):
                    assert not registers(earlier.split(",")[0]) & use, (name, earlier, text)
        elif text.startswith("s_nop"):
            since += int(text.split()[1], 0) + 1
        elif text.startswith("v_accvgpr_read"):
            assert since >= 19, (name, text)          # a product of eight passes, and what is behind it in the pipe
        before.append(text)
    assert kernels and products >= 576 * len(kernels)
