"""What the kernels of csrc/stream_deep.h need of their machine code.  Their accumulators are accumulation registers by number, of whose
contents the compiler knows nothing: no instruction but the products and the reads of their results may name one, and the wait states
that the compiler would put between its own products and their neighbours have to be there.  The build refuses an object that breaks this."""

import os
import re
import subprocess
import tempfile

KERNEL = "stream_deep_kernel"
LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")
_ACC = re.compile(r"\ba(?:\d+|\[\d+:\d+\])(?![\w\[])")
_PRODUCT = re.compile(r"v_mfma_f32_16x16x32_(?:bf16|f16) a\[(\d+):(\d+)\], v\[\d+:\d+\], v\[\d+:\d+\], (0|a\[(\d+):(\d+)\])$")
_READ = re.compile(r"v_accvgpr_read_b32 v\d+, a\d+$")


def _registers(text):
    out = set()
    for lo, hi, one in re.findall(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b", text):
        out |= set(range(int(lo), int(hi) + 1)) if lo else {int(one)}
    return out


def accumulator_faults(listing):
    """``listing``: llvm-objdump -d of a code object -> (its kernels of stream_deep.h, their products, what is wrong with them)."""
    kernels, products, faults = set(), 0, []
    name, since, before = "", 99, []
    for line in listing.splitlines():
        if head := re.match(r"^[0-9a-f]+ <(\S+)>:", line):
            name, since, before = head.group(1), 99, []
            continue
        text = line.split("//")[0].strip()
        if KERNEL not in name or not text:
            continue
        kernels.add(name)
        if text.startswith("scratch_"):
            faults.append(f"{name}: {text}: registers spilled")
        if text.startswith("v_mfma"):
            products += 1
            since = 0
            form = _PRODUCT.match(text)
            if not form or int(form[1]) % 4 or int(form[2]) != int(form[1]) + 3 or (form[3] != "0" and form.group(4, 5) != form.group(1, 2)):
                faults.append(f"{name}: {text}: not a product of the source's")
            use = _registers(text.split(",", 1)[1])
            for earlier in before[-2:]:
                if earlier.startswith("v_") and not earlier.startswith("v_mfma") and _registers(earlier.split(",")[0]) & use:
                    faults.append(f"{name}: {earlier}: too close to {text}")
        elif text.startswith("s_nop"):
            since += int(text.split()[1], 0) + 1
        elif text.startswith("v_accvgpr_read"):
            if since < 19:      # a product of eight passes, and what is behind it in the pipe
                faults.append(f"{name}: {text}: {since} wait states behind a product")
        if not text.startswith("v_mfma") and _ACC.search(text) and not _READ.match(text):
            faults.append(f"{name}: {text}: names an accumulator")
        before.append(text)
    return kernels, products, faults


def listing(obj):
    """The gfx950 code of an object file of hipcc's, disassembled."""
    tools = [os.path.join(LLVM, t) for t in ("llvm-objcopy", "clang-offload-bundler", "llvm-objdump")]
    with tempfile.TemporaryDirectory() as d:
        fat, code = os.path.join(d, "fat"), os.path.join(d, "code")
        subprocess.check_call([tools[0], "--dump-section", f".hip_fatbin={fat}", obj, os.path.join(d, "copy")])
        subprocess.check_call([tools[1], "--unbundle", "--type=o", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--input={fat}",
                               f"--output={code}"])
        return subprocess.run([tools[2], "-d", "--no-show-raw-insn", code], capture_output=True, text=True, check=True).stdout


def has_deep_tiles(obj):
    with open(obj, "rb") as f:
        return KERNEL.encode() in f.read()


def check_object(obj):
    """Raises if ``obj`` has kernels of stream_deep.h whose accumulators something else may touch."""
    if not has_deep_tiles(obj):
        return
    kernels, products, faults = accumulator_faults(listing(obj))
    if not kernels or products < 576 * len(kernels):
        faults.append(f"{len(kernels)} kernels with {products} products: not all of them were read")
    if faults:
        raise RuntimeError(f"{os.path.basename(obj)}: {len(faults)} instructions against stream_deep.h's use of accumulation registers:\n"
                           + "\n".join(faults[:20]))
