"""Builds byox_vllm_amd/libnv_hip.so from csrc/*.hip with hipcc for gfx950 (cross-compiles without a GPU).

``build_library()`` compiles what is stale and links every source.  ``ensure(sources)`` is what entry points call that
must work from a fresh checkout: when no library is there it compiles only the named sources (what one model needs)
and links those; the binding (byox_vllm_amd/_C.py) then offers the entry points the library has, and a later full build
replaces it."""

import glob
import os
import subprocess

from byox_vllm_amd import build_check

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "byox_vllm_amd", "csrc")
LIB = os.path.join(ROOT, "byox_vllm_amd", "libnv_hip.so")

# -fno-slp-vectorize: the SLP vectoriser pairs the dequantisation's scalar fp32 FMAs into v_pk_fma_f32, which (unlike
# scalar VALU instructions) does not execute in the shadow of an MFMA on gfx950.  -packed-fp32-ops off: no
# v_pk_{add,mul,fma}_f32 from ordinary float code either.
# No -D flag: the measurement switches of the sources (NV_ABL_* leave one activity out of the GEMM loop and give wrong
# results, NV_STAMP writes cycle stamps, NV_GEMM_WNT / NV_ATTN_DEPTH* change cache policy and pipeline depth) exist
# only in libraries built by scripts/build_variant.py under another file name; the shipped libnv_hip.so is compiled
# with none of them defined.
HIPCC_FLAGS = ["-O3", "-std=c++17", "-fno-slp-vectorize", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
               "--offload-arch=gfx950", "-fPIC"]


def _stale(target, sources):
    if not os.path.exists(target):
        return True
    t = os.path.getmtime(target)
    return any(os.path.getmtime(s) > t for s in sources)


def _headers():
    return glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(ROOT, "include", "*.h"))


def compile_sources(sources, force=False, jobs=None):
    """hipcc -c each stale source (in parallel) -> the object files, whose machine code is looked over where it has to be (build_check.py)."""
    jobs = jobs or max(1, min(16, os.cpu_count() or 1))
    headers = _headers()
    objs, todo = [], []
    for src in sources:
        obj = src[:-4] + ".o"
        objs.append(obj)
        if force or _stale(obj, [src] + headers):
            cmd = ["hipcc"] + HIPCC_FLAGS + ["-c", src, "-o", obj]
            assert not any(a.startswith("-D") for a in cmd)
            todo.append((src, cmd))
    running = []
    while todo or running:
        while todo and len(running) < jobs:
            src, cmd = todo.pop(0)
            running.append((src, subprocess.Popen(cmd, stdout=subprocess.DEVNULL, stderr=subprocess.PIPE)))
        src, p = running.pop(0)
        _, err = p.communicate()
        if p.returncode != 0:
            for _, q in running:
                q.kill()
            raise RuntimeError(f"hipcc failed on {src}:\n{err.decode(errors='replace')[-4000:]}")
        try:
            build_check.check_object(src[:-4] + ".o")
        except Exception:
            os.remove(src[:-4] + ".o")      # not to be linked by a later call
            for _, q in running:
                q.kill()
            raise
    return objs


def link(objs):
    tmp = LIB + f".{os.getpid()}.tmp"
    subprocess.check_call(["hipcc", "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp] + objs)
    os.replace(tmp, LIB)


def build_library(force: bool = False) -> str:
    sources = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    before = {o: os.path.getmtime(o) for o in (s[:-4] + ".o" for s in sources) if os.path.exists(o)}
    objs = compile_sources(sources, force)
    changed = any(before.get(o) != os.path.getmtime(o) for o in objs)
    if force or changed or _stale(LIB, objs) or not _has_all(sources):
        link(objs)
    if os.path.exists(_marker()):
        os.remove(_marker())      # the note of a partial build: this library is whole
    return LIB


def _marker():
    return LIB + ".sources"


def _has_all(sources) -> bool:
    """Was the library at hand linked from (at least) these sources?"""
    try:
        with open(_marker()) as f:
            have = set(f.read().split())
    except OSError:
        return True          # a library without a note is a full build
    return {os.path.basename(s) for s in sources} <= have


def _with_needed(names):
    """``names`` and what their sources call in others."""
    needs = {"linear": ("linear_deep", "linear_eight", "linear_split")}
    return list(dict.fromkeys(m for n in names for m in (n,) + needs.get(n, ())))


def ensure(names) -> str:
    """Make sure a library with the kernels of csrc/<name>.hip, name in ``names``, is there.  An existing library is
    used as it is when it holds them and none of them is stale; otherwise exactly these sources are compiled and
    linked (beside whatever objects of an earlier partial build are current)."""
    sources = [os.path.join(CSRC, n + ".hip") for n in _with_needed(names)]
    if os.path.exists(LIB) and _has_all(sources) and not _stale(LIB, sources + _headers()):
        return LIB
    objs = compile_sources(sources)
    have = set()
    if os.path.exists(_marker()):
        with open(_marker()) as f:
            have = set(f.read().split())
    # keep what an earlier partial build already compiled, if still current
    for other in sorted(have - {os.path.basename(s) for s in sources}):
        src = os.path.join(CSRC, other)
        obj = src[:-4] + ".o"
        if os.path.exists(src) and os.path.exists(obj) and not _stale(obj, [src] + _headers()):
            sources.append(src)
            objs.append(obj)
    link(objs)
    with open(_marker(), "w") as f:
        f.write("\n".join(sorted(os.path.basename(s) for s in sources)) + "\n")
    return LIB
