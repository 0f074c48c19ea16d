"""The build targets gfx950 and nothing else (CPU only, no GPU needed).

The kernels rely on gfx950 specifics -- MFMA shapes, LDS size, the 8-XCD
workgroup mapping and the hardware ordering the cross-workgroup split-K
exchange depends on -- so the recipe must name that one target, every
compile must disable packed-fp32 VALU ops, and a device compile for any other
target must stop at the guard in nibble_common.h.
"""
from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

from nibblegemm_amd import build

HAVE_HIPCC = os.path.exists(build._hipcc()) or shutil.which("hipcc") is not None


def _arch_flags(flags):
    return [f for f in flags if f.startswith("--offload-arch") or f.startswith("--amdgpu-target")]


def test_recipe_names_gfx950_only():
    assert build.ARCH == "gfx950"
    assert _arch_flags(build.HIPCC_FLAGS) == ["--offload-arch=gfx950"]
    i = build.HIPCC_FLAGS.index("-packed-fp32-ops")
    assert build.HIPCC_FLAGS[i - 3:i] == ["-Xclang", "-target-feature", "-Xclang"]


def test_every_hip_source_is_built_and_includes_the_guard():
    on_disk = sorted(f for f in os.listdir(build.CSRC) if f.endswith(".hip"))
    assert sorted(build.HIP_SOURCES) == on_disk
    for src in on_disk:
        with open(os.path.join(build.CSRC, src)) as f:
            text = f.read()
        assert '#include "nibble_common.h"' in text, src


def _device_compile(tmp_path, arch):
    src = tmp_path / "guard.hip"
    src.write_text('#include "nibble_common.h"\n__global__ void k(int* p) { *p = 1; }\n')
    cmd = [build._hipcc(), "-std=c++17", f"--offload-arch={arch}", "--cuda-device-only", "-c",
           "-I", build.CSRC, "-I", build.INCLUDE, str(src), "-o", str(tmp_path / "guard.o")]
    return subprocess.run(cmd, capture_output=True, text=True, timeout=300)


@pytest.mark.skipif(not HAVE_HIPCC, reason="hipcc not installed")
def test_guard_rejects_another_target(tmp_path):
    r = _device_compile(tmp_path, "gfx942")
    assert r.returncode != 0
    assert "built for gfx950 only" in r.stderr


@pytest.mark.skipif(not HAVE_HIPCC, reason="hipcc not installed")
def test_guard_passes_gfx950(tmp_path):
    r = _device_compile(tmp_path, "gfx950")
    assert r.returncode == 0, r.stderr


OBJDUMP = os.path.join(os.path.dirname(os.path.dirname(build._hipcc())), "llvm", "bin", "llvm-objdump")


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="llvm-objdump not installed")
def test_direct_kernel_waits_match_its_loads(tmp_path):
    """The prefill kernel waits for its copies by count: its loop lets a step's
    loads stay in flight (COPIES copies, 4 word loads, a scale load), and is
    right only if the compiler emits exactly those between one barrier and the
    next.  Counted in the built code, for every tile form: before the first
    barrier, before the loop's first, between its four, and from its last to
    the branch back."""
    lib = shutil.copy(build.LIB, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=tmp_path, capture_output=True, check=True)
    objects = [p for p in sorted(tmp_path.iterdir())
               if "gfx950" in p.name and b"gemm_direct_kernel" in p.read_bytes()]
    assert len(objects) == 1
    text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(objects[0])], capture_output=True,
                          text=True, check=True).stdout
    parts = re.split(r"\n[0-9a-f]+ <([^>]+)>:\n", text)
    forms = 0
    for name, body in zip(parts[1::2], parts[2::2]):
        form = re.search(r"gemm_direct_kernelILi(\d+)ELi(\d+)ELi(\d+)E", name)
        if form is None:
            continue
        forms += 1
        tm, wn = int(form[1]), int(form[3])
        copies = 32 * tm // 8 // wn
        words, part = 5, copies // 4
        step = copies + words
        counts, waits, n, wait = [], [], 0, None
        for line in body.splitlines():
            op = line.split("//")[0].strip()
            if re.match(r"(buffer|global|flat|scratch)_", op):
                n += 1
            elif op.startswith("s_waitcnt") and "vmcnt" in op:
                wait = int(re.search(r"vmcnt\((\d+)\)", op)[1])
            elif op.startswith("s_barrier") and len(counts) < 5:
                counts.append(n)
                waits.append(wait)
                n = 0
            elif op.startswith("s_cbranch") and len(counts) == 5:
                break  # the loop's: back to its first slice
        assert waits == [step + 2 * words + part] + [step] * 4, name
        assert counts == [4 * words + 2 * copies + part, step - 2 - part, step, step, step], name
        assert n == 2 + part, name
    assert forms == 2 * 16  # tile forms and groups
