"""Registers of the built kernels, read from the library's own metadata: a
kernel that spills them to scratch memory pays for it on every launch."""

import os
import re
import subprocess

from conftest import PKG

LLVM = "/opt/rocm/llvm/bin/"
LIB = os.path.join(PKG, "soraku_amd", "libsoraku_mi355x.so")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
# The 1.7B pair's MLP half with FP32 weights, whose rows do not fit in the registers.
SPILLS = r"lx_mlp8_kernelI.*WF32.*Li2048ELi6144E"


def _kernels(tmp_path):
    fat, out = tmp_path / "fat", {}
    subprocess.run([LLVM + "llvm-objcopy", "--dump-section", f".hip_fatbin={fat}", LIB, str(tmp_path / "x")], check=True)
    for i, part in enumerate(fat.read_bytes().split(MAGIC)[1:]):
        src, obj = tmp_path / f"b{i}", tmp_path / f"b{i}.o"
        src.write_bytes(MAGIC + part)
        subprocess.run([LLVM + "clang-offload-bundler", "--unbundle", "--type=o", f"--input={src}", f"--output={obj}",
                        "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
        notes = subprocess.run([LLVM + "llvm-readelf", "--notes", str(obj)], capture_output=True, text=True, check=True)
        for block in re.split(r"\n  - \.a", notes.stdout)[1:]:
            field = dict(re.findall(r"\.(name|vgpr_spill_count|private_segment_fixed_size):\s+(\S+)", block))
            out[field["name"]] = (int(field["vgpr_spill_count"]), int(field["private_segment_fixed_size"]))
    return out


def test_kernels_do_not_spill(tmp_path):
    kernels = _kernels(tmp_path)
    assert len(kernels) > 500 and any("skinny_kernel" in k for k in kernels)
    bad = {k: v for k, v in kernels.items() if v != (0, 0) and not re.search(SPILLS, k)}
    assert not bad, bad
