"""The prefill GEMM's device code and tile rule, checked without a GPU: small
programs around csrc/sk_gemm.h are compiled here (gfx950 assembly, or the host
side run on the CPU)."""

import os
import re
import subprocess

import pytest

from conftest import PKG, ROOT

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-w", "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(PKG, "csrc")]


def _hipcc(tmp_path, text, *args):
    src = tmp_path / "t.hip"
    src.write_text(text)
    out = tmp_path / "t.out"
    r = subprocess.run([HIPCC, *FLAGS, *args, str(src), "-o", str(out)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return out


@pytest.mark.parametrize("use", ["__builtin_amdgcn_s_sendmsg(1, v);",
                                 "__builtin_amdgcn_global_load_lds((gv*)(g + threadIdx.x * 4), (lv*)(lds + 1024), 4, 0, 0);"])
def test_lds_load_declares_m0(tmp_path, use):
    """A value kept in M0 across lds_load16 (which puts its LDS address there)
    is set again before its next use."""
    s = _hipcc(tmp_path, """
#include "sk_gemm.h"
typedef __attribute__((address_space(1))) const void gv;
typedef __attribute__((address_space(3))) void lv;
__global__ void k(const char* g, float* out, int v) {
  __shared__ __attribute__((aligned(1024))) char lds[2048];
  %s
  sk::lds_load16(g, threadIdx.x * 16, lds);
  %s
  out[threadIdx.x] = lds[threadIdx.x];
}
""" % (use, use), "--offload-device-only", "-S").read_text()
    body = re.search(r"^_Z1kPKcPfi:(.*?)s_endpgm", s, re.S | re.M).group(1)
    after = body[body.index("global_load_lds_dwordx4"):]
    after = after[:re.search(r"s_sendmsg|global_load_lds_dword ", after).start()]
    assert re.search(r"s_\w+ m0,", after), body


def test_plan_evaluates_every_tile_for_short_k(tmp_path):
    """K of fewer than four 64-byte units still gets the tile with the smallest
    estimate, in one slice (not whichever comes first in the table)."""
    exe = _hipcc(tmp_path, """
#include <stdio.h>
#include "sk_gemm.h"
int main() {
  for (int bf = 0; bf < 2; ++bf)
    for (int sw = 0; sw < 2; ++sw)
      for (int K : {32, 64, 96, 128})
        for (int M : {2, 40, 300, 5000}) {
          const sk::GemmPlan p = sk::plan_gemm(bf, sw, M, 160, K, 16);
          const sk::GemmTile t = bf ? sk::GEMM_BF16[p.tile] : sk::GEMM_F32[p.tile];
          printf("%d %d %d %d %d %d %d %d\\n", bf, sw, K, M, t.bm, t.bn, (int)t.swiglu, p.ksplit);
        }
}
""", "--offload-host-only")
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout
    rows = [tuple(int(x) for x in line.split()) for line in out.splitlines()]
    assert len(rows) == 64
    for bf, sw, K, M, bm, bn, ok, ks in rows:
        assert ks == 1 or K * (2 if bf else 4) >= 4 * 64 * ks, (bf, sw, K, M, ks)
        assert ok or not sw
        if M <= 40:
            assert bm <= 64 and bn <= 128, (bf, sw, K, M, bm, bn)   # not a tile 4 times the rows
