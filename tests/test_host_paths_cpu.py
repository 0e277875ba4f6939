"""The engine's host side on a stand-in HIP runtime (hip_host_stub.cpp), no GPU:
what a failing call leaves behind, and which kernels a shape is given."""

import os
import subprocess
import sys

import pytest

from conftest import ROOT

HERE = os.path.join(ROOT, "tests")


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    d = tmp_path_factory.mktemp("hip")
    so = str(d / "stub.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "hip_host_stub.cpp"), "-o", so], check=True)

    def run(script, **env):
        f = d / "script.py"
        f.write_text(script)
        r = subprocess.run([sys.executable, os.path.join(HERE, "host_engine.py"), so, str(f)], capture_output=True,
                           text=True, env=dict(os.environ, **env))
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout

    return run


STEP = """
s = TINY
h = engine(s)
for r in range(2):
    assert stage(h, s, r) == 0, error()
assert L.sk_prefill_run(h) == 0 and L.sk_capture(h) == 0, error()
codes = (C.c_int64 * s.n_codebooks)()
logits = (C.c_float * (s.n_codebooks * s.audio_vocab))()
step = lambda: L.sk_step_frame(h, 1, None, None, codes, logits)
calls()
"""


@pytest.mark.parametrize("name,after", [("hipLaunchKernel", 0), ("hipGraphLaunch", 0), ("hipLaunchKernel", 1),
                                        ("hipMemcpyAsync", 0)])
def test_failing_step_waits_for_what_it_queued(host, name, after):
    """A stepped frame that fails after its first launch waits for the stream
    before it returns: that launch reads the pinned buffer which the next step
    fills."""
    host(STEP + f"""
assert L.sk_set_debug(h, 1) == 0 and step() == 0, error()
calls()
stub.stub_fail(b"{name}", {after})
rc = step()
cs = [c[0] for c in calls()]
assert rc == _lib.SK_EHIP, (rc, cs)
text = error()
assert "{name}" in cs and "stub error" in text, (cs, text)
assert cs[-1] == "hipStreamSynchronize", cs
stub.stub_fail(b"", -1)
assert step() == 0, error()
""")


def test_prefix_without_host_memory_is_refused(host):
    """Prefixes are kept in host memory until the prefill runs: where there is
    none, staging and the prefill report it (no C++ exception leaves the C
    interface) and the engine goes on with what it had."""
    host("""
s = TINY
h = engine(s)
for r in range(2):
    assert stage(h, s, r) == 0, error()
stub.stub_new_limit(200)
rc, text = stage(h, s, 1, 3, 30), error()
assert rc == _lib.SK_EHIP and "host memory" in text, (rc, text)
stub.stub_new_limit(-1)
calls()
assert L.sk_prefill_run(h) == 0, error()
tokens = [g[0] for n, g in kernels(calls()) if "pf_embed" in n]
assert tokens == [8], tokens            # two rows of 3 + 1 tokens, as staged before
for r in range(2):
    assert stage(h, s, r, 3, 30) == 0, error()
stub.stub_new_limit(600)
rc, text = L.sk_prefill_run(h), error()
assert rc == _lib.SK_EHIP and "host memory" in text, (rc, text)
stub.stub_new_limit(-1)
assert L.sk_prefill_run(h) == 0, error()
""")


@pytest.mark.parametrize("name,bf16", [("QWEN3_06B", False), ("QWEN3_06B", True), ("QWEN3_17B", False),
                                       ("QWEN3_17B", True)])
def test_code_table_vocabularies(host, name, bf16):
    """Depth steps by code tables for every vocabulary whose sampler fits in
    LDS, with no more logits per thread than it needs."""
    out = host(f"""
import re
for rows in (1, 2):
    for V in (100, 512, 513, 1024, 1025, 1536, 1537, 2051, 2560, 2561, 3840, 3841, 4096):
        s = replace({name}, n_layers=1, n_codebooks=3, codebook_size=V - 3, text_vocab=64)
        h = engine(s, cfg_rows=rows, bf16={bf16})
        calls()
        assert L.sk_capture(h) == 0, error()
        steps = [re.search(r"depth_step_kernelI.*?Li(\\d+)ELi(\\d)ELi\\d+ELi\\d+ELi(\\d)E", n) for n, _ in kernels(calls())]
        steps = [tuple(int(x) for x in m.groups()) for m in steps if m]
        print(rows, V, sorted(set(p for p, m, mode in steps if mode == 2)), sorted(set(m for _, m, _ in steps)))
        L.sk_destroy(h)
""")
    want = {100: 1, 512: 1, 513: 2, 1024: 2, 1025: 3, 1536: 3, 1537: 5, 2051: 5, 2560: 5, 2561: 8, 3840: 8}
    for line in out.splitlines():
        rows, V, rest = line.split(" ", 2)
        n = want.get(int(V))
        assert rest == (f"[{n}] [{rows}]" if n else "[] []"), line


def test_xcd_layers_rule(host):
    """Which engines run the XCD-resident layers."""
    out = host("""
for name, s in (("06b", QWEN3_06B), ("17b", QWEN3_17B)):
    for rows in (1, 2, 3):
        for bf16 in (False, True):
            h = engine(replace(s, n_layers=3, n_codebooks=2, text_vocab=64), n_utts=3 if rows == 3 else 1,
                       cfg_rows=1 if rows == 3 else rows, bf16=bf16)
            print(name, rows, bf16, L.sk_xcd_layers(h))
            L.sk_destroy(h)
""")
    got = {tuple(line.split()[:3]): line.split()[3] for line in out.splitlines()}
    assert len(got) == 12
    for (name, rows, bf16), lx in got.items():
        want = rows == "2" or (rows == "1" and (name == "06b" or bf16 == "True"))
        assert lx == str(int(want)), (name, rows, bf16, lx)


def test_prefill_gemms_have_gpu_cases(host):
    """Every GEMM kernel (epilogue, weight type, tile) that a prefill launches
    at either trunk shape, up to 6,000 tokens, is launched by a case of
    test_gpu_prefill_tiles.py; the short shape's cases reach the half stage."""
    host("""
import re
import test_gpu_prefill_tiles as t

def gemms(shape, lens, bf16):
    h = engine(shape, n_utts=len(lens), cfg_rows=1, max_ctx=max(lens) + 4, bf16=bf16)
    for r, n in enumerate(lens):
        assert stage(h, shape, r, n - 1, 1) == 0, error()
    calls()
    assert L.sk_prefill_run(h) == 0, error()
    names = [re.search(r"gemm_kernelILi(\\d)E.*?(WF32|WBF16)E((?:Li\\d+E)+)", n) for n, _ in kernels(calls())]
    L.sk_destroy(h)
    return {m.groups() for m in names if m}

fields = [f.name for f in dataclasses.fields(QWEN3_06B)]
tested = {}
for name, total, bf16 in t.CASES:
    s = replace(QWEN3_06B, **{f: getattr(t.shape(name), f) for f in fields})
    tested.setdefault(name, set()).update(gemms(s, t.lens_of(total), bf16))
used = set()
for s in (QWEN3_06B, QWEN3_17B):
    for total in list(range(16, 400, 9)) + list(range(400, 6000, 75)):
        for bf16 in (False, True):
            used |= gemms(replace(s, n_layers=1, text_vocab=512), t.lens_of(total), bf16)
assert len(used) >= 28 and used <= tested["ragged"], used - tested["ragged"]
half = {k for k in tested["short"] if k[2].endswith("Li2E")}
assert {k[0] for k in half} == {"0", "1"}, half      # stages of 128 bytes, both epilogues
""")


def test_attention_split_rule(host):
    """Workgroups per (row, KV head) of the many-row attention: one for short
    caches, else as many as fit 256 CUs; 17 to 31 rows two for long caches."""
    out = host("""
for rows, ctx, kv_bf16 in ((6, 256, 0), (6, 257, 0), (8, 640, 0), (8, 513, 1), (12, 640, 0), (16, 640, 0), (32, 65536, 1),
                           (17, 2000, 0), (17, 18432, 0), (17, 18433, 0), (21, 36864, 1), (21, 36865, 1),
                           (22, 6144, 0), (22, 6145, 0), (25, 12288, 1), (25, 12289, 1),
                           (26, 3072, 0), (26, 3073, 0), (31, 6144, 1), (31, 6145, 1)):
    s = replace(QWEN3_06B, n_layers=1, n_codebooks=2, text_vocab=64)
    h = engine(s, n_utts=rows, cfg_rows=1, max_ctx=ctx, kv_bf16=bool(kv_bf16))
    calls()
    assert L.sk_capture(h) == 0, error()
    grids = [g for n, g in kernels(calls()) if "attention_stream_kernel" in n]
    assert len(grids) == 1 and grids[0][1:] == (8, rows), grids
    print(rows, ctx, kv_bf16, grids[0][0])
    L.sk_destroy(h)
""")
    got = [int(line.split()[3]) for line in out.splitlines()]
    assert got == [1, 5, 4, 4, 2, 2, 1, 1, 1, 2, 1, 2, 1, 2, 1, 2, 1, 2, 1, 2], out


@pytest.mark.parametrize("name,after", [("hipMemsetAsync", 0), ("hipMemsetAsync", 2), ("hipLaunchKernel", 5)])
def test_failing_prefill_waits_for_its_table(host, name, after):
    """A prefill that fails after its table's copy was queued waits for the
    stream: the copy reads host memory that goes away with the call."""
    host(f"""
s = TINY
h = engine(s)
for r in range(2):
    assert stage(h, s, r) == 0, error()
calls()
stub.stub_fail(b"{name}", {after})
rc = L.sk_prefill_run(h)
cs = [c[0] for c in calls()]
assert rc == _lib.SK_EHIP and "hipMemcpyAsync" in cs and cs[-1] == "hipStreamSynchronize", (rc, cs)
stub.stub_fail(b"", -1)
assert L.sk_prefill_run(h) == 0, error()   # the rows are still staged
""")


def test_operator_rows_rule(host):
    """Which projections of many rows run as GEMV launches of 4 rows and which
    in one pass of up to 32."""
    out = host("""
p = C.c_void_p(4096)
def run(op, B, N, K, bf16):
    calls()
    dt = int(bf16)
    if op == "bias": rc = L.sk_op_classifier_gemv(None, B, N, K, dt, p, p, p, p)
    elif op == "resid": rc = L.sk_op_down_residual_gemv(None, B, N, K, dt, p, p, p, p)
    else: rc = L.sk_op_swiglu_gemv(None, B, N, K, dt, p, p, p, p)
    assert rc == 0, error()
    return ["one" if "skinny" in n else "gemv" for n, _ in kernels(calls())]
for case in (("bias", 4, 1024, 2048, 0), ("bias", 5, 1024, 2048, 0), ("bias", 5, 1024, 2040, 0), ("bias", 7, 1024, 2048, 0),
             ("resid", 8, 1024, 3072, 0), ("resid", 8, 1536, 3072, 0), ("resid", 5, 1537, 3072, 0), ("resid", 5, 1025, 3080, 0),
             ("resid", 9, 1024, 3072, 0), ("bias", 5, 1024, 4096, 1), ("resid", 5, 1024, 4096, 1), ("resid", 7, 1024, 6144, 1),
             ("resid", 5, 16, 6152, 0), ("swiglu", 6, 1024, 1024, 0), ("swiglu", 6, 1536, 2048, 0), ("swiglu", 6, 1536, 2056, 0),
             ("swiglu", 7, 1024, 4096, 1), ("swiglu", 7, 1024, 4088, 1), ("swiglu", 7, 6144, 2048, 1),
             ("bias", 20, 2051, 1024, 0), ("bias", 40, 2051, 1024, 0)):
    print(*case, *run(*case))
""")
    g, o = "gemv", "one"
    want = [[g], [g, g], [o], [o], [g, g], [g, g], [o], [o], [o], [o], [g, g], [o], [o], [g, g], [g, g], [o], [g, g], [o],
            [o], [o], [o, o]]
    assert [line.split()[5:] for line in out.splitlines()] == want, out
