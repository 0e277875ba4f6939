"""An engine on the stand-in HIP runtime (hip_host_stub.cpp), in a process of
its own: python host_engine.py STUB.so SCRIPT runs SCRIPT with the names below.
Weights are addresses that nothing reads; kernels are only written down."""

import ctypes as C
import dataclasses
import sys

stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)   # before the library: its definitions come first
stub.stub_calls.restype = C.c_char_p
stub.stub_new_limit.argtypes = [C.c_long]

from conftest import PKG  # noqa: E402,F401
from soraku_amd import _lib  # noqa: E402
from soraku_amd.config import QWEN3_06B, QWEN3_17B, TINY, to_sk_config  # noqa: E402,F401
from soraku_amd.synthetic import is_matrix, weight_shapes  # noqa: E402

L = _lib.lib()


def calls():
    """The calls since the last look, one list of words each."""
    out = [c.split() for c in stub.stub_calls().decode().splitlines()]
    stub.stub_clear()
    return out


def kernels(cs):
    """(demangled-enough name, grid) of the launches among calls cs."""
    return [(c[5], tuple(int(x) for x in c[1:4])) for c in cs if c[0] == "hipLaunchKernel"]


def engine(shape, *, n_utts=1, cfg_rows=2, max_ctx=64, bf16=False, kv_bf16=False, max_frames=8):
    cfg = to_sk_config(shape, n_utts=n_utts, cfg_rows=cfg_rows, max_ctx=max_ctx, max_frames=max_frames, bf16=bf16,
                       kv_bf16=kv_bf16)
    h = C.c_void_p()
    _lib.check(L.sk_create(C.byref(cfg), None, C.byref(h)))
    for key, shp in weight_shapes(shape).items():
        dt = _lib.SK_BF16 if bf16 and is_matrix(key) else _lib.SK_F32
        _lib.check(L.sk_bind_weight(h, key.encode(), C.c_void_p(4096), dt, (C.c_int64 * len(shp))(*shp), len(shp)))
    return h


def stage(h, shape, row, n_text=3, n_frames=1):
    ids = (C.c_int64 * n_text)(*([1] * n_text))
    codes = (C.c_int64 * (n_frames * shape.n_codebooks))()
    return L.sk_prefill_row(h, row, ids, n_text, codes, n_frames)


def error():
    return L.sk_last_error().decode()


replace = dataclasses.replace
exec(compile(open(sys.argv[2]).read(), sys.argv[2], "exec"))
