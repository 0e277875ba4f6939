"""Every GEMM kernel that a prefill is planned for, at widths that leave partial
tiles and an odd number of 64-byte units of K (d 1056, SwiGLU 3104), and at K
that ends in half a stage with the SwiGLU product (d 160): the second layer's K
and V of every token, and the last tokens' hidden states, against the float64
oracle.  test_host_paths_cpu.py checks that these cases launch every kernel the
plan picks over both trunk shapes.

Bounds, of the largest value: FP32 sums of up to 3,104 products in another order
over two layers 2e-5; with BF16 weights activations are hi + lo pairs, 2^-17 per
value: 1e-4."""

import numpy as np
import pytest

import oracle.model as om

pytestmark = pytest.mark.gpu

SHAPES = {
    "ragged": dict(d_model=1056, n_layers=2, n_q_heads=14, n_kv_heads=7, head_dim=128, trunk_inter=3104),
    "short": dict(d_model=160, n_layers=2, n_q_heads=6, n_kv_heads=3, head_dim=16, trunk_inter=224),
    "06b": dict(n_layers=2),
}
CASES = ([("ragged", t, True) for t in (41, 81, 140, 180, 353, 651, 1101, 1401, 1801, 2201, 2601, 3601)]
         + [("ragged", t, False) for t in (20, 61, 101, 140, 180, 401)]
         + [("short", t, b) for t in (20, 61) for b in (False, True)])


def shape(name):
    return om.Shape(n_codebooks=4, codebook_size=32, text_vocab=512, **SHAPES[name])


def lens_of(total, rows=8):
    """`rows` ragged prefix lengths of `total` tokens."""
    w = np.arange(1, rows + 1)
    lens = np.maximum(2, total * w // w.sum())
    lens[-1] += total - lens.sum()
    return [int(x) for x in lens]


def _weights(s, bf16):
    from soraku_amd.synthetic import is_matrix

    w = om.synthetic_weights(s, 5, norm_gain_std=0.1)
    return {k: om.round_bf16(v) if is_matrix(k) else v for k, v in w.items()} if bf16 else w


def _engine(dev, s, w, n_utts, max_len, bf16):
    from soraku_amd import GraphFrameEngine
    from soraku_amd.config import DecodeShape

    return GraphFrameEngine(device=dev, max_cache_len=max_len, cfg_scale=1.0, batch=1, state_dict=w, n_utts=n_utts,
                            shape=DecodeShape(**{k: getattr(s, k) for k in DecodeShape.__dataclass_fields__}), bf16=bf16)


def _kv(e, layer):
    """K and V of `layer`, FP32 [2][rows][kv heads][max_len][head_dim]."""
    import ctypes as C

    from soraku_amd._lib import check, lib

    hip = C.CDLL("libamdhip64.so.7")
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    out = np.empty((2, e.rows, e.shape.n_kv_heads, e.max_len, e.shape.head_dim), np.float32)
    for kv in (0, 1):
        p = C.c_void_p()
        check(lib().sk_kv_ptr(e._h, layer, kv, C.byref(p)))
        e.synchronize()
        assert hip.hipMemcpy(out[kv].ctypes.data, p, out[kv].nbytes, 2) == 0   # device to host
    return out


def _err(got, ref):
    return float(np.abs(got - ref).max() / np.abs(ref).max())


@pytest.mark.parametrize("name,total,bf16", CASES)
def test_every_planned_gemm_matches_oracle(hip_device, name, total, bf16):
    s = shape(name)
    w = _weights(s, bf16)
    lens = lens_of(total)
    rng = np.random.default_rng(total)
    items = [(rng.integers(0, s.text_vocab, n - 1), None, None) for n in lens]
    print(f"prefill {name} {lens} bf16={bf16}", flush=True)
    e = _engine(hip_device, s, w, len(lens), max(lens) + 4, bf16)
    got = e.prefill_utterances(items).cpu().numpy()
    kv = _kv(e, 1)
    e.close()
    m = om.OracleModel(s, w, np.float64)
    tol = 1e-4 if bf16 else 2e-5
    for r, (text, _, _) in enumerate(items):
        st = om.RowState(s, lens[r] + 1, np.float64)
        ref = m.prefill(st, m.prefix_embeds(text, None))
        errs = _err(got[r], ref), _err(kv[0, r, :, :lens[r]], st.k[1, :, :lens[r]]), _err(kv[1, r, :, :lens[r]], st.v[1, :, :lens[r]])
        assert max(errs) < tol, (r, lens[r], errs)


@pytest.mark.parametrize("bf16", [False, True])
def test_prefix_alone_in_a_batch_and_as_refill(hip_device, bf16):
    """GEMM tiles, K slices and the attention's key split go by the tokens of
    the whole call, so one prefix's results may differ in the last bits with
    what is prefilled beside it, and in no more."""
    s = shape("06b")
    w = _weights(s, bf16)
    rng = np.random.default_rng(3)
    text = rng.integers(0, s.text_vocab, 37)
    others = [(rng.integers(0, s.text_vocab, n), None, None) for n in (201, 90, 333, 150, 18, 260, 77)]
    outs = []
    e = _engine(hip_device, s, w, 1, 400, bf16)
    outs.append((e.prefill_utterances([(text, None, None)]).cpu().numpy()[0], _kv(e, 1)[:, 0, :, :38]))
    e.close()
    e = _engine(hip_device, s, w, 8, 400, bf16)
    outs.append((e.prefill_utterances([(text, None, None)] + others).cpu().numpy()[0], _kv(e, 1)[:, 0, :, :38]))
    e.prefill_utterances([others[0]] + others)
    e.refill({0: (text, None, None)})
    outs.append((e.hidden()[0], _kv(e, 1)[:, 0, :, :38]))
    e.close()
    for hid, kv in outs[1:]:
        print(f"bf16={bf16}: hidden {_err(hid, outs[0][0]):.2e}, K/V {_err(kv, outs[0][1]):.2e}", flush=True)
        assert _err(hid, outs[0][0]) < (1e-4 if bf16 else 2e-5) and _err(kv, outs[0][1]) < (1e-4 if bf16 else 2e-5)
