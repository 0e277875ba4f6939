"""Decode rows and widths that the XCD-resident layers (all but one FP32 row at
d 2048) and the code-table depth steps take beside the CFG pair in FP32 (0.6B) and BF16 (1.7B): one row without
CFG (beside an inactive row of zeros), BF16 weights at d 1024 (half-width inner
pieces), FP32 weights at d 2048 (double-width ones).  Four trunk layers of the
real widths, teacher-forced frames against the float64 oracle; a second prefill
on the same engine and a retired row equal a fresh engine bit for bit.

Bounds: FP32 sums in another order over ~10 projections deep: 2e-5; with BF16
weights the prefix goes through hi + lo activation pairs, 2^-17 each: 1e-4."""

import numpy as np
import pytest

import oracle.model as om
from oracle.generate import Record, generate
from oracle.sampler import apply_masks

pytestmark = pytest.mark.gpu

SHAPES = {"06b": om.Shape(n_layers=4, text_vocab=512, n_codebooks=6),
          "17b": om.Shape(d_model=2048, trunk_inter=6144, n_layers=4, text_vocab=512, n_codebooks=4)}


def _engine(dev, s, w, rows, bf16, frames=8, max_len=160):
    from soraku_amd import GraphFrameEngine
    from soraku_amd.config import DecodeShape

    e = GraphFrameEngine(device=dev, max_cache_len=max_len, cfg_scale=1.5 if rows == 2 else 1.0, batch=rows,
                         state_dict=w, shape=DecodeShape(**{k: getattr(s, k) for k in DecodeShape.__dataclass_fields__}),
                         bf16=bf16, max_frames=frames)
    e.set_temperature(0.9)
    e.set_sampling(sampled=True, top_k=50, top_p=0.95)
    e.set_debug(True)
    return e


def _frames(e, item, codes, u):
    e.prefill_utterances([item])
    if e.graph is None:
        e.capture()
    return np.stack([e.step_frame(mask_eos_q0=True, uniforms=u[f], forced_codes=codes[f], return_logits=True)[1][0]
                     for f in range(len(codes))])


@pytest.mark.parametrize("name,rows,bf16", [("06b", 1, False), ("06b", 1, True), ("06b", 2, True), ("17b", 1, True),
                                            ("17b", 1, False), ("17b", 2, False)])
def test_row_counts_and_widths_match_oracle(hip_device, name, rows, bf16):
    from soraku_amd.synthetic import is_matrix

    s = SHAPES[name]
    w = om.synthetic_weights(s, 21, norm_gain_std=0.1, bias_std=0.02)
    if bf16:
        w = {k: om.round_bf16(v) if is_matrix(k) else v for k, v in w.items()}
    rng = np.random.default_rng(4)
    V, Q, F = s.codebook_size, s.n_codebooks, 3
    items = [(rng.integers(0, 512, n), np.array([1], np.int64), rng.integers(0, V, (p, Q))) for n, p in ((70, 25), (5, 0))]
    codes, u = rng.integers(0, V, (F, Q)), rng.random((F, Q))
    print(f"{name} rows {rows} bf16 {bf16}", flush=True)
    e = _engine(hip_device, s, w, rows, bf16)
    assert e.xcd_layers == (not (name == "17b" and rows == 1 and not bf16))   # that one keeps five kernels per layer
    got = _frames(e, items[0], codes, u)
    m = om.OracleModel(s, w, np.float64)
    rec = Record()
    generate(m, input_ids=items[0][0], prompt_codes=items[0][2], uncond_input_ids=items[0][1] if rows == 2 else None,
             max_new_frames=F, min_new_frames=F, temperature=0.0, cfg_scale=1.5 if rows == 2 else 1.0, batched=True,
             record=rec, forced_codes=codes)
    for f in range(F):
        ref = np.stack([apply_masks(x, q=q, frame_index=f, min_new_frames=F, bos_id=s.bos_id, eos_id=s.eos_id,
                                    pad_id=s.pad_id) for q, x in enumerate(rec.merged[f])]).astype(np.float64)
        fin = np.isfinite(ref)
        assert (np.isfinite(got[f]) == fin).all()
        err = np.abs(got[f][fin] - ref[fin]).max() / np.abs(ref[fin]).max()
        print(f"frame {f}: {err:.2e}", flush=True)
        assert err < (1e-4 if bf16 else 2e-5)
    # the engine again, on a shorter prefix, after a frame with its rows
    # retired: as a fresh engine
    e.retire(0)
    e.step_frame(mask_eos_q0=True, uniforms=u[0], forced_codes=codes[0])
    again = _frames(e, items[1], codes, u)
    e.close()
    e = _engine(hip_device, s, w, rows, bf16)
    fresh = _frames(e, items[1], codes, u)
    e.close()
    np.testing.assert_array_equal(again, fresh)
