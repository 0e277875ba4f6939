"""Values without a finite number on the way through the trunk: a codebook row
that holds NaN, infinity or a number past the fixed-point residual stream's
range reaches that frame's later logits and every later frame's as NaN, with the
XCD-resident layers as with the five kernels per layer (where the number, still
finite in FP32, stays finite), and a new prefill starts clean."""

import numpy as np
import pytest

import oracle.model as om

pytestmark = pytest.mark.gpu

BAD = 7   # the code whose row of codebook 0 holds the value
WIDTH = {"06b": dict(), "17b": dict(d_model=2048, trunk_inter=6144)}


@pytest.mark.parametrize("name,rows,bf16,layers", [("06b", 1, False, True), ("06b", 1, True, True),
                                                   ("06b", 2, False, True), ("06b", 1, False, False),
                                                   ("17b", 1, True, True), ("17b", 2, True, True)])
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf, 3e9])
def test_bad_value_reaches_the_logits(hip_device, monkeypatch, name, rows, bf16, layers, value):
    from soraku_amd import GraphFrameEngine
    from soraku_amd.config import DecodeShape

    s = om.Shape(n_layers=3, text_vocab=512, n_codebooks=4, codebook_size=61, tie_audio_head=False, **WIDTH[name])
    w = om.synthetic_weights(s, 17, norm_gain_std=0.1, bias_std=0.02)
    w["audio_codebooks.table"][0, BAD, 5] = value
    rng = np.random.default_rng(8)
    item = (rng.integers(0, 512, 9), np.array([1], np.int64), None)
    codes = rng.integers(BAD + 1, 61, (4, 4))
    print(f"{name} rows {rows} bf16 {bf16} layers {layers} value {value}", flush=True)
    if not layers:
        monkeypatch.setenv("SORAKU_XCD_LAYERS", "0")
    e = GraphFrameEngine(device=hip_device, max_cache_len=32, cfg_scale=1.5 if rows == 2 else 1.0, batch=rows,
                         state_dict=w, shape=DecodeShape(**{k: getattr(s, k) for k in DecodeShape.__dataclass_fields__}),
                         bf16=bf16, max_frames=8)
    assert e.xcd_layers == layers
    e.set_debug(True)
    kept = [v for v in range(s.audio_vocab) if v not in (s.bos_id, s.eos_id, s.pad_id)]

    def run(forced):
        e.prefill_utterances([item])
        if e.graph is None:
            e.capture()
        return np.stack([e.step_frame(mask_eos_q0=True, forced_codes=f, return_logits=True)[1][0] for f in forced])

    clean = run(codes)
    assert np.isfinite(clean[:, :, kept]).all()
    bad = codes.copy()
    bad[1, 0] = BAD
    got = run(bad)[:, :, kept]
    assert np.array_equal(got[0], clean[0][:, kept]) and np.array_equal(got[1, 0], clean[1, 0][kept])
    if layers or not np.isfinite(value):
        assert np.isnan(got[2:]).all()
    else:
        assert np.isfinite(got).all()
    if not np.isfinite(value):
        assert np.isnan(got[1, 1:]).all()   # the frame's own prefix holds it
    assert np.array_equal(run(codes), clean, equal_nan=True)
    e.close()
