"""Depth steps of one utterance over the range of vocabularies: code tables up
to V = 3,840 (1, 2, 3, 5 or 8 logits per thread), the launches per codebook
past it, one and two rows, with the XCD-resident layers and with the five
kernels per layer (the frame then ends with an FP32 trunk output).

The codes are the sampler's own: each must be what the oracle draws from the
logits the engine recorded, and those must be the float64 oracle's for the same
codes.  Bounds: FP32 sums in another order over a few projections 2e-5; with
BF16 weights the prefix goes through hi + lo activation pairs, 2^-17 each: 1e-4."""

import numpy as np
import pytest

import oracle.model as om
from oracle.generate import Record, generate
from oracle.sampler import apply_masks, sample

pytestmark = pytest.mark.gpu

TEMP, TOP_K, TOP_P, CFG = 0.9, 50, 0.95, 1.5
WIDTH = {"06b": dict(), "17b": dict(d_model=2048, trunk_inter=6144)}


@pytest.mark.parametrize("name,rows,bf16,V,layers", [
    ("06b", 2, False, 500, True), ("06b", 2, False, 1500, True), ("06b", 2, False, 2560, True),
    ("06b", 2, False, 2561, True), ("06b", 2, False, 3840, True), ("06b", 2, False, 3841, True),
    ("06b", 2, False, 2561, False), ("06b", 1, True, 500, True), ("06b", 1, True, 2051, True),
    ("06b", 1, True, 2561, True), ("06b", 1, True, 2051, False), ("06b", 1, False, 2051, False),
    ("17b", 2, True, 2561, True), ("17b", 1, True, 2051, True), ("17b", 1, True, 2051, False),
    ("17b", 1, False, 2051, False), ("17b", 1, False, 3840, False)])
def test_sampled_frames_match_oracle(hip_device, monkeypatch, name, rows, bf16, V, layers):
    from soraku_amd import GraphFrameEngine
    from soraku_amd.config import DecodeShape
    from soraku_amd.synthetic import is_matrix

    s = om.Shape(n_layers=1, text_vocab=512, n_codebooks=4, codebook_size=V - 3, **WIDTH[name])
    w = om.synthetic_weights(s, 31, norm_gain_std=0.1, bias_std=0.02)
    if bf16:
        w = {k: om.round_bf16(v) if is_matrix(k) else v for k, v in w.items()}
    rng = np.random.default_rng(V + rows)
    text, uncond = rng.integers(0, 512, 11), np.array([1], np.int64)
    F, Q = 3, s.n_codebooks
    u = rng.random((F, Q))
    print(f"{name} rows {rows} bf16 {bf16} V {V} layers {layers}", flush=True)
    if not layers:
        monkeypatch.setenv("SORAKU_XCD_LAYERS", "0")
    e = GraphFrameEngine(device=hip_device, max_cache_len=32, cfg_scale=CFG if rows == 2 else 1.0, batch=rows,
                         state_dict=w, shape=DecodeShape(**{k: getattr(s, k) for k in DecodeShape.__dataclass_fields__}),
                         bf16=bf16, max_frames=8)
    assert e.xcd_layers == layers
    e.set_temperature(TEMP)
    e.set_sampling(sampled=True, top_k=TOP_K, top_p=TOP_P)
    e.set_debug(True)
    e.prefill_utterances([(text, uncond, None)])
    e.capture()
    codes, logits = zip(*(e.step_frame(mask_eos_q0=True, uniforms=u[f], return_logits=True) for f in range(F)))
    e.close()
    codes = np.stack([c.numpy() for c in codes])
    for f in range(F):
        for q in range(Q):
            assert codes[f, q] == sample(logits[f][0][q], temperature=TEMP, top_k=TOP_K, top_p=TOP_P, u=u[f][q]), (f, q)
    rec = Record()
    generate(om.OracleModel(s, w, np.float64), input_ids=text, uncond_input_ids=uncond if rows == 2 else None,
             max_new_frames=F, min_new_frames=F, temperature=0.0, cfg_scale=CFG if rows == 2 else 1.0, batched=True,
             record=rec, forced_codes=codes)
    for f in range(F):
        ref = np.stack([apply_masks(x, q=q, frame_index=f, min_new_frames=F, bos_id=s.bos_id, eos_id=s.eos_id,
                                    pad_id=s.pad_id) for q, x in enumerate(rec.merged[f])]).astype(np.float64)
        fin = np.isfinite(ref)
        assert (np.isfinite(logits[f][0]) == fin).all()
        err = np.abs(logits[f][0][fin] - ref[fin]).max() / np.abs(ref[fin]).max()
        print(f"frame {f}: {err:.2e}", flush=True)
        assert err < (1e-4 if bf16 else 2e-5)
