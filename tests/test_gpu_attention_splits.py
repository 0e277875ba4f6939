"""Many-row decode attention on both sides of its rule for one or several
workgroups per (row, KV head): the KV capacity at which one takes a row whole,
and row counts whose workgroups just fit the 256 CUs.  Four trunk layers of the
0.6B widths, ragged prefixes long enough that every split holds tokens,
teacher-forced frames against the float64 oracle.

Bounds: FP32 sums in another order over ~10 projections deep: 2e-5.  A BF16
cache rounds K and V (2^-9 each): the two capacities against each other, whose
few FP32 differences may move a rounding of the appended tokens: 1e-3."""

import numpy as np
import pytest

import oracle.model as om
from oracle.generate import Record, generate
from oracle.sampler import apply_masks

pytestmark = pytest.mark.gpu

S = om.Shape(n_layers=4, text_vocab=512, n_codebooks=4)
F = 3


def _weights():
    return om.synthetic_weights(S, 23, norm_gain_std=0.1, bias_std=0.02)


def _inputs(utts):
    rng = np.random.default_rng(6)
    V, Q = S.codebook_size, S.n_codebooks
    items = [(rng.integers(0, 512, 20 + 9 * i), np.array([1], np.int64), rng.integers(0, V, (180 - 17 * i, Q)))
             for i in range(utts)]
    return items, rng.integers(0, V, (F, utts, Q)), rng.random((F, utts, Q))


def _run(dev, w, utts, max_len, items, codes, u, bf16=False, shape=S):
    from soraku_amd import GraphFrameEngine
    from soraku_amd.config import DecodeShape

    e = GraphFrameEngine(device=dev, max_cache_len=max_len, cfg_scale=1.5, batch=2, state_dict=w,
                         shape=DecodeShape(**{k: getattr(shape, k) for k in DecodeShape.__dataclass_fields__}),
                         n_utts=utts, bf16=bf16, kv_bf16=bf16, max_frames=8)
    e.set_temperature(0.9)
    e.set_sampling(sampled=True, top_k=50, top_p=0.95)
    e.set_debug(True)
    e.prefill_utterances(items)
    e.capture()
    out = np.stack([e.step_frame(mask_eos_q0=True, uniforms=u[f], forced_codes=codes[f], return_logits=True)[1]
                    for f in range(F)])
    e.close()
    return out


@pytest.mark.parametrize("utts,max_len", [(3, 256), (3, 257), (4, 256), (4, 257), (4, 1100), (5, 640), (6, 640), (9, 640)])
def test_split_rule_matches_oracle(hip_device, utts, max_len):
    w = _weights()
    items, codes, u = _inputs(utts)
    print(f"utts {utts} capacity {max_len}", flush=True)
    got = _run(hip_device, w, utts, max_len, items, codes, u)
    m = om.OracleModel(S, w, np.float64)
    for i in (0, utts - 1):
        rec = Record()
        generate(m, input_ids=items[i][0], prompt_codes=items[i][2], uncond_input_ids=items[i][1], max_new_frames=F,
                 min_new_frames=F, temperature=0.0, cfg_scale=1.5, batched=True, record=rec, forced_codes=codes[:, i])
        for f in range(F):
            ref = np.stack([apply_masks(x, q=q, frame_index=f, min_new_frames=F, bos_id=S.bos_id, eos_id=S.eos_id,
                                        pad_id=S.pad_id) for q, x in enumerate(rec.merged[f])]).astype(np.float64)
            fin = np.isfinite(ref)
            assert (np.isfinite(got[f, i]) == fin).all()
            err = np.abs(got[f, i][fin] - ref[fin]).max() / np.abs(ref[fin]).max()
            print(f"utterance {i} frame {f}: {err:.2e}", flush=True)
            assert err < 2e-5


def test_split_rule_bf16_cache(hip_device):
    w = _weights()
    items, codes, u = _inputs(4)
    one, split = (_run(hip_device, w, 4, n, items, codes, u, bf16=True) for n in (512, 513))
    fin = np.isfinite(one)
    assert (np.isfinite(split) == fin).all()
    assert np.abs(one[fin] - split[fin]).max() < 1e-3 * np.abs(one[fin]).max()


@pytest.mark.parametrize("utts,max_len", [(9, 18500), (11, 6100), (11, 6200), (14, 3000), (14, 3100)])
def test_two_splits_for_long_caches_match_oracle(hip_device, utts, max_len):
    """18, 22 and 28 rows on both sides of the capacity from which two
    workgroups share a row (18 rows: past it)."""
    s = om.Shape(n_layers=1, text_vocab=512, n_codebooks=4)
    w = om.synthetic_weights(s, 23, norm_gain_std=0.1, bias_std=0.02)
    rng = np.random.default_rng(7)
    items = [(rng.integers(0, 512, 20 + 9 * i), np.array([1], np.int64), rng.integers(0, s.codebook_size, (190 - 13 * i, 4)))
             for i in range(utts)]
    codes, u = rng.integers(0, s.codebook_size, (F, utts, 4)), rng.random((F, utts, 4))
    print(f"utts {utts} capacity {max_len}", flush=True)
    got = _run(hip_device, w, utts, max_len, items, codes, u, shape=s)
    m = om.OracleModel(s, w, np.float64)
    for i in (0, utts - 1):
        rec = Record()
        generate(m, input_ids=items[i][0], prompt_codes=items[i][2], uncond_input_ids=items[i][1], max_new_frames=F,
                 min_new_frames=F, temperature=0.0, cfg_scale=1.5, batched=True, record=rec, forced_codes=codes[:, i])
        for f in range(F):
            ref = np.stack([apply_masks(x, q=q, frame_index=f, min_new_frames=F, bos_id=s.bos_id, eos_id=s.eos_id,
                                        pad_id=s.pad_id) for q, x in enumerate(rec.merged[f])]).astype(np.float64)
            fin = np.isfinite(ref)
            assert (np.isfinite(got[f, i]) == fin).all()
            assert np.abs(got[f, i][fin] - ref[fin]).max() < 2e-5 * np.abs(ref[fin]).max()
