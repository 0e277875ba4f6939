"""The batched prefill over K slices and the smaller GEMM tiles: prefixes of a
few to a thousand tokens in several ragged rows against the float64 oracle.  The
token counts sit at and around the tile heights, the widths take the trunk
shapes and an odd one with short K (96 and 160); test_gpu_prefill_tiles.py has a
case for every tile.

Bounds: FP32 sums of K = 6144 products in another order differ by ~sqrt(K) *
2^-24 = 5e-6 of a row's size per projection, 2e-5 over two layers; with BF16
weights the activations are hi + lo pairs, good to 2^-17 per value, 1e-4."""

import numpy as np
import pytest

from oracle.model import OracleModel, RowState, Shape, synthetic_weights

pytestmark = pytest.mark.gpu

SHAPES = {
    "06b": Shape(n_layers=2, text_vocab=512),
    "17b": Shape(d_model=2048, trunk_inter=6144, n_layers=1, text_vocab=512),
    "odd": Shape(d_model=96, n_layers=2, n_q_heads=6, n_kv_heads=3, head_dim=16, trunk_inter=160, n_codebooks=4,
                 codebook_size=32, text_vocab=512),
    "hd32": Shape(d_model=128, n_layers=2, n_q_heads=8, n_kv_heads=1, head_dim=32, trunk_inter=192, n_codebooks=4,
                  codebook_size=32, text_vocab=512),
    "hd64": Shape(d_model=128, n_layers=2, n_q_heads=4, n_kv_heads=4, head_dim=64, trunk_inter=192, n_codebooks=4,
                  codebook_size=32, text_vocab=512),
}


def _lens(total, rows):
    """`rows` ragged prefix lengths (text + BOS frame) of `total` tokens."""
    rows = min(rows, total // 2) or 1
    w = np.arange(1, rows + 1)
    lens = np.maximum(2, total * w // w.sum())
    lens[-1] += total - lens.sum()
    return [int(x) for x in lens]


@pytest.mark.parametrize("name,total", [("06b", t) for t in (2, 31, 33, 65, 129, 257, 401, 1150)]
                         + [("17b", 70), ("17b", 530), ("odd", 5), ("odd", 70), ("odd", 300)])
@pytest.mark.parametrize("bf16", [False, True])
def test_prefill_sizes_match_oracle(hip_device, name, total, bf16):
    _check(hip_device, name, total, bf16, False)


@pytest.mark.parametrize("name", ["odd", "hd32", "hd64", "06b"])
@pytest.mark.parametrize("total", [17, 130])
@pytest.mark.parametrize("kv_bf16", [False, True])
def test_prefill_attention_shapes_match_oracle(hip_device, name, total, kv_bf16):
    """Head sizes, group sizes and cache types of the attention: partial key
    tiles, rows shorter than a query block, waves without a key."""
    _check(hip_device, name, total, False, kv_bf16)


def _check(hip_device, name, total, bf16, kv_bf16):
    from oracle.model import round_bf16
    from soraku_amd import GraphFrameEngine
    from soraku_amd.config import DecodeShape
    from soraku_amd.synthetic import is_matrix

    s = SHAPES[name]
    w = synthetic_weights(s, 5, norm_gain_std=0.1)
    if bf16:
        w = {k: round_bf16(v) if is_matrix(k) else v for k, v in w.items()}
    lens = _lens(total, 4)
    rng = np.random.default_rng(total)
    items = [(rng.integers(0, s.text_vocab, n - 1), None, None) for n in lens]
    print(f"prefill {name} {lens} bf16={bf16}", flush=True)
    e = GraphFrameEngine(device=hip_device, max_cache_len=max(lens) + 4, cfg_scale=1.0, batch=1, state_dict=w,
                         shape=DecodeShape(**{k: getattr(s, k) for k in DecodeShape.__dataclass_fields__}),
                         n_utts=len(lens), bf16=bf16, kv_bf16=kv_bf16)
    got = e.prefill_utterances(items).cpu().numpy()
    e.close()
    m = OracleModel(s, w, np.float64, kv_bf16=kv_bf16)
    for r, (text, _, _) in enumerate(items):
        ref = m.prefill(RowState(s, lens[r] + 1, np.float64), m.prefix_embeds(text, None))
        err = np.abs(got[r] - ref).max() / np.abs(ref).max()
        # a BF16 cache: a few K/V values round the other way (2^-9 of the value each)
        assert err < (4e-3 if kv_bf16 else 1e-4 if bf16 else 2e-5), (r, lens[r], err)
