"""Performance cases of the decode engine and the operator API.

Each case is one call (or one short program of calls) that a user of the
package makes through its public entry points: the operator factories of
``soraku_amd.ops`` and ``soraku_amd.GraphFrameEngine`` (prefill, then frames).
``listed()`` names the fixed cases, ``draw(rng)`` gives more of the same
ranges; ``prepare`` / ``run`` / ``exact`` / ``work`` / ``tolerance`` make, run,
check and price one case.

Kinds of cases:

* ``norm``      add + RMSNorm of a few rows: the smallest call, all latency.
* ``depth``     one codebook step of the depth head as a chain of operators
                (add + norm, SwiGLU, down + residual, norm, classifier, sampler,
                prefix advance), the way a program drives the operator API.
* ``mlp``       SwiGLU + down projection of 1 to 32 decode rows.
* ``head``      one codebook's classifier for 1 to 32 decode rows.
* ``prefill``   the prefixes of one call through the trunk, from one short row
                to 16 ragged utterances with CFG.
* ``utterance`` prefill, then frames one at a time as ``generate`` steps them.
                The codes of every frame are given (teacher forcing), so that a
                last-bit difference in the logits cannot send the rest of the
                run down another path; every frame still samples.

Weights are random with the initialiser's spread (N(0, 0.02), norm gains near
1) at the two trunk shapes of the package, text ids and codes are uniform.
"""

from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "soraku-tts_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

from soraku_amd import QWEN3_06B, QWEN3_17B, GraphFrameEngine, ops  # noqa: E402
from soraku_amd.config import FLT_EPS  # noqa: E402
from soraku_amd.synthetic import is_matrix, weight_shapes  # noqa: E402

DEV = "cuda:0"
V = QWEN3_06B.audio_vocab
Q = QWEN3_06B.n_codebooks
SHAPES = {"06b": QWEN3_06B, "17b": QWEN3_17B}
CFG, TEMP, TOP_K, TOP_P = 1.5, 0.9, 50, 0.95
TEXT_BOS = 151643
MIN_NEW = 4


def listed():
    return [
        # one norm of a CFG pair: what a single small launch costs
        dict(name="norm_pair", kind="norm", rows=2, d=1024),
        # the operator API driving one codebook step of one utterance with CFG
        dict(name="depth_pair_f32", kind="depth", rows=2, d=1024, inner=2048, bf16=False),
        # the wider trunk's MLP for an odd number of decode rows
        dict(name="mlp_7rows_bf16", kind="mlp", rows=7, d=2048, inner=6144, bf16=True),
        # a codebook classifier for ten utterances with CFG
        dict(name="head_20rows_f32", kind="head", rows=20, d=1024, bf16=False),
        # voice-cloning prefix of one utterance with CFG (text + prompt audio)
        dict(name="prefill_pair_f32", kind="prefill", model="06b", bf16=False, kv_bf16=False, utts=1, cfg=2,
             text=96, prompt=144),
        # a serving batch: 16 ragged prefixes at once
        dict(name="prefill_16utts_bf16", kind="prefill", model="06b", bf16=True, kv_bf16=True, utts=16, cfg=2,
             text=96, prompt=143),
        # a long text with a long prompt, no CFG, on the wider trunk
        dict(name="prefill_long_17b_bf16", kind="prefill", model="17b", bf16=True, kv_bf16=False, utts=1, cfg=1,
             text=701, prompt=612),
        # one utterance with CFG, FP32: the interactive case
        dict(name="utt_pair_f32", kind="utterance", model="06b", bf16=False, kv_bf16=False, utts=1, cfg=2,
             text=96, prompt=144, frames=48),
        # one utterance without CFG (the default of generate), BF16, no prompt
        dict(name="utt_single_bf16", kind="utterance", model="06b", bf16=True, kv_bf16=False, utts=1, cfg=1,
             text=57, prompt=0, frames=48),
        # one utterance with CFG on the wider trunk
        dict(name="utt_pair_17b_bf16", kind="utterance", model="17b", bf16=True, kv_bf16=False, utts=1, cfg=2,
             text=95, prompt=144, frames=48),
        # a few utterances with CFG in FP32
        dict(name="utts_4_f32", kind="utterance", model="06b", bf16=False, kv_bf16=False, utts=4, cfg=2,
             text=80, prompt=75, frames=32),
        # the throughput batch: 16 utterances with CFG, BF16 weights and cache
        dict(name="utts_16_bf16", kind="utterance", model="06b", bf16=True, kv_bf16=True, utts=16, cfg=2,
             text=96, prompt=143, frames=48),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["norm", "depth", "mlp", "head", "prefill", "prefill", "utterance", "utterance"])
    bf16 = rng.random() < 0.5
    if kind == "norm":
        return dict(kind=kind, rows=_log_int(rng, 1, 32), d=32 * rng.randint(2, 64))
    if kind == "depth":
        d = rng.choice([1024, 2048, 32 * rng.randint(8, 64)])
        return dict(kind=kind, rows=rng.randint(1, 2), d=d, inner=2 * d, bf16=bf16)
    if kind == "mlp":
        d = rng.choice([1024, 2048, 32 * rng.randint(8, 64)])
        return dict(kind=kind, rows=_log_int(rng, 1, 32), d=d, inner=rng.choice([2, 3]) * d, bf16=bf16)
    if kind == "head":
        return dict(kind=kind, rows=_log_int(rng, 1, 32), d=rng.choice([1024, 2048, 32 * rng.randint(8, 64)]), bf16=bf16)
    top = max(_cost(c) for c in listed() if c["kind"] == kind)
    while True:
        c = dict(kind=kind, model=rng.choice(["06b", "06b", "17b"]), bf16=bf16, kv_bf16=bf16 and rng.random() < 0.5,
                 utts=rng.choice([1, 1, _log_int(rng, 1, 16)]), cfg=rng.choice([1, 2, 2]),
                 text=_log_int(rng, 6, 800), prompt=rng.choice([0, _log_int(rng, 12, 640)]))
        if kind == "utterance":
            c["frames"] = _log_int(rng, 8, 48)
        if _cost(c) <= top:
            return c


def _cost(case):
    w = work(case)
    return w["bytes"] / 6e12 + w["flops"] * (1 if case["bf16"] else 8) / 8e14


# ------------------------------------------------------------------ inputs

def _lens(case):
    """(text ids, prompt frames) of each utterance: ragged from half to all of
    the case's sizes when there are several."""
    n = case["utts"]
    out = []
    for u in range(n):
        f = 1.0 if n == 1 else 0.5 + 0.5 * ((7 * u) % n) / (n - 1)
        out.append((max(1, round(case["text"] * f)), round(case["prompt"] * f)))
    return out


def _row_lens(case):
    """Prefix tokens of each decode row: text, the BOS frame, the prompt; the
    uncond row's text is one id."""
    rows = []
    for t, p in _lens(case):
        rows.append(t + 1 + p)
        if case["cfg"] == 2:
            rows.append(1 + 1 + p)
    return rows


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 1000003 + 17)


def _randn(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32).mul_(scale)


def _mat(g, bf16, *shape):
    w = _randn(g, *shape, scale=0.02)
    return w.to(torch.bfloat16) if bf16 else w


def _gain(g, n):
    return _randn(g, n, scale=0.1).add_(1.0)


def _weights(case, seed):
    g = _gen(seed)
    out = {}
    for key, shp in weight_shapes(SHAPES[case["model"]]).items():
        if is_matrix(key):
            out[key] = _mat(g, case["bf16"], *shp)
        elif key == "depth_head.bias":
            out[key] = _randn(g, *shp, scale=0.02)
        else:
            out[key] = _gain(g, shp[0])
    return out


def _items(case, seed):
    """(cond ids, uncond ids, prompt codes) per utterance, and the frames'
    codes and uniforms."""
    rng = np.random.default_rng([int(seed), 5])
    s = SHAPES[case["model"]]
    items = []
    for t, p in _lens(case):
        text = rng.integers(0, s.text_vocab, t)
        text[0] = TEXT_BOS
        prompt = rng.integers(0, s.codebook_size, (p, Q))
        items.append((text, np.array([TEXT_BOS], np.int64), prompt))
    n = case.get("frames", 0)
    codes = rng.integers(0, s.codebook_size, (n, case["utts"], Q))
    return items, codes, rng.random((n, case["utts"], Q))


def _op_inputs(case, seed):
    g, b, d = _gen(seed), case["rows"], case["d"]
    kind = case["kind"]
    x = {"x": _randn(g, b, d)}
    if kind == "norm":
        x.update(prefix=_randn(g, b, d, scale=0.1), w=_gain(g, d))
        return x
    bf = case["bf16"]
    if kind in ("depth", "mlp"):
        i = case["inner"]
        x.update(wg=_mat(g, bf, i, d), wu=_mat(g, bf, i, d), wd=_mat(g, bf, d, i), res=_randn(g, b, d))
    if kind in ("depth", "head"):
        # the classifier's rows: in the weights' type; the prefix table of the operator API is FP32
        x.update(table=_mat(g, bf, V, d), bias=_randn(g, V, scale=0.02))
    if kind == "depth":
        x.update(prefix=_randn(g, b, d, scale=0.1), w_in=_gain(g, d), w_out=_gain(g, d),
                 table32=x["table"].float(), code=torch.randint(0, V - 3, (1,), generator=g, device=DEV),
                 u=float(np.random.default_rng([int(seed), 6]).random()))
    return x


def prepare(case, seed):
    if case["kind"] in ("prefill", "utterance"):
        items, codes, u = _items(case, seed)
        n = case.get("frames", 0)
        e = GraphFrameEngine(device=DEV, max_cache_len=max(_row_lens(case)) + n + 8, cfg_scale=CFG if case["cfg"] == 2 else 1.0,
                             batch=case["cfg"], state_dict=_weights(case, seed), shape=SHAPES[case["model"]],
                             n_utts=case["utts"], bf16=case["bf16"], kv_bf16=case["kv_bf16"], max_frames=max(n, 1))
        e.set_temperature(TEMP)
        e.set_sampling(sampled=True, top_k=TOP_K, top_p=TOP_P)
        if n:
            e.set_debug(True)
            e.prefill_utterances(items)
            e.capture()
        return dict(case=case, engine=e, items=items, codes=codes, u=u)
    x = _op_inputs(case, seed)
    b, d = case["rows"], case["d"]
    k = {}
    if case["kind"] == "norm":
        k["add_norm"] = ops.add_rmsnorm(b, d, FLT_EPS)
    if case["kind"] in ("depth", "mlp"):
        k["swiglu"] = ops.swiglu_gemv(b, case["inner"], d)
        k["down"] = ops.down_residual_gemv(b, d, case["inner"])
    if case["kind"] in ("depth", "head"):
        k["head"] = ops.classifier_gemv(b, V, d)
    if case["kind"] == "depth":
        s = QWEN3_06B
        k.update(add_norm=ops.add_rmsnorm(b, d, FLT_EPS), norm=ops.rmsnorm(b, d, FLT_EPS),
                 sample=ops.sample(V, s.bos_id, s.eos_id, s.pad_id), prefix=ops.prefix_add(b, V, d, s.frame_scale))
    return dict(case=case, k=k, **x)


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "prefill":
        return st["engine"].prefill_utterances(st["items"])
    if kind == "utterance":
        e, n = st["engine"], case["frames"]
        e.prefill_utterances(st["items"])
        codes = []
        for f in range(n):
            kw = dict(mask_eos_q0=f < MIN_NEW, uniforms=st["u"][f], forced_codes=st["codes"][f])
            if f + 1 < n:
                codes.append(e.step_frame(**kw))
            else:
                c, logits = e.step_frame(**kw, return_logits=True)
                codes.append(c)
        return {"codes": torch.stack(codes), "logits": logits, "hidden": e.hidden()}
    k = st["k"]
    if kind == "norm":
        return k["add_norm"](st["x"], st["prefix"], st["w"])
    if kind == "mlp":
        return k["down"](k["swiglu"](st["x"], st["wg"], st["wu"]), st["wd"], st["res"])
    if kind == "head":
        return k["head"](st["x"], st["table"], st["bias"])
    a = k["add_norm"](st["x"], st["prefix"], st["w_in"])
    y = k["down"](k["swiglu"](a, st["wg"], st["wu"]), st["wd"], a)
    logits = k["head"](k["norm"](y, st["w_out"]), st["table"], st["bias"])
    code = k["sample"](logits, cfg_scale=CFG if case["rows"] == 2 else 1.0, q=3, mask_eos_q0=False,
                       temperature=TEMP, top_k=TOP_K, top_p=TOP_P, u=st["u"])
    return {"logits": logits, "code": code, "prefix": k["prefix"](st["prefix"], st["table32"], st["code"])}


# ------------------------------------------------------------------ the same in 64 bits

def _rms(x, w, eps):
    return w.double() * (x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps))


def _lin(x, w):
    return x @ w.double().t()


def _mlp64(x, wg, wu, wd):
    gate = _lin(x, wg)
    return _lin(gate * torch.sigmoid(gate) * _lin(x, wu), wd)


def _trunk64(case, w, embeds):
    """The trunk over each row's whole sequence; final-normed hidden states."""
    s = SHAPES[case["model"]]
    lens = [x.shape[0] for x in embeds]
    h = torch.cat(embeds)
    hd, hq, hk = s.head_dim, s.n_q_heads, s.n_kv_heads
    # the model's rotary table: FP32 inverse frequencies and FP32 angles
    ex = np.arange(0, hd, 2, dtype=np.float32) / np.float32(hd)
    inv = (np.float32(1.0) / np.float32(s.rope_theta) ** ex).astype(np.float32)
    pos = np.concatenate([np.arange(n, dtype=np.float32) for n in lens])
    ang = torch.from_numpy((pos[:, None] * inv[None, :]).astype(np.float64)).to(DEV)
    cos, sin = ang.cos()[:, None, :], ang.sin()[:, None, :]

    def rope(x):
        a, b = x[..., : hd // 2], x[..., hd // 2:]
        return torch.cat((a * cos - b * sin, b * cos + a * sin), -1)

    def cached(x):
        return x.float().to(torch.bfloat16).double() if case["kv_bf16"] else x

    for i in range(s.n_layers):
        p = f"trunk.layers.{i}."
        x = _rms(h, w[p + "input_layernorm.weight"], s.trunk_eps)
        q = _lin(x, w[p + "self_attn.q_proj.weight"]).view(-1, hq, hd)
        k = _lin(x, w[p + "self_attn.k_proj.weight"]).view(-1, hk, hd)
        v = cached(_lin(x, w[p + "self_attn.v_proj.weight"]).view(-1, hk, hd))
        q = rope(_rms(q, w[p + "self_attn.q_norm.weight"], s.trunk_eps))
        k = cached(rope(_rms(k, w[p + "self_attn.k_norm.weight"], s.trunk_eps)))
        outs, at = [], 0
        for n in lens:
            qr = q[at:at + n].transpose(0, 1)
            kr = k[at:at + n].transpose(0, 1).repeat_interleave(hq // hk, 0)
            vr = v[at:at + n].transpose(0, 1).repeat_interleave(hq // hk, 0)
            sc = torch.matmul(qr, kr.transpose(1, 2).contiguous()) * hd ** -0.5
            sc.masked_fill_(torch.ones(n, n, dtype=torch.bool, device=DEV).triu_(1), -math.inf)
            outs.append(torch.matmul(sc.softmax(-1), vr.contiguous()).transpose(0, 1).reshape(n, hq * hd))
            at += n
        h = h + _lin(torch.cat(outs), w[p + "self_attn.o_proj.weight"])
        x = _rms(h, w[p + "post_attention_layernorm.weight"], s.trunk_eps)
        h = h + _mlp64(x, w[p + "mlp.gate_proj.weight"], w[p + "mlp.up_proj.weight"], w[p + "mlp.down_proj.weight"])
    return torch.split(_rms(h, w["trunk.norm.weight"], s.trunk_eps), lens)


def _frames64(w, codes):
    """Embedding of codes [n, Q]: the codebooks' rows summed, times Q^-1/2."""
    t = w["audio_codebooks.table"]
    c = torch.from_numpy(np.ascontiguousarray(codes)).to(DEV)
    return sum(t[j][c[:, j]].double() for j in range(Q)) * Q ** -0.5


def _exact_engine(case, seed):
    s = SHAPES[case["model"]]
    w = _weights(case, seed)
    items, codes, _ = _items(case, seed)
    n = case.get("frames", 0)
    bos = np.full((1, Q), s.bos_id, np.int64)
    embeds = []
    for u, (text, uncond, prompt) in enumerate(items):
        frames = _frames64(w, np.concatenate((bos, prompt, codes[:, u])))
        for ids in (text, uncond)[: case["cfg"]]:
            te = w["trunk.embed_tokens.weight"][torch.from_numpy(ids).to(DEV)].double()
            embeds.append(torch.cat((te, frames)))
    hid = _trunk64(case, w, embeds)
    last = torch.stack([h[-1] for h in hid])
    if not n:
        return last
    h = torch.stack([x[-2] for x in hid])           # what the last frame's depth steps read
    prefix = torch.zeros_like(h)
    logits = torch.empty(case["utts"], Q, s.audio_vocab, dtype=torch.float64, device=DEV)
    for q in range(Q):
        a = _rms(h + prefix, w["depth_head.norm_in.weight"], FLT_EPS)
        y = a + _mlp64(a, *(w[f"depth_head.mlp.{m}_proj.weight"] for m in ("gate", "up", "down")))
        body = _rms(y, w["depth_head.norm_out.weight"], FLT_EPS)
        lg = _lin(body, w["audio_codebooks.table"][q]) + w["depth_head.bias"][q].double()
        if case["cfg"] == 2:
            c, un = lg[0::2], lg[1::2]
            lg = un + CFG * (c - un)
        logits[:, q] = lg
        step = w["audio_codebooks.table"][q][torch.from_numpy(codes[-1, :, q]).to(DEV)].double() * s.frame_scale
        prefix = prefix + step.repeat_interleave(case["cfg"], 0)
    logits[:, :, s.bos_id] = -math.inf
    logits[:, :, s.pad_id] = -math.inf
    logits[:, 0 if n <= MIN_NEW else 1:, s.eos_id] = -math.inf   # EOS only at codebook 0, past the first frames
    c = torch.from_numpy(codes if case["utts"] > 1 else codes[:, 0])
    return {"codes": c, "logits": logits.cpu().numpy(), "hidden": last.cpu().numpy()}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("prefill", "utterance"):
        return _exact_engine(case, seed)
    x = _op_inputs(case, seed)
    x64 = x["x"].double()
    if kind == "norm":
        return _rms(x64 + x["prefix"].double(), x["w"], FLT_EPS)
    if kind == "mlp":
        return _mlp64(x64, x["wg"], x["wu"], x["wd"]) + x["res"].double()
    if kind == "head":
        return _lin(x64, x["table"]) + x["bias"].double()
    a = _rms(x64 + x["prefix"].double(), x["w_in"], FLT_EPS)
    y = a + _mlp64(a, x["wg"], x["wu"], x["wd"])
    logits = _lin(_rms(y, x["w_out"], FLT_EPS), x["table"]) + x["bias"].double()
    return {"logits": logits, "code": None,
            "prefix": x["prefix"].double() + x["table32"].double()[x["code"]] * QWEN3_06B.frame_scale}


# ------------------------------------------------------------------ work and tolerance

def work(case):
    kind = case["kind"]
    if kind in ("prefill", "utterance"):
        return _engine_work(case)
    b, d = case["rows"], case["d"]
    if kind == "norm":
        return {"bytes": 4 * d * (3 * b + 1), "flops": 5 * b * d}
    wb = 2 if case["bf16"] else 4
    nbytes, mats = 4 * b * d, 0
    if kind in ("depth", "mlp"):
        mats += 3 * d * case["inner"]
    if kind in ("depth", "head"):
        mats += V * d
        nbytes += 4 * V + 4 * b * V
    if kind == "mlp":
        nbytes += 8 * b * d
    if kind == "depth":
        nbytes += 4 * d * (2 * b + 3)
    return {"bytes": nbytes + wb * mats, "flops": 2 * b * mats}


def _engine_work(case):
    """Prefill: the trunk's weights once, the prefix embeddings, K/V written
    and read back once.  Frames: every weight once per frame (the depth MLP
    counted once though it runs for every codebook), the live K/V."""
    s = SHAPES[case["model"]]
    wb, kb = (2 if case["bf16"] else 4), (2 if case["kv_bf16"] else 4)
    hq, hk = s.n_q_heads * s.head_dim, s.n_kv_heads * s.head_dim
    trunk = s.n_layers * (2 * hq * s.d_model + 2 * hk * s.d_model + 3 * s.trunk_inter * s.d_model)
    lens = _row_lens(case)
    rows, tokens = len(lens), sum(lens)
    kv_token = s.n_layers * 2 * hk * kb
    nbytes = trunk * wb + tokens * (s.d_model * wb + 2 * kv_token) + rows * s.d_model * 4
    flops = 2 * trunk * tokens + sum(2 * s.n_layers * hq * n * n for n in lens)
    n = case.get("frames", 0)
    if n:
        depth, table = 3 * s.depth_inner * s.d_model, Q * s.audio_vocab * s.d_model
        ctx = sum(n * x + n * (n - 1) // 2 for x in lens)
        nbytes += n * ((trunk + depth + table) * wb + Q * s.audio_vocab * 4 + rows * kv_token) + ctx * kv_token
        flops += n * rows * 2 * (trunk + Q * depth + table) + 4 * s.n_layers * hq * ctx
        nbytes += n * case["utts"] * Q * 24
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # about four times the error against 64 bits that the engine shows
    kind = case["kind"]
    if kind in ("prefill", "utterance"):
        if case["kv_bf16"]:
            # K and V are rounded to BF16: a last-bit change flips some of them by one place
            return {"rel": 6e-3, "max": 6e-2, "differ": 0.0}
        if case["bf16"]:
            # activations of a prefill and of many rows go through the GEMMs as BF16 hi + lo pairs
            return {"rel": 1.2e-4, "max": 1.2e-3, "differ": 0.0}
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.0}
    if kind == "norm":
        return {"rel": 5e-7, "max": 5e-6}
    return {"rel": 1e-6, "max": 1e-5, "differ": 0.0}
