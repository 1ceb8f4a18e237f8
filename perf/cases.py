"""The work a user of this framework has it do, as measurable cases.

A case is one pass through a public entry point at the Qwen3-VL-2B shapes: the
decode kernels a swapped layer or a hand-written loop calls one at a time, the
one-launch decoder layer, and the engines' whole calls (prompt prefill, one
decode step at batch 1, one step of a ragged batch).  ``listed()`` gives the
measured cases, ``draw(rng)`` one more from the same ranges.
"""

from __future__ import annotations

import dataclasses
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "aicasgc-2026_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import cuda_decode_attention  # noqa: E402
import cuda_decode_gemv  # noqa: E402
from qwen3vl_hip import synthetic as syn  # noqa: E402
from qwen3vl_hip.config import QWEN3VL_2B as S  # noqa: E402
from qwen3vl_hip.engine import BatchDecodeEngine, DecodeEngine, rope_inv_freq  # noqa: E402

QKV, D, HQ, HKV, HID, INTER = S.qkv_rows, S.head_dim, S.num_heads, S.num_kv_heads, S.hidden, S.intermediate


# ------------------------------------------------------------------ the cases

def listed() -> list:
    return [
        # One projection of one layer: RMSNorm + QKV GEMV of a decode token.  The
        # smallest call of the drop-in chain; launch and host latency count.
        {"name": "rmsnorm_qkv", "path": "norm_matvec", "n": QKV, "k": HID},
        # The post-attention MLP of one layer (add + RMSNorm, gate_up + SiLU, down).
        {"name": "post_attn_mlp", "path": "mlp"},
        # The tied lm_head of the drop-in loop (FastLmHead): the largest GEMV.
        {"name": "lm_head", "path": "matvec", "n": S.vocab, "k": HID},
        # Decode attention behind a 1024-position prompt, an odd length inside a
        # larger static cache.
        {"name": "attention_1029", "path": "attention", "length": 1029, "capacity": 1281},
        # Decode attention late in a long document, near the largest cache served.
        {"name": "attention_30001", "path": "attention", "length": 30001, "capacity": 32768},
        # One swapped decoder layer (the one-launch layer) behind a 1024-position
        # prompt.
        {"name": "layer_1029", "path": "layer", "length": 1029, "capacity": 1281},
        # Time to first token of a short text question.
        {"name": "prefill_text_37", "path": "prefill", "grid_h": 0, "grid_w": 0, "n_text": 37},
        # Prefill of the 1024-position multimodal prompt: 24 x 32 vision rows + 256 ids.
        {"name": "prefill_1024", "path": "prefill", "grid_h": 24, "grid_w": 32, "n_text": 256},
        # Prefill of a large picture and a longer text, an odd total length.
        {"name": "prefill_4001", "path": "prefill", "grid_h": 48, "grid_w": 64, "n_text": 929},
        # One greedy step of the whole 28-layer model at batch 1, context 4096.
        {"name": "decode_4096", "path": "decode", "length": 4096, "capacity": 4160},
        # One step of 8 ragged sequences, KV lengths in [2048, 4096].
        {"name": "batch8_4096", "path": "batch", "batch": 8, "low": 2048, "high": 4096, "capacity": 4160},
        # One step of 3 ragged chats early in their conversations.
        {"name": "batch3_700", "path": "batch", "batch": 3, "low": 40, "high": 700, "capacity": 1024},
    ]


def _log(rng, low: int, high: int) -> int:
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng) -> dict:
    path = rng.choice(["norm_matvec", "matvec", "attention", "layer", "prefill", "prefill", "decode", "batch"])
    if path in ("norm_matvec", "matvec"):
        return {"path": path, "n": _log(rng, 1000, S.vocab), "k": HID if path == "norm_matvec" else rng.choice([HID, INTER])
                if rng.random() < 0.3 else HID}
    if path in ("attention", "layer", "decode"):
        length = _log(rng, 2, {"attention": 32768, "layer": 16384, "decode": 8192}[path])
        return {"path": path, "length": length, "capacity": length + rng.randrange(0, 300)}
    if path == "prefill":
        gh, gw = (0, 0) if rng.random() < 0.4 else (rng.randrange(2, 49), rng.randrange(2, 65))
        return {"path": path, "grid_h": gh, "grid_w": gw, "n_text": _log(rng, 2, 4001 - gh * gw)}
    batch = rng.randrange(2, 9)
    high = _log(rng, 64, 4096)
    low = max(2, high // rng.randrange(2, 9))
    return {"path": path, "batch": batch, "low": low, "high": high, "capacity": high + rng.randrange(1, 65)}


# ------------------------------------------------------------------ inputs

def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape, std: float = 1.0, mean: float = 0.0) -> torch.Tensor:
    return torch.empty(shape, dtype=torch.float16, device="cuda").normal_(mean, std, generator=g)


def _layer_weights(g) -> syn.LayerWeights:
    """Random-init weights as the repository's configurations have them."""
    return syn.LayerWeights(
        qkv_weight=_randn(g, QKV, HID, std=0.02), o_proj_weight=_randn(g, HID, S.q_size, std=0.02),
        gate_up_weight=_randn(g, 2 * INTER, HID, std=0.02), down_proj_weight=_randn(g, HID, INTER, std=0.02),
        input_layernorm_weight=_randn(g, HID, std=0.02, mean=1.0),
        post_attn_layernorm_weight=_randn(g, HID, std=0.02, mean=1.0),
        q_norm_weight=_randn(g, D, std=0.02, mean=1.0), k_norm_weight=_randn(g, D, std=0.02, mean=1.0))


def _model_weights(g) -> syn.ModelWeights:
    return syn.ModelWeights([_layer_weights(g) for _ in range(S.num_layers)], _randn(g, S.vocab, HID, std=0.02),
                            _randn(g, HID, std=0.02, mean=1.0), S)


def _cache(g, rows: int, capacity: int, batch: int = 1) -> torch.Tensor:
    c = torch.zeros(batch, HKV, capacity, D, dtype=torch.float16, device="cuda")
    c[:, :, :rows].normal_(generator=g)
    return c


def _long(v: int) -> torch.Tensor:
    return torch.tensor([v], dtype=torch.int64, device="cuda")


def _rope(position: int):
    """fp16 cos / sin of one text position, as a model's rotary embedding hands them over."""
    f = rope_inv_freq(S).cuda() * float(position)
    e = torch.cat([f, f])
    return e.cos().half(), e.sin().half()


def _prompt(case: dict, seed: int) -> syn.MultimodalPrompt:
    grid_t = 1 if case["grid_h"] else 0
    p = syn.multimodal_prompt(seed, grid_t, case["grid_h"], case["grid_w"], case["n_text"])
    return dataclasses.replace(p, vision_embeds=p.vision_embeds.cuda())


def _lengths(case: dict) -> list:
    """Valid KV lengths of the batch (the row written by the step included)."""
    return syn.batch8_kv_lengths(4, case["batch"], case["low"], case["high"]).tolist()


def _tokens(g, n: int) -> list:
    return torch.randint(0, S.vocab, (n,), generator=g, device="cuda").tolist()


def prepare(case: dict, seed: int) -> dict:
    g, path = _gen(seed), case["path"]
    st = {"case": case}
    if path in ("norm_matvec", "matvec"):
        n, k = case["n"], case["k"]
        st.update(x=_randn(g, 1, 1, k), w=_randn(g, n, k, std=0.02), gamma=_randn(g, k, std=0.02, mean=1.0),
                  ws={"type": "nosplit", "out": torch.empty(n, dtype=torch.float16, device="cuda")})
    elif path == "mlp":
        st.update(w=_layer_weights(g), residual=_randn(g, 1, 1, HID), attn=_randn(g, 1, 1, HID),
                  ws={"type": "fused_post_attn_mlp_softsync",
                      "hidden_out": torch.empty(INTER, dtype=torch.float16, device="cuda"),
                      "out": torch.empty(HID, dtype=torch.float16, device="cuda")})
    elif path == "attention":
        st.update(q=_randn(g, 1, HQ, 1, D), k=_cache(g, case["length"], case["capacity"]),
                  v=_cache(g, case["length"], case["capacity"]), pos=_long(case["length"] - 1), ws={})
    elif path == "layer":
        st.update(w=_layer_weights(g), x=_randn(g, 1, 1, HID), k=_cache(g, case["length"] - 1, case["capacity"]),
                  v=_cache(g, case["length"] - 1, case["capacity"]), pos=_long(case["length"] - 1), ws={})
        st["cos"], st["sin"] = _rope(case["length"] - 1)
    elif path == "prefill":
        p = _prompt(case, seed)
        st.update(prompt=p, engine=DecodeEngine(_model_weights(g), capacity=p.length + 64))
    elif path == "decode":
        e = DecodeEngine(_model_weights(g), capacity=case["capacity"], keep_logits=True)
        for k, v in zip(e.k_caches, e.v_caches):
            k[:, :, :case["length"] - 1].normal_(generator=g)
            v[:, :, :case["length"] - 1].normal_(generator=g)
        st.update(engine=e, token=_tokens(g, 1)[0])
        e.reserve_tokens(1)
        e.capture()
    else:
        e = BatchDecodeEngine(_model_weights(g), case["batch"], case["capacity"], keep_logits=True)
        lens = _lengths(case)
        for k, v in zip(e.k_caches, e.v_caches):
            for b, n in enumerate(lens):
                k[b, :, :n - 1].normal_(generator=g)
                v[b, :, :n - 1].normal_(generator=g)
        st.update(engine=e, lens=lens, tokens=_tokens(g, case["batch"]))
        e.reserve_tokens(1)
        e.capture()
    return st


# ------------------------------------------------------------------ one pass

def run(st: dict):
    path = st["case"]["path"]
    if path == "norm_matvec":
        return cuda_decode_gemv.fused_rmsnorm_qkv_half(st["x"], st["gamma"], st["w"], None, S.rms_eps)
    if path == "matvec":
        return cuda_decode_gemv.nosplit_matvec_half(st["x"], st["w"], None, workspace=st["ws"])
    if path == "mlp":
        w = st["w"]
        return cuda_decode_gemv.fused_post_attn_mlp_softsync_half(
            st["residual"], st["attn"], w.post_attn_layernorm_weight, w.gate_up_weight, w.down_proj_weight, None,
            S.rms_eps, st["ws"])
    if path == "attention":
        return cuda_decode_attention.decode_attn_v4_cta_qhead_splitkv_fused(
            st["q"], st["k"], st["v"], S.scaling, S.groups, st["pos"], split_k=4, workspace=st["ws"])
    if path == "layer":
        w = st["w"]
        out = cuda_decode_gemv.fused_decode_full_layer_softsync_half(
            st["x"], w.qkv_weight, w.input_layernorm_weight, w.q_norm_weight, w.k_norm_weight, st["cos"], st["sin"],
            st["k"], st["v"], st["pos"], w.o_proj_weight, None, w.post_attn_layernorm_weight, w.gate_up_weight,
            w.down_proj_weight, None, S.rms_eps, S.scaling, st["ws"])
        return [out, st["k"], st["v"]]
    e = st["engine"]
    if path == "prefill":
        token = e.prefill(st["prompt"])
        return {"token": token, "k": e.k_caches, "v": e.v_caches}
    # a step's logits and caches, not its token: random-init weights give near
    # ties now and then, and the logits say everything the token does
    if path == "decode":
        e.decode(st["token"], st["case"]["length"] - 1, 0, 1)
    else:
        pos = [n - 1 for n in st["lens"]]
        e.decode(st["tokens"], pos, pos, 1)
    return {"logits": e.logits, "k": e.k_caches, "v": e.v_caches}


# ------------------------------------------------------------------ bounds

_LAYER_WEIGHTS = QKV * HID + HID * S.q_size + 3 * INTER * HID   # elements of one layer's matrices
_NORMS = 2 * HID + 2 * D


def work(case: dict) -> dict:
    """Each weight, K/V row and activation once; two flops per multiply-add."""
    path = case["path"]
    if path in ("norm_matvec", "matvec"):
        n, k = case["n"], case["k"]
        return {"bytes": 2 * (n * k + n + k * (2 if path == "norm_matvec" else 1)), "flops": 2 * n * k}
    if path == "mlp":
        return {"bytes": 2 * (3 * INTER * HID + 4 * HID + INTER), "flops": 6 * INTER * HID}
    if path == "attention":
        n = case["length"]
        return {"bytes": 2 * (2 * HKV * n * D + 2 * HQ * D), "flops": 4 * HQ * n * D}
    if path == "layer":
        n = case["length"]
        return {"bytes": 2 * (_LAYER_WEIGHTS + _NORMS + 2 * HKV * n * D + 2 * HID),
                "flops": 2 * _LAYER_WEIGHTS + 4 * HQ * n * D}
    if path == "prefill":
        n = case["grid_h"] * case["grid_w"] + case["n_text"]
        kv = S.num_layers * 2 * HKV * n * D
        return {"bytes": 2 * (S.num_layers * (_LAYER_WEIGHTS + _NORMS) + S.vocab * HID + HID + n * HID + kv),
                "flops": 2 * n * S.num_layers * _LAYER_WEIGHTS + 4 * HQ * D * S.num_layers * n * (n + 1) // 2
                + 2 * S.vocab * HID}
    lens = [case["length"]] if path == "decode" else _lengths(case)
    b, total = len(lens), sum(lens)
    return {"bytes": 2 * (S.num_layers * (_LAYER_WEIGHTS + _NORMS + 2 * HKV * total * D) + S.vocab * HID + HID
                          + b * (HID + S.vocab)),
            "flops": b * 2 * (S.num_layers * _LAYER_WEIGHTS + S.vocab * HID) + 4 * HQ * D * S.num_layers * total}


# Largest differences two correct implementations show, about four times those
# measured (against 64 bits; for the engines also between the chain and the
# persistent step, and between prefills that sum in another order).  An fp16
# result is off by its rounding, 2.1e-4 (MLP and layer 3e-4); a prefill's fp16
# caches differ only where a last bit flips (6e-5); the batch-1 step rounds its
# GEMV inputs to fp16 (logits 2.3e-3 after 28 layers); the batch step carries
# fp32 (logits 6e-5, caches a flipped bit).  "max" covers one fp16 step of the
# largest values.
_TOLERANCE = {
    "norm_matvec": {"rel": 8e-4, "max": 4e-3}, "matvec": {"rel": 8e-4, "max": 4e-3},
    "attention": {"rel": 8e-4, "max": 4e-3}, "mlp": {"rel": 1.2e-3, "max": 8e-3},
    "layer": {"rel": 1.5e-3, "max": 1e-2}, "prefill": {"rel": 2.5e-4, "max": 4e-3},
    "decode": {"rel": 8e-3, "max": 4e-2}, "batch": {"rel": 3e-4, "max": 4e-3},
}


def tolerance(case: dict) -> dict:
    return dict(_TOLERANCE[case["path"]])


# ------------------------------------------------------------------ the same in 64 bits

def _d(t: torch.Tensor) -> torch.Tensor:
    return t.double()


def _rms64(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + S.rms_eps) * _d(w)


def _rotate64(x, cos, sin):
    h = x.shape[-1] // 2
    return x * cos + torch.cat([-x[..., h:], x[..., :h]], -1) * sin


def _mlp64(r, w):
    gu = _rms64(r, w.post_attn_layernorm_weight) @ _d(w.gate_up_weight).T
    return torch.nn.functional.silu(gu[..., :INTER]) * gu[..., INTER:]


def _qkv64(x, w, cos, sin):
    """Rotated q [n, HQ, D], rotated k and v [n, HKV, D] of the rows x [n, HID]."""
    n = x.shape[0]
    q, k, v = (_rms64(x, w.input_layernorm_weight) @ _d(w.qkv_weight).T).split([S.q_size, S.kv_size, S.kv_size], -1)
    q = _rotate64(_rms64(q.reshape(n, HQ, D), w.q_norm_weight), cos, sin)
    k = _rotate64(_rms64(k.reshape(n, HKV, D), w.k_norm_weight), cos, sin)
    return q, k, v.reshape(n, HKV, D)


def _attend64(q, k, v):
    """q [HQ, D] over k, v [HKV, L, D]."""
    out = []
    for h in range(HKV):
        sc = q[h * S.groups:(h + 1) * S.groups] @ k[h].T * S.scaling
        out.append(torch.softmax(sc, -1) @ v[h])
    return torch.cat(out)


def _step64(x, w, kc, vc, pos, cos, sin):
    """One layer of one decode token x [HID]: its output and the caches with the new row."""
    q, k, v = _qkv64(x[None], w, cos, sin)
    kc, vc = _d(kc).clone(), _d(vc).clone()
    kc[:, pos], vc[:, pos] = _d(k[0].half()), _d(v[0].half())   # attended as the fp16 cache holds it
    o = _attend64(q[0], kc[:, :pos + 1], vc[:, :pos + 1]).reshape(-1)
    kc[:, pos], vc[:, pos] = k[0], v[0]
    r = x + _d(w.o_proj_weight) @ o
    return r + _d(w.down_proj_weight) @ _mlp64(r, w), kc, vc


def _angles64(pos):
    """cos / sin [n, 1, D] of M-RoPE positions [3, n]."""
    stream = torch.zeros(D // 2, dtype=torch.long, device="cuda")
    for dim in (1, 2):
        stream[dim:S.mrope_section[dim] * 3:3] = dim
    f = _d(pos.cuda())[stream].T * _d(rope_inv_freq(S).cuda())
    e = torch.cat([f, f], -1)
    return e.cos()[:, None], e.sin()[:, None]


def _logits64(x, weights):
    return _rms64(x, weights.final_norm_weight) @ _d(weights.embed_tokens).T


def _prefill64(case: dict, st: dict) -> dict:
    e, p = st["engine"], st["prompt"]
    n, w = p.length, e.w
    x = torch.cat([_d(p.vision_embeds), _d(w.embed_tokens[p.text_ids.cuda()])])
    cos, sin = _angles64(p.position_ids)
    mask = torch.full((n, n), float("-inf"), dtype=torch.float64, device="cuda").triu(1)
    ks, vs = [], []
    for lw in w.layers:
        q, k, v = _qkv64(x, lw, cos, sin)
        for out, t in ((ks, k), (vs, v)):
            c = torch.zeros(1, HKV, e.capacity, D, dtype=torch.float64, device="cuda")
            c[0, :, :n] = t.transpose(0, 1)
            out.append(c)
        heads = []
        for h in range(HQ):
            sc = q[:, h].contiguous() @ k[:, h // S.groups].contiguous().T * S.scaling + mask
            heads.append(torch.softmax(sc, -1) @ v[:, h // S.groups].contiguous())
        r = x + torch.cat(heads, -1) @ _d(lw.o_proj_weight).T
        x = r + _mlp64(r, lw) @ _d(lw.down_proj_weight).T
    return {"token": None, "k": ks, "v": vs}


def exact(case: dict, seed: int):
    with torch.no_grad():
        st, path = prepare(case, seed), case["path"]
        if path in ("norm_matvec", "matvec"):
            x = _d(st["x"])
            return (_rms64(x, st["gamma"]) if path == "norm_matvec" else x) @ _d(st["w"]).T
        if path == "mlp":
            r = _d(st["residual"]) + _d(st["attn"])
            hidden = _mlp64(r, st["w"])
            return hidden, r + hidden @ _d(st["w"].down_proj_weight).T
        if path == "attention":
            n = case["length"]
            return _attend64(_d(st["q"][0, :, 0]), _d(st["k"][0, :, :n]), _d(st["v"][0, :, :n])).view(1, 1, HQ, D)
        if path == "layer":
            out, k, v = _step64(_d(st["x"]).view(-1), st["w"], st["k"][0], st["v"][0], case["length"] - 1,
                                _d(st["cos"]), _d(st["sin"]))
            return [out.view(1, 1, HID), k[None], v[None]]
        if path == "prefill":
            return _prefill64(case, st)
        e = st["engine"]
        lens = [case["length"]] if path == "decode" else st["lens"]
        tokens = [st["token"]] if path == "decode" else st["tokens"]
        ks, vs = [_d(k) for k in e.k_caches], [_d(v) for v in e.v_caches]
        rows = []
        for b, (tok, n) in enumerate(zip(tokens, lens)):
            cos, sin = (t[0, 0] for t in _angles64(torch.full((3, 1), n - 1)))
            x = _d(e.w.embed_tokens[tok])
            for i, lw in enumerate(e.w.layers):
                x, ks[i][b], vs[i][b] = _step64(x, lw, e.k_caches[i][b], e.v_caches[i][b], n - 1, cos, sin)
            rows.append(_logits64(x, e.w))
        return {"logits": rows[0] if path == "decode" else torch.stack(rows), "k": ks, "v": vs}
