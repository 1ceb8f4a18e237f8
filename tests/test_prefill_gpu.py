"""The native prefill (qd_prefill) on the GPU against the oracle's prefill.

Row counts sit at the edges of the kernels' tiles (64 K/V and q rows, 64 / 128 /
256 GEMM rows, K splits for few rows); shapes cover GQA groups 1, 2 and 4 and
inputs of very different magnitudes.  The cache holds fp16, so a K/V element may
be off by half an fp16 step (2^-11 of itself) plus the difference of two fp32
evaluations, whose sums of 2048 to 6144 terms leave about 3e-6 of a row's rms per
layer: 2e-5 of the largest value covers the extremes of all elements.
"""

from __future__ import annotations

import dataclasses

import pytest
import torch

from oracle import qwen3vl_oracle as O

pytestmark = pytest.mark.gpu

SMALL = {"hidden": 512, "num_heads": 4, "num_kv_heads": 4, "intermediate": 512, "vocab": 512}
GROUP4 = {"hidden": 1024, "num_heads": 8, "num_kv_heads": 2, "intermediate": 1536, "vocab": 512}
MODEL = {"vocab": 2048}
WIDE = {"hidden": 512, "num_heads": 32, "num_kv_heads": 8, "intermediate": 512, "vocab": 512}


def _check(w, prompt, eng, token, per_row=False):
    """``per_row``: the bound on each row relative to that row's largest value."""
    s = w.shape
    shape = O.OracleShape(**{f.name: getattr(s, f.name) for f in dataclasses.fields(O.OracleShape)})
    n, cap = prompt.length, eng.capacity
    caches = [tuple(torch.zeros(1, s.num_kv_heads, cap, 128) for _ in "kv") for _ in range(s.num_layers)]
    last = O.prefill(w, O.embed_prompt(w, prompt), prompt.position_ids, caches, shape=shape)
    for li in range(s.num_layers):
        for got, ref in zip((eng.k_caches[li], eng.v_caches[li]), caches[li]):
            got = got.cpu().float()
            assert torch.equal(got[:, :, n:], torch.zeros_like(got[:, :, n:])), "rows past the prompt were written"
            top = ref[:, :, :n].abs().amax((1, 3), keepdim=True) if per_row else ref.abs().max()
            got, ref = got[:, :, :n], ref[:, :, :n]
            # an fp16 step is 2^-24 at the least
            err, bound = (got - ref).abs(), ref.abs() * 2 ** -11 + 2e-5 * top + (2 ** -25 if per_row else 0)
            print(f"[parity] layer {li}: worst {float((err / bound).max()):.3f} of the bound", flush=True)
            assert bool((err <= bound).all())
    logits = O.rms_norm(last, w.final_norm_weight, s.rms_eps) @ w.embed_tokens.float().T
    assert float(logits.max() - logits[token]) <= 1e-4 * float(logits.abs().max())


def _not_native(prompt):
    raise AssertionError("not the native route")


def _run(case, shape_kw, grid, n_text, layers=2, scale=None, weights=None, per_row=False):
    from qwen3vl_hip import synthetic as syn
    from qwen3vl_hip.config import Qwen3VLTextShape
    from qwen3vl_hip.engine import DecodeEngine

    print(f"case prefill {case}", flush=True)
    shape = Qwen3VLTextShape(num_layers=layers, **shape_kw)
    w = syn.model_weights(11, shape)
    if weights is not None:
        weights(w)
    p = syn.multimodal_prompt(11, *((1, *grid) if grid else (0, 0, 0)), n_text, shape=shape)
    if scale is not None:
        p = dataclasses.replace(p, vision_embeds=p.vision_embeds.float() * scale(p.vision_embeds.shape[0])[:, None])
    eng = DecodeEngine(w, capacity=p.length + 5)
    eng._prefill_general = _not_native
    token = eng.prefill(p)
    _check(w, p, eng, token, per_row)
    before = [t.clone() for t in eng.k_caches + eng.v_caches]
    assert eng.prefill(p) == token
    assert all(torch.equal(a, b) for a, b in zip(before, eng.k_caches + eng.v_caches)), "a second pass differs"
    return w, p, eng


@pytest.mark.parametrize("n", [1, 2, 16, 17, 63, 64, 65, 127, 129, 257, 513])
def test_prefill_text_lengths(cuda, n):
    _run(f"text {n}", MODEL, None, n)


@pytest.mark.parametrize("n", [15, 33, 49, 193, 256, 300, 700, 1300])
def test_prefill_tile_shapes(cuda, n):
    """Lengths at which the four products take the 16-, 32- and 64-row tiles, the
    192-wide ones and K ranges of unequal length; 256 is the last with 1024 threads
    per SiLU row on 256 CUs."""
    _run(f"tiles {n}", MODEL, None, n)


# Rows, columns and bk of the GEMM's tile table
GEMM_TILES = [(256, 256, 32), (256, 192, 32), (192, 192, 32), (128, 256, 32), (128, 128, 64), (64, 256, 64),
              (64, 192, 64), (64, 128, 64), (64, 64, 128), (32, 128, 128), (32, 64, 128), (16, 128, 128)]


@pytest.mark.parametrize("tile", range(len(GEMM_TILES)))
def test_prefill_gemm_tiles(cuda, tile):
    """Every tile with every K split of the plan, at the edges of its rows, columns
    and K ranges (one to three blocks, the depth of the ring, and more; ranges of
    unequal length), so that no plan can choose one that ran nowhere.  An accumulator
    is rounded some k / 16 times, by 2^-24 of a partial sum that random signs keep
    below 4 / sqrt(k) of the sum of the products' sizes: sqrt(k) / 4 times 2^-24 of
    that, and 3 more for short sums, the scale and the planes.  (Without the lo plane:
    5 times as much at the largest k.)"""
    from qwen3vl_hip import _lib

    bm, bn, bk = GEMM_TILES[tile]
    g, worst = torch.Generator().manual_seed(tile), 0.0
    for z in (1, 2, 3, 4, 6, 8, 12, 16):
        for m, n, kb in ((1, 4, z), (bm - 1, bn + 4, z + 1), (bm + 1, bn - 4, 2 * z + 1), (2 * bm, 2 * bn, 3 * z),
                         (2 * bm + 7, bn, 5 * z + max(1, z - 1))):
            k = kb * bk
            print(f"case gemm tile {tile} z {z} {m} x {n} x {k}", flush=True)
            x = torch.randn(m, k, generator=g) * 2.0 ** 12
            hi = x.half()
            lo = (x - hi.float()).half()
            w = torch.randn(n, k, generator=g).mul_(0.02).half()
            scale = 2.0 ** -torch.randint(0, 20, (m,), generator=g).float()
            dev = [t.to(cuda) for t in (hi, lo, scale, w)]
            y = torch.full((z, m, n), float("nan"), device=cuda)
            _lib.check(_lib.lib().qd_prefill_gemm(dev[0].data_ptr(), dev[1].data_ptr(), dev[2].data_ptr(),
                                                  dev[3].data_ptr(), y.data_ptr(), m, n, k, tile, z, _lib.stream(cuda)),
                       "qd_prefill_gemm")
            # the reference in 64 bits on the GPU: torch's own product
            h, l, s, wd = (t.double() for t in dev)
            ref, size = ((h + l) @ wd.T) * s[:, None], ((h.abs() + l.abs()) @ wd.abs().T) * s[:, None]
            err = (y.double().sum(0) - ref).abs()
            assert not bool(err.isnan().any())
            worst = max(worst, float((err / size).max()) / ((k ** 0.5 / 4 + 3) * 2.0 ** -24))
            assert worst <= 1, worst
    print(f"[parity] gemm tile {tile}: worst {worst:.3f} of the bound", flush=True)
    bad = _lib.lib().qd_prefill_gemm(dev[0].data_ptr(), dev[1].data_ptr(), dev[2].data_ptr(), dev[3].data_ptr(),
                                     y.data_ptr(), m, n, bk, tile, 2, _lib.stream(cuda))
    assert bad == _lib.QD_ERR_SHAPE


@pytest.mark.parametrize("n", [2432, 2433, 2560])
def test_prefill_attention_tile_rows(cuda, n):
    """Both sides of the step from 64 to 128 q rows per attention workgroup (16
    heads, 256 CUs), and an even multiple of the larger tile; two layers, since the
    last one runs its last tile alone and the next layer's K/V rows show every row."""
    _run(f"q tiles {n}", MODEL, None, n)


@pytest.mark.parametrize("n", [1152, 1153, 1217, 1345])
def test_prefill_attention_tile_rows_of_more_heads(cuda, n):
    """The same step with 32 q heads, and 65 and 1 rows in the last of the larger tiles."""
    _run(f"q tiles of 32 heads {n}", WIDE, None, n)


@pytest.mark.parametrize("grid,n_text", [((3, 5), 1), ((7, 9), 2), ((24, 32), 330), ((40, 44), 351)])
def test_prefill_multimodal(cuda, grid, n_text):
    _run(f"grid {grid} text {n_text}", MODEL, grid, n_text)


@pytest.mark.parametrize("kw", [SMALL, GROUP4])
@pytest.mark.parametrize("n", [1, 70, 200])
def test_prefill_other_shapes(cuda, kw, n):
    _run(f"{kw} n={n}", kw, None, n)


def test_prefill_rows_of_very_different_magnitude(cuda):
    """fp32 embedding rows from 1e-4 to 1e4 of the usual size, in one prompt."""
    _run("scaled rows", MODEL, (8, 11), 9,
         scale=lambda n: 10.0 ** (torch.arange(n) % 9 - 4).float())


@pytest.mark.parametrize("kw,n_text", [(SMALL, 70), (GROUP4, 200), (WIDE, 1100)])
@pytest.mark.parametrize("small", [(0, 64), (64, 128)])
def test_prefill_rows_far_below_the_rest(cuda, kw, n_text, small):
    """A run of embedding rows 2^-36 of the others' size, below what RMSNorm's eps
    levels: their V rows are about 2^-26 of the layer's largest, and the attention
    outputs of a first run depend on them alone, so layer 1's K rows must hold
    to fp16 and fp32 rounding of each row.  128 q rows per workgroup (32 heads,
    1228 rows) and 64 (the others)."""
    lo, hi = small
    _run(f"rows {lo}..{hi} far below, {kw}", kw, (8, 16), n_text, per_row=True,
         scale=lambda n: torch.where((torch.arange(n) >= lo) & (torch.arange(n) < hi), 2.0 ** -36, 1.0))


@pytest.mark.parametrize("kw,grid", [(MODEL, (32, 64)), (WIDE, (64, 64))])
def test_prefill_large_rows_at_the_end(cuda, kw, grid):
    """The same with the large rows behind more V tiles than a wave's first loads of
    their exponents cover (256 of 8 heads with 64 q rows, 512 with 128), where a
    missed one would overflow the last rows."""
    _run(f"large rows behind {grid}, {kw}", kw, grid, 130, per_row=True, scale=lambda n: torch.full((n,), 2.0 ** -36))


@pytest.mark.parametrize("n", [5, 70])
def test_prefill_zero_head_norms(cuda, n):
    """q and k norm weights of zero: all scores equal, attention the causal mean."""
    _run(f"zero head norms {n}", SMALL, None, n,
         weights=lambda w: [t.zero_() for lw in w.layers for t in (lw.q_norm_weight, lw.k_norm_weight)])


def test_prefill_forms_outside_the_native_route(cuda):
    """Float positions, one position for all rows and float64 embeddings keep
    their results: the first two by the general path, the last natively."""
    w, p, eng = _run("forms", SMALL, (2, 3), 4)
    token, k = eng.prefill(p), [t.clone() for t in eng.k_caches]
    general, calls = type(eng)._prefill_general, []

    def again(q, native):
        for t in eng.k_caches + eng.v_caches:
            t.zero_()
        eng._prefill_general = _not_native if native else lambda prompt: calls.append(0) or general(eng, prompt)
        before = len(calls)
        _check(w, dataclasses.replace(q, position_ids=q.position_ids.long().expand(3, q.length)), eng, eng.prefill(q))
        assert native or len(calls) == before + 1

    again(dataclasses.replace(p, position_ids=p.position_ids.double()), False)
    again(dataclasses.replace(p, position_ids=torch.full((3, 1), 7)), False)
    again(dataclasses.replace(p, vision_embeds=p.vision_embeds.double()), True)
    assert eng.prefill(p) == token and all(torch.equal(a, b) for a, b in zip(k, eng.k_caches))
    with pytest.raises(ValueError):
        eng.prefill(dataclasses.replace(p, text_ids=p.text_ids * 0 + SMALL["vocab"]))


@pytest.mark.parametrize("dtype", [torch.int32, torch.int16, torch.uint8, torch.float32, torch.float64])
def test_prefill_text_id_types(cuda, dtype):
    """Ids of a type that does not index an embedding table are refused."""
    w, p, eng = _run("id types", {**SMALL, "vocab": 200}, (2, 3), 4)
    q = dataclasses.replace(p, text_ids=p.text_ids.to(dtype))
    if dtype == torch.int32:
        assert eng.prefill(q) == eng.prefill(p)
    else:
        del eng._prefill_general
        with pytest.raises(IndexError):
            eng.prefill(q)


@pytest.mark.parametrize("form", ["field", "data", "layer", "embedding", "fp32", "transposed", "cache"])
@pytest.mark.parametrize("i", [0, 4])
def test_prefill_reads_the_weights_of_its_call(cuda, form, i):
    """Weights and caches rebound after the engine was made are the ones used,
    whatever route their type and layout take; a wrong shape is refused.  The call
    looks at the first four layers before its first launch, at the others after."""
    from qwen3vl_hip import synthetic as syn
    from qwen3vl_hip.config import Qwen3VLTextShape
    from qwen3vl_hip.engine import DecodeEngine

    shape = Qwen3VLTextShape(num_layers=5, **SMALL)
    other = syn.model_weights(12, shape, device=cuda)
    p = syn.multimodal_prompt(11, 1, 2, 3, 9, shape=shape)
    eng = DecodeEngine(syn.model_weights(11, shape), capacity=p.length + 5)
    w, held = eng.w, [(lw, lw.down_proj_weight, lw.qkv_weight) for lw in eng.w.layers]   # no old weight is freed
    held.append((eng.w.embed_tokens, list(eng.k_caches)))
    first = eng.prefill(p)
    if form == "field":
        w.layers[i].down_proj_weight = other.layers[i].down_proj_weight
    elif form == "data":
        held.append(w.layers[i].qkv_weight.data)
        w.layers[i].qkv_weight.data = other.layers[i].qkv_weight
    elif form == "layer":
        w.layers[i] = other.layers[i]
    elif form == "embedding":
        w.embed_tokens = other.embed_tokens
    elif form == "fp32":
        w.layers[i].down_proj_weight = other.layers[i].down_proj_weight.float()
    elif form == "transposed":
        w.layers[i].down_proj_weight = other.layers[i].down_proj_weight.T.contiguous().T
    else:
        eng.k_caches[i] = torch.zeros_like(eng.k_caches[i])
    token = eng.prefill(p)
    _check(w.to("cpu"), p, eng, token)
    if form == "cache":
        assert token == first
    else:
        fresh = DecodeEngine(w, capacity=eng.capacity)
        assert fresh.prefill(p) == token
        for a, b in zip(eng.k_caches + eng.v_caches, fresh.k_caches + fresh.v_caches):
            assert torch.equal(a, b)
    w.layers[4 - i].o_proj_weight = w.layers[4 - i].o_proj_weight[:, :-64].contiguous()
    with pytest.raises(RuntimeError):
        eng.prefill(p)


@pytest.mark.parametrize("cuts", [(0, 5), (0, 1, 5), (0, 2, 4, 5)])
def test_prefill_in_parts(cuda, cuts):
    """The C entries: a whole prefill and one in parts, bit for bit the engine's (whose
    own parts are of four layers and the rest), with a workspace full of NaN."""
    import ctypes

    from qwen3vl_hip import _lib

    w, p, eng = _run(f"parts {cuts}", SMALL, (2, 3), 70, layers=5)
    token, before = eng.prefill(p), [t.clone() for t in eng.k_caches + eng.v_caches]
    for t in eng.k_caches + eng.v_caches:
        t.zero_()
    lib, d, n = _lib.lib(), ctypes.byref(eng.desc), p.length
    nbytes = lib.qd_prefill_workspace_bytes(d, n)
    ws = torch.full((nbytes,), 255, dtype=torch.uint8, device=cuda)
    out = torch.full((1,), -1, dtype=torch.int64, device=cuda)
    vis, ids, pos = (t.to(cuda).contiguous() for t in (p.vision_embeds, p.text_ids, p.position_ids))
    args = (vis.data_ptr(), _lib.QD_F16, vis.shape[0], ids.data_ptr(), pos.data_ptr(), n, out.data_ptr(), ws.data_ptr(),
            nbytes, _lib.stream(cuda))
    for first, count in ((-1, 2), (0, 0), (0, 6), (5, 1), (4, 2)):
        assert lib.qd_prefill_layers(d, first, count, *args) == _lib.QD_ERR_SHAPE
    if len(cuts) == 2:
        _lib.check(lib.qd_prefill(d, *args), "qd_prefill")
    for a, b in zip(cuts, cuts[1:]) if len(cuts) > 2 else ():
        assert int(out) == -1
        _lib.check(lib.qd_prefill_layers(d, a, b - a, *args), "qd_prefill_layers")
    assert int(out) == token
    assert all(torch.equal(a, b) for a, b in zip(before, eng.k_caches + eng.v_caches))
