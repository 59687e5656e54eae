"""Prefill kernels at the edges of their tiles and splits, against the oracle.

One-layer models: the 1B and 4B models' layers and one whose row counts are odd
multiples of 64 (the last 256-row tile is mostly past the edge).  Two-layer
ones where the norm handed between GEMMs counts, and small ones for the other
head groupings.
"""
import dataclasses
import os

import numpy as np
import pytest

from conftest import model_root

pytestmark = pytest.mark.gpu
ABS_TOL, REL_TOL = 2e-3, 1e-3  # the logit tolerance of every parity test


@pytest.fixture(scope="module")
def mods():
    import oracle.oracle as O
    import tinyminigo_amd as T
    from tinyminigo_amd import workloads as W

    O.set_attn_threads(max(1, min(16, os.cpu_count() or 1)))
    yield T, O, W
    O.set_attn_threads(1)


_open = {}


def _models(mods, which):
    if which in _SHAPES or which[4:] in _SHAPES:
        return _shaped(mods, which)
    if which not in _open:
        T, O, W = mods
        if which.startswith("i8-"):
            wl = _models(mods, which[3:])[2]
            p = W.ensure_model(wl, model_root())
            os.environ["TMG_I8"] = "1"
            try:
                _open[which] = T.Model.load(p), O.OracleModel.load(p, i8=True), wl
            finally:
                del os.environ["TMG_I8"]
            return _open[which]
        if which.startswith("f32-"):
            from f32models import variant
            wl = _models(mods, which[4:])[2]
            p = variant(W.ensure_model(wl, model_root()), model_root(), "f32")
            _open[which] = T.Model.load(p), O.OracleModel.load(p), wl
            return _open[which]
        if which == "1b":
            wl = dataclasses.replace(W.ONE_B, name="minicpm5-1b-synthetic-l1", num_hidden_layers=1)
        elif which == "4b":
            wl = dataclasses.replace(W.FOUR_B, name="minicpm5-4b-synthetic-l1", num_hidden_layers=1)
        else:
            wl = dataclasses.replace(W.ONE_B, name="llama-h1088-i2112-l1", num_hidden_layers=1, hidden_size=1088,
                                     num_attention_heads=8, num_key_value_heads=4, intermediate_size=2112,
                                     vocab_size=777, weight_seed=29)
        p = W.ensure_model(wl, model_root())
        _open[which] = T.Model.load(p), O.OracleModel.load(p), wl
    return _open[which]


def _close(a, b, what):
    d = np.abs(np.asarray(a, np.float64) - np.asarray(b, np.float64))
    assert np.all(d <= ABS_TOL + REL_TOL * np.abs(b)), f"{what}: max abs {d.max():.3e}"


def _check(mods, which, pieces):
    T, _, _ = mods
    g, o, wl = _models(mods, which)
    total = sum(pieces)
    ids = [int(t) for t in T.synth_tokens(83, total, wl.vocab_size)]
    gc, oc = T.KvCache(g, total), o.new_cache()
    at, first = 0, None
    for n in pieces:
        print(f"{which} prefill {n} at {at}", flush=True)
        a = g.forward_seq(ids[at:at + n], gc)
        first = a if first is None else first
        _close(a, o.forward_seq(ids[at:at + n], oc), f"{which} prefill {n} at {at}")
        at += n
    _close(gc.keys_flat(0), oc.keys_flat(0), "keys")
    _close(gc.values_flat(0), oc.values_flat(0), "values")
    # the order of every sum is fixed: a rerun is bitwise identical
    gc2 = T.KvCache(g, total)
    assert np.array_equal(first, g.forward_seq(ids[:pieces[0]], gc2))
    gc.close()
    gc2.close()


# lengths at and past the tiles' edges, whatever kernels they take (at 257 the
# short-prompt ones alone, at 640 four different ones;
# test_gemm_kernels_as_planned names the kernel of each of its cases)
@pytest.mark.parametrize("which,n", [("1b", 257), ("1b", 577), ("1b", 640), ("1b", 1025), ("1b", 1408),
                                     ("h1088", 577), ("h1088", 1100)])
def test_tiled_gemm_spans(mods, which, n):
    _check(mods, which, [n])


# attention with a query block's keys dealt to several workgroups: the fp32
# kernel of pieces under 256 tokens (one row and a partial column tile after a
# long context, pieces and contexts at and past the 64-key block, runs that
# lie past some of the queries), the split-bf16 kernel above
@pytest.mark.parametrize("which,pieces", [("1b", [959, 1, 64]), ("1b", [1000, 45, 130, 300]), ("1b", [448, 16, 17, 200, 65]),
                                          ("1b", [320]), ("1b", [255, 255]), ("4b", [700, 33, 2, 128])])
def test_attention_key_runs(mods, which, pieces):
    _check(mods, which, pieces)


# f32 weight matrices: the whole range of token counts takes the span kernel,
# from one row (one live wavefront column) to several tiles
@pytest.mark.parametrize("which,pieces", [("f32-1b", [1, 16]), ("f32-1b", [129, 64]), ("f32-1b", [640]),
                                          ("f32-h1088", [2, 255]), ("f32-h1088", [300])])
def test_f32_weight_gemm(mods, which, pieces):
    _check(mods, which, pieces)


# int8 codes: the row scales in the epilogues of whole and of split tiles
@pytest.mark.parametrize("n", [130, 577, 1025])
def test_i8_spans(mods, n):
    _check(mods, "i8-1b", [n])


def test_rows_before_a_non_finite_one(mods):
    # a token whose embedding is infinite makes its own row NaN and no earlier
    # one: its keys and values are masked for them, whose attention must not
    # meet 0 * NaN (the fp32 kernel's key-by-key block)
    import shutil

    from f32models import write_safetensors
    T, O, W = mods
    wl = dataclasses.replace(W.ONE_B, name="minicpm5-1b-synthetic-l2-v512", num_hidden_layers=2, vocab_size=512,
                             weight_seed=31)
    src = W.ensure_model(wl, model_root())
    d = os.path.join(model_root(), wl.name + "-inf-row")
    path = os.path.join(d, "model.safetensors")
    if not os.path.exists(path):
        os.makedirs(d, exist_ok=True)
        tensors = {}
        for name, t in O.load_safetensors(src).items():
            data = np.array(t.data)
            if name == "model.embed_tokens.weight":
                data.reshape(wl.vocab_size, -1)[7] = 0x7F80
            tensors[name] = (t.dtype, t.shape, data.tobytes())
        shutil.copy(os.path.join(os.path.dirname(src), "config.json"), os.path.join(d, "config.json"))
        write_safetensors(path, tensors)
    g = T.Model.load(path)
    ids = [8 + int(t) % 500 for t in T.synth_tokens(89, 1064, wl.vocab_size)]
    kv = []
    for last in (ids[-1], 7):
        c = T.KvCache(g, 1064)
        g.forward_seq(ids[:1000], c)
        g.forward_seq(ids[1000:1063] + [last], c)
        kv.append((c.keys_flat(1).reshape(1064, -1)[:1063], c.values_flat(1).reshape(1064, -1)[:1063]))
        c.close()
    for a, b in zip(*kv):
        assert np.all(np.isfinite(b))
        _close(b, a, "rows before the NaN one")
    g.close()


def _non_finite_model(mods):
    """Two layers; token 7's embedding is infinite, so its rows are NaN from
    the first norm on."""
    from f32models import edited
    T, O, W = mods
    wl = dataclasses.replace(W.ONE_B, name="minicpm5-1b-synthetic-l2-v512", num_hidden_layers=2, vocab_size=512,
                             weight_seed=31)

    def edit(name, w):
        if name == "model.embed_tokens.weight":
            w[7] = 0x7F80

    return edited(W.ensure_model(wl, model_root()), model_root(), wl.name + "-inf-row", edit)


# pieces that take the split-bf16 kernel, with key runs and in whole query
# blocks (as many workgroups as the chip has CUs)
@pytest.mark.parametrize("pieces", [(700, 300), (2112,), (256, 257)])
def test_rows_before_a_non_finite_one_in_a_long_piece(mods, pieces):
    T, O, W = mods
    g = T.Model.load(_non_finite_model(mods))
    n = sum(pieces)
    ids = [8 + int(t) % 500 for t in T.synth_tokens(89, n, 512)]
    kv = []
    for last in (ids[-1], 7):
        c, at = T.KvCache(g, n), 0
        for p in pieces:
            print(f"rows before token {last}: {p} at {at}", flush=True)
            g.forward_seq((ids[:-1] + [last])[at:at + p], c)
            at += p
        kv.append((c.keys_flat(1).reshape(n, -1), c.values_flat(1).reshape(n, -1)))
        c.close()
    for a, b in zip(*kv):
        assert np.all(np.isnan(b[-1])) and np.all(np.isfinite(b[:-1]))
        _close(b[:-1], a[:-1], "rows before the NaN one")
    g.close()


@pytest.mark.parametrize("piece", [64, 300])
def test_rows_after_a_run_of_non_finite_ones(mods, piece):
    # 256 tokens whose keys and values are all NaN: a run of key blocks may
    # hold nothing else, and its NaN has to reach every later row all the same
    T, O, W = mods
    g = T.Model.load(_non_finite_model(mods))
    ids = [8 + int(t) % 500 for t in T.synth_tokens(97, 640 + piece, 512)]
    ids[256:512] = [7] * 256
    c = T.KvCache(g, len(ids))
    print(f"after NaN rows: {piece}", flush=True)
    g.forward_seq(ids[:640], c)
    g.forward_seq(ids[640:], c)
    k, v = c.keys_flat(1).reshape(len(ids), -1), c.values_flat(1).reshape(len(ids), -1)
    assert np.all(np.isfinite(k[:256])) and np.all(np.isfinite(v[:256]))
    assert np.all(np.isnan(k[256:])) and np.all(np.isnan(v[256:]))
    c.close()
    g.close()


@pytest.mark.parametrize("pieces", [(1024, 64), (1024, 300)])
def test_first_keys_at_minus_infinity(mods, pieces):
    # 512 tokens whose keys score -inf against every other query (their q . k
    # overflows): the first runs of key blocks hold no weight, the later ones
    # all of it
    from f32models import edited
    T, O, W = mods
    wl = dataclasses.replace(W.ONE_B, name="minicpm5-1b-synthetic-l1-v512-s37", num_hidden_layers=1, vocab_size=512,
                             weight_seed=37)
    hd, slow = wl.head_dim, wl.head_dim // 2 - 1  # the slowest RoPE pair's first dim

    def bf16(x):
        return np.float32(x).view(np.uint32) >> 16

    def edit(name, w):
        if name == "model.embed_tokens.weight":
            w[:, :2] = 0
            w[:8, 0] = bf16(1.0)  # tokens 0-7: these keys
            w[8:, 1] = bf16(1.0)  # the others: their queries
        elif name.endswith("k_proj.weight"):
            w[slow::hd] = 0
            w[slow::hd, 0] = bf16(-5e36)
        elif name.endswith("q_proj.weight"):
            w[slow::hd] = 0
            w[slow::hd, 1] = bf16(4.0)

    p = edited(W.ensure_model(wl, model_root()), model_root(), wl.name + "-minus-inf", edit)
    g, o = T.Model.load(p), O.OracleModel.load(p)
    n = sum(pieces)
    ids = [8 + int(t) % 500 for t in T.synth_tokens(101, n, 512)]
    ids[:512] = [int(t) % 8 for t in T.synth_tokens(103, 512, 512)]
    gc, oc, at = T.KvCache(g, n), o.new_cache(), 0
    for m in pieces:
        print(f"first keys at -inf: {m} at {at}", flush=True)
        a, b = g.forward_seq(ids[at:at + m], gc), o.forward_seq(ids[at:at + m], oc)
        assert np.all(np.isfinite(b))
        _close(a, b, f"piece of {m} at {at}")
        at += m
    gc.close()
    g.close()


_SHAPES = {
    # two layers: the norm handed to QKV and from down
    "1b-l2": dict(name="minicpm5-1b-synthetic-l2-v512", num_hidden_layers=2, vocab_size=512, weight_seed=31),
    "4b-l2": dict(name="minicpm5-4b-synthetic-l2-v512", num_hidden_layers=2, vocab_size=512, weight_seed=47),
    # row counts that end a quarter into a 256-row tile, and K that is an odd
    # number of 32-wide steps there
    "h1088-i4160": dict(name="llama-h1088-i4160-l1", num_hidden_layers=1, hidden_size=1088, num_attention_heads=8,
                        num_key_value_heads=4, intermediate_size=4160, vocab_size=777, weight_seed=53),
    "h1056": dict(name="llama-h1056-i2080-l1", num_hidden_layers=1, hidden_size=1056, num_attention_heads=8,
                  num_key_value_heads=4, intermediate_size=2080, vocab_size=777, weight_seed=59),
    # one and eight query heads per KV head
    "g1": dict(name="llama-h512-q4-k4-l1", num_hidden_layers=1, hidden_size=512, num_attention_heads=4,
               num_key_value_heads=4, intermediate_size=1024, vocab_size=777, weight_seed=61),
    "g8": dict(name="llama-h512-q8-k1-l1", num_hidden_layers=1, hidden_size=512, num_attention_heads=8,
               num_key_value_heads=1, intermediate_size=1024, vocab_size=777, weight_seed=67),
}


def _shaped(mods, which):
    if which not in _open:
        T, O, W = mods
        f32 = which.startswith("f32-")
        shape = which[4:] if f32 else which
        wl = dataclasses.replace(W.FOUR_B if shape.startswith("4b") else W.ONE_B, **_SHAPES[shape])
        p = W.ensure_model(wl, model_root())
        if f32:
            from f32models import variant
            p = variant(p, model_root(), "f32")
        _open[which] = T.Model.load(p), O.OracleModel.load(p), wl
    return _open[which]


def _plan(mods, which, n, start=0):
    """{launch kind: (kernel, "whole" or "split")}; a line of tiles cut into
    spans counts as split."""
    T = mods[0]
    plan = T.prefill_plan(_shaped(mods, which)[2], n, start, which.startswith("f32-"))
    return {k: (kernel, "whole" if tiles == wgs else "split") for k, (kernel, tiles, wgs) in plan.items()}


# every GEMM kernel above 64 tokens with each epilogue and norm hand-off that it
# meets; the plan is asserted, so that a change of the estimates cannot leave a
# case on another kernel
@pytest.mark.parametrize("which,n,plan", [
    ("1b-l2", 768, {"qkv": ("gemm_dma", "whole"), "o": ("gemm_skinny_wide", "whole"), "gate_up": ("gemm_span", "split"),
                    "down": ("gemm_span", "split")}),
    ("1b-l2", 1025, {"qkv": ("gemm_span", "whole"), "o": ("gemm_dma", "whole"), "gate_up": ("gemm_big", "whole"),
                     "down": ("gemm_span", "split")}),
    ("1b-l2", 2049, {"qkv": ("gemm_span", "split"), "o": ("gemm_span", "split"), "gate_up": ("gemm_big", "whole"),
                     "down": ("gemm_span", "split")}),
    ("1b-l2", 301, {"qkv": ("gemm_skinny_wide", "whole"), "o": ("gemm_skinny_pair", "whole"),
                    "gate_up": ("gemm_skinny_wide", "whole"), "down": ("gemm_skinny_wide", "split")}),
    ("4b-l2", 128, {"qkv": ("gemm_skinny_wide", "split"), "gate_up": ("gemm_span", "split")}),
    ("4b-l2", 700, {"qkv": ("gemm_span", "split"), "o": ("gemm_skinny_wide", "whole"), "gate_up": ("gemm_big", "whole"),
                    "down": ("gemm_span", "split")}),
    ("h1088-i4160", 1025, {"qkv": ("gemm_dma", "whole"), "down": ("gemm_span", "split")}),
    ("f32-h1056", 2, {k: ("gemm_f32w_span", "split") for k in ("qkv", "o", "gate_up", "down")}),
    ("f32-h1056", 300, {k: ("gemm_f32w_span", "split") for k in ("qkv", "o", "gate_up", "down")}),
])
def test_gemm_kernels_as_planned(mods, which, n, plan):
    got = _plan(mods, which, n)
    assert {k: got[k] for k in plan} == plan
    _check(mods, which, [n])


# the attention kernels at every number of query heads per KV head, with the
# keys of a query tile dealt to several workgroups: the fp32 kernel (a partial
# column tile, one row), the split-bf16 one (a partial query block)
@pytest.mark.parametrize("which", ["g1", "1b-l2", "4b-l2", "g8"])
def test_attention_runs_per_group(mods, which):
    pieces = [1000, 67, 300, 1]
    at = pieces[0]
    for n, kernel in zip(pieces[1:], ["attn_f32", "attn_prefill", "attn_f32"]):
        assert _plan(mods, which, n, at)["attention"] == (kernel, "split")
        at += n
    _check(mods, which, pieces)
