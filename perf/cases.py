"""The workloads this library's speed is measured on, through its public API.

A case is a dict of plain values.  Three kinds cover what a program does with
the library:

- "session": one KV cache; per turn one `Model.forward_seq` of the turn's
  tokens (the first turn is a prompt, later ones continue a conversation or
  feed a long input in pieces), then `steps` calls of `Model.forward_token`
  with given ids.  Every call hands its logits to the caller, who samples or
  scores on the host.
- "generate": `generate`, greedy or sampled, with its own cache, as a
  command-line program or a one-shot request calls it.
- "batch": `generate_batch` of drafts for several prompts, then the first
  draft read into a session's cache to go on from, whose logits are returned.

Model shapes are the benchmark's (tinyminigo_amd/workloads.py): random-init
weights N(0, 0.02).  `exact` is the same model in float64 torch.
"""
from __future__ import annotations

import dataclasses
import json
import math
import os
import shutil
import struct
import tempfile

import numpy as np
import torch

import tinyminigo_amd as T
from tinyminigo_amd import workloads as W

SHAPES = {
    "tiny": W.TINY,
    "1b": W.ONE_B,
    "4b": W.FOUR_B,
    # four layers of the 1B shape, for the checkpoint type whose matrices are
    # held as f32 rows
    "1b4": dataclasses.replace(W.ONE_B, name="minicpm5-1b-synthetic-l4", num_hidden_layers=4),
}


def _session(name, model, turns, steps=0, weights="bf16"):
    return {"name": name, "kind": "session", "model": model, "weights": weights, "turns": turns, "steps": steps}


def listed():
    return [
        # the smallest model (16-token prompt, 40 tokens): every call is
        # launch and host latency
        _session("tiny_decode", "tiny", "16", 40),
        # token-by-token decoding with the caller's own sampler, short context
        _session("decode_1b", "1b", "64", 24),
        # the same after a document of some thousand tokens
        _session("decode_1b_ctx3k", "1b", "3001", 40),
        # prompts: the benchmark's short one, a ragged one of a paragraph, one
        # of a page or two, and the benchmark's longest
        _session("prefill_1b_64", "1b", "64"),
        _session("prefill_1b_301", "1b", "301"),
        _session("prefill_1b_1000", "1b", "1000"),
        _session("prefill_1b_8192", "1b", "8192"),
        # a conversation over a document: each turn continues the cache
        _session("chat_1b", "1b", "1500,45,130,20,300,75"),
        # an F16 checkpoint: a prompt and a short answer
        _session("f16_200", "1b4", "200", 12, "f16"),
        # the benchmark's sampled 4B request, 64 of its tokens
        {"name": "generate_4b", "kind": "generate", "model": "4b", "weights": "bf16", "prompt": 128, "tokens": 64,
         "temperature": 0.8, "top_k": 50, "top_p": 0.9, "penalty": 1.1},
        # nucleus sampling over the whole vocabulary; a trained model's
        # distribution is peaked, which the low temperature stands for
        {"name": "generate_1b_nucleus", "kind": "generate", "model": "1b", "weights": "bf16", "prompt": 40,
         "tokens": 48, "temperature": 0.1, "top_k": 0, "top_p": 0.95, "penalty": 1.0},
        # drafts for a queue of requests of mixed lengths
        {"name": "batch_1b", "kind": "batch", "model": "1b", "weights": "bf16",
         "prompts": "64,17,160,90,33,210,48,75,120,29,64,140", "tokens": 24},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))


def draw(rng):
    kind = rng.choice(["prefill", "prefill", "prefill", "chat", "decode", "generate", "batch"])
    model = rng.choice(["1b", "1b", "1b", "4b", "tiny"])
    most = {"1b": 8192, "4b": 2500, "tiny": 8192}[model]
    if kind == "prefill":
        pick = rng.random()
        if pick < 0.15:
            c = _session("", "1b4", str(_log(rng, 2, 1000)), rng.randint(0, 8), "f16")
        elif pick < 0.3:
            c = _session("", "1b", str(_log(rng, 2, 4000)), 0, "i8")
        else:
            c = _session("", model, str(_log(rng, 1, most)))
    elif kind == "chat":
        turns = [_log(rng, 10, most // 2)] + [_log(rng, 2, 600) for _ in range(rng.randint(1, 4))]
        c = _session("", model, ",".join(map(str, turns)), rng.randint(0, 2))
    elif kind == "decode":
        c = _session("", model, str(_log(rng, 1, 3000 if model != "4b" else 1000)), rng.randint(4, 24))
    elif kind == "generate":
        c = {"kind": "generate", "model": model, "weights": "bf16", "prompt": _log(rng, 1, 1500),
             "tokens": _log(rng, 4, 48), "temperature": rng.choice([0.0, 0.1]), "top_k": rng.choice([0, 20, 50, 200]),
             "top_p": rng.choice([0.9, 0.95, 1.0]), "penalty": rng.choice([1.0, 1.1])}
    else:
        model = rng.choice(["1b", "tiny"])
        lens = [_log(rng, 4, 300) for _ in range(_log(rng, 2, 20))]
        c = {"kind": "batch", "model": model, "weights": "bf16", "prompts": ",".join(map(str, lens)),
             "tokens": rng.randint(4, 24)}
    c.pop("name", None)
    return c


# ---- models -----------------------------------------------------------------

def _root():
    d = os.environ.get("TMG_MODEL_DIR") or os.path.join(tempfile.gettempdir(), "tmg_models")
    os.makedirs(d, exist_ok=True)
    return d


def _tensors(path):
    """name -> (dtype, shape, memory-mapped array) of a safetensors file."""
    with open(path, "rb") as f:
        n = struct.unpack("<Q", f.read(8))[0]
        head = json.loads(f.read(n))
    raw = np.memmap(path, np.uint8, "r")
    kinds = {"BF16": np.uint16, "F16": np.float16, "F32": np.float32}
    out = {}
    for name, e in head.items():
        if name != "__metadata__":
            a, b = e["data_offsets"]
            out[name] = (e["dtype"], tuple(e["shape"]), raw[8 + n + a:8 + n + b].view(kinds[e["dtype"]]))
    return out


def _f16_path(path):
    """The checkpoint with every tensor stored as F16, values below F16's
    normal range as zeros: the reference's loader reads F16 subnormals with
    another exponent than IEEE's, and the library follows it."""
    src = os.path.dirname(path)
    d = src + "-f16-flushed"
    out = os.path.join(d, "model.safetensors")
    if os.path.exists(out):
        return out
    os.makedirs(d, exist_ok=True)
    shutil.copy(os.path.join(src, "config.json"), os.path.join(d, "config.json"))
    tensors, head, off = _tensors(path), {}, 0
    for name, (_, shape, data) in tensors.items():
        head[name] = {"dtype": "F16", "shape": list(shape), "data_offsets": [off, off + 2 * data.size]}
        off += 2 * data.size
    text = json.dumps(head).encode()
    text += b" " * ((8 - len(text) % 8) % 8)
    with open(out + ".part", "wb") as f:
        f.write(struct.pack("<Q", len(text)) + text)
        for name, (kind, _, data) in tensors.items():
            wide = (data.astype(np.uint32) << 16).view(np.float32) if kind == "BF16" else np.asarray(data, np.float32)
            f.write(np.where(np.abs(wide) < 2.0 ** -14, np.float32(0), wide).astype(np.float16).tobytes())
    os.replace(out + ".part", out)
    return out


def _path(case):
    p = W.ensure_model(SHAPES[case["model"]], _root())
    return _f16_path(p) if case["weights"] == "f16" else p


_models = {}


def _model(case):
    """The loaded model: a program loads it once and serves every request."""
    key = (case["model"], case["weights"])
    if key not in _models:
        os.environ["TMG_I8"] = "1" if case["weights"] == "i8" else "0"
        try:
            _models[key] = T.Model.load(_path(case))
        finally:
            del os.environ["TMG_I8"]
    return _models[key]


# ---- one pass ---------------------------------------------------------------

def _ints(text):
    return [int(x) for x in text.split(",")]


def _ids(case, seed, n, salt=0):
    return T.synth_tokens(1 + seed * 64 + salt, n, SHAPES[case["model"]].vocab_size)


def prepare(case, seed):
    m = _model(case)
    s = {"case": case, "model": m}
    if case["kind"] == "session":
        turns = _ints(case["turns"])
        s["turns"] = [_ids(case, seed, n, i) for i, n in enumerate(turns)]
        s["forced"] = [[int(t) for t in _ids(case, seed, case["steps"], 32 + i)] for i in range(len(turns))]
        total = sum(turns) + len(turns) * case["steps"]
        s["cache"] = m.new_cache((total + 63) // 64 * 64)
    elif case["kind"] == "generate":
        s["prompt"] = _ids(case, seed, case["prompt"])
        s["params"] = T.GenParams(max_tokens=case["tokens"], temperature=case["temperature"], top_k=case["top_k"],
                                  top_p=case["top_p"], repetition_penalty=case["penalty"], seed=seed)
    else:
        lens = _ints(case["prompts"])
        s["prompts"] = [_ids(case, seed, n, i) for i, n in enumerate(lens)]
        s["cache"] = m.new_cache((lens[0] + case["tokens"] + 63) // 64 * 64)
    return s


def run(s):
    case, m = s["case"], s["model"]
    if case["kind"] == "session":
        cache, out = s["cache"], []
        cache.reset()
        for turn, forced in zip(s["turns"], s["forced"]):
            out.append(m.forward_seq(turn, cache))
            for t in forced:
                out.append(m.forward_token(t, cache))
        return out
    if case["kind"] == "generate":
        g = T.generate(m, s["prompt"], s["params"])
        return {"tokens": np.asarray(g.tokens, np.int64), "logits": g.logits_first_step}
    drafts, _ = T.generate_batch(m, s["prompts"], case["tokens"])
    s["cache"].reset()
    text = np.concatenate([s["prompts"][0], np.asarray(drafts[0], np.uint32)])
    logits = m.forward_seq(text, s["cache"])
    return {"tokens": np.asarray([t for d in drafts for t in d], np.int64), "logits": logits}


# ---- what a pass cannot do without ------------------------------------------

def _call(w, case, new, ctx):
    """(bytes, flops) of one call that takes `new` tokens after `ctx`: the
    weights and the cached K/V once, the new K/V rows and one row of logits."""
    H, I, V, L = w.hidden_size, w.intermediate_size, w.vocab_size, w.num_hidden_layers
    qd, kvd = w.num_attention_heads * w.head_dim, w.num_key_value_heads * w.head_dim
    per_layer = qd * H + 2 * kvd * H + H * qd + 3 * H * I
    size = {"bf16": 2, "f16": 2, "i8": 1}[case["weights"]]
    head = 2 * V * H
    nbytes = L * per_layer * size + head + (2 * L + 1) * H * 4 + 2 * L * (ctx + new) * kvd * 4 + new * H * 2 + V * 4
    pairs = new * ctx + new * (new + 1) / 2
    flops = 2.0 * new * per_layer * L + 2.0 * V * H + 4.0 * L * qd * pairs
    return nbytes, flops


def work(case):
    w = SHAPES[case["model"]]
    calls = []
    if case["kind"] == "session":
        at = 0
        for n in _ints(case["turns"]):
            calls.append((n, at))
            at += n
            for _ in range(case["steps"]):
                calls.append((1, at))
                at += 1
        costs = [_call(w, case, n, at) for n, at in calls]
        return {"bytes": sum(c[0] for c in costs), "flops": sum(c[1] for c in costs)}
    if case["kind"] == "generate":
        costs = [_call(w, case, case["prompt"], 0)]
        costs += [_call(w, case, 1, case["prompt"] + i) for i in range(case["tokens"])]
        return {"bytes": sum(c[0] for c in costs), "flops": sum(c[1] for c in costs)}
    lens, n = _ints(case["prompts"]), case["tokens"]
    kvd = w.num_key_value_heads * w.head_dim
    one = _call(w, case, 1, 0)[0]
    # the prompts together, each step's sequences together, then the first draft
    nbytes = one + 2 * w.num_hidden_layers * kvd * 4 * sum(lens)
    flops = sum(_call(w, case, p, 0)[1] for p in lens)
    for i in range(n - 1):
        nbytes += one + 2 * w.num_hidden_layers * kvd * 4 * sum(p + i for p in lens)
        flops += sum(_call(w, case, 1, p + i)[1] for p in lens)
    last = _call(w, case, lens[0] + n, 0)
    return {"bytes": nbytes + last[0], "flops": flops + last[1]}


def tolerance(case):
    """Prompts go through the matrix cores as split-bf16 pairs, which leave
    2^-18 of an activation out; after the layers the logits are 1.1e-5 to
    3.1e-5 from float64 (1.2e-6 to 4e-6 for the tiny model), and two ways of
    summing are up to that much apart.  Four times this, and a largest
    difference of five times the 2-norm's."""
    rel = 1.6e-5 if case["model"] == "tiny" else 1.2e-4
    return {"rel": rel, "max": 5 * rel, "differ": 0.01}


# ---- the same in float64 ----------------------------------------------------

def _rope(w, n):
    """cos and sin of the f32 angles a Llama RoPE table holds."""
    half = w.head_dim // 2
    freq = np.array([np.float32(1) / np.float32(w.rope_theta ** (2.0 * i / w.head_dim)) for i in range(half)], np.float32)
    ang = (np.arange(n, dtype=np.float32)[:, None] * freq[None, :]).astype(np.float64)
    return torch.from_numpy(np.cos(ang)).cuda(), torch.from_numpy(np.sin(ang)).cuda()


def _wide(entry, i8=False):
    kind, shape, data = entry
    t = torch.from_numpy(np.array(data.view(np.int16) if kind == "BF16" else data)).cuda()
    t = (t.view(torch.bfloat16) if kind == "BF16" else t).reshape(shape)
    if not i8:
        return t.double()
    f = t.float()
    top = f.abs().amax(1, keepdim=True)
    # a tensor divisor: torch multiplies by the reciprocal of a number, and
    # codes at exact halves hang on the last bit of the scale
    scale = torch.where(top > 0, top / torch.full_like(top, 127.0), torch.ones_like(top))
    q = f / scale
    q = torch.sign(q) * torch.floor(q.abs().double() + 0.5)
    return q.clamp(-127, 127) * scale.double()


def _logits64(case, ids, rows):
    """Logits of the given positions of one causal pass over ids."""
    w, ts = SHAPES[case["model"]], _tensors(_path(case))
    i8 = case["weights"] == "i8"
    n, hd, nq, nkv = len(ids), w.head_dim, w.num_attention_heads, w.num_key_value_heads
    cos, sin = (t[:, None, :] for t in _rope(w, n))

    def norm(x, name):
        g = _wide(ts[name])
        return x / torch.sqrt((x * x).mean(1, keepdim=True) + float(np.float32(w.rms_norm_eps))) * g

    def turn(x):
        a, b = x[..., :hd // 2], x[..., hd // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    table = _wide(ts["model.embed_tokens.weight"])
    x = table[torch.from_numpy(np.asarray(ids, np.int64)).cuda()]
    for l in range(w.num_hidden_layers):
        p = "model.layers.%d." % l

        def mat(name):
            return _wide(ts[p + name], i8).t().contiguous()

        h = norm(x, p + "input_layernorm.weight")
        q = turn((h @ mat("self_attn.q_proj.weight")).reshape(n, nq, hd)).permute(1, 0, 2).contiguous()
        k = turn((h @ mat("self_attn.k_proj.weight")).reshape(n, nkv, hd)).permute(1, 2, 0).contiguous()
        v = (h @ mat("self_attn.v_proj.weight")).reshape(n, nkv, hd).permute(1, 0, 2).contiguous()
        o = torch.empty(n, nq * hd, dtype=torch.float64, device="cuda")
        step, group = 512, nq // nkv
        for i in range(0, n, step):
            e = min(n, i + step)
            late = torch.arange(e, device="cuda")[None, :] > torch.arange(i, e, device="cuda")[:, None]
            for g in range(nkv):
                a = q[g * group:(g + 1) * group, i:e].reshape(-1, hd) @ k[g, :, :e].contiguous() / math.sqrt(hd)
                a = a.reshape(group, e - i, e).masked_fill(late, -math.inf).softmax(-1)
                b = (a.reshape(-1, e) @ v[g, :e]).reshape(group, e - i, hd)
                o[i:e, g * group * hd:(g + 1) * group * hd] = b.permute(1, 0, 2).reshape(e - i, group * hd)
        x = x + o @ mat("self_attn.o_proj.weight")
        h = norm(x, p + "post_attention_layernorm.weight")
        g = h @ mat("mlp.gate_proj.weight")
        x = x + (g * torch.sigmoid(g) * (h @ mat("mlp.up_proj.weight"))) @ mat("mlp.down_proj.weight")
    h = norm(x, "model.norm.weight")[torch.tensor(rows, device="cuda")]
    head = table if "lm_head.weight" not in ts else _wide(ts["lm_head.weight"])
    return (h @ head.t().contiguous()).cpu().numpy()


def exact(case, seed):
    if case["kind"] == "generate":
        ids = _ids(case, seed, case["prompt"])
        return {"tokens": None, "logits": _logits64(case, ids, [len(ids) - 1])[0]}
    if case["kind"] == "batch":
        return None  # the drafts decide what the logits are of
    ids, rows = [], []
    for i, n in enumerate(_ints(case["turns"])):
        ids += [int(t) for t in _ids(case, seed, n, i)]
        rows.append(len(ids) - 1)
        for t in _ids(case, seed, case["steps"], 32 + i):
            ids.append(int(t))
            rows.append(len(ids) - 1)
    return list(_logits64(case, ids, rows))
