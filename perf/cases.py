"""What a user of this library has it do, as cases to time and to compare.

The shapes are the Qwen2.5-0.5B decoder's (hidden 896, 14 query and 2 KV heads of 64,
intermediate 4,864, vocabulary 151,936, 24 layers) over 16-token KV pages. Kinds of case,
each through the package's public calls:

  decode   one layer's decode step on the cache (RoPE + append + attention): one launch for
           16-bit caches, rope_and_cache + attention for f32 ones, with a host-built work
           list, as the engine runs it
  prompt   one layer's prompt step on the cache (RoPE + append + prefill attention), the
           rows continuing `start` cached positions
  proj     the projections around attention: rmsnorm + q/k/v, and o_proj into the residual
  mlp      rmsnorm + gate/up + SiLU, and down into the residual
  head     final norm, LM head and greedy token of the rows that want one
  step     a whole forward step of a 24-layer model, decode (a recorded graph, replayed
           per step as the engine does) or prompt, to logits and tokens

Every number is drawn on the GPU from the seed alone.
"""
from __future__ import annotations

import importlib
import math

import numpy as np
import torch

ie = importlib.import_module("llm-inference-engine_amd")

HIDDEN, INTER, VOCAB, LAYERS = 896, 4864, 151936, 24
NH, NKV, HD, THETA, EPS, PAGE = 14, 2, 64, 1e6, 1e-6, 16
QD, KVD = NH * HD, NKV * HD
KV = {"f32": (ie.KV_F32, torch.float32), "f16": (ie.KV_F16, torch.float16),
      "bf16": (ie.KV_BF16, torch.bfloat16)}
KV_BYTES = {"f32": 4, "f16": 2, "bf16": 2}
W_BYTES = {"bf16": 2, "int8": 1}
DEV = "cuda"


# ------------------------------------------------------------------ cases ----
def listed():
    return [
        # The smallest call: one user's short chat, one layer's step on the cache.
        dict(name="decode_b1_short", kind="decode", rows=1, lo=600, hi=600, kv="f16"),
        # A full serving batch of ragged contexts, the engine's headline step.
        dict(name="decode_b64", kind="decode", rows=64, lo=128, hi=4096, kv="f16"),
        # One user with a long document in its context.
        dict(name="decode_b1_32k", kind="decode", rows=1, lo=32768, hi=32768, kv="bf16"),
        # The default f32 cache, a batch of middling contexts.
        dict(name="decode_b48_f32", kind="decode", rows=48, lo=256, hi=2048, kv="f32"),
        # A long prompt into an empty 16-bit cache.
        dict(name="prompt_4000", kind="prompt", rows=4000, start=0, kv="f16"),
        # The next turn of a chat on the default f32 cache: an odd number of rows that
        # continues a cached history.
        dict(name="prompt_1333_f32", kind="prompt", rows=1333, start=1000, kv="f32"),
        # Projections of a long prompt.
        dict(name="proj_4000", kind="proj", rows=4000, weights="bf16"),
        # The MLP of a small decode batch, and of an odd prompt with INT8 weights.
        dict(name="mlp_8", kind="mlp", rows=8, weights="bf16"),
        dict(name="mlp_1501_int8", kind="mlp", rows=1501, weights="int8"),
        # The vocabulary projection and the greedy choice of a full decode batch.
        dict(name="head_64", kind="head", rows=64, weights="bf16"),
        # Whole steps: a full decode batch, and the prompt a chat opens with.
        dict(name="step_b64", kind="step", mode="decode", rows=64, lo=128, hi=4096, kv="f16",
             weights="bf16"),
        dict(name="step_prompt_600_int8", kind="step", mode="prompt", rows=600, start=0, kv="f16",
             weights="int8"),
    ]


def _log_int(rng, lo, hi):
    return int(min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the listed ones' ranges: batches 1 to 64, contexts to 32,768 (the
    batch's total kept to 262,144), prompts of 16 to 4,000 rows, every cache and weight type."""
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "proj", "mlp", "mlp", "head", "step"])
    kv = rng.choice(["f32", "f16", "bf16"])
    weights = rng.choice(["bf16", "int8"])
    if kind == "decode":
        rows = _log_int(rng, 1, 64)
        hi = _log_int(rng, 64, min(32768, 262144 // rows))
        return dict(kind=kind, rows=rows, lo=max(1, hi // rng.choice([1, 3, 16])), hi=hi, kv=kv)
    if kind == "prompt":
        rows = _log_int(rng, 16, 4000 if kv != "f32" else 2000)
        start = rng.choice([0, _log_int(rng, 1, 2000)])
        return dict(kind=kind, rows=rows, start=min(start, 4000 - rows), kv=kv)
    if kind in ("proj", "mlp"):
        return dict(kind=kind, rows=_log_int(rng, 1, 4000), weights=weights)
    if kind == "head":
        return dict(kind=kind, rows=_log_int(rng, 1, 64), weights=weights)
    if rng.random() < 0.6:
        rows = _log_int(rng, 1, 64)
        hi = _log_int(rng, 64, 4096)
        return dict(kind=kind, mode="decode", rows=rows, lo=max(1, hi // 8), hi=hi,
                    kv=rng.choice(["f16", "bf16"]), weights=weights)
    return dict(kind=kind, mode="prompt", rows=_log_int(rng, 16, 600), start=0,
                kv=rng.choice(["f16", "bf16"]), weights=weights)


# ----------------------------------------------------------------- inputs ----
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _normal(g, shape, scale=1.0):
    return torch.randn(shape, generator=g, device=DEV) * scale


def _activations(g, rows, cols):
    """Residual-stream rows: unit scale, with a few channels some ten times larger, as
    decoders have them."""
    x = _normal(g, (rows, cols))
    x[:, torch.randperm(cols, generator=g, device=DEV)[: cols // 128]] *= 12.0
    return x


def _weights(g, rows, cols, fmt):
    """(values, row scales or None) of a [rows, cols] matrix that keeps unit scale."""
    w = _normal(g, (rows, cols), 1.0 / math.sqrt(cols))
    if fmt == "bf16":
        return w.bfloat16(), None
    scale = w.abs().amax(dim=1) / 127.0
    return torch.round(w / scale[:, None]).to(torch.int8), scale.contiguous()


def _lens(case, seed):
    """Contexts evenly spread over [lo, hi] (its end always among them), in a drawn order."""
    n = np.linspace(case["hi"], case["lo"], case["rows"]).astype(np.int64)
    return np.random.default_rng(seed).permutation(n)


def _cache(g, seed, lens, kv, layers=1):
    """Pools of normal values and block tables whose pages are a shuffled permutation."""
    max_pages = (int(max(lens)) + PAGE - 1) // PAGE
    need = [(int(n) + PAGE - 1) // PAGE for n in lens]
    num_pages = sum(need)
    order = np.random.default_rng(seed + 1).permutation(num_pages).astype(np.int32)
    tables = np.zeros((len(lens), max_pages), np.int32)
    at = 0
    for s, n in enumerate(need):
        tables[s, :n] = order[at:at + n]
        at += n
    shape = (num_pages * PAGE, KVD)
    pools = [(_normal(g, shape).to(KV[kv][1]), _normal(g, shape).to(KV[kv][1]))
             for _ in range(layers)]
    return tables, max_pages, pools


def _row_ids(case, seed):
    """Sequence lengths after the step, and each row's position and sequence."""
    if case["kind"] == "prompt" or case.get("mode") == "prompt":
        lens = [case["start"] + case["rows"]]
        pos = np.arange(case["start"], lens[0], dtype=np.int32)
        return lens, pos, np.zeros(case["rows"], np.int32)
    lens = _lens(case, seed)
    return lens, (lens - 1).astype(np.int32), np.arange(case["rows"], dtype=np.int32)


def _to(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _matrix(w):
    return ie.matrix(w[0], w[1])


def _layer_weights(g, fmt):
    return dict(norm1=1.0 + _normal(g, (HIDDEN,), 0.1), norm2=1.0 + _normal(g, (HIDDEN,), 0.1),
                wqkv=_weights(g, QD + 2 * KVD, HIDDEN, fmt), bqkv=_normal(g, (QD + 2 * KVD,), 0.5),
                wo=_weights(g, HIDDEN, QD, fmt), wg=_weights(g, INTER, HIDDEN, fmt),
                wu=_weights(g, INTER, HIDDEN, fmt), wd=_weights(g, HIDDEN, INTER, fmt))


def _inputs(case, seed):
    """The case's inputs, from the seed alone: what both prepare() and exact() start from."""
    g, kind, rows = _gen(seed), case["kind"], case["rows"]
    i = {}
    if kind in ("decode", "prompt", "step"):
        lens, i["pos"], i["seq"] = _row_ids(case, seed)
        i["tables"], i["max_pages"], i["pools"] = _cache(g, seed, lens, case["kv"],
                                                         LAYERS if kind == "step" else 1)
        i["max_len"] = int(max(lens))
    if kind in ("decode", "prompt"):
        i["q"], i["k"], i["v"] = (_normal(g, (rows, n)) for n in (QD, KVD, KVD))
    if kind in ("proj", "mlp"):
        i["x"] = _activations(g, rows, HIDDEN)
        i["attn"] = _normal(g, (rows, QD))
        i["w"] = _layer_weights(g, case["weights"])
    if kind in ("head", "step"):
        i["final_norm"] = 1.0 + _normal(g, (HIDDEN,), 0.1)
        i["embed"] = _weights(g, VOCAB, HIDDEN, case["weights"])
    if kind == "head":
        i["x"] = _activations(g, rows, HIDDEN)
    if kind == "step":
        i["ids"] = torch.randint(0, VOCAB, (rows,), generator=g, device=DEV, dtype=torch.int32)
        i["layers"] = [_layer_weights(g, case["weights"]) for _ in range(LAYERS)]
    return i


# ------------------------------------------------------------ the calls ----
class _Paged:
    """What a program keeps for its cache: device tables, rows, work list, workspace."""

    def __init__(self, case, i):
        self.prompt = case["kind"] == "prompt" or case.get("mode") == "prompt"
        self.f32 = case["kv"] == "f32"
        self.max_pages, self.pools = i["max_pages"], i["pools"]
        self.pos, self.seq, self.tables = _to(i["pos"]), _to(i["seq"]), _to(i["tables"])
        self.rope = ie.rope_table(i["max_len"], HD, THETA).to(DEV)
        self.out = torch.empty((case["rows"], QD), device=DEV)
        if not self.prompt:
            self.chunk = ie.attention_chunk_tokens(case["rows"], case["hi"], KV[case["kv"]][0])
            self.chunks = ie.attention_chunks(i["max_len"], self.chunk)
            self.workspace = ie.attention_workspace(case["rows"], NH, HD, self.chunks)
            self.plan = _to(ie.attention_plan(i["pos"], i["seq"], i["tables"], self.chunks,
                                              self.chunk))

    def attend(self, q, k, v, layer=0):
        kp, vp = self.pools[layer]
        rows = (self.pos, self.seq, self.tables, self.max_pages)
        heads = (NH, NKV, HD)
        if self.f32:
            ie.rope_and_cache(q, k, v, kp, vp, self.rope, *rows, *heads)
        if self.prompt:
            if self.f32:
                ie.attention_prefill(self.out, q, kp, vp, *rows, *heads)
            else:
                ie.rope_cache_attention_prefill(self.out, q, k, v, kp, vp, self.rope, *rows, *heads)
            return self.out
        split = (self.chunks, self.chunk, self.workspace, self.plan)
        if self.f32:
            ie.attention_planned(self.out, q, kp, vp, *rows, *split, *heads)
        else:
            ie.rope_cache_attention_planned(self.out, q, k, v, kp, vp, self.rope, *rows, *split,
                                            *heads)
        return self.out


def _layer_handles(w):
    return dict(w, wqkv=_matrix(w["wqkv"]), wo=_matrix(w["wo"]), wg=_matrix(w["wg"]),
                wu=_matrix(w["wu"]), wd=_matrix(w["wd"]))


def _project(s, x, w):
    ie.rmsnorm_qkv_proj(s["q"], s["k"], s["v"], x, w["norm1"], EPS, w["wqkv"], w["bqkv"])


def _mlp(s, x, w):
    ie.rmsnorm_gate_up_silu(s["mid"], x, w["norm2"], EPS, w["wg"], w["wu"])
    ie.matmul(x, s["mid"], w["wd"], accumulate=True)


def _head(s):
    ie.gather_rows(s["xg"], s["x"], s["logit_rows"])
    ie.rmsnorm(s["xg"], s["xg"], s["final_norm"], EPS)
    ie.matmul(s["logits"], s["xg"], s["head"])
    ie.argmax_rows(s["tokens"], s["logits"])


def _forward(s):
    """A whole step of the model, the work the engine and its LayerBody enqueue."""
    ie.embedding(s["x"], s["ids"], s["head"])
    for l, w in enumerate(s["layers"]):
        _project(s, s["x"], w)
        attn = s["paged"].attend(s["q"], s["k"], s["v"], l)
        ie.matmul(s["x"], attn, w["wo"], accumulate=True)
        _mlp(s, s["x"], w)
    _head(s)


def prepare(case, seed):
    i = _inputs(case, seed)
    rows, kind = case["rows"], case["kind"]
    s = dict(kind=kind, keep=i)
    empty = lambda *shape: torch.empty(shape, device=DEV)
    if kind in ("decode", "prompt"):
        s.update(paged=_Paged(case, i), q=i["q"], k=i["k"], v=i["v"])
        if case["kv"] == "f32":  # rope_and_cache rotates q in place
            s["q_rot"] = empty(rows, QD)
    if kind in ("proj", "step"):
        s.update(q=empty(rows, QD), k=empty(rows, KVD), v=empty(rows, KVD))
    if kind in ("mlp", "step"):
        s["mid"] = empty(rows, INTER)
    if kind in ("proj", "mlp"):
        s.update(x=i["x"], attn=i["attn"], residual=empty(rows, HIDDEN), w=_layer_handles(i["w"]))
    if kind in ("head", "step"):
        n = rows if kind == "head" or case["mode"] == "decode" else 1
        s.update(xg=empty(n, HIDDEN), logits=empty(n, VOCAB), final_norm=i["final_norm"],
                 head=_matrix(i["embed"]), tokens=torch.empty(n, dtype=torch.int32, device=DEV),
                 logit_rows=torch.arange(rows - n, rows, dtype=torch.int32, device=DEV))
    if kind == "head":
        s["x"] = i["x"]
    if kind == "step":
        s.update(x=empty(rows, HIDDEN), ids=i["ids"], paged=_Paged(case, i),
                 layers=[_layer_handles(w) for w in i["layers"]])
        if case["mode"] == "decode":  # decode steps replay a recorded graph
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                _forward(s)
            side.synchronize()
            s["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s["graph"], stream=side):
                _forward(s)
    return s


def run(s):
    kind = s["kind"]
    if kind in ("decode", "prompt"):
        q = s["q"]
        if "q_rot" in s:
            q = s["q_rot"]
            q.copy_(s["q"])
        return [s["paged"].attend(q, s["k"], s["v"]), *s["paged"].pools[0]]
    if kind == "proj":
        _project(s, s["x"], s["w"])
        s["residual"].copy_(s["x"])
        ie.matmul(s["residual"], s["attn"], s["w"]["wo"], accumulate=True)
        return [s["q"], s["k"], s["v"], s["residual"]]
    if kind == "mlp":
        s["residual"].copy_(s["x"])
        _mlp(s, s["residual"], s["w"])
        return [s["mid"], s["residual"]]
    if kind == "head":
        _head(s)
        return [s["logits"], s["tokens"]]
    if "graph" in s:
        s["graph"].replay()
    else:
        _forward(s)
    return [s["logits"], s["tokens"], s["x"]]


# ------------------------------------------------------------- the cost ----
def _dense_work(T, rows, cols, fmt):
    return rows * cols * W_BYTES[fmt] + (rows * 4 if fmt == "int8" else 0), 2 * T * rows * cols


def _attention_work(case):
    """K/V rows read, rows appended, q read and out written; the products of scores and values."""
    T, b = case["rows"], 2 * KVD * KV_BYTES[case["kv"]]
    if case["kind"] == "prompt" or case.get("mode") == "prompt":
        keys = case["start"]
        pairs = T * case["start"] + T * (T + 1) // 2
    else:
        keys = pairs = int(_lens(case, 0).sum())
    io = T * (2 * QD + 2 * KVD) * 4 + T * 8 + keys // PAGE * 4
    return keys * b + T * b + io, 4 * NH * HD * pairs


def work(case):
    T, kind = case["rows"], case["kind"]
    if kind in ("decode", "prompt"):
        b, f = _attention_work(case)
        return {"bytes": b, "flops": f}
    fmt = case["weights"]
    qkv, o = _dense_work(T, QD + 2 * KVD, HIDDEN, fmt), _dense_work(T, HIDDEN, QD, fmt)
    gu, down = _dense_work(T, 2 * INTER, HIDDEN, fmt), _dense_work(T, HIDDEN, INTER, fmt)
    if kind == "proj":
        io = T * (2 * HIDDEN + 2 * QD + 2 * KVD + HIDDEN) * 4
        return {"bytes": qkv[0] + o[0] + io, "flops": qkv[1] + o[1]}
    if kind == "mlp":
        io = T * (2 * HIDDEN + INTER) * 4
        return {"bytes": gu[0] + down[0] + io, "flops": gu[1] + down[1]}
    n = T if kind == "head" or case["mode"] == "decode" else 1
    head = _dense_work(n, VOCAB, HIDDEN, fmt)
    if kind == "head":
        return {"bytes": head[0] + n * (HIDDEN + VOCAB + 1) * 4, "flops": head[1]}
    b, f = _attention_work(case)
    b -= T * (2 * QD + 2 * KVD) * 4  # activations between the ops need not leave the chip
    dense = [sum(p[j] for p in (qkv, o, gu, down)) for j in (0, 1)]
    return {"bytes": LAYERS * (b + dense[0]) + head[0] + n * VOCAB * 4 + T * HIDDEN * W_BYTES[fmt],
            "flops": LAYERS * (f + dense[1]) + head[1]}


def tolerance(case):
    kind, kv = case["kind"], case.get("kv")
    if kind == "step":
        # Pages (and, in prompts on f16 caches, attention weights) are rounded to 16 bits,
        # and a value that rounds the other way travels through the layers after it: 6e-5
        # against float64 on f16 caches, a few times that on bf16 ones. Tokens may differ
        # where two logits tie to that error.
        return {"rel": 1e-3, "max": 2e-2, "differ": 0.05}
    if kind == "head":
        return {"rel": 1e-6, "max": 2e-5, "differ": 0.02}  # f32 sums: 2e-7 against float64
    if kind in ("proj", "mlp"):
        return {"rel": 1e-6, "max": 2e-5}  # as the head's
    if kv == "f32":
        return {"rel": 3e-6, "max": 1e-4}  # 2e-7 (decode) to 8e-7 (prompt) against float64
    if kind == "prompt" and kv == "f16":
        return {"rel": 1e-3, "max": 2e-2}  # weights and q enter as f16: 2.5e-4
    return {"rel": 2e-5, "max": 8e-3}  # 3e-6 (bf16); a page value may round the other way


# ------------------------------------------------- the same in 64 bits ----
def _rope64(x, pos, heads):
    """Rotated rows in float64, by the float32 angles that the rotation table is defined by."""
    expo = (np.arange(0, HD, 2, dtype=np.float32) / np.float32(HD)).astype(np.float64)
    inv = np.float32(1) / (THETA ** expo).astype(np.float32)
    ang = (np.asarray(pos, np.float32)[:, None] * inv[None, :]).astype(np.float32)
    c = torch.from_numpy(np.cos(ang.astype(np.float64))).to(DEV)[:, None, :]
    s = torch.from_numpy(np.sin(ang.astype(np.float64))).to(DEV)[:, None, :]
    x = x.double().view(len(pos), heads, HD)
    a, b = x[..., : HD // 2], x[..., HD // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], dim=-1).reshape(len(pos), heads * HD)


def _attend64(i, q, k, v, kv, prompt, layer=0):
    """The step's attention in float64 over pages that hold values of the cache's own type."""
    dt = KV[kv][1]
    kp, vp = (p.clone() for p in i["pools"][layer])
    pos, seq, tables = i["pos"], i["seq"], i["tables"]
    slots = _to((tables[seq, pos // PAGE].astype(np.int64) * PAGE + pos % PAGE))
    kp[slots] = _rope64(k, pos, NKV).float().to(dt)
    vp[slots] = v.float().to(dt)
    q = _rope64(q, pos, NH).view(-1, NH, HD)
    out = torch.empty_like(q)

    def rows_of(s, n):
        p = np.arange(n)
        at = _to(tables[s, p // PAGE].astype(np.int64) * PAGE + p % PAGE)
        return kp[at].double().view(n, NKV, HD), vp[at].double().view(n, NKV, HD)

    if prompt:
        kk, vv = rows_of(0, int(pos[-1]) + 1)
        hidden = torch.arange(kk.shape[0], device=DEV)[None, :] > _to(pos.astype(np.int64))[:, None]
        for h in range(NH):
            kv_h = h // (NH // NKV)
            sc = (q[:, h] @ kk[:, kv_h].t()) / math.sqrt(HD)
            out[:, h] = torch.softmax(sc.masked_fill(hidden, -math.inf), dim=-1) @ vv[:, kv_h]
    else:
        for t in range(len(pos)):
            kk, vv = rows_of(int(seq[t]), int(pos[t]) + 1)
            for j in range(NKV):
                hs = slice(j * (NH // NKV), (j + 1) * (NH // NKV))
                w = torch.softmax((q[t, hs] @ kk[:, j].t()) / math.sqrt(HD), dim=-1)
                out[t, hs] = w @ vv[:, j]
    return out.view(-1, QD), kp, vp


def _dense64(x, w):
    y = x @ w[0].double().t()
    return y if w[1] is None else y * w[1].double()[None, :]


def _norm64(x, w):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + EPS) * w.double()


def _project64(x, w):
    y = _dense64(_norm64(x, w["norm1"]), w["wqkv"]) + w["bqkv"].double()
    return torch.split(y, [QD, KVD, KVD], dim=1)


def _mlp64(x, w):
    xn = _norm64(x, w["norm2"])
    mid = torch.nn.functional.silu(_dense64(xn, w["wg"])) * _dense64(xn, w["wu"])
    return mid, x + _dense64(mid, w["wd"])


def exact(case, seed):
    i = _inputs(case, seed)
    kind, prompt = case["kind"], case["kind"] == "prompt" or case.get("mode") == "prompt"
    if kind in ("decode", "prompt"):
        return list(_attend64(i, i["q"], i["k"], i["v"], case["kv"], prompt))
    if kind == "proj":
        x = i["x"].double()
        return [*_project64(x, i["w"]), x + _dense64(i["attn"].double(), i["w"]["wo"])]
    if kind == "mlp":
        return list(_mlp64(i["x"].double(), i["w"]))
    if kind == "head":
        x = i["x"].double()
    else:
        ids = i["ids"].long()
        x = i["embed"][0][ids].double()
        if i["embed"][1] is not None:
            x = x * i["embed"][1][ids].double()[:, None]
        for l, w in enumerate(i["layers"]):
            q, k, v = _project64(x, w)
            x = x + _dense64(_attend64(i, q, k, v, case["kv"], prompt, l)[0], w["wo"])
            x = _mlp64(x, w)[1]
    last = x[-1:] if kind == "step" and prompt else x
    logits = _dense64(_norm64(last, i["final_norm"]), i["embed"])
    out = [logits, torch.argmax(logits, dim=-1).int()]
    return out + [x] if kind == "step" else out
