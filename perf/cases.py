"""The work that users of this library have it do, as cases that can be timed and checked.

Kinds of case (key "kind"), each one pass through public entry points:

  decode        Ops.paged_attention: one query per sequence over its paged KV
  mixed         Ops.paged_attention_varlen: prompt chunks and decodes in one batch
  kv            Ops.paged_kv_append_gather: one new token per sequence into its
                page, then every context out as rows
  attention     Ops.self_attention over contiguous keys (L queries, S keys)
  layer         a decoder layer written with the ops: norm, q/k/v, RoPE into the
                caches, self_attention, o, residual, norm, gate, up, SwiGLU,
                down, residual
  linear        Ops.linear
  head          the last rows' norm, the packed LM head and the argmax
  model_decode  Qwen2.fork / step / free: teacher-forced decode steps of a batch
  model_prompt  Qwen2.create_sequence / step / free: fresh prompts

Sizes are the Qwen2-1.5B shape the benchmark and the tests use (hidden 1536, 12
query and 2 KV heads of 128, FFN 8960, vocabulary 151936) and odd neighbours of
it; the models have few layers, because a rounding difference in one layer
travels through all that follow. Lengths within a batch are spread evenly over
their range and shuffled by the seed, so a case's work does not depend on it.
"""
import math

import numpy as np
import torch

from llaisys_amd import DataType, DeviceType, MemcpyKind, Ops, RuntimeAPI, Tensor
from llaisys_amd.models import Qwen2
from llaisys_amd.models.qwen2 import Qwen2Meta

HEAD = 128   # the paged KV's head dim
PAGE = 16    # tokens of a page
THETA = 10000.0
EPS = 1e-6

_TYPES = {"f32": (torch.float32, DataType.F32), "f16": (torch.float16, DataType.F16),
          "bf16": (torch.bfloat16, DataType.BF16)}
_LL = {torch.float32: DataType.F32, torch.float16: DataType.F16, torch.bfloat16: DataType.BF16,
       torch.int32: DataType.I32, torch.int64: DataType.I64}
_BYTES = {"f32": 4, "f16": 2, "bf16": 2}


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # A single chat's next token: one sequence, a short context; latency.
        {"name": "decode_one", "kind": "decode", "batch": 1, "ctx_lo": 700, "ctx_hi": 700, "nh": 12, "nkvh": 2,
         "out": "bf16"},
        # The benchmark's decode batch: 64 sequences of very different lengths.
        {"name": "decode_batch", "kind": "decode", "batch": 64, "ctx_lo": 512, "ctx_hi": 8192, "nh": 12, "nkvh": 2,
         "out": "bf16"},
        # The benchmark's mixed step of a server: 4 prompt chunks and 60 decodes.
        {"name": "mixed_step", "kind": "mixed", "chunks": 4, "chunk": 512, "prior": 4096, "decodes": 60,
         "ctx_lo": 256, "ctx_hi": 4096, "nh": 12, "nkvh": 2},
        # The benchmark's append and gather of one layer's cache.
        {"name": "kv_append_gather", "kind": "kv", "batch": 32, "ctx_lo": 1, "ctx_hi": 2048, "nkvh": 2},
        # One token against a contiguous cache of 512 + itself, 32-bit.
        {"name": "attention_token_f32", "kind": "attention", "q": 1, "keys": 513, "nh": 12, "nkvh": 2, "d": 128,
         "dtype": "f32"},
        # A prompt through the contiguous op.
        {"name": "attention_prompt", "kind": "attention", "q": 1000, "keys": 1000, "nh": 12, "nkvh": 2, "d": 128,
         "dtype": "bf16"},
        # A generate loop written with the ops: one layer, one token.
        {"name": "layer_token", "kind": "layer", "q": 1, "past": 300, "hs": 1536, "nh": 12, "nkvh": 2, "di": 8960,
         "dtype": "bf16"},
        # The same layer over a prompt.
        {"name": "layer_prompt", "kind": "layer", "q": 777, "past": 0, "hs": 1536, "nh": 12, "nkvh": 2, "di": 8960,
         "dtype": "bf16"},
        # The largest projection of a long prefill step.
        {"name": "linear_prompt", "kind": "linear", "m": 8192, "n": 17920, "k": 1536, "dtype": "bf16", "bias": False},
        # The end of a decode step of 48 sequences.
        {"name": "head_batch", "kind": "head", "rows": 48, "voc": 151936},
        # Continuations of 32 cached prompts, 4 steps.
        {"name": "model_decode", "kind": "model_decode", "batch": 32, "ctx_lo": 600, "ctx_hi": 1800, "steps": 4,
         "layers": 4},
        # Three fresh prompts of different lengths in one step.
        {"name": "model_prompt", "kind": "model_prompt", "prompts": 3, "len_lo": 200, "len_hi": 1100, "layers": 4},
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def draw(rng):
    kind = rng.choice(["decode", "mixed", "kv", "attention", "layer", "linear", "head", "model_decode",
                       "model_prompt"])
    if kind == "decode":
        batch, hi = _log(rng, 1, 128), _log(rng, 32, 16384)
        hi = min(hi, max(32, 560_000 // batch))
        nh, nkvh = rng.choice([(12, 2), (12, 2), (12, 2), (8, 2), (16, 1), (4, 4)])
        return {"kind": kind, "batch": batch, "ctx_lo": rng.randint(1, hi), "ctx_hi": hi, "nh": nh, "nkvh": nkvh,
                "out": rng.choice(["bf16", "bf16", "bf16", "f32"])}
    if kind == "mixed":
        chunk, chunks = _log(rng, 17, 2048), rng.randint(1, 6)
        chunk = min(chunk, 3072 // chunks)
        hi = _log(rng, 64, 4096)
        nh, nkvh = rng.choice([(12, 2), (12, 2), (8, 2)])
        return {"kind": kind, "chunks": chunks, "chunk": chunk, "prior": rng.choice([0, _log(rng, 16, 4096)]),
                "decodes": rng.choice([0, _log(rng, 1, 100)]), "ctx_lo": rng.randint(1, hi), "ctx_hi": hi, "nh": nh,
                "nkvh": nkvh}
    if kind == "kv":
        batch, hi = _log(rng, 1, 128), _log(rng, 32, 8192)
        hi = min(hi, max(32, 80_000 // batch))
        return {"kind": kind, "batch": batch, "ctx_lo": rng.randint(1, hi), "ctx_hi": hi,
                "nkvh": rng.choice([2, 2, 2, 1, 4])}
    if kind == "attention":
        nh, nkvh = rng.choice([(12, 2), (12, 2), (8, 2), (4, 4)])
        what = rng.choice(["token", "prompt", "chunk"])
        if what == "token":
            q, keys = 1, _log(rng, 16, 8192)
        elif what == "prompt":
            q = keys = _log(rng, 16, 1024)
        else:
            q = _log(rng, 2, 512)
            keys = q + _log(rng, 16, 1536)
        return {"kind": kind, "q": q, "keys": keys, "nh": nh, "nkvh": nkvh, "d": rng.choice([128, 128, 128, 64]),
                "dtype": rng.choice(["bf16", "bf16", "f16", "f32"])}
    if kind == "layer":
        hs, nh, nkvh, di = rng.choice([(1536, 12, 2, 8960), (1536, 12, 2, 8960), (1024, 8, 2, 2752)])
        q = rng.choice([1, _log(rng, 2, 800)])
        return {"kind": kind, "q": q, "past": rng.choice([0, _log(rng, 16, 800)]), "hs": hs, "nh": nh, "nkvh": nkvh,
                "di": di, "dtype": rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])}
    if kind == "linear":
        dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
        n, k = rng.choice([(2048, 1536), (1536, 1536), (17920, 1536), (1536, 8960),
                           (_log(rng, 100, 9000), 8 * _log(rng, 16, 512))])
        return {"kind": kind, "m": _log(rng, 1, 8192 if dtype != "f32" else 1024), "n": n, "k": k, "dtype": dtype,
                "bias": rng.random() < 0.5}
    if kind == "head":
        return {"kind": kind, "rows": _log(rng, 1, 128), "voc": rng.choice([151936, 151936, 16 * rng.randint(500, 4000)])}
    if kind == "model_decode":
        hi = _log(rng, 64, 2048)
        return {"kind": kind, "batch": _log(rng, 1, 40), "ctx_lo": rng.randint(max(1, hi // 4), hi), "ctx_hi": hi,
                "steps": rng.randint(2, 4), "layers": rng.randint(2, 4)}
    prompts = rng.randint(1, 4)
    hi = min(_log(rng, 20, 2000), 2000 // prompts)
    return {"kind": kind, "prompts": prompts, "len_lo": rng.randint(max(2, hi // 4), hi), "len_hi": hi,
            "layers": rng.randint(2, 4)}


# ------------------------------------------------- torch and the library

_API = None


def _api():
    global _API
    if _API is None:
        _API = RuntimeAPI(DeviceType.AMD)
    return _API


def _tensor(shape, dtype):
    return Tensor(tuple(shape), dtype=dtype, device=DeviceType.AMD)


def _to(t):
    """A library tensor holding a copy of the torch tensor t."""
    t = t.contiguous()
    lt = _tensor(t.shape, _LL[t.dtype])
    if t.numel():
        torch.cuda.current_stream().synchronize()
        _api().memcpy_sync(lt.data_ptr(), t.data_ptr(), t.numel() * t.element_size(), MemcpyKind.D2D)
    return lt


class _Memory:
    def __init__(self, ptr, shape, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": tuple(shape), "typestr": typestr,
                                         "strides": None, "version": 3}


_TYPESTR = {DataType.F32: ("<f4", torch.float32), DataType.F16: ("<f2", torch.float16),
            DataType.BF16: ("<i2", torch.bfloat16), DataType.I32: ("<i4", torch.int32),
            DataType.I64: ("<i8", torch.int64)}


def _view(lt):
    """The library tensor's own memory as a torch tensor."""
    typestr, dtype = _TYPESTR[lt.dtype()]
    return torch.as_tensor(_Memory(lt.data_ptr(), lt.shape(), typestr, lt), device="cuda:0").view(dtype)


def _gen(seed, salt=0):
    return torch.Generator(device="cuda:0").manual_seed((int(seed) * 1_000_003 + salt) & ((1 << 62) - 1))


def _normal(g, shape, dtype, std=1.0, mean=0.0):
    return torch.empty(tuple(shape), dtype=torch.float32, device="cuda:0").normal_(mean, std, generator=g).to(dtype)


def _spread(lo, hi, n, seed=None):
    """n lengths evenly over [lo, hi], in the seed's order (None: rising)."""
    v = [int(round(lo + (hi - lo) * ((i + 0.5) / n if n > 1 else 1.0))) for i in range(n)]
    if seed is not None:
        v = [v[i] for i in np.random.RandomState(int(seed) % (1 << 31)).permutation(n)]
    return v


# ------------------------------------------------------------ paged inputs

def _rows(g, lens, nkvh):
    """K and V rows of contexts of the given lengths, one after the other: [sum, nkvh, 128] each."""
    shape = (sum(lens), nkvh, HEAD)
    return _normal(g, shape, torch.bfloat16), _normal(g, shape, torch.bfloat16)


def _pool(seed, lens, k, v, nkvh, extra=0):
    """The pools that hold these contexts in randomly placed pages, and the
    block table, with `extra` more tokens mapped."""
    pages = [max(1, (n + extra + PAGE - 1) // PAGE) for n in lens]
    blocks = sum(pages) + 3
    order = np.random.RandomState((int(seed) + 17) % (1 << 31)).permutation(blocks)
    table = np.full((len(lens), max(pages)), -1, np.int32)
    at = 0
    for b, p in enumerate(pages):
        table[b, :p] = order[at:at + p]
        at += p
    zero = torch.zeros((blocks, nkvh, PAGE, HEAD), dtype=torch.bfloat16, device="cuda:0")
    kp, vp = _to(zero), _to(zero)
    tab = _to(torch.from_numpy(table).cuda())
    cu = np.zeros(len(lens) + 1, np.int32)
    cu[1:] = np.cumsum(lens)
    none = _to(torch.zeros(len(lens), dtype=torch.int32, device="cuda:0"))
    Ops.paged_kv_append(kp, vp, _to(k), _to(v), tab, none, _to(torch.from_numpy(cu).cuda()))
    _api().device_synchronize()
    return kp, vp, tab


def _mixed_shape(case, seed):
    """(queries per sequence, contexts) of a mixed batch, in the seed's order."""
    # contexts before the chunks: from none to the longest
    last = max(1, case["chunks"] - 1)
    priors = [case["prior"] * i // last if case["chunks"] > 1 else case["prior"] for i in range(case["chunks"])]
    # ragged chunks: each a little shorter than the one before
    q = [max(1, case["chunk"] - 3 * i) for i in range(case["chunks"])]
    ctx = [p + n for p, n in zip(priors, q)]
    q += [1] * case["decodes"]
    ctx += _spread(case["ctx_lo"], case["ctx_hi"], case["decodes"]) if case["decodes"] else []
    if seed is not None:
        o = np.random.RandomState(int(seed) % (1 << 31)).permutation(len(q))
        q, ctx = [q[i] for i in o], [ctx[i] for i in o]
    return q, ctx


# ------------------------------------------------------------------- layers

def _layer_weights(case, seed):
    t = _TYPES[case["dtype"]][0]
    g = _gen(seed, 5)
    hs, di = case["hs"], case["di"]
    q, kv = case["nh"] * HEAD, case["nkvh"] * HEAD
    w = {"norm1": _normal(g, (hs,), t, 0.1, 1.0), "norm2": _normal(g, (hs,), t, 0.1, 1.0)}
    for name, shape in (("q", (q, hs)), ("k", (kv, hs)), ("v", (kv, hs)), ("o", (hs, q)), ("gate", (di, hs)),
                        ("up", (di, hs)), ("down", (hs, di))):
        w[name] = _normal(g, shape, t, 0.02)
    for name, n in (("qb", q), ("kb", kv), ("vb", kv)):
        w[name] = _normal(g, (n,), t, 0.1)
    return w


def _layer_inputs(case, seed):
    t = _TYPES[case["dtype"]][0]
    g = _gen(seed, 6)
    x = _normal(g, (case["q"], case["hs"]), t)
    kc = _normal(g, (case["past"], case["nkvh"], HEAD), t)
    vc = _normal(g, (case["past"], case["nkvh"], HEAD), t)
    return x, kc, vc


# -------------------------------------------------------------------- model

_MODEL = {"hs": 1536, "nh": 12, "nkvh": 2, "di": 8960, "voc": 151936}


def _model_weights(layers, seed):
    """(name, bf16 tensor) of every weight, one after the other."""
    m = _MODEL
    q, kv = m["nh"] * HEAD, m["nkvh"] * HEAD
    g = _gen(seed, 7)
    bf = torch.bfloat16
    yield "model.embed_tokens.weight", _normal(g, (m["voc"], m["hs"]), bf, 0.02)
    yield "lm_head.weight", _normal(g, (m["voc"], m["hs"]), bf, 0.02)
    yield "model.norm.weight", _normal(g, (m["hs"],), bf, 0.1, 1.0)
    for i in range(layers):
        p = f"model.layers.{i}."
        yield p + "input_layernorm.weight", _normal(g, (m["hs"],), bf, 0.1, 1.0)
        for n, rows in (("q", q), ("k", kv), ("v", kv)):
            yield p + f"self_attn.{n}_proj.weight", _normal(g, (rows, m["hs"]), bf, 0.02)
            yield p + f"self_attn.{n}_proj.bias", _normal(g, (rows,), bf, 0.1)
        yield p + "self_attn.o_proj.weight", _normal(g, (m["hs"], q), bf, 0.02)
        yield p + "post_attention_layernorm.weight", _normal(g, (m["hs"],), bf, 0.1, 1.0)
        yield p + "mlp.gate_proj.weight", _normal(g, (m["di"], m["hs"]), bf, 0.02)
        yield p + "mlp.up_proj.weight", _normal(g, (m["di"], m["hs"]), bf, 0.02)
        yield p + "mlp.down_proj.weight", _normal(g, (m["hs"], m["di"]), bf, 0.02)


def _model(layers, blocks, seed):
    meta = Qwen2Meta(nlayer=layers, hs=_MODEL["hs"], nh=_MODEL["nh"], nkvh=_MODEL["nkvh"], di=_MODEL["di"],
                     voc=_MODEL["voc"], maxseq=8192, epsilon=EPS, theta=THETA)
    model = Qwen2(meta=meta, num_blocks=blocks)
    for name, t in _model_weights(layers, seed):
        h = Tensor(tensor=model.weight_handle(name))
        torch.cuda.current_stream().synchronize()
        _api().memcpy_sync(h.data_ptr(), t.data_ptr(), t.numel() * 2, MemcpyKind.D2D)
        h._tensor = None  # the model owns the handle
    return model


def _model_tokens(case, seed):
    """(prompts, continuation tokens [steps][batch]) of a model case."""
    r = np.random.RandomState((int(seed) + 29) % (1 << 31))
    if case["kind"] == "model_prompt":
        lens = _spread(case["len_lo"], case["len_hi"], case["prompts"], seed)
        return [r.randint(0, _MODEL["voc"], n).astype(np.int64) for n in lens], []
    lens = _spread(case["ctx_lo"], case["ctx_hi"], case["batch"], seed)
    prompts = [r.randint(0, _MODEL["voc"], n).astype(np.int64) for n in lens]
    return prompts, [r.randint(0, _MODEL["voc"], case["batch"]).astype(np.int64) for _ in range(case["steps"])]


# ------------------------------------------------------------------ prepare

def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "decode":
        g = _gen(seed)
        lens = _spread(case["ctx_lo"], case["ctx_hi"], case["batch"], seed)
        k, v = _rows(g, lens, case["nkvh"])
        s["kp"], s["vp"], s["table"] = _pool(seed, lens, k, v, case["nkvh"])
        s["q"] = _to(_normal(g, (case["batch"], case["nh"], HEAD), torch.bfloat16))
        s["ctx"] = _to(torch.tensor(lens, dtype=torch.int32, device="cuda:0"))
        s["out"] = _tensor((case["batch"], case["nh"], HEAD), _TYPES[case["out"]][1])
        s["views"] = _view(s["out"])
    elif kind == "mixed":
        g = _gen(seed)
        q, ctx = _mixed_shape(case, seed)
        k, v = _rows(g, ctx, case["nkvh"])
        s["kp"], s["vp"], s["table"] = _pool(seed, ctx, k, v, case["nkvh"])
        s["q"] = _to(_normal(g, (sum(q), case["nh"], HEAD), torch.bfloat16))
        cu = np.zeros(len(q) + 1, np.int32)
        cu[1:] = np.cumsum(q)
        s["cu"] = _to(torch.from_numpy(cu).cuda())
        s["ctx"] = _to(torch.tensor(ctx, dtype=torch.int32, device="cuda:0"))
        s["out"] = _tensor((sum(q), case["nh"], HEAD), DataType.BF16)
        s["views"] = _view(s["out"])
    elif kind == "kv":
        g = _gen(seed)
        lens = _spread(case["ctx_lo"], case["ctx_hi"], case["batch"], seed)
        k, v = _rows(g, lens, case["nkvh"])
        s["kp"], s["vp"], s["table"] = _pool(seed, lens, k, v, case["nkvh"], extra=1)
        s["kn"] = _to(_normal(g, (case["batch"], case["nkvh"], HEAD), torch.bfloat16))
        s["vn"] = _to(_normal(g, (case["batch"], case["nkvh"], HEAD), torch.bfloat16))
        s["ctx"] = _to(torch.tensor(lens, dtype=torch.int32, device="cuda:0"))
        cu = np.zeros(len(lens) + 1, np.int32)
        cu[1:] = np.cumsum([n + 1 for n in lens])
        s["cu"] = _to(torch.from_numpy(cu).cuda())
        rows = (int(cu[-1]), case["nkvh"], HEAD)
        s["ko"], s["vo"] = _tensor(rows, DataType.BF16), _tensor(rows, DataType.BF16)
        s["views"] = {"k": _view(s["ko"]), "v": _view(s["vo"]), "k_pool": _view(s["kp"]), "v_pool": _view(s["vp"])}
    elif kind == "attention":
        g, t = _gen(seed), _TYPES[case["dtype"]]
        s["q"] = _to(_normal(g, (case["q"], case["nh"], case["d"]), t[0]))
        s["k"] = _to(_normal(g, (case["keys"], case["nkvh"], case["d"]), t[0]))
        s["v"] = _to(_normal(g, (case["keys"], case["nkvh"], case["d"]), t[0]))
        s["out"] = _tensor((case["q"], case["nh"], case["d"]), t[1])
        s["views"] = _view(s["out"])
    elif kind == "layer":
        t = _TYPES[case["dtype"]][1]
        L, P, hs, di = case["q"], case["past"], case["hs"], case["di"]
        q, kv = case["nh"] * HEAD, case["nkvh"] * HEAD
        s["w"] = {n: _to(w) for n, w in _layer_weights(case, seed).items()}
        x, kc, vc = _layer_inputs(case, seed)
        s["x"] = _to(x)
        pad = torch.zeros((L, case["nkvh"], HEAD), dtype=x.dtype, device="cuda:0")
        s["kc"], s["vc"] = _to(torch.cat([kc, pad])), _to(torch.cat([vc, pad]))
        s["pos"] = _to(torch.arange(P, P + L, dtype=torch.int64, device="cuda:0"))
        # the caches' rows of this call, written in place by RoPE and the v projection
        s["k_rows"] = s["kc"].slice(0, P, P + L)
        s["v_rows"] = s["vc"].slice(0, P, P + L).view(L, kv)
        for name, shape in (("h", (L, hs)), ("qp", (L, q)), ("kp", (L, kv)), ("qr", (L, case["nh"], HEAD)),
                            ("a", (L, case["nh"], HEAD)), ("p", (L, hs)), ("y", (L, hs)), ("h2", (L, hs)),
                            ("g", (L, di)), ("u", (L, di)), ("act", (L, di)), ("dn", (L, hs)), ("out", (L, hs))):
            s[name] = _tensor(shape, t)
        s["q3"], s["k3"] = s["qp"].view(L, case["nh"], HEAD), s["kp"].view(L, case["nkvh"], HEAD)
        s["a2"] = s["a"].view(L, q)
        s["views"] = {"out": _view(s["out"]), "k": _view(s["kc"]), "v": _view(s["vc"])}
    elif kind == "linear":
        g, t = _gen(seed), _TYPES[case["dtype"]]
        s["x"] = _to(_normal(g, (case["m"], case["k"]), t[0]))
        s["w"] = _to(_normal(g, (case["n"], case["k"]), t[0], 0.02))
        s["b"] = _to(_normal(g, (case["n"],), t[0], 0.1)) if case["bias"] else None
        s["y"] = _tensor((case["m"], case["n"]), t[1])
        s["views"] = _view(s["y"])
    elif kind == "head":
        g = _gen(seed)
        hs, bf = _MODEL["hs"], DataType.BF16
        s["x"] = _to(_normal(g, (case["rows"], hs), torch.bfloat16))
        s["nw"] = _to(_normal(g, (hs,), torch.bfloat16, 0.1, 1.0))
        w = _to(_normal(g, (case["voc"], hs), torch.bfloat16, 0.02))
        s["w"] = _tensor((case["voc"], hs), bf)
        Ops.linear_pack_weight(s["w"], w)
        _api().device_synchronize()
        s["h"], s["y"] = _tensor((case["rows"], hs), bf), _tensor((case["rows"], case["voc"]), bf)
        s["idx"], s["val"] = _tensor((case["rows"],), DataType.I64), _tensor((case["rows"],), bf)
        # The index is not among the outputs: logits that round to the same
        # value, or nearly, take its place from one correct sum to another.
        # The value that it points at is.
        s["views"] = {"logits": _view(s["y"]), "max": _view(s["val"])}
    elif kind == "model_decode":
        prompts, cont = _model_tokens(case, seed)
        pages = sum((len(p) + case["steps"] + PAGE - 1) // PAGE + 2 for p in prompts)
        s["model"] = m = _model(case["layers"], pages + 16, seed)
        s["ids"] = [m.create_sequence()[0] for _ in prompts]
        at = 0
        while at < len(prompts):  # the cached prompts, in steps of up to 16k tokens
            n, total = 0, 0
            while at + n < len(prompts) and (n == 0 or total + len(prompts[at + n]) <= 16384):
                total += len(prompts[at + n])
                n += 1
            m.step(s["ids"][at:at + n], prompts[at:at + n])
            at += n
        s["cont"] = [[[int(t)] for t in c] for c in cont]
    elif kind == "model_prompt":
        prompts, _ = _model_tokens(case, seed)
        pages = sum((len(p) + PAGE - 1) // PAGE + 2 for p in prompts)
        s["model"] = _model(case["layers"], pages + 16, seed)
        s["prompts"] = prompts
    return s


# ---------------------------------------------------------------------- run

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        Ops.paged_attention(s["out"], s["q"], s["kp"], s["vp"], s["table"], s["ctx"], 1.0 / math.sqrt(HEAD))
    elif kind == "mixed":
        Ops.paged_attention_varlen(s["out"], s["q"], s["kp"], s["vp"], s["table"], s["cu"], s["ctx"],
                                   1.0 / math.sqrt(HEAD))
    elif kind == "kv":
        Ops.paged_kv_append_gather(s["ko"], s["vo"], s["kp"], s["vp"], s["kn"], s["vn"], s["table"], s["ctx"], s["cu"])
    elif kind == "attention":
        Ops.self_attention(s["out"], s["q"], s["k"], s["v"], 1.0 / math.sqrt(case["d"]))
    elif kind == "layer":
        w = s["w"]
        Ops.rms_norm(s["h"], s["x"], w["norm1"], EPS)
        Ops.linear(s["qp"], s["h"], w["q"], w["qb"])
        Ops.linear(s["kp"], s["h"], w["k"], w["kb"])
        Ops.linear(s["v_rows"], s["h"], w["v"], w["vb"])
        Ops.rope(s["qr"], s["q3"], s["pos"], THETA)
        Ops.rope(s["k_rows"], s["k3"], s["pos"], THETA)
        Ops.self_attention(s["a"], s["qr"], s["kc"], s["vc"], 1.0 / math.sqrt(HEAD))
        Ops.linear(s["p"], s["a2"], w["o"], None)
        Ops.add(s["y"], s["x"], s["p"])
        Ops.rms_norm(s["h2"], s["y"], w["norm2"], EPS)
        Ops.linear(s["g"], s["h2"], w["gate"], None)
        Ops.linear(s["u"], s["h2"], w["up"], None)
        Ops.swiglu(s["act"], s["g"], s["u"])
        Ops.linear(s["dn"], s["act"], w["down"], None)
        Ops.add(s["out"], s["y"], s["dn"])
    elif kind == "linear":
        Ops.linear(s["y"], s["x"], s["w"], s["b"])
    elif kind == "head":
        Ops.rms_norm(s["h"], s["x"], s["nw"], EPS)
        Ops.linear_packed(s["y"], s["h"], s["w"])
        Ops.argmax(s["idx"], s["val"], s["y"])
    elif kind == "model_decode":
        m = s["model"]
        ids = [m.fork(i) for i in s["ids"]]
        for tokens in s["cont"]:
            m.step(ids, tokens)
        logits = m.logits()
        for i in ids:
            m.free(i)
        return _view(logits)
    elif kind == "model_prompt":
        m = s["model"]
        ids = [m.create_sequence()[0] for _ in s["prompts"]]
        m.step(ids, s["prompts"])
        logits = m.logits()
        for i in ids:
            m.free(i)
        return _view(logits)
    return s["views"]


# --------------------------------------------------------------------- work

def _attention_work(pairs, nh, d):
    return 4.0 * pairs * nh * d


def _layer_work(T, pairs, kv_read, hs, nh, nkvh, di):
    """(weight elements, flops) of one decoder layer over T new tokens."""
    q, kv = nh * HEAD, nkvh * HEAD
    w = hs * (q + 2 * kv) + q * hs + 3 * hs * di
    return w, 2.0 * T * w + _attention_work(pairs, nh, HEAD)


def work(case):
    kind = case["kind"]
    if kind == "decode":
        lens = _spread(case["ctx_lo"], case["ctx_hi"], case["batch"])
        n, rows = sum(lens), case["batch"] * case["nh"] * HEAD
        return {"bytes": n * case["nkvh"] * HEAD * 4 + rows * (2 + _BYTES[case["out"]]) + n // PAGE * 4,
                "flops": _attention_work(n, case["nh"], HEAD)}
    if kind == "mixed":
        q, ctx = _mixed_shape(case, None)
        pairs = sum(n * c - n * (n - 1) // 2 for n, c in zip(q, ctx))
        return {"bytes": sum(ctx) * case["nkvh"] * HEAD * 4 + sum(q) * case["nh"] * HEAD * 4,
                "flops": _attention_work(pairs, case["nh"], HEAD)}
    if kind == "kv":
        n = sum(_spread(case["ctx_lo"], case["ctx_hi"], case["batch"])) + case["batch"]
        return {"bytes": (n + case["batch"]) * case["nkvh"] * HEAD * 8, "flops": 0}
    if kind == "attention":
        L, S, e = case["q"], case["keys"], _BYTES[case["dtype"]]
        return {"bytes": e * case["d"] * 2 * (L * case["nh"] + S * case["nkvh"]),
                "flops": _attention_work(L * S - L * (L - 1) // 2, case["nh"], case["d"])}
    if kind == "layer":
        L, S, e = case["q"], case["q"] + case["past"], _BYTES[case["dtype"]]
        w, f = _layer_work(L, L * S - L * (L - 1) // 2, S, case["hs"], case["nh"], case["nkvh"], case["di"])
        return {"bytes": e * (w + 2 * L * case["hs"] + 2 * (S + L) * case["nkvh"] * HEAD), "flops": f}
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _BYTES[case["dtype"]] * (m * k + n * k + m * n), "flops": 2.0 * m * n * k}
    m = _MODEL
    if kind == "head":
        return {"bytes": 2 * (case["voc"] * m["hs"] + case["rows"] * (m["hs"] + case["voc"])),
                "flops": 2.0 * case["rows"] * case["voc"] * m["hs"]}
    total = {"bytes": 0.0, "flops": 0.0}
    if kind == "model_decode":
        lens = _spread(case["ctx_lo"], case["ctx_hi"], case["batch"])
        steps = [([1] * len(lens), [n + t + 1 for n in lens]) for t in range(case["steps"])]
    else:
        lens = _spread(case["len_lo"], case["len_hi"], case["prompts"])
        steps = [(lens, lens)]
    for q, ctx in steps:
        pairs = sum(n * c - n * (n - 1) // 2 for n, c in zip(q, ctx))
        w, f = _layer_work(sum(q), pairs, sum(ctx), m["hs"], m["nh"], m["nkvh"], m["di"])
        total["flops"] += case["layers"] * f + 2.0 * len(q) * m["voc"] * m["hs"]
        total["bytes"] += case["layers"] * (2 * w + sum(ctx) * m["nkvh"] * HEAD * 4)
        total["bytes"] += 2 * (m["voc"] * m["hs"] + len(q) * m["voc"] + sum(q) * m["hs"])
    return total


# ---------------------------------------------------------------- tolerance

def tolerance(case):
    kind = case["kind"]
    if kind == "kv":
        return "exact"  # copies
    if kind in ("decode", "mixed"):
        # bf16 results of 32-bit sums; 32-bit results carry the probabilities'
        # two bf16 halves (2^-17)
        return {"rel": 1e-2, "max": 0.1} if case.get("out") != "f32" else {"rel": 1e-4, "max": 1e-3}
    if kind in ("attention", "linear"):
        return {"f32": {"rel": 1e-5, "max": 2e-4}, "f16": {"rel": 2e-3, "max": 2e-2},
                "bf16": {"rel": 1e-2, "max": 0.1}}[case["dtype"]]
    if kind == "layer":  # a dozen roundings to the type, one after the other
        return {"f32": {"rel": 2e-5, "max": 4e-4}, "f16": {"rel": 3e-3, "max": 3e-2},
                "bf16": {"rel": 2e-2, "max": 0.2}}[case["dtype"]]
    if kind == "head":
        return {"rel": 1e-2, "max": 0.1}
    return {"rel": 3e-2, "max": 0.3}  # whole models in bf16


# -------------------------------------------------------------------- exact

def _attend64(q, k, v, scale):
    """q [L, nh, d], k, v [S, nkvh, d] in 64 bits, causal, the last rows aligned."""
    L, nh, d = q.shape
    S, nkvh, _ = k.shape
    out = torch.empty((L, nh, v.shape[2]), dtype=torch.float64, device=q.device)
    see = torch.arange(S, device=q.device)[None, :] <= torch.arange(L, device=q.device)[:, None] + (S - L)
    for h in range(nh):
        kh = h // (nh // nkvh)
        a = (q[:, h] @ k[:, kh].t().contiguous()) * scale
        a = torch.softmax(a.masked_fill(~see, -math.inf), dim=-1)
        out[:, h] = a @ v[:, kh].contiguous()
    return out


def _norm64(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _rope64(x, pos):
    """x [T, nh, d] rotated by pos, the angles as the op's formula gives them in 32 bits."""
    half = x.shape[2] // 2
    e = (2.0 * torch.arange(half, dtype=torch.float32, device=x.device)) / x.shape[2]
    phi = (pos.float()[:, None] / torch.pow(torch.tensor(THETA, dtype=torch.float32, device=x.device), e)).double()
    c, s = torch.cos(phi)[:, None, :], torch.sin(phi)[:, None, :]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _mlp64(x, w):
    h = _norm64(x, w["norm2"])
    g = h @ w["gate"].t()
    return x + (g / (1 + torch.exp(-g)) * (h @ w["up"].t())) @ w["down"].t()


def exact(case, seed):
    kind = case["kind"]
    d64 = torch.float64
    if kind in ("decode", "mixed", "kv"):
        g = _gen(seed)
        if kind == "mixed":
            qn, lens = _mixed_shape(case, seed)
        else:
            lens = _spread(case["ctx_lo"], case["ctx_hi"], case["batch"], seed)
            qn = [1] * len(lens)
        k, v = _rows(g, lens, case["nkvh"])
        at = np.concatenate([[0], np.cumsum(lens)])
        if kind == "kv":
            kn = _normal(g, (case["batch"], case["nkvh"], HEAD), torch.bfloat16)
            vn = _normal(g, (case["batch"], case["nkvh"], HEAD), torch.bfloat16)
            rows = lambda old, new: torch.cat([t for b in range(len(lens)) for t in (old[at[b]:at[b + 1]], new[b:b + 1])])  # noqa: E731
            return {"k": rows(k, kn).to(d64), "v": rows(v, vn).to(d64), "k_pool": None, "v_pool": None}
        q = _normal(g, (sum(qn), case["nh"], HEAD), torch.bfloat16)
        out, r = [], 0
        for b, n in enumerate(qn):
            out.append(_attend64(q[r:r + n].to(d64), k[at[b]:at[b + 1]].to(d64), v[at[b]:at[b + 1]].to(d64),
                                 1.0 / math.sqrt(HEAD)))
            r += n
        return torch.cat(out)
    if kind == "attention":
        g, t = _gen(seed), _TYPES[case["dtype"]][0]
        q = _normal(g, (case["q"], case["nh"], case["d"]), t).to(d64)
        k = _normal(g, (case["keys"], case["nkvh"], case["d"]), t).to(d64)
        v = _normal(g, (case["keys"], case["nkvh"], case["d"]), t).to(d64)
        return _attend64(q, k, v, 1.0 / math.sqrt(case["d"]))
    if kind == "layer":
        w = {n: t.to(d64) for n, t in _layer_weights(case, seed).items()}
        x, kc, vc = (t.to(d64) for t in _layer_inputs(case, seed))
        L, P = case["q"], case["past"]
        pos = torch.arange(P, P + L, device="cuda:0")
        h = _norm64(x, w["norm1"])
        q = _rope64((h @ w["q"].t() + w["qb"]).view(L, case["nh"], HEAD), pos)
        k = torch.cat([kc, _rope64((h @ w["k"].t() + w["kb"]).view(L, case["nkvh"], HEAD), pos)])
        v = torch.cat([vc, (h @ w["v"].t() + w["vb"]).view(L, case["nkvh"], HEAD)])
        y = x + _attend64(q, k, v, 1.0 / math.sqrt(HEAD)).reshape(L, -1) @ w["o"].t()
        return {"out": _mlp64(y, w), "k": k, "v": v}
    if kind == "linear":
        g, t = _gen(seed), _TYPES[case["dtype"]][0]
        x = _normal(g, (case["m"], case["k"]), t).to(d64)
        w = _normal(g, (case["n"], case["k"]), t, 0.02).to(d64)
        y = x @ w.t()
        return y + _normal(g, (case["n"],), t, 0.1).to(d64) if case["bias"] else y
    if kind == "head":
        g, bf = _gen(seed), torch.bfloat16
        x = _normal(g, (case["rows"], _MODEL["hs"]), bf).to(d64)
        nw = _normal(g, (_MODEL["hs"],), bf, 0.1, 1.0).to(d64)
        w = _normal(g, (case["voc"], _MODEL["hs"]), bf, 0.02).to(d64)
        y = _norm64(x, nw) @ w.t()
        return {"logits": y, "max": y.max(-1).values}
    prompts, cont = _model_tokens(case, seed)
    hist = [np.concatenate([p, np.array([c[i] for c in cont], np.int64)]) for i, p in enumerate(prompts)]
    w = dict(_model_weights(case["layers"], seed))
    lens = [len(t) for t in hist]
    ids = torch.from_numpy(np.concatenate(hist)).cuda()
    pos = torch.from_numpy(np.concatenate([np.arange(n) for n in lens])).cuda()
    x = w["model.embed_tokens.weight"][ids].to(d64)
    T = x.shape[0]
    for i in range(case["layers"]):
        p = f"model.layers.{i}."
        a = {n: w[p + f"self_attn.{n}_proj.weight"].to(d64) for n in "qkvo"}
        b = {n: w[p + f"self_attn.{n}_proj.bias"].to(d64) for n in "qkv"}
        h = _norm64(x, w[p + "input_layernorm.weight"].to(d64))
        q = _rope64((h @ a["q"].t() + b["q"]).view(T, _MODEL["nh"], HEAD), pos)
        k = _rope64((h @ a["k"].t() + b["k"]).view(T, _MODEL["nkvh"], HEAD), pos)
        v = (h @ a["v"].t() + b["v"]).view(T, _MODEL["nkvh"], HEAD)
        rows, at = [], 0
        for n in lens:
            rows.append(_attend64(q[at:at + n], k[at:at + n], v[at:at + n], 1.0 / math.sqrt(HEAD)).reshape(n, -1))
            at += n
        x = x + torch.cat(rows) @ a["o"].t()
        x = _mlp64(x, {"norm2": w[p + "post_attention_layernorm.weight"].to(d64),
                       **{n: w[p + f"mlp.{n}_proj.weight"].to(d64) for n in ("gate", "up", "down")}})
    last = torch.from_numpy(np.cumsum(lens) - 1).cuda()
    return _norm64(x[last], w["model.norm.weight"].to(d64)) @ w["lm_head.weight"].to(d64).t()
