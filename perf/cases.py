"""The work a user of this framework has it do, as measurable cases.

Attention by itself, through the C ABI on device rows (what a C engine that keeps its
activations on the device calls), and whole models through the host engine.  Head shapes are
those of the benchmark (16/8/128, 32/8/128, 32/8/64, 8/4/256, 16/8/256); models are the
Qwen3-0.6B-shaped GGUF model and the pre-norm mixer stack of width 2048 of the engine's timing
programs, random weights; experts are those of the width-2048 stacks.

kinds:
  decode    one query row for each of several sessions over their caches: the attention of a
            decode step
  prefill   `rows` new positions behind `ctx` cached ones, appended and attended: a prompt, a
            later turn of a conversation, a portion of a long prompt, a sliding-window layer
  chat      a request from start to end: a session, its prompt, `steps` tokens one by one, the
            session's end
  serve     `steps` batched steps of running sessions
  experts   a mixture-of-experts feed-forward over `rows` rows: choice, both products, sum

Contexts inside [lo, hi] are drawn from the seed.
"""
from __future__ import annotations

import ctypes as C
import json
import math
import os
import tempfile

import numpy as np
import torch

from wayruntime_amd import engine as E
from wayruntime_amd import gguf_writer as gw
from wayruntime_amd import hipattn
from wayruntime_amd import mix_timing
from wayruntime_amd import mix_writer as mw

_u32, _vp = C.c_uint32, C.c_void_p
MODELS = ("qwen3-0.6b", "taredra-w2048")
WIDTH, EXPERTS, TOP, EXPERT_FF = 2048, 64, 6, 1024           # the experts of the width-2048 stacks
SESSION_CTX = 4352                                           # positions a session of the engine has room for


def listed():
    return [
        # one session early in its answer: a layer's attention of a lone decode step, latency alone
        dict(name="decode-one", kind="decode", nq=16, nkv=8, hd=128, sessions=1, lo=600, hi=600),
        # a served batch at mixed ages
        dict(name="decode-ragged16", kind="decode", nq=32, nkv=8, hd=128, sessions=16, lo=256, hi=4096),
        # long documents, wide heads: the stream of the cache and nothing else
        dict(name="decode-long16", kind="decode", nq=8, nkv=4, hd=256, sessions=16, lo=32768, hi=32768),
        # a prompt into an empty cache
        dict(name="prefill-2048", kind="prefill", nq=32, nkv=8, hd=128, ctx=0, rows=2048, window=0),
        # the next turn of a long conversation: few new rows, many cached ones
        dict(name="prefill-turn", kind="prefill", nq=32, nkv=8, hd=128, ctx=8192, rows=177, window=0),
        # a sliding-window layer with wide heads over an odd-sized prompt
        dict(name="prefill-window", kind="prefill", nq=8, nkv=4, hd=256, ctx=0, rows=1501, window=512),
        # a short question and a short answer
        dict(name="chat-short", kind="chat", model="qwen3-0.6b", prompt=45, steps=24),
        # a long prompt, one token out: time to first token
        dict(name="chat-prompt", kind="chat", model="qwen3-0.6b", prompt=2047, steps=1),
        # a full batch of running sessions
        dict(name="serve-16", kind="serve", model="qwen3-0.6b", sessions=16, lo=100, hi=1500, steps=8),
        # the same two for the recurrent family
        dict(name="stack-prompt", kind="chat", model="taredra-w2048", prompt=2047, steps=1),
        dict(name="stack-serve", kind="serve", model="taredra-w2048", sessions=16, lo=100, hi=1500, steps=8),
        # the experts of a prompt portion
        dict(name="experts-512", kind="experts", rows=512),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "chat", "serve", "experts"])
    if kind == "decode":
        nq, nkv, hd = rng.choice([(16, 8, 128), (32, 8, 128), (8, 4, 256), (32, 8, 64)])
        lo = _log(rng, 32, 16384)
        return dict(kind=kind, nq=nq, nkv=nkv, hd=hd, sessions=rng.randint(1, 16), lo=lo, hi=min(32768, _log(rng, lo, 4 * lo)))
    if kind == "prefill":
        nq, nkv, hd = rng.choice([(16, 8, 128), (32, 8, 128), (8, 4, 256), (16, 8, 256), (32, 8, 64)])
        ctx = rng.choice([0, _log(rng, 32, 16384)])
        return dict(kind=kind, nq=nq, nkv=nkv, hd=hd, ctx=ctx, rows=_log(rng, 3, 4096), window=rng.choice([0, 0, _log(rng, 128, 4096)]))
    if kind == "experts":
        return dict(kind=kind, rows=_log(rng, 1, 4096))
    model = rng.choice(MODELS)
    if kind == "chat":
        prompt = _log(rng, 4, 2047)
        return dict(kind=kind, model=model, prompt=prompt, steps=1 if prompt > 1024 else rng.randint(1, 16))
    lo = _log(rng, 16, 512)
    return dict(kind=kind, model=model, sessions=rng.randint(1, 16), lo=lo, hi=2 * lo, steps=rng.randint(4, 8))


# ------------------------------------------------------------------ what a program keeps

_kept = {}


def _engine():
    """One engine per process; it brings the device library up."""
    if "engine" not in _kept:
        _kept["engine"] = E.Engine()
        _bind_mix(hipattn.lib())
    return _kept["engine"]


def _lib():
    _engine()
    return hipattn.lib()


def _ok(rc):
    if rc != 0:
        raise RuntimeError("status %d" % rc)


def _model_path(name):
    """The model's file or folder, written once per machine (random weights of a fixed seed)."""
    gguf = name == "qwen3-0.6b"
    path = os.path.join(tempfile.gettempdir(), "wayruntime_amd_cases_" + name + (".gguf" if gguf else ""))
    if not os.path.exists(path):
        part = "%s.part%d" % (path, os.getpid())
        if gguf:
            gw.write_model(part, gw.QWEN3_0_6B)
        else:
            mw.write_model(part, _stack_config(), rank=mix_timing.RANK)
        try:
            os.rename(part, path)
        except OSError:                                      # another process was first
            if not os.path.exists(path):
                raise
    return path


def _stack_config():
    return mix_timing.SIZES["w2048"][mix_timing.KINDS.index("taredra")]


def _model(name):
    if name not in _kept:
        m = _engine().load(_model_path(name), max_context=SESSION_CTX)
        if name != "qwen3-0.6b":
            m.set_cache_pool(64 * SESSION_CTX, 64)
        _kept[name] = m
    return _kept[name]


class _Raw:
    """Device memory of the library, given back with its last user."""

    def __init__(self, shape, dtype):
        n = math.prod(shape) * dtype.itemsize
        self.p = _lib().wr_hip_attn_dev_alloc(max(n, 16))
        if not self.p:
            raise MemoryError("out of memory: %d bytes on the device" % n)
        kind = {torch.float32: "<f4", torch.int32: "<i4", torch.int16: "<i2"}[dtype]
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": kind, "data": (self.p, False), "version": 2}

    def __del__(self):
        if getattr(self, "p", None):
            hipattn.lib().wr_hip_attn_dev_free(self.p)


class _Memory:
    """Such memory, its address and a torch tensor over it."""

    def __init__(self, shape, dtype=torch.float32):
        raw = _Raw(shape, dtype)
        self.p, self.t = raw.p, torch.as_tensor(raw, device="cuda")   # the tensor holds on to the memory

    @classmethod
    def of(cls, x):
        m = cls(x.shape, x.dtype)
        m.t.copy_(x)
        return m


class _Cache:
    """One session's cache of one layer."""

    def __init__(self, hd, nkv, max_ctx):
        h = _vp()
        _ok(_lib().wr_hip_attn_kv_create(1, (_u32 * 1)(hd), nkv, max_ctx, C.byref(h)))
        self.h = h

    def __del__(self):
        if getattr(self, "h", None):
            hipattn.lib().wr_hip_attn_kv_destroy(self.h)


class _Sessions:
    """Running sessions; `fill` brings them to their contexts."""

    def __init__(self, model, prompts):
        self.model, self.prompts, self.open = model, prompts, []
        self.fill()

    def fill(self):
        self.close()
        for p in self.prompts:
            s = self.model.session()
            self.open.append(s)
            if s.prefill(p) != len(p):
                raise RuntimeError("prompt refused: %d" % s.status)

    def close(self):
        for s in self.open:
            s.close()
        self.open = []

    def __del__(self):
        self.close()


class _Lent(np.ndarray):
    """A view of memory that its owner gives back."""

    owner = None


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _contexts(case, seed):
    r = np.random.default_rng([seed, 7])
    return [int(c) for c in r.integers(case["lo"], case["hi"] + 1, case["sessions"])]


def _tokens(seed, i, n, vocab):
    return np.random.default_rng([seed, 11, i]).integers(0, vocab, n).astype(np.uint32)


def _vocab(name):
    return gw.QWEN3_0_6B.vocab if name == "qwen3-0.6b" else mix_timing.VOCAB


def _token_array(ids):
    return (_u32 * len(ids))(*[int(t) for t in ids])


# ------------------------------------------------------------------ attention

def _decode_rows(case, seed):
    """Per session (K, V) [ctx, nkv, hd], then the query rows."""
    g = _gen(seed)
    for c in _contexts(case, seed):
        yield _normal(g, c, case["nkv"], case["hd"]), _normal(g, c, case["nkv"], case["hd"])
    yield _normal(g, case["sessions"], case["nq"], case["hd"])


def _fill_cache(cache, k, v):
    for at in range(0, len(k), 8192):                        # a long context comes in portions
        a, b = _Memory.of(k[at:at + 8192].contiguous()), _Memory.of(v[at:at + 8192].contiguous())
        torch.cuda.synchronize()
        _ok(_lib().wr_hip_attn_append_dev(cache.h, 0, at, len(a.t), a.p, b.p))
        _ok(_lib().wr_hip_attn_sync())


def _prepare_decode(case, seed):
    ctx = _contexts(case, seed)
    s = dict(kind="decode", n=len(ctx), nq=case["nq"], caches=[])
    for c, rows in zip(ctx + [0], _decode_rows(case, seed)):
        if isinstance(rows, tuple):
            s["caches"].append(_Cache(case["hd"], case["nkv"], c))
            _fill_cache(s["caches"][-1], *rows)
        else:
            s["q"] = _Memory.of(rows)
    s["out"] = _Memory((len(ctx), case["nq"], case["hd"]))
    s["kv"] = (_vp * len(ctx))(*[c.h for c in s["caches"]])
    s["seq_k"] = (_u32 * len(ctx))(*ctx)
    return s


def _run_decode(s):
    _ok(hipattn.lib().wr_hip_attn_decode_batched_dev(s["n"], s["kv"], 0, s["seq_k"], s["q"].p, s["out"].p, s["nq"], 0.0, 0))
    return s["out"].t


def _prefill_rows(case, seed):
    g, n = _gen(seed), case["ctx"] + case["rows"]
    return (_normal(g, n, case["nkv"], case["hd"]), _normal(g, n, case["nkv"], case["hd"]),
            _normal(g, case["rows"], case["nq"], case["hd"]))


def _prepare_prefill(case, seed):
    k, v, q = _prefill_rows(case, seed)
    ctx = case["ctx"]
    cache = _Cache(case["hd"], case["nkv"], len(k))
    if ctx:
        _fill_cache(cache, k[:ctx], v[:ctx])
    return dict(kind="prefill", case=case, cache=cache, q=_Memory.of(q), k=_Memory.of(k[ctx:].contiguous()),
                v=_Memory.of(v[ctx:].contiguous()), out=_Memory((case["rows"], case["nq"], case["hd"])))


def _run_prefill(s):
    c, lib = s["case"], hipattn.lib()
    _ok(lib.wr_hip_attn_append_dev(s["cache"].h, 0, c["ctx"], c["rows"], s["k"].p, s["v"].p))
    _ok(lib.wr_hip_attn_prefill_dev(s["cache"].h, 0, c["ctx"], c["rows"], s["q"].p, s["out"].p, c["nq"], 0.0, c["window"]))
    return s["out"].t


def _stored(x):
    """What the cache keeps of 32-bit values: binary16 with the low bits dropped, tiny values as zeros."""
    x = x.float().contiguous()
    y = (x.view(torch.int32) & ~0x1FFF).view(torch.float32)
    return torch.where(y.abs() < 2.0 ** -14, torch.zeros_like(y), y).double()


def _attend(q, k, v, first, window):
    """[T, nq, hd] rows at positions first .. over k, v [n, nkv, hd], causal, in float64."""
    T, nq, hd = q.shape
    group = nq // k.shape[1]
    out = torch.empty(T, nq, hd, dtype=torch.float64, device=q.device)
    pos, keys = torch.arange(T, device=q.device)[:, None] + first, torch.arange(len(k), device=q.device)[None]
    seen = (keys <= pos) & (keys > pos - window) if window else keys <= pos
    for h in range(nq):
        w = (q[:, h].double() @ k[:, h // group].t().contiguous()) * hd ** -0.5
        out[:, h] = torch.softmax(w.masked_fill_(~seen, -math.inf), dim=1) @ v[:, h // group].contiguous()
    return out


def _exact_decode(case, seed):
    rows = list(_decode_rows(case, seed))
    return torch.cat([_attend(rows[-1][i:i + 1], _stored(k), _stored(v), len(k) - 1, 0) for i, (k, v) in enumerate(rows[:-1])])


def _exact_prefill(case, seed):
    k, v, q = _prefill_rows(case, seed)
    return _attend(q, _stored(k), _stored(v), case["ctx"], case["window"])


# ------------------------------------------------------------------ whole models

def _prepare_chat(case, seed):
    m, vocab = _model(case["model"]), _vocab(case["model"])
    ids = _tokens(seed, 0, case["prompt"] + case["steps"], vocab)
    return dict(kind="chat", model=m, prompt=_token_array(ids[:case["prompt"]]), steps=[int(t) for t in ids[case["prompt"]:]],
                logits=np.empty(vocab, dtype=np.float32))


def _run_chat(s):
    m = s["model"]
    session = m.session()
    rc = m.lib.wr_prefill(session.h, s["prompt"], len(s["prompt"]))
    if rc != len(s["prompt"]):
        raise RuntimeError("prompt refused: %d" % rc)
    for t in s["steps"]:
        p = m.lib.wr_step(session.h, t)
        if not p:
            raise RuntimeError("step refused: %d" % session.status)
    s["logits"][:] = np.ctypeslib.as_array(p, shape=s["logits"].shape)
    session.close()
    return s["logits"]


def _serve_tokens(case, seed):
    """Per session its prompt, then what it is fed: tokens the sampler has picked."""
    vocab = _vocab(case["model"])
    ids = [_tokens(seed, i, c + case["steps"], vocab) for i, c in enumerate(_contexts(case, seed))]
    return [t[:-case["steps"]] for t in ids], [t[-case["steps"]:] for t in ids]


def _prepare_serve(case, seed):
    prompts, feed = _serve_tokens(case, seed)
    n, vocab = case["sessions"], _vocab(case["model"])
    return dict(kind="serve", vocab=vocab, n=n, sessions=_Sessions(_model(case["model"]), prompts),
                feed=[_token_array([f[k] for f in feed]) for k in range(case["steps"])], out=(C.POINTER(C.c_float) * n)())


def _run_serve(s):
    ss, n = s["sessions"], s["n"]
    if max(x.pos for x in ss.open) + len(s["feed"]) > SESSION_CTX:   # full: new requests take their places
        ss.fill()
    h = (_vp * n)(*[x.h for x in ss.open])
    for t in s["feed"]:
        rc = ss.model.lib.wr_batch_step(h, t, n, s["out"])
        if rc != n:
            raise RuntimeError("step refused: %d" % rc)
    rows = [np.ctypeslib.as_array(s["out"][i], shape=(s["vocab"],)).view(_Lent) for i in range(n)]
    for r in rows:
        r.owner = ss
    return rows


def _norm(x, w, eps=1e-6):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _turn_halves(x, pos, base, dims, series=False):
    """[T, heads, hd]: dimension i turns with i + dims / 2.  GGUF models define their sine and cosine as short power series
    of the angle inside [-pi, pi] (four terms each)."""
    half = dims // 2
    a = pos.double()[:, None, None] * base ** (-2.0 * torch.arange(half, device=x.device, dtype=torch.float64) / dims)
    if series:
        a = a - 2 * math.pi * torch.round(a / (2 * math.pi))
        b = a * a
        c, s = 1 - b / 2 + b ** 2 / 24 - b ** 3 / 720, a * (1 - b / 6 + b ** 2 / 120 - b ** 3 / 5040)
    else:
        c, s = a.cos(), a.sin()
    u, v = x[..., :half], x[..., half:dims]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., dims:]], -1)


def _mm(x, w):
    """x . w^T for a matrix kept as rows of outputs."""
    return x @ w.double().t().contiguous()


def _qwen_weights():
    """Device tensors of the file, its data in the order in which its tensors are listed."""
    plan = gw.tensor_plan(gw.QWEN3_0_6B)
    sizes = [math.prod(d) * (4 if t == gw.GGML_F32 else 2) for _, d, t in plan]
    places = [-(-n // gw.ALIGN) * gw.ALIGN for n in sizes]
    raw = np.memmap(_model_path("qwen3-0.6b"), dtype=np.uint8, mode="r")
    at, out = len(raw) - sum(places), {}
    for (name, dims, typ), n, place in zip(plan, sizes, places):
        x = np.array(raw[at:at + n]).view(np.float32 if typ == gw.GGML_F32 else np.float16)
        out[name] = torch.from_numpy(x.reshape(dims[::-1])).cuda()
        at += place
    return out


def _qwen_exact(requests):
    """Logits of each request's last token, float64; the cache keeps what it keeps."""
    m, w = gw.QWEN3_0_6B, _qwen_weights()
    ids = torch.from_numpy(np.concatenate(requests).astype(np.int64)).cuda()
    ends = np.cumsum([len(r) for r in requests])
    parts = [slice(e - len(r), e) for e, r in zip(ends, requests)]
    pos = torch.cat([torch.arange(len(r), device="cuda") for r in requests])
    x = w["token_embd.weight"][ids].double()
    for i in range(m.n_layers):
        p = "blk.%d." % i
        h = _norm(x, w[p + "attn_norm.weight"].double(), m.rms_eps)
        q, k, v = (_mm(h, w[p + "attn_%s.weight" % n]).reshape(len(ids), -1, m.head_dim) for n in "qkv")
        q = _turn_halves(_norm(q, w[p + "attn_q_norm.weight"].double(), m.rms_eps), pos, m.rope_base, m.head_dim, True)
        k = _stored(_turn_halves(_norm(k, w[p + "attn_k_norm.weight"].double(), m.rms_eps), pos, m.rope_base, m.head_dim, True))
        v = _stored(v)
        o = torch.cat([_attend(q[s], k[s], v[s], 0, 0) for s in parts]).reshape(len(ids), -1)
        x = x + _mm(o, w[p + "attn_output.weight"])
        h = _norm(x, w[p + "ffn_norm.weight"].double(), m.rms_eps)
        u = torch.nn.functional.silu(_mm(h, w[p + "ffn_gate.weight"])) * _mm(h, w[p + "ffn_up.weight"])
        x = x + _mm(u, w[p + "ffn_down.weight"])
    last = _norm(x[torch.from_numpy(ends - 1).cuda()], w["output_norm.weight"].double(), m.rms_eps)
    return _mm(last, w["token_embd.weight"])


def _stack_weights():
    folder = _model_path("taredra-w2048")
    raw = np.memmap(os.path.join(folder, "model.safetensors"), dtype=np.uint8, mode="r")
    n = int(np.array(raw[:8]).view(np.uint64)[0])
    out = {}
    for name, d in json.loads(raw[8:8 + n].tobytes()).items():
        a, b = (8 + n + o for o in d["data_offsets"])
        out[name] = torch.from_numpy(np.array(raw[a:b]).view(np.int16)).cuda().view(torch.bfloat16).reshape(d["shape"])
    return out


def _unit(x, eps=1e-6):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _state_walk(r, k, v, decay, bonus=None, rate=None):
    """Outputs [T, H, D] of a matrix state per head: a bonus for the token itself, or a removal along the unit key."""
    T, H, D = r.shape
    S, o = torch.zeros(H, D, D, dtype=torch.float64, device=r.device), torch.empty_like(r)
    if rate is not None:
        u = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + 1e-6)
        away = rate * u
    for t in range(T):
        kv = k[t][:, :, None] * v[t][:, None, :]
        if rate is None:
            o[t] = (r[t][:, None] @ (S + bonus[:, :, None] * kv))[:, 0]
            S = torch.addcmul(kv, decay[t][:, :, None], S)
        else:
            S = torch.addcmul(kv - away[t][:, :, None] * (u[t][:, None] @ S), decay[t][:, :, None], S)
            o[t] = (r[t][:, None] @ S)[:, 0]
    return o


def _stack_exact_one(cfg, w, ids):
    """Logits of the last token of one request through the pre-norm stack."""
    f64, W, T = torch.float64, cfg["width"], len(ids)
    one = lambda n: 1.0 + w[n].double()  # noqa: E731
    pos = torch.arange(T, device="cuda")
    x = w["embed"][torch.from_numpy(ids.astype(np.int64)).cuda()].double() * cfg["embedding"]["scale"]
    for i, layer in enumerate(cfg["layers"]):
        p, m = "l%d." % i, layer["mixer"]
        h = _norm(x, one(p + "norm1"))
        if layer["type"] == "wkv":
            q, H, D = p + "mix.", m["heads"], m["dim"]
            before = torch.cat([torch.zeros(1, W, dtype=f64, device="cuda"), h[:-1]])
            mix = {n: h + (before - h) * w[q + "mu." + n].double() for n in "rkvgw"}
            r, k, v = (_mm(mix[n], w[q + n]).reshape(T, H, D) for n in "rkv")
            z = _mm(torch.tanh(_mm(mix["w"], w[q + "w1"])), w[q + "w2"]) + w[q + "w0"].double()
            o = _state_walk(r, k, v, torch.exp(-torch.exp(z)).reshape(T, H, D), bonus=w[q + "u"].double())
            o = _unit(o).reshape(T, -1) * w[q + "norm"].double() * torch.nn.functional.silu(_mm(mix["g"], w[q + "g"]))
            x = x + _mm(o, w[q + "o"])
        else:
            a, q = m["left"], p + "mix.left."
            qh, kh = (_turn_halves(_mm(h, w[q + n]).reshape(T, -1, a["dim"]), pos, a["rot"]["base"], a["rot"]["dims"]) for n in "qk")
            v = _unit(_mm(h, w[q + "v"]).reshape(T, -1, a["vdim"]))
            gap = pos[:, None] - pos[None]
            seen, o = (gap >= 0) & (gap < a["mask"]["size"]), torch.empty(T, a["heads"], a["vdim"], dtype=f64, device="cuda")
            for n in range(a["heads"]):
                j = n // (a["heads"] // a["kv_heads"])
                s = ((qh[:, n] @ kh[:, j].t().contiguous()) * a["scale"]).masked_fill_(~seen, -math.inf)
                s = torch.cat([s, w[q + "sink"][n].double().expand(T, 1)], 1)
                o[:, n] = torch.softmax(s, 1)[:, :-1] @ v[:, j].contiguous()
            left = _mm(o.reshape(T, -1), w[q + "o"])
            b, q = m["right"], p + "mix.right."
            H, D = b["heads"], b["dim"]
            r, k, v = (_mm(h, w[q + n]).reshape(T, H, D) for n in "rkv")
            z = _mm(torch.tanh(_mm(h, w[q + "w1"])), w[q + "w2"]) + w[q + "w0"].double()
            rate = torch.sigmoid(_mm(h, w[q + "a"]) + w[q + "a.b"].double()).reshape(T, H, D)
            o = _state_walk(r, k, v, torch.exp(-math.exp(-0.5) * torch.sigmoid(z)).reshape(T, H, D), rate=rate)
            o = _unit(o).reshape(T, -1) * w[q + "norm"].double() * torch.sigmoid(_mm(h, w[q + "g"]))
            x = x + m["left_scale"] * left + m["right_scale"] * _mm(o, w[q + "o"])
        h = _norm(x, one(p + "norm2"))
        g = torch.nn.functional.gelu(_mm(h, w[p + "mlp.gate"]), approximate="tanh")
        x = x + _mm(g * _mm(h, w[p + "mlp.up"]), w[p + "mlp.down"])
    return _mm(_norm(x[-1:], one("final.norm")), w["embed"])


def _exact_logits(case, requests):
    if case["model"] == "qwen3-0.6b":
        return _qwen_exact(requests)
    if sum(len(r) for r in requests) > 20000:                # the recurrences walk token by token
        return None
    cfg, w = _stack_config(), _stack_weights()
    return torch.cat([_stack_exact_one(cfg, w, r) for r in requests])


def _exact_chat(case, seed):
    rows = _exact_logits(case, [_tokens(seed, 0, case["prompt"] + case["steps"], _vocab(case["model"]))])
    return None if rows is None else rows[0]


def _exact_serve(case, seed):
    rows = _exact_logits(case, [np.concatenate(p) for p in zip(*_serve_tokens(case, seed))])
    return None if rows is None else list(rows)


# ------------------------------------------------------------------ experts

class _Gemm(C.Structure):
    _fields_ = [("w", _vp), ("x", _vp), ("x_kt", _u32), ("x_kt_z", _u32), ("rows", _u32), ("group_expert", _vp),
                ("tile_groups", _u32), ("out", _u32), ("y_f32", _vp), ("y_act", _vp), ("ldy", _u32), ("h", _vp), ("h_kt", _u32),
                ("col_z", _u32), ("n_split", _u32), ("silu_end", _u32), ("sigmoid_end", _u32), ("relu2", _u32),
                ("scale", C.c_float), ("tanh_end", _u32), ("gelu", _u32), ("x_kt0", _u32), ("bias", _vp), ("limit", C.c_float),
                ("slope", C.c_float), ("up_bias", C.c_float), ("x_perm", _vp), ("h_kt0", _u32), ("x_scale", _vp)]


class _Router(C.Structure):
    _fields_ = [("experts", _u32), ("identity", _u32), ("top", _u32), ("groups", _u32), ("keep", _u32), ("softmax_all", _u32),
                ("shared_gate", _u32), ("scale", C.c_float), ("correction", _vp), ("logistic", _u32)]


class _Resid(C.Structure):
    _fields_ = [("width", _u32), ("eps", C.c_float), ("x", _vp), ("y", _vp), ("post", _vp), ("add", _vp), ("next", _vp),
                ("gate", _vp), ("slot", _vp), ("top", _u32), ("wanted", _u32), ("h", _vp), ("side", _vp), ("ident", _vp),
                ("shared", _vp), ("pair_y", _vp * 2), ("pair_post", _vp * 2)]


class _Seq(C.Structure):
    _fields_ = [("rows", _u32), ("pos0", _u32), ("slot", _u32), ("buf_in", _u32), ("buf_out", _u32), ("n_pages", _u32),
                ("pages", C.POINTER(_u32))]


OUT_ROWS_F32, OUT_FRAG = 0, 2


def _bind_mix(lib):
    lib.wr_hip_mix_mat_create.argtypes = [_u32, _u32, _u32, _vp, C.POINTER(_vp)]
    lib.wr_hip_mix_pool_create.argtypes = [C.c_int, _u32, C.POINTER(_u32), _u32, _u32, _vp, _u32, C.POINTER(_vp)]
    lib.wr_hip_mix_step_create.argtypes = [_u32, C.POINTER(_vp)]
    lib.wr_hip_mix_step_set.argtypes = [_vp, _vp, _u32, C.POINTER(_Seq), C.POINTER(_u32), _u32, _u32, _vp]
    lib.wr_hip_mix_route.argtypes = [_vp, _vp, _u32, C.POINTER(_Router), _u32, _vp, _vp, _vp, _vp, _vp, _vp]
    lib.wr_hip_mix_route_gather.argtypes = [_vp, C.c_int, _vp, _u32, _u32, _vp, _vp, _vp]
    lib.wr_hip_mix_route_groups.argtypes = [_u32, _u32, _u32, _u32]
    lib.wr_hip_mix_route_groups.restype = _u32
    lib.wr_hip_mix_gemm_run.argtypes = [C.c_int, C.POINTER(_Gemm)]
    lib.wr_hip_mix_residual.argtypes = [_vp, C.c_int, C.POINTER(_Resid)]
    for n in ("mat", "pool", "step"):
        f = getattr(lib, "wr_hip_mix_%s_destroy" % n)
        f.argtypes, f.restype = [_vp], None


def _expert_weights():
    """(up [experts, ff, width], down [experts, width, ff]) bfloat16, of a fixed seed."""
    g = _gen(1)
    up = _normal(g, EXPERTS, EXPERT_FF, WIDTH) * WIDTH ** -0.5
    return up.bfloat16(), (_normal(g, EXPERTS, WIDTH, EXPERT_FF) * EXPERT_FF ** -0.5).bfloat16()


def _expert_mats():
    if "experts" not in _kept:
        mats = []
        for x in _expert_weights():
            bits, h = x.view(torch.int16).cpu().numpy(), _vp()
            _ok(_lib().wr_hip_mix_mat_create(x.shape[0], x.shape[1], x.shape[2], bits.ctypes.data, C.byref(h)))
            mats.append(h)
        _kept["experts"] = mats
    return _kept["experts"]


def _expert_inputs(case, seed):
    """Residual rows, normed rows and router logits, as the launches ahead of a feed-forward leave them."""
    g, R = _gen(seed), case["rows"]
    return _normal(g, R, WIDTH), _normal(g, R, WIDTH).bfloat16(), _normal(g, R, EXPERTS)


class _StepRows:
    """A step of one request of `rows` rows, and the pool it is checked against."""

    def __init__(self, rows):
        lib, pages = _lib(), -(-rows // 64)
        self.pool, self.h = _vp(), _vp()
        _ok(lib.wr_hip_mix_pool_create(0, 1, (_u32 * 1)(32), pages, 0, None, 1, C.byref(self.pool)))
        _ok(lib.wr_hip_mix_step_create(pages, C.byref(self.h)))
        self.pages = (_u32 * pages)(*range(pages))
        _ok(lib.wr_hip_mix_step_set(self.h, self.pool, 1, C.byref(_Seq(rows, 0, 0, 0, 1, pages, self.pages)), (_u32 * rows)(), 1, 0, None))

    def __del__(self):
        hipattn.lib().wr_hip_mix_step_destroy(self.h)
        hipattn.lib().wr_hip_mix_pool_destroy(self.pool)


def _prepare_experts(case, seed):
    up, down = _expert_mats()
    x, h, z = _expert_inputs(case, seed)
    R, lib = case["rows"], _lib()
    tile = 8 if R * TOP >= EXPERTS * 32 else 1               # experts whose rows fill whole tiles take runs of eight groups
    groups = lib.wr_hip_mix_route_groups(R, EXPERTS, TOP, tile)
    slots, r16 = groups * 16, -(-R // 16) * 16
    f = torch.zeros(r16, WIDTH, dtype=torch.bfloat16, device="cuda")
    f[:R] = h
    f = f.reshape(r16 // 16, 16, WIDTH // 32, 4, 8).permute(0, 2, 3, 1, 4).contiguous()      # operand order
    s = dict(kind="experts", R=R, tile=tile, groups=groups, step=_StepRows(R), x=_Memory.of(x), h=_Memory.of(f.view(torch.int16)),
             z=_Memory.of(z), gate=_Memory((R, TOP)), slot=_Memory((R, TOP), torch.int32), perm=_Memory((slots,), torch.int32),
             expert=_Memory((groups,), torch.int32), xs=_Memory((slots, WIDTH), torch.int16), act=_Memory((slots, EXPERT_FF), torch.int16),
             ys=_Memory((slots, WIDTH)), y=_Memory((R, WIDTH)))
    s["router"] = _Router(experts=EXPERTS, top=TOP)
    few = tile == 1                                          # few rows: the product fetches them where they are
    s["up"] = _Gemm(w=up, x=s["h"].p if few else s["xs"].p, x_perm=s["perm"].p if few else None, x_kt=WIDTH // 32, rows=slots,
                    group_expert=s["expert"].p, tile_groups=tile, out=OUT_FRAG, h=s["act"].p, h_kt=EXPERT_FF // 32, relu2=1)
    s["down"] = _Gemm(w=down, x=s["act"].p, x_kt=EXPERT_FF // 32, rows=slots, group_expert=s["expert"].p, tile_groups=tile,
                      out=OUT_ROWS_F32, y_f32=s["ys"].p, ldy=WIDTH)
    s["resid"] = _Resid(width=WIDTH, eps=1e-6, x=s["x"].p, y=s["ys"].p, gate=s["gate"].p, slot=s["slot"].p, top=TOP)
    return s


def _run_experts(s):
    """Returns the residual's change on top of what earlier passes left: x grows by the same rows each time."""
    lib, step = hipattn.lib(), s["step"].h
    _ok(lib.wr_hip_mix_route(step, s["z"].p, EXPERTS, C.byref(s["router"]), s["tile"], s["gate"].p, None, None, s["slot"].p, s["perm"].p,
                             s["expert"].p))
    if s["tile"] > 1:
        _ok(lib.wr_hip_mix_route_gather(step, 0, s["h"].p, WIDTH // 32, s["groups"], s["perm"].p, s["expert"].p, s["xs"].p))
    _ok(lib.wr_hip_mix_gemm_run(0, C.byref(s["up"])))
    _ok(lib.wr_hip_mix_gemm_run(0, C.byref(s["down"])))
    _ok(lib.wr_hip_mix_residual(step, 0, C.byref(s["resid"])))
    return dict(x=s["x"].t, gate=s["gate"].t)


def _exact_experts(case, seed):
    x, h, z = _expert_inputs(case, seed)
    up, down = _expert_weights()
    best, chosen = torch.topk(z.double(), TOP, dim=1)
    gate, y = torch.softmax(best, 1), x.double()
    for e in range(EXPERTS):
        r, t = (chosen == e).nonzero(as_tuple=True)
        if len(r):
            a = _mm(h[r].double(), up[e]).clamp_min(0) ** 2
            y.index_add_(0, r, gate[r, t][:, None] * _mm(a, down[e]))
    return dict(x=y, gate=gate)


# ------------------------------------------------------------------ the cases as they are asked for

_PREPARE = dict(decode=_prepare_decode, prefill=_prepare_prefill, chat=_prepare_chat, serve=_prepare_serve, experts=_prepare_experts)
_RUN = dict(decode=_run_decode, prefill=_run_prefill, chat=_run_chat, serve=_run_serve, experts=_run_experts)
_EXACT = dict(decode=_exact_decode, prefill=_exact_prefill, chat=_exact_chat, serve=_exact_serve, experts=_exact_experts)


def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, seed)
    torch.cuda.synchronize()
    return state


def run(state):
    return _RUN[state["kind"]](state)


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


def _pairs(rows, first, window):
    """Keys seen by rows first .. first + rows - 1, summed."""
    return sum(min(first + i + 1, window or first + i + 1) for i in range(rows))


def _qwen_work(requests, logit_rows):
    """requests: (rows, position of the first) of one pass over the weights."""
    m = gw.QWEN3_0_6B
    layer = m.hidden * (m.n_q + 2 * m.n_kv) * m.head_dim + m.n_q * m.head_dim * m.hidden + 3 * m.hidden * m.ffn
    rows, head = sum(r for r, _ in requests), m.hidden * m.vocab
    seen = sum(_pairs(r, p, 0) for r, p in requests)
    kv = sum(r + p + r for r, p in requests) * 4 * m.n_kv * m.head_dim
    return dict(bytes=2 * (m.n_layers * layer + (head if logit_rows else 0)) + m.n_layers * kv + 4 * logit_rows * m.vocab,
                flops=2 * rows * m.n_layers * layer + 4 * seen * m.n_q * m.head_dim * m.n_layers + 2 * logit_rows * head)


def _stack_work(requests, logit_rows):
    cfg = _stack_config()
    W, rows = cfg["width"], sum(r for r, _ in requests)
    seen, kv = sum(_pairs(r, p, 0) for r, p in requests), sum(r + p + r for r, p in requests)
    weights = sum(math.prod(s) for n, s in mw.tensor_shapes(cfg, mix_timing.RANK).items() if len(s) == 2 and n != "embed")
    work = dict(bytes=2 * weights, flops=2 * rows * weights)
    for layer in cfg["layers"]:
        m = layer["mixer"]
        b = m.get("right", m)
        state = b["heads"] * b["dim"] ** 2
        work["bytes"] += 2 * 4 * state * len(requests)
        work["flops"] += 6 * state * rows
        if "left" in m:
            a = m["left"]
            work["bytes"] += 2 * kv * a["kv_heads"] * (a["dim"] + a["vdim"])
            work["flops"] += 2 * seen * a["heads"] * (a["dim"] + a["vdim"])
    if logit_rows:
        work["bytes"] += 2 * W * cfg["vocab"] + 4 * logit_rows * cfg["vocab"]
        work["flops"] += 2 * logit_rows * W * cfg["vocab"]
    return work


def _sum(parts):
    return {k: float(sum(p[k] for p in parts)) for k in ("bytes", "flops")}


def work(case):
    kind = case["kind"]
    if kind == "decode":
        n, keys = case["sessions"], case["sessions"] * (case["lo"] + case["hi"]) / 2
        return dict(bytes=4 * keys * case["nkv"] * case["hd"] + 8 * n * case["nq"] * case["hd"], flops=4 * keys * case["nq"] * case["hd"])
    if kind == "prefill":
        T, ctx, kv = case["rows"], case["ctx"], case["nkv"] * case["hd"]
        old = min(ctx, case["window"] or ctx)                # cached rows that any new row sees
        return dict(bytes=8 * T * case["nq"] * case["hd"] + 2 * T * kv * (4 + 2) + 4 * old * kv,
                    flops=4 * case["nq"] * case["hd"] * _pairs(T, ctx, case["window"]))
    if kind == "experts":
        used = EXPERTS * (1 - (1 - TOP / EXPERTS) ** case["rows"])           # experts that some row chose
        return dict(bytes=4 * used * WIDTH * EXPERT_FF + case["rows"] * (10 * WIDTH + 4 * EXPERTS + 8 * TOP),
                    flops=4 * case["rows"] * TOP * WIDTH * EXPERT_FF)
    step = _qwen_work if case["model"] == "qwen3-0.6b" else _stack_work
    if kind == "chat":
        return _sum([step([(case["prompt"], 0)], 0)] + [step([(1, case["prompt"] + i)], 1) for i in range(case["steps"])])
    at = [(case["lo"] + case["hi"]) // 2] * case["sessions"]
    return _sum([step([(1, p + i) for p in at], len(at)) for i in range(case["steps"])])


def tolerance(case):
    """About four times the distance from 64-bit arithmetic that the path shows."""
    kind = case["kind"]
    if kind == "decode":
        return {"rel": 2e-6}                                 # 32-bit sums over binary16 keys and values: 2.3e-7 to 4.1e-7
    if kind == "prefill":
        return {"rel": 1.2e-3}                               # queries and weights in binary16: 2.1e-4 to 3.0e-4
    if kind == "experts":
        return {"rel": 3e-3}                                 # bfloat16 units between the products: 8e-4
    # prompts attend with binary16 queries: 1.6e-4 to 5.2e-4; bfloat16 operands throughout: 4.3e-3 to 9.5e-3
    return {"rel": 2e-3} if case["model"] == "qwen3-0.6b" else {"rel": 0.03}
