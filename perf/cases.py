"""What a user of this framework has the GPU do, as measurable cases.

A case is one call (or, for a whole model, one token or one prompt) through the
public entry points: the C ABI of include/gq_hip.h as guanaco_amd.hip exposes
it.  Inputs are made on the GPU from a seed; weights are blocks of the K-quant
formats with the statistics of trained ones (zero mean, standard deviation
about 0.02, scales that vary from block to block).  `exact` evaluates the same
mathematics in float64 with torch alone.

Shapes come from guanaco_amd.spec: the 8B and the 1.1B Llama shapes that the
benchmark and the tests run, in the Q4_K_M mix and in Q8_0.
"""
import ctypes as C
import math
import random

import numpy as np
import torch

import guanaco_amd.hip as H
from guanaco_amd import spec as S

DEV = "cuda"
PAD = 256  # weights carry this much tail padding (include/gq_hip.h)
EPS = 1e-6
QK = {n: S.BLOCK[d] for n, d in (("q4_k", S.Q4_K), ("q6_k", S.Q6_K), ("q8_0", S.Q8_0))}
CODE = {"q4_k": S.Q4_K, "q6_k": S.Q6_K, "q8_0": S.Q8_0}
# model shapes by name, with the dtype rule of the layers
SHAPES = {"8b": (S.LLAMA8B, "q4_k_m"), "1.1b": (S.TINYLLAMA, "q4_k_m"), "1.1b_q8": (S.TINYLLAMA_Q8, "q8_0")}


# ------------------------------------------------------------------- inputs
def _gen(seed, tag):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + int(tag) * 7919 + 12345) % (1 << 62))
    return g


def _half_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(v.shape + (2,))


def quant(dtype, rows, cols, seed, tag, role=""):
    """rows x cols random blocks of a dtype (uint8, tail padding included).
    role: "residual" for the o and down projections, which depth-scaled
    initialisation makes smaller (here by four), "embed" for embeddings of
    standard deviation about one."""
    qk, bb = QK[dtype]
    n = rows * (cols // qk)
    g = _gen(seed, tag)
    out = torch.zeros(n * bb + PAD, dtype=torch.uint8, device=DEV)
    blk = out[:n * bb].view(n, bb)
    # the block scale varies by +-25 %
    var = 0.75 + 0.5 * torch.rand(n, generator=g, device=DEV)
    res, emb = role == "residual", 40.0 if role == "embed" else 1.0
    rnd = lambda k, hi=256: torch.randint(0, hi, (n, k), generator=g, device=DEV, dtype=torch.uint8)  # noqa: E731
    if dtype == "q4_k":  # w = d sc q - dmin m; m = sc and dmin = 7.5 d: zero mean
        d = 1.2e-4 * emb * var
        blk[:, 0:2] = _half_bytes(d)
        blk[:, 2:4] = _half_bytes(7.5 * d.to(torch.float16).float())
        sc = rnd(8, 16 if res else 64)
        hi = (sc[:, 4:] >> 4) << 6
        blk[:, 4:8] = sc[:, :4] | hi
        blk[:, 8:12] = sc[:, :4] | hi
        blk[:, 12:16] = (sc[:, 4:] & 15) | ((sc[:, 4:] & 15) << 4)
        blk[:, 16:] = rnd(128)
    elif dtype == "q6_k":  # w = d sc (q - 32), sc of either sign
        blk[:, 0:192] = rnd(192)
        blk[:, 192:208] = rnd(16, 16) - 8  # wraps to int8 -8 .. 7
        blk[:, 208:210] = _half_bytes((6.4e-5 if res else 2.3e-4) * var)
    else:  # w = d q
        blk[:, 0:2] = _half_bytes((6.8e-5 if res else 2.7e-4) * emb * var)
        blk[:, 2:] = rnd(32)
    return out


def normal(shape, seed, tag, scale=1.0):
    return torch.randn(shape, generator=_gen(seed, tag), device=DEV, dtype=torch.float32) * scale


def norm_weight(n, seed, tag):
    return 1.0 + normal((n,), seed, tag, 1.0 / 16)


def dequant(dtype, w, rows, cols):
    """The weights of `quant` in float64, rows x cols."""
    qk, bb = QK[dtype]
    n = rows * (cols // qk)
    b = w[:n * bb].view(n, bb)
    half = lambda a: b[:, a:a + 2].contiguous().view(torch.float16).double()  # noqa: E731, (n, 1)
    if dtype == "q4_k":
        d, dm = half(0), half(2)
        s = b[:, 4:16].long()
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        q = b[:, 16:].view(n, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).double()  # (n, chunk, nibble, 32): sub-block 2 chunk + nibble
        out = (d * sc).view(n, 4, 2, 1) * q - (dm * mn).view(n, 4, 2, 1)
    elif dtype == "q6_k":
        ql = b[:, 0:128].view(n, 2, 2, 32)  # half, 32-byte group, l
        qh = b[:, 128:192].view(n, 2, 1, 32)
        q = torch.cat([ql & 15, ql >> 4], 2)  # (n, half, group, l)
        sh = torch.tensor([0, 2, 4, 6], device=DEV, dtype=torch.uint8).view(1, 1, 4, 1)
        q = (q | (((qh >> sh) & 3) << 4)).double() - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double().view(n, 2, 4, 2, 1)
        out = half(208).view(n, 1, 1, 1, 1) * sc * q.view(n, 2, 4, 2, 16)
    else:
        out = half(0) * b[:, 2:].contiguous().view(torch.int8).double()
    return out.reshape(rows, cols)


def qbytes(dtype, rows, cols):
    qk, bb = QK[dtype]
    return rows * (cols // qk) * bb


# ------------------------------------------------------------------- models
def layer_dtypes(mix, layer):
    if mix == "q8_0":
        return ["q8_0"] * 7
    six = "q6_k" if layer % 2 == 0 else "q4_k"  # Q4_K_M: half of the v and down projections
    return ["q4_k", "q4_k", six, "q4_k", "q4_k", "q4_k", six]


def model_shape(case):
    s, mix = SHAPES[case["shape"]]
    kvd = s.n_kv_heads * s.head_dim
    Hd, F = s.hidden, s.ff
    return s, mix, [(Hd, Hd), (kvd, Hd), (kvd, Hd), (Hd, Hd), (F, Hd), (F, Hd), (Hd, F)]


def head_dtypes(mix):
    return ("q8_0", "q8_0") if mix == "q8_0" else ("q4_k", "q6_k")  # embedding, LM head


def model_weights(case, seed):
    """Every tensor of the case's model: a generator of (layer or -1, list)."""
    s, mix, shapes = model_shape(case)
    for l in range(case["layers"]):
        dts = layer_dtypes(mix, l)
        yield l, [quant(dts[i], *shapes[i], seed, 100 * l + i, "residual" if i in (3, 6) else "") for i in range(7)] + [
            norm_weight(s.hidden, seed, 100 * l + 7), norm_weight(s.hidden, seed, 100 * l + 8)]
    ed, hd = head_dtypes(mix)
    yield -1, [quant(ed, s.vocab, s.hidden, seed, 90001, "embed"), quant(hd, s.vocab, s.hidden, seed, 90002),
               norm_weight(s.hidden, seed, 90003)]


def history(s, layer, n, seed):
    """K and V rows of positions 0 .. n-1 of one layer (n_kv x n x head_dim)."""
    return (normal((s.n_kv_heads, n, s.head_dim), seed, 50000 + 2 * layer),
            normal((s.n_kv_heads, n, s.head_dim), seed, 50001 + 2 * layer))


def prompt_tokens(case, seed):
    s = model_shape(case)[0]
    r = random.Random(seed * 31 + 7)
    return np.array([r.randrange(s.vocab) for _ in range(case["T"])], np.int32)


class View:
    """A device array of another owner, as torch sees it."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = dict(shape=shape, strides=None, typestr="<f4", data=(ptr, False), version=3)


def slab(ptr, heads, max_seq, hd):
    """A layer's K or V slab; only valid while its context is open."""
    return torch.as_tensor(View(ptr, (heads, max_seq, hd)), device=DEV)


class Rows(list):
    """Views of a context's cache with the state that owns the context, which
    has to outlive them (a closed context frees its cache)."""

    owner = None


class Buf:
    """A torch tensor as the methods of guanaco_amd.hip take a buffer."""

    def __init__(self, t):
        self.t, self.ptr = t, t.data_ptr()


class ModelState:
    """One context with a bound model and its KV cache, as a program holds."""

    def __init__(self, case, seed, past, max_seq):
        s, mix, shapes = model_shape(case)
        n = case["layers"]
        self.ctx = H.Context(0)
        self.ctx.kv_init(n, s.n_kv_heads, s.head_dim, max_seq, s.rope_theta)
        self.max_seq, self.s, self.n = max_seq, s, n
        self.keep = []
        layers = (H.GqLayer * n)()
        for l, ts in model_weights(case, seed):
            self.keep += ts
            if l >= 0:
                dts = layer_dtypes(mix, l)
                for i, f in enumerate(("wq", "wk", "wv", "wo", "w_gate", "w_up", "w_down")):
                    setattr(layers[l], f, H.GqWeight(ts[i].data_ptr(), CODE[dts[i]], *shapes[i]))
                layers[l].rms_att, layers[l].rms_ffn = ts[7].data_ptr(), ts[8].data_ptr()
                if past:
                    for t, p in zip(history(s, l, past, seed), (H.lib.gq_hip_kv_k, H.lib.gq_hip_kv_v)):
                        slab(p(self.ctx.h, l), s.n_kv_heads, max_seq, s.head_dim)[:, :past] = t
            else:
                ed, hd = head_dtypes(mix)
                m = H.GqModel(n, s.hidden, s.ff, s.n_heads, s.n_kv_heads, s.head_dim, s.vocab, s.rope_theta, EPS,
                              C.cast(layers, C.POINTER(H.GqLayer)), H.GqWeight(ts[0].data_ptr(), CODE[ed], s.vocab, s.hidden),
                              H.GqWeight(ts[1].data_ptr(), CODE[hd], s.vocab, s.hidden), ts[2].data_ptr())
        torch.cuda.synchronize()  # the weights are written before the model is bound
        self.ctx.check(H.lib.gq_hip_model_bind(self.ctx.h, C.byref(m)), "model_bind")
        self.logits = np.zeros(s.vocab, np.float32)
        self.hidden = np.zeros(s.hidden, np.float32)

    def rows(self, layer, pos, n):
        """K and V of positions pos .. pos + n - 1 of a layer (views)."""
        s = self.s
        r = Rows(slab(p(self.ctx.h, layer), s.n_kv_heads, self.max_seq, s.head_dim)[:, pos:pos + n]
                 for p in (H.lib.gq_hip_kv_k, H.lib.gq_hip_kv_v))
        r.owner = self
        return r

    def __del__(self):
        if getattr(self, "ctx", None) and H is not None and H.lib is not None:  # not at interpreter exit
            self.ctx.close()


_shared = {}


def shared_ctx(key=None, kv=None):
    """One context for all states of a geometry, as one program has one: its
    calls run in order on one stream.  kv: (layers, kv heads, head_dim,
    max_seq, theta) of its cache; a state owns one layer of it."""
    if key not in _shared:
        for k in [k for k, v in _shared.items() if k is not None and len(v[1]) == v[2]]:
            _shared.pop(k)[0].close()
        ctx = H.Context(0)
        if kv:
            ctx.kv_init(*kv)
        n = kv[0] if kv else 0
        _shared[key] = (ctx, list(range(n)), n)
    return _shared[key]


class Slot:
    """One layer of a shared context's cache, given back with the state."""

    def __init__(self, key, kv):
        self.ctx, self.free, _ = shared_ctx(key, kv)
        self.layer = self.free.pop(0)

    def __del__(self):
        self.free.append(self.layer)


# -------------------------------------------------------------------- cases
def listed():
    return [
        # one projection of the 1.1B model through the matvec entry: the smallest call there is
        dict(name="matvec_q4k_2048", kind="matvec", dtype="q4_k", rows=2048, cols=2048),
        # a down projection of the 8B model on its own, as the per-layer host split calls it
        dict(name="matvec_q6k_down_8b", kind="matvec", dtype="q6_k", rows=4096, cols=14336),
        # final RMSNorm + LM head of a Q8_0 model
        dict(name="head_q8_32000", kind="head", dtype="q8_0", rows=32000, cols=2048),
        # attention of one token over a long context (8B heads)
        dict(name="attention_8b_32k", kind="attention", heads=32, kv_heads=8, hd=128, pos=32767, max_seq=32832),
        # attention of a prompt's last chunk (the runtime's chunk of 512 tokens) over 4096 positions
        dict(name="prompt_attention_8b", kind="prompt_attention", heads=32, kv_heads=8, hd=128, T=512, pos=3584, max_seq=4160),
        # attention of a short chat turn in the 1.1B model
        dict(name="prompt_attention_turn", kind="prompt_attention", heads=32, kv_heads=4, hd=64, T=77, pos=301, max_seq=2048),
        # the reference's default sampler over a real vocabulary
        dict(name="sample_topk40", kind="sample", vocab=128256, mode="top_k", k=40, p=0.9, temp=0.7),
        # one decode step through two layers and the head of the Q8_0 model, short context
        dict(name="token_1b_q8", kind="token", shape="1.1b_q8", layers=2, pos=301, max_seq=2048),
        # a chat turn's prompt through two layers of the Q8_0 model
        dict(name="turn_1b_q8", kind="prompt", shape="1.1b_q8", layers=2, T=37, pos=301, max_seq=2048),
        # one full chunk through two layers of the 8B model
        dict(name="chunk_8b", kind="prompt", shape="8b", layers=2, T=512, pos=0, max_seq=2048),
        # the benchmark's decode step: the whole 8B model at context 8192
        dict(name="token_8b", kind="token", shape="8b", layers=32, pos=8192, max_seq=8320),
        # a long prompt through the whole 8B model, chunks and a ragged rest
        dict(name="prompt_8b", kind="prompt", shape="8b", layers=32, T=1500, pos=0, max_seq=2048),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["matvec", "head", "attention", "prompt_attention", "sample", "token", "prompt", "prompt"])
    if kind in ("matvec", "head"):
        dtype = rng.choice(["q4_k", "q6_k", "q8_0"])
        cols = 256 * _log(rng, 2, 112 if kind == "matvec" else 32)
        if dtype == "q8_0" and rng.random() < 0.3:
            cols += 32 * rng.randrange(1, 8)  # Q8_0 rows need only whole 32-weight blocks
        rows = _log(rng, 64, 16384) if kind == "matvec" else _log(rng, 1000, 128256)
        return dict(kind=kind, dtype=dtype, rows=rows, cols=cols)
    if kind in ("attention", "prompt_attention"):
        hd, group = rng.choice([64, 128]), rng.choice([1, 2, 4, 8])
        kv = rng.choice([2, 4, 8]) if group > 1 else rng.choice([4, 8, 16, 32])
        if kind == "attention":
            pos = _log(rng, 1, 32768) - 1
            ms = min(32832, max(64, rng.choice([pos + 1, pos + 100, 2 * (pos + 1)])))
            return dict(kind=kind, heads=kv * group, kv_heads=kv, hd=hd, pos=pos, max_seq=max(ms, pos + 1))
        T, pos = _log(rng, 1, 512), rng.choice([0, _log(rng, 1, 7500)])
        return dict(kind=kind, heads=kv * group, kv_heads=kv, hd=hd, T=T, pos=pos, max_seq=pos + T + rng.randrange(0, 200))
    if kind == "sample":
        return dict(kind=kind, vocab=_log(rng, 1000, 131072), mode=rng.choice(["top_k", "top_k", "top_p", "temperature"]),
                    k=_log(rng, 1, 200), p=round(rng.uniform(0.5, 0.98), 3), temp=round(rng.uniform(0.4, 1.3), 2))
    shape = rng.choice(["8b", "1.1b", "1.1b_q8"])
    if kind == "token":
        pos = _log(rng, 1, 16384) - 1
        return dict(kind=kind, shape=shape, layers=rng.randrange(1, 5), pos=pos, max_seq=pos + 1 + rng.randrange(0, 600))
    T, pos = _log(rng, 2, 1500), rng.choice([0, 0, _log(rng, 1, 6000)])
    return dict(kind=kind, shape=shape, layers=rng.randrange(1, 4), T=T, pos=pos, max_seq=pos + T + rng.randrange(0, 600))


# ------------------------------------------------------------ prepare / run
def _logits(case, seed):
    """Logits as a language model's: a broad body and a few likely tokens."""
    n = case["vocab"]
    x = normal((n,), seed, 1, 2.2)
    top = torch.randint(0, n, (max(4, n // 2000),), generator=_gen(seed, 2), device=DEV)
    x[top] += 4.0 + 3.0 * torch.rand(top.shape, generator=_gen(seed, 3), device=DEV)
    return x


def _rnd(seed):
    return random.Random(seed * 17 + 3).randrange(1 << 31)


class State:
    pass


def prepare(case, seed):
    kind = case["kind"]
    if kind == "token":
        st = ModelState(case, seed, case["pos"], case["max_seq"])
        st.token = random.Random(seed).randrange(st.s.vocab)
    elif kind == "prompt":
        st = ModelState(case, seed, case["pos"], case["max_seq"])
        st.tokens = prompt_tokens(case, seed)
    else:
        st = State()
        if kind in ("matvec", "head"):
            st.ctx = shared_ctx()[0]
            st.w = quant(case["dtype"], case["rows"], case["cols"], seed, 1)
            st.x = Buf(normal((case["cols"],), seed, 2, 1.0 if kind == "matvec" else 3.0))
            st.y = Buf(torch.zeros(case["rows"], device=DEV))
            st.nw = Buf(norm_weight(case["cols"], seed, 3))
        elif kind == "sample":
            st.ctx = shared_ctx()[0]
            st.x = Buf(_logits(case, seed))
            st.rnd = _rnd(seed)
        else:
            nh, nkv, hd, ms = case["heads"], case["kv_heads"], case["hd"], case["max_seq"]
            st.slot = Slot((nkv, hd, ms), (8, nkv, hd, ms, S.LLAMA8B.rope_theta))
            st.ctx = st.slot.ctx
            past = case["pos"] + (1 if kind == "attention" else 0)
            for p, tag in ((H.lib.gq_hip_kv_k, 1), (H.lib.gq_hip_kv_v, 2)):
                if past:
                    slab(p(st.ctx.h, st.slot.layer), nkv, ms, hd)[:, :past] = normal((nkv, past, hd), seed, tag)
            T = case.get("T", 1)
            st.q0 = Buf(normal((T, nh, hd), seed, 3))
            st.q = Buf(st.q0.t.clone())
            st.k, st.v = Buf(normal((T, nkv, hd), seed, 4)), Buf(normal((T, nkv, hd), seed, 5))
            st.out = Buf(torch.zeros((T, nh, hd), device=DEV))
    st.case = case
    torch.cuda.synchronize()
    return st


def _ints(a):
    return a.ctypes.data_as(C.POINTER(C.c_int32))


def run(st):
    case, kind = st.case, st.case["kind"]
    if kind == "matvec":
        st.ctx.matvec_dev(CODE[case["dtype"]], st.w.data_ptr(), case["rows"], case["cols"], st.x, st.y)
        return st.y.t
    if kind == "head":
        st.ctx.matvec_norm_dev(CODE[case["dtype"]], st.w.data_ptr(), case["rows"], case["cols"], st.x, st.nw, EPS, st.y)
        return st.y.t
    if kind == "sample":
        mode = case["mode"]
        tok = H.lib.gq_hip_sample_dev(st.ctx.h, st.x.ptr, case["vocab"], case["temp"],
                                      case["k"] if mode == "top_k" else 0, case["p"] if mode == "top_p" else 1.0, st.rnd)
        if tok < 0:
            st.ctx.raise_last("sample_dev", tok)
        return tok
    if kind == "attention":
        st.ctx.check(st.ctx.attention_dev(st.slot.layer, case["pos"], case["heads"], st.q, st.out), "attention_dev")
        return st.out.t
    if kind == "prompt_attention":
        # q is rotated in place: the projection's fresh output each time
        st.ctx.check(H.lib.gq_hip_copy_dev(st.ctx.h, st.q.ptr, st.q0.ptr, 4 * st.q0.t.numel()), "copy_dev")
        st.ctx.check(st.ctx.prefill_attention_dev(st.slot.layer, case["pos"], case["T"], case["heads"], st.q, st.k, st.v,
                                                  st.out), "prefill_attention_dev")
        return st.out.t
    if kind == "token":
        tok = H.lib.gq_hip_forward_token(st.ctx.h, st.token, case["pos"], H._f(st.logits), None)
        if tok < 0:
            st.ctx.raise_last("forward_token", tok)
        return {"logits": st.logits, "kv": st.rows(st.n - 1, case["pos"], 1)}
    tok = H.lib.gq_hip_prefill(st.ctx.h, _ints(st.tokens), case["T"], case["pos"], H._f(st.logits), H._f(st.hidden), None)
    if tok < 0:
        st.ctx.raise_last("prefill", tok)
    return {"logits": st.logits, "hidden": st.hidden, "kv": st.rows(st.n - 1, case["pos"], case["T"])}


# ------------------------------------------------------------ work, tolerance
def work(case):
    kind = case["kind"]
    if kind in ("matvec", "head"):
        n = qbytes(case["dtype"], case["rows"], case["cols"])
        return {"bytes": n + 4 * (case["rows"] + case["cols"] * (2 if kind == "head" else 1)),
                "flops": 2 * case["rows"] * case["cols"]}
    if kind == "sample":
        return {"bytes": 4 * case["vocab"], "flops": case["vocab"]}
    if kind in ("attention", "prompt_attention"):
        T, nh, nkv, hd = case.get("T", 1), case["heads"], case["kv_heads"], case["hd"]
        n = case["pos"] + T
        keys = T * case["pos"] + T * (T + 1) // 2 if kind == "prompt_attention" else n
        return {"bytes": 4 * hd * (2 * nkv * n + 2 * nh * T + (2 * nkv * T if kind == "prompt_attention" else 0)),
                "flops": 4 * hd * nh * keys}
    s, mix, shapes = model_shape(case)
    T, L = case.get("T", 1), case["layers"]
    wb, params = 0, 0
    for l in range(L):
        for dt, (r, c) in zip(layer_dtypes(mix, l), shapes):
            wb += qbytes(dt, r, c)
            params += r * c
    ed, hd = head_dtypes(mix)
    head = qbytes(hd, s.vocab, s.hidden)
    keys = T * case["pos"] + T * (T + 1) // 2
    kv = 8 * s.n_kv_heads * s.head_dim * L * (case["pos"] + T)
    return {"bytes": wb + head + T * qbytes(ed, 1, s.hidden) + 4 * s.hidden * (2 * L + 1) + kv + 4 * s.vocab,
            "flops": 2 * params * T + 2 * s.vocab * s.hidden + 4 * s.head_dim * s.n_heads * keys * L}


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    if kind in ("matvec", "head", "attention", "prompt_attention"):
        return {"rel": 4e-6}  # fp32 sums: 1.4e-7 .. 6e-7 from float64
    if kind == "token":
        return {"rel": 3e-5}  # fp32 throughout: 6.4e-6 from float64 after 32 layers
    # bf16 GEMM inputs: 1.3e-3 .. 3.7e-3 from float64 after two layers, 1.5e-2
    # after 32, where another order of the sums moves the outputs by 1.1e-2
    return {"rel": 3e-2 if case["layers"] > 8 else 1.5e-2}


# -------------------------------------------------------------------- exact
def _rope(x, pos0, theta):
    """x: T x heads x hd in float64; the angles are the reference's fp32 ones."""
    T, _, hd = x.shape
    p = (theta ** (np.arange(0, hd, 2, dtype=np.float32) / np.float32(hd)).astype(np.float64)).astype(np.float32)
    f = np.float32(1.0) / p
    a = (np.arange(pos0, pos0 + T, dtype=np.float32)[:, None] * f[None]).astype(np.float64)
    c, s = (torch.from_numpy(v).to(DEV)[:, None, :] for v in (np.cos(a), np.sin(a)))
    e, o = x[..., 0::2], x[..., 1::2]
    return torch.stack([e * c - o * s, e * s + o * c], -1).reshape(x.shape)


def _attend(q, k, v, pos):
    """q: T x heads x hd; k, v: kv x n x hd; token t sees positions 0 .. pos + t."""
    T, nh, hd = q.shape
    nkv, n, _ = k.shape
    out = torch.empty_like(q)
    mask = torch.arange(n, device=DEV)[None] > (pos + torch.arange(T, device=DEV))[:, None]
    for h in range(nh):
        kk, vv = k[h // (nh // nkv)], v[h // (nh // nkv)]
        s = q[:, h] @ kk.T.contiguous() / math.sqrt(hd)
        s.masked_fill_(mask, -math.inf)
        out[:, h] = torch.softmax(s, 1) @ vv
    return out


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("matvec", "head"):
        w = dequant(case["dtype"], quant(case["dtype"], case["rows"], case["cols"], seed, 1), case["rows"], case["cols"])
        x = normal((case["cols"],), seed, 2, 1.0 if kind == "matvec" else 3.0).double()
        return w @ (x if kind == "matvec" else _rms(x, norm_weight(case["cols"], seed, 3)))
    if kind == "sample":
        return None
    if kind in ("attention", "prompt_attention"):
        nh, nkv, hd, pos, T = case["heads"], case["kv_heads"], case["hd"], case["pos"], case.get("T", 1)
        past = pos + (1 if kind == "attention" else 0)
        k, v = (normal((nkv, past, hd), seed, t).double() for t in (1, 2))
        q = normal((T, nh, hd), seed, 3).double()
        if kind == "prompt_attention":
            kn, vn = (normal((T, nkv, hd), seed, t).double() for t in (4, 5))
            q, kn = _rope(q, pos, S.LLAMA8B.rope_theta), _rope(kn, pos, S.LLAMA8B.rope_theta)
            k, v = torch.cat([k, kn.transpose(0, 1)], 1), torch.cat([v, vn.transpose(0, 1)], 1)
        return _attend(q, k, v, pos)
    s, mix, shapes = model_shape(case)
    pos = case["pos"]
    tokens = prompt_tokens(case, seed) if kind == "prompt" else np.array([random.Random(seed).randrange(s.vocab)])
    T, (ed, hdt) = len(tokens), head_dtypes(mix)
    rb = qbytes(ed, 1, s.hidden)
    emb = quant(ed, s.vocab, s.hidden, seed, 90001, "embed")[:s.vocab * rb].view(s.vocab, rb)
    x = dequant(ed, emb[torch.from_numpy(tokens.astype(np.int64)).to(DEV)].reshape(-1), T, s.hidden)
    for l, ts in model_weights(case, seed):
        if l < 0:
            last = x[-1]
            logits = dequant(hdt, ts[1], s.vocab, s.hidden) @ _rms(last, ts[2])
            break
        dts = layer_dtypes(mix, l)
        mm = lambda i, a: a @ dequant(dts[i], ts[i], *shapes[i]).T  # noqa: E731,B023
        h = _rms(x, ts[7])
        q = _rope(mm(0, h).view(T, s.n_heads, s.head_dim), pos, s.rope_theta)
        kn = _rope(mm(1, h).view(T, s.n_kv_heads, s.head_dim), pos, s.rope_theta).transpose(0, 1)
        vn = mm(2, h).view(T, s.n_kv_heads, s.head_dim).transpose(0, 1)
        kp, vp = history(s, l, pos, seed)
        att = _attend(q, torch.cat([kp.double(), kn], 1), torch.cat([vp.double(), vn], 1), pos)
        x = x + mm(3, att.reshape(T, s.hidden))
        h = _rms(x, ts[8])
        g = mm(4, h)
        x = x + mm(6, g * torch.sigmoid(g) * mm(5, h))
    out = {"logits": logits, "kv": [kn, vn]}
    if kind == "prompt":
        out["hidden"] = last
    return out
