"""Performance cases of the RWKV-7 forward step, through the public entry points.

A case is one block of a layer (the feed-forward block, the time-mix block,
the head with the sampler, the WKV7 scan) issued as the model driver issues
it over the C-ABI of include/rsv_hip.h, or one whole call of the Bundle API on
a model of a few layers.  Widths and LoRA ranks are those of synth.TINY and
synth.THREE_B and widths between them; row counts run from one decoded token
to a packed prefill chunk of 4096 rows (the driver's default).

Layer weights are int8 in the reference's per-row or per-group format, or
fp16.  Weights are made per state from the seed; the whole-call cases keep one
model per process, as a program does, and take their prompts from the seed.
All states share one backend context (one stream), as a program's calls do.
"""
import ctypes
import functools
import math
import os
import random
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rwkv-rsv_amd"))

import rsv  # noqa: E402
import synth  # noqa: E402

NONE = rsv.NONE
N = 64  # head size
VOCAB = synth.THREE_B["vocab"]
LN_EPS, GN_EPS, L2_EPS = 1e-5, 64e-5, 1e-12
DECAY = -1.0 / math.sqrt(math.e)
WIDTHS = (768, 1024, 1536, 2048, 2560)
SMALL_PROMPT = 128  # rows up to which a prefill chunk runs on the decode GEMMs (the driver's own line)


def listed():
    return [
        # one decoded token of the small model: the smallest call, latency and launches
        dict(name="ffn_decode_1", kind="ffn", c=768, rows=1, weights="int8"),
        # one step of 64 concurrent sessions through the feed-forward block
        dict(name="ffn_decode_64", kind="ffn", c=2560, rows=64, weights="int8"),
        # a short prompt, on the decode GEMMs
        dict(name="ffn_prompt_100", kind="ffn_prompt", c=2560, rows=100, weights="int8"),
        # a full packed prefill chunk
        dict(name="ffn_prompt_4096", kind="ffn_prompt", c=2560, rows=4096, weights="fp16"),
        # one decoded token, 8 and 64 sessions through the time-mix block (projections, LoRA, WKV7, output)
        dict(name="tmix_decode_1", kind="tmix", c=2560, rows=1, weights="int8"),
        dict(name="tmix_decode_8", kind="tmix", c=2560, rows=8, weights="int8"),
        dict(name="tmix_decode_64", kind="tmix", c=2560, rows=64, weights="int8"),
        # one long prompt alone, and a chunk packed from the pieces of several prompts
        dict(name="tmix_prompt_1x700", kind="tmix_prompt", c=2560, rows=700, segs=1, weights="int8"),
        dict(name="tmix_prompt_24x4096", kind="tmix_prompt", c=2560, rows=4096, segs=24, weights="int8"),
        # final norm, head and top-p sampler of 8 sessions
        dict(name="head_sample_8", kind="head", c=2560, rows=8, weights="int8", pick="top_p"),
        # whole calls on a two-layer model of the 3B widths: token-by-token inference, and ragged prompts
        # prefilled with their last logits
        dict(name="model_tokens_24", kind="model_tokens", rows=24),
        dict(name="model_prompts_5x1500", kind="model_prompts", rows=1500, segs=5),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["ffn", "ffn", "ffn_prompt", "ffn_prompt", "tmix", "tmix", "tmix_prompt", "tmix_prompt",
                       "scan", "head", "model_tokens", "model_prompts"])
    c, weights = rng.choice(WIDTHS), rng.choice(["int8", "int8", "int8_group", "fp16"])
    if kind in ("ffn", "tmix"):  # sessions of a decode step
        return dict(kind=kind, c=c, rows=_log_int(rng, 1, 64), weights=weights)
    if kind == "ffn_prompt":
        return dict(kind=kind, c=c, rows=_log_int(rng, 2, 4096), weights=weights)
    if kind in ("tmix_prompt", "scan"):
        rows = _log_int(rng, 2, 4096)
        return dict(kind=kind, c=c, rows=rows, segs=_log_int(rng, 1, min(64, rows)), weights=weights)
    if kind == "head":
        return dict(kind=kind, c=c, rows=_log_int(rng, 1, 8), weights=weights,
                    pick=rng.choice(["top_p", "top_k", "argmax"]))
    if kind == "model_tokens":
        return dict(kind=kind, rows=rng.randint(1, 24))
    rows = _log_int(rng, 8, 1500)
    return dict(kind=kind, rows=rows, segs=_log_int(rng, 1, 5))


# ---------------------------------------------------------------- inputs
def _ranks(c):
    cfg = synth.THREE_B if c >= 2048 else synth.TINY
    return cfg["wm"], cfg["am"], cfg["vm"], cfg["gm"]


def _lens(case):
    """Segment lengths of a packed chunk: fixed by the case, ragged, each at least 1."""
    rows, segs = case["rows"], case["segs"]
    rng = random.Random(rows * 1009 + segs)
    part = [rng.uniform(0.3, 1.0) for _ in range(segs)]
    lens = [1 + int((rows - segs) * p / sum(part)) for p in part]
    lens[0] += rows - sum(lens)
    return lens


class _Gen:
    """Seeded inputs on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator("cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0):
        return torch.randn(*shape, generator=self.g, device="cuda") * std + mean

    def uniform(self, *shape):
        return torch.rand(*shape, generator=self.g, device="cuda")

    def ints(self, n, hi):
        return torch.randint(0, hi, (n,), generator=self.g, device="cuda")

    def matrix(self, m, k, weights):
        """A weight [m, k] ~ N(0, 0.02^2): ("fp16", w), or ("int8", idx u8, sz i32) in the reference's format:
        symmetric per row, or min/max per group of 128."""
        w = self.normal(m, k, std=0.02)
        if weights == "fp16":
            return "fp16", w.half()
        if weights == "int8":
            s = (w.abs().amax(1, keepdim=True) / 127).half()
            q = torch.clamp(torch.round(w / s.float()), -127, 127) + 128
            s = s.expand(m, k // 128)
            z = (-128.0 * s.float()).half()
        else:
            g = w.view(m, k // 128, 128)
            lo, hi = g.amin(2), g.amax(2)
            sc = (hi - lo) / 255.0
            q = torch.clamp(torch.round((g - lo[..., None]) / sc[..., None]), 0, 255).view(m, k)
            s, z = sc.half(), lo.half()
        bits = lambda t: t.contiguous().view(torch.int16).int() & 0xFFFF  # noqa: E731
        return "int8", q.to(torch.uint8), bits(s) | (bits(z) << 16)


def _f64(w):
    """A weight of _Gen.matrix in 64 bits."""
    if w[0] == "fp16":
        return w[1].double()
    q, sz = w[1].double(), w[2]
    half = lambda t: t.to(torch.int16).view(torch.float16).double()  # noqa: E731
    s, z = half(sz & 0xFFFF), half((sz >> 16) & 0xFFFF)
    m, k = q.shape
    return (q.view(m, k // 128, 128) * s[..., None] + z[..., None]).view(m, k)


def _ffn_inputs(g, c, weights):
    f = 4 * c
    return dict(ln_w=g.normal(c, std=0.1, mean=1.0), ln_b=g.normal(c, std=0.1), mix=g.uniform(c),
                key=g.matrix(f, c, weights), value=g.matrix(c, f, weights))


def _tmix_inputs(g, c, weights):
    p = dict(ln_w=g.normal(c, std=0.1, mean=1.0), ln_b=g.normal(c, std=0.1))
    p.update({"x_" + n: g.uniform(c) for n in "rwkvag"})
    p.update({n: g.matrix(c, c, weights) for n in ("r", "k", "v", "o")})
    for n, rank in zip("wavg", _ranks(c)):
        p[n + "1"] = g.normal(rank, c, std=0.02).half()
        p[n + "2"] = g.normal(c, rank, std=0.1).half()
    # decays from slow to fast channels, in-context rates and gates around their middle
    p.update(w0=g.normal(c, std=2.0, mean=-1.5), a0=g.normal(c), v0=g.normal(c, mean=0.5), k_k=g.normal(c, 1, std=0.1, mean=0.85).view(c),
             k_a=g.uniform(c), r_k=g.normal(c, std=0.1), gn_w=g.normal(c, std=0.1, mean=1.0), gn_b=g.normal(c, std=0.1))
    return p


# ---------------------------------------------------------------- device side
@functools.lru_cache(None)
def _backend():
    return rsv.Backend(0)


class _Mem:
    """A tensor of the backend, freed when nothing refers to it; torch views it in place."""

    def __init__(self, n, dtype, made=None):
        self.be = _backend()
        self.id = self.be.tensor(n=n, dtype=dtype) if made is None else made
        p = ctypes.c_void_p()
        self.be.call("rsv_tensor_ptr", self.id, ctypes.byref(p))
        self.__cuda_array_interface__ = dict(shape=(n,), typestr={rsv.F32: "<f4", rsv.F16: "<f2", rsv.U32: "<i4"}[dtype],
                                             data=(p.value, False), version=2, strides=None)

    def __del__(self):
        rsv.hip_lib().rsv_tensor_free(self.be.ctx, self.id)


_made = []  # the memory of the state that prepare() is making


class _Dev:
    """A backend tensor's id and its torch view (which keeps the memory alive)."""

    def __init__(self, shape, dtype):
        mem = _Mem(math.prod(shape), dtype)
        _made.append(mem)
        self.id, self.t = mem.id, torch.as_tensor(mem, device="cuda").view(shape)


_KIND = {torch.float32: rsv.F32, torch.float16: rsv.F16, torch.int32: rsv.U32}


def _put(t):
    if t.dtype == torch.uint8:
        t = t.contiguous().view(torch.int32)
    d = _Dev(t.shape, _KIND[t.dtype])
    d.t.copy_(t)
    return d


def _f32(*shape):
    return _Dev(shape, rsv.F32)


def _f16(*shape):
    return _Dev(shape, rsv.F16)


def _u32(values):
    return _put(torch.tensor(np.asarray(values, np.uint32).view(np.int32), device="cuda"))


class _Weight:
    """A layer weight as the driver holds it: row-major, MFMA-tiled (batched decode), and an fp16 copy (prefill)."""

    def __init__(self, w, tiled=False, prompt=False):
        self.m, self.k = w[1].shape
        ids = [_put(t).id for t in w[1:]]
        self.i8 = None if w[0] == "fp16" else rsv.Int8Handle(*ids, self.m, self.k)
        self.w16 = ids[0] if w[0] == "fp16" else NONE
        self.tiled = int(tiled)
        torch.cuda.synchronize()
        if tiled and self.i8:
            self.i8 = rsv.Int8Handle(self.tile(self.i8.idx, 1), self.tile(self.i8.sz, 4), self.m, self.k)
        elif tiled:
            self.w16 = self.tile(self.w16, 2)
        elif prompt and self.i8:
            self.w16 = _f16(self.m, self.k).id
            _backend().call("rsv_dequant_int8_to_f16", ctypes.byref(self.i8), self.w16, self.m, self.k)
            self.i8 = None

    def tile(self, src, esz):
        out = ctypes.c_uint32()
        _backend().call("rsv_tile_weights", src, self.m, self.k, esz, ctypes.byref(out))
        _made.append(_Mem(0, rsv.U32, made=out.value))
        return out.value

    @property
    def w8(self):
        return ctypes.pointer(self.i8) if self.i8 else None


class _State:
    """What a case's pass needs: its launches in order, and its outputs."""

    def __init__(self):
        self.steps, self.keep, self.out = [], [], None

    def op(self, name, *args):
        self.keep.append(args)
        self.steps.append(functools.partial(getattr(rsv.hip_lib(), name), _backend().ctx, *args))

    def run(self):
        for step in self.steps:
            if step():
                raise rsv.RsvError(rsv.hip_lib().rsv_last_error().decode())
        return self.out


def _ids(*devs):
    return (ctypes.c_uint32 * len(devs))(*[d.id if d is not None else NONE for d in devs])


def _gemv_job(w, x, y, pro, epi, **more):
    j = rsv.GemvJob()
    ctypes.memset(ctypes.byref(j), 0xFF, ctypes.sizeof(j))
    j.w16, j.w8, j.m, j.k, j.x, j.y, j.prologue, j.epilogue = w.w16 if not w.i8 else NONE, w.w8, w.m, w.k, x.id, y.id, pro, epi
    for name, d in more.items():
        setattr(j, name, d if isinstance(d, float) else d.id)
    return j


def _gemv(st, jobs, side=(None, None), n=0):
    st.op("rsv_gemv_multi", (rsv.GemvJob * len(jobs))(*jobs), len(jobs), *[d.id if d else NONE for d in side], n, 1)


def _mm_job(w, x, y, epi, bias=None, aux=None, scale=None):
    ids = [d.id if d is not None else NONE for d in (bias, aux, scale)]
    return rsv.MmJob(NONE if w.i8 else w.w16, w.w8, w.m, w.k, x.id, y.id, NONE, epi, *ids, w.tiled)


def _mm(st, name, jobs, rows):
    st.op(name, (rsv.MmJob * len(jobs))(*jobs), len(jobs), rows)


def _kslices(st, w, x, part, nsl, rows):
    job = _mm_job(w, x, part, 0)
    st.op("rsv_gemm_skinny_kslices", ctypes.pointer(job), nsl, rows)


def _vslices(c):
    """k-slices of the feed-forward value product on the batched decode path (the driver's rule)."""
    return (4 * c + 2559) // 2560


# the epilogue codes of include/rsv_hip.h
E_STORE, E_RELU2, E_ADD, E_TANH = 0, 1, 2, 3
G_STORE, G_ADD, G_RELU2, G_TANH, G_WDECAY, G_SIGB, G_VLERP, G_SIG = 0, 2, 3, 4, 5, 6, 7, 8
P_NONE, P_LN, P_GN = 0, 3, 4


def _chunk(case):
    """Row bookkeeping of a packed chunk."""
    lens = _lens(case) if "segs" in case else [case["rows"]]
    start = np.concatenate([[0], np.cumsum(lens)[:-1]])
    prev = np.arange(case["rows"], dtype=np.int64) - 1
    prev[start] = 0x80000000 + np.arange(len(lens))
    return dict(n=len(lens), start=_u32(start), len=_u32(lens), slot=_u32(range(len(lens))),
                last=_u32(start + np.asarray(lens) - 1), prev=_u32(prev))


def _prepare_ffn(case, g):
    c, rows = case["c"], case["rows"]
    p = _ffn_inputs(g, c, case["weights"])
    x0, prev0, part0 = g.normal(rows, c), g.normal(rows, c), g.normal(2, rows, c, std=0.3)
    st = _State()
    x, state, lw, lb, mix = _put(x0), _put(prev0), _put(p["ln_w"]), _put(p["ln_b"]), _put(p["mix"])
    key, value = (_Weight(p[n], tiled=rows > 1) for n in ("key", "value"))
    if rows == 1:
        r2, ln = _f32(1, 4 * c), _f32(1, c)
        _gemv(st, [_gemv_job(key, x, r2, P_LN, E_RELU2, gamma=lw, beta=lb, prev=state, coef=mix, lnout=ln)])
        _gemv(st, [_gemv_job(value, r2, x, P_NONE, E_ADD)], (ln, state), c)
        st.out = [x.t, state.t]
    else:
        nsl = _vslices(c)
        part, xout, xb, r2, vpart = _put(part0), _f32(rows, c), _f16(rows, c), _f16(rows, 4 * c), _f32(nsl, rows, c)
        st.op("rsv_ln_mix_f16_acc", x.id, part.id, 2, xout.id, state.id, lw.id, lb.id, _ids(mix), _ids(xb), 1, c, LN_EPS, rows)
        _mm(st, "rsv_gemm_skinny", [_mm_job(key, xb, r2, G_RELU2)], rows)
        _kslices(st, value, r2, vpart, nsl, rows)
        st.out = [xout.t, state.t, vpart.t]
    return st


def _prepare_ffn_prompt(case, g):
    c, rows = case["c"], case["rows"]
    small = rows <= SMALL_PROMPT
    p = _ffn_inputs(g, c, case["weights"])
    x0, prev0 = g.normal(rows, c), g.normal(1, c)
    st = _State()
    x, state, lw, lb, mix = _put(x0), _put(prev0), _put(p["ln_w"]), _put(p["ln_b"]), _put(p["mix"])
    key, value = (_Weight(p[n], tiled=small, prompt=not small) for n in ("key", "value"))
    xb, r2, seg = _f16(rows, c), _f16(rows, 4 * c), _chunk(case)
    st.op("rsv_seq_norm_mix", x.id, state.id, lw.id, lb.id, _ids(mix), _ids(xb), 1, seg["prev"].id, rows, c, LN_EPS)
    st.op("rsv_seq_state_store", x.id, state.id, lw.id, lb.id, seg["last"].id, seg["slot"].id, 1, c, LN_EPS)
    if small:
        _mm(st, "rsv_gemm_skinny", [_mm_job(key, xb, r2, G_RELU2)], rows)
        _mm(st, "rsv_gemm_skinny", [_mm_job(value, r2, x, G_ADD)], rows)
    else:
        st.op("rsv_gemm_ex", xb.id, key.w16, None, r2.id, rows, 4 * c, c, G_RELU2, NONE, NONE, NONE)
        st.op("rsv_gemm_ex", r2.id, value.w16, None, x.id, rows, c, 4 * c, G_ADD, NONE, NONE, NONE)
    st.out = [x.t, state.t]
    return st


def _lora_struct(d, c, rows, mids, f16):
    """rsv_wkv_lora of include/rsv_hip.h as raw bytes, filled by field."""
    class Op(ctypes.Structure):
        _fields_ = ([(n, ctypes.c_uint32) for n in (
            "state", "r", "k", "v", "v_first", "w_mid", "a_mid", "v_mid", "g_mid", "w2", "a2", "v2", "g2", "w0", "a0",
            "v0", "scale_w", "k_k", "k_a", "r_k", "ln_x_w", "ln_x_b", "yg", "side_src", "side_dst")]
            + [(n, ctypes.c_uint64) for n in ("n_head", "w_rank", "a_rank", "v_rank", "g_rank")]
            + [("eps", ctypes.c_float), ("gn_eps", ctypes.c_float), ("f16_io", ctypes.c_int),
               ("y_bonus", ctypes.c_uint32), ("y_gate", ctypes.c_uint32)])
    op = Op()
    for n in ("side_src", "side_dst", "y_bonus", "y_gate"):
        setattr(op, n, NONE)
    for n, v in d.items():
        setattr(op, n, v.id)
    for n, m in zip("wavg", mids):
        setattr(op, n + "_mid", m.id)
    op.n_head = c // N
    op.w_rank, op.a_rank, op.v_rank, op.g_rank = _ranks(c)
    op.eps, op.gn_eps, op.f16_io = L2_EPS, GN_EPS, int(f16)
    return op


def _prepare_tmix(case, g):
    c, rows = case["c"], case["rows"]
    p = _tmix_inputs(g, c, case["weights"])
    x0, prev0, vf0 = g.normal(rows, c), g.normal(rows, c), g.normal(rows, c)
    s0 = g.normal(rows, c // N, N, N, std=0.1)
    st = _State()
    x, state, vf, rnn = _put(x0), _put(prev0), _put(vf0), _put(s0)
    vec = {n: _put(p[n]) for n in ("ln_w", "ln_b", "x_r", "x_w", "x_k", "x_v", "x_a", "x_g", "w0", "a0", "v0", "k_k",
                                   "k_a", "r_k", "gn_w", "gn_b")}
    scale = _put(torch.tensor([DECAY], device="cuda"))
    W = {n: _Weight(p[n], tiled=rows > 1) for n in ("r", "k", "v", "o")}
    for n in "wavg":
        W[n + "1"] = _Weight(("fp16", p[n + "1"]), tiled=rows > 1)
    up = {n + "2": _put(p[n + "2"]) for n in "wavg"}
    r, k, v = _f32(rows, c), _f32(rows, c), _f32(rows, c)
    common = dict(state=rnn, r=r, k=k, v=v, v_first=vf, w0=vec["w0"], a0=vec["a0"], v0=vec["v0"], scale_w=scale,
                  k_k=vec["k_k"], k_a=vec["k_a"], r_k=vec["r_k"], ln_x_w=vec["gn_w"], ln_x_b=vec["gn_b"], **up)
    if rows == 1:
        mid = {n: _f32(1, rank) for n, rank in zip("wavg", _ranks(c))}
        ln, yn, bonus, gate = _f32(1, c), _f32(1, c), _f32(1, c), _f32(1, c)
        jobs = []
        for n, y, epi, coef in (("r", r, E_STORE, "x_r"), ("k", k, E_STORE, "x_k"), ("v", v, E_STORE, "x_v"),
                                ("v1", mid["v"], E_STORE, "x_v"), ("w1", mid["w"], E_TANH, "x_w"),
                                ("a1", mid["a"], E_STORE, "x_a"), ("g1", mid["g"], E_STORE, "x_g")):
            jobs.append(_gemv_job(W[n], x, y, P_LN, epi, gamma=vec["ln_w"], beta=vec["ln_b"], prev=state,
                                  coef=vec[coef], **({"lnout": ln} if n == "r" else {})))
        _gemv(st, jobs)
        op = _lora_struct(dict(common, yg=yn, side_src=ln, side_dst=state, y_bonus=bonus, y_gate=gate), c, 1,
                          [mid[n] for n in "wavg"], False)
        st.op("rsv_wkv7_lora_decode", ctypes.cast(ctypes.pointer(op), ctypes.c_void_p), 1)
        _gemv(st, [_gemv_job(W["o"], yn, x, P_GN, E_ADD, gamma=vec["gn_w"], beta=vec["gn_b"], prev=bonus, xmul=gate,
                             gn_eps=GN_EPS)])
        st.out = [x.t, rnn.t, state.t]
    else:
        mix = [_f16(rows, c) for _ in range(6)]  # r w k v a g
        mid = {n: _f16(rows, rank) for n, rank in zip("wavg", _ranks(c))}
        yg, part = _f16(rows, c), _f32(2, rows, c)
        st.op("rsv_ln_mix_f16", x.id, state.id, vec["ln_w"].id, vec["ln_b"].id, _ids(*[vec["x_" + n] for n in "rwkvag"]),
              _ids(*mix), 6, c, LN_EPS, rows)
        _mm(st, "rsv_gemm_skinny", [_mm_job(W["r"], mix[0], r, G_STORE), _mm_job(W["k"], mix[2], k, G_STORE),
                                    _mm_job(W["v"], mix[3], v, G_STORE), _mm_job(W["v1"], mix[3], mid["v"], G_STORE),
                                    _mm_job(W["w1"], mix[1], mid["w"], G_TANH), _mm_job(W["a1"], mix[4], mid["a"], G_STORE),
                                    _mm_job(W["g1"], mix[5], mid["g"], G_SIG)], rows)
        op = _lora_struct(dict(common, yg=yg), c, rows, [mid[n] for n in "wavg"], True)
        st.op("rsv_wkv7_lora_decode", ctypes.cast(ctypes.pointer(op), ctypes.c_void_p), rows)
        _kslices(st, W["o"], yg, part, 2, rows)
        st.out = [part.t, rnn.t, state.t]
    return st


def _prepare_tmix_prompt(case, g):
    c, rows = case["c"], case["rows"]
    small = rows <= SMALL_PROMPT
    p = _tmix_inputs(g, c, case["weights"])
    seg = _chunk(case)
    x0, prev0, vf0 = g.normal(rows, c), g.normal(seg["n"], c), g.normal(rows, c)
    s0 = g.normal(seg["n"], c // N, N, N, std=0.1)
    st = _State()
    x, state, vf, rnn = _put(x0), _put(prev0), _put(vf0), _put(s0)
    vec = {n: _put(p[n]) for n in ("ln_w", "ln_b", "x_r", "x_w", "x_k", "x_v", "x_a", "x_g", "w0", "a0", "v0", "k_k",
                                   "k_a", "r_k", "gn_w", "gn_b")}
    scale = _put(torch.tensor([DECAY], device="cuda"))
    W = {n: _Weight(p[n], tiled=small, prompt=not small) for n in ("r", "k", "v", "o")}
    for n in "wavg":
        for d in "12":
            W[n + d] = _Weight(("fp16", p[n + d]), tiled=small)
    mix = [_f16(rows, c) for _ in range(6)]  # r w k v a g
    r, k, v, w, a, gate, yw = (_f32(rows, c) for _ in range(7))
    mid = {n: _f16(rows, rank) for n, rank in zip("wavg", _ranks(c))}
    bonus, yg = _f32(rows, c // N), _f16(rows, c)
    st.op("rsv_seq_norm_mix", x.id, state.id, vec["ln_w"].id, vec["ln_b"].id, _ids(*[vec["x_" + n] for n in "rwkvag"]),
          _ids(*mix), 6, seg["prev"].id, rows, c, LN_EPS)
    st.op("rsv_seq_state_store", x.id, state.id, vec["ln_w"].id, vec["ln_b"].id, seg["last"].id, seg["slot"].id,
          seg["n"], c, LN_EPS)
    mm = "rsv_gemm_skinny" if small else "rsv_gemm_multi"
    _mm(st, mm, [_mm_job(W["r"], mix[0], r, G_STORE), _mm_job(W["k"], mix[2], k, G_STORE),
                 _mm_job(W["v"], mix[3], v, G_STORE), _mm_job(W["v1"], mix[3], mid["v"], G_STORE),
                 _mm_job(W["w1"], mix[1], mid["w"], G_TANH), _mm_job(W["a1"], mix[4], mid["a"], G_STORE),
                 _mm_job(W["g1"], mix[5], mid["g"], G_SIG)], rows)
    _mm(st, mm, [_mm_job(W["w2"], mid["w"], w, G_WDECAY, vec["w0"], None, scale),
                 _mm_job(W["a2"], mid["a"], a, G_SIGB, vec["a0"]),
                 _mm_job(W["v2"], mid["v"], v, G_VLERP, vec["v0"], vf), _mm_job(W["g2"], mid["g"], gate, G_STORE)], rows)
    _scan_op(st, rnn, r, w, k, v, a, gate, yw, bonus, yg, vec, seg, rows, c)
    if small:
        _mm(st, "rsv_gemm_skinny", [_mm_job(W["o"], yg, x, G_ADD)], rows)
    else:
        st.op("rsv_gemm_ex", yg.id, W["o"].w16, None, x.id, rows, c, c, G_ADD, NONE, NONE, NONE)
    st.out = [x.t, rnn.t, state.t]
    return st


def _scan_op(st, rnn, r, w, k, v, a, gate, yw, bonus, yg, vec, seg, rows, c):
    st.op("rsv_wkv7_seq_ragged_gate", rnn.id, r.id, w.id, k.id, v.id, a.id, vec["k_k"].id, vec["k_a"].id, vec["r_k"].id,
          vec["gn_w"].id, vec["gn_b"].id, gate.id, yw.id, bonus.id, yg.id, seg["start"].id, seg["len"].id,
          seg["slot"].id, seg["n"], rows, c // N, N, GN_EPS)


def _scan_inputs(case, g):
    c, rows, segs = case["c"], case["rows"], case["segs"]
    p = dict(k_k=g.normal(c, std=0.1, mean=0.85), k_a=g.uniform(c), r_k=g.normal(c, std=0.1),
             gn_w=g.normal(c, std=0.1, mean=1.0), gn_b=g.normal(c, std=0.1))
    x = dict(r=g.normal(rows, c), k=g.normal(rows, c), v=g.normal(rows, c),
             w=torch.exp(DECAY * torch.sigmoid(g.normal(rows, c, std=2.0, mean=-1.5))),
             a=torch.sigmoid(g.normal(rows, c)), gate=g.normal(rows, c, std=0.5))
    return p, x, g.normal(segs, c // N, N, N, std=0.1)


def _prepare_scan(case, g):
    c, rows = case["c"], case["rows"]
    p, x, s0 = _scan_inputs(case, g)
    st, seg = _State(), _chunk(case)
    vec, d, rnn = {n: _put(t) for n, t in p.items()}, {n: _put(t) for n, t in x.items()}, _put(s0)
    yw, bonus, yg = _f32(rows, c), _f32(rows, c // N), _f16(rows, c)
    _scan_op(st, rnn, d["r"], d["w"], d["k"], d["v"], d["a"], d["gate"], yw, bonus, yg, vec, seg, rows, c)
    st.out = [yg.t, rnn.t]
    return st


def _head_inputs(case, g):
    c, rows = case["c"], case["rows"]
    # a gamma of 3 gives logits of standard deviation 3, about as peaked as a trained model's
    return dict(x=g.normal(rows, c), ln_w=g.normal(c, std=0.3, mean=3.0 * math.sqrt(2560 / c)), ln_b=g.normal(c, std=0.1),
                head=g.matrix(VOCAB, c, case["weights"]))


def _prepare_head(case, g):
    c, rows = case["c"], case["rows"]
    p = _head_inputs(case, g)
    st = _State()
    x, lw, lb, head = _put(p["x"]), _put(p["ln_w"]), _put(p["ln_b"]), _Weight(p["head"], tiled=rows > 1)
    logits, tok = _f32(rows, VOCAB), _Dev((rows,), rsv.U32)
    if rows == 1:
        xn = _f32(1, c)
        st.op("rsv_norm", x.id, lw.id, lb.id, xn.id, c, 1, LN_EPS, 1)
        if head.i8:
            st.op("rsv_gemv_int8_plain", head.w8, xn.id, logits.id, VOCAB, c, 1)
        else:
            st.op("rsv_gemv_f16", head.w16, xn.id, logits.id, VOCAB, c, 1)
    else:
        xn = _f16(rows, c)
        st.op("rsv_ln_mix_f16", x.id, NONE, lw.id, lb.id, None, _ids(xn), 1, c, LN_EPS, rows)
        _mm(st, "rsv_gemm_skinny", [_mm_job(head, xn, logits, G_STORE)], rows)
    if case["pick"] == "argmax":
        st.op("rsv_argmax_batch", logits.id, tok.id, VOCAB, rows)
    else:
        temp, counter, sampler, hist = _f32(rows, VOCAB), _Dev((rows, VOCAB), rsv.U32), _f32(rows, 8), _Dev((rows,), rsv.U32)
        seeds = (ctypes.c_uint32 * rows)(*[1000 + 7 * q for q in range(rows)])
        top_k, top_p = (0, 0.9) if case["pick"] == "top_p" else (50, 1.0)
        st.op("rsv_store_sampler_async_batch", sampler.id, 0, 1.0, top_k, top_p, seeds, rows, 1.0, 0.0, 0.0, 0)
        st.op("rsv_sample_into_host_seeded_batch", logits.id, tok.id, VOCAB, temp.id, NONE, counter.id, sampler.id, hist.id, rows)
    st.out = [logits.t, tok.t]
    return st


# ---------------------------------------------------------------- whole calls
MODEL = dict(synth.THREE_B, n_layer=2)


def _model_tensors():
    """(key, kind, data) of the model file's tensors, on the GPU, the same ones each time: random weights in
    synth.py's layout, with its N(0, 0.02^2) matrices; kind is the safetensors type."""
    g = _Gen(1)
    for key, shape in synth.shapes(MODEL):
        if synth._is_norm(key):
            yield key, "F32", torch.full(shape, float(key.endswith("weight")), device="cuda")
        elif key.endswith(synth.LINEARS) or key == "head.weight":
            _, idx, sz = g.matrix(*shape, "int8")
            yield key + ".int8_idx", "U8", idx
            yield key + ".int8_sz", "U32", sz
        elif key == "emb.weight":
            yield key, "F16", g.normal(*shape, std=0.02).half()
        else:
            yield key, "F32", g.normal(*shape, std=0.02)


@functools.lru_cache(None)
def _model():
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "model.st")
        size = {"F32": 4, "F16": 2, "U8": 1, "U32": 4}
        w = synth._Writer(path, [(k, t, tuple(x.shape), x.numel() * size[t]) for k, t, x in _model_tensors()])
        for _, _, x in _model_tensors():
            w.write(x.cpu().numpy())
        w.close()
        return rsv.ModelBuilder(path).build()


class _Tokens:
    """infer_tokens of a conversation, on an instance of its own that shares the model's weights: the last logits
    and the state it leaves."""

    def __init__(self, case, g):
        self.bundle, self.tokens = _model().build_shared(), g.ints(case["rows"], VOCAB).cpu().numpy().astype(np.uint32)

    def run(self):
        logits = self.bundle.infer_tokens(self.tokens)
        return [logits, self.bundle.state_back()]


class _Prompts:
    """forward_seq_batch of several conversations: every prompt's last token and last logits."""

    def __init__(self, case, g):
        self.bundle, lens = _model(), _lens(case)
        flat = g.ints(case["rows"], VOCAB).cpu().numpy().astype(np.uint32)
        self.prompts = np.split(flat, np.cumsum(lens)[:-1])
        self.state = self.bundle.create_batch_state(len(lens))

    def run(self):
        seeds, logits = self.bundle.forward_seq_batch(self.state, self.prompts, want_logits=True)
        return [seeds, logits]

    def __del__(self):
        if hasattr(self, "state"):
            self.state.free()


def prepare(case, seed):
    g = _Gen(seed)
    _made.clear()
    made = {"ffn": _prepare_ffn, "ffn_prompt": _prepare_ffn_prompt, "tmix": _prepare_tmix,
            "tmix_prompt": _prepare_tmix_prompt, "scan": _prepare_scan, "head": _prepare_head,
            "model_tokens": _Tokens, "model_prompts": _Prompts}[case["kind"]](case, g)
    torch.cuda.synchronize()
    if isinstance(made, _State):
        made.keep.append(list(_made))
    _made.clear()
    return made


def run(state):
    return state.run()


# ---------------------------------------------------------------- work and tolerance
def _wbytes(m, k, weights):
    return m * k * (2 if weights == "fp16" else 1 + 4 / 128)


def work(case):
    kind, rows = case["kind"], case["rows"]
    if kind.startswith("model"):
        m, c, n = MODEL, MODEL["c"], case.get("segs", 1)
        lin = m["n_layer"] * (4 * c * c + 2 * c * m["ffn"])
        lora = m["n_layer"] * 2 * c * sum(_ranks(c))
        state = n * m["n_layer"] * (c * N + 2 * c) * 4
        wkv = m["n_layer"] * rows * c // N * 36864
        if kind == "model_tokens":  # every token reads the layers and the state; logits are asked for the last only
            return dict(bytes=rows * (lin * 33 / 32 + lora * 2 + 2 * state) + VOCAB * c * 33 / 32 + rows * c * 4 + VOCAB * 4,
                        flops=rows * 2 * (lin + lora) + 2 * VOCAB * c + wkv)
        return dict(bytes=lin * 33 / 32 + lora * 2 + VOCAB * c * 33 / 32 + 2 * state + rows * c * 4 + n * VOCAB * 4,
                    flops=rows * 2 * (lin + lora) + n * 2 * VOCAB * c + wkv)
    c, w = case["c"], case["weights"]
    if kind in ("ffn", "ffn_prompt"):
        out = (1 + _vslices(c) + 2 + 2) if kind == "ffn" and rows > 1 else 2  # slice sums in and out beside the rows
        return dict(bytes=2 * _wbytes(4 * c, c, w) + rows * c * 4 * (out + (2 if kind == "ffn" else 0)), flops=16 * rows * c * c)
    if kind == "head":
        return dict(bytes=_wbytes(VOCAB, c, w) + rows * (c + VOCAB) * 4, flops=2 * rows * VOCAB * c)
    segs = case.get("segs", rows)
    wkv = rows * (c // N) * 36864
    state = 2 * segs * c * N * 4
    if kind == "scan":
        return dict(bytes=rows * c * (6 * 4 + 2) + state, flops=wkv)
    lora = 2 * c * sum(_ranks(c))
    rowsio = rows * c * 4 * (5 if kind == "tmix" else 3) + 2 * segs * c * 4
    return dict(bytes=4 * _wbytes(c, c, w) + 2 * lora + state + rowsio, flops=rows * 2 * (4 * c * c + lora) + wkv)


def tolerance(case):
    """About four times the error against exact(): 32-bit sums at one token, 16-bit activations beyond."""
    kind, rows = case["kind"], case["rows"]
    if kind == "model_tokens":
        return dict(rel=1e-5)
    if rows == 1 and kind in ("ffn", "tmix", "head"):
        return dict(rel=1e-5)
    return dict(rel=3.5e-3 if kind == "tmix" else 2.5e-3 if kind == "model_prompts" else 1.6e-3)


# ---------------------------------------------------------------- the same in 64 bits
def _ln64(x, w, b, eps):
    mu = x.mean(-1, keepdim=True)
    d = x - mu
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps) * w + b


def _shift64(ln, prev, lens):
    """Each row's predecessor: the row before it in its segment, or the segment's carried row."""
    out, at = torch.empty_like(ln), 0
    for i, n in enumerate(lens):
        out[at] = prev[i]
        out[at + 1:at + n] = ln[at:at + n - 1]
        at += n
    return out, ln[np.cumsum(lens) - 1].clone()


def _wkv64(S, r, w, k, v, a, p, lens):
    """The WKV7 recurrence over packed segments; returns y = GroupNorm(S r) + bonus and the states."""
    rows, c = r.shape
    H = c // N
    kk = (k * p["k_k"]).view(rows, H, N)
    kk = kk / kk.norm(dim=2, keepdim=True).clamp_min(L2_EPS)
    kmod = (k * (1 + (a - 1) * p["k_a"])).view(rows, H, N)
    r, w, v, a = (t.reshape(rows, H, N) for t in (r, w, v, a))
    b = -kk * a
    y, start = torch.empty_like(r), torch.tensor(np.concatenate([[0], np.cumsum(lens)[:-1]]), device=r.device)
    n = torch.tensor(lens, device=r.device)
    S = S.clone()
    for t in range(max(lens)):
        live = torch.nonzero(n > t).view(-1)
        at, s = start[live] + t, S[live]
        sk = s @ kk[at][..., None]
        s = s * w[at][:, :, None, :] + sk * b[at][:, :, None, :] + v[at][..., None] * kmod[at][:, :, None, :]
        S[live] = s
        y[at] = (s @ r[at][..., None])[..., 0]
    yn = _ln64(y, p["gn_w"].view(H, N), p["gn_b"].view(H, N), GN_EPS)
    yn = yn + (r * kmod * p["r_k"].view(H, N)).sum(2, keepdim=True) * v
    return yn.reshape(rows, c), S


def _tmix64(p, x, prev, vf, S, lens):
    """One time-mix block: its output product (added to x by the caller), the states, and v."""
    D = {n: (_f64(t) if isinstance(t, tuple) else t.double()) for n, t in p.items()}
    ln = _ln64(x, D["ln_w"], D["ln_b"], LN_EPS)
    before, last = _shift64(ln, prev, lens)
    mix = {n: ln + D["x_" + n] * (before - ln) for n in "rwkvag"}
    r, k, v = (mix[n] @ D[n].T for n in "rkv")
    if vf is not None:
        v = v + torch.sigmoid(mix["v"] @ D["v1"].T @ D["v2"].T + D["v0"]) * (vf - v)
    w = torch.exp(DECAY * torch.sigmoid(torch.tanh(mix["w"] @ D["w1"].T) @ D["w2"].T + D["w0"]))
    a = torch.sigmoid(mix["a"] @ D["a1"].T @ D["a2"].T + D["a0"])
    gate = torch.sigmoid(mix["g"] @ D["g1"].T) @ D["g2"].T
    y, S = _wkv64(S, r, w, k, v, a, D, lens)
    return y * gate, D["o"], S, last, v


def _ffn64(p, x, prev, lens):
    D = {n: (_f64(t) if isinstance(t, tuple) else t.double()) for n, t in p.items()}
    ln = _ln64(x, D["ln_w"], D["ln_b"], LN_EPS)
    before, last = _shift64(ln, prev, lens)
    return torch.relu((ln + D["mix"] * (before - ln)) @ D["key"].T) ** 2, D["value"], last


def _slices64(x, w, n):
    """The products of the n equal k-slices of x w^T."""
    k = x.shape[1] // n
    return torch.stack([x[:, i * k:(i + 1) * k] @ w[:, i * k:(i + 1) * k].T for i in range(n)])


def _model64(tokens, lens):
    """The two-layer model over packed new conversations: the last logits of each, and the layers' states."""
    T = {}
    for key, kind, x in _model_tensors():
        if key.endswith("int8_idx"):
            T[key[:-9]] = ("int8", x)
        elif key.endswith("int8_sz"):
            T[key[:-8]] += (x,)
        else:
            T[key] = x
    vec = lambda name: T[name].reshape(-1)  # noqa: E731
    segs, c = len(lens), MODEL["c"]
    x = T["emb.weight"][torch.from_numpy(tokens.astype(np.int64)).cuda()].double()
    x = _ln64(x, vec("blocks.0.ln0.weight").double(), vec("blocks.0.ln0.bias").double(), LN_EPS)
    vf, states, zero = None, [], torch.zeros(segs, c, dtype=torch.float64, device="cuda")
    for i in range(MODEL["n_layer"]):
        b = "blocks.%d." % i
        p = {"x_" + n: vec(b + "att.x_" + n) for n in "rwkvag"}
        p.update({n: vec(b + "att." + n) for n in ("w0", "a0", "v0", "k_k", "k_a", "r_k")})
        p.update(ln_w=vec(b + "ln1.weight"), ln_b=vec(b + "ln1.bias"), gn_w=vec(b + "att.ln_x.weight"),
                 gn_b=vec(b + "att.ln_x.bias"), r=T[b + "att.receptance.weight"], k=T[b + "att.key.weight"],
                 v=T[b + "att.value.weight"], o=T[b + "att.output.weight"])
        for n in "wavg":  # the file holds [in, out]; the loader keeps fp16
            p[n + "1"], p[n + "2"] = (T[b + "att." + n + d].half().T for d in "12")
        S0 = torch.zeros(segs, c // N, N, N, dtype=torch.float64, device="cuda")
        y, o, S, tx, v = _tmix64(p, x, zero, vf, S0, lens)
        vf = v if vf is None else vf
        x = x + y @ o.T
        f = dict(ln_w=vec(b + "ln2.weight"), ln_b=vec(b + "ln2.bias"), mix=vec(b + "ffn.x_k"),
                 key=T[b + "ffn.key.weight"], value=T[b + "ffn.value.weight"])
        r2, value, cx = _ffn64(f, x, zero, lens)
        x = x + r2 @ value.T
        states += [tx, S.reshape(segs, -1), cx]
    last = np.cumsum(lens) - 1
    xn = _ln64(x[last], vec("ln_out.weight").double(), vec("ln_out.bias").double(), LN_EPS)
    return xn @ _f64(T["head.weight"]).T, torch.cat(states + [vf[last]], 1)


def exact(case, seed):
    g, kind, rows = _Gen(seed), case["kind"], case["rows"]
    if kind.startswith("model"):
        tokens = g.ints(rows, VOCAB).cpu().numpy()
        logits, state = _model64(tokens, _lens(case) if kind == "model_prompts" else [rows])
        return [logits[0].cpu(), state[0].cpu()] if kind == "model_tokens" else [None, logits.cpu()]
    c = case["c"]
    if kind == "ffn":
        p = _ffn_inputs(g, c, case["weights"])
        x, prev, part = g.normal(rows, c).double(), g.normal(rows, c).double(), g.normal(2, rows, c, std=0.3).double()
        if rows == 1:
            r2, value, last = _ffn64(p, x, prev, [1])
            return [x + r2 @ value.T, last]
        x = x + part.sum(0)
        r2, value, last = _ffn64(p, x, prev, [1] * rows)
        return [x, last, _slices64(r2, value, _vslices(c))]
    if kind == "ffn_prompt":
        p = _ffn_inputs(g, c, case["weights"])
        x, prev = g.normal(rows, c).double(), g.normal(1, c).double()
        r2, value, last = _ffn64(p, x, prev, [rows])
        return [x + r2 @ value.T, last]
    if kind in ("tmix", "tmix_prompt"):
        lens = [1] * rows if kind == "tmix" else _lens(case)
        p = _tmix_inputs(g, c, case["weights"])
        x, prev, vf = g.normal(rows, c).double(), g.normal(len(lens), c).double(), g.normal(rows, c).double()
        S = g.normal(len(lens), c // N, N, N, std=0.1).double()
        y, o, S, last, _ = _tmix64(p, x, prev, vf, S, lens)
        return [_slices64(y, o, 2) if kind == "tmix" and rows > 1 else x + y @ o.T, S, last]
    if kind == "scan":
        p, x, S = _scan_inputs(case, g)
        p, x = {n: t.double() for n, t in p.items()}, {n: t.double() for n, t in x.items()}
        y, S = _wkv64(S.double(), x["r"], x["w"], x["k"], x["v"], x["a"], p, _lens(case))
        return [y * x["gate"], S]
    p = _head_inputs(case, g)
    xn = _ln64(p["x"].double(), p["ln_w"].double(), p["ln_b"].double(), LN_EPS)
    return [xn @ _f64(p["head"]).T, None]
