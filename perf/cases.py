"""The work that programs on this framework run, as cases to time and compare.

Each case is one call, or the few calls of one block, through the C ABI
(include/krafla_hip.h) or the model API (include/krafla.h) as the Python
binding exposes them, at the sizes of the repository's own configurations
(stories15M, the 0.5B, 1B and 8B shapes, Gemma-like heads) or generic ones.
Buffers are torch tensors on the GPU; the library runs on its own stream.
"""
import ctypes as C
import math
import os
import random
import shutil
import sys
import tempfile
import weakref

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "isa-lm_amd"))   # run from the repository's root
import krafla as K  # noqa: E402

QK = 32
KV_TYPES = {"f32": K.ML_F32, "f16": K.ML_F16, "q8": K.ML_Q8_0}
EPS = 1e-5


def listed():
    return [
        # the smallest block of a token step: a 15M model's FFN (f32 scales)
        dict(name="ffn_token_15m", kind="ffn_token", dim=288, hidden=768, up="q8", down="q8", d16=False),
        # the isolated decode matvec of the benchmark (its Q4_0 large shape)
        dict(name="matvec_q4_14336x4096", kind="matvec", rows=14336, cols=4096, wtype="q4", d16=True),
        # the FFN of one decoded token, 8B shape
        dict(name="ffn_token_8b", kind="ffn_token", dim=4096, hidden=14336, up="q8", down="q8", d16=True),
        # the attention block of one decoded token: projections, cache row,
        # attention over the cache, output projection; 8B shape, F32 cache
        dict(name="attn_token_8b_f32", kind="attn_token", dim=4096, heads=32, kv_heads=8, head_dim=128, wtype="q8",
             pos=2111, kv="f32"),
        # the same at the end of a long context over a Q8 cache, 1B shape
        dict(name="attn_token_1b_q8", kind="attn_token", dim=2048, heads=32, kv_heads=8, head_dim=64, wtype="q4",
             pos=4050, kv="q8"),
        # a short prompt's product (a ragged handful of tokens, quantized first), 8B down projection
        dict(name="matmul_37_tokens", kind="matmul", rows=4096, cols=14336, wtype="q8", tokens=37),
        # the FFN of a whole prompt step, 8B shape
        dict(name="ffn_prompt_8b", kind="ffn_prompt", dim=4096, hidden=14336, up="q8", down="q8", tokens=2047),
        # the second step of a long prompt's attention, 1B shape
        dict(name="attn_prompt_1b_f32", kind="attn_prompt", heads=32, kv_heads=8, head_dim=64, pos0=2048,
             tokens=1951, window=0, softcap=0.0, kv="f32"),
        # sliding-window attention with soft-capped scores over 256-wide heads (Gemma)
        dict(name="attn_prompt_window_f16", kind="attn_prompt", heads=8, kv_heads=4, head_dim=256, pos0=1000,
             tokens=1021, window=1024, softcap=50.0, kv="f16"),
        # sixteen top-p draws over a 128k vocabulary (ml_run's default -p 0.9)
        dict(name="draw_top_p", kind="draw", vocab=128256, temperature=0.8, topp=0.9, topk=0, draws=16),
        # whole calls: a 15M model's short greedy run, and the 0.5B model's
        # 512-token prompt and the tokens after it
        dict(name="generate_15m", kind="generate", model="stories15m_q8", prompt=8, steps=136, kv="f32"),
        dict(name="generate_05b", kind="generate", model="qwen05b_mixed", prompt=512, steps=544, kv="f32"),
    ]


def _log(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["matvec", "ffn_token", "attn_token", "matmul", "ffn_prompt", "attn_prompt", "attn_prompt",
                       "draw", "generate"])
    if kind == "matvec":
        return dict(kind=kind, rows=_log(rng, 896, 14336), cols=_log(rng, 896, 14336, 32),
                    wtype=rng.choice(["q8", "q4"]), d16=rng.random() < 0.7)
    if kind == "ffn_token":
        return dict(kind=kind, dim=_log(rng, 288, 4096, 32), hidden=_log(rng, 768, 14336, 32),
                    up=rng.choice(["q8", "q4"]), down="q8", d16=rng.random() < 0.7)
    if kind in ("attn_token", "attn_prompt"):
        hd = rng.choice([48, 64, 64, 80, 96, 128, 128, 256])
        nkv = rng.choice([1, 2, 4, 8])
        heads = nkv * rng.choice([1, 2, 3, 4, 7] if kind == "attn_token" else [1, 2, 3, 4])
        if kind == "attn_token":
            if heads * hd % 32:
                heads *= 2
            return dict(kind=kind, dim=_log(rng, 288, 4096, 32), heads=heads, kv_heads=nkv, head_dim=hd,
                        wtype=rng.choice(["q8", "q4"]), pos=_log(rng, 8, 4090), kv=rng.choice(["f32", "f16", "q8"]))
        tokens = _log(rng, 16, 2047)
        windowed = rng.random() < 0.5
        return dict(kind=kind, heads=heads, kv_heads=nkv, head_dim=hd, pos0=rng.randrange(0, 2049), tokens=tokens,
                    window=_log(rng, 64, 2048) if windowed else 0,
                    softcap=50.0 if windowed and rng.random() < 0.3 else 0.0, kv=rng.choice(["f32", "f16", "q8"]))
    if kind == "matmul":
        return dict(kind=kind, rows=_log(rng, 288, 14336), cols=_log(rng, 288, 14336, 32),
                    wtype=rng.choice(["q8", "q4"]), tokens=_log(rng, 2, 2047))
    if kind == "ffn_prompt":
        return dict(kind=kind, dim=_log(rng, 512, 4096, 32), hidden=_log(rng, 2048, 14336, 32),
                    up=rng.choice(["q8", "q4"]), down="q8", tokens=_log(rng, 256, 2047))
    if kind == "draw":
        topk = rng.choice([0, 0, 0, 1, 40, 40, 200])
        return dict(kind=kind, vocab=_log(rng, 512, 151936), temperature=round(rng.uniform(0.5, 1.3), 2),
                    topp=rng.choice([1.0, 0.8, 0.9, 0.95]), topk=topk, draws=rng.randrange(4, 17))
    prompt = _log(rng, 2, 512)
    return dict(kind=kind, model="qwen05b_mixed", prompt=prompt, steps=prompt + _log(rng, 4, 31),
                kv=rng.choice(["f32", "f16", "q8"]))


# ---- inputs ----

def _gen(seed, salt=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000003 + salt)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


class Mat:
    """A quantized weight matrix as the .mlb format lays it out (blocks of 32
    along the columns; Q4: byte j holds elements j and j + 16), of N(0,
    0.02^2) values by the format's writer rules, with its descriptor."""

    def __init__(self, g, rows, cols, wtype, d16):
        w = (_randn(g, rows, cols) * 0.02).view(rows, cols // QK, QK)
        if wtype == "q8":
            d = w.abs().amax(2) / 127
            self.d = d.to(torch.float16) if d16 else d
            ds = self.d.float().unsqueeze(2)
            self.n = torch.clamp(torch.round(w / torch.where(ds > 0, ds, torch.ones_like(ds))), -127, 127).to(
                torch.int8)
            self.q = self.n.contiguous()
        else:
            at = w.abs().argmax(2, keepdim=True)
            d = torch.gather(w, 2, at).squeeze(2) / -8
            self.d = d.to(torch.float16) if d16 else d
            ds = self.d.float().unsqueeze(2)
            n = torch.clamp(torch.round(w / torch.where(ds != 0, ds, torch.ones_like(ds))) + 8, 0, 15).to(torch.uint8)
            self.n = n.to(torch.int8) - 8
            self.q = (n[:, :, :16] | n[:, :, 16:] << 4).contiguous()
        self.n = None   # exact() takes the values from q
        self.rows, self.cols, self.wtype = rows, cols, wtype
        self.m = K.KrhMat(self.q.data_ptr(), self.d.data_ptr(), rows, cols,
                          K.ML_Q8_0 if wtype == "q8" else K.ML_Q4_0, int(d16))
        self.ref = C.byref(self.m)

    def exact(self):
        if self.wtype == "q8":
            n = self.q.double()
        else:
            n = torch.cat([self.q & 15, self.q >> 4], 2).double() - 8
        return (n * self.d.double().unsqueeze(2)).view(self.rows, self.cols)


def _rope(max_seq, hd, theta=5e5):
    inv = theta ** (-2.0 * torch.arange(hd // 2, dtype=torch.float64) / hd)
    ang = torch.arange(max_seq, dtype=torch.float64).unsqueeze(1) * inv
    return ang.cos().float().cuda().contiguous(), ang.sin().float().cuda().contiguous()


def _quant_rows(x):
    """int8 rows and one scale a row (the Q8 cache's rule), x [..., hd]"""
    m = x.abs().amax(-1, keepdim=True)
    q = torch.trunc(x * (127 / m) + torch.copysign(torch.full_like(x, 0.5), x)).clamp(-127, 127)
    return q.to(torch.int8).contiguous(), (m / 127).squeeze(-1).contiguous()


def _cache(g, kv, rows, nkv, hd):
    """one layer's cache of `rows` positions with its ml_kv_layer view"""
    k, v = _randn(g, rows, nkv, hd), _randn(g, rows, nkv, hd)
    s = {}
    view = K.MlKvLayer()
    if kv == "f32":
        s["k"], s["v"] = k, v
        view.k, view.v = k.data_ptr(), v.data_ptr()
    elif kv == "f16":
        s["k"], s["v"] = k.half(), v.half()
        view.kh, view.vh = s["k"].data_ptr(), s["v"].data_ptr()
    else:
        s["k"], s["kd"] = _quant_rows(k)
        s["v"], s["vd"] = _quant_rows(v)
        view.kq, view.vq, view.kd, view.vd = (s[n].data_ptr() for n in ("k", "v", "kd", "vd"))
    s["view"] = view
    return s


def _cache_exact(s, kv):
    k, v = s["k"].double(), s["v"].double()
    if kv == "q8":
        k, v = k * s["kd"].double().unsqueeze(-1), v * s["vd"].double().unsqueeze(-1)
    return k, v


def _f32(*shape):
    return torch.zeros(*shape, device="cuda", dtype=torch.float32)


def _i8(*shape):
    return torch.zeros(*shape, device="cuda", dtype=torch.int8)


def _ldx(t):
    return (t + 127) // 128 * 128


def _close(model, state, path):
    if state is not None:
        state.close()
    if model is not None:
        model.close()
    shutil.rmtree(path, ignore_errors=True)


class Run:
    """a loaded model with its decoding state; both go with this object"""

    def __init__(self, case, seed):
        spec = dict(K.CONFIGS[case["model"]], seed=seed + 11, device=1)
        d = tempfile.mkdtemp(prefix="krcase_", dir="/dev/shm" if os.path.isdir("/dev/shm") else None)
        path = os.path.join(d, "m.mlb")
        self.model = self.state = None
        try:
            K.gen_mlb(path, **spec)
            self.model = K.Model(path)
            self.state = K.State(self.model, KV_TYPES[case["kv"]])
        finally:
            self.end = weakref.finalize(self, _close, self.model, self.state, d)
            if os.path.exists(path):
                os.unlink(path)


def prepare(case, seed):
    K.init_device()
    kind = case["kind"]
    g = _gen(seed)
    s = dict(case)
    if kind == "matvec":
        s["W"] = Mat(g, case["rows"], case["cols"], case["wtype"], case["d16"])
        s["x"], s["y"] = _randn(g, case["cols"]), _f32(case["rows"])
    elif kind == "ffn_token":
        d, h = case["dim"], case["hidden"]
        s["w1"], s["w3"] = Mat(g, h, d, case["up"], case["d16"]), Mat(g, h, d, case["up"], case["d16"])
        s["w2"] = Mat(g, d, h, case["down"], case["d16"])
        s["x"], s["nw"] = _randn(g, d), 1 + 0.01 * _randn(g, d)
        s["h"], s["y"] = _f32(h), _f32(d)
    elif kind == "attn_token":
        d, nh, nkv, hd, pos = case["dim"], case["heads"], case["kv_heads"], case["head_dim"], case["pos"]
        ms = s["max_seq"] = 4096
        s["wq"], s["wk"] = Mat(g, nh * hd, d, case["wtype"], True), Mat(g, nkv * hd, d, case["wtype"], True)
        s["wv"], s["wo"] = Mat(g, nkv * hd, d, "q8", True), Mat(g, d, nh * hd, "q8", True)
        s["x"], s["nw"] = _randn(g, d), 1 + 0.01 * _randn(g, d)
        s["cos"], s["sin"] = _rope(ms, hd)
        s["cache"] = _cache(g, case["kv"], ms, nkv, hd)
        s["q"], s["ao"], s["y"], s["att"] = _f32(nh * hd), _f32(nh * hd), _f32(d), _f32(nh, ms)
        s["ks"], s["vs"] = _f32(nkv * hd), _f32(nkv * hd)
        s["pos_dev"] = torch.tensor([pos], dtype=torch.int32, device="cuda")
    elif kind == "matmul":
        T, r, c = case["tokens"], case["rows"], case["cols"]
        L = _ldx(T)
        s["W"] = Mat(g, r, c, case["wtype"], True)
        s["xq"], s["xd"], s["y"] = _i8(L, c), _f32(c // QK, L), _f32(T, r)
        s["x"] = _randn(g, T, c)
    elif kind == "ffn_prompt":
        T, d, h = case["tokens"], case["dim"], case["hidden"]
        L = _ldx(T)
        s["w1"], s["w3"] = Mat(g, h, d, case["up"], True), Mat(g, h, d, case["up"], True)
        s["w2"] = Mat(g, d, h, case["down"], True)
        s["x"], s["nw"] = _randn(g, T, d), 1 + 0.01 * _randn(g, d)
        s["xq"], s["xd"] = _i8(L, d), _f32(d // QK, L)
        s["hq"], s["hd"], s["y"] = _i8(L, h), _f32(h // QK, L), _f32(T, d)
    elif kind == "attn_prompt":
        nh, nkv, hd, T = case["heads"], case["kv_heads"], case["head_dim"], case["tokens"]
        ms = s["max_seq"] = 4096
        s["cache"] = _cache(g, case["kv"], ms, nkv, hd)
        s["cache"]["view"].window = case["window"]
        s["q"], s["ao"], s["att"] = _randn(g, T, nh * hd), _f32(T, nh * hd), _f32(T, nh, ms)
        s["pos_dev"] = torch.tensor([case["pos0"]], dtype=torch.int32, device="cuda")
    elif kind == "draw":
        # logits of a trained model's spread: most of the mass on a few hundred ids
        n, v = case["draws"], case["vocab"]
        s["rows"] = _randn(g, n, v) * 2.5
        s["logits"] = _f32(n, v)
        s["ids"] = torch.zeros(n + 1, dtype=torch.int32, device="cuda")
        s["tok"], s["at"] = (torch.zeros(1, dtype=torch.int32, device="cuda") for _ in range(2))
        s["opts"] = K.sampler_opts(temperature=case["temperature"], topp=case["topp"], topk=case["topk"],
                                   seed=seed + 1)
    else:
        s["run"] = Run(case, seed)
        s["tokens"] = np.random.RandomState(seed).randint(1, s["run"].model.cfg.vocab, case["prompt"]).astype(
            np.int32)
    torch.cuda.synchronize()
    return s


def run(s):
    kind, h = s["kind"], K.hip
    if kind == "matvec":
        h.krh_matvec_f(s["y"].data_ptr(), s["W"].ref, s["x"].data_ptr(), 0)
        return s["y"]
    if kind == "ffn_token":
        h.krh_rmsnorm_matvec_swiglu(s["h"].data_ptr(), s["w1"].ref, s["w3"].ref, s["x"].data_ptr(),
                                    s["nw"].data_ptr(), EPS)
        h.krh_matvec_f(s["y"].data_ptr(), s["w2"].ref, s["h"].data_ptr(), 0)
        return {"h": s["h"], "y": s["y"]}
    if kind == "attn_token":
        return _run_attn_token(s)
    if kind == "matmul":
        T, L = s["tokens"], _ldx(s["tokens"])
        h.krh_quantize_q8_t(s["xq"].data_ptr(), s["xd"].data_ptr(), L, s["x"].data_ptr(), s["cols"], T)
        h.krh_matmul(s["y"].data_ptr(), s["rows"], s["W"].ref, s["xq"].data_ptr(), s["xd"].data_ptr(), L, T, 0)
        return s["y"]
    if kind == "ffn_prompt":
        T, d, hid = s["tokens"], s["dim"], s["hidden"]
        L = _ldx(T)
        h.krh_rmsnorm_q8_t(s["xq"].data_ptr(), s["xd"].data_ptr(), L, None, s["x"].data_ptr(), s["nw"].data_ptr(), d,
                           EPS, T)
        h.krh_matmul_swiglu(s["hq"].data_ptr(), s["hd"].data_ptr(), s["w1"].ref, s["w3"].ref, s["xq"].data_ptr(),
                            s["xd"].data_ptr(), L, T)
        h.krh_matmul(s["y"].data_ptr(), d, s["w2"].ref, s["hq"].data_ptr(), s["hd"].data_ptr(), L, T, 0)
        return {"hd": s["hd"][:, :T], "y": s["y"]}
    if kind == "attn_prompt":
        hd, T = s["head_dim"], s["tokens"]
        args = (s["ao"].data_ptr(), s["att"].data_ptr(), s["q"].data_ptr(), C.byref(s["cache"]["view"]), s["heads"],
                s["kv_heads"], hd, s["max_seq"], hd ** -0.5, s["pos_dev"].data_ptr(), T, s["pos0"] + T - 1)
        if s["softcap"] > 0:
            h.krh_attention_kv_softcap(*args, s["softcap"])
        else:
            h.krh_attention_kv(*args)
        return s["ao"]
    if kind == "draw":
        v = s["vocab"]
        h.krh_copy_d2d_async(s["logits"].data_ptr(), s["rows"].data_ptr(), s["rows"].nbytes)
        h.krh_set_int(s["at"].data_ptr(), 0)
        smp = K.Sampler(v, s["opts"])
        for i in range(s["draws"]):
            smp.sample(s["tok"].data_ptr(), s["logits"].data_ptr() + 4 * v * i, v, s["at"].data_ptr(),
                       s["ids"].data_ptr())
        smp.close()
        return {"ids": s["ids"][1:], "last": s["tok"]}
    st = s["run"].state
    ids, _, _ = st.generate(s["tokens"], s["steps"])
    return {"ids": ids, "logits": st.buffer("logits", np.float32, s["run"].model.cfg.vocab)}


def _run_attn_token(s):
    h, kv = K.hip, s["kv"]
    c, hd, nkv, pos = s["cache"], s["head_dim"], s["kv_heads"], s["pos"]
    p = s["pos_dev"].data_ptr()
    kc, vc = c["k"].data_ptr(), c["v"].data_ptr()
    tail = (s["wq"].ref, s["wk"].ref, s["wv"].ref, None, None, None, s["x"].data_ptr(), s["nw"].data_ptr(), EPS,
            s["cos"].data_ptr(), s["sin"].data_ptr(), hd, p)
    q, ao, att, scale = s["q"].data_ptr(), s["ao"].data_ptr(), s["att"].data_ptr(), hd ** -0.5
    if kv == "f32":
        h.krh_rmsnorm_matvec_qkv(q, kc, vc, *tail)
        h.krh_attention(ao, None, None, att, q, kc, vc, s["heads"], nkv, hd, s["max_seq"], 0, scale, p)
    elif kv == "f16":
        h.krh_rmsnorm_matvec_qkv_f16(q, kc, vc, *tail)
        h.krh_attention_kv(ao, att, q, C.byref(c["view"]), s["heads"], nkv, hd, s["max_seq"], scale, p, 1,
                           s["max_seq"] - 1)
    else:
        h.krh_rmsnorm_matvec_qkv_stage(q, s["ks"].data_ptr(), s["vs"].data_ptr(), *tail)
        h.krh_attention_q8_store(ao, att, q, C.byref(c["view"]), s["ks"].data_ptr(), s["vs"].data_ptr(), s["heads"],
                                 nkv, hd, s["max_seq"], scale, p)
    h.krh_matvec_f(s["y"].data_ptr(), s["wo"].ref, ao, 0)
    return {"q": s["q"], "k": c["k"][pos], "v": c["v"][pos], "ao": s["ao"], "y": s["y"]}


# ---- what a pass cannot do without ----

def _wbytes(rows, cols, wtype, sb=2):
    n = rows * cols
    return (n if wtype == "q8" else n // 2) + n // QK * sb


def _kvbytes(kv, nkv, hd):
    """one position's K and V"""
    return nkv * (hd * {"f32": 8, "f16": 4, "q8": 2}[kv] + (8 if kv == "q8" else 0))


def _attended(pos0, tokens, window):
    """(score pairs, distinct positions read) of tokens at pos0.."""
    pairs = sum(min(pos0 + t + 1, window) if window else pos0 + t + 1 for t in range(tokens))
    first = max(0, pos0 - window + 1) if window else 0
    return pairs, pos0 + tokens - first


def _model_work(case):
    c = K.CONFIGS[case["model"]]
    L, d, hid, V = c["n_layers"], c["dim"], c["hidden_dim"], c["vocab"]
    hd = d // c["n_heads"]
    kvd = c["n_kv_heads"] * hd
    q4 = c["wtype"] == K.ML_Q4_0
    a, b = ("q4" if q4 else "q8"), "q8"
    sb = 2 if c["scale_f16"] else 4
    layer = (_wbytes(d, d, a, sb) + _wbytes(kvd, d, a, sb) + _wbytes(kvd, d, b, sb) + _wbytes(d, d, b, sb)
             + 2 * _wbytes(hid, d, a, sb) + _wbytes(d, hid, b, sb))
    per = 2 * (2 * d * d + 2 * kvd * d + 3 * hid * d)
    np_, n = case["prompt"], case["steps"] - (case["prompt"] - 1)
    kvb = _kvbytes(case["kv"], c["n_kv_heads"], hd)
    ctx = sum(np_ + i for i in range(n))
    pairs = _attended(0, case["steps"], 0)[0]
    return dict(bytes=(n + (np_ > 1)) * L * layer + n * _wbytes(V, d, a, sb) + L * kvb * (ctx + case["steps"]),
                flops=case["steps"] * L * per + n * 2 * V * d + 4 * L * pairs * d)


def work(case):
    kind = case["kind"]
    if kind == "matvec":
        r, c = case["rows"], case["cols"]
        return dict(bytes=_wbytes(r, c, case["wtype"], 2 if case["d16"] else 4) + 4 * (r + c), flops=2 * r * c)
    if kind == "ffn_token":
        d, h = case["dim"], case["hidden"]
        sb = 2 if case["d16"] else 4
        return dict(bytes=2 * _wbytes(h, d, case["up"], sb) + _wbytes(d, h, case["down"], sb) + 4 * (3 * d + h),
                    flops=6 * d * h)
    if kind == "attn_token":
        d, nh, nkv, hd, n = case["dim"], case["heads"], case["kv_heads"], case["head_dim"], case["pos"] + 1
        w = (_wbytes(nh * hd, d, case["wtype"]) + _wbytes(nkv * hd, d, case["wtype"]) + _wbytes(nkv * hd, d, "q8")
             + _wbytes(d, nh * hd, "q8"))
        return dict(bytes=w + n * _kvbytes(case["kv"], nkv, hd) + 4 * (3 * d + 2 * nh * hd),
                    flops=2 * d * hd * (2 * nh + 2 * nkv) + 4 * nh * hd * n)
    if kind == "matmul":
        r, c, T = case["rows"], case["cols"], case["tokens"]
        return dict(bytes=_wbytes(r, c, case["wtype"]) + 4 * T * (c + r), flops=2 * r * c * T)
    if kind == "ffn_prompt":
        d, h, T = case["dim"], case["hidden"], case["tokens"]
        return dict(bytes=2 * _wbytes(h, d, case["up"]) + _wbytes(d, h, case["down"]) + T * 8 * d, flops=6 * d * h * T)
    if kind == "attn_prompt":
        nh, nkv, hd, T = case["heads"], case["kv_heads"], case["head_dim"], case["tokens"]
        pairs, rows = _attended(case["pos0"], T, case["window"])
        return dict(bytes=rows * _kvbytes(case["kv"], nkv, hd) + 8 * T * nh * hd, flops=4 * pairs * nh * hd)
    if kind == "draw":
        return dict(bytes=case["draws"] * case["vocab"] * 8, flops=case["draws"] * case["vocab"] * 4)
    return _model_work(case)


def tolerance(case):
    # 32-bit sums are within 2.1e-7 (products) and 1.3e-6 (attention) of 64
    # bits. Where activations are quantized to 8 bits inside the block, a last
    # bit decides a few of those roundings: 1e-4 over a product's tokens,
    # 2.3e-4 over a prompt's FFN, one element of 4096 (4e-4) for one token.
    return {"matvec": {"rel": 1e-5}, "matmul": {"rel": 4e-4}, "attn_prompt": {"rel": 1e-5}, "draw": "exact",
            "generate": {"rel": 1e-3, "differ": 0.01}}.get(case["kind"], {"rel": 1e-3})


# ---- the same in 64 bits ----

def _q8_exact(x):
    """the values of x's Q8_0 blocks"""
    b = x.reshape(*x.shape[:-1], x.shape[-1] // QK, QK)
    m = b.abs().amax(-1, keepdim=True)
    q = torch.trunc(b * (127 / m) + torch.copysign(torch.full_like(b, 0.5), b)).clamp(-127, 127)
    return (q * (m / 127)).reshape(x.shape)


def _norm_exact(x, w):
    x = x.double()
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rotate(x, c, s):
    """pairs (2i, 2i + 1) of each head by row c, s"""
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * c - b * s, b * c + a * s], -1).reshape(x.shape)


def _ffn_exact(s):
    a = _q8_exact(_norm_exact(s["x"], s["nw"]))
    g, u = a @ s["w1"].exact().t(), a @ s["w3"].exact().t()
    h = g / (1 + torch.exp(-g)) * u
    return h, _q8_exact(h) @ s["w2"].exact().t()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("draw", "generate"):
        return None
    s = prepare(case, seed)
    if kind == "matvec":
        return s["W"].exact() @ _q8_exact(s["x"].double())
    if kind == "ffn_token":
        h, y = _ffn_exact(s)
        return {"h": h, "y": y}
    if kind == "matmul":
        return _q8_exact(s["x"].double()) @ s["W"].exact().t()
    if kind == "ffn_prompt":
        h, y = _ffn_exact(s)
        m = h.view(h.shape[0], -1, QK).abs().amax(-1) / 127
        return {"hd": m.t().contiguous(), "y": y}
    nh, nkv, hd = case["heads"], case["kv_heads"], case["head_dim"]
    k, v = _cache_exact(s["cache"], case["kv"])
    if kind == "attn_prompt":
        ao = []
        q = s["q"].double().view(-1, nh, hd)
        for t0 in range(0, case["tokens"], 256):
            ao.append(_attend(q[t0:t0 + 256], k, v, case["pos0"] + t0, case["window"], case["softcap"], case["kv"]))
        return torch.cat(ao)
    a, p = _q8_exact(_norm_exact(s["x"], s["nw"])), case["pos"]
    c, sn = s["cos"][p].double(), s["sin"][p].double()
    q = _rotate((s["wq"].exact() @ a).view(nh, hd), c, sn)
    kn = _rotate((s["wk"].exact() @ a).view(nkv, hd), c, sn)
    vn = (s["wv"].exact() @ a).view(nkv, hd)
    if case["kv"] == "f16":
        kn, vn = kn.half().double(), vn.half().double()
    if case["kv"] == "q8":
        (kq, kd), (vq, vd) = _quant_rows(kn), _quant_rows(vn)
        kn, vn = kq.double() * kd.unsqueeze(-1), vq.double() * vd.unsqueeze(-1)
    k[p], v[p] = kn, vn
    ao = _attend(q.view(1, nh, hd), k, v, p, 0, 0.0, case["kv"]).view(-1)
    whole = case["kv"] == "q8"
    return {"q": q.reshape(-1), "k": None if whole else kn, "v": None if whole else vn, "ao": ao,
            "y": s["wo"].exact() @ _q8_exact(ao)}


def _attend(q, k, v, pos0, window, softcap, kv):
    T, nh, hd = q.shape
    nkv = k.shape[1]
    n = pos0 + T
    if kv == "q8":   # each query head quantized with one scale
        m = q.abs().amax(-1, keepdim=True)
        q = torch.trunc(q * (127 / m) + torch.copysign(torch.full_like(q, 0.5), q)) * (m / 127)
    q = q.view(T, nkv, nh // nkv, hd).permute(1, 2, 0, 3).reshape(nkv, -1, hd)
    sc = torch.matmul(q, k[:n].permute(1, 2, 0).contiguous()) * hd ** -0.5
    if softcap > 0:
        sc = softcap * torch.tanh(sc / softcap)
    at = torch.arange(n, device=q.device)
    own = pos0 + torch.arange(T, device=q.device).unsqueeze(1)
    ok = at <= own
    if window:
        ok &= at > own - window
    sc = sc.view(nkv, nh // nkv, T, n).masked_fill(~ok, -math.inf).softmax(-1).view(nkv, -1, n)
    o = torch.matmul(sc, v[:n].permute(1, 0, 2).contiguous())
    return o.view(nkv, nh // nkv, T, hd).permute(2, 0, 1, 3).reshape(T, nh * hd)


if __name__ == "__main__":
    for seed in range(3):
        print(draw(random.Random(seed)))
