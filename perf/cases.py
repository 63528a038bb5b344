"""The work a program gives this backend, as cases that can be timed and compared.

Three ways in are covered, each through the calls a program makes (common_amd.hardware.HipContext and
common_amd.qwen3.Qwen3):

* stand-alone operators on device buffers: decode attention, a projection (dense), the SwiGLU hidden
  layer, the prompt-row products (gemm_bf16, gemm_f32) and token sampling;
* prompts: reset, set_prompt, prefill, with the last row's logits;
* generation: a prompt, then greedy tokens, with the logits of the last step.

A program holds one context, its buffers and one model per checkpoint, and feeds the model one prompt
after another: the context and the latest model are therefore kept in this module, weights are the
model's own (they do not follow the seed), and a state of a model case is a prompt.

Model weights are N(0, 0.02) as in common_amd.synthetic, with the two projections that write the
residual stream scaled by 1/sqrt(2 layers) and a wider embedding.  The tied head then prefers the last
token by a wide margin, so the greedy tokens of a generation do not hang on roundings.
"""
import math

import numpy as np
import torch

from common_amd import config as C
from common_amd import hardware as hw
from common_amd.qwen3 import Qwen3

# dim, FFN width, query heads, KV heads, head size
SHAPES = {
    "tiny": (256, 768, 4, 2, 64),          # C1
    "110M": (768, 2048, 12, 12, 64),       # the stories110M checkpoint's
    "0.6B": (1024, 3072, 16, 8, 128),      # C3
    "1.7B": (2048, 6144, 16, 8, 128),      # C4
    "4B": (2560, 9728, 32, 8, 128),        # C5
}
THETA = 1_000_000.0
EPS = 1e-6
EMBED_STD = 0.25


def listed():
    return [
        # one decode step's attention of a small model early in its context: launch latency
        {"name": "attention-short", "op": "attention", "heads": 4, "kv_heads": 2, "head_size": 64, "max_seq": 48,
         "pos": 20, "per_head": False},
        # the decode attention op at 4096 cached rows (C2)
        {"name": "attention-4k", "op": "attention", "heads": 16, "kv_heads": 8, "head_size": 128, "max_seq": 4097,
         "pos": 4096, "per_head": False},
        # long context with four query heads per KV head, at a row in the middle of a larger cache
        {"name": "attention-30k", "op": "attention", "heads": 32, "kv_heads": 8, "head_size": 128, "max_seq": 32768,
         "pos": 30010, "per_head": True},
        # the vocabulary projection of the 0.6B shape with its RMSNorm, fp32, one sequence
        {"name": "head-f32", "op": "dense", "rows": 151936, "cols": 1024, "batch": 1, "bf16": False, "norm": True,
         "bias": False},
        # the FFN hidden layer of the 4B shape for eight sequences
        {"name": "ffn-bf16-b8", "op": "swiglu", "rows": 9728, "cols": 2560, "batch": 8, "bf16": True, "norm": True},
        # prompt rows: the gate/up product of the 1.7B shape over a 2048-token prompt (C4)
        {"name": "gemm-bf16-gate-up", "op": "gemm_bf16", "m": 2048, "n": 6144, "k": 2048, "swiglu": True,
         "bias": False},
        # prompt rows in fp32: the QKV product of the 0.6B shape over a ragged prompt
        {"name": "gemm-f32-qkv", "op": "gemm_f32", "m": 1021, "n": 4096, "k": 1024, "swiglu": False, "bias": True},
        # nucleus sampling of eight sequences over the full vocabulary
        {"name": "sample-top-p-b8", "op": "sample", "rows": 8, "n": 151936, "mode": hw.SAMPLE_TOKEN,
         "temperature": 0.8, "top_p": 0.9},
        # fp32 prompt of the 0.6B shape (odd length), four layers, vocabulary in proportion
        {"name": "prompt-f32", "op": "prompt", "shape": "0.6B", "layers": 4, "vocab": 21696, "bf16": False,
         "kv16": False, "per_head": False, "bias": False, "batch": 1, "prompt": 1531},
        # bf16 prompt of the 1.7B shape (C4's length), four layers, vocabulary in proportion
        {"name": "prompt-bf16", "op": "prompt", "shape": "1.7B", "layers": 4, "vocab": 21696, "bf16": True,
         "kv16": False, "per_head": True, "bias": False, "batch": 1, "prompt": 2048},
        # C3: the whole 0.6B shape in fp32, one sequence, 128-token prompt, greedy tokens
        {"name": "generate-f32-b1", "op": "generate", "shape": "0.6B", "layers": 28, "vocab": 151936, "bf16": False,
         "kv16": False, "per_head": False, "bias": False, "batch": 1, "prompt": 128, "steps": 32},
        # eight sequences of the 4B shape, four layers: a 1024-token prompt each, then greedy tokens
        {"name": "generate-bf16-b8", "op": "generate", "shape": "4B", "layers": 4, "vocab": 16896, "bf16": True,
         "kv16": False, "per_head": True, "bias": False, "batch": 8, "prompt": 1024, "steps": 32},
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["attention", "attention", "dense", "swiglu", "gemm_bf16", "gemm_f32", "sample", "prompt",
                     "prompt", "generate"])
    if op == "attention":
        kv = rng.choice([2, 4, 8, 12])
        max_seq = _log(rng, 32, 32768)
        return {"op": op, "heads": kv * rng.choice([1, 2, 4]), "kv_heads": kv, "head_size": rng.choice([64, 128]),
                "max_seq": max_seq, "pos": rng.randrange(max_seq // 2, max_seq), "per_head": rng.random() < 0.5}
    if op == "dense":
        return {"op": op, "rows": _log(rng, 512, 32000), "cols": 8 * _log(rng, 32, 1216), "batch": rng.randint(1, 8),
                "bf16": rng.random() < 0.5, "norm": rng.random() < 0.5, "bias": rng.random() < 0.3}
    if op == "swiglu":
        return {"op": op, "rows": _log(rng, 512, 9728), "cols": 8 * _log(rng, 32, 320), "batch": rng.randint(1, 8),
                "bf16": rng.random() < 0.5, "norm": rng.random() < 0.5}
    if op == "gemm_bf16":
        swiglu = rng.random() < 0.5
        return {"op": op, "m": _log(rng, 16, 4096), "n": 128 * _log(rng, 4, 64), "k": 64 * _log(rng, 4, 64),
                "swiglu": swiglu, "bias": not swiglu and rng.random() < 0.5}
    if op == "gemm_f32":
        swiglu = rng.random() < 0.5
        return {"op": op, "m": _log(rng, 16, 2048), "n": 64 * _log(rng, 8, 64), "k": 32 * _log(rng, 8, 96),
                "swiglu": swiglu, "bias": not swiglu and rng.random() < 0.5}
    if op == "sample":
        return {"op": op, "rows": rng.randint(1, 8), "n": _log(rng, 1000, 151936),
                "mode": rng.choice([hw.SAMPLE_TOKEN, hw.SAMPLE_TOKEN, hw.SAMPLE_MODEL]),
                "temperature": round(rng.uniform(0.5, 1.2), 2), "top_p": round(rng.uniform(0.8, 1.0), 2)}
    bf16 = rng.random() < 0.6
    shape = rng.choice(["110M", "0.6B", "1.7B", "4B"] if bf16 else ["tiny", "110M", "0.6B", "1.7B"])
    case = {"op": op, "shape": shape, "layers": rng.randint(2, 3), "vocab": 8 * _log(rng, 500, 4000), "bf16": bf16,
            "kv16": bf16 and rng.random() < 0.4, "per_head": rng.random() < 0.5, "bias": rng.random() < 0.2}
    if op == "prompt":
        case["batch"] = rng.choice([1, 1, 1, 2, 4])
        case["prompt"] = _log(rng, 16, 2048 // case["batch"])
    else:
        case["batch"] = rng.choice([1, 1, 2, 3, 5, 8])
        case["prompt"] = _log(rng, 16, 2048 // case["batch"])
        case["steps"] = rng.randint(8, 48)
    return case


# ---- device memory ---------------------------------------------------------------------------------

_kept = {}


def _context():
    if "ctx" not in _kept:
        _kept["ctx"] = hw.HipContext()
    return _kept["ctx"]


class _View:
    """A device buffer's bytes for torch.as_tensor; the tensors made from it hold it, and the buffer is
    freed with the last of them."""

    def __init__(self, buf, shape, kind):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": shape, "typestr": kind, "data": (buf.ptr, False), "version": 2}

    def __del__(self):
        self.buf.free()


class _Buffers:
    """Device buffers of the context's memory provider, by name, with torch views to fill and return them."""

    KINDS = {torch.float32: "<f4", torch.int32: "<i4", torch.int64: "<i8", torch.bfloat16: "<i2"}

    def __init__(self):
        self.ctx = _context()
        self.buf, self.view = {}, {}

    def add(self, name, t):
        """A buffer holding the tensor's values."""
        b = self.ctx.allocate(max(t.numel() * t.element_size(), 16))
        v = torch.as_tensor(_View(b, tuple(t.shape), self.KINDS[t.dtype]), device="cuda")
        v = v.view(torch.bfloat16) if t.dtype == torch.bfloat16 else v
        assert v.data_ptr() == b.ptr
        v.copy_(t)
        self.buf[name], self.view[name] = b, v

    def __getitem__(self, name):
        return self.buf.get(name)

    def ready(self):
        """The fills ran on torch's stream: they end here, before the context's stream reads."""
        torch.cuda.synchronize()
        return self


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape, std=1.0, mean=0.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).mul_(std).add_(mean)


# ---- operator inputs (the same for prepare and exact) ------------------------------------------------

def _inputs(case, seed):
    """The operator's inputs by name, on the GPU."""
    g, op, t = _gen(seed), case["op"], {}
    if op == "attention":
        H, KV, D, S = case["heads"], case["kv_heads"], case["head_size"], case["max_seq"]
        t["q"], t["k"], t["v"] = _randn(g, H * D), _randn(g, KV * D), _randn(g, KV * D, std=0.6)
        t["q_norm"], t["k_norm"] = _randn(g, H * D, std=0.02, mean=1.0), _randn(g, KV * D, std=0.02, mean=1.0)
        t["k_cache"], t["v_cache"] = _randn(g, KV, S, D), _randn(g, KV, S, D, std=0.6)
    elif op in ("dense", "swiglu"):
        R, N, B = case["rows"], case["cols"], case["batch"]
        for name in ("w", "w2") if op == "swiglu" else ("w",):
            t[name] = _randn(g, R, N, std=0.02)
        if case["bf16"]:
            t = {k: v.bfloat16() for k, v in t.items()}
        t["x"] = _randn(g, B, N)
        if case["norm"]:
            t["norm"] = _randn(g, N, std=0.02, mean=1.0)
        if case.get("bias"):
            t["bias"] = _randn(g, R, std=0.1)
    elif op in ("gemm_bf16", "gemm_f32"):
        M, N, K = case["m"], case["n"], case["k"]
        t["a"], t["w"] = _randn(g, M, K), _randn(g, N, K, std=0.02)
        if case["swiglu"]:
            t["w2"] = _randn(g, N, K, std=0.02)
        if op == "gemm_bf16":
            t = {k: v.bfloat16() for k, v in t.items()}
        if case["bias"]:
            t["bias"] = _randn(g, N, std=0.1)
    elif op == "sample":
        # logits of a model: a few likely tokens over a wide floor
        t["logits"] = _randn(g, case["rows"], case["n"], std=2.0)
        t["rng"] = torch.tensor([hw.java_random_state(seed * 8 + r) for r in range(case["rows"])], dtype=torch.int64)
    return t


# ---- models ------------------------------------------------------------------------------------------

MODEL_KEYS = ("shape", "layers", "vocab", "bf16", "kv16", "per_head", "bias")


def _weights(case):
    """(key, fp32 GPU tensor) of every weight, bf16-rounded for bf16 models."""
    d, f, h, kv, hd = SHAPES[case["shape"]]
    g = _gen(4242 + case["layers"] + case["vocab"])
    out_std = 0.02 / math.sqrt(2 * case["layers"])

    def mat(n, k, std=0.02):
        t = _randn(g, n, k, std=std)
        return t.bfloat16().float() if case["bf16"] else t

    yield "model.embed_tokens.weight", mat(case["vocab"], d, EMBED_STD)
    yield "model.norm.weight", _randn(g, d, std=0.02, mean=1.0)
    for i in range(case["layers"]):
        p = "model.layers.%d." % i
        yield p + "input_layernorm.weight", _randn(g, d, std=0.02, mean=1.0)
        yield p + "self_attn.q_proj.weight", mat(h * hd, d)
        yield p + "self_attn.k_proj.weight", mat(kv * hd, d)
        yield p + "self_attn.v_proj.weight", mat(kv * hd, d)
        yield p + "self_attn.o_proj.weight", mat(d, h * hd, out_std)
        yield p + "self_attn.q_norm.weight", _randn(g, h, hd, std=0.02, mean=1.0)
        yield p + "self_attn.k_norm.weight", _randn(g, kv, hd, std=0.02, mean=1.0)
        yield p + "post_attention_layernorm.weight", _randn(g, d, std=0.02, mean=1.0)
        yield p + "mlp.gate_proj.weight", mat(f, d)
        yield p + "mlp.up_proj.weight", mat(f, d)
        yield p + "mlp.down_proj.weight", mat(d, f, out_std)
        if case["bias"]:
            for n, rows in (("q", h * hd), ("k", kv * hd), ("v", kv * hd)):
                yield p + "self_attn.%s_proj.bias" % n, _randn(g, rows, std=0.1)


def _positions(case):
    return case["prompt"] + case.get("steps", 0)


def _model(case):
    """The loaded model of this case; the one before it is closed."""
    key = tuple(case[k] for k in MODEL_KEYS) + (case["batch"], _positions(case))
    if _kept.get("key") != key:
        if "model" in _kept:
            _kept.pop("key")
            _kept.pop("model").close()
        d, f, h, kv, hd = SHAPES[case["shape"]]
        cfg = C.Qwen3Config(dim=d, hidden_dim=f, layer_count=case["layers"], head_count=h, kv_head_count=kv,
                            vocab_size=case["vocab"], seq_len=_positions(case), head_size=hd, rope_theta=THETA,
                            epsilon=EPS, qk_norm_mode=C.QK_NORM_PER_HEAD if case["per_head"] else C.QK_NORM_WHOLE,
                            weight_dtype=C.DTYPE_BF16 if case["bf16"] else C.DTYPE_F32,
                            kv_dtype=C.DTYPE_F16 if case["kv16"] else C.DTYPE_F32, max_batch=case["batch"],
                            qkv_bias=case["bias"])
        _kept["model"] = Qwen3(cfg, ((k, t.cpu().numpy()) for k, t in _weights(case)), ctx=_context())
        _kept["key"] = key
    return _kept["model"]


def _prompts(case, seed):
    r = np.random.RandomState(seed % (1 << 32))
    return r.randint(0, case["vocab"], (case["batch"], case["prompt"])).astype(np.int32)


# ---- the measured call -------------------------------------------------------------------------------

def prepare(case, seed):
    op = case["op"]
    if op in ("prompt", "generate"):
        return {"case": case, "model": _model(case).model, "prompts": _prompts(case, seed)}
    s = _Buffers()
    for name, t in _inputs(case, seed).items():
        s.add(name, t)
    new = lambda dtype, *shape: torch.zeros(*shape, dtype=dtype, device="cuda")  # noqa: E731
    if op == "attention":
        s.add("out", new(torch.float32, case["heads"] * case["head_size"]))
    elif op in ("dense", "swiglu"):
        s.add("y", new(torch.float32, case["batch"], case["rows"]))
    elif op in ("gemm_bf16", "gemm_f32"):
        s.add("c", new(torch.bfloat16 if op == "gemm_bf16" and case["swiglu"] else torch.float32,
                       case["m"], case["n"]))
    else:
        s.add("out", new(torch.int32, case["rows"]))
    return {"case": case, "buffers": s.ready()}


def run(state):
    case = state["case"]
    op = case["op"]
    if op in ("prompt", "generate"):
        am = state["model"]
        am.reset()
        for b in range(case["batch"]):
            am.set_prompt(state["prompts"][b], b)
        if op == "prompt":
            logits = am.prefill(return_logits=True)
            return {"logits": logits, "hidden": am.hidden()}
        am.prefill()
        tokens = am.run(case["steps"] - 1)
        last, logits = am.next(return_logits=True)
        return {"tokens": tokens, "last": last, "logits": logits, "hidden": am.hidden()}
    s = state["buffers"]
    ctx = s.ctx
    if op == "attention":
        ctx.attention_decode(s["q"], s["k"], s["v"], s["q_norm"], s["k_norm"], EPS,
                             C.QK_NORM_PER_HEAD if case["per_head"] else C.QK_NORM_WHOLE, s["k_cache"], s["v_cache"],
                             case["max_seq"], case["pos"], case["heads"], case["kv_heads"], case["head_size"], THETA,
                             s["out"])
        return {k: s.view[k] for k in ("out", "k_cache", "v_cache")}
    if op == "dense":
        ctx.dense(s["w"], hw.DTYPE_BF16 if case["bf16"] else hw.DTYPE_F32, s["x"], s["y"], case["rows"], case["cols"],
                  case["batch"], s["bias"], s["norm"], EPS)
        return s.view["y"]
    if op == "swiglu":
        ctx.swiglu(s["w"], s["w2"], hw.DTYPE_BF16 if case["bf16"] else hw.DTYPE_F32, s["x"], s["y"], case["rows"],
                   case["cols"], case["batch"], s["norm"], EPS)
        return s.view["y"]
    if op == "gemm_bf16":
        if case["swiglu"]:
            ctx.gemm_bf16(s["a"], s["w"], case["m"], case["n"], case["k"], hw.GEMM_SWIGLU, W2=s["w2"], O=s["c"])
        else:
            ctx.gemm_bf16(s["a"], s["w"], case["m"], case["n"], case["k"], hw.GEMM_STORE, bias=s["bias"], C=s["c"])
        return s.view["c"]
    if op == "gemm_f32":
        ctx.gemm_f32(s["a"], s["w"], case["m"], case["n"], case["k"],
                     hw.GEMM_SWIGLU if case["swiglu"] else hw.GEMM_STORE, W2=s["w2"], bias=s["bias"], C=s["c"])
        return s.view["c"]
    ctx.sample(s["logits"], case["rows"], case["n"], case["mode"], case["temperature"], case["top_p"], s["rng"],
               s["out"])
    return {"tokens": s.view["out"], "rng": s.view["rng"]}


# ---- what a pass cannot do without -------------------------------------------------------------------

def work(case):
    op = case["op"]
    if op == "attention":
        rows, H, KV, D = case["pos"] + 1, case["heads"], case["kv_heads"], case["head_size"]
        return {"bytes": 4 * (2 * rows * KV * D + 2 * KV * D + 3 * H * D + 3 * KV * D), "flops": 4 * rows * H * D}
    if op in ("dense", "swiglu"):
        R, N, B, n = case["rows"], case["cols"], case["batch"], 2 if op == "swiglu" else 1
        return {"bytes": n * R * N * (2 if case["bf16"] else 4) + 4 * B * (R + N), "flops": 2 * n * R * N * B}
    if op in ("gemm_bf16", "gemm_f32"):
        M, N, K, n = case["m"], case["n"], case["k"], 2 if case["swiglu"] else 1
        e = 2 if op == "gemm_bf16" else 4
        return {"bytes": e * (M * K + n * N * K) + (2 if op == "gemm_bf16" and case["swiglu"] else 4) * M * N,
                "flops": 2 * n * M * N * K}
    if op == "sample":
        return {"bytes": 4 * case["rows"] * case["n"], "flops": 4 * case["rows"] * case["n"]}
    d, f, h, kv, hd = SHAPES[case["shape"]]
    B, T, L, V, steps = case["batch"], case["prompt"], case["layers"], case["vocab"], case.get("steps", 0)
    e, ke = 2 if case["bf16"] else 4, 2 if case["kv16"] else 4
    layer, head = d * (h + 2 * kv) * hd + d * h * hd + 3 * d * f, V * d
    row = 2 * kv * hd * ke  # a position's K and V in one layer
    nbytes = e * (L * layer + head) + B * T * L * row + 4 * B * (V + d)
    flops = 2 * B * T * L * layer + 2 * B * head + 4 * B * L * h * hd * T * (T + 1) // 2
    seen = sum(T + i + 1 for i in range(steps))
    nbytes += steps * e * (L * layer + head) + B * L * row * (seen + steps)
    flops += 2 * B * steps * (L * layer + head) + 4 * B * L * h * hd * seen
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    op = case["op"]
    if op == "sample":
        return "exact"
    if op == "gemm_bf16":
        # a bf16 output (1.7e-3 from 64 bits), or fp32 sums of exact products (3e-7)
        return {"rel": 7e-3} if case["swiglu"] else {"rel": 2e-6}
    if op in ("dense", "swiglu") and case["bf16"]:
        return {"rel": 1.5e-5}  # three or more sequences split the input into two bf16 planes (3.6e-6)
    if op in ("attention", "dense", "swiglu", "gemm_f32"):
        return {"rel": 2e-6}  # 1e-7 to 6e-7 from 64 bits
    # whole passes: fp16 MFMA operands in a bf16 model's prompt (1e-4 to 7e-4 from 64 bits), an fp16 cache
    # where the case has one; fp32 throughout otherwise (3e-7 to 6e-7)
    return {"rel": 3e-3, "max": 0.05} if case["bf16"] else {"rel": 5e-6, "max": 2e-4}


# ---- the same in 64 bits, in plain torch -------------------------------------------------------------

def _rms(x, w):
    return w * x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)


def _rope(x, pos):
    """Split-half rotation of (..., rows, heads, hd) at the positions `pos` (rows)."""
    half = x.shape[-1] // 2
    freq = torch.exp(torch.arange(half, dtype=torch.float64, device=x.device) * (-2.0 * math.log(THETA) / x.shape[-1]))
    ang = pos.to(torch.float64)[:, None] * freq
    c, s = torch.cos(ang)[:, None, :], torch.sin(ang)[:, None, :]
    a, b = x[..., :half], x[..., half:]
    return torch.cat((a * c - b * s, a * s + b * c), -1)


def _qk_norm(x, w, per_head):
    """x (rows, heads, hd) normalised over each head, or over all of a row."""
    if per_head:
        return _rms(x, w.view(x.shape[-2:]))
    return _rms(x.flatten(-2), w.flatten()).view(x.shape)


def _silu(x):
    return x / (1 + torch.exp(-x))


def _exact_model(case, seed):
    d, f, h, kv, hd = SHAPES[case["shape"]]
    w = {k: t.double() for k, t in _weights(case)}
    steps = case.get("steps", 0)
    prompts = _prompts(case, seed)
    outs = {"tokens": [], "last": [], "logits": [], "hidden": []}
    for b in range(case["batch"]):
        cache = [None] * case["layers"]

        def forward(ids, start):
            pos = torch.arange(start, start + len(ids), device="cuda")
            x = w["model.embed_tokens.weight"][torch.as_tensor(ids, device="cuda", dtype=torch.long)]
            mask = torch.arange(start + len(ids), device="cuda")[None, :] > pos[:, None]
            for i in range(case["layers"]):
                p = "model.layers.%d." % i
                y = _rms(x, w[p + "input_layernorm.weight"])
                q, k, v = (y @ w[p + "self_attn.%s_proj.weight" % n].T for n in "qkv")
                if case["bias"]:
                    q, k, v = (t + w[p + "self_attn.%s_proj.bias" % n] for n, t in zip("qkv", (q, k, v)))
                q = _rope(_qk_norm(q.view(-1, h, hd), w[p + "self_attn.q_norm.weight"], case["per_head"]), pos)
                k = _rope(_qk_norm(k.view(-1, kv, hd), w[p + "self_attn.k_norm.weight"], case["per_head"]), pos)
                v = v.view(-1, kv, hd)
                if cache[i] is not None:
                    k, v = torch.cat((cache[i][0], k)), torch.cat((cache[i][1], v))
                cache[i] = (k, v)
                o = torch.empty_like(q)
                for j in range(h):
                    s = (q[:, j] @ k[:, j // (h // kv)].T / math.sqrt(hd)).masked_fill(mask, -math.inf)
                    o[:, j] = torch.softmax(s, -1) @ v[:, j // (h // kv)]
                x = x + o.flatten(1) @ w[p + "self_attn.o_proj.weight"].T
                y = _rms(x, w[p + "post_attention_layernorm.weight"])
                y = _silu(y @ w[p + "mlp.gate_proj.weight"].T) * (y @ w[p + "mlp.up_proj.weight"].T)
                x = x + y @ w[p + "mlp.down_proj.weight"].T
            return x[-1], _rms(x[-1], w["model.norm.weight"]) @ w["model.embed_tokens.weight"].T

        x, logits = forward(prompts[b].tolist(), 0)
        fed = []
        for i in range(steps):
            fed.append(int(logits.argmax()))
            x, logits = forward([fed[-1]], case["prompt"] + i)
        outs["tokens"].append(fed[:-1])
        outs["last"].append(fed[-1:])
        outs["logits"].append(logits)
        outs["hidden"].append(x)
    logits, hidden = torch.stack(outs["logits"]).cpu(), torch.stack(outs["hidden"]).cpu()
    if case["op"] == "prompt":
        return {"logits": logits, "hidden": hidden}
    return {"tokens": torch.tensor(outs["tokens"], dtype=torch.int32),
            "last": torch.tensor(outs["last"], dtype=torch.int32).view(-1), "logits": logits, "hidden": hidden}


def exact(case, seed):
    op = case["op"]
    if op in ("prompt", "generate"):
        return _exact_model(case, seed)
    if op == "sample":
        return None  # whole numbers
    t = {k: v.double() for k, v in _inputs(case, seed).items()}
    if op == "attention":
        H, KV, D, pos = case["heads"], case["kv_heads"], case["head_size"], case["pos"]
        at = torch.tensor([pos], device="cuda")
        q = _rope(_qk_norm(t["q"].view(1, H, D), t["q_norm"], case["per_head"]), at)[0]
        k = _rope(_qk_norm(t["k"].view(1, KV, D), t["k_norm"], case["per_head"]), at)[0]
        kc, vc = t["k_cache"], t["v_cache"]
        kc[:, pos], vc[:, pos] = k, t["v"].view(KV, D)
        out = torch.empty_like(q)
        for j in range(H):
            kk, vv = kc[j // (H // KV), :pos + 1], vc[j // (H // KV), :pos + 1]
            out[j] = torch.softmax(kk @ q[j] / math.sqrt(D), 0) @ vv
        return {"out": out.flatten(), "k_cache": kc, "v_cache": vc}
    if op in ("dense", "swiglu"):
        x = _rms(t["x"], t["norm"]) if case["norm"] else t["x"]
        y = x @ t["w"].T
        if op == "swiglu":
            return (x @ t["w2"].T) * _silu(y)
        return y + t["bias"] if case["bias"] else y
    y = t["a"] @ t["w"].T
    if case["swiglu"]:
        return (t["a"] @ t["w2"].T) * _silu(y)
    return y + t["bias"] if case["bias"] else y
