"""The work that a user of this library has it do, as measurable cases.

The library is the prefill path of a Qwen3.5-style hybrid decoder (three Gated DeltaNet layers to
one full-attention layer): a program keeps weights and activation buffers on the GPU and calls the
cs1_* operations layer by layer, or lets the native runner (qwen3_5_native.model) do it.  The cases
are the layers' blocks, each through the operations that the runner itself calls in that order, the
attention operation alone at head dim 128, and two whole calls of the runner.

Sizes are the repository's own: configurations 0 to 4 of the benchmark, the prompt lengths 107, 936
and 3399 of the GDN benchmark, and the ranges around them.  Prompts are 64 to 4096 tokens (attention
and GDN layers up to 8192), candidate continuations 8 of 64 to 256 tokens over a 2048-token prefix.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "system1-omni_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from qwen3_5_native import hip  # noqa: E402
from qwen3_5_native import model as QM  # noqa: E402

BF = torch.bfloat16
F64 = torch.float64
EPS = 1e-6
D = 128  # Gated DeltaNet head dim
DH = 256  # the decoder's attention head dim
HALF = 32  # rotary frequencies per head
VOCAB_4B, VOCAB_27B = 151936, 248320
SIZES = {"4b": (2560, 9728, VOCAB_4B), "27b": (5120, 17408, VOCAB_27B)}  # hidden, SwiGLU width, vocabulary
# One period of each decoder (three GDN layers, one attention layer) at full width: a model of 32 or
# 64 such layers repeats it, and over one period the roundings of the layers stay comparable.
PERIOD = {
    "4b": QM.Config(**{**QM.CFG3_4B.__dict__, "layers": 4}),
    "27b": QM.Config(**{**QM.CFG4_27B.__dict__, "layers": 4}),
}


def listed():
    return [
        # the headline layer: gated causal GQA attention with log-sum-exp, one 2048-token prompt
        {"name": "attn-d128-2048", "kind": "attn", "T": 2048, "hq": 16, "hk": 4, "dh": 128, "gate": True, "lse": True},
        # an attention layer of a short chat prompt in the 27B-class decoder
        {"name": "attnlayer-333", "kind": "attnlayer", "T": 333, "hq": 24, "hk": 4},
        # an attention layer of the 4096-token decision prompt in the 4B-class decoder
        {"name": "attnlayer-4096", "kind": "attnlayer", "T": 4096, "hq": 16, "hk": 4},
        # candidate scoring: eight continuations of one cached 2048-token prefix, one packed call
        {"name": "attncands-8x", "kind": "attncands", "pre": 2048, "n": 8, "lo": 64, "hi": 256, "lens": 5, "hq": 24,
         "hk": 4},
        # a GDN layer of the shortest prompt of the GDN benchmark (48 value heads): latency
        {"name": "gdn-107", "kind": "gdn", "T": 107, "hk": 16, "h": 48, "state": False},
        # the GDN benchmark's middle prompt
        {"name": "gdn-936", "kind": "gdn", "T": 936, "hk": 16, "h": 48, "state": False},
        # a long document through a GDN layer that continues from a state and leaves one
        {"name": "gdn-8192", "kind": "gdn", "T": 8192, "hk": 16, "h": 32, "state": True},
        # the GDN layer of candidate scoring: packed continuations of one state
        {"name": "gdncands-8x", "kind": "gdncands", "n": 8, "lo": 64, "hi": 256, "lens": 5, "hk": 16, "h": 48},
        # the MLP of a short prompt in the 4B-class decoder
        {"name": "mlp-4b-333", "kind": "mlp", "T": 333, "size": "4b"},
        # the MLP of a packed candidate batch in the 27B-class decoder
        {"name": "mlp-27b-1217", "kind": "mlp", "T": 1217, "size": "27b"},
        # the decision call: a 4096-token prompt, the last hidden state and its label logits
        {"name": "decide-4b-4096", "kind": "decide", "T": 4096, "size": "4b", "labels": 64},
        # scoring a short text: the log-probability of each of its tokens
        {"name": "logprobs-27b-250", "kind": "logprobs", "T": 250, "size": "27b"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attn", "attnlayer", "attnlayer", "attncands", "attncands", "gdn", "gdn", "gdncands", "mlp",
                       "mlp", "decide", "logprobs"])
    c = {"kind": kind}
    if kind == "attn":
        c.update(T=_log_int(rng, 64, 8192), hq=rng.choice([8, 16, 32]), hk=4, dh=128, gate=rng.random() < 0.7,
                 lse=rng.random() < 0.5)
        if c["hq"] == 32:
            c["hk"] = 8
    elif kind == "attnlayer":
        hq = rng.choice([16, 24])
        c.update(T=_log_int(rng, 64, 8192), hq=hq, hk=4)
    elif kind == "attncands":
        hi = rng.choice([16, 64, 256])
        c.update(pre=64 * _log_int(rng, 4, 64), n=rng.randint(2, 12), lo=rng.choice([1, hi // 4]), hi=hi,
                 lens=rng.randint(0, 1 << 20), hq=rng.choice([16, 24]), hk=4)
    elif kind == "gdn":
        c.update(T=_log_int(rng, 64, 8192), hk=16, h=rng.choice([16, 32, 48]), state=rng.random() < 0.5)
    elif kind == "gdncands":
        hi = rng.choice([64, 256])
        c.update(n=rng.randint(2, 12), lo=rng.choice([1, hi // 4]), hi=hi, lens=rng.randint(0, 1 << 20), hk=16,
                 h=rng.choice([32, 48]))
    elif kind == "mlp":
        size = rng.choice(["4b", "27b"])
        c.update(T=_log_int(rng, 64, 4096 if size == "4b" else 2048), size=size)
    elif kind == "decide":
        c.update(T=_log_int(rng, 64, 4096), size="4b", labels=rng.randint(48, 96))
    else:
        c.update(T=_log_int(rng, 64, 512), size="27b")
    return c


# ---------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape, std=1.0):
    return (torch.randn(*shape, generator=g, device="cuda") * std).to(BF)


def _empty(*shape, dtype=BF):
    return torch.empty(*shape, dtype=dtype, device="cuda")


def _lens(c):
    """The candidates' lengths, uniform on [lo, hi]."""
    return [int(x) for x in np.random.default_rng(c["lens"]).integers(c["lo"], c["hi"] + 1, c["n"])]


def _offsets(lens):
    return np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)


def _rotary(positions):
    inv = 1.0 / (1e7 ** (torch.arange(HALF, dtype=F64, device="cuda") / HALF))
    a = positions.to(F64)[:, None] * inv
    return a.cos().to(BF), a.sin().to(BF)


def _ids(seed, T, vocab):
    return np.random.default_rng(seed).integers(0, vocab, T).astype(np.int32)


def _attn_inputs(c, seed):
    g = _gen(seed)
    T, hq, hk, dh = c["T"], c["hq"], c["hk"], c["dh"]
    s = {"q": _randn(g, T, hq, dh), "k": _randn(g, T, hk, dh), "v": _randn(g, T, hk, dh)}
    s["gate"] = _randn(g, T, hq, dh) if c["gate"] else None
    return s


def _attnlayer_inputs(c, seed):
    # one row holds what the QKV projection writes: per q head (q | gate), then k, then v
    g = _gen(seed)
    T, hq, hk = c["T"], c["hq"], c["hk"]
    cos, sin = _rotary(torch.arange(T, device="cuda"))
    return {"x": _randn(g, T, 2 * hq * DH + 2 * hk * DH), "qw": _randn(g, DH, std=0.1), "kw": _randn(g, DH, std=0.1),
            "cos": cos, "sin": sin}


def _attncands_inputs(c, seed):
    g = _gen(seed)
    R, hq, hk = sum(_lens(c)), c["hq"], c["hk"]
    return {"q": _randn(g, R, hq, DH), "k": _randn(g, R, hk, DH), "v": _randn(g, R, hk, DH), "gate": _randn(g, R, hq, DH),
            "kp": _randn(g, c["pre"], hk, DH), "vp": _randn(g, c["pre"], hk, DH)}


def _gdn_inputs(c, seed, T):
    # one row holds what the input projection writes: q | k | v | z | b | a.  The gates' decay is spread
    # as the layer's parameters are set up: softplus(dt_bias) log-uniform on [1e-3, 1e-1], A on [1, 16].
    g = _gen(seed)
    hk, h = c["hk"], c["h"]
    conv = (2 * hk + h) * D
    u = torch.rand(h, generator=g, device="cuda")
    dt = torch.exp(math.log(1e-3) + u * (math.log(1e-1) - math.log(1e-3)))
    a_log = torch.log(1 + 15 * torch.rand(h, generator=g, device="cuda")).to(BF)
    s = {"x": _randn(g, T, conv + h * D + 2 * h), "cw": (torch.rand(conv, 4, generator=g, device="cuda") - 0.5).to(BF),
         "a_log": a_log, "dt_bias": torch.log(torch.expm1(dt)).to(BF), "gw": (1 + _randn(g, D, std=0.1).float()).to(BF)}
    s["x"][:, -h:] *= 0.5
    return s, g, conv


def _mlp_inputs(c, seed):
    g = _gen(seed)
    hidden, inter, vocab = SIZES[c["size"]]
    ids = torch.from_numpy(_ids(seed, c["T"], vocab)).cuda()
    return {"ids": ids, "table": _randn(g, vocab, hidden, std=0.02), "delta": _randn(g, c["T"], hidden),
            "norm": _randn(g, hidden, std=0.1), "next": _randn(g, hidden, std=0.1),
            "gate_up": _randn(g, 2 * inter, hidden, std=0.02), "down": _randn(g, hidden, inter, std=0.02)}


class _Gemm:
    """The GEMM handle that a program keeps, with the runner's 32 MiB workspace."""

    def __init__(self):
        self.handle = hip.api().cs1_gemm_create(32 << 20)

    def __del__(self):
        if self.handle and hip is not None:  # (None: the interpreter is ending)
            hip.api().cs1_gemm_destroy(self.handle)


def prepare(case, seed):
    hip.load()
    c = dict(case)
    kind = c["kind"]
    api = hip.api()
    s = {"case": c}
    if kind == "attn":
        s.update(_attn_inputs(c, seed))
        s["out"] = _empty(c["T"], c["hq"], c["dh"])
        s["lse"] = _empty(c["hq"], c["T"], dtype=torch.float32) if c["lse"] else None
    elif kind == "attnlayer":
        s.update(_attnlayer_inputs(c, seed))
        T, hq, hk = c["T"], c["hq"], c["hk"]
        s.update(q=_empty(T, hq, DH), gate=_empty(T, hq, DH), k=_empty(T, hk, DH), out=_empty(T, hq, DH))
    elif kind == "attncands":
        s.update(_attncands_inputs(c, seed))
        s["cu"] = _offsets(_lens(c))
        R = int(s["cu"][-1])
        s.update(out=_empty(R, c["hq"], DH), lse=_empty(c["hq"], R, dtype=torch.float32))
    elif kind in ("gdn", "gdncands"):
        if kind == "gdn":
            T = rows = c["T"]
            nstates = 1
        else:
            s["cu"] = _offsets(_lens(c))
            T, nstates = int(s["cu"][-1]), c["n"]
            rows = 64 * sum((n + 63) // 64 for n in _lens(c))
        inputs, g, conv = _gdn_inputs(c, seed, T)
        s.update(inputs)
        h = c["h"]
        s["s_in"] = (torch.randn(h, D, D, generator=g, device="cuda") * 0.1) if kind == "gdncands" or c["state"] else None
        s["hist"] = _randn(g, 3, s["x"].shape[1]) if kind == "gdncands" else None
        s.update(q=_empty(T, c["hk"], D), k=_empty(T, c["hk"], D), v=_empty(T, h, D), o=_empty(T, h, D),
                 out=_empty(T, h, D), s_out=_empty(nstates, h, D, D, dtype=torch.float32),
                 ws=_empty(api.cs1_gdn_workspace_floats(rows, h), dtype=torch.float32), conv=conv)
    elif kind == "mlp":
        s.update(_mlp_inputs(c, seed))
        hidden, inter, _ = SIZES[c["size"]]
        T = c["T"]
        s.update(res=_empty(T, hidden), xn=_empty(T, hidden), gu=_empty(T, 2 * inter), act=_empty(T, inter),
                 d2=_empty(T, hidden), out=_empty(T, hidden), gemm=_Gemm())
    else:
        cfg = PERIOD[c["size"]]
        s["model"] = QM.Model(cfg, seed=seed, max_tokens=c["T"])
        s["ids"] = _ids(seed, c["T"], cfg.vocab)
        if kind == "decide":
            # a server answers prompt after prompt: it keeps the label rows and replays a captured graph
            s["model"].set_graph(True)
            labels = _ids(seed + 1, c["labels"], cfg.vocab)
            s["letters"] = _weight(s["model"], cfg, QM.EMBED, 0, rows=labels).float().cpu().numpy()
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------- one pass

def _p(t):
    return None if t is None else t.data_ptr()


def run(s):
    c = s["case"]
    kind = c["kind"]
    api = hip.api()
    st = torch.cuda.current_stream().cuda_stream
    if kind == "attn":
        hip.check(api.cs1_attention_ex(_p(s["q"]), _p(s["k"]), _p(s["v"]), c["hk"] * c["dh"], _p(s["gate"]), _p(s["out"]),
                                       _p(s["lse"]), c["T"], c["hq"], c["hk"], c["dh"], c["dh"] ** -0.5, 0, st),
                  "cs1_attention_ex")
        return [s["out"], s["lse"]] if c["lse"] else [s["out"]]
    if kind == "attnlayer":
        T, hq, hk = c["T"], c["hq"], c["hk"]
        ld = s["x"].shape[1]
        kr = _p(s["x"]) + 2 * (2 * hq * DH)
        vr = kr + 2 * hk * DH
        hip.check(api.cs1_attn_prep(_p(s["x"]), kr, ld, _p(s["qw"]), _p(s["kw"]), _p(s["cos"]), _p(s["sin"]), _p(s["q"]),
                                    _p(s["gate"]), _p(s["k"]), T, hq, hk, DH, HALF, EPS, st), "cs1_attn_prep")
        hip.check(api.cs1_attention_gated(_p(s["q"]), _p(s["k"]), vr, ld, _p(s["gate"]), _p(s["out"]), T, hq, hk, DH,
                                          DH ** -0.5, st), "cs1_attention_gated")
        return [s["out"], s["k"]]
    if kind == "attncands":
        hq, hk = c["hq"], c["hk"]
        hip.check(api.cs1_attention_prefix_varlen(_p(s["q"]), _p(s["k"]), _p(s["v"]), hk * DH, _p(s["kp"]), _p(s["vp"]),
                                                  hk * DH, c["pre"], _p(s["gate"]), _p(s["out"]), _p(s["lse"]),
                                                  s["cu"].ctypes.data, len(s["cu"]) - 1, hq, hk, DH, DH ** -0.5, st),
                  "cs1_attention_prefix_varlen")
        return [s["out"], s["lse"]]
    if kind in ("gdn", "gdncands"):
        hk, h = c["hk"], c["h"]
        T, ld = s["x"].shape
        z = _p(s["x"]) + 2 * s["conv"]
        b = z + 2 * h * D
        a = b + 2 * h
        scale = D ** -0.5
        if kind == "gdn":
            hip.check(api.cs1_gdn_conv(_p(s["x"]), ld, _p(s["cw"]), _p(s["q"]), _p(s["k"]), _p(s["v"]), T, hk * D, h * D,
                                       st), "cs1_gdn_conv")
            hip.check(api.cs1_gdn_prefill_gated_x(_p(s["q"]), _p(s["k"]), _p(s["v"]), b, a, ld, _p(s["a_log"]),
                                                  _p(s["dt_bias"]), _p(s["o"]), _p(s["ws"]), T, h, hk, scale,
                                                  _p(s["s_in"]), _p(s["s_out"]), st), "cs1_gdn_prefill_gated_x")
        else:
            cu, n = s["cu"].ctypes.data, len(s["cu"]) - 1
            hip.check(api.cs1_gdn_conv_varlen(_p(s["x"]), ld, _p(s["cw"]), _p(s["q"]), _p(s["k"]), _p(s["v"]), cu, n,
                                              _p(s["hist"]), hk * D, h * D, st), "cs1_gdn_conv_varlen")
            hip.check(api.cs1_gdn_prefill_gated_varlen(_p(s["q"]), _p(s["k"]), _p(s["v"]), b, a, ld, _p(s["a_log"]),
                                                       _p(s["dt_bias"]), _p(s["o"]), _p(s["ws"]), cu, n, h, hk, scale,
                                                       _p(s["s_in"]), 0, _p(s["s_out"]), h * D * D, st),
                      "cs1_gdn_prefill_gated_varlen")
        hip.check(api.cs1_gated_rms_norm(_p(s["o"]), z, ld, _p(s["gw"]), _p(s["out"]), T, h, D, EPS, st),
                  "cs1_gated_rms_norm")
        return [s["out"], s["s_out"]]
    if kind == "mlp":
        hidden, inter, _ = SIZES[c["size"]]
        T, gm = c["T"], s["gemm"].handle
        hip.check(api.cs1_embed(_p(s["ids"]), _p(s["table"]), _p(s["res"]), T, hidden, st), "cs1_embed")
        hip.check(api.cs1_add_rms_norm(_p(s["res"]), _p(s["delta"]), _p(s["norm"]), _p(s["xn"]), T, hidden, EPS, st),
                  "cs1_add_rms_norm")
        hip.check(api.cs1_gemm(gm, _p(s["xn"]), _p(s["gate_up"]), _p(s["gu"]), T, 2 * inter, hidden, 2 * inter, st),
                  "cs1_gemm")
        hip.check(api.cs1_silu_mul(_p(s["gu"]), 2 * inter, _p(s["act"]), T, inter, st), "cs1_silu_mul")
        hip.check(api.cs1_gemm(gm, _p(s["act"]), _p(s["down"]), _p(s["d2"]), T, hidden, inter, hidden, st), "cs1_gemm")
        hip.check(api.cs1_add_rms_norm(_p(s["res"]), _p(s["d2"]), _p(s["next"]), _p(s["out"]), T, hidden, EPS, st),
                  "cs1_add_rms_norm")
        return [s["out"], s["res"]]
    if kind == "decide":
        last = s["model"].forward(s["ids"])
        return [last, QM.letter_logits(s["letters"], last, c["labels"])]
    return [s["model"].logprobs(s["ids"])]


# ---------------------------------------------------------------- what a pass cannot do without

def _pairs(T):
    return T * (T + 1) / 2


def _gdn_flops(T, h):
    # per token and value head in chunks of 64: the lower triangles of k k^T and q k^T, of the inverse and
    # its two products, and three products with the 128 x 128 state
    return T * h * 139264.0


def _gdn_work(c, T, states):
    hk, h = c["hk"], c["h"]
    row = (2 * hk + h) * D + h * D + 2 * h
    b = 2.0 * T * (row + h * D) + 4.0 * states * h * D * D
    return {"bytes": b, "flops": _gdn_flops(T, h) + 2.0 * 4 * T * (2 * hk + h) * D}


def _layer_flops(cfg, T, i):
    mlp = 2.0 * T * 3 * cfg.hidden * cfg.intermediate
    if cfg.is_full(i):
        w = 2 * cfg.heads * DH + 2 * cfg.kv_heads * DH
        return mlp + 2.0 * T * cfg.hidden * (w + cfg.heads * DH) + 4.0 * DH * cfg.heads * _pairs(T)
    vd = cfg.lin_v_heads * D
    w = 2 * cfg.lin_k_heads * D + 2 * vd + 2 * cfg.lin_v_heads
    return mlp + 2.0 * T * cfg.hidden * (w + vd) + _gdn_flops(T, cfg.lin_v_heads)


def _layer_bytes(cfg, i):
    mlp = 3 * cfg.hidden * cfg.intermediate
    if cfg.is_full(i):
        return 2.0 * (mlp + cfg.hidden * (3 * cfg.heads * DH + 2 * cfg.kv_heads * DH))
    vd = cfg.lin_v_heads * D
    return 2.0 * (mlp + cfg.hidden * (2 * cfg.lin_k_heads * D + 3 * vd + 2 * cfg.lin_v_heads))


def work(case):
    c = case
    kind = c["kind"]
    if kind == "attn":
        T, hq, hk, dh = c["T"], c["hq"], c["hk"], c["dh"]
        return {"bytes": 2.0 * T * dh * ((3 if c["gate"] else 2) * hq + 2 * hk) + (4.0 * T * hq if c["lse"] else 0),
                "flops": 4.0 * dh * hq * _pairs(T)}
    if kind == "attnlayer":
        T, hq, hk = c["T"], c["hq"], c["hk"]
        return {"bytes": 2.0 * T * DH * (3 * hq + 3 * hk) + 4.0 * T * HALF, "flops": 4.0 * DH * hq * _pairs(T)}
    if kind == "attncands":
        lens, hq, hk = _lens(c), c["hq"], c["hk"]
        R = sum(lens)
        return {"bytes": 2.0 * DH * (R * (3 * hq + 2 * hk) + 2 * c["pre"] * hk) + 4.0 * R * hq,
                "flops": 4.0 * DH * hq * sum(n * c["pre"] + _pairs(n) for n in lens)}
    if kind == "gdn":
        return _gdn_work(c, c["T"], 2 if c["state"] else 1)
    if kind == "gdncands":
        return _gdn_work(c, sum(_lens(c)), 1 + c["n"])
    if kind == "mlp":
        hidden, inter, _ = SIZES[c["size"]]
        T = c["T"]
        return {"bytes": 2.0 * (3 * hidden * inter + T * hidden * 4), "flops": 2.0 * T * 3 * hidden * inter}
    cfg, T = PERIOD[c["size"]], c["T"]
    w = {"bytes": sum(_layer_bytes(cfg, i) for i in range(cfg.layers)) + 2.0 * T * cfg.hidden,
         "flops": sum(_layer_flops(cfg, T, i) for i in range(cfg.layers))}
    if kind == "logprobs":
        w["bytes"] += 2.0 * cfg.vocab * cfg.hidden
        w["flops"] += 2.0 * T * cfg.vocab * cfg.hidden
    return w


def tolerance(case):
    """About four times what two correct orders of the same sums differ by.  GEMM cases: measured with the handle's
    tuned plans (mlp 8e-5, logprobs 8e-4), with room for a hidden element that moves by a bf16 step and for the layers
    that follow it.  Attention and GDN: the order decides how the 16-bit probabilities and operands round, about as far
    from each other as each is from 64 bits (measured: 3e-3 to 4e-3, and 5e-3 to 6e-3)."""
    return {
        "attn": {"rel": 5e-3, "max": 0.15},
        "attnlayer": {"rel": 5e-3, "max": 0.15},
        "attncands": {"rel": 5e-3, "max": 0.15},
        "gdn": {"rel": 8e-3, "max": 0.2},
        "gdncands": {"rel": 8e-3, "max": 0.2},
        "mlp": {"rel": 4e-3, "max": 0.1},
        "decide": {"rel": 3e-2, "max": 0.2},
        "logprobs": {"rel": 3e-3, "max": 0.02},
    }[case["kind"]]


# ---------------------------------------------------------------- the same in 64 bits

def _weight(model, cfg, which, layer, rows=None):
    """A weight tensor of the runner (an input, like the ids), on the GPU in bf16."""
    ptr, n = ctypes.c_void_p(), ctypes.c_size_t()
    hip.check(model.lib.q35m_tensor(model.handle, layer, which, ctypes.byref(ptr), ctypes.byref(n)), "q35m_tensor")
    st = model.stream()
    t = _empty(n.value) if rows is None else _empty(len(rows), cfg.hidden)
    torch.cuda.synchronize()  # the model copies on its own stream; what last used this memory is done
    if rows is not None:
        for i, r in enumerate(rows):
            hip.check(hip.api().cs1_copy_dd(t[i].data_ptr(), ptr.value + 2 * int(r) * cfg.hidden, 2 * cfg.hidden, st), "copy")
    else:
        hip.check(hip.api().cs1_copy_dd(t.data_ptr(), ptr.value, 2 * n.value, st), "copy")
    hip.check(hip.api().cs1_stream_sync(st), "sync")
    return t


def _attention64(q, k, v, gate, scale, causal_from):
    """Rows i of q [R, hq, dh] see keys 0 .. causal_from + i; float64. Returns out, lse [hq, R]."""
    R, hq, dh = q.shape
    rep = hq // k.shape[1]
    out = torch.empty(R, hq, dh, dtype=F64, device="cuda")
    lse = torch.empty(hq, R, dtype=F64, device="cuda")
    keys = torch.arange(k.shape[0], device="cuda")
    for h in range(hq):
        kh = k[:, h // rep].to(F64).contiguous()
        vh = v[:, h // rep].to(F64).contiguous()
        for r0 in range(0, R, 2048):
            qh = q[r0:r0 + 2048, h].to(F64).contiguous()
            sc = (qh @ kh.t().contiguous()) * scale
            rows = torch.arange(r0, r0 + qh.shape[0], device="cuda")
            sc.masked_fill_(keys[None, :] > causal_from + rows[:, None], -math.inf)
            m = torch.logsumexp(sc, 1)
            lse[h, r0:r0 + 2048] = m
            out[r0:r0 + 2048, h] = torch.exp(sc - m[:, None]) @ vh
    if gate is not None:
        out = out * torch.sigmoid(gate.to(F64))
    return out, lse


def _norm64(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * (1 + w.to(F64))


def _prep64(x, hq, hk, qw, kw, cos, sin):
    T = x.shape[0]
    x = x.to(F64)
    qg = x[:, :2 * hq * DH].reshape(T, hq, 2 * DH)
    kr = x[:, 2 * hq * DH:(2 * hq + hk) * DH].reshape(T, hk, DH)
    c, s = cos.to(F64)[:, None], sin.to(F64)[:, None]

    def rope(y):
        a, b = y[..., :HALF], y[..., HALF:2 * HALF]
        return torch.cat([a * c - b * s, b * c + a * s, y[..., 2 * HALF:]], -1)

    return rope(_norm64(qg[..., :DH], qw)), qg[..., DH:], rope(_norm64(kr, kw)), x[:, (2 * hq + hk) * DH:].reshape(T, hk, DH)


def _gdn64(x, cw, a_log, dt_bias, gw, hk, h, s_in, hist):
    """Conv, gates, delta rule token by token and gated norm of one sequence; returns out and the final state."""
    T = x.shape[0]
    conv = (2 * hk + h) * D
    pre = torch.zeros(3, conv, dtype=F64, device="cuda") if hist is None else hist[:, :conv].to(F64)
    p = torch.cat([pre, x[:, :conv].to(F64)])
    w = cw.to(F64)
    y = sum(p[j:j + T] * w[:, j] for j in range(4))
    y = y * torch.sigmoid(y)
    q, k, v = y[:, :hk * D].reshape(T, hk, D), y[:, hk * D:2 * hk * D].reshape(T, hk, D), y[:, 2 * hk * D:].reshape(T, h, D)
    q = q * torch.rsqrt((q * q).sum(-1, keepdim=True) + 1e-6) * D ** -0.5
    k = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + 1e-6)
    rep = h // hk
    q, k = q.repeat_interleave(rep, 1).contiguous(), k.repeat_interleave(rep, 1).contiguous()
    zba = x[:, conv:].to(F64)
    z, b, a = zba[:, :h * D].reshape(T, h, D), zba[:, h * D:h * D + h], zba[:, h * D + h:]
    beta = torch.sigmoid(b)
    decay = torch.exp(-torch.exp(a_log.to(F64)) * torch.nn.functional.softplus(a + dt_bias.to(F64)))
    S = torch.zeros(h, D, D, dtype=F64, device="cuda") if s_in is None else s_in.to(F64).clone()
    o = torch.empty(T, h, 1, D, dtype=F64, device="cuda")
    kr, kc = k.unsqueeze(2), k.unsqueeze(3)
    qr, vr = q.unsqueeze(2), v.unsqueeze(2)
    dec, bt = decay[:, :, None, None], beta[:, :, None, None]
    for t in range(T):
        S.mul_(dec[t])
        d = (vr[t] - torch.bmm(kr[t], S)) * bt[t]
        S.baddbmm_(kc[t], d)
        torch.bmm(qr[t], S, out=o[t])
    o = o.reshape(T, h, D)
    out = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + EPS) * gw.to(F64) * (z * torch.sigmoid(z))
    return out, S


def _mm64(x, w):
    """x [T, K] w [N, K]^T in float64, the weight widened a block of rows at a time."""
    return torch.cat([x @ w[i:i + 16384].to(F64).t().contiguous() for i in range(0, w.shape[0], 16384)], 1)


def _swiglu64(x, gate_up, down):
    gu = _mm64(x, gate_up)
    g, u = gu[:, :gu.shape[1] // 2], gu[:, gu.shape[1] // 2:]
    return _mm64(g * torch.sigmoid(g) * u, down)


def _decoder64(m, cfg, ids):
    """Final-norm hidden rows of the runner's model in float64."""
    T, hid = len(ids), cfg.hidden
    get = lambda which, i=0: _weight(m, cfg, which, i)  # noqa: E731
    res = get(QM.EMBED).view(-1, hid)[torch.from_numpy(ids).long().cuda()].to(F64)
    cos, sin = _rotary(torch.arange(T, device="cuda"))
    vd = cfg.lin_v_heads * D
    x = _norm64(res, get(QM.INPUT_NORM, 0))
    for i in range(cfg.layers):
        if cfg.is_full(i):
            q, gate, k, v = _prep64(_mm64(x, get(QM.ATTN_QKV, i).view(-1, hid)), cfg.heads, cfg.kv_heads,
                                    get(QM.ATTN_Q_NORM, i), get(QM.ATTN_K_NORM, i), cos, sin)
            o, _ = _attention64(q, k, v, gate, DH ** -0.5, 0)
            res = res + _mm64(o.reshape(T, -1), get(QM.ATTN_O, i).view(hid, -1))
        else:
            o, _ = _gdn64(_mm64(x, get(QM.GDN_IN, i).view(-1, hid)), get(QM.GDN_CONV, i).view(-1, 4), get(QM.GDN_A_LOG, i),
                          get(QM.GDN_DT_BIAS, i), get(QM.GDN_NORM, i), cfg.lin_k_heads, cfg.lin_v_heads, None, None)
            res = res + _mm64(o.reshape(T, vd), get(QM.GDN_OUT, i).view(hid, vd))
        res = res + _swiglu64(_norm64(res, get(QM.POST_NORM, i)), get(QM.MLP_GATE_UP, i).view(-1, hid),
                              get(QM.MLP_DOWN, i).view(hid, -1))
        x = _norm64(res, get(QM.INPUT_NORM, i + 1) if i + 1 < cfg.layers else get(QM.FINAL_NORM))
    return x


def exact(case, seed):
    c = dict(case)
    kind = c["kind"]
    if kind == "attn":
        s = _attn_inputs(c, seed)
        out, lse = _attention64(s["q"], s["k"], s["v"], s["gate"], c["dh"] ** -0.5, 0)
        return [out, lse] if c["lse"] else [out]
    if kind == "attnlayer":
        s = _attnlayer_inputs(c, seed)
        q, gate, k, v = _prep64(s["x"], c["hq"], c["hk"], s["qw"], s["kw"], s["cos"], s["sin"])
        return [_attention64(q, k, v, gate, DH ** -0.5, 0)[0], k]
    if kind == "attncands":
        s = _attncands_inputs(c, seed)
        outs, lses, r0 = [], [], 0
        for n in _lens(c):
            r = slice(r0, r0 + n)
            o, l = _attention64(s["q"][r], torch.cat([s["kp"], s["k"][r]]), torch.cat([s["vp"], s["v"][r]]), s["gate"][r],
                                DH ** -0.5, c["pre"])
            outs.append(o)
            lses.append(l)
            r0 += n
        return [torch.cat(outs), torch.cat(lses, 1)]
    if kind in ("gdn", "gdncands"):
        lens = [c["T"]] if kind == "gdn" else _lens(c)
        s, g, _ = _gdn_inputs(c, seed, sum(lens))
        h = c["h"]
        s_in = (torch.randn(h, D, D, generator=g, device="cuda") * 0.1) if kind == "gdncands" or c["state"] else None
        hist = _randn(g, 3, s["x"].shape[1]) if kind == "gdncands" else None
        outs, states, r0 = [], [], 0
        for n in lens:
            o, S = _gdn64(s["x"][r0:r0 + n], s["cw"], s["a_log"], s["dt_bias"], s["gw"], c["hk"], h, s_in, hist)
            outs.append(o)
            states.append(S)
            r0 += n
        return [torch.cat(outs), torch.stack(states)]
    if kind == "mlp":
        s = _mlp_inputs(c, seed)
        res = s["table"][s["ids"].long()].to(F64) + s["delta"].to(F64)
        res = res + _swiglu64(_norm64(res, s["norm"]), s["gate_up"], s["down"])
        return [_norm64(res, s["next"]), res]
    cfg = PERIOD[c["size"]]
    m = QM.Model(cfg, seed=seed, max_tokens=c["T"])
    ids = _ids(seed, c["T"], cfg.vocab)
    x = _decoder64(m, cfg, ids)
    if kind == "decide":
        letters = _weight(m, cfg, QM.EMBED, 0, rows=_ids(seed + 1, c["labels"], cfg.vocab)).to(F64)
        return [x[-1].cpu().numpy(), (letters @ x[-1]).cpu().numpy()]
    head = _weight(m, cfg, QM.LM_HEAD, 0).view(cfg.vocab, cfg.hidden)
    logits = _mm64(x[:-1].contiguous(), head)
    nxt = torch.from_numpy(ids[1:]).long().cuda()
    return [(logits.gather(1, nxt[:, None])[:, 0] - torch.logsumexp(logits, 1)).cpu().numpy()]
