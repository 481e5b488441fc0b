"""Timed cases of the fused LTX-2.3 DiT block ops on one GPU: what a denoise
loop calls through `opengenie_amd`, from one latent frame (18 x 32 = 576
tokens) to a 576p clip (16 x 18 x 32 = 9216) and its continuation window
(16 x 22 x 40 = 14080).

listed() names the cases, draw(rng) gives one more of the same ranges,
prepare() makes what the program holds before the call (activations, weights,
tables; distributions as in bench.py), run() makes the call, work() counts
what the call cannot do without, tolerance() says how far another correct
implementation may be off and exact() evaluates the call in float64.

The library is an inference path: there is no backward direction. Hidden size
4096, 32 heads of 128, feed-forward width 16384 throughout."""

import math

import torch

from opengenie_amd import attention as A
from opengenie_amd import block as B
from opengenie_amd import ltx_ops as L
from opengenie_amd.rope import video_rope_cos_sin

C, HEADS, HEAD_DIM, FF = 4096, 32, 128, 16384
EPS = 1e-6
FP8 = torch.float8_e4m3fn
DEV = "cuda"


# --------------------------------------------------------------------------
# the cases
# --------------------------------------------------------------------------
def listed():
    return [
        # AdaZero on one latent frame: the smallest call of the loop, where
        # the launch and the host path count.
        {"name": "adazero_576", "op": "adazero", "tokens": 576, "table": "bf16"},
        # The text cross-attention's K (or V) projection of a 256-token
        # prompt: few rows against a whole 4096 x 4096 weight.
        {"name": "text_linear_256", "op": "linear", "tokens": 256, "k": C, "n": C, "dtype": "bf16"},
        # A 4096 -> 4096 projection on one GPU's 9216 / 8 tokens.
        {"name": "linear_1152", "op": "linear", "tokens": 1152, "k": C, "n": C, "dtype": "bf16"},
        # The feed-forward up-projection of a quarter-size clip.
        {"name": "ffn_up_2304", "op": "linear", "tokens": 2304, "k": C, "n": FF, "dtype": "bf16"},
        # GELU-tanh inside the quantizer and the down-projection, 576p clip.
        {"name": "ffn_down_9216", "op": "ffn_down", "tokens": 9216},
        # Q/K RMSNorm + split RoPE before the self-attention, 576p clip.
        {"name": "preattention_9216", "op": "preattention", "t": 16, "h": 18, "w": 32, "rope": "bf16"},
        # The video tokens' cross-attention to a 256-token prompt.
        {"name": "text_attention_9216x256", "op": "attention", "tokens": 9216, "keys": 256},
        # Self-attention of a quarter-size clip and of the 576p clip.
        {"name": "self_attention_2304", "op": "attention", "tokens": 2304, "keys": 2304},
        {"name": "self_attention_9216", "op": "attention", "tokens": 9216, "keys": 9216},
        # The FP8 attention path (per-head quantizers, then the e4m3
        # products) at a token count that divides nothing.
        {"name": "fp8_attention_4999", "op": "fp8_attention", "tokens": 4999},
        # Gated residual with the attention's output bias and a timestep of
        # its own for every token: the continuation window.
        {"name": "residual_bias_14080", "op": "residual_bias", "tokens": 14080, "table": "bf16"},
        # The block's three video branches with every fusion, at ragged token
        # and prompt lengths: what one denoise step repeats per layer.
        {"name": "block_1537x200", "op": "block", "tokens": 1537, "text": 200},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["adazero", "linear", "linear", "linear", "ffn_down", "preattention", "attention", "attention",
                     "text_attention", "fp8_attention", "residual_bias", "block"])
    if op == "adazero":
        return {"op": op, "tokens": _log_int(rng, 64, 14080), "table": rng.choice(["bf16", "f32"])}
    if op == "linear":
        # prompt lengths up to whole clips, every linear of the block
        k, n = rng.choice([(C, C), (C, C), (C, FF), (FF, C)])
        return {"op": op, "tokens": _log_int(rng, 64, 9216), "k": k, "n": n,
                "dtype": rng.choice(["bf16", "bf16", "bf16", "fp16"])}
    if op == "ffn_down":
        return {"op": op, "tokens": _log_int(rng, 512, 9216)}
    if op == "preattention":
        return {"op": op, "t": rng.randint(1, 16), "h": rng.randint(9, 18), "w": rng.randint(16, 32),
                "rope": rng.choice(["bf16", "f32"])}
    if op == "attention":
        n = _log_int(rng, 512, 9000)
        return {"op": op, "tokens": n, "keys": n}
    if op == "text_attention":
        return {"op": "attention", "tokens": _log_int(rng, 512, 9216), "keys": _log_int(rng, 32, 512)}
    if op == "fp8_attention":
        return {"op": op, "tokens": _log_int(rng, 512, 9000)}
    if op == "residual_bias":
        return {"op": op, "tokens": _log_int(rng, 512, 14080), "table": rng.choice(["bf16", "f32"])}
    return {"op": op, "tokens": _log_int(rng, 512, 2500), "text": rng.randint(64, 256)}


def _tokens(case):
    return case["t"] * case["h"] * case["w"] if case["op"] == "preattention" else case["tokens"]


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed))

    def normal(self, *shape, std=1.0, mean=0.0, dtype=torch.bfloat16):
        t = torch.randn(shape, generator=self.g, device=DEV, dtype=torch.float32)
        return t.mul_(std).add_(mean).to(dtype)

    def outliers(self, *shape, dtype=torch.bfloat16):
        """N(0, 1) with 0.1 % of the entries 50 times larger."""
        t = torch.randn(shape, generator=self.g, device=DEV, dtype=torch.float32)
        big = torch.rand(shape, generator=self.g, device=DEV) < 1e-3
        return torch.where(big, t * 50.0, t).to(dtype)

    def linear(self, n, k, input_scale, dtype=torch.bfloat16):
        """FP8 linear of a loaded model: e4m3 weight with a per-tensor scale."""
        w = torch.randn((n, k), generator=self.g, device=DEV, dtype=torch.float32).mul_(0.02)
        ws = (w.abs().amax() / 448.0).reshape(())
        codes = w.div_(ws).clamp_(-448.0, 448.0).to(FP8)
        s = input_scale if isinstance(input_scale, torch.Tensor) else torch.tensor(float(input_scale), device=DEV)
        return B.FP8Linear(codes, ws, s, self.normal(n, std=0.01, dtype=dtype))

    def timestep_tokens(self, tokens, width):
        """e(t) = a + t b with a t of its own for every token; the first
        three sixteenths (the clean prefix) share t = 0."""
        a = self.normal(width, std=0.5, dtype=torch.float32)
        b = self.normal(width, std=0.5, dtype=torch.float32)
        t = torch.rand((tokens, 1), generator=self.g, device=DEV)
        t[: tokens * 3 // 16] = 0.0
        return (a + t * b).to(torch.bfloat16).unsqueeze(0)


def _dtype(name):
    return {"bf16": torch.bfloat16, "fp16": torch.float16, "f32": torch.float32}[name]


def _rope(t, h, w, dtype=torch.bfloat16):
    return video_rope_cos_sin((t, h, w), heads=HEADS, head_dim=HEAD_DIM, device=DEV, dtype=dtype)


def prepare(case, seed):
    r, op, n = _Rand(seed), case["op"], _tokens(case)
    if op == "adazero":
        ts = r.normal(1, 1, 6 * C, std=0.5)
        return {"op": op, "x": r.normal(1, n, C), "table": r.normal(6, C, std=0.02, dtype=_dtype(case["table"])),
                "ts": ts.expand(1, n, 6 * C)}
    if op == "linear":
        x = r.outliers(1, n, case["k"], dtype=_dtype(case["dtype"]))
        scale = (x.float().abs().amax() / 448.0).reshape(())
        return {"op": op, "x": x, "lin": r.linear(case["n"], case["k"], scale, dtype=x.dtype)}
    if op == "ffn_down":
        return {"op": op, "x": r.normal(1, n, FF), "lin": r.linear(C, FF, 4.0 / 448)}
    if op == "preattention":
        cos, sin = _rope(case["t"], case["h"], case["w"], _dtype(case["rope"]))
        return {"op": op, "q": r.normal(1, n, C), "k": r.normal(1, n, C), "qw": r.normal(C, std=0.05, mean=1.0),
                "kw": r.normal(C, std=0.05, mean=1.0), "cos": cos, "sin": sin}
    if op == "attention":
        return {"op": op, "q": r.normal(1, n, C), "k": r.normal(1, case["keys"], C), "v": r.normal(1, case["keys"], C)}
    if op == "fp8_attention":
        return {"op": op, **{name: r.normal(1, n, HEADS, HEAD_DIM) for name in "qkv"}}
    if op == "residual_bias":
        return {"op": op, "x": r.normal(1, n, C), "y": r.normal(1, n, C), "bias": r.normal(C, std=0.01),
                "table": r.normal(9, C, std=0.02, dtype=_dtype(case["table"])), "ts": r.timestep_tokens(n, 9 * C)}

    def attention():
        return B.VideoAttention(
            to_q=r.linear(C, C, 8.0 / 448), to_k=r.linear(C, C, 8.0 / 448), to_v=r.linear(C, C, 8.0 / 448),
            to_out=r.linear(C, C, 2.0 / 448), q_norm_weight=r.normal(C, std=0.05, mean=1.0),
            k_norm_weight=r.normal(C, std=0.05, mean=1.0), heads=HEADS)

    # the linears' scales are a loaded model's: fixed
    L.set_frozen_fp8_scales(True)
    blk = B.VideoBlock(table=r.normal(9, C, std=0.02), prompt_table=r.normal(2, C, std=0.02), attn1=attention(),
                       attn2=attention(), ff_up=r.linear(FF, C, 8.0 / 448), ff_down=r.linear(C, FF, 4.0 / 448),
                       eps=EPS)
    cos, sin = _rope(n, 1, 1)
    text = case["text"]
    # the residual stream is larger than what one branch adds to it
    return {"op": op, "block": blk, "x": r.normal(1, n, C, std=2.0), "context": r.normal(1, text, C),
            "ts": r.normal(1, 1, 9 * C, std=0.5).expand(1, n, 9 * C),
            "pts": r.normal(1, 1, 2 * C, std=0.5).expand(1, text, 2 * C), "cos": cos, "sin": sin}


# --------------------------------------------------------------------------
# the call
# --------------------------------------------------------------------------
def run(s):
    op = s["op"]
    if op == "adazero":
        return L.fused_adazero_from_ada(s["x"], EPS, s["table"], s["ts"], shift_index=0, scale_index=1)
    if op == "linear":
        return L.fp8_linear_forward(s["lin"], s["x"])
    if op == "ffn_down":
        q = L.fused_gelu_tanh_fp8_quantize_e4m3(s["x"], s["lin"].input_scale)
        return L.fp8_linear_from_quantized_e4m3(s["lin"], q, out_dtype=s["x"].dtype)
    if op == "preattention":
        return L.fused_video_qk_rmsnorm_rope(s["q"], s["k"], s["qw"], s["kw"], EPS, s["cos"], s["sin"])
    if op == "attention":
        return A.attention_video(s["q"], s["k"], s["v"], HEADS)
    if op == "fp8_attention":
        (q, qs), (k, ks), (v, vs) = (L.fused_fp8_quantize_e4m3_per_head_4d(s[name]) for name in "qkv")
        return A.flash_attn_func(q, k, v, q_descale=qs, k_descale=ks, v_descale=vs)
    if op == "residual_bias":
        return L.fused_residual_gate_bias_from_ada(s["x"], s["y"], s["bias"], s["table"], s["ts"], gate_index=2)
    return B.video_block_forward(s["block"], s["x"], s["context"], s["ts"], s["pts"], s["cos"], s["sin"],
                                 fuse_gelu_quant=True, qkv_grouped=True, fuse_norm=True, fuse_ada_quant=True,
                                 fuse_residual_ada=True, fuse_out_quant=True)


# --------------------------------------------------------------------------
# what it cannot do without, and how far off it may be
# --------------------------------------------------------------------------
def work(case):
    op, n = case["op"], _tokens(case)
    row = 2 * n * C  # bytes of one bf16 activation
    if op == "adazero":
        return {"bytes": 2 * row + 4 * C * 2, "flops": 0}
    if op in ("linear", "ffn_down"):
        k, m = (FF, C) if op == "ffn_down" else (case["k"], case["n"])
        return {"bytes": 2 * n * k + m * k + 2 * m + 2 * n * m, "flops": 2.0 * n * m * k}
    if op == "preattention":
        rope = 4 if case["rope"] == "f32" else 2
        return {"bytes": 4 * row + 2 * n * HEADS * (HEAD_DIM // 2) * rope + 4 * C, "flops": 0}
    if op in ("attention", "fp8_attention"):
        keys = case.get("keys", n)
        return {"bytes": 2 * row + 4 * keys * C, "flops": 4.0 * n * keys * C}
    if op == "residual_bias":
        return {"bytes": 4 * row + 4 * C, "flops": 0}
    text = case["text"]
    flops = 2.0 * n * C * C * 6 + 4.0 * n * C * FF + 2.0 * text * C * C * 2 + 4.0 * n * n * C + 4.0 * n * text * C
    return {"bytes": 8 * C * C + 2 * C * FF + 2 * row + 2 * text * C + n * HEADS * HEAD_DIM * 2, "flops": flops}


def tolerance(case):
    """About four times the difference seen when the sums run in another
    order (K of a linear, the keys of an attention, or the block's tokens and
    prompt permuted; torch's own rms_norm for the norms)."""
    op = case["op"]
    if op == "residual_bias":
        return "exact"  # elementwise, every rounding prescribed
    if op in ("adazero", "preattention"):  # seen: 1.7e-5, one bf16 step
        return {"rel": 1e-4, "max": 6e-2}
    if op in ("linear", "ffn_down"):  # 5.2e-4, one bf16 step
        return {"rel": 2e-3, "max": 6e-2}
    if op == "attention":  # 3.1e-3, 0.019
        return {"rel": 1.2e-2, "max": 8e-2}
    if op == "fp8_attention":  # 0.033 (P in e4m3, rounded against another running max), 0.21
        return {"rel": 3e-2, "max": 8e-1}
    return {"rel": 3e-2, "max": 9e-1}  # 0.011, 0.3: re-quantized three times on the way


# --------------------------------------------------------------------------
# float64
# --------------------------------------------------------------------------
def _rms(x, weight=None):
    y = x / torch.sqrt(x.square().mean(dim=-1, keepdim=True) + EPS)
    return y if weight is None else y * weight.double()


def _ada(table, ts, i):
    ts = ts.reshape(ts.shape[0], ts.shape[1], table.shape[0], -1)
    return table[i].double() + ts[:, :, i, :].double()


def _quant(x, scale):
    """The FP8 linear's input quantizer, its roundings prescribed by x's dtype."""
    return torch.clamp(x * scale.reciprocal(), -448.0, 448.0).to(FP8)


def _mm(lin, codes, bias=True):
    w, rows = lin.weight.double(), codes.reshape(-1, codes.shape[-1])
    out = torch.cat([rows[i:i + 2048].double() @ w.t() for i in range(0, rows.shape[0], 2048)])
    out = (out * (lin.input_scale.double() * lin.weight_scale.double())).reshape(*codes.shape[:-1], -1)
    return out + lin.bias.double() if bias else out


def _rope64(x, cos, sin):
    b, n, _ = x.shape
    x = x.reshape(b, n, HEADS, HEAD_DIM).transpose(1, 2)
    first, second = x[..., : HEAD_DIM // 2], x[..., HEAD_DIM // 2:]
    cos, sin = cos.double(), sin.double()
    out = torch.cat([first * cos - second * sin, second * cos + first * sin], dim=-1)
    return out.transpose(1, 2).reshape(b, n, C)


def _attend(q, k, v):
    """q, k, v [1, N, HEADS, HEAD_DIM] in any dtype; one head at a time."""
    out = torch.empty((1, q.shape[1], HEADS, HEAD_DIM), device=DEV, dtype=torch.float64)
    for h in range(HEADS):
        kh, vh = k[0, :, h].double().t().contiguous(), v[0, :, h].double().contiguous()
        for i in range(0, q.shape[1], 4096):
            p = torch.softmax((q[0, i:i + 4096, h].double() @ kh) * HEAD_DIM ** -0.5, dim=-1)
            out[0, i:i + 4096, h] = p @ vh
    return out


def _heads(x):
    return x.reshape(1, -1, HEADS, HEAD_DIM)


def _per_head(x):
    scale = x.float().abs().amax(dim=(1, 3)).clamp_min(1e-12) / 448.0
    codes = torch.clamp(x.float() / scale[:, None, :, None], -448.0, 448.0).to(FP8)
    return codes.double() * scale.double()[:, None, :, None]


def exact(case, seed):
    s = prepare(case, seed)
    op = s["op"]
    bf = torch.bfloat16
    if op == "adazero":
        return _rms(s["x"].double()) * (1 + _ada(s["table"], s["ts"], 1)) + _ada(s["table"], s["ts"], 0)
    if op == "linear":
        return _mm(s["lin"], _quant(s["x"], s["lin"].input_scale))
    if op == "ffn_down":
        g = torch.nn.functional.gelu(s["x"], approximate="tanh")
        return _mm(s["lin"], _quant(g, s["lin"].input_scale))
    if op == "preattention":
        return (_rope64(_rms(s["q"].double(), s["qw"]), s["cos"], s["sin"]),
                _rope64(_rms(s["k"].double(), s["kw"]), s["cos"], s["sin"]))
    if op == "attention":
        return _attend(_heads(s["q"]), _heads(s["k"]), _heads(s["v"])).reshape(1, -1, C)
    if op == "fp8_attention":
        return _attend(_per_head(s["q"]), _per_head(s["k"]), _per_head(s["v"]))
    if op == "residual_bias":
        gate = _ada(s["table"], s["ts"], 2)
        return s["x"].double() + (s["y"].double() + s["bias"].double()) * gate
    # The block in float64 between its quantizers, whose inputs are bf16.
    blk = s["block"]
    x, a1, a2 = s["x"].double(), blk.attn1, blk.attn2

    def lin(layer, v, bias=True):
        return _mm(layer, _quant(v.to(bf), layer.input_scale), bias)

    def ada(i):
        return _ada(blk.table, s["ts"][:, :1], i)

    h = _rms(x) * (1 + ada(1)) + ada(0)
    q = _rope64(_rms(lin(a1.to_q, h), a1.q_norm_weight), s["cos"], s["sin"])
    k = _rope64(_rms(lin(a1.to_k, h), a1.k_norm_weight), s["cos"], s["sin"])
    o = _attend(_heads(q), _heads(k), _heads(lin(a1.to_v, h))).reshape(1, -1, C)
    x = x + lin(a1.to_out, o) * ada(2)
    h = _rms(x) * (1 + ada(7)) + ada(6)
    enc = s["context"].double() * (1 + _ada(blk.prompt_table, s["pts"], 1)) + _ada(blk.prompt_table, s["pts"], 0)
    q = _rms(lin(a2.to_q, h), a2.q_norm_weight)
    k = _rms(lin(a2.to_k, enc), a2.k_norm_weight)
    o = _attend(_heads(q), _heads(k), _heads(lin(a2.to_v, enc))).reshape(1, -1, C)
    x = x + lin(a2.to_out, o) * ada(8)
    h = _rms(x) * (1 + ada(4)) + ada(3)
    h = torch.nn.functional.gelu(lin(blk.ff_up, h), approximate="tanh")
    return x + lin(blk.ff_down, h) * ada(5)
