"""GPU parity at the full shapes of the benchmark configurations.

The small-shape parity tests give every wave of the token-row kernels a
single row. At the configured shapes the kernels stream several rows per
wave (AdaZero from 9216 tokens, the continuation ops at 14080 tokens), with
later rows' loads in flight and a short last group; these tests run those
schedules against the oracle, bit for bit, and assert from the library's own
schedule query that the multi-row path is reached. Inputs are drawn on the
CPU with seeded generators, so the oracle and the kernels see the same bits.

Shapes:
  AdaZero            (1, 2304, 4096), bf16 table, one timestep row for all
                     tokens; (1, 9216, 4096) and (1, 9217, 4096) (3 and 4 rows
                     per wave); (2, 1537, 4096) per-token timesteps with a
                     float32 table; (1, 2305, 4096) float32 timesteps
  continuation ops   (1, 14080, 4096) (workgroups streaming one or two rows)
                     and (1, 4999, 4096), per-token 9-row timestep embeddings
                     with a t = 0 prefix
  Q/K RMSNorm+RoPE   (1, 9216, 4096) with the (16, 18, 32) grid table
  per-head FP8       (1, 9216, 32, 128)
  FP8 quantizer      (9216, 4096) with 0.1 % outliers x50, amax/448 scale
  FP8 linear         9216 x 4096 -> 16384 (nine whole rounds), 16384 -> 4096
                     (a split-K tail) and 4096 -> 4096 (three whole rounds of
                     smaller tiles), grouped Q/K/V 4096 -> 3 x 4096: every
                     output against a full-size checker
                     (decoded e4m3 codes, a float32 device matmul, the
                     reference's two roundings), sampled rows against the
                     oracle (which also pins the checker there), the bias
                     epilogue on every element
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from oracle import ltx_ops as O
from oracle.numerics import T, bf16_round
from tests.helpers import assert_same_bits, gen, nan_canon, np32, randn, to_T

pytestmark = pytest.mark.gpu

DEV = "cuda"
C = 4096


@pytest.fixture(autouse=True)
def _strict(monkeypatch):
    monkeypatch.setenv("OPENGENIE_AMD_STRICT", "1")
    from opengenie_amd import ltx_ops

    ltx_ops.reset_hip_calls()
    yield


def _ran(name: str) -> None:
    from opengenie_amd import ltx_ops

    assert ltx_ops.collect_hip_calls().get(name, 0) > 0, f"{name} did not take the HIP path"


def g(t: torch.Tensor) -> torch.Tensor:
    return t.to(DEV)


def out_np(t: torch.Tensor) -> np.ndarray:
    torch.cuda.synchronize()
    return t.float().cpu().numpy()


def rows_per_wave(kind: int, batch: int, tokens: int) -> int:
    from opengenie_amd import _lib

    return int(_lib.load().oga_rows_per_wave(kind, batch, tokens, C))


def timestep_embeddings(tokens: int, params: int, prefix: int, seed: int) -> torch.Tensor:
    """(1, tokens, params*C) bf16: e(t) = a + t*b with t ~ U(0,1) per token and
    t = 0 for the first `prefix` tokens (the clean conditioning frames)."""
    gg = gen(seed)
    a = torch.randn((params * C,), generator=gg) * 0.5
    b = torch.randn((params * C,), generator=gg) * 0.5
    t = torch.rand((tokens, 1), generator=gg)
    t[:prefix] = 0.0
    out = torch.empty((1, tokens, params * C), dtype=torch.bfloat16)
    for r0 in range(0, tokens, 2048):  # bounded float32 temporaries
        out[0, r0:r0 + 2048] = (a + t[r0:r0 + 2048] * b).to(torch.bfloat16)
    return out


def ada_rows(table: torch.Tensor, ts: torch.Tensor, indices) -> tuple[T, T]:
    """The table rows and timestep rows of `indices` only, as oracle inputs
    (the kernels read the full tensors; the values are the same bits)."""
    b, n, w = ts.shape
    p = table.shape[0]
    sub = ts.view(b, n, p, w // p)[:, :, list(indices), :].reshape(b, n, len(indices) * (w // p))
    return to_T(table[list(indices)]), to_T(sub)


# ------------------------------------------------------------------ AdaZero
ADA_CASES = [
    # batch, tokens, table dtype, ts dtype, broadcast ts, several rows per wave
    (1, 2304, torch.bfloat16, torch.bfloat16, True, False),  # config 1 (one row per wave)
    (1, 9216, torch.bfloat16, torch.bfloat16, True, True),   # the 576p block shape, next row in flight
    (1, 9217, torch.float32, torch.bfloat16, True, True),    # ragged: waves with 4 and with 3 rows
    (2, 1537, torch.float32, torch.bfloat16, False, True),   # per-token timesteps, two batches
    (1, 2305, torch.bfloat16, torch.float32, True, False),   # float32 Ada values
]


@pytest.mark.parametrize("batch,tokens,tdt,sdt,bc,multi", ADA_CASES)
def test_adazero_from_ada_config_shape(batch, tokens, tdt, sdt, bc, multi):
    from opengenie_amd import _lib
    from opengenie_amd.ltx_ops import fused_adazero_from_ada

    rpw = rows_per_wave(_lib.ROWS_ADAZERO, batch, tokens)
    assert rpw >= (2 if multi else 1), rpw
    x = randn((batch, tokens, C), 20260101)
    table = randn((6, C), 20260102, dtype=tdt, std=0.02)
    ts = randn((batch, 1 if bc else tokens, 6 * C), 20260103, dtype=sdt, std=0.5)
    tsg = g(ts).expand(batch, tokens, 6 * C) if bc else g(ts)
    out = fused_adazero_from_ada(g(x), 1e-6, g(table), tsg, shift_index=0, scale_index=1)
    _ran("fused_adazero_from_ada")
    ref = O.adazero_from_ada(to_T(x), 1e-6, to_T(table), to_T(ts), 0, 1)
    assert_same_bits(out_np(out), bf16_round(ref.v), f"adazero {batch}x{tokens}")


# ------------------------------------------------------- continuation block
@pytest.fixture(scope="module", params=[(14080, 2640), (4999, 880)], ids=["14080", "4999"])
def continuation(request):
    tokens, prefix = request.param
    x = randn((1, tokens, C), 20260401)
    y = randn((1, tokens, C), 20260402)
    table = randn((9, C), 20260403, std=0.02)
    bias = randn((C,), 20260404, std=0.01)
    ts = timestep_embeddings(tokens, 9, prefix, 20260405)
    return {"tokens": tokens, "x": x, "y": y, "table": table, "bias": bias, "ts": ts,
            "gx": g(x), "gy": g(y), "gtable": g(table), "gbias": g(bias), "gts": g(ts)}


def _multi_row(tokens: int) -> None:
    """At the configured 14080 tokens some workgroups stream two rows (the
    loop over rows runs); 4999 tokens give every workgroup one row."""
    from opengenie_amd import _lib

    if tokens == 14080:
        assert rows_per_wave(_lib.ROWS_ELEMENTWISE, 1, tokens) >= 2


def test_adaln_affine_config_shape(continuation):
    from opengenie_amd.ltx_ops import fused_adaln_affine_from_ada

    c = continuation
    _multi_row(c["tokens"])
    out = fused_adaln_affine_from_ada(c["gx"], c["gtable"], c["gts"], shift_index=6, scale_index=7)
    _ran("fused_adaln_affine_from_ada")
    tab, ts = ada_rows(c["table"], c["ts"], (6, 7))
    ref = O.adaln_affine_from_ada(to_T(c["x"]), tab, ts, 0, 1)
    assert_same_bits(out_np(out), ref.v, "adaln affine")


def test_residual_gate_bias_config_shape(continuation):
    from opengenie_amd.ltx_ops import fused_residual_gate_bias_from_ada

    c = continuation
    _multi_row(c["tokens"])
    out = fused_residual_gate_bias_from_ada(c["gx"], c["gy"], c["gbias"], c["gtable"], c["gts"], gate_index=2)
    _ran("fused_residual_gate_bias_from_ada")
    tab, ts = ada_rows(c["table"], c["ts"], (2,))
    ref = O.residual_gate_bias_from_ada(to_T(c["x"]), to_T(c["y"]), to_T(c["bias"]), tab, ts, 0)
    assert_same_bits(out_np(out), ref.v, "residual gate + bias")


def test_residual_gate_config_shape(continuation):
    from opengenie_amd.ltx_ops import fused_residual_gate_from_ada

    c = continuation
    _multi_row(c["tokens"])
    out = fused_residual_gate_from_ada(c["gx"], c["gy"], c["gtable"], c["gts"], gate_index=8,
                                       count_video_ada=False)
    _ran("fused_residual_gate_from_ada")
    tab, ts = ada_rows(c["table"], c["ts"], (8,))
    ref = O.residual_gate_from_ada(to_T(c["x"]), to_T(c["y"]), tab, ts, 0)
    assert_same_bits(out_np(out), ref.v, "residual gate")


def test_mul_from_ada_config_shape(continuation):
    from opengenie_amd.ltx_ops import fused_mul_from_ada

    c = continuation
    out = fused_mul_from_ada(c["gx"], c["gtable"], c["gts"], gate_index=5)
    _ran("fused_mul_from_ada")
    tab, ts = ada_rows(c["table"], c["ts"], (5,))
    ref = O.mul_from_ada(to_T(c["x"]), tab, ts, 0)
    assert_same_bits(out_np(out), ref.v, "mul from ada")


# ------------------------------------------------------- Q/K preattention
def test_video_qk_rmsnorm_rope_config_shape():
    from opengenie_amd.ltx_ops import fused_video_qk_rmsnorm_rope
    from opengenie_amd.rope import video_rope_cos_sin

    n = 9216
    q = randn((1, n, C), 20260301)
    k = randn((1, n, C), 20260302)
    qw = randn((C,), 20260303, std=0.05, mean=1.0)
    kw = randn((C,), 20260304, std=0.05, mean=1.0)
    cos, sin = video_rope_cos_sin((16, 18, 32), heads=32, head_dim=128)
    oq, ok = fused_video_qk_rmsnorm_rope(g(q), g(k), g(qw), g(kw), 1e-6, g(cos), g(sin))
    _ran("fused_video_qk_rmsnorm_rope")
    rq, rk = O.video_qk_rmsnorm_rope(to_T(q), to_T(k), to_T(qw), to_T(kw), 1e-6, to_T(cos), to_T(sin))
    assert_same_bits(out_np(oq), rq.v, "q")
    assert_same_bits(out_np(ok), rk.v, "k")


# ------------------------------------------------------------ FP8 quantizers
def test_fp8_per_head_config_shape():
    from opengenie_amd.ltx_ops import fused_fp8_quantize_e4m3_per_head_4d

    x = randn((1, 9216, 32, 128), 20260501)
    q, s = fused_fp8_quantize_e4m3_per_head_4d(g(x))
    _ran("fused_fp8_quantize_e4m3_per_head_4d")
    torch.cuda.synchronize()
    qr, sr = O.fp8_per_head_quantize(np32(x))
    assert_same_bits(s.cpu().numpy(), sr, "per-head scale")
    assert np.array_equal(q.view(torch.uint8).cpu().numpy(), qr)


@pytest.mark.parametrize("zero_dim", [True, False])
def test_fp8_quantize_config_shape(zero_dim):
    """Config 2's input: (9216, 4096) ~N(0,1) with 0.1 % of the entries x50,
    scale = amax/448 (0-dim as the harness passes it, and (1,))."""
    from opengenie_amd.ltx_ops import fused_fp8_quantize_e4m3

    gg = gen(20260201)
    xf = torch.randn((9216, C), generator=gg)
    idx = torch.randperm(9216 * C, generator=gg)[: 9216 * C // 1000]
    xf.view(-1)[idx] *= 50.0
    x = xf.to(torch.bfloat16)
    s = (x.float().abs().amax() / 448.0).reshape(())
    if not zero_dim:
        s = s.reshape(1)
    q = fused_fp8_quantize_e4m3(g(x), g(s))
    _ran("fused_fp8_quantize_e4m3")
    torch.cuda.synchronize()
    ref = O.fp8_quantize_e4m3(to_T(x), float(s), zero_dim, device="cuda")
    got = q.view(torch.uint8).cpu().numpy()
    assert np.array_equal(nan_canon(got), nan_canon(ref))
    assert (np.abs(x.float().numpy()) > 40).sum() > 9216 * C // 5000  # the outliers are there


# ------------------------------------------------------------ FP8 linear at 9216 tokens
def _device_fp8_linear(a8: torch.Tensor, w8: torch.Tensor, sa: torch.Tensor, sb: torch.Tensor,
                       bias: torch.Tensor | None) -> torch.Tensor:
    """Full-size checker of the FP8 linear, fixed by the mathematics: e4m3
    codes decode exactly to float32 and every product of two e4m3 values is
    exact in float32, so a float32 device matmul (TF32 off) computes the
    reference's accumulator up to float32 summation rounding; then the
    reference's two roundings, R(acc * sa * sb) and R(out + R(bias))
    (triton_ltx_ops.py:1691-1709)."""
    prev = torch.backends.cuda.matmul.allow_tf32
    torch.backends.cuda.matmul.allow_tf32 = False
    try:
        acc = a8.float() @ w8.float().t()
    finally:
        torch.backends.cuda.matmul.allow_tf32 = prev
    out = (acc * (sa.float().reshape(()) * sb.float().reshape(()))).to(torch.bfloat16)
    del acc
    if bias is not None:
        out = (out.float() + bias.to(torch.bfloat16).float()).to(torch.bfloat16)
    return out


def _bf16_steps_t(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """Distance in bf16 steps between two bf16 tensors (monotone integer map
    of the bit patterns), on the device."""
    def key(x):
        u = x.contiguous().view(torch.int16).to(torch.int32) & 0xFFFF
        return torch.where(u >= 0x8000, 0x8000 - u, u)
    return (key(a) - key(b)).abs()


def _linear_full_check(got: torch.Tensor, ref: torch.Tensor, what: str) -> None:
    """The GEMM bar of _linear_rows_check on every output, on the device."""
    g32, r32 = got.float(), ref.float()
    close = torch.isclose(g32, r32, rtol=1e-2, atol=1e-3 * float(r32.abs().max()))
    far = int((~close).sum())
    steps = _bf16_steps_t(got, ref)
    over1 = float((steps > 1).float().mean())
    worst_far = int(steps[~close].max()) if far else 0
    print(f"{what}: {got.numel()} outputs, {far} outside rtol 1e-2 (worst {worst_far} steps), "
          f"{over1:.2e} more than one step away")
    assert far / got.numel() < 1e-5, (what, far)
    assert worst_far <= 2, (what, worst_far)
    assert over1 < 1e-2, (what, over1)


def _linear_rows_check(got_rows: np.ndarray, ref_rows: np.ndarray) -> None:
    """The FP8 linear's bar against the float64-accumulated oracle (as the
    small-shape tests): rtol 1e-2 with an outlier allowance of 1e-5 at most
    two bf16 steps (the MFMA's own accumulation rounding next to a power of
    two), and fewer than 1 % of outputs more than one step away."""
    from tests.helpers import bf16_ulp_distance

    close = np.isclose(got_rows, ref_rows, rtol=1e-2, atol=1e-3 * float(np.abs(ref_rows).max()))
    assert (~close).mean() < 1e-5, int((~close).sum())
    assert (bf16_ulp_distance(got_rows[~close], ref_rows[~close]) <= 2).all()
    assert (bf16_ulp_distance(got_rows, ref_rows) > 1).mean() < 1e-2


@pytest.mark.parametrize("n,k", [(16384, 4096), (4096, 16384), (4096, 4096)],
                         ids=["up_4096_to_16384", "down_16384_to_4096", "proj_4096_to_4096"])
def test_fp8_linear_config_shapes(n, k):
    """The FP8 linear at 9216 tokens on the schedules the benchmark times:
    4096 -> 16384 is 2304 tiles, nine whole rounds of the persistent kernel on
    256 CUs; 16384 -> 4096 two whole rounds, then 64 tiles in 4 K-chunks and
    their reduce; 4096 -> 4096 three whole rounds of 192 x 256. Config 2's data: x ~N(0,1) with
    0.1 % of the entries x50, per-tensor amax/448 scales, W from N(0,0.02),
    bf16 bias ~N(0,0.01). Every output against the full-size device checker
    at the GEMM bar; every 127th row (and the last) against the oracle, and
    the checker against the oracle on those rows; every element of the
    biased output equal to R(out_nobias + R(bias)) from the unbiased call on
    the same schedule."""
    from opengenie_amd import _lib
    from opengenie_amd.ltx_ops import fp8_scaled_mm

    m = 9216
    lib = _lib.load()
    plan = (ctypes.c_int64 * 4)()
    ws_bytes = int(lib.oga_fp8_linear_workspace_bytes(m, n, k))
    assert lib.oga_fp8_linear_plan(m, n, k, ws_bytes, 0, plan) == 0
    split = plan[3] > 1
    assert split == (ws_bytes > 0) == (k == 16384)
    assert tuple(plan) == {(16384, 4096): (256, 256, 2304, 1), (4096, 16384): (256, 256, 512, 4),
                           (4096, 4096): (192, 256, 768, 1)}[n, k]
    gg = gen(20260601 + n + k)
    xf = torch.randn((m, k), generator=gg)
    idx = torch.randperm(m * k, generator=gg)[: m * k // 1000]
    xf.view(-1)[idx] *= 50.0
    x = xf.to(torch.bfloat16)
    sa = (x.float().abs().amax() / 448.0).reshape(())
    a = torch.clamp(x.float() / sa, -448, 448).to(torch.float8_e4m3fn)
    wf = torch.randn((n, k), generator=gg) * 0.02
    sb = (wf.abs().amax() / 448.0).reshape(())
    w = torch.clamp(wf / sb, -448, 448).to(torch.float8_e4m3fn)
    bias = (torch.randn((n,), generator=gg) * 0.01).to(torch.bfloat16)
    ga, gw, gsa, gsb, gb = g(a), g(w), g(sa), g(sb), g(bias)
    out = fp8_scaled_mm(ga, gw, gsa, gsb, gb)
    out0 = fp8_scaled_mm(ga, gw, gsa, gsb, None)
    _ran("fp8_scaled_mm")
    want = (out0.float() + gb.float()).to(torch.bfloat16)  # R(out_nobias + R(bias)), bias already bf16
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
    del out0, want
    full = _device_fp8_linear(ga, gw, gsa, gsb, gb)
    _linear_full_check(out, full, f"FP8 linear 9216x{k}->{n}")
    rows = np.unique(np.concatenate([np.arange(0, m, 127), [m - 1]]))
    a_codes = a.view(torch.uint8).numpy()
    ref = O.fp8_linear(a_codes[rows], w.view(torch.uint8).numpy(), float(sa), float(sb), to_T(bias))
    got = out_np(out)[rows]
    _linear_rows_check(got, ref)
    _linear_rows_check(out_np(full)[rows], ref)  # the checker itself, against the oracle


def test_fp8_grouped_qkv_config_shape():
    """The grouped Q/K/V projection at 9216 tokens (one launch over the 1728
    tiles of the three 4096 -> 4096 linears, 6.75 rounds of the CUs, no split)
    with each linear's own weight scale and bias: every output of q, k and v
    against the full-size device checker, every 127th row against the oracle
    at the GEMM bar."""
    from opengenie_amd import ltx_ops as L
    from opengenie_amd.block import random_video_block

    blk = random_video_block(C, 32, seed=41, gated=False)
    a = blk.attn1
    x = (torch.randn((1, 9216, C), generator=gen(20260611))).to(torch.bfloat16)
    qkv = L.fp8_qkv_from_grouped_mm(a, g(x))
    assert qkv is not None
    _ran("fp8_grouped_linear")
    rows = np.unique(np.concatenate([np.arange(0, 9216, 127), [9215]]))
    for lin, got_t in zip((a.to_q, a.to_k, a.to_v), qkv):
        # the input codes as torch computes them on the GPU (x times the
        # float32 reciprocal of the 0-dim scale; torch's CPU division differs
        # in about 2 % of the codes)
        s_in = float(lin.input_scale.float().cpu())
        xq = O.fp8_quantize_e4m3(to_T(x), s_in, True, device="cuda").reshape(9216, C)
        ref = O.fp8_linear(xq[rows], lin.weight.cpu().view(torch.uint8).numpy(), s_in,
                           float(lin.weight_scale.float().cpu()), to_T(lin.bias.cpu()))
        got = out_np(got_t).reshape(9216, -1)[rows]
        _linear_rows_check(got, ref)
        xq_d = torch.from_numpy(xq).to(DEV).view(torch.float8_e4m3fn)
        full = _device_fp8_linear(xq_d, lin.weight, lin.input_scale, lin.weight_scale, lin.bias)
        _linear_full_check(got_t.reshape(9216, -1), full, "grouped Q/K/V 9216x4096->4096")
