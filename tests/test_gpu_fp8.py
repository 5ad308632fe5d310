"""BASELINE config 4 at its real size: the FP8 e4m3fn W8A8 linears of one decoder layer on
8 x 1024 packed prefill tokens (M = 8192), FP8Linear (kernels/fp8_linear.py:66-126) against
the oracle on the same quantised operands.

Shapes (K -> N): QKV 1536 -> 2048 (with the q|k|v bias), O 1536 -> 1536, gate/up
1536 -> 17920, down 8960 -> 1536; x ~ N(0, 1) fp16, W ~ N(0, 0.02) fp16 (config 4).  At
M = 8192 every config-4 shape runs a persistent grid of 256-row big tiles (gate/up: 32 x 70
tiles of 256 x 256 on 256 workgroups, 9 rounds; O and down 256 tiles of 256 x 192, one
per CU); the 256 x 128 pipeline takes the down shape at M = 4096 (big tiles would fill half
the grid) and a ragged M (a partial tile in the last round); K < 512 takes the
one-tile-per-workgroup kernel.  ``omni_fp8_gemm_plan`` names the kernel and grid each case
runs, so the test states which path it covered.

The oracle's product is computed for 8 rows of every 256-row block (one row in each of
the four 64-row wave bands, several 16-row sub-tiles and lane positions) and every column:
every output tile of every round is compared.  All M rows are checked against a
size-independent property: sum_n y[m, n] equals sa[m] * (xq[m] . (Wq^T sw)) up to the
roundings of each term."""

import pytest
import torch

from oracle import qwen2_ref as ref

pytestmark = pytest.mark.gpu

KIND = {0: "one tile per workgroup", 1: "pipelined 256x128 persistent",
        2: "persistent 256x256 tiles", 3: "persistent 256x192 tiles"}
COLS = {0: 128, 1: 128, 2: 256, 3: 192}
BLOCK_ROWS = (0, 17, 63, 98, 133, 228, 239, 255)    # within each 256-row block


def say(msg):
    print(f"[gpu-test] {msg}", flush=True)


def f16(shape, seed, std=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * std).to(torch.float16)


def sample_rows(M):
    rows = sorted({b + r for b in range(0, M, 256) for r in BLOCK_ROWS if b + r < M} | {M - 1})
    return torch.tensor(rows, dtype=torch.long)


def plan(M, N, K):
    from omniserver_amd._lib import lib
    import ctypes
    g = ctypes.c_int(0)
    kind = lib().omni_fp8_gemm_plan(M, N, K, ctypes.byref(g))
    return kind, g.value


def abs_product(xq, sa, wq, sw):
    return (xq.float().abs() @ wq.float().abs().t()) * sa.view(-1, 1) * sw.view(1, -1)


CASES = [
    # name, M, K, N, bias
    ("qkv", 8192, 1536, 2048, True),
    ("o", 8192, 1536, 1536, False),
    ("gate_up", 8192, 1536, 17920, False),
    ("gate_up biased", 8192, 1536, 17920, True),   # 192-column tail tiles with biases
    ("down", 8192, 8960, 1536, False),
    ("256-wide", 8192, 4096, 2048, True),
    ("down half grid", 4096, 8960, 1536, False),
    ("gate_up ragged", 8192 + 100, 1536, 17920, False),
    ("down ragged", 2000, 8960, 1536, True),
    ("short K", 1000, 384, 2048, True),
]


@pytest.mark.parametrize("name,M,K,N,bias", CASES, ids=[c[0] for c in CASES])
def test_fp8_config4_linear(gpu, name, M, K, N, bias):
    from omniserver_amd.linear import FP8Linear
    kind, grid = plan(M, N, K)
    tiles = -(-M // (256 if kind else 128)) * (N // COLS[kind])
    say(f"fp8 {name}: M={M} K={K} N={N} bias={bias} -> {KIND[kind]}, grid {grid}, "
        f"{tiles} tiles ({-(-tiles // grid)} rounds)")
    W = f16((N, K), 400 + N % 97, 0.02)
    b = f16((N,), 401, 0.02) if bias else None
    x = f16((M, K), 402 + K % 89)
    lin = FP8Linear(W.to(gpu), None if b is None else b.to(gpu), rowwise=True)
    y = lin(x.to(gpu)).cpu()
    torch.cuda.synchronize()
    wq, sw = ref.fp8_weight_rowwise(W.float())
    assert torch.equal(lin.weight_fp8.cpu(), wq.view(torch.uint8))
    xq, sa = ref.quant_fp8(x.float())

    # every tile: sampled rows, all columns, against the oracle
    rows = sample_rows(M)
    e = ref.fp8_linear_rowwise(xq[rows], sa[rows], wq, sw, None if b is None else b.float())
    e0 = ref.fp8_linear_rowwise(xq[rows], sa[rows], wq, sw, None)
    yc = y[rows].float()
    d = (yc - e).abs()
    tol = (e0.abs() * 2.0 ** -7 + e.abs() * 2.0 ** -10
           + abs_product(xq[rows], sa[rows], wq, sw) * 2.0 ** -14)
    assert (d <= tol + 1e-6).all(), (d - tol).max().item()
    same = (d == 0).float().mean().item()
    assert same > 0.95, same

    # every row: the row sum against the closed form (each output within one bf16 step,
    # one fp16 step and the bias rounding of its exact value)
    exact_sum = sa.view(-1) * (xq.float() @ (wq.float().t() @ sw))
    if b is not None:
        exact_sum = exact_sum + b.float().sum()
    ysum = y.float().sum(1)
    ymag = y.float().abs().sum(1)
    bound = (ymag * (2.0 ** -8 + 2.0 ** -10) + 1e-3
             + (xq.float().abs() @ (wq.float().abs().t() @ sw)) * sa.view(-1) * 2.0 ** -14)
    assert ((ysum - exact_sum).abs() <= bound).all(), ((ysum - exact_sum).abs() - bound).max()
    say(f"fp8 {name}: {len(rows)} sampled rows x {N} columns, {100 * same:.2f}% bit-equal; "
        f"{M} row sums within bounds")


def test_fp8_prequant_bias_bf16(gpu):
    """forward_prequant with a bias (fp8_linear.py:99-108): bf16 product + bias.to(bf16) as
    a bf16 add, at a size that runs the persistent pipelined kernel."""
    from omniserver_amd import fused_ops as F
    from omniserver_amd.linear import FP8Linear
    M, H, N = 1024, 1536, 4096
    say(f"fp8 prequant + bias M={M} N={N}")
    x, r = f16((M, H), 410), f16((M, H), 411)
    w = torch.ones(H, dtype=torch.float16)
    W = f16((N, H), 412, 0.02)
    b = f16((N,), 413, 0.05)
    lin = FP8Linear(W.to(gpu), b.to(gpu), rowwise=True)
    q, s, _ = F.add_rms_norm_fp8(x.to(gpu), r.to(gpu), w.to(gpu), 1e-6)
    y = lin.forward_prequant(q, s)
    torch.cuda.synchronize()
    assert y.dtype == torch.bfloat16
    wq, sw = ref.fp8_weight_rowwise(W.float())
    qc = q.cpu().view(torch.float8_e4m3fn)
    e = ref.fp8_linear_prequant(qc, s.cpu(), wq, sw, b.float())
    e0 = ref.fp8_linear_prequant(qc, s.cpu(), wq, sw, None)
    d = (y.cpu().float() - e).abs()
    tol = (e0.abs() + e.abs()) * 2.0 ** -7 + abs_product(qc, s.cpu(), wq, sw) * 2.0 ** -14
    assert (d <= tol + 1e-6).all(), (d - tol).max().item()
    assert (d == 0).float().mean().item() > 0.95


def test_bf16_rounding_exhaustive(gpu):
    """The FP8 epilogues round to bf16 with the device's packed conversion: on every one of
    the 2^32 float bit patterns it equals the integer round-to-nearest-even with quieted NaNs
    (the rounding of the reference's bf16 outputs), NaN inputs included."""
    from omniserver_amd._lib import call, ptr, stream
    say("bf16 rounding: all 2^32 float inputs")
    mism = torch.zeros(2, device=gpu, dtype=torch.int64)
    call("omni_bf16_rne_check", ptr(mism), stream())
    torch.cuda.synchronize()
    assert mism.tolist() == [0, 0]


def test_fp8_codes_exhaustive(gpu):
    """The quantisers' hardware e4m3 conversion against the integer rounding on every fp32 value
    that is not NaN, and their corrected quotients against fp32 division: every pair of
    significands for 11-bit numerators, 2^31 pairs for 24-bit ones."""
    from omniserver_amd._lib import call, ptr, stream
    say("e4m3 conversion on all fp32 inputs, quotients on all significand pairs")
    mism = torch.zeros(3, dtype=torch.int64, device=gpu)
    call("omni_fp8_codes_check", ptr(mism), stream())
    torch.cuda.synchronize()
    assert mism.tolist() == [0, 0, 0]


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("M,K,N", [(1, 512, 128), (16, 640, 2048), (17, 8960, 1536),
                                   (64, 8960, 1536), (65, 1536, 2048), (130, 8960, 1536),
                                   (300, 1536, 1536), (33, 1536, 17920), (1000, 8960, 1536)])
def test_fp8_few_rows(gpu, M, K, N, bias):
    """The few-row kernel in each of its forms (row blocks with one row and one row short of
    full, K steps that do not divide over its waves, more than one round of workgroups) and
    every output form, against a float64 product of the same codes: the MFMA's reduced
    intermediate precision (2^-14 of the absolute product) and the output's roundings; the
    output's padding columns stay untouched."""
    from omniserver_amd.linear import FP8Linear
    kind, grid = plan(M, N, K)
    say(f"fp8 few rows M={M} K={K} N={N} bias={bias} -> kind {kind}, grid {grid}")
    assert kind == 4
    b = f16((N,), 410, 0.5).to(gpu) if bias else None
    lin = FP8Linear(f16((N, K), 411, 0.02).to(gpu), b, rowwise=True)
    xq, sa = lin.quantize_input(f16((M, K), 412).to(gpu))
    e4 = lambda t: t.view(torch.float8_e4m3fn).double()
    sc = sa.double().view(-1, 1) * lin.weight_scale.double().view(1, -1)
    v = e4(xq) @ e4(lin.weight_fp8).t() * sc
    mag = e4(xq).abs() @ e4(lin.weight_fp8).abs().t() * sc
    bb = b.double() if bias else torch.zeros(N, device=gpu, dtype=torch.float64)
    for mode, eps in ((lin.OUT_F16_VIA_BF16, 2.0 ** -8), (lin.OUT_BF16, 2.0 ** -8),
                      (lin.OUT_F16, 2.0 ** -11)):
        dt = torch.bfloat16 if mode == lin.OUT_BF16 else torch.float16
        buf = torch.full((M, N + 4), 5.0, device=gpu, dtype=dt)
        lin.gemm_out(xq, sa, buf[:, :N], mode)
        d = (buf[:, :N].double() - (v + bb)).abs()
        # v, b (bf16 form) and their sum each rounded once, plus v's fp16 rounding
        tol = mag * 2.0 ** -14 + (eps + 2.0 ** -11) * (2 * v.abs() + 2 * bb.abs()) + 1e-6
        assert (d <= tol).all(), (mode, (d - tol).max().item())
        assert (buf[:, N:] == 5.0).all()


@pytest.mark.parametrize("ldo", [2 ** 22 + 4, 2 ** 25 + 4])
def test_fp8_big_tiles_wide_rows(gpu, ldo):
    """A ragged shape of the big tiles whose output rows are further apart than their 32-bit
    offsets reach: bit-equal to the same product in packed rows, in every output form; the
    SiLU form refuses such rows."""
    from omniserver_amd._lib import lib, ptr, stream
    from omniserver_amd.linear import FP8Linear
    M, N, K = 300, 36864, 1024
    assert plan(M, N, K)[0] in (2, 3)
    say(f"fp8 big tiles wide rows ldo={ldo}")
    lin = FP8Linear(f16((N, K), 420, 0.02).to(gpu), f16((N,), 421).to(gpu), rowwise=True)
    xq, sa = lin.quantize_input(f16((M, K), 422).to(gpu))
    buf = torch.empty((M - 1) * ldo + N, device=gpu, dtype=torch.float16)
    for mode in (lin.OUT_F16_VIA_BF16, lin.OUT_BF16, lin.OUT_F16):
        dt = torch.bfloat16 if mode == lin.OUT_BF16 else torch.float16
        wide = buf.view(dt).as_strided((M, N), (ldo, 1))
        lin.gemm_out(xq, sa, wide, mode)
        want = lin.gemm_out(xq, sa, torch.empty(M, N, device=gpu, dtype=dt), mode)
        assert torch.equal(wide.contiguous().view(torch.int16), want.view(torch.int16)), mode
    assert lib().omni_fp8_gemm_silu_grid(M, N, K) > 0
    assert lib().omni_fp8_gemm_silu(ptr(xq), ptr(sa), ptr(lin.weight_fp8), ptr(lin.weight_scale),
                                    ptr(buf), ldo, None, M, N, K, lin.OUT_BF16, stream()) == -2
