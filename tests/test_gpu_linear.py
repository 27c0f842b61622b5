"""GPU parity: block_fp8_linear (fp8.py:254-299) and the SwiGLU epilogue."""

from __future__ import annotations

import ctypes
import hashlib
import json
from pathlib import Path

import numpy as np
import pytest

from conftest import assert_parity, from_bits, random_codes, submodule, to_bits

pytestmark = pytest.mark.gpu
GOLDEN = Path(__file__).resolve().parent / "golden"


def _linear(M, dev, x_bits, codes, scale):
    import torch

    x = from_bits(x_bits, dev)
    w = torch.from_numpy(codes).to(dev)
    s = torch.from_numpy(scale).to(dev)
    return to_bits(M.block_fp8_linear(x, w, s))


def test_config1_gemv_matches_oracle(M, O, dev):
    """x bf16 [1,4096] ~N(0,1), W E4M3 [4096,4096] from N(0,0.02)."""
    rng = np.random.default_rng(1)
    w = rng.normal(0.0, 0.02, size=(4096, 4096)).astype(np.float32)
    codes, scale = O.quantize_e4m3_blocks(w)
    x = O.f32_to_bf16(rng.normal(size=(1, 4096)).astype(np.float32))
    got = _linear(M, dev, x, codes, scale)
    want = O.fp8_linear(x, codes, scale)
    assert_parity(got, want, O, exact_fraction=0.97)


@pytest.mark.parametrize("k,n", [(1024, 256), (1536, 512), (2048, 130), (4096, 64)])
def test_gemv_random_codes_decode_like_reference_lut(M, O, dev, k, n):
    """Random codes 0..246 include 0x7F, which the reference LUT decodes to
    480 (fp8.py:22-27); the exact E4M3->FP16 register decode must agree."""
    rng = np.random.default_rng(k + n)
    codes = random_codes(rng, (n, k))
    scale = (rng.uniform(size=(-(-n // 128), k // 128)) * 0.002).astype(np.float32)
    x = O.f32_to_bf16((rng.normal(size=(1, k)) * 2).astype(np.float32))
    got = _linear(M, dev, x, codes, scale)
    want = O.fp8_linear(x, codes, scale)
    assert_parity(got, want, O, exact_fraction=0.98)


@pytest.mark.parametrize("k,n", [(12288, 200), (16384, 130), (65536, 8)])
@pytest.mark.parametrize("with_480", [False, True])
def test_wide_gemv_split_k_matches_oracle(M, O, dev, k, n, with_480):
    """One-row linear with K a multiple of 4096 above 8192 (an attention
    output projection is 16384 wide): one wavefront per 4096-wide K part,
    parts added in order.  Codes with 0x7F/0xFF take the exact software
    decode, codes without them the hardware one."""
    rng = np.random.default_rng(k + n + with_480)
    if with_480:
        codes = random_codes(rng, (n, k))
    else:
        codes = (rng.integers(0, 0x7F, size=(n, k)) | (rng.integers(0, 2, size=(n, k)) << 7)).astype(np.uint8)
    scale = (rng.uniform(size=(-(-n // 128), k // 128)) * 0.002).astype(np.float32)
    x = O.f32_to_bf16((rng.normal(size=(1, k)) * 2).astype(np.float32))
    got = _linear(M, dev, x, codes, scale)
    want = O.fp8_linear(x, codes, scale)
    assert_parity(got, want, O, exact_fraction=0.98)


def test_reference_kat_non_aligned_129x257(M, O, dev):
    """tests/test_fp8_metal.py:23-39: 129 x 257 crosses both block edges;
    error vs the dequantised matmul <= 0.03125."""
    rng = np.random.default_rng(7)
    m, k = 129, 257
    codes = random_codes(rng, (m, k))
    scale = (rng.uniform(size=(2, 3)) * 0.02).astype(np.float32)
    x = O.f32_to_bf16(rng.normal(size=(2, k)).astype(np.float32))
    got = _linear(M, dev, x, codes, scale)
    dense = O.dequantize(codes, scale)
    expected = O.f32_to_bf16((O.bf16_to_f32(x).astype(np.float64) @ dense.T).astype(np.float32))
    err = np.max(np.abs(O.bf16_to_f32(got) - O.bf16_to_f32(expected)))
    assert err <= 0.03125
    assert_parity(got, O.fp8_linear(x, codes, scale), O, exact_fraction=0.97)


@pytest.mark.parametrize("rows", [2, 7, 8, 9, 33, 100])
def test_multi_row_mfma_path_matches_oracle(M, O, dev, rows):
    """M > 1 with K % 128 == 0 runs the FP8 MFMA GEMM on the exact hi/lo
    activation split; the result must match the FP32-exact oracle."""
    rng = np.random.default_rng(rows)
    k, n = 512, 144
    w = rng.normal(0.0, 0.02, size=(n, k)).astype(np.float32)
    codes, scale = O.quantize_e4m3_blocks(w)
    x = O.f32_to_bf16(rng.normal(size=(rows, k)).astype(np.float32))
    got = _linear(M, dev, x, codes, scale)
    assert_parity(got, O.fp8_linear(x, codes, scale), O, exact_fraction=0.97)


@pytest.mark.parametrize("with_480", [False, True])
@pytest.mark.parametrize("rows,k", [(2, 128), (17, 4224), (250, 1152), (499, 1152), (999, 1152), (1999, 640),
                                    (2800, 256), (4801, 384), (11000, 128), (16500, 256)])
def test_dense_tiles_ragged_edges_match_oracle(M, O, dev, rows, k, with_480):
    """Row counts that take one output tile of the several-row linear after
    the other at 272 columns (16 x 16 to 64 x 128, then 128 x 256 and 128 x 512),
    the last row and column tiles ragged, K of 1 to 33 blocks.
    Without a code flag a few 0x7F / 0xFF in one tile must be found."""
    rng = np.random.default_rng(rows + k)
    n = 272
    codes = (rng.integers(0, 0x7F, size=(n, k)) | (rng.integers(0, 2, size=(n, k)) << 7)).astype(np.uint8)
    if with_480:
        codes[0, 0], codes[n - 1, k - 1], codes[40, 64] = 0x7F, 0xFF, 0xFF
    scale = (rng.uniform(size=(-(-n // 128), k // 128)) * 0.002).astype(np.float32)
    x = O.f32_to_bf16(rng.normal(size=(rows, k)).astype(np.float32))
    assert_parity(_linear(M, dev, x, codes, scale), O.fp8_linear(x, codes, scale), O, exact_fraction=0.95)


@pytest.mark.parametrize("rows,k", [(17, 3712), (17, 9344), (250, 4224), (250, 9344), (499, 4224), (499, 3712),
                                    (999, 4224), (999, 3712)])
def test_few_row_tiles_over_long_k_match_oracle(M, O, dev, rows, k):
    """16 x 16, 16 x 32, 32 x 32 and 32 x 64 tiles through more than one turn
    of their K loop and several folds, the last step of K whole or ragged over
    the wavefronts; 0x7F / 0xFF in a middle and in the last K block, found
    without a code flag."""
    rng = np.random.default_rng(rows + k)
    n = 272
    codes = (rng.integers(0, 0x7F, size=(n, k)) | (rng.integers(0, 2, size=(n, k)) << 7)).astype(np.uint8)
    scale = (rng.uniform(size=(-(-n // 128), k // 128)) * 0.002).astype(np.float32)
    x = O.f32_to_bf16(rng.normal(size=(rows, k)).astype(np.float32))
    assert_parity(_linear(M, dev, x, codes, scale), O.fp8_linear(x, codes, scale), O, exact_fraction=0.95)
    codes[3, k // 2], codes[100, k - 1], codes[n - 1, k - 128] = 0x7F, 0xFF, 0x7F
    assert_parity(_linear(M, dev, x, codes, scale), O.fp8_linear(x, codes, scale), O, exact_fraction=0.95)


@pytest.mark.parametrize("marked", ["none", "gate_proj", "up_proj"])
@pytest.mark.parametrize("rows", [33, 150, 300])
def test_mlp_over_long_k_equals_its_parts_and_the_oracle(M, O, dev, rows, marked):
    """The 16 x 32, 32 x 32 and 32 x 64 SwiGLU tiles through 33 K blocks: the
    bytes of the projections called in turn, with the code flags and without
    (0x7F / 0xFF in a middle and in the last K block, looked for), and the
    oracle's chain."""
    import torch

    hidden, inter, limit = 4224, 640, 2.0
    gen = torch.Generator().manual_seed(rows)
    mlp = M.ClampedMLP(hidden, inter, limit, device=dev)
    for name in ("gate_proj", "up_proj", "down_proj"):
        proj = getattr(mlp, name)
        codes = torch.randint(0, 0x7F, tuple(proj.weight.shape), generator=gen, dtype=torch.uint8)
        codes |= torch.randint(0, 2, tuple(codes.shape), generator=gen, dtype=torch.uint8) << 7
        if name == marked:
            codes[7, hidden // 2], codes[-1, -1], codes[200, -128] = 0x7F, 0xFF, 0x7F
        proj.weight.copy_(codes)
        proj.weight_scale_inv.copy_(torch.rand(tuple(proj.weight_scale_inv.shape), generator=gen) * 0.002)
    x = torch.randn((rows, hidden), generator=gen).to(dev, torch.bfloat16)
    y = mlp(x)
    parts = mlp.down_proj(M.swiglu(mlp.gate_proj(x), mlp.up_proj(x), limit))
    assert mlp._one_call(x) and torch.equal(y.view(torch.int16), parts.view(torch.int16))
    N = submodule("_native")
    plain = mlp.as_c_struct()
    for linear in (plain.gate, plain.up, plain.down):
        linear.code_flags = None
    size = N.lib().glm53_mlp_workspace_bytes(rows, hidden, inter)
    ws, looked = N.workspace(size, dev), torch.empty_like(y)
    N.check(N.lib().glm53_mlp(ctypes.byref(plain), limit, N.ptr(x), rows, N.ptr(looked), N.ptr(ws), size,
                              N.stream_handle(dev)))
    assert torch.equal(looked.view(torch.int16), y.view(torch.int16))
    at = [(p.weight.cpu().numpy(), p.weight_scale_inv.cpu().numpy()) for p in (mlp.gate_proj, mlp.up_proj, mlp.down_proj)]
    bits = to_bits(x)
    h = O.swiglu(O.fp8_linear(bits, *at[0]), O.fp8_linear(bits, *at[1]), limit)
    want = O.fp8_linear(h, *at[2])
    assert_parity(to_bits(y), want, O, elementwise=False)
    # An output of one step (2^-7) apart, plus what the hidden values bring:
    # about 2.4% of them are a step off (1.2% of gate and of up each), so the
    # sum is off by sqrt(0.024) 2^-7 = 1.2e-3 of the outputs' RMS (one
    # deviation); six of them.
    got, want = O.bf16_to_f32(to_bits(y)).astype(np.float64), O.bf16_to_f32(want).astype(np.float64)
    assert (np.abs(got - want) <= 2.0 ** -7 * np.abs(want) + 7.3e-3 * np.sqrt(np.mean(want ** 2))).all()


@pytest.mark.parametrize("with_480", [False, True])
@pytest.mark.parametrize("rows,n,k", [(450, 4112, 256), (1100, 4112, 256), (2100, 4112, 128), (190, 4112, 1664),
                                      (195, 4112, 1664), (1500, 3088, 256), (600, 2064, 384), (230, 8208, 2176),
                                      (300, 8208, 4224), (33, 16400, 2176), (2, 65552, 1024), (32, 65552, 896),
                                      (33, 65552, 1024), (3, 131088, 128), (40, 131088, 128)])
def test_dense_tile_rule_on_wide_outputs_matches_oracle(M, O, dev, rows, n, k, with_480):
    """Both sides of the tile rule's lines: 128 x 128 and wider over many
    columns, 32 x 128 by its rows, 64 x 128 by columns, matrix size and row
    groups, few rows over more columns than a round of 128 x 256 holds; the
    last row and column tiles ragged.  Checked on 64 of the rows and a run of
    columns at either end and in the middle (columns do not mix), taken
    together: about 1.2% of the outputs lie one BF16 step off, and over the
    544 outputs of the smallest case 5% is more than five deviations away."""
    rng = np.random.default_rng(rows + n + k)
    codes = rng.integers(0, 0x7F, size=(n, k), dtype=np.uint8)
    if with_480:
        codes[0, 0], codes[n - 1, k - 1], codes[n // 2, k // 2] = 0x7F, 0xFF, 0xFF
    scale = (rng.uniform(size=(-(-n // 128), k // 128)) * 0.002).astype(np.float32)
    x = O.f32_to_bf16(rng.normal(size=(rows, k)).astype(np.float32))
    got = _linear(M, dev, x, codes, scale)
    keep = np.unique(np.concatenate([np.arange(min(rows, 8)), np.linspace(0, rows - 1, 48, dtype=int),
                                     np.arange(max(rows - 8, 0), rows)]))
    runs = [slice(c0, min(c0 + 128, n)) for c0 in (0, n // 256 * 128, (n - 1) // 128 * 128)]
    want = [O.fp8_linear(x[keep], codes[c], scale[c.start // 128:c.start // 128 + 1]) for c in runs]
    assert_parity(np.concatenate([got[keep, c] for c in runs], axis=1), np.concatenate(want, axis=1), O,
                  exact_fraction=0.95)


@pytest.mark.parametrize("rows,n,k", [(3, 128, 128), (16, 272, 1152), (40, 2064, 8192), (250, 272, 640), (3, 64, 8320)])
def test_few_rows_split_in_the_kernel_equals_the_split_launch(M, O, dev, rows, n, k):
    """Rows that are 16-byte aligned are split inside the few-row product (K
    up to 8192), others by a launch of their own: the same bytes, with zero
    blocks, subnormal and huge blocks, NaN and infinities among them."""
    import torch

    rng = np.random.default_rng(rows + n + k)
    codes = rng.integers(0, 0x7F, size=(n, k), dtype=np.int64).astype(np.uint8)
    scale = (rng.uniform(size=(-(-n // 128), k // 128)) * 0.002).astype(np.float32)
    w, s = torch.from_numpy(codes).to(dev), torch.from_numpy(scale).to(dev)
    x = rng.normal(size=(rows, k)) * 2.0 ** rng.integers(-20, 20, size=(rows, 1))
    bits = O.f32_to_bf16(x.astype(np.float32)).reshape(rows, k)
    bits[0, :128] = 0
    bits[1, :128] = rng.integers(0, 0x80, size=128)  # subnormal
    bits[2, 5], bits[2, k - 3], bits[2, 40], bits[rows - 1, k - 1] = 0x7F80, 0xFFC1, 0x7F01, 0xFF80
    aligned = from_bits(bits, dev)
    shifted = torch.empty(rows * k + 1, dtype=torch.bfloat16, device=dev)[1:].view(rows, k)
    shifted.copy_(aligned)
    assert aligned.data_ptr() % 16 == 0 and shifted.data_ptr() % 16 == 2
    needed = submodule("_native").lib().glm53_fp8_linear_workspace_needed
    assert (needed(aligned.data_ptr(), rows, n, k) == 0) == (k <= 8192) and needed(shifted.data_ptr(), rows, n, k) > 0
    got, want = (M.block_fp8_linear(v, w, s) for v in (aligned, shifted))
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("with_480", [False, True])
@pytest.mark.parametrize("rows", [2, 33, 150, 300, 700, 1300, 6000, 12000])
def test_mlp_in_one_call_equals_its_parts(M, dev, rows, with_480):
    """ClampedMLP over two or more rows runs as one native call: the bytes of
    gate_proj, up_proj, swiglu and down_proj called in turn (a hook on one of
    them keeps the parts), in every tile of the SwiGLU form and of the down
    product, rows and columns ragged, codes 0x7F / 0xFF in one matrix each."""
    import torch

    hidden, inter = 256, 640
    gen = torch.Generator().manual_seed(rows)
    for marked in ("gate_proj", "up_proj", "down_proj") if with_480 else ("none",):
        mlp = M.ClampedMLP(hidden, inter, 2.0, device=dev)
        for name in ("gate_proj", "up_proj", "down_proj"):
            proj = getattr(mlp, name)
            codes = torch.randint(0, 0x7F, tuple(proj.weight.shape), generator=gen, dtype=torch.uint8)
            codes |= torch.randint(0, 2, tuple(codes.shape), generator=gen, dtype=torch.uint8) << 7
            if name == marked:
                codes[-1, -1], codes[3, 200] = 0xFF, 0x7F
            proj.weight.copy_(codes)
            proj.weight_scale_inv.copy_(torch.rand(tuple(proj.weight_scale_inv.shape), generator=gen) * 0.002)
        x = torch.randn((1, rows, 2 * hidden), generator=gen).to(dev, torch.bfloat16)[..., ::2]
        assert mlp._one_call(x)
        y = mlp(x)
        hook = mlp.up_proj.register_forward_hook(lambda module, args, out: None)
        assert not mlp._one_call(x)
        assert torch.equal(y.view(torch.int16), mlp(x).view(torch.int16)), (rows, marked)
        hook.remove()
    assert not mlp._one_call(x[:, :1]) and not mlp._one_call(x.float())
    with pytest.raises(ValueError):
        mlp(x[..., :128])


@pytest.mark.parametrize("name", ["gate_proj", "up_proj", "down_proj"])
def test_mlp_with_a_scale_table_on_the_host_is_refused(M, dev, name):
    """A projection whose scale table stayed on the host raises, whatever the
    number of rows."""
    import torch

    mlp = M.ClampedMLP(256, 128, 2.0, device=dev)
    proj = getattr(mlp, name)
    proj.weight_scale_inv = proj.weight_scale_inv.cpu()
    for rows in (1, 5):
        x = torch.zeros((rows, 256), dtype=torch.bfloat16, device=dev)
        assert not mlp._one_call(x)
        with pytest.raises(ValueError, match="ROCm device"):
            mlp(x)


@pytest.mark.parametrize("rows", [1, 5, 64])
def test_both_480_codes_gemv_and_mfma(M, O, dev, rows):
    """Codes over the whole byte range, so 0x7F (+480) and 0xFF (-480) both
    occur: the reference LUT decodes them as finite +-480 (fp8.py:22-27),
    OCP E4M3 (and the MFMA) as NaN.  M = 1 takes the register-decode GEMV,
    M > 1 the MFMA GEMM with its chained +-32 correction."""
    rng = np.random.default_rng(480 + rows)
    k, n = 1024, 272
    codes = random_codes(rng, (n, k), high=256)
    codes[:, :8] = 0xFF  # every row carries both signs
    codes[:, 8:16] = 0x7F
    scale = (rng.uniform(size=(-(-n // 128), k // 128)) * 0.002).astype(np.float32)
    x = O.f32_to_bf16(rng.normal(size=(rows, k)).astype(np.float32))
    got = _linear(M, dev, x, codes, scale)
    want = O.fp8_linear(x, codes, scale)
    assert np.isfinite(O.bf16_to_f32(got)).all()
    # full-range codes spread the products over ~2^16: more FP32 sums land
    # one BF16 ulp from the exact one than for checkpoint-like weights
    assert_parity(got, want, O, exact_fraction=0.95)


def test_input_layout_invariance(M, O, dev):
    """tests/test_metal_input_layout.py:27-95: strided / offset inputs give
    byte-identical results to row-contiguous ones."""
    import torch

    rng = np.random.default_rng(3)
    k, n = 1024, 256
    codes = random_codes(rng, (n, k))
    scale = (rng.uniform(size=(2, 8)) * 0.002).astype(np.float32)
    w = torch.from_numpy(codes).to(dev)
    s = torch.from_numpy(scale).to(dev)
    for tokens in (1, 7, 8, 9, 127, 128, 129, 255, 256, 1023, 1024):
        base = from_bits(O.f32_to_bf16(rng.normal(size=(tokens, 2 * k)).astype(np.float32)), dev)
        strided = base[:, ::2]
        contiguous = strided.contiguous()
        a = M.block_fp8_linear(strided, w, s)
        b = M.block_fp8_linear(contiguous, w, s)
        assert torch.equal(a.view(torch.int16), b.view(torch.int16)), tokens


def test_sigmoid_matches_reference_exhaustive_sweep_hash(M, dev):
    """The device sigmoid over all 33,346 finite BF16 values in [-10, 10]
    hashes to the MLX reference hash recorded by the reference's sweep."""
    import torch

    golden = json.loads((GOLDEN / "sigmoid_sweep.json").read_text())
    bits = np.arange(1 << 16, dtype=np.uint16)
    vals = (bits.astype(np.uint32) << 16).view(np.float32)
    domain = bits[np.isfinite(vals) & (np.abs(vals) <= np.float32(10.0))]
    assert hashlib.sha256(domain.tobytes()).hexdigest() == golden["domain_bits_sha256"]
    N = submodule("_native")
    g = from_bits(domain, dev)
    out = torch.empty_like(g)
    N.check(N.lib().glm53_sigmoid_bf16(N.ptr(g), g.numel(), N.ptr(out), N.stream_handle(dev)))
    got = to_bits(out)
    assert hashlib.sha256(got.tobytes()).hexdigest() == golden["reference_sigmoid_sha256"]


def test_sigmoid_every_bf16_pattern_matches_oracle(O, dev):
    """The device sigmoid (the hardware-exponential form every SwiGLU uses,
    with its correctly rounding fallback for |g| > 87 and the fast::exp
    point) on all 65,536 BF16 patterns equals the oracle's MLX sigmoid bit
    for bit on every non-NaN input (NaN in, NaN out)."""
    import torch

    N = submodule("_native")
    bits = np.arange(1 << 16, dtype=np.uint16)
    vals = (bits.astype(np.uint32) << 16).view(np.float32)
    g = from_bits(bits, dev)
    out = torch.empty_like(g)
    N.check(N.lib().glm53_sigmoid_bf16(N.ptr(g), g.numel(), N.ptr(out), N.stream_handle(dev)))
    got = to_bits(out)
    ok = ~np.isnan(vals)
    want = O.sigmoid_bf16(bits[ok])
    bad = np.flatnonzero(got[ok] != want)
    assert bad.size == 0, [(hex(int(bits[ok][i])), hex(int(got[ok][i])), hex(int(want[i]))) for i in bad[:8]]
    nan_out = (got[~ok] & 0x7F80) == 0x7F80
    assert nan_out.all() and (got[~ok] & 0x007F).all()


def test_swiglu_bit_exact_against_oracle(M, O, dev):
    rng = np.random.default_rng(11)
    bits = np.arange(1 << 16, dtype=np.uint16)
    vals = (bits.astype(np.uint32) << 16).view(np.float32)
    gate = bits[np.isfinite(vals) & (np.abs(vals) <= 40.0)]
    up = O.f32_to_bf16(rng.normal(scale=6.0, size=gate.size).astype(np.float32))
    for limit in (10.0, 3.0, 20.0):
        got = to_bits(M.swiglu(from_bits(gate, dev), from_bits(up, dev), limit))
        assert np.array_equal(got, O.swiglu(gate, up, limit)), limit


def test_swiglu_every_gate_pattern_matches_oracle(M, O, dev):
    """The straight-line SwiGLU (two values per conversion, the form of the
    grouped GEMM epilogues) with its fall-back to the exact sequence, over
    all 65,536 BF16 gate patterns (NaN, +-inf, |g| > 87 and 0xC0DB included)
    against up values with +-0, +-inf, NaN and values past the clamp: equal
    to the oracle bit for bit wherever the oracle's result is not NaN, NaN
    where it is."""
    rng = np.random.default_rng(12)
    gate = np.arange(1 << 16, dtype=np.uint16)
    up = O.f32_to_bf16(rng.normal(scale=12.0, size=gate.size).astype(np.float32))
    special = np.array([0x0000, 0x8000, 0x7F80, 0xFF80, 0x7FC0, 0xFFC1, 0x3F80, 0xBF80, 0x4120, 0xC120],
                       dtype=np.uint16)
    pick = rng.choice(gate.size, size=4096, replace=False)
    up[pick] = special[rng.integers(0, special.size, size=pick.size)]
    # an odd count: the last value is paired with itself
    gate, up = gate[:-1], up[:-1]
    for limit in (7.0, 10.0, float("inf")):
        got = to_bits(M.swiglu(from_bits(gate, dev), from_bits(up, dev), limit))
        want = O.swiglu(gate, up, limit)
        nan_want = (want & 0x7F80) == 0x7F80
        nan_want &= (want & 0x007F) != 0
        bad = np.flatnonzero(~nan_want & (got != want))
        assert bad.size == 0, (limit, [(hex(int(gate[i])), hex(int(up[i])), hex(int(got[i])), hex(int(want[i])))
                                       for i in bad[:8]])
        assert ((got[nan_want] & 0x7F80) == 0x7F80).all() and (got[nan_want] & 0x007F).all(), limit
