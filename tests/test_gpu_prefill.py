"""bf16 matrix-core prefill GEMM (Int8Linear's large-M path) through the C ABI.

Two oracles (oracle/math_ref.int8_linear_prefill_f64):
  * with x rounded to bfloat16 (ties to even), the product the kernel computes exactly up to
    its float32 accumulation: rel-L2 <= 2e-6 and max-abs <= 2e-5 * max|y|;
  * the plain weight-only product over float32 x (the reference's dequant GEMM, quant.py:71-72
    and :78-79): the stated bf16 tolerance, rel-L2 <= 5e-3.
At BASELINE config 3 sizes (M = 2048) the float64 oracles run on a seeded subset of rows.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import capi_util as cu
from oracle import math_ref as mr
from oracle import quant as oq

pytestmark = pytest.mark.gpu
F32 = np.float32
TIGHT_L2, TIGHT_MAX, BF16_L2 = 2e-6, 2e-5, 5e-3


def rel_l2(got, ref):
    got = np.asarray(got, np.float64)
    return float(np.linalg.norm(got - ref) / np.linalg.norm(ref))


def check(y, x, q, s, rows=None):
    y = y.cpu().numpy()
    if rows is not None:
        x, y = x[rows], y[rows]
    exact = mr.int8_linear_prefill_f64(x, q, s)
    assert rel_l2(y, exact) <= TIGHT_L2, rel_l2(y, exact)
    assert np.abs(y - exact).max() <= TIGHT_MAX * np.abs(exact).max()
    plain = mr.int8_linear_prefill_f64(x, q, s, round_x=False)
    err = rel_l2(y, plain)
    assert err <= BF16_L2, err
    return err


def make(seed, M, N, K):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((M, K)).astype(F32)
    q, s = oq.int8_quantize((rng.standard_normal((N, K)) * 0.02).astype(F32))
    return x, q, s


@pytest.mark.parametrize("M,N,K", [(1, 1, 64), (37, 100, 64), (256, 256, 128), (300, 520, 192),
                                   (513, 257, 320), (64, 2048, 1024), (200, 300, 4096),
                                   (2048, 6000, 128)])
def test_shapes(gpu, M, N, K):
    x, q, s = make(M * 7 + N, M, N, K)
    y = cu.int8_linear_prefill(cu.dev(x), cu.dev(q), cu.dev(s))
    check(y, x, q, s)


# The 256-row tiles with their last row and column tiles partly past M and N, above the line to the
# small tiles: four K splits, 192-wide tiles (a 48-column last one), and K off the 128 grid.
@pytest.mark.parametrize("M,N,K,splits", [(777, 2040, 8192, 4), (2040, 6000, 2048, 1), (33, 1000, 704, 1)])
def test_partial_large_tiles(gpu, M, N, K, splits):
    x, q, s = make(M + N, M, N, K)
    copy = (M * K * 2 + 255) // 256 * 256
    partials = splits * M * N * 4 if splits > 1 else 0
    assert cu.capi().llmserve_int8_linear_prefill_workspace_bytes(M, N, K) == copy + partials
    y = cu.int8_linear_prefill(cu.dev(x), cu.dev(q), cu.dev(s))
    rows = np.concatenate([np.arange(min(M, 40)), np.arange(M)[-40:]])
    check(y, x, q, s, rows)


@pytest.mark.parametrize("N,K", [(6144, 2048), (16384, 2048), (2048, 8192)])
def test_config3_shapes(gpu, N, K):
    """BASELINE config 3 (SmolLM2-1.7B qkv, gate_up, down) at M = 2048; 96 seeded rows checked
    against float64, every row against the torch bf16 product of the same operands."""
    M = 2048
    g = torch.Generator(device="cuda").manual_seed(N + K)
    xd = torch.randn(M, K, device="cuda", generator=g)
    wd = torch.randn(N, K, device="cuda", generator=g) * 0.02
    q, s = cu.int8_quantize(wd)
    y = cu.int8_linear_prefill(xd, q, s)
    rows = np.random.default_rng(N).choice(M, 96, replace=False)
    err = check(y, xd.cpu().numpy(), q.cpu().numpy(), s.cpu().numpy(), rows)
    print(f"config 3 N={N} K={K}: rel-L2 vs fp32-x weight-only product {err:.2e}")
    # all rows: float32 GEMM of the same bf16-rounded operands (torch, fp32 accumulate)
    ref = (xd.to(torch.bfloat16).float() @ q.float().t()) * s[None, :]
    assert torch.linalg.norm(y - ref) / torch.linalg.norm(ref) <= 1e-5


def test_module_prefill_and_dequant_agree(gpu):
    from torch import nn

    from llmserve.quant import Int8Linear

    torch.manual_seed(0)
    lin = nn.Linear(512, 384, bias=True)
    m = Int8Linear(lin, device="cuda")
    x = torch.randn(2, 150, 512, device="cuda")
    y = m(x)  # auto: 300 rows -> prefill GEMM
    Int8Linear.kernel = "dequant"
    try:
        y_ref = m(x)
    finally:
        Int8Linear.kernel = "auto"
    assert y.shape == (2, 150, 384)
    assert (torch.linalg.norm(y - y_ref) / torch.linalg.norm(y_ref)).item() <= BF16_L2


def test_rejects_bad_k(gpu):
    x = torch.randn(4, 96, device="cuda")
    q = torch.zeros(8, 96, dtype=torch.int8, device="cuda")
    s = torch.ones(8, device="cuda")
    with pytest.raises(RuntimeError, match="multiple of 64"):
        cu.int8_linear_prefill(x, q, s)


# Both sides of the line between the small tiles and the 256-wide ones, at the small tiles' edges (16 x 64,
# 32 x 128, 64 x 256 with 4, 2 and 1 K parts), odd row and channel counts and K block counts that
# pad; K off the 128 grid stays with the 256-wide tiles.
@pytest.mark.parametrize("M,N,K", [(1, 1, 128), (17, 63, 256), (16, 65, 384), (33, 1000, 640), (129, 257, 1152),
                                   (777, 1025, 512), (1290, 4161, 384), (2048, 6144, 1024),
                                   (2049, 6144, 1024), (33, 1000, 704)])
def test_small_tiles(gpu, M, N, K):
    x, q, s = make(M + N + K, M, N, K)
    x[:, 3] *= 1000  # a channel far above the others
    y = cu.int8_linear_prefill(cu.dev(x), cu.dev(q), cu.dev(s))
    check(y, x, q, s, np.random.default_rng(M).permutation(M)[:200])


def test_small_tiles_rows_are_independent(gpu):
    """Rows of 1e-30 .. 1e30, a zero row, an infinity (beside the largest finite values) and a NaN: each
    row as float32 arithmetic on bf16(x) has it."""
    x, q, s = make(3, 40, 96, 256)
    x[:8] *= np.logspace(-30, 30, 8).astype(F32)[:, None]
    x[8] = 0
    x[9] = 1e38
    x[9, 200], x[10, 3] = np.inf, np.nan
    y = cu.int8_linear_prefill(cu.dev(x), cu.dev(q), cu.dev(s)).cpu().numpy()
    want = np.where(q[:, 200] == 0, np.nan, np.sign(q[:, 200]) * np.inf)
    np.testing.assert_array_equal(y[9], want.astype(F32))
    assert np.isnan(y[10]).all() and not y[8].any()
    for r in (r for r in range(40) if r not in (8, 9, 10)):
        exact = mr.int8_linear_prefill_f64(x[r:r + 1], q, s)
        assert rel_l2(y[r:r + 1], exact) <= TIGHT_L2, r
