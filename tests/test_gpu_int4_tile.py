"""The tiled int4 GEMM (llmserve_int4_linear_tile, Int4Linear's large-M path) against float64.

Bound: x' is held to 2^-22 of each element (two fp16 pieces), the zero term's operands to 2^-22
as well, and fp32 adds at most K / 32 partial sums of exact products: with random signs about
2^-22 + 2^-24 sqrt(K / 32), below 1e-6 relative (2-norm) for K up to 8192; 2e-6 is asked, and ten
times that of the largest value.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import capi_util as cu
from llmserve.kernels import load_int8_gemv
from oracle import math_ref as mr
from oracle import quant as oq

pytestmark = pytest.mark.gpu
F32 = np.float32


def make(seed, M, N, K, group, awq):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((M, K)).astype(F32)
    x[:, rng.permutation(K)[: max(1, K // 100)]] *= 20
    act = (np.abs(rng.standard_normal(K)) + 0.2).astype(F32) if awq else None
    w = (rng.standard_normal((N, K)) * 0.02).astype(F32)
    return (x, *oq.int4_quantize_pack(w, group, act))


def run(x, nib, gs, gz, group, inv, packed):
    ops = load_int8_gemv()
    t = [torch.from_numpy(a).cuda() if a is not None else None for a in (x, nib, gs, gz, inv)]
    pk = ops.int4_gemm_pack(t[1], t[2], t[3], group) if packed else None
    return ops.int4_linear_tile(t[0], t[1], t[2], t[3], group, t[4], pk), t


def check(y, x, nib, gs, gz, group, inv):
    ref = mr.int4_linear_f64(x, nib, gs, gz, group, inv)
    y = y.cpu().numpy().astype(np.float64)
    assert np.linalg.norm(y - ref) <= 2e-6 * np.linalg.norm(ref)
    assert np.abs(y - ref).max() <= 2e-5 * np.abs(ref).max()


# tile edges (16, 32, 64 rows; 64, 128, 256 channels), odd sizes, an odd count of K blocks, groups of
# 64 / 128 / 192 / 256 / the whole row, more than 64 units of K, each tile of the dispatch
@pytest.mark.parametrize("M,N,K,group,packed", [
    (1, 1, 128, 64, False), (17, 63, 128, 128, False), (16, 64, 256, 64, False),
    (33, 65, 384, 192, False), (31, 129, 640, 128, True), (65, 300, 1152, 64, False),
    (129, 257, 512, 256, True), (100, 1000, 8320, 64, False), (70, 200, 1024, 1024, True),
    (300, 1464, 1664, 128, True), (257, 4100, 256, 64, False), (513, 2049, 384, 128, False),
    (1030, 6100, 256, 64, False), (1281, 4160, 384, 128, True)])
def test_tile_vs_f64(gpu, M, N, K, group, packed):
    x, nib, gs, gz, inv = make(M + N + K, M, N, K, group, M % 2 == 1)
    y, t = run(x, nib, gs, gz, group, inv, packed)
    check(y, x, nib, gs, gz, group, inv)
    if packed:  # the caller's packing and the call's own give the same bits
        assert torch.equal(y, run(x, nib, gs, gz, group, inv, False)[0])
    off = torch.zeros(t[0].numel() + 1, device="cuda")[1:].view(t[0].shape)  # 4-byte aligned rows
    off.copy_(t[0])
    assert torch.equal(y, load_int8_gemv().int4_linear_tile(off, t[1], t[2], t[3], group, t[4]))


def test_rows_are_independent_and_wide_ranges_hold(gpu):
    """Rows of 1e-30 .. 1e30, a zero row, a row with a NaN and one with an infinity: each row's
    result is its own, and finite rows keep their precision."""
    x, nib, gs, gz, inv = make(5, 40, 96, 256, 64, True)
    x[:8] *= np.logspace(-30, 30, 8).astype(F32)[:, None]
    x[8] = 0
    x[9, 3], x[10, 200] = np.nan, np.inf
    y = run(x, nib, gs, gz, 64, inv, False)[0].cpu().numpy()
    fine = [r for r in range(40) if r not in (9, 10)]
    assert not np.isfinite(y[[9, 10]]).any() and not y[8].any()
    ref = mr.int4_linear_f64(x[fine], nib, gs, gz, 64, inv)
    err = np.linalg.norm(y[fine] - ref, axis=1)
    assert (err <= 3e-6 * np.linalg.norm(ref, axis=1)).all()


@pytest.mark.parametrize("group,rows,path", [(64, 16, "gemv"), (64, 17, "tile"), (128, 256, "gemm"),
                                             (128, 257, "tile")])
def test_module_dispatch(gpu, group, rows, path):
    from llmserve.quant import Int4Linear

    base = torch.nn.Linear(256, 200, device="cuda")
    m = Int4Linear(base, group)
    x = torch.randn(rows, 256, device="cuda")
    assert m._path(rows, load_int8_gemv(), x) == path
    with torch.inference_mode():
        y = m(x)
    ref = x.double() @ m.dequantize().double().t() + m.bias.double()
    assert (y - ref).norm() <= 1e-5 * ref.norm()
    # gradients, other types and K off the 128 grid keep the torch ops
    xg = x.clone().requires_grad_()
    assert m._path(rows, load_int8_gemv(), xg) != "tile"
    assert not m._tile_ok(x.bfloat16())
    assert not Int4Linear(torch.nn.Linear(192, 8, device="cuda"), 64)._tile_ok(x[:, :192])
    assert torch.ops.llmserve_hip.int4_linear_tile(
        *(t.to("meta") for t in (x, m.nibbles, m.g_scale, m.g_zero)), group).shape == y.shape


@pytest.mark.parametrize("name", ["x", "g_scale", "g_zero"])
def test_gradients_and_autocast_keep_the_torch_ops(gpu, name):
    from llmserve.quant import Int4Linear

    m = Int4Linear(torch.nn.Linear(256, 40, bias=False, device="cuda"), 64)
    x = torch.randn(33, 256, device="cuda")
    assert m._tile_ok(x)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not m._tile_ok(x) and m(x).dtype == torch.bfloat16
    t = (x if name == "x" else getattr(m, name)).requires_grad_()
    m(x).sum().backward()
    assert t.grad is not None and t.grad.abs().sum() > 0
    with torch.no_grad():
        assert m._tile_ok(x)


# each tile (16 x 64, 32 x 128, 64 x 256) with its last row tile partly past M, down to one row in it
@pytest.mark.parametrize("M,N,K", [(1, 60, 128), (17, 64, 256), (33, 70, 128), (65, 136, 384), (33, 12200, 128),
                                   (65, 12300, 128), (65, 41000, 128), (1281, 4100, 128)])
@pytest.mark.parametrize("weights", ["int4", "int8"])
def test_nothing_is_written_behind_y(gpu, M, N, K, weights):
    """The bytes behind y and behind the workspace stay as they were."""
    pad = 64 * N  # floats: more than the rows a tile can have past M
    rng = np.random.default_rng(M + N)
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(F32)).cuda()
    w = torch.from_numpy((rng.standard_normal((N, K)) * 0.02).astype(F32)).cuda()
    y = torch.full((M * N + pad,), -7.5, device="cuda")
    lib = cu.capi()
    if weights == "int8":
        q, s = cu.int8_quantize(w)
        need = lib.llmserve_int8_linear_prefill_workspace_bytes(M, N, K)
    else:
        q, gs, gz, _ = cu.int4_quantize(w, 64)
        need = lib.llmserve_int4_linear_tile_workspace_bytes(M, N, K, 64)
    ws = torch.full((need + 4096,), 0x5A, dtype=torch.uint8, device="cuda")
    if weights == "int8":
        cu.check(lib.llmserve_int8_linear_prefill(cu._p(x), cu._p(q), cu._p(s), cu._p(y), M, N, K, cu._p(ws), need,
                                                  cu._stream()))
        ref = x.bfloat16().double() @ (q.double() * s.double()[:, None]).t()
    else:
        cu.check(lib.llmserve_int4_linear_tile(cu._p(x), None, cu._p(q), cu._p(gs), cu._p(gz), None, cu._p(y), M, N,
                                               K, 64, cu._p(ws), need, cu._stream()))
        ref = mr.int4_linear_f64(*(t.cpu().numpy() for t in (x, q, gs, gz)), 64)
        ref = torch.from_numpy(ref).cuda()
    assert (y[M * N:] == -7.5).all() and (ws[need:] == 0x5A).all()
    assert (y[: M * N].view(M, N) - ref).norm() <= 2e-6 * ref.norm()


def follows(m, x):
    """The module's output is the product of the buffers it holds now."""
    with torch.no_grad():
        y, ref = m(x), x.double() @ m.dequantize().double().t()
    return (y - ref).norm() <= 1e-5 * ref.norm()


@pytest.mark.parametrize("group,rows", [(128, 300), (64, 300), (64, 40)])
def test_large_batches_follow_the_buffers(gpu, group, rows):
    """After a state dict, an in-place change, one through .data (that no version counter sees), a new
    buffer and under functional_call."""
    from llmserve.quant import Int4Linear

    a, b = (Int4Linear(torch.nn.Linear(256, 208, bias=False, device="cuda"), group) for _ in range(2))
    x = torch.randn(rows, 256, device="cuda")
    old = a(x)
    with torch.no_grad():
        swapped = torch.func.functional_call(a, dict(b.state_dict()), (x,))
        assert torch.equal(swapped, b(x)) and torch.equal(a(x), old)
    a.load_state_dict(b.state_dict())
    assert follows(a, x) and not torch.equal(a(x), old)
    a.g_scale.mul_(3)
    assert follows(a, x)
    a.g_zero.data.add_(0.5)
    assert follows(a, x)
    a.nibbles = torch.flip(a.nibbles, (0,)).contiguous()
    assert follows(a, x)


def test_transforms_through_the_module(gpu):
    """A forward-mode derivative, and a gradient taken outside of a vmap (which no tensor inside shows)."""
    from llmserve.quant import Int4Linear

    m = Int4Linear(torch.nn.Linear(256, 40, bias=False, device="cuda"), 64)
    w = m.dequantize()
    x, dx = torch.randn(2, 3, 33, 256, device="cuda")
    _, t = torch.func.jvp(m, (x[0],), (dx[0],))
    assert (t - dx[0] @ w.t()).norm() <= 1e-5 * t.norm()
    g = torch.func.grad(lambda x: torch.vmap(m)(x).square().sum())(x)
    assert (g - 2 * (x @ w.t()) @ w).norm() <= 1e-5 * g.norm()


def test_buffers_of_other_types_and_strides_keep_the_torch_ops(gpu):
    """Scales in 16 bits (a module moved with .half()), and buffers that are views of other memory."""
    from llmserve.quant import Int4Linear

    lin = torch.nn.Linear(256, 40, bias=False, device="cuda")
    act = torch.rand(256, device="cuda") + 0.5
    x = torch.randn(33, 256, device="cuda")
    m = Int4Linear(lin, 64, act).half()
    xs = x * m.inv_act_scale
    assert torch.equal(m(x), xs @ m.dequantize().t()) and m(x).dtype == torch.float32
    for name in ("nibbles", "g_scale", "g_zero", "inv_act_scale"):
        m = Int4Linear(lin, 64, act)
        y = m(x)
        t = getattr(m, name)
        setattr(m, name, t.repeat_interleave(2, -1)[..., ::2])
        assert (m(x) - y).norm() <= 2e-6 * y.norm()


@pytest.mark.parametrize("M,N,K,group,packed", [(40, 96, 256, 64, False), (129, 1000, 384, 128, True),
                                                (300, 12300, 128, 64, False)])
def test_infinities_keep_their_signs(gpu, M, N, K, group, packed):
    """A row with infinities is what arithmetic on the dequantized weight gives: signed infinities, NaN
    where opposite ones meet or the weight is 0; the other rows are as they were."""
    x, nib, gs, gz, inv = make(M + K, M, N, K, group, True)
    clean = run(x, nib, gs, gz, group, inv, packed)[0]
    gz[3, 0], gs[5, 0] = 0, 0  # code 8 of channel 3 is a weight of 0
    nib[3, 0], gz[5, 0] = 0x88, 0
    bad = {1: {0: np.inf}, 2: {7: -np.inf}, M - 1: {1: np.inf, K - 1: np.inf}, 9: {3: np.inf, 5: np.nan}}
    for r, where in bad.items():
        for k, v in where.items():
            x[r, k] = v
    x[4, 2] = 3e38  # an infinity from the AWQ product
    inv[2] = 4
    rows = sorted([*bad, 4])
    y = run(x, nib, gs, gz, group, inv, packed)[0].cpu().numpy()
    with np.errstate(invalid="ignore", over="ignore"):
        want = mr.int4_linear_f64(x[rows], nib, gs, gz, group, inv)
    assert not np.isfinite(want).any() and np.isinf(want[0]).any()
    np.testing.assert_array_equal(y[rows], want.astype(F32))
    fine = [r for r in range(M) if r not in rows]
    ref = mr.int4_linear_f64(x[fine], nib, gs, gz, group, inv)
    assert np.linalg.norm(y[fine] - ref) <= 2e-6 * np.linalg.norm(ref)
