"""The tiled prefill attention (llmserve_paged_attention_prefill) against float64.

Bound: scores and sums are fp32 sums of exact products of 22-bit operands, as the row kernel's are
fp32 products: the same 1e-5 of the largest value that its tests ask, and 2e-6 in the 2-norm
(measured 1.3e-7 to 4.5e-7; the widest scale range below has the largest).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import capi_util as cu
from llmserve import attention as at
from llmserve.kernels import load_paged_attention
from oracle import math_ref as mr
from oracle import quant as oq

pytestmark = pytest.mark.gpu
F32 = np.float32


def make(seed, q_lens, ctx, geom, int8, spread=0.0):
    hq, hk, d, bs = geom
    rng = np.random.default_rng(seed)
    need = [-(-c // bs) for c in ctx]
    order = rng.permutation(sum(need) + 3).astype(np.int64)
    tables, used = [], 0
    for n in need:
        tables.append(order[used: used + n].tolist())
        used += n
    slots = order.size * bs
    k, v = (rng.standard_normal((slots, hk, d)).astype(F32) for _ in range(2))
    if spread:  # rows of very different size
        v *= np.exp(rng.standard_normal((slots, hk, 1)) * spread).astype(F32)
        k *= np.exp(rng.standard_normal((slots, hk, 1)) * spread / 4).astype(F32)
    q = rng.standard_normal((sum(q_lens), hq, d)).astype(F32)
    meta = at.AttentionMetadata.build(q_lens, ctx, tables, bs, "cuda", "hip")
    cache, mult = (k, v, None, None), None
    if int8:
        (kq, ks), (vq, vs) = oq.kv_quantize(k), oq.kv_quantize(v)
        cache = (kq, vq, ks, vs)
        k, v = mr.kv_dequantize(kq, ks), mr.kv_dequantize(vq, vs)
        mult = (0.5 + rng.random((hq, d))).astype(F32)
    dev = tuple(None if t is None else torch.from_numpy(t).cuda() for t in cache)
    return q, k, v, tables, meta, dev, mult


def reference(q, k, v, q_lens, ctx, tables, geom, mult):
    hq, hk, d, bs = geom
    row_tab = np.repeat(np.arange(len(q_lens)), q_lens)
    row_ctx = np.concatenate([np.arange(c - n, c) + 1 for n, c in zip(q_lens, ctx)])
    bt = np.zeros((len(tables), max(map(len, tables))), np.int64)
    for i, t in enumerate(tables):
        bt[i, : len(t)] = t
    qd = q if mult is None else q * mult
    return mr.paged_rows_f64(qd, k, v, bt, row_tab, row_ctx, bs, d ** -0.5)


@pytest.fixture(autouse=True)
def every_batch_in_tiles(monkeypatch):
    """The dispatch's estimate would leave small batches to the row kernel."""
    monkeypatch.setattr(at, "ROW_US", 1e6)


def run(q, meta, dev, mult, d):
    m = None if mult is None else torch.from_numpy(mult).cuda()
    return at._attend_native(load_paged_attention(), torch.from_numpy(q).cuda(), dev, m, meta, d ** -0.5)


def close(out, ref):
    out = out.cpu().numpy().astype(np.float64)
    assert np.linalg.norm(out - ref) <= 2e-6 * np.linalg.norm(ref)
    assert np.abs(out - ref).max() <= 1e-5 * np.abs(ref).max()


# query tiles of 1 .. 64 tokens, contexts around the context tiles (32 / 64) and over several chunks,
# odd head counts per kv head, block sizes that divide nothing, decode rows beside prompts
@pytest.mark.parametrize("int8", [True, False])
@pytest.mark.parametrize("q_lens,ctx,geom", [
    ([16], [16], (2, 1, 128, 16)), ([65], [65], (8, 8, 64, 16)), ([64, 1, 17], [64, 40, 300], (4, 2, 64, 4)),
    ([127, 128], [127, 1000], (9, 3, 64, 5)), ([40], [2500], (16, 8, 128, 16)),
    ([193, 1, 1, 20], [321, 1, 77, 20], (7, 1, 128, 24)), ([33, 15], [33, 500], (6, 2, 128, 1)),
    ([600], [1900], (16, 2, 128, 32))])
def test_prefill_vs_f64(gpu, q_lens, ctx, geom, int8):
    q, k, v, tables, meta, dev, mult = make(sum(ctx), q_lens, ctx, geom, int8)
    assert meta.prefill_tiles is not None
    close(run(q, meta, dev, mult, geom[2]), reference(q, k, v, q_lens, ctx, tables, geom, mult))


@pytest.mark.parametrize("int8", [True, False])
def test_rows_of_very_different_size(gpu, int8):
    geom = (8, 2, 128, 16)
    q, k, v, tables, meta, dev, mult = make(3, [200], [700], geom, int8, spread=3.0)
    close(run(q, meta, dev, mult, 128), reference(q, k, v, [200], [700], tables, geom, mult))


@pytest.mark.parametrize("int8", [True, False])
def test_blocks_outside_the_cache_and_bad_rows(gpu, int8):
    """A block id outside the cache adds nothing (as in the row kernel); a key or value row that is
    not finite reaches the tokens that see it and no other."""
    geom, n = (4, 2, 64, 16), 100
    q, k, v, tables, meta, dev, mult = make(4, [n], [n], geom, int8)
    meta.block_tables[0, 2] = 10**6
    got = run(q, meta, dev, mult, 64)
    rows = at._tiles_ok
    try:
        at._tiles_ok = lambda *a: False
        want = run(q, meta, dev, mult, 64)
    finally:
        at._tiles_ok = rows
    assert (got - want).norm() <= 1e-6 * want.norm()
    meta.block_tables[0, 2] = tables[0][2]
    clean = run(q, meta, dev, mult, 64)
    slot = tables[0][3] * 16 + 5  # token 53
    for i, t in enumerate(dev[2:] if int8 else dev[:2]):
        # an infinite key scale is left out: it gives scores of +-inf, and -inf is a weight of 0
        for bad in (float("nan"), float("inf")) if i else (float("nan"),):
            was = t[slot].clone()
            t[slot] = bad
            out = run(q, meta, dev, mult, 64)
            t[slot] = was
            assert torch.equal(out[:53], clean[:53]) and not torch.isfinite(out[53:]).any()


def test_dispatch(gpu, monkeypatch):
    """Sequences of at least TILE_ROWS new tokens go to the tiles, the rest to the row kernel; head
    sizes and groups the tiles do not take keep the row kernel for all, and so does work too small
    for a tiled launch (and a sequence with less context than new tokens)."""
    def tiled(q_lens, ctx):
        tabs = [list(range(-(-c // 16))) for c in ctx]
        return at.AttentionMetadata.build(q_lens, ctx, tabs, 16, "cuda", "hip").prefill_tiles is not None

    monkeypatch.undo()
    assert [tiled([n], [1024]) for n in (32, 64)] == [False, True]
    assert not tiled([64, 1], [1024, 10]) and tiled([200, 1], [1024, 10])
    assert not tiled([4] * 8, [4096] * 8) and tiled([8] * 8, [4096] * 8)
    assert not tiled([2000], [1000])
    monkeypatch.setattr(at, "ROW_US", 1e6)
    few, many = at.TILE_ROWS - 1, at.TILE_ROWS
    meta = at.AttentionMetadata.build([few, many, 1], [50, 70, 9], [[0] * 4, [1] * 5, [2]], 16, "cuda", "hip")
    assert meta.prefill_tiles_host.tolist() == [[few, many, 70 - many + 1, 1]]
    assert torch.equal(meta.prefill_tiles.cpu(), meta.prefill_tiles_host)
    assert meta.rest_rows.tolist() == [*range(few), few + many]
    assert meta.rest_context.tolist() == [*range(50 - few + 1, 51), 9]
    k = torch.zeros(96, 2, 128, device="cuda")
    assert at._tiles_ok(torch.zeros(few + many + 1, 4, 128), k, meta)
    assert not at._tiles_ok(torch.zeros(few + many + 1, 4, 32), k, meta)
    assert not at._tiles_ok(torch.zeros(few + many + 1, 18, 128), k, meta)
    assert at.AttentionMetadata.build([1], [9], [[0]], 16, "cuda", "hip").prefill_tiles is None
    ops = load_paged_attention()
    q = torch.zeros(4, 4, 128, device="cuda")
    with pytest.raises(RuntimeError, match="tile 0 outside"):  # more tokens than the batch has
        ops.paged_attention_prefill_(torch.empty_like(q), q, k, k, None, None, meta.block_tables,
                                     meta.prefill_tiles, meta.prefill_tiles_host, 16, 1.0)


@pytest.mark.parametrize("int8", [True, False])
@pytest.mark.parametrize("q_lens,ctx,geom", [([100], [100], (4, 2, 64, 16)), ([70, 1], [1500, 30], (3, 1, 128, 16))])
def test_infinities_stay_where_they_are(gpu, int8, q_lens, ctx, geom):
    """An infinite value reaches its own channel only, an infinite key the tokens it scores +inf or NaN
    (-inf is a weight of 0), an infinite value scale the channels whose code is not 0, also where
    the weight is small (down to e^-40), over one chunk and several: as float64 has it."""
    q, k, v, tables, meta, dev, mult = make(9, q_lens, ctx, geom, int8)
    n, inf = ctx[0], np.inf
    a, b, c = (tables[0][t // 16] * 16 + t % 16 for t in (n - 90, n - 40, n - 3))
    if int8:
        kq, vq, ks, vs = (t.cpu().numpy() for t in dev)
        vs[[a, b], 0], ks[b, 0], vq[a, 0, 5] = inf, 12 * ks[b, 0], 0
        with np.errstate(invalid="ignore"):
            k, v = mr.kv_dequantize(kq, ks), mr.kv_dequantize(vq, vs)
        host = kq, vq, ks, vs
    else:
        v[a, 0, 7], v[b, 0, 9], k[c, 0, 11] = inf, -inf, inf
        k[b] *= 12
        host = k, v, None, None
    for t, h in zip(dev, host):
        if t is not None:
            t.copy_(torch.from_numpy(h))
    got = run(q, meta, dev, mult, geom[2]).cpu().numpy()
    with np.errstate(invalid="ignore"):
        want = reference(q, k, v, q_lens, ctx, tables, geom, mult)
    fine = np.isfinite(want)
    np.testing.assert_array_equal(got[~fine], want[~fine].astype(F32))
    assert np.linalg.norm(got[fine] - want[fine]) <= 2e-6 * np.linalg.norm(want[fine])
    last = want[q_lens[0] - 2: q_lens[0], : geom[0] // geom[1]]
    assert np.isinf(want).any() and (int8 or (np.isfinite(last).any() and np.isnan(last).any()))


# many chunks of one tile beside tiles of one chunk, more chunks than a merge round takes, a context of
# about the most chunks, tiles out of order; and partly filled tiles of one chunk
@pytest.mark.parametrize("q_lens,ctx,geom,order", [
    ([700, 20, 130], [700, 3000, 400], (4, 2, 64, 16), 1), ([700, 20, 130], [700, 3000, 400], (4, 2, 64, 16), -1),
    ([20], [17000], (2, 1, 128, 16), 1), ([300, 300], [300, 1500], (6, 2, 128, 16), -1),
    ([17, 33], [17, 64], (3, 1, 64, 16), 1)])
def test_chunks_of_ragged_tiles(gpu, q_lens, ctx, geom, order):
    q, k, v, tables, meta, dev, mult = make(11, q_lens, ctx, geom, True)
    tiles = meta.prefill_tiles_host.flip(0) if order < 0 else meta.prefill_tiles_host
    tiles = tiles.contiguous()
    lib, d = cu.capi(), geom[2]
    need = lib.llmserve_paged_attention_prefill_workspace_bytes(tiles.data_ptr(), len(tiles), *geom[:3])
    assert (need > 0) == (max(ctx) > 64)  # some tile is split
    qd, td, md = torch.from_numpy(q).cuda(), tiles.cuda(), torch.from_numpy(mult).cuda()
    out = torch.full((q.size + 4096,), -7.5, device="cuda")
    ws = torch.full((need + 4096,), 0x5A, dtype=torch.uint8, device="cuda")
    cu.check(lib.llmserve_paged_attention_prefill(
        cu._p(qd), *(cu._p(t) for t in dev), cu._p(meta.block_tables), len(ctx), cu._p(td), tiles.data_ptr(), len(tiles),
        cu._p(out), len(q), *geom[:3], dev[0].shape[0], meta.block_tables.shape[1], geom[3], d ** -0.5, cu._p(md),
        cu._p(ws), need, cu._stream()))
    assert (out[q.size:] == -7.5).all() and (ws[need:] == 0x5A).all()
    close(out[: q.size].view(q.shape), reference(q, k, v, q_lens, ctx, tables, geom, mult))
