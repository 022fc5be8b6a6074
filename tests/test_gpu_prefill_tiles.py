"""Prefill over tile images: segment edges, row remainders and the running max (GPU).

The kernels that multiply from pre-dequantized page images cut the row blocks
into segments of any length from one page up, visit a segment's pages in a
rotated order and run several pages at once, so the cases below have segments
of one, two and more pages, a last block with few rows, a last page with few
keys, and scores that keep rising so that the running max moves late and often.
"""
from __future__ import annotations

import math

import numpy as np
import pytest
import torch

from gpu_cases import DEV, Cache, assert_close, fill_sequence, random_tables, seeded_normal
from k8v4_v030.layout import PAGE, PageLayout
from k8v4_v030.prefill import hip_prefill
from oracle import torch_cpu
from oracle.paged import Geometry

pytestmark = pytest.mark.gpu


def _run(cache, q, row, seq_len):
    out = torch.full(q.shape, float("nan"), dtype=torch.float32, device=DEV)
    hip_prefill(q.to(DEV), cache.views, row.to(device=DEV, dtype=torch.int32), seq_len, 1,
                1.0 / math.sqrt(q.shape[2]), out=out)
    torch.cuda.synchronize()
    return out.cpu().numpy()


def _want(cache, q, row, seq_len):
    lay = cache.layout
    views = torch_cpu.region_views(torch.from_numpy(cache.blob().copy()), Geometry(lay.hkv, lay.head_dim))
    return torch_cpu.prefill(views, q, row.long(), seq_len, 1.0 / math.sqrt(lay.head_dim)).numpy()


@pytest.mark.parametrize("hkv,d,q_len,seq_len", [
    # whole prompts: 27 steps a work-group over blocks of 1 to 68 pages
    (2, 256, 4300, 4300), (4, 256, 2817, 3901),
    # one key in the last page, six rows in the last block
    (2, 256, 2049, 16385),
    (4, 128, 129, 129), (2, 128, 171, 65), (4, 128, 683, 1985), (2, 128, 1999, 1999),
    # 64-row waves of 128 dims: 40 pages a segment or more
    (4, 128, 1025, 12801), (2, 128, 2100, 14913), (2, 128, 5000, 6000),
])
def test_segments_of_every_length(gpu_ops, hkv, d, q_len, seq_len):
    seq_len = max(q_len, seq_len)
    print("prefill tiles hkv=%d d=%d q=%d seq=%d" % (hkv, d, q_len, seq_len), flush=True)
    assert gpu_ops.prefill_uses_tiles(seq_len, q_len, hkv, d)
    lay = PageLayout(hkv, d)
    gen = torch.Generator().manual_seed(q_len + seq_len + hkv + d)
    pages = -(-seq_len // PAGE)
    cache = Cache(pages + 3, lay)
    table = random_tables(gen, [seq_len], pages + 3)
    fill_sequence(gpu_ops, cache, gen, table[0], seq_len)
    q = seeded_normal(gen, (q_len, lay.hq, d))
    assert_close(_run(cache, q, table[0], seq_len), _want(cache, q, table[0], seq_len), what="tiles")


@pytest.mark.parametrize("vmax", [65504.0, 1.0])
@pytest.mark.parametrize("d,q_len,seq_len", [(256, 2100, 8192), (128, 200, 8192), (128, 2100, 8192)])
def test_running_max_moves_late_and_often(gpu_ops, d, q_len, seq_len, vmax):
    """Each 32-token chunk scores 0.25 (log2 units) above the one before, with
    V rows of +-vmax whose sign alternates from chunk to chunk: with the widest
    V an fp16 row can hold P' = p * v_scale overflows past a lag of 2.9, with a
    small one the lag may grow to 8.

    Tolerance: scores reach 64 log2 units, the keys of the tile images are
    rounded to fp16 once (2^-12 relative), so two neighbouring chunks' weights
    may shift against each other by 2 * 64 * 2^-12 log2 units = 2.2 %."""
    print("prefill rising d=%d q=%d vmax=%g" % (d, q_len, vmax), flush=True)
    lay = PageLayout(2, d)
    gen = torch.Generator().manual_seed(d + q_len)
    pages = seq_len // PAGE
    cache = Cache(pages + 3, lay)
    table = random_tables(gen, [seq_len], pages + 3)
    t = torch.arange(seq_len)
    per_c = math.sqrt(d) * 1.4426950408889634  # log2 score of a ones query per unit of c
    c = (t // 32).float() * (0.25 / per_c)
    k = (c[:, None, None] * torch.ones((seq_len, 2, d))).to(torch.float16)
    sign = 1.0 - 2.0 * ((t // 32) % 2).float()
    v = (sign[:, None, None] * torch.full((seq_len, 2, d), vmax)).to(torch.float16)
    v[:, :, 1::2] = -v[:, :, 1::2]
    slots = (table[0].long()[t // PAGE] * PAGE + t % PAGE).to(DEV)
    cache.store(gpu_ops, k.to(DEV), v.to(DEV), slots)
    q = torch.ones((q_len, 12, d), dtype=torch.float16)
    assert gpu_ops.prefill_uses_tiles(seq_len, q_len, 2, d)
    want = _want(cache, q, table[0], seq_len)
    assert np.abs(want).max() > 0.05 * vmax
    assert_close(_run(cache, q, table[0], seq_len), want, atol=0.022 * vmax, rtol=1e-2, what="rising scores")


def test_a_workspace_for_one_head_still_serves_the_call(gpu_ops):
    """The images of one KV head at a time fit a workspace of the partial
    states of a one-head launch plus one head's images; a larger one lets
    several heads share a launch.  Both give the oracle's rows."""
    lay = PageLayout(4, 128)
    q_len = seq_len = 1025
    gen = torch.Generator().manual_seed(1025)
    pages = -(-seq_len // PAGE)
    cache = Cache(pages + 3, lay)
    table = random_tables(gen, [seq_len], pages + 3)
    fill_sequence(gpu_ops, cache, gen, table[0], seq_len)
    q = seeded_normal(gen, (q_len, lay.hq, 128))
    want = _want(cache, q, table[0], seq_len)
    blocks = -(-q_len * 6 // 256)
    steps = sum(min(q_len - 1, (256 * b + 255) // 6) // PAGE + 1 for b in range(blocks))
    grid = min(256, steps // 4) // 8 * 8
    one_head = (grid * 2 * 256 * 130 * 4 + 255) // 256 * 256 + pages * 35 * 1024
    full = gpu_ops.prefill_workspace_bytes(seq_len, q_len, 4, 128)
    assert full > one_head
    row = table[0].to(device=DEV, dtype=torch.int32)
    for nbytes in (one_head, full):
        ws = torch.empty(nbytes // 4, dtype=torch.float32, device=DEV)
        out = torch.full(q.shape, float("nan"), dtype=torch.float32, device=DEV)
        gpu_ops.prefill_paged(q.to(DEV), *cache.region_args(), row, seq_len, 1, 1.0 / math.sqrt(128), out, ws)
        torch.cuda.synchronize()
        assert_close(out.cpu().numpy(), want, what="%d bytes" % nbytes)
    with pytest.raises(RuntimeError, match="prefill workspace holds"):
        gpu_ops.prefill_paged(q.to(DEV), *cache.region_args(), row, seq_len, 1, 1.0 / math.sqrt(128),
                              torch.empty(q.shape, dtype=torch.float32, device=DEV),
                              torch.empty(one_head // 4 - 64, dtype=torch.float32, device=DEV))


@pytest.mark.parametrize("d", [128, 256])
def test_batch_of_blocks_of_very_different_length(gpu_ops, d):
    """Row blocks of one page beside blocks of many in one launch: work-groups
    take many short blocks or a part of a long one, and a work-group's range may
    begin or end within the steps that stand for a block's fixed cost."""
    q_lens, ctxs = [11, 64, 128, 17, 33, 90, 12, 100], [0, 0, 9000, 47, 640, 2000, 52, 0]
    lens = [q + c for q, c in zip(q_lens, ctxs)]
    lay = PageLayout(2, d)
    gen = torch.Generator().manual_seed(77 + d)
    pool = sum(-(-n // PAGE) for n in lens) + 3
    cache = Cache(pool, lay)
    table = random_tables(gen, lens, pool)
    for b, n in enumerate(lens):
        fill_sequence(gpu_ops, cache, gen, table[b], n)
    q = seeded_normal(gen, (sum(q_lens), lay.hq, d))
    out = torch.full(q.shape, float("nan"), dtype=torch.float32, device=DEV)
    ws = torch.empty(gpu_ops.prefill_batch_workspace_bytes(2, d) // 4, dtype=torch.float32, device=DEV)
    tok0 = [sum(q_lens[:i]) for i in range(len(q_lens))]
    gpu_ops.prefill_paged_batch(q.to(DEV), *cache.region_args(), table.to(DEV), tok0, q_lens, lens,
                                list(range(len(lens))), 1, 1.0 / math.sqrt(d), out, ws)
    torch.cuda.synchronize()
    for b, n in enumerate(lens):
        rows = slice(tok0[b], tok0[b] + q_lens[b])
        assert_close(out[rows].cpu().numpy(), _want(cache, q[rows], table[b], n), what="sequence %d" % b)


@pytest.mark.parametrize("q_len,ctx", [(129, 26000), (150, 24001), (700, 3000), (1300, 0)])
def test_d256_chunks_over_images_where_the_workspace_has_room(gpu_ops, q_len, ctx):
    """Head dim 256, chunks that run over tile images if the workspace holds
    them and in place otherwise, through the single and the batched entry."""
    hkv, d, seq_len = 4, 256, q_len + ctx
    lay = PageLayout(hkv, d)
    assert not gpu_ops.prefill_uses_tiles(seq_len, q_len, hkv, d)
    gen = torch.Generator().manual_seed(q_len + ctx)
    lens = [seq_len, 200]
    pool = sum(-(-n // PAGE) for n in lens) + 3
    cache = Cache(pool, lay)
    table = random_tables(gen, lens, pool)
    for b, n in enumerate(lens):
        fill_sequence(gpu_ops, cache, gen, table[b], n)
    q = seeded_normal(gen, (q_len + 20, lay.hq, d))
    want = [_want(cache, q[:q_len], table[0], seq_len), _want(cache, q[q_len:], table[1], 200)]
    batch = gpu_ops.prefill_batch_workspace_bytes(hkv, d)
    full = gpu_ops.prefill_workspace_bytes(seq_len, q_len, hkv, d)
    pages = -(-seq_len // PAGE)
    assert full > pages * 66 * 1024  # with the images
    for nbytes in (batch, max(batch, full)):
        ws = torch.empty(nbytes // 4, dtype=torch.float32, device=DEV)
        out = torch.full(q.shape, float("nan"), dtype=torch.float32, device=DEV)
        gpu_ops.prefill_paged(q[:q_len].to(DEV), *cache.region_args(), table[0].to(device=DEV, dtype=torch.int32),
                              seq_len, 1, 1.0 / 16, out[:q_len], ws)
        torch.cuda.synchronize()
        assert_close(out[:q_len].cpu().numpy(), want[0], what="single, %d bytes" % nbytes)
        out.fill_(float("nan"))
        gpu_ops.prefill_paged_batch(q.to(DEV), *cache.region_args(), table.to(DEV), [0, q_len], [q_len, 20], lens,
                                    [0, 1], 1, 1.0 / 16, out, ws)
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        assert_close(got[:q_len], want[0], what="batch, %d bytes" % nbytes)
        assert_close(got[q_len:], want[1], what="batch, second sequence")
