"""GPU parity: partial-prefill attention against the fp32 oracle.

bf16 / fp16 outputs must be within 2e-2 absolute of the fp32 reference; fp32 inputs within
the reference suite's own 1e-4 absolute / 1e-3 relative. Cases restate
synapse_kv_connector/tests/test_triton_kernels.py:396-493 and add GQA + paged cases up to the
Qwen2.5-7B shape (28 q heads / 4 KV heads, head_dim 128, 16384-token context).
"""

from __future__ import annotations

import math

import pytest
import torch

import bench
from oracle import ref_cpu as ref
from semblend_amd import triton_kernels as tk
from tests.helpers import assert_attn_close, gen, randn, recompute_set

pytestmark = pytest.mark.gpu


# ---- dense drop-in (triton_kernels.py:655-734) ----

def test_dense_all_compute_fp32(dev):
    q, k, v = (randn((2, 8, 16), torch.float32, s) for s in (1, 2, 3))
    mask = torch.ones(8, dtype=torch.bool)
    got = tk.partial_prefill_attention(q.to(dev), k.to(dev), v.to(dev), mask.to(dev),
                                       1.0 / math.sqrt(16))
    assert_attn_close(got, ref.partial_prefill_attention(q, k, v, mask, 1.0 / math.sqrt(16)))


def test_dense_reuse_rows_zero_and_full_context(dev):
    q, k, v = (randn((2, 8, 16), torch.float32, s) for s in (4, 5, 6))
    mask = torch.tensor([True, False, True, False, True, False, True, False])
    got = tk.partial_prefill_attention(q.to(dev), k.to(dev), v.to(dev), mask.to(dev)).cpu()
    for p in (1, 3, 5, 7):
        assert torch.all(got[:, p] == 0)
    assert_attn_close(got, ref.partial_prefill_attention(q, k, v, mask))
    q1, k1, v1 = (randn((1, 4, 8), torch.float32, s) for s in (7, 8, 9))
    m1 = torch.tensor([False, False, False, True])
    got1 = tk.partial_prefill_attention(q1.to(dev), k1.to(dev), v1.to(dev), m1.to(dev))
    assert_attn_close(got1, ref.partial_prefill_attention(q1, k1, v1, m1))


def test_dense_empty_mask(dev):
    q = randn((2, 4, 8), torch.float32, 10).to(dev)
    got = tk.partial_prefill_attention(q, q, q, torch.zeros(4, dtype=torch.bool, device=dev))
    assert torch.all(got == 0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("seq_len", [1, 77, 300, 1000])
def test_dense_mfma(dev, dtype, head_dim, seq_len):
    h = 3
    q, k, v = (randn((h, seq_len, head_dim), dtype, 20 + s) for s in range(3))
    mask = torch.rand(seq_len, generator=gen(seq_len)) < 0.3
    mask[-1] = True
    got = tk.partial_prefill_attention(q.to(dev), k.to(dev), v.to(dev), mask.to(dev))
    want = ref.partial_prefill_attention(q, k, v, mask)
    assert got.dtype == dtype
    assert torch.all(got.cpu()[:, ~mask] == 0)
    assert_attn_close(got, want)


@pytest.mark.parametrize("n_rows", [1, 40, 700])
def test_dense_split_from_device_row_count(dev, n_rows):
    """The dense drop-in knows its row count only on the device, so its kernels derive the
    key-range split from that count: a few rows of a long context run in many chunks (40
    rows of 8192 keys: 512-key chunks, merged by the general path past four chunks), more
    rows in fewer; the launch and the workspace cover every count."""
    h, s = 4, 8192
    q, k, v = (randn((h, s, 128), torch.bfloat16, 320 + i) for i in range(3))
    mask = torch.zeros(s, dtype=torch.bool)
    mask[torch.randperm(s, generator=gen(323 + n_rows))[:n_rows]] = True
    mask[s - 1] = True
    got = tk.partial_prefill_attention(q.to(dev), k.to(dev), v.to(dev), mask.to(dev))
    assert torch.all(got.cpu()[:, ~mask] == 0)
    assert_attn_close(got, ref.partial_prefill_attention(q, k, v, mask))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_dense_other_head_dim(dev, dtype):
    """head_dim 96 takes the general (non-MFMA) kernel."""
    q, k, v = (randn((2, 130, 96), dtype, 30 + s) for s in range(3))
    mask = torch.rand(130, generator=gen(31)) < 0.5
    got = tk.partial_prefill_attention(q.to(dev), k.to(dev), v.to(dev), mask.to(dev), 0.3)
    assert_attn_close(got, ref.partial_prefill_attention(q, k, v, mask, 0.3))


# ---- GQA over a paged cache ----

def _paged_case(hq, hkv, d, seq_len, n_rows, dtype, seed, nb=None, bs=16):
    nblk = (seq_len + bs - 1) // bs
    nb = nb or nblk + 7
    kv = randn((nb, 2, hkv, bs, d), dtype, seed)
    bt = torch.randperm(nb, generator=gen(seed + 1))[:nblk].to(torch.int32)
    pos = recompute_set(seq_len, n_rows, seed + 2, chunk=min(256, seq_len // 4 or 1))
    q = randn((pos.shape[0], hq, d), dtype, seed + 3)
    return q, kv, bt, pos


def test_paged_gqa_qwen05b_fp32(dev):
    """Qwen2.5-0.5B attention: 14 q heads / 2 KV heads, head_dim 64, fp32, 1024 tokens,
    154 query rows drawn without replacement."""
    kv = randn((128, 2, 2, 16, 64), torch.float32, 40)
    bt = torch.randperm(128, generator=gen(41))[:64].to(torch.int32)
    pos = torch.randperm(1024, generator=gen(42))[:154].sort().values.to(torch.int32)
    q = randn((154, 14, 64), torch.float32, 43)
    got = tk.partial_prefill_attention_paged(q.to(dev), kv.to(dev), bt.to(dev), pos.to(dev))
    assert_attn_close(got, ref.partial_attention_paged(q, kv, bt, pos))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d", [(28, 4, 128), (32, 8, 128), (14, 2, 64), (8, 8, 128)])
def test_paged_gqa_mfma(dev, dtype, hq, hkv, d):
    q, kv, bt, pos = _paged_case(hq, hkv, d, 2048, 300, dtype, 50)
    got = tk.partial_prefill_attention_paged(q.to(dev), kv.to(dev), bt.to(dev), pos.to(dev))
    assert_attn_close(got, ref.partial_attention_paged(q, kv, bt, pos))


@pytest.mark.parametrize("bs", [24, 32, 1])
def test_paged_gqa_block_sizes(dev, bs):
    """Block sizes other than 16. 24 is not a power of two, so the block of a key is found
    by division and its offset with 64-bit products; 1 puts every key in its own block."""
    q, kv, bt, pos = _paged_case(28, 4, 128, 1500, 200, torch.bfloat16, 80 + bs, bs=bs)
    got = tk.partial_prefill_attention_paged(q.to(dev), kv.to(dev), bt.to(dev), pos.to(dev))
    assert_attn_close(got, ref.partial_attention_paged(q, kv, bt, pos))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("seq_len", [384, 383])
def test_paged_gqa_every_tile_count(dev, dtype, seq_len):
    """Every position of a short context is a query row, so the row tiles' key ranges grow
    from one 64-key tile to six (and, at 383, end one key short of a tile): the tile loop
    runs its two-tile body zero to two times and finishes with one or two tiles, for every
    combination."""
    q, kv, bt, _ = _paged_case(28, 4, 128, seq_len, 8, dtype, 70 + seq_len)
    pos = torch.arange(seq_len, dtype=torch.int32)
    q = randn((seq_len, 28, 128), dtype, 71 + seq_len)
    got = tk.partial_prefill_attention_paged(q.to(dev), kv.to(dev), bt.to(dev), pos.to(dev))
    assert_attn_close(got, ref.partial_attention_paged(q, kv, bt, pos))


def test_paged_gqa_position_major_layout(dev):
    """A cache stored [blocks, block_size, 2, kv_heads, head_dim] and viewed as
    [blocks, 2, kv_heads, block_size, head_dim]: the position stride (2·H·D) exceeds the
    head stride, and K and V of a position sit next to each other."""
    q, kv, bt, pos = _paged_case(32, 8, 128, 1200, 150, torch.bfloat16, 90)
    store = kv.permute(0, 3, 1, 2, 4).contiguous()        # [nb, bs, 2, H, D]
    view = store.to(dev).permute(0, 2, 3, 1, 4)           # [nb, 2, H, bs, D]
    assert not view.is_contiguous()
    got = tk.partial_prefill_attention_paged(q.to(dev), view, bt.to(dev), pos.to(dev))
    assert_attn_close(got, ref.partial_attention_paged(q, kv, bt, pos))


def test_paged_gqa_no_rows(dev):
    q, kv, bt, _ = _paged_case(28, 4, 128, 256, 8, torch.bfloat16, 95)
    got = tk.partial_prefill_attention_paged(q[:0].to(dev), kv.to(dev), bt.to(dev),
                                             torch.zeros(0, dtype=torch.int32, device=dev))
    assert got.shape == (0, 28, 128)


def test_paged_gqa_long_context_many_chunks(dev):
    """A 65536-token context with few rows: the planner splits the key range into 512-key
    chunks to fill the GPU, so the last rows span 128 chunks that the merge combines. Rows
    at the start, at chunk limits and at the last position, plus random ones."""
    ctx, bs = 65536, 16
    nblk = ctx // bs
    kv = randn((nblk + 3, 2, 1, bs, 128), torch.bfloat16, 96)
    bt = torch.randperm(nblk + 3, generator=gen(97))[:nblk].to(torch.int32)
    pos = torch.cat([torch.tensor([0, 1, 16383, 16384, 32767, 49152, 65534, 65535]),
                     torch.randint(0, ctx, (40,), generator=gen(98))]).unique()
    pos = pos.sort().values.to(torch.int32)
    q = randn((pos.shape[0], 8, 128), torch.bfloat16, 99)
    got = tk.partial_prefill_attention_paged(q.to(dev), kv.to(dev), bt.to(dev), pos.to(dev))
    assert_attn_close(got, ref.partial_attention_paged(q, kv, bt, pos))


def test_paged_gqa_unsorted_positions(dev):
    q, kv, bt, pos = _paged_case(28, 4, 128, 1024, 200, torch.bfloat16, 60)
    perm = torch.randperm(pos.shape[0], generator=gen(61))
    q, pos = q[perm].contiguous(), pos[perm].contiguous()
    got = tk.partial_prefill_attention_paged(q.to(dev), kv.to(dev), bt.to(dev), pos.to(dev))
    assert_attn_close(got, ref.partial_attention_paged(q, kv, bt, pos))


def test_paged_gqa_full_size_7b(dev):
    """The 7B attention workload at full size: 16384-token context, 2458 query rows
    (first 256 tokens, two random 256-token chunks, the rest scattered), 28/4 heads, bf16.
    Every output row is compared with the oracle."""
    q, kv, bt, pos = _paged_case(28, 4, 128, 16384, 2458, torch.bfloat16, 70, nb=2048)
    assert pos.shape[0] == 2458
    got = tk.partial_prefill_attention_paged(q.to(dev), kv.to(dev), bt.to(dev), pos.to(dev))
    want = ref.partial_attention_paged(q, kv, bt, pos)
    assert_attn_close(got.cpu(), want)


def test_paged_gqa_bench_workload(dev):
    """The attention phase that bench.py times, on its own inputs (built by the same seeded
    code on the device): all 2458 rows of all 28 q-heads against the oracle."""
    inp = bench.build_inputs(dev)
    q, kv, pos = inp["attn_q"], inp["attn_kv"], inp["attn_pos"]
    bt = inp["block_table"]
    got = tk.partial_prefill_attention_paged(q, kv, bt, pos)
    want = ref.partial_attention_paged(q.cpu(), kv.cpu(), bt.cpu(), pos.cpu())
    assert_attn_close(got.cpu(), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_paged_gqa_rising_scores_rescale(dev, dtype):
    """Scores that keep rising along the context, so the kernel's reference max must move
    (O and l rescaled, the next tile's scores shifted) many times within one row: K rows are
    scaled from 1 to 24 (bf16) or 1 to 4 (fp16) along the positions, so a late tile's
    scores exceed the first tile's maximum by far more than the 2^64 (bf16) or 2^8 (fp16)
    tile-sum bound of P. Rows at every 64-key tile boundary and at the end of the context,
    with several key chunks for the long rows."""
    hq, hkv, d, bs, ctx = 8, 2, 128, 16, 4096
    nb = ctx // bs
    top = 24.0 if dtype == torch.bfloat16 else 4.0
    kv = randn((nb, 2, hkv, bs, d), torch.float32, 120)
    scale = torch.linspace(1.0, top, ctx).view(nb, bs)          # per position
    kv[:, 0] *= scale[:, None, :, None]
    kv = kv.to(dtype)
    bt = torch.arange(nb, dtype=torch.int32)
    pos = torch.cat([torch.arange(63, ctx, 256), torch.tensor([0, 64, 4094, 4095]),
                     torch.randint(0, ctx, (60,), generator=gen(121))]).unique()
    pos = pos.sort().values.to(torch.int32)
    q = randn((pos.shape[0], hq, d), dtype, 122)
    got = tk.partial_prefill_attention_paged(q.to(dev), kv.to(dev), bt.to(dev), pos.to(dev))
    want = ref.partial_attention_paged(q, kv, bt, pos)
    # the softmax is peaked: most rows put nearly all weight on a few late keys
    assert float(want.abs().amax()) > 1.0
    assert_attn_close(got, want)


# ---- host-planned launches (split + longest-first order) ----

def test_paged_gqa_planned_bench_workload(dev):
    """The planned launch on the bench's 7B inputs: every row against the oracle, and a
    plan of other positions (same shape) is still correct, only slower."""
    inp = bench.build_inputs(dev)
    q, kv, pos, bt = inp["attn_q"], inp["attn_kv"], inp["attn_pos"], inp["block_table"]
    plan = tk.plan_partial_attention_paged(inp["pos_cpu"], 28, 4, 128, 16, bt.shape[0],
                                           torch.bfloat16, dev)
    assert plan.max_chunks >= 2 and plan.ks_rest < plan.ks_first
    got = tk.partial_prefill_attention_paged(q, kv, bt, pos, plan=plan)
    want = ref.partial_attention_paged(q.cpu(), kv.cpu(), bt.cpu(), pos.cpu())
    assert_attn_close(got.cpu(), want)
    other = recompute_set(16384, pos.shape[0], 5)
    plan2 = tk.plan_partial_attention_paged(other, 28, 4, 128, 16, bt.shape[0], torch.bfloat16,
                                            dev)
    got2 = tk.partial_prefill_attention_paged(q, kv, bt, pos, plan=plan2)
    assert_attn_close(got2.cpu(), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d,seq,rows,bs", [(28, 4, 128, 4096, 600, 16),
                                                   (32, 8, 128, 8192, 800, 16),
                                                   (14, 2, 64, 3000, 450, 32),
                                                   (8, 8, 128, 2048, 300, 24)])
def test_paged_gqa_planned_shapes(dev, dtype, hq, hkv, d, seq, rows, bs):
    q, kv, bt, pos = _paged_case(hq, hkv, d, seq, rows, dtype, 130 + hq + bs, bs=bs)
    plan = tk.plan_partial_attention_paged(pos, hq, hkv, d, bs, bt.shape[0], dtype, dev)
    got = tk.partial_prefill_attention_paged(q.to(dev), kv.to(dev), bt.to(dev), pos.to(dev),
                                             plan=plan)
    assert_attn_close(got, ref.partial_attention_paged(q, kv, bt, pos))


def test_paged_gqa_planned_unsorted_and_fp32(dev):
    """Positions in any order (the plan reads them as given); fp32 takes the VALU kernel,
    for which the plan is empty."""
    q, kv, bt, pos = _paged_case(28, 4, 128, 2048, 400, torch.bfloat16, 140)
    perm = torch.randperm(pos.shape[0], generator=gen(141))
    q, pos = q[perm].contiguous(), pos[perm].contiguous()
    plan = tk.plan_partial_attention_paged(pos, 28, 4, 128, 16, bt.shape[0], torch.bfloat16, dev)
    got = tk.partial_prefill_attention_paged(q.to(dev), kv.to(dev), bt.to(dev), pos.to(dev),
                                             plan=plan)
    assert_attn_close(got, ref.partial_attention_paged(q, kv, bt, pos))
    q32, kv32 = q.float(), kv.float()
    plan32 = tk.plan_partial_attention_paged(pos, 28, 4, 128, 16, bt.shape[0], torch.float32,
                                             dev)
    assert plan32.max_chunks == 0 and plan32.order.numel() == 0
    got32 = tk.partial_prefill_attention_paged(q32.to(dev), kv32.to(dev), bt.to(dev),
                                               pos.to(dev), plan=plan32)
    assert_attn_close(got32, ref.partial_attention_paged(q32, kv32, bt, pos))
    with pytest.raises(ValueError, match="another shape"):
        tk.partial_prefill_attention_paged(q.to(dev)[:10], kv.to(dev), bt.to(dev),
                                           pos.to(dev)[:10], plan=plan)


# ---- fp32 on the fp32 matrix cores (head_dim 64 and 128) ----

@pytest.mark.parametrize("hq,hkv,d,seq,rows,bs", [
    (14, 2, 64, 65, 1, 16),       # one row, one key past a 64-key tile
    (14, 2, 64, 64, 9, 16),       # 63 flattened rows: one short of a row tile
    (32, 8, 128, 700, 17, 16),    # 68 flattened rows: a second row tile of 4
    (28, 4, 128, 33, 33, 24),     # every row; blocks that are no power of two
    (4, 4, 128, 4096, 3, 32),     # few rows of a long context: many key chunks
    (4, 4, 64, 700, 700, 16),     # no GQA, every row
    (64, 16, 64, 2000, 1100, 16)])  # enough row tiles to run unsplit
def test_paged_fp32_tiles_and_splits(dev, hq, hkv, d, seq, rows, bs):
    """Row tiles of 64, key tiles of 4096 / head_dim and the key split at their edges (the shortest
    contexts take the one-launch kernel); a call whose caller sized no workspace (an empty launch
    plan through the C entry) runs unsplit."""
    q, kv, bt, pos = _paged_case(hq, hkv, d, seq, rows, torch.float32, 400 + d + rows, bs=bs)
    qd, kvd, btd, posd = q.to(dev), kv.to(dev), bt.to(dev), pos.to(dev)
    want = ref.partial_attention_paged(q, kv, bt, pos)
    got = tk.partial_prefill_attention_paged(qd, kvd, btd, posd)
    # two orders of summing d products and up to seq weighted values: a few 2^-24 of |out| <= 1
    assert float((got.cpu() - want).abs().max()) <= 5e-6 * max(1.0, float(want.abs().max()))
    out = torch.full_like(qd, float("nan"))
    from semblend_amd import _lib
    _lib.call("sb_partial_attention_paged_planned", out.data_ptr(), qd.data_ptr(),
              kvd.data_ptr(), btd.data_ptr(), posd.data_ptr(), None, 0, 0, 0, 0, None, 0,
              q.shape[0], hq, hkv, d, bs, kv.shape[0], bt.shape[0], 1.0 / math.sqrt(d),
              _lib.strides(qd), _lib.strides(out), _lib.strides(kvd), _lib.dtype_code(qd),
              _lib.stream_handle(dev))
    assert float((out.cpu() - want).abs().max()) <= 5e-6 * max(1.0, float(want.abs().max()))


@pytest.mark.parametrize("d", [64, 128])
def test_fp32_masked_keys_never_reach_a_row(dev, d):
    """NaN and infinite K / V at positions past a row (but inside its key tile) leave the row as
    it is without them; a row that does attend them takes the same non-finite elements."""
    h, s = 2, 200
    q, k, v = (randn((h, s, d), torch.float32, 430 + i) for i in range(3))
    v[0, 100, 3], v[1, 150, 5] = float("nan"), float("inf")
    k[0, 120, 1], v[0, 199] = float("nan"), float("-inf")
    for rows in ([90, 99, 100, 119, 120, 149, 150, 198, 199], [60, 110]):
        mask = torch.zeros(s, dtype=torch.bool)
        mask[rows] = True
        got = tk.partial_prefill_attention(q.to(dev), k.to(dev), v.to(dev), mask.to(dev)).cpu()
        for hh in range(h):
            for p in rows:
                w = torch.softmax((k[hh, :p + 1].double() @ q[hh, p].double()) / math.sqrt(d), 0)
                want = (w[:, None] * v[hh, :p + 1].double()).sum(0)
                fin = torch.isfinite(want)
                assert torch.equal(torch.isnan(got[hh, p]), torch.isnan(want)), (hh, p)
                assert torch.equal(torch.isfinite(got[hh, p]), fin), (hh, p)
                assert float((got[hh, p].double() - want)[fin].abs().max().nan_to_num(0)
                             if fin.any() else 0) <= 1e-5


def test_fp32_rising_scores_and_strided_inputs(dev):
    """Scores that rise along the context move the row maximum in every tile; query and cache
    are views with a wider head stride."""
    hq, hkv, d, ctx = 8, 2, 64, 1500
    kv = randn((100, 2, hkv, 16, 2 * d), torch.float32, 440)[..., :d]
    kv[:, 0] *= torch.linspace(0.2, 8.0, 100)[:, None, None, None]
    bt = torch.arange(94, dtype=torch.int32)
    pos = recompute_set(ctx, 130, 441, chunk=16)
    q = randn((pos.shape[0], hq, 2 * d), torch.float32, 442)[..., :d]
    big = torch.zeros((100, 2, hkv, 16, 2 * d), device=dev)
    big[..., :d] = kv.to(dev)
    bq = torch.zeros((pos.shape[0], hq, 2 * d), device=dev)
    bq[..., :d] = q.to(dev)
    got = tk.partial_prefill_attention_paged(bq[..., :d], big[..., :d], bt.to(dev), pos.to(dev))
    assert_attn_close(got, ref.partial_attention_paged(q, kv, bt, pos))


# ---- small calls: fine key splits and the merge that spreads a row's chunks over lanes ----

@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d,ctx,rows,bs", [
    (4, 2, 64, 384, 3, 16),      # whole: one chunk
    (4, 2, 128, 400, 3, 16),     # four chunks of 128: the merge of few chunks
    (4, 2, 128, 900, 2, 24),     # eight chunks: the last holds 4 keys
    (14, 2, 64, 8000, 1, 16),    # 63 chunks: two batches of the wide merge
    (32, 8, 128, 3200, 40, 32)])
def test_small_calls_split_and_merge(dev, dtype, hq, hkv, d, ctx, rows, bs):
    g = gen(500 + ctx)
    nb = -(-ctx // bs)
    kv = randn((nb + 3, 2, hkv, bs, d), dtype, 501)
    bt = torch.randperm(nb + 3, generator=g)[:nb].to(torch.int32)
    pos = torch.cat([torch.tensor([0, ctx - 1])[:rows],
                     torch.randperm(ctx - 2, generator=g)[:max(0, rows - 2)] + 1])
    pos = pos.sort().values.to(torch.int32)
    q = randn((pos.numel(), hq, d), dtype, 502)
    got = tk.partial_prefill_attention_paged(q.to(dev), kv.to(dev), bt.to(dev), pos.to(dev))
    assert_attn_close(got, ref.partial_attention_paged(q, kv, bt, pos))
    half = tk.partial_prefill_attention_paged_varlen(
        torch.cat([q, q]).to(dev), kv.to(dev), torch.stack([bt, bt]).to(dev),
        torch.cat([pos, pos]).to(dev), [pos.numel()] * 2, [nb] * 2)
    assert_attn_close(half[pos.numel():], ref.partial_attention_paged(q, kv, bt, pos))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows", [[2999], [0, 1500, 2999], list(range(0, 3000, 9))])
def test_dense_few_rows_of_a_long_context(dev, dtype, rows):
    """The device-derived split of few rows (fine chunks, wide strided merge) and of many."""
    q, k, v = (randn((2, 3000, 64), dtype, 510 + i) for i in range(3))
    mask = torch.zeros(3000, dtype=torch.bool)
    mask[rows] = True
    got = tk.partial_prefill_attention(q.to(dev), k.to(dev), v.to(dev), mask.to(dev)).cpu()
    want = ref.partial_prefill_attention(q.float(), k.float(), v.float(), mask)
    assert_attn_close(got[:, rows], want[:, rows].to(dtype))
    assert not bool(got[:, ~mask].any())


@pytest.mark.parametrize("hq,hkv,d,ctx,rows", [
    (32, 8, 128, 4000, 600),    # ten row tiles: one item per slot at most
    (28, 4, 128, 9000, 1500),   # an average slot of 2300-5500 keys: about two rounds
    (28, 4, 64, 20000, 2200),   # more than that
    (28, 28, 64, 1500, 2000)])  # more row tiles than slots
def test_key_split_rules_cover_every_key(dev, hq, hkv, d, ctx, rows):
    """Sampled rows of each split rule against the oracle, the same rows through the batched
    entry (its own split) beside a short request, and all rows against a planned launch."""
    g = gen(600 + ctx)
    rows = min(rows, ctx)
    nb = -(-ctx // 16)
    kv = randn((nb + 40, 2, hkv, 16, d), torch.bfloat16, 601)
    bt = torch.randperm(nb + 40, generator=g)[:nb].to(torch.int32)
    pos = torch.randperm(ctx, generator=g)[:rows].sort().values.to(torch.int32)
    q = randn((rows, hq, d), torch.bfloat16, 602)
    qd, kvd, btd, posd = q.to(dev), kv.to(dev), bt.to(dev), pos.to(dev)
    got = tk.partial_prefill_attention_paged(qd, kvd, btd, posd)
    sel = torch.randperm(rows, generator=g)[:12].sort().values
    sel[0], sel[-1] = 0, rows - 1
    want = ref.partial_attention_paged(q[sel], kv, bt, pos[sel])
    assert_attn_close(got.cpu()[sel], want)
    plan = tk.plan_partial_attention_paged(pos, hq, hkv, d, 16, nb, torch.bfloat16, dev)
    planned = tk.partial_prefill_attention_paged(qd, kvd, btd, posd, plan=plan)
    assert_attn_close(got, planned.float().cpu())
    short = min(rows, 40)
    tables = torch.stack([btd, btd])
    both = tk.partial_prefill_attention_paged_varlen(
        torch.cat([qd, qd[:short]]), kvd, tables, torch.cat([posd, posd[:short]]),
        [rows, short], [nb, nb])
    assert_attn_close(both[:rows].cpu()[sel], want)
    assert_attn_close(both[rows:], got[:short].float().cpu())


@pytest.mark.parametrize("hq,hkv,d,ctx,rows", [
    (28, 4, 128, 6573, 273),    # few row tiles: even chunks longer than 512 keys
    (28, 4, 128, 2630, 490),    # few row tiles: one round in chunks of 512
    (32, 8, 128, 513, 300),     # one key past the contexts that stay whole
    (28, 4, 128, 8247, 786),    # late rows: even chunks
    (28, 4, 64, 15291, 1304)])  # late rows: the average work of a slot
@pytest.mark.parametrize("order", ["uniform", "late", "late first"])
def test_key_split_by_the_first_position(dev, hq, hkv, d, ctx, rows, order):
    """Splits chosen by the row count and by the first row's position: uniform rows, the last rows
    of the context, and a first row past 3/8 of it before rows that are not."""
    g = gen(640 + ctx)
    nb = -(-ctx // 16)
    kv = randn((nb + 8, 2, hkv, 16, d), torch.bfloat16, 641)
    bt = torch.randperm(nb + 8, generator=g)[:nb].to(torch.int32)
    if order == "late":
        pos = torch.arange(ctx - rows, ctx, dtype=torch.int32)
    else:
        pos = torch.randperm(ctx, generator=g)[:rows].sort().values.to(torch.int32)
    if order == "late first":
        pos = pos.flip(0)
    q = randn((rows, hq, d), torch.bfloat16, 642)
    got = tk.partial_prefill_attention_paged(q.to(dev), kv.to(dev), bt.to(dev), pos.to(dev)).cpu()
    sel = torch.randperm(rows, generator=g)[:10].sort().values
    sel[0], sel[-1] = 0, rows - 1
    assert_attn_close(got[sel], ref.partial_attention_paged(q[sel], kv, bt, pos[sel]))


@pytest.mark.parametrize("first,rows", [(1535, 500), (1536, 500), (3500, 596), (4095, 1), (0, 4096)])
def test_dense_split_by_the_first_position(dev, first, rows):
    """The device-derived split on both sides of 3/8 of the context (28 heads: 56 to 84 row tiles
    of 2 and 3 per head)."""
    h, s, d = 28, 4096, 64
    q, k, v = (randn((h, s, d), torch.bfloat16, 650 + i) for i in range(3))
    mask = torch.zeros(s, dtype=torch.bool)
    mask[first:first + rows] = True
    got = tk.partial_prefill_attention(q.to(dev), k.to(dev), v.to(dev), mask.to(dev)).cpu()
    sel = torch.tensor(sorted({first, first + rows // 3, first + rows - 1}))
    for hh in (0, h - 1):
        for p in sel.tolist():
            w = torch.softmax((k[hh, :p + 1].double() @ q[hh, p].double()) / math.sqrt(d), 0)
            want = (w[:, None] * v[hh, :p + 1].double()).sum(0)
            assert_attn_close(got[hh, p][None, None], want.float()[None, None])
    assert not bool(got[:, ~mask].any())


@pytest.mark.parametrize("hq,hkv,d,seq,rows,bs", [
    (14, 2, 64, 160, 9, 16), (14, 2, 64, 161, 9, 16),    # the smallest calls: up to 160 x 64
    (28, 4, 128, 80, 25, 16), (28, 4, 128, 80, 26, 16),  # ... and 7340032 products
    (14, 2, 64, 193, 1, 16), (14, 2, 64, 192, 9, 16),    # key tiles of 64, one key past and whole
    (32, 8, 128, 97, 17, 16),                            # key tiles of 32, one key past
    (28, 4, 128, 150, 33, 24)])                          # blocks that are no power of two
def test_paged_fp32_smallest_calls(dev, hq, hkv, d, seq, rows, bs):
    from semblend_amd import _lib

    q, kv, bt, _ = _paged_case(hq, hkv, d, seq, seq, torch.float32, 660 + seq, bs=bs)
    pos = torch.randperm(seq, generator=gen(661))[:rows].sort().values.to(torch.int32)
    pos[-1] = seq - 1
    q = q[:rows]
    want = ref.partial_attention_paged(q, kv, bt, pos)
    args = [t.to(dev) for t in (q, kv, bt, pos)]
    _lib.kernel_timing(True)
    try:
        got = tk.partial_prefill_attention_paged(*args)
        torch.cuda.synchronize()
        valu = _lib.kernel_time("attn_valu")[1]
    finally:
        _lib.kernel_timing(False)
    keys = bt.numel() * kv.shape[3]
    assert valu == (keys * d <= 160 * 64 and rows * hq * keys * d <= 7 << 20)
    # two orders of summing d products and up to seq weighted values: a few 2^-24 of |out| <= 1
    assert float((got.cpu() - want).abs().max()) <= 5e-6 * max(1.0, float(want.abs().max()))
