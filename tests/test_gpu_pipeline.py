"""GPU parity of whole pipelines against the oracle:

* the one-layer Qwen2.5-0.5B pipeline (fp32, 1024 tokens): scatter into a permuted paged
  cache, per-token RoPE deltas in [-64, 64] applied in place, 154-row GQA attention over that
  same cache; every step checked, and the RoPE step also through ``rope_correct_k`` on the
  flat donor K and the dense drop-in attention on GQA-expanded K/V;
* the single-layer orchestrator ``partial_prefill`` on the reference suite's own cases
  (synapse_kv_connector/tests/test_triton_kernels.py:504-762: basic, full reuse, no reuse,
  sparse reuse, timing fields) in fp16 as there, and in bf16 and fp32, plus a larger bf16
  case that takes the MFMA projection;
* the full-size Llama-3-8B batch (32 layers, four requests of 8K-32K tokens, deltas in
  [-4096, 4096]): V bit-exact and K within the RoPE bar on sampled pairs of every layer,
  attention on sampled rows of every request in two layers.
"""

from __future__ import annotations

import pytest
import torch

import bench
from oracle import ref_cpu as ref
from semblend_amd import rope_correction as rc
from semblend_amd import triton_kernels as tk
from tests.helpers import (ATTN_F32_ATOL, ATTN_F32_RTOL, ATTN_16_ATOL, assert_attn_close,
                           assert_bit_exact, assert_rope_close, gen, randn)

pytestmark = pytest.mark.gpu


# ---- Qwen2.5-0.5B one-layer pipeline ------------------------------------------------------

def test_qwen05b_pipeline_step_by_step(dev):
    inp = bench.qwen05b_pipeline_inputs(seed=0)
    c = bench.QWEN05B
    assert inp["deltas"].abs().max() <= 64 and inp["rows"].unique().numel() == 154
    # (1) scatter, bit-exact
    want = inp["cache"].clone()
    ref.scatter_donor_kv_paged(want, inp["donor"], inp["block_table"], inp["positions"],
                               inp["positions"])
    kv = inp["cache"].to(dev)
    bt = inp["block_table"].to(dev)
    pos = inp["positions"].to(dev)
    tk.scatter_donor_kv_paged(kv, inp["donor"].to(dev), bt, pos, pos)
    assert_bit_exact(kv, want)
    # (2) per-token RoPE, one in-place call per distinct delta; V untouched
    groups = bench.delta_groups(inp["deltas"])
    assert 100 < len(groups) <= 128
    for dl, where in groups:
        n_want = ref.apply_rope_delta_inplace(want, inp["block_table"], where, dl,
                                              rope_base=c["theta"])
        n_got = rc.apply_rope_delta_inplace(kv, bt, where, dl, rope_base=c["theta"])
        assert n_got == n_want == len(where)
    got = kv.cpu()
    assert_bit_exact(got[:, 1], want[:, 1])
    assert_rope_close(got[:, 0], want[:, 0])
    # the same rotation applied to the flat donor K (rope_correct_k) lands the same rows
    d = inp["positions"]
    t = d + inp["deltas"].to(torch.int32)
    k_flat = rc.rope_correct_k(inp["donor"][0].to(dev), d.to(dev), t.to(dev), head_dim=64,
                               rope_base=c["theta"])
    k_want = ref.rope_correct_k(inp["donor"][0], d, t, head_dim=64, rope_base=c["theta"])
    assert_rope_close(k_flat, k_want)
    k_paged, _ = ref.gather_paged_kv(got, inp["block_table"], c["ctx"])
    assert_bit_exact(k_paged, k_flat.cpu())
    # (3) 154-row GQA attention over the corrected cache
    out = tk.partial_prefill_attention_paged(inp["q"].to(dev), kv, bt, inp["rows"].to(dev))
    want_attn = ref.partial_attention_paged(inp["q"], want, inp["block_table"], inp["rows"])
    assert_attn_close(out, want_attn)
    # the dense drop-in on the GQA-expanded cache gives the same rows, zeros elsewhere
    g = c["hq"] // c["hkv"]
    kd, vd = ref.gather_paged_kv(got, inp["block_table"], c["ctx"])
    qd = torch.zeros((c["hq"], c["ctx"], c["d"]))
    qd[:, inp["rows"].long()] = inp["q"].permute(1, 0, 2)
    mask = torch.zeros(c["ctx"], dtype=torch.bool)
    mask[inp["rows"].long()] = True
    dense = tk.partial_prefill_attention(qd.to(dev), kd.repeat_interleave(g, 0).to(dev),
                                         vd.repeat_interleave(g, 0).to(dev), mask.to(dev))
    dense = dense.cpu()
    assert_attn_close(dense[:, inp["rows"].long()].permute(1, 0, 2), want_attn)
    assert not bool(dense[:, ~mask].any())


def test_qwen05b_pipeline_function_matches_oracle(dev):
    """The bench's pipeline function run through the HIP entry points and through the oracle
    (the CPU baseline it times) on another seed."""
    inp = bench.qwen05b_pipeline_inputs(seed=3)
    kv, out = bench.qwen05b_pipeline(tk, rc, inp, device=dev)
    kv_want, out_want = bench.qwen05b_pipeline(ref, ref, inp)
    got = kv.cpu()
    assert_bit_exact(got[:, 1], kv_want[:, 1])
    assert_rope_close(got[:, 0], kv_want[:, 0])
    assert_attn_close(out, out_want)


# ---- partial_prefill, the single-layer orchestrator ---------------------------------------

def _prefill_case(name: str, dtype: torch.dtype, seed: int):
    """The reference suite's cases (same sizes, masks and pairs; seeded N(0,1) inputs in the
    reference's unscaled form), and a larger one at a realistic scale."""
    g = gen(seed)

    def rn(*shape, scale=1.0):
        return (torch.randn(shape, generator=g) * scale).to(dtype)

    if name == "basic":
        s, hid, h, d, layers, dl = 8, 32, 4, 8, 2, 8
        dp = torch.tensor([0, 1, 2, 3]); tp = dp.clone()
        cm = torch.tensor([False] * 4 + [True] * 4)
    elif name == "full_reuse":
        s, hid, h, d, layers, dl = 4, 16, 2, 8, 1, 4
        dp = torch.arange(s); tp = dp.clone()
        cm = torch.zeros(s, dtype=torch.bool)
    elif name == "no_reuse":
        s, hid, h, d, layers, dl = 4, 16, 2, 8, 1, 4
        dp = torch.zeros(0, dtype=torch.int64); tp = dp.clone()
        cm = torch.ones(s, dtype=torch.bool)
    elif name == "sparse":
        s, hid, h, d, layers, dl = 16, 32, 4, 8, 2, 10
        dp = torch.tensor([0, 2, 4, 6, 8]); tp = torch.tensor([0, 3, 6, 9, 12])
        cm = torch.ones(s, dtype=torch.bool)
        cm[tp] = False
    elif name == "timing":
        s, hid, h, d, layers, dl = 64, 128, 8, 16, 4, 32
        dp = torch.arange(16); tp = dp.clone()
        cm = torch.ones(s, dtype=torch.bool)
        cm[:16] = False
    elif name == "large":
        s, hid, h, d, layers, dl = 384, 512, 8, 64, 2, 384
        perm = torch.randperm(s, generator=g)
        cm = torch.ones(s, dtype=torch.bool)
        cm[perm[:270]] = False
        tp = (~cm).nonzero().flatten()
        dp = torch.randperm(dl, generator=g)[:tp.numel()]
        hs = rn(s, hid)
        donor = rn(layers, 2, h, dl, d)
        wq = rn(3 * h * d, hid, scale=hid ** -0.5)
        wo = rn(hid, h * d, scale=(h * d) ** -0.5)
        return hs, donor, wq, wo, dp.to(torch.int32), tp.to(torch.int32), cm, h, d
    else:
        raise ValueError(name)
    hs = rn(s, hid)
    donor = rn(layers, 2, h, dl, d)
    wq = rn(3 * h * d, hid)
    wo = rn(hid, h * d)
    return hs, donor, wq, wo, dp.to(torch.int32), tp.to(torch.int32), cm, h, d


def _ulp(x: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    if dtype == torch.float32:
        return x.abs() * 2.0 ** -23 + 1e-38
    mant = 7 if dtype == torch.bfloat16 else 10
    e = torch.floor(torch.log2(x.abs().clamp_min(2.0 ** -14)))
    return torch.pow(2.0, e - mant)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("case", ["basic", "full_reuse", "no_reuse", "sparse", "timing",
                                  "large"])
def test_partial_prefill_matches_oracle(dev, case, dtype):
    seed = {"basic": 1, "full_reuse": 2, "no_reuse": 3, "sparse": 4, "timing": 5, "large": 6}
    hs, donor, wq, wo, dp, tp, cm, h, d = _prefill_case(case, dtype, seed=seed[case])
    res = tk.partial_prefill(hs.to(dev), donor.to(dev), wq.to(dev), wo.to(dev), dp.to(dev),
                             tp.to(dev), cm.to(dev), h, d)
    out_w, kv_w, computed, reused, ratio = ref.partial_prefill(hs, donor, wq, wo, dp, tp, cm,
                                                               h, d)
    # the reference suite's structural assertions
    assert isinstance(res, tk.PartialPrefillResult)
    assert (res.positions_computed, res.positions_reused) == (computed, reused)
    assert res.computation_ratio == pytest.approx(ratio, abs=1e-6)
    assert res.output.shape == out_w.shape and res.output.dtype == dtype
    assert res.kv_cache.shape == kv_w.shape and res.kv_cache.dtype == dtype
    assert res.total_time_ms > 0 and res.scatter_time_ms >= 0
    assert res.projection_time_ms >= 0 and res.attention_time_ms >= 0
    out = res.output.cpu()
    kv = res.kv_cache.cpu()
    # donor rows copied bit-exact into every layer (reference: exact equality)
    reuse = (~cm).nonzero().flatten()
    for i in range(dp.numel()):
        assert_bit_exact(kv[:, :, :, int(tp[i])], donor[:, :, :, int(dp[i])])
    # positions neither reused nor computed stay zero; reuse rows of the output are zero
    untouched = torch.ones(cm.numel(), dtype=torch.bool)
    untouched[cm] = False
    untouched[tp.long()] = False
    assert not bool(kv[:, :, :, untouched].any())
    assert not bool(out[reuse].any())
    # new K/V of the computed rows (same in every layer): fp32 projection rounded once; two
    # correct GEMMs may round a near-tie apart by one ulp of the dtype
    comp = cm.nonzero().flatten()
    if comp.numel():
        got_kv = kv[:, :, :, comp].float()
        want_kv = kv_w[:, :, :, comp].float()
        dot = torch.nn.functional.linear(hs.float().abs(), wq.float().abs())  # sum |x w|
        kvbound = dot[comp][:, h * d:].reshape(-1, 2, h, d).permute(1, 2, 0, 3)
        tol = _ulp(want_kv, dtype) + 2.0 ** -16 * kvbound.unsqueeze(0)
        assert bool(((got_kv - want_kv).abs() <= tol).all()), "new K/V outside the bar"
        # output rows: the attention bar carried through the output projection, plus an
        # ulp of the output for the final rounding
        # (attention rows are convex combinations of V rows, so |attn| <= max |V|)
        attn_bar = ATTN_16_ATOL if dtype != torch.float32 else ATTN_F32_ATOL
        rel = 0.0 if dtype != torch.float32 else ATTN_F32_RTOL
        vmax = float(kv_w[0, 1].float().abs().max())
        bound = (attn_bar + rel * vmax) * wo.float().abs().sum(dim=1)
        diff = (out[comp].float() - out_w[comp].float()).abs()
        tol = bound.unsqueeze(0) + _ulp(out_w[comp].float(), dtype)
        assert bool((diff <= tol).all()), \
            f"output outside the bar: max excess {float((diff - tol).max())}"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("s,hid,h,d,layers,feats,share", [
    (1, 64, 1, 64, 1, 4, 1.0),          # one position, one feature quad
    (33, 48, 3, 64, 2, 36, 0.5),        # hidden no multiple of 64; a second row tile of one row
    (257, 128, 5, 128, 3, 100, 0.0),    # nothing computed: donor rows and zeros only
    (1025, 192, 2, 128, 1, 68, 0.4),    # one position past an index workgroup
    (700, 256, 4, 64, 1, 16384, 0.3)])  # wide output tiles
def test_partial_prefill_stages_match_composed(dev, dtype, s, hid, h, d, layers, feats, share):
    """The stage kernels against the composition of the module's functions, over tile edges,
    strided donors, repeated and out-of-range pairs and biases."""
    g = gen(900 + s)
    f = h * d
    wide = torch.randn((layers, 2, h, s + 9, 2 * d), generator=g).to(dtype).to(dev)
    donor = wide[..., d:]                                       # strided rows
    x = torch.randn((s, hid), generator=g).to(dtype).to(dev)
    wq = (torch.randn((3 * f, hid), generator=g) * hid ** -0.5).to(dtype).to(dev)
    bq = (torch.randn(3 * f, generator=g) * 0.1).to(dtype).to(dev)
    wo = (torch.randn((feats, f), generator=g) * f ** -0.5).to(dtype).to(dev)
    bo = torch.randn(feats, generator=g).to(dtype).to(dev)
    cm = torch.rand(s, generator=g) < share
    tp = torch.cat([torch.arange(0, s, 2), torch.tensor([-1, s, s + 5])])
    dp = torch.cat([torch.randperm(s + 9, generator=g)[:tp.numel() - 3], torch.tensor([0, 1, 2])])
    if s > 8:
        dp[:4] = torch.tensor([-3, s + 9, 1 << 30, 0])          # out of range: not moved
        tp[3], dp[5] = tp[2], 7                                 # a target named twice
    args = (x, donor, wq, wo, dp.to(torch.int32).to(dev), tp.to(torch.int32).to(dev),
            cm.to(dev), h, d, bq, bo, None)
    assert tk._prefill_stages_ok(*args)
    got = tk.partial_prefill(*args)
    want = tk._prefill_composed(x.device, *args)
    assert (got.positions_computed, got.positions_reused) == (int(cm.sum()), int((~cm).sum()))
    assert not bool(got.output.cpu()[~cm].any())
    # donor rows and zeros are the same bits; new K/V come from one projection kernel on the
    # same rows (fp32: the library's GEMM, which may sum in another order for another shape)
    assert_bit_exact(got.kv_cache[:, :, :, ~cm.to(dev)].cpu(),
                     want.kv_cache[:, :, :, ~cm.to(dev)].cpu())
    if not cm.any():
        return
    eps = {torch.float32: 2.0 ** -20, torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}[dtype]
    for a, b in ((got.kv_cache, want.kv_cache), (got.output, want.output)):
        a, b = a.float(), b.float()
        # one rounding to the dtype on each side, of fp32 results that differ in the last bits
        assert float((a - b).abs().max()) <= eps * float(b.abs().max())


def _stage_args(dev, dtype=torch.float32, s=70, hid=64, h=2, d=64, layers=1, feats=40, seed=950):
    """Arguments of a call that takes the stage kernels: pairs, 40% computed, both biases."""
    g = gen(seed)
    f = h * d
    rand = lambda *shape, scale=1.0: (torch.randn(shape, generator=g) * scale).to(dtype).to(dev)
    pos = torch.arange(0, s, 2, dtype=torch.int32).to(dev)
    return [rand(s, hid), rand(layers, 2, h, s, d), rand(3 * f, hid, scale=hid ** -0.5),
            rand(feats, f, scale=f ** -0.5), pos, pos.flip(0), (torch.rand(s, generator=g) < 0.4).to(dev),
            h, d, rand(3 * f, scale=0.1), rand(feats), None]


@pytest.mark.parametrize("at", [3, 10])  # output_projection, output_bias
def test_partial_prefill_forward_derivatives_and_vmap(dev, at):
    """The output is linear in the output projection and its bias: the forward-mode tangent is
    the output of a call with the tangent in that input's place, and vmap over that input the
    calls one by one."""
    from torch.autograd import forward_ad

    args = _stage_args(dev)
    assert tk._prefill_stages_ok(*args)
    zero = list(args)
    zero[3], zero[10] = torch.zeros_like(args[3]), torch.zeros_like(args[10])
    zero[at] = torch.randn(args[at].shape, generator=gen(951)).to(dev)
    want = tk.partial_prefill(*zero).output
    with forward_ad.dual_level():
        dual = list(args)
        dual[at] = forward_ad.make_dual(args[at], zero[at])
        out = forward_ad.unpack_dual(tk.partial_prefill(*dual).output)
        assert out.tangent is not None
    tol = 2.0 ** -18 * float(want.abs().max())  # fp32 sums of 128 products in another order
    assert float((out.tangent - want).abs().max()) <= tol
    both = torch.stack([args[at], zero[at]])
    got = torch.vmap(lambda x: tk.partial_prefill(*args[:at], x, *args[at + 1:]).output)(both)
    for x, y in zip(both, got):
        one = tk.partial_prefill(*args[:at], x, *args[at + 1:]).output
        assert float((y - one).abs().max()) <= 2.0 ** -18 * float(one.abs().max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_partial_prefill_without_a_donor(dev, dtype):
    """No donor found: a donor of zero positions and no pairs is the composed form's result, and
    that of a donor from which nothing is taken."""
    args = _stage_args(dev, dtype)
    args[4] = args[5] = torch.zeros(0, dtype=torch.int32, device=dev)
    full = tk.partial_prefill(*args)
    args[1] = args[1][:, :, :, :0]
    for empty in (args[1], args[1].contiguous()):
        args[1] = empty
        got = tk.partial_prefill(*args)
        want = tk._prefill_composed(dev, *args)
        assert got.positions_computed == full.positions_computed
        assert_bit_exact(got.kv_cache.cpu(), want.kv_cache.cpu())
        assert_bit_exact(got.output.cpu(), want.output.cpu())
        eps = 2.0 ** -18 if dtype == torch.float32 else 2.0 ** -7
        for a, b in ((got.kv_cache, full.kv_cache), (got.output, full.output)):
            assert float((a.float() - b.float()).abs().max()) <= eps * float(b.float().abs().max())


@pytest.mark.parametrize("offset", [1, 2, 3])
def test_partial_prefill_output_bias_at_any_offset(dev, offset):
    """An fp32 output bias that is a view at an address of no multiple of 16 bytes."""
    args = _stage_args(dev)
    want = tk.partial_prefill(*args).output
    flat = torch.zeros(44, device=dev)
    flat[offset:offset + 40] = args[10]
    args[10] = flat[offset:offset + 40]
    assert args[10].data_ptr() % 16 and tk._prefill_stages_ok(*args)
    assert_bit_exact(tk.partial_prefill(*args).output.cpu(), want.cpu())


@pytest.mark.parametrize("form", ["stages", "composed"])
def test_partial_prefill_times_the_attention_alone(dev, form, monkeypatch):
    """attention_time_ms spans the attention launches and not the output projection, the total
    everything, in both forms."""
    log = []

    class Event(torch.cuda.Event):
        def record(self, *args):
            log.append(self)
            super().record(*args)

        def elapsed_time(self, end):
            return float(log.index(end) * 1000 + log.index(self))

    call, linear = tk._lib.call, torch.nn.functional.linear
    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(tk._lib, "call", lambda name, *a: (log.append(name), call(name, *a))[1])
    monkeypatch.setattr(torch.nn.functional, "linear",
                        lambda *a: (log.append("linear"), linear(*a))[1])
    args = _stage_args(dev, torch.bfloat16)
    res = tk.partial_prefill(*args) if form == "stages" else tk._prefill_composed(dev, *args)
    end, start = divmod(int(res.attention_time_ms), 1000)
    within = [x for x in log[start:end] if isinstance(x, str)]
    assert within == ["sb_partial_attention_rows_f32" if form == "stages"
                      else "sb_partial_prefill_attention"]
    end, start = divmod(int(res.total_time_ms), 1000)
    assert (start, end) == (0, len(log) - 1)
    assert log.count("linear") == (0 if form == "stages" else 1)


# ---- Llama-3-8B batch at full size --------------------------------------------------------

def test_llama3_8b_batch_full_size(dev):
    """The benched batch exactly: 32 layers, requests of 8192/16384/24576/32768 tokens with
    10/15/20/30% recompute and chunk-constant deltas in [-4096, 4096], pool of 8192 blocks.
    After one RoPE scatter step: for 192 sampled pairs per request, the cache rows of every
    layer against the oracle (V bit-exact, K within the RoPE bar); then batched attention of
    layers 0 and 31, 48 sampled rows per request against the oracle."""
    from semblend_amd.batch import KVReuseBatch

    caches, reqs, theta = bench.llama_batch(dev)
    c = bench.LLAMA
    assert [int(r.block_table.numel()) * 16 for r in reqs] == list(c["ctx"])
    batch = KVReuseBatch(caches, reqs, rope_base=theta)
    batch.scatter_rope()
    torch.cuda.synchronize()
    g = gen(77)
    for r in reqs:
        n = r.donor_positions.numel()
        sel = torch.randperm(n, generator=g)[:192].to(dev)
        d = r.donor_positions[sel].long()
        t = r.target_positions[sel].long()
        assert int((t - d).abs().max()) <= 4096
        pb = r.block_table[t // 16].long()
        off = t % 16
        d_cpu, t_cpu = d.cpu().to(torch.int32), t.cpu().to(torch.int32)
        idx = torch.arange(d.numel(), dtype=torch.int32)
        for layer in range(c["layers"]):
            got = caches[layer][pb, :, :, off, :].cpu()          # [n, 2, H, D]
            donor_rows = r.donor_kvs[layer][:, :, d, :].cpu()     # [2, H, n, D]
            assert_bit_exact(got[:, 1], donor_rows[1].permute(1, 0, 2))
            # oracle: row i rotated by t_i - d_i (rope_correct_k on the gathered rows)
            k_want = ref.rope_correct_k(donor_rows[0], idx, idx + (t_cpu - d_cpu),
                                        head_dim=c["d"], rope_base=theta)
            assert_rope_close(got[:, 0], k_want.permute(1, 0, 2))
    q = randn((batch.num_rows, c["hq"], c["d"]), torch.bfloat16, 78).to(dev)
    for layer in (0, c["layers"] - 1):
        out = batch.attention(layer, q).cpu()
        kv = caches[layer].cpu()
        for i, r in enumerate(reqs):
            a = batch.row_offsets[i]
            nr = r.compute_positions.numel()
            rows = torch.randperm(nr, generator=g)[:48].sort().values
            pos = r.compute_positions.cpu()[rows]
            want = ref.partial_attention_paged(q[a:a + nr].cpu()[rows], kv,
                                               r.block_table.cpu(), pos)
            assert_attn_close(out[a + rows], want)
        del kv
