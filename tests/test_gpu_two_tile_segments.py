"""On the GPU: how the kernels of two column tiles cut their rows in the split path."""
import ctypes
import math
import statistics

import pytest
import torch

import _segment_policy as P
from flash_attention_factory_amd import _cabi, runner, workloads as W
from flash_attention_factory_amd.lib import paged_attention_fp8_reduce, paged_attention_reduce
from _torch_ref import assert_close_to_reference

pytestmark = pytest.mark.gpu

MARK_BITS, MARK_MASK = 0x7FD3A600, 0xFFFFFF00  # segment_mark
MAX_PARTITIONS = 64                            # kSegmentMaxPartitions


def two_tile_segment(lens, psize, heads, units):
    """two_tile_partitions_per_segment; 0: no opinion."""
    parts = [-(-n // psize) for n in lens]
    items, longest = sum(parts) * heads, max(parts)
    if longest <= MAX_PARTITIONS and 3 * longest * units <= 4 * items:
        return max(longest, 1)
    if sum(p > 0 for p in parts) * heads > units:
        return 0
    mean = -(-items // units)
    m = max(mean, 1)
    while m <= MAX_PARTITIONS and (m == mean or 3 * m * units <= 4 * items):
        if sum(-(-n // (m * psize)) for n in lens) * heads <= units:
            return m
        m += 1
    return 0


@pytest.mark.parametrize("name", ["whole", "one_per_unit", "no_opinion"])
def test_two_tile_segments(oracle, name):
    """Four query tokens of eight heads a kv head (two column tiles): the segment length that the marks in max_logits hold
    is the rule's, and the output the oracle's."""
    dev = torch.device("cuda:0")
    units = torch.cuda.get_device_properties(dev).multi_processor_count
    H, Hk, D, QL, psize = 64, 8, 64, 4, 64
    lens = {"whole": [2100 + (331 * s) % 400 for s in range(units // Hk + 8)],
            "one_per_unit": [1500 + 190 * s for s in range(max(2, units // Hk // 4))],
            "no_opinion": [2600] + [300 + (97 * s) % 200 for s in range(units // Hk + 8)]}[name]
    want = two_tile_segment(lens, psize, Hk, units)
    assert (want == 0) == (name == "no_opinion"), want
    S, keys = len(lens), max(lens)
    w_cpu = W.make_test_shaped(batch_size=S, nheads=H, nheads_k=Hk, d=D, seqlen_k=keys, varlen=False, has_sinks=False,
                               block_size=16, seed=3, layout=W.HEAD_MAJOR)
    w_cpu.context_lens = torch.tensor(lens, dtype=torch.int32)
    query = torch.randn(S, QL, H, D, generator=torch.Generator().manual_seed(4)).to(w_cpu.query.dtype)
    ref = oracle.attention_ref(query, w_cpu.key_cache, w_cpu.value_cache, w_cpu.block_tables, w_cpu.context_lens,
                               scale=w_cpu.scale, block_size=16, kv_strides=w_cpu.kv_strides(), num_kv_heads=Hk, want_f32=True)[1]
    w = w_cpu.to(dev)
    NP = -(-keys // psize)
    nan = dict(fill_value=math.nan, dtype=torch.float32, device=dev)
    ml, es, tmp = torch.full((S * QL, H, NP), **nan), torch.full((S * QL, H, NP), **nan), torch.full((S * QL, H, NP, D), **nan)
    out = torch.zeros((S, QL, H, D), dtype=query.dtype, device=dev)
    paged_attention_reduce.run(ml, es, tmp, out, None, query.to(dev), runner.logical_cache_view(w, w.key_cache),
                               runner.logical_cache_view(w, w.value_cache), w.block_tables, w.context_lens, H // Hk, w.scale, 16,
                               keys, None, None, 0.0, partition_size=psize)
    torch.cuda.synchronize()
    bits = ml.view(torch.int32).cpu()
    marks = bits[(bits & MARK_MASK) == MARK_BITS] & 0xFF
    if want:
        assert set(marks.tolist()) == {want}, (set(marks.tolist()), want)
    assert_close_to_reference(out.float().cpu(), ref, name)


def _lognormal(n, median, most, spread=0.75):
    normal = statistics.NormalDist()
    return [min(most, int(median * math.exp(spread * normal.inv_cdf((k + 0.5) / n)))) for k in range(n)]


def _uniform(n, lo, hi):
    return [lo + (hi - lo) * k // max(n - 1, 1) for k in range(n)]


@pytest.mark.parametrize("lens, hk, group, d, fp8, token_major, query_len, whole", [
    # rows of which a few are much longer than the others: left whole, the longest would meet others on its unit
    (_lognormal(157, 2000, 16384), 8, 8, 128, True, False, 4, False),
    (_lognormal(157, 2000, 16384), 8, 8, 128, False, False, 4, False),
    (_lognormal(200, 1000, 8192), 8, 4, 128, True, True, 8, False),   # teams of two kv heads
    (_lognormal(64, 1200, 8192), 16, 8, 64, False, False, 4, False),
    (_lognormal(90, 1200, 8192), 16, 8, 64, False, True, 4, False),   # teams
    (_lognormal(198, 828, 9584), 8, 8, 64, True, False, 4, False),
    # rows that balance
    (_uniform(48, 257, 6000), 8, 8, 128, True, False, 4, True),
    (_uniform(78, 517, 13330), 8, 8, 128, True, False, 4, True),       # a sixth of the mean above it
    (_uniform(150, 300, 3000), 8, 8, 128, True, True, 4, True),        # teams
    (_lognormal(50, 632, 2419), 16, 5, 128, True, False, 6, True),
    ([1800] * 250, 8, 5, 64, True, False, 6, True),
    # a row per unit at most
    ([1623] * 9, 8, 4, 128, False, False, 5, False),
    (_uniform(16, 745, 3191), 8, 7, 128, True, False, 4, None),
    (_uniform(3, 1000, 5000), 32, 8, 64, False, False, 3, None),
    ([7000], 2, 8, 64, True, False, 4, None),
    (_uniform(34, 4748, 10618), 8, 4, 64, False, True, 5, False),      # teams
    ([0, 5, 0], 4, 8, 128, True, False, 4, True),
])
def test_two_tile_choice_equals_the_host_restatement(lens, hk, group, d, fp8, token_major, query_len, whole):
    """The length that the marks hold is the restated rule's; a work-group with the longest and others of the rows left whole
    has no more above the mean than the rule's bound (and 32 keys a row, the step it counts in); with a local window the rule is
    the same."""
    dev = torch.device("cuda:0")
    block, psize = 16, 512 if d == 128 else 256
    S, H, mb, npart = len(lens), hk * group, -(-max(lens) // block), -(-max(lens) // psize)
    nb = 512
    shape = (nb, block, hk, d) if token_major else (nb, hk, block, d)
    pool = torch.zeros(shape, dtype=torch.uint8 if fp8 else torch.float16, device=dev)
    pool = pool if token_major else pool.permute(0, 2, 1, 3)
    tables = torch.randint(0, nb, (S, mb), generator=torch.Generator().manual_seed(0), dtype=torch.int32).to(dev)
    query = torch.zeros((S, query_len, H, d), dtype=torch.float16, device=dev)
    es, ml = (torch.full((S * query_len, H, npart), math.nan, device=dev) for _ in range(2))
    tmp = torch.empty((S * query_len, H, npart, d), device=dev)
    order = torch.randperm(S, generator=torch.Generator().manual_seed(1))
    at = torch.tensor(lens, dtype=torch.int32)[order].to(dev)
    sh, op, plan = _cabi.Shape(), _cabi.Options(), _cabi.SplitPlan()
    op.query_len = query_len
    sh.num_seqs, sh.num_heads, sh.num_kv_heads, sh.head_size, sh.block_size = S, H, hk, d, block
    sh.max_blocks_per_seq, sh.max_num_partitions, sh.partition_size = mb, npart, psize
    sh.kv_block_stride, sh.kv_token_stride, sh.kv_head_stride = pool.stride(0), pool.stride(1), pool.stride(2)
    sh.q_dtype, sh.num_pool_blocks = _cabi.FA_DTYPE_F16, nb
    op.schedule = _cabi.FA_SCHEDULE_SPLIT
    _cabi.check(_cabi.load().fa_paged_attention_reduce_plan(ctypes.byref(sh), ctypes.byref(op), 0, int(fp8), 0, ctypes.byref(plan)))
    assert plan.form == _cabi.FA_SPLIT_FORM_SEGMENT
    geo = dict(partition_size=psize, max_num_partitions=npart, max_ctx=mb * block, num_kv_heads=hk // plan.kv_heads_per_item)
    want = P.two_tile_partitions_per_segment(
        lens, head_size=d, groups=plan.work_groups, cus=plan.compute_units, rows_apart=token_major, teams=plan.kv_heads_per_item > 1,
        partition_bytes=2 * psize * d * (1 if fp8 else 2) * plan.kv_heads_per_item, **geo)
    longest = max(-(-n // psize) for n in lens)
    if whole is not None:
        assert (want >= longest) == whole, (want, longest)
    if want >= longest and sum(n > 0 for n in lens) * geo["num_kv_heads"] >= 2 * plan.work_groups:
        keys = P.dealt_keys(lens, want, groups=plan.work_groups, **geo)
        mean = sum(keys) / len(keys)
        key_bytes = 2 * d * (1 if fp8 else 2) * plan.kv_heads_per_item
        assert keys[0] - mean <= max((192 if plan.kv_heads_per_item > 1 else 480) * 1024 / key_bytes, mean / 6) + 32 * len(lens), (keys[0], mean)
    for window in (None, 700):
        ml.fill_(math.nan)
        out = torch.empty_like(query)
        head = [ml, es, tmp, out, None, query, pool, pool, tables, at, group, d ** -0.5] + ([1.0] if fp8 else [])
        mod = paged_attention_fp8_reduce if fp8 else paged_attention_reduce
        mod.run(*head, block, 0, None, None, 0.0, partition_size=psize, timed=False, window_left=window, schedule=_cabi.FA_SCHEDULE_SPLIT)
        torch.cuda.synchronize()
        bits = ml.view(torch.int32).cpu()
        marks = set((bits[(bits & MARK_MASK) == MARK_BITS] & 0xFF).tolist())
        assert marks == ({want} if want > 1 and longest > 1 else set()), (marks, want, plan.work_groups, plan.kv_heads_per_item)


def test_skewed_rows_against_the_oracle(oracle):
    """Byte cache, head size 128, rows of which few are long (not left whole) and rows that are, with a window and without."""
    dev = torch.device("cuda:0")
    units = torch.cuda.get_device_properties(dev).multi_processor_count
    H, Hk, D, QL, psize = 32, 4, 128, 4, 64
    S = 3 * units // Hk
    for lens in ([1024] * (S // 16) + [150 + (7 * s) % 90 for s in range(S - S // 16)], [500 + (7 * s) % 90 for s in range(S)]):
        w_cpu = W.make_test_shaped(batch_size=S, nheads=H, nheads_k=Hk, d=D, seqlen_k=max(lens), varlen=False, has_sinks=True,
                                   fp8=True, block_size=16, seed=3, layout=W.HEAD_MAJOR)
        w_cpu.context_lens = torch.tensor(lens, dtype=torch.int32)
        query = torch.randn(S, QL, H, D, generator=torch.Generator().manual_seed(4)).to(w_cpu.query.dtype)
        w = w_cpu.to(dev)
        NP = -(-max(lens) // psize)
        nan = dict(fill_value=math.nan, dtype=torch.float32, device=dev)
        ml, es, tmp = torch.full((S * QL, H, NP), **nan), torch.full((S * QL, H, NP), **nan), torch.full((S * QL, H, NP, D), **nan)
        for window in (None, 300):
            ref = oracle.attention_ref(query, w_cpu.key_cache, w_cpu.value_cache, w_cpu.block_tables, w_cpu.context_lens,
                                       scale=w_cpu.scale, block_size=16, kv_strides=w_cpu.kv_strides(), num_kv_heads=Hk, sinks=w_cpu.sinks,
                                       fp8_scale=1.0, want_f32=True, window_left=-1 if window is None else window)[1]
            out = torch.zeros((S, QL, H, D), dtype=query.dtype, device=dev)
            paged_attention_fp8_reduce.run(ml, es, tmp, out, None, query.to(dev), runner.logical_cache_view(w, w.key_cache),
                                           runner.logical_cache_view(w, w.value_cache), w.block_tables, w.context_lens, H // Hk, w.scale,
                                           1.0, 16, max(lens), None, w.sinks, 0.0, partition_size=psize, window_left=window,
                                           schedule=_cabi.FA_SCHEDULE_SPLIT)
            torch.cuda.synchronize()
            assert_close_to_reference(out.float().cpu(), ref, f"window {window}")
