"""On the GPU: how the kernels of two column tiles cut their rows in the split path."""
import math

import pytest
import torch

from flash_attention_factory_amd import runner, workloads as W
from flash_attention_factory_amd.lib import paged_attention_reduce
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
