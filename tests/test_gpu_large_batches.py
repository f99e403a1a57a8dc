"""On the GPU: loop calls of more sequences than the persistent kernel ranks, from 16-bit caches, on both sides of the rule that
gives them to the grid form (head size, rows per compute unit, bound on the keys of a row), against the oracle."""
import pytest
import torch

from flash_attention_factory_amd import lib, runner, workloads as W
from _torch_ref import assert_close_to_reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,H,Hk,D,keys,layout", [
    (129, 4, 2, 64, 300, W.HEAD_MAJOR),
    (131, 6, 3, 64, 2048, W.TOKEN_MAJOR),     # the longest rows of the grid form
    (131, 6, 3, 64, 2049, W.TOKEN_MAJOR),     # sub-batches
    (160, 8, 8, 128, 100, W.HEAD_MAJOR),      # 1280 rows: five for each of 256 units
    (161, 8, 8, 128, 100, W.HEAD_MAJOR),      # more: sub-batches (bf16: groups of one head in fp16 have a kernel of their own)
    (300, 4, 1, 128, 513, W.TOKEN_MAJOR),
    (176, 64, 32, 64, 40, W.TOKEN_MAJOR),     # 88 x 32 rows in each of two sub-batches: eleven for each unit
    (177, 64, 32, 64, 40, W.TOKEN_MAJOR),     # more: sub-batches
    (177, 64, 32, 64, 40, W.HEAD_MAJOR),      # sub-batches if modified
    (192, 8, 4, 128, 60, W.HEAD_MAJOR),       # 96 x 4: one and a half
    (193, 8, 4, 128, 60, W.HEAD_MAJOR),       # sub-batches if modified
])
@pytest.mark.parametrize("mods", [{}, dict(softcap=20.0, apply_softcap=True, window_left=90)], ids=["plain", "modified"])
def test_against_the_oracle(oracle, S, H, Hk, D, keys, layout, mods):
    w = W.make_test_shaped(batch_size=S, nheads=H, nheads_k=Hk, d=D, seqlen_k=keys, varlen=False, has_sinks=True, block_size=16,
                           seed=S, dtype=torch.bfloat16, layout=layout)
    edge = [keys, 0, 1, 31, 32, 33, 255, 256, 257, keys - 1]
    w.context_lens = torch.tensor([min(keys, edge[s % 10]) for s in range(S)], dtype=torch.int32)
    w.sinks = torch.linspace(-2, 2, H).to(w.query.dtype)
    wd = w.to(torch.device("cuda:0"))
    for query_len in (1, 2):
        query = w.query if query_len == 1 else torch.randn(S, 2, H, D, generator=torch.Generator().manual_seed(1)).to(w.query.dtype)
        ref = oracle.attention_ref(query, w.key_cache, w.value_cache, w.block_tables, w.context_lens, scale=w.scale, block_size=16,
                                   kv_strides=w.kv_strides(), num_kv_heads=Hk, sinks=w.sinks, want_f32=True,
                                   softcap=mods.get("softcap", 0.0), window_left=mods.get("window_left", -1))[1]
        out = torch.full_like(query, 7.0, device="cuda:0")
        kw = dict(mods)
        lib.paged_attention_loop.run(None, None, None, out, None, query.to("cuda:0"), runner.logical_cache_view(wd, wd.key_cache),
                                     runner.logical_cache_view(wd, wd.value_cache), wd.block_tables, wd.context_lens, H // Hk, w.scale,
                                     16, keys, None, wd.sinks, kw.pop("softcap", 0.0), **kw)
        torch.cuda.synchronize()
        live = w.context_lens > 0
        assert (out.cpu()[~live] == 7.0).all(), "rows without keys are not written"
        assert_close_to_reference(out.float().cpu()[live], ref[live], f"{query_len} query tokens")
