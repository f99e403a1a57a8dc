"""On the GPU: the forms of the reduce kernel behind the segment kernels, on both sides of the numbers of (row, head) pairs
and of slots between which the launcher chooses."""
import pytest
import torch

from flash_attention_factory_amd import runner, workloads as W
from _torch_ref import assert_close_to_reference, call_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,H,Hk,D,keys,m", [
    (4, 32, 4, 128, 65 * 64, 1),   # 128 pairs: rows asked for ahead, and one slot beyond the 64 that are
    (1, 8, 1, 64, 128 * 64, 3),    # the most slots of that form
    (1, 8, 1, 128, 128 * 64, 1),   # and every one a partial
    (1, 8, 1, 64, 129 * 64, 3),    # one more: four wavefronts a pair
    (5, 32, 4, 128, 700, 2),       # more pairs: four wavefronts a pair
    (3, 40, 5, 128, 90, 1),        # two slots for sixteen wavefronts
    (117, 35, 5, 64, 400, 2),      # 4095 pairs: four wavefronts a pair
    (118, 35, 5, 64, 400, 2),      # 4130: one wavefront a pair, eight pairs a work-group, the last of which has two
])
def test_reduce_forms(oracle, S, H, Hk, D, keys, m):
    """Partitions of 64 keys, m of them a segment; the scratch arrays hold NaN before (a row of tmp_out that no piece has
    written must not reach the result), one sequence is empty and some rows have a single partial."""
    w_cpu = W.make_test_shaped(batch_size=S, nheads=H, nheads_k=Hk, d=D, seqlen_k=keys, varlen=False, has_sinks=True,
                               block_size=16, seed=S + m)
    w_cpu.partition_size = 64
    edge = [keys, 0, 64, 65, 1, keys - 1, 64 * m, 64 * m + 1, 129]
    w_cpu.context_lens = torch.tensor([min(keys, edge[s % len(edge)]) for s in range(S)], dtype=torch.int32)
    w_cpu.sinks = torch.linspace(-2, 2, H).to(w_cpu.query.dtype)
    _, ref = call_oracle(oracle.attention_ref, w_cpu, want_f32=True)
    w = w_cpu.to(torch.device("cuda:0"))
    bufs = runner.alloc_buffers(w, max_num_partitions=-(-keys // 64))
    for _ in range(2):  # the second call finds what the first has left
        bufs.out.zero_()
        runner.run_workload(w, "reduce", bufs, segment_partitions=m)
        torch.cuda.synchronize()
        got = bufs.out.float().cpu()
        live = w_cpu.context_lens > 0
        assert (got[~live] == 0).all()
        assert_close_to_reference(got[live], ref[live], f"{S}x{H} pairs, {keys} keys, m = {m}")


@pytest.mark.parametrize("D", [64, 128])
def test_scratch_wider_than_the_rows(oracle, D):
    """Sixteen wavefronts a pair ask for the first 16 rows of tmp_out before they know the length and for the next ones behind it:
    rows of 1, 2, 15 to 17, 32, 33, 64, 65, 80 and 81 partitions in scratch of 128, all of it NaN before."""
    lens = [64 * n - d for n, d in ((1, 0), (2, 0), (15, 3), (16, 0), (17, 63), (32, 0), (33, 1), (64, 0), (65, 63), (80, 0), (81, 5))] + [0]
    w_cpu = W.make_test_shaped(batch_size=len(lens), nheads=4, nheads_k=2, d=D, seqlen_k=max(lens), varlen=False, has_sinks=True,
                               block_size=16, seed=D)
    w_cpu.partition_size = 64
    w_cpu.context_lens = torch.tensor(lens, dtype=torch.int32)
    _, ref = call_oracle(oracle.attention_ref, w_cpu, want_f32=True)
    w = w_cpu.to(torch.device("cuda:0"))
    wide = torch.zeros((len(lens), 128 * 4), dtype=torch.int32, device="cuda:0")
    wide[:, :w.block_tables.shape[1]] = w.block_tables
    w.block_tables = wide
    for m in (1, 2):
        bufs = runner.alloc_buffers(w, max_num_partitions=128)
        bufs.out.zero_()
        runner.run_workload(w, "reduce", bufs, segment_partitions=m)
        torch.cuda.synchronize()
        got = bufs.out.float().cpu()
        assert (got[-1] == 0).all()
        assert_close_to_reference(got[:-1], ref[:-1], f"m = {m}")
