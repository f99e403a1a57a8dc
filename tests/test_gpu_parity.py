"""Parity of the HIP kernels (through lib.paged_attention_*.run -> C ABI) with the CPU
oracle on the same seeded inputs.  Tolerance: atol = rtol = 1e-2 on fp16/bf16 outputs,
as the benchmark contract states; the upstream relative rule
(err <= 3 * err_of_a_16-bit-torch-evaluation + 1e-5, test_paged.py:603-604) is checked
in the form err <= 3 * err(oracle kernel model) + 1e-5 where the kernel model rounds
where the upstream kernels round."""
import math
import os

import pytest
import torch

from flash_attention_factory_amd import _cabi, workloads as W
from _torch_ref import call_oracle, out_pt_reference

pytestmark = pytest.mark.gpu

ATOL = RTOL = 1e-2


def _dev():
    assert torch.cuda.is_available(), "these tests need the GPU"
    return torch.device("cuda:0")


def _run(w_cpu, kernel, max_context_len=None, schedule=0, spin_limit=0, timed=True, segment_partitions=0, **kw):
    from flash_attention_factory_amd import runner
    w = w_cpu.to(_dev())
    bufs = runner.alloc_buffers(w, **kw)
    times = runner.run_workload(w, kernel, bufs, max_context_len=max_context_len, schedule=schedule,
                                spin_limit=spin_limit, timed=timed, segment_partitions=segment_partitions)
    if "reduce" in kernel and timed and times[1] == 0.0:
        # rows so short that the split entry ran the single-pass kernel (tests/test_gpu_segment_policy.py
        # covers that); the tests here are after the split kernels
        bufs = runner.alloc_buffers(w, **kw)
        times = runner.run_workload(w, kernel, bufs, max_context_len=max_context_len, schedule=3,
                                    spin_limit=spin_limit)
    torch.cuda.synchronize()
    return bufs, times


def _wide(block_tables, columns):
    table = torch.zeros((block_tables.shape[0], columns), dtype=torch.int32)
    table[:, :block_tables.shape[1]] = block_tables
    return table


def _check(out, w_cpu, oracle, label, literal_rule=False):
    ref16, ref32 = call_oracle(oracle.attention_ref, w_cpu, want_f32=True)
    got = out.float().cpu()
    err = (got - ref32).abs().max().item()
    mag = ref32.abs().max().item()
    print(f"{label}: max|out-ref| = {err:.3e}, max|ref| = {mag:.3e}, rel = {err / mag:.3e}", flush=True)
    assert torch.isfinite(got).all(), label
    torch.testing.assert_close(got, ref32, atol=ATOL, rtol=RTOL, msg=lambda m: f"{label}: {m}")
    # upstream-style relative gate against the rounding-faithful kernel model
    _, model32 = call_oracle(oracle.kernel_loop, w_cpu, partition_size=w_cpu.partition_size, want_f32=True)
    ulp = 2.0 ** (-8 if w_cpu.query.dtype == torch.bfloat16 else -11) * mag
    bar = 3 * max((model32 - ref32).abs().max().item(), ulp) + 1e-5
    assert err <= bar, f"{label}: err {err:.3e} above relative bar {bar:.3e}"
    if literal_rule:
        # upstream's own assertion, word for word (test_paged.py:603-604): both errors against the
        # upcast reference rounded to the 16-bit type
        live = w_cpu.context_lens > 0
        err16 = (out.cpu()[live].float() - ref16[live].float()).abs().max().item()
        err_pt = (out_pt_reference(w_cpu)[live].float() - ref16[live].float()).abs().max().item()
        assert err16 <= 3 * err_pt + 1e-5, f"{label}: err {err16:.3e} above upstream's 3 x {err_pt:.3e} + 1e-5"


SMALL = {  # measured configurations cut down so the oracle finishes in seconds
    0: dict(),
    1: dict(num_seqs=4, pool_blocks=512),
    2: dict(num_seqs=1, pool_blocks=2048),
    3: dict(num_seqs=4, pool_blocks=512),
    4: dict(num_seqs=6, pool_blocks=8192),
}


@pytest.mark.parametrize("index", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("layout", [W.HEAD_MAJOR, W.TOKEN_MAJOR])
def test_measured_configs(oracle, index, layout):
    w = W.make_config(index, layout=layout, **SMALL[index])
    kernel = W.CONFIG_KERNEL[index]
    bufs, times = _run(w, kernel)
    assert len(times) == (2 if "reduce" in kernel else 1) and all(t > 0 for t in times)
    _check(bufs.out, w, oracle, f"{w.name}/{layout}")


@pytest.mark.parametrize("index", [0, 1, 3])
def test_other_kernel_on_same_config(oracle, index):
    """Every configuration also runs through the other kernel of its cache type."""
    w = W.make_config(index, **SMALL[index])
    kernel = {"loop": "reduce", "fp8_loop": "fp8_reduce"}[W.CONFIG_KERNEL[index]]
    bufs, _ = _run(w, kernel)
    _check(bufs.out, w, oracle, f"{w.name} via {kernel}")


GRID = [  # a slice of the upstream grid (test_paged.py:211-256): groups 8,8,5,7,6,4,3,2,1
    dict(batch_size=2, nheads=8, nheads_k=1, d=128, seqlen_k=339, varlen=True, has_sinks=True),
    dict(batch_size=1, nheads=16, nheads_k=2, d=64, seqlen_k=1024, varlen=False, has_sinks=False),
    dict(batch_size=2, nheads=10, nheads_k=2, d=128, seqlen_k=800, varlen=True, has_sinks=False),
    dict(batch_size=2, nheads=14, nheads_k=2, d=64, seqlen_k=799, varlen=True, has_sinks=True),
    dict(batch_size=1, nheads=12, nheads_k=2, d=128, seqlen_k=2048, varlen=False, has_sinks=True),
    dict(batch_size=2, nheads=8, nheads_k=2, d=64, seqlen_k=128, varlen=True, has_sinks=False),
    dict(batch_size=2, nheads=6, nheads_k=2, d=128, seqlen_k=256, varlen=False, has_sinks=True),
    dict(batch_size=1, nheads=4, nheads_k=2, d=64, seqlen_k=20000, varlen=True, has_sinks=False),
    dict(batch_size=2, nheads=2, nheads_k=2, d=128, seqlen_k=2048, varlen=True, has_sinks=True),
]


@pytest.mark.parametrize("case", GRID, ids=lambda c: "h{nheads}x{nheads_k}_d{d}_s{seqlen_k}".format(**c))
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("split", [False, True])
def test_upstream_grid_slice(oracle, case, fp8, split):
    w = W.make_test_shaped(fp8=fp8, **case)
    kernel = ("fp8_" if fp8 else "") + ("reduce" if split else "loop")
    bufs, _ = _run(w, kernel)
    _check(bufs.out, w, oracle, f"{w.name}/{kernel}")


@pytest.mark.parametrize("fp8", [False, True])
def test_partition_scratch_matches_kernel_model(oracle, fp8):
    """exp_sums / max_logits / tmp_out against the restated upstream arithmetic; slots of
    partitions past a sequence's length stay untouched (paged_attention_kernel_v2.hpp:577-579)."""
    w = W.make_test_shaped(batch_size=2, nheads=8, nheads_k=2, d=128, seqlen_k=1300, varlen=True,
                           has_sinks=True, fp8=fp8, seed=7)
    w.context_lens = torch.tensor([1300, 700], dtype=torch.int32)
    NP = 5  # one slot more than any sequence needs
    bufs, _ = _run(w, "fp8_reduce" if fp8 else "reduce", max_num_partitions=NP)
    es, ml, tmp = call_oracle(oracle.kernel_partition, w, partition_size=w.partition_size,
                              max_num_partitions=NP)
    g_es, g_ml, g_tmp = bufs.exp_sums.cpu(), bufs.max_logits.cpu(), bufs.tmp_out.cpu()
    for s in range(2):
        live = math.ceil(int(w.context_lens[s]) / w.partition_size)
        torch.testing.assert_close(g_ml[s, :, :live], ml[s, :, :live], atol=1e-4, rtol=1e-5)
        torch.testing.assert_close(g_es[s, :, :live], es[s, :, :live], atol=1e-4, rtol=1e-4)
        torch.testing.assert_close(g_tmp[s, :, :live], tmp[s, :, :live], atol=2e-3, rtol=1e-2)
        assert torch.isnan(g_ml[s, :, live:]).all() and torch.isnan(g_tmp[s, :, live:]).all()


@pytest.mark.parametrize("schedule", [1, 2])
@pytest.mark.parametrize("fp8", [False, True])
def test_schedule_option(oracle, fp8, schedule):
    """options->schedule: the grid form (upstream's own decomposition, one work-group per (sequence, kv
    head[, partition])) and, for FP8 caches, its variant with K/V staged through LDS by direct-to-LDS
    loads -- on a batch the library would by itself run in the persistent forms.  Same `out`; in the
    split path every live slot of the scratch arrays holds upstream's per-partition values."""
    w = W.make_config(4 if fp8 else 2, num_seqs=5, pool_blocks=4096, lens=[1, 33, 2048, 1537, 700])
    if not fp8:
        w = W.make_config(2, num_seqs=5, pool_blocks=4096, lens=[1, 33, 2048, 1537, 700], layout=W.TOKEN_MAJOR)
    w.sinks = torch.linspace(-1, 2, w.num_heads).to(w.query.dtype)
    for kernel in ("loop", "reduce"):
        kernel = ("fp8_" if fp8 else "") + kernel
        bufs, _ = _run(w, kernel, schedule=schedule)
        _check(bufs.out, w, oracle, f"{w.name}/{kernel}/schedule{schedule}")
        if "reduce" in kernel:
            es, ml, tmp = call_oracle(oracle.kernel_partition, w, partition_size=w.partition_size,
                                      max_num_partitions=w.max_num_partitions)
            # The kernels round the probabilities to the query dtype against a reference maximum that
            # may lag the true one by a few units, the oracle against the true one: the same values,
            # rounded differently.  bf16 keeps 8 significant bits, and a partition of one or a few
            # tokens does not average that out.
            tmp_atol = 2e-3 if w.query.dtype == torch.float16 else 4e-3
            for s in range(w.num_seqs):
                live = math.ceil(int(w.context_lens[s]) / w.partition_size)
                torch.testing.assert_close(bufs.max_logits[s, :, :live].cpu(), ml[s, :, :live], atol=1e-4, rtol=1e-5)
                torch.testing.assert_close(bufs.exp_sums[s, :, :live].cpu(), es[s, :, :live], atol=1e-4, rtol=1e-4)
                torch.testing.assert_close(bufs.tmp_out[s, :, :live].cpu(), tmp[s, :, :live], atol=tmp_atol, rtol=1e-2)
                assert torch.isnan(bufs.max_logits[s, :, live:]).all()


@pytest.mark.parametrize("fp8", [False, True], ids=["kv16", "fp8"])
def test_dot_product_kernel_for_single_head_groups(oracle, fp8):
    """schedule = FA_SCHEDULE_GRID_VALU: the loop path for query groups of one head by lane dot products
    and fp32 multiply-adds instead of the matrix cores.  Edge lengths around its 32-token chunks and the
    rows of one load instruction, an empty sequence, sinks, both layouts, E4M3 bytes -- and the whole of
    the benchmark configuration of its cache type."""
    lens = [1, 3, 4, 5, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 255, 256, 257, 700, 2048, 0]
    cfg = 3 if fp8 else 1
    variants = [dict(), dict(layout=W.TOKEN_MAJOR)] + ([dict(fp8_dtype=torch.float8_e4m3fn)] if fp8 else [])
    for schedule in (_cabi.FA_SCHEDULE_GRID_VALU, _cabi.FA_SCHEDULE_VALU):  # grid form, persistent form
        for kw in variants:
            w = W.make_config(cfg, num_seqs=len(lens), pool_blocks=4096, lens=lens, **kw)
            assert w.num_heads == w.num_kv_heads and w.head_size == 128
            w.sinks = torch.linspace(-1, 2, w.num_heads).to(w.query.dtype)
            bufs, _ = _run(w, ("fp8_" if fp8 else "") + "loop", schedule=schedule)
            _check(bufs.out, w, oracle, f"{w.name}/valu{schedule}/{kw}")
        # few items of few chunks: work-groups with one item, wavefronts without a chunk of their own
        w = W.make_config(cfg, num_seqs=3, pool_blocks=512, lens=[40, 0, 97])
        bufs, _ = _run(w, ("fp8_" if fp8 else "") + "loop", schedule=schedule)
        _check(bufs.out, w, oracle, f"{w.name}/valu{schedule}/few")
        w = W.make_config(cfg)
        bufs, _ = _run(w, ("fp8_" if fp8 else "") + "loop", schedule=schedule)
        _check(bufs.out, w, oracle, f"{w.name}/valu{schedule}/full")
        # more sequences than one resident launch lists (with a 16-bit cache the library's own choice is the grid
        # form of these kernels then: schedule 0 below)
        gen = torch.Generator().manual_seed(11)
        many = [int(x) for x in torch.randint(0, 300, (150,), generator=gen)]
        w = W.make_config(cfg, num_seqs=len(many), pool_blocks=4096, lens=many)
        w.sinks = torch.linspace(-2, 1, w.num_heads).to(w.query.dtype)
        for sched in (schedule, 0):
            bufs, _ = _run(w, ("fp8_" if fp8 else "") + "loop", schedule=sched)
            _check(bufs.out, w, oracle, f"{w.name}/valu{sched}/150 sequences")
        # a group of several heads is not these kernels': the call runs on the matrix cores
        w = W.make_config(4 if fp8 else 2, num_seqs=3, pool_blocks=4096, lens=[700, 33, 1537])
        bufs, _ = _run(w, ("fp8_" if fp8 else "") + "loop", schedule=schedule)
        _check(bufs.out, w, oracle, f"{w.name}/valu{schedule}/fallback")


@pytest.mark.parametrize("shape", [(16, 128, True), (32, 64, True), (16, 64, False), (64, 128, True), (24, 128, True)],
                         ids=lambda s: f"hk{s[0]}_d{s[1]}_{'fp8' if s[2] else 'kv16'}")
def test_loop_items_listed_by_memory_stack(oracle, shape):
    """Head-major pools whose per-head chunks are 1, 2 or 4 KiB: the persistent loop kernels list a sequence's kv
    heads so that a work-group's XCC reads one memory stack (csrc/paged_attention_utils.h: stack_affine_head).
    Whatever the order, every (sequence, kv head) must come out right -- shapes on which the map permutes the
    heads, one with a head count it does not take (24), several items per work-group and fewer than work-groups."""
    hk, d, fp8 = shape
    for S in (3, 40):
        w = W.make_test_shaped(batch_size=S, nheads=hk, nheads_k=hk, d=d, seqlen_k=300, varlen=True, has_sinks=True,
                               fp8=fp8, block_size=16, layout=W.HEAD_MAJOR, seed=S)
        bufs, _ = _run(w, ("fp8_" if fp8 else "") + "loop")
        _check(bufs.out, w, oracle, f"{w.name}/stack-affine item order")


def test_unknown_pool_size(oracle, monkeypatch):
    """shape.num_pool_blocks = 0, as a caller passes who does not know how many blocks the pools hold: the
    persistent kernels need the size (they request block ids before they know the lengths), so every
    schedule runs a grid form, block-table columns past a context are never read and ids are not clamped.
    The Python modules always know the size; the shape is edited on its way into the library."""
    L = _cabi.load()
    edited = []
    for entry in ("fa_paged_attention_loop", "fa_paged_attention_reduce", "fa_paged_attention_fp8_loop",
                  "fa_paged_attention_fp8_reduce"):
        def without_pool_size(*args, _real=getattr(L, entry), _entry=entry):
            args[-2]._obj.num_pool_blocks = 0   # the fa_paged_attention_shape behind byref()
            edited.append(_entry)
            return _real(*args)
        monkeypatch.setattr(L, entry, without_pool_size)
    lens = [1, 33, 700, 0, 1537, 2048]
    for cfg, kernel, schedules in ((1, "loop", (0, 1, 4, 5)), (2, "loop", (0,)), (2, "reduce", (0, 1)),
                                   (3, "fp8_loop", (0, 2, 4, 5)), (4, "fp8_reduce", (0, 1, 2))):
        w = W.make_config(cfg, num_seqs=len(lens), pool_blocks=4096, lens=lens)
        w.sinks = torch.linspace(-1, 2, w.num_heads).to(w.query.dtype)
        # columns of the block table past a context hold ids no pool has: nobody may read them
        for s, n in enumerate(lens):
            w.block_tables[s, -(-n // w.block_size):] = 0x7FFFFFF0
        for schedule in schedules:
            bufs, _ = _run(w, kernel, schedule=schedule)
            _check(bufs.out, w, oracle, f"{w.name}/{kernel}/unknown pool size, schedule {schedule}")
    assert len(edited) == 14 and len(set(edited)) == 4


def test_lds_staged_kernel_full_size(oracle):
    """The LDS-staged grid kernel on the whole FP8 loop configuration, both layouts, and E4M3 bytes."""
    for kw in (dict(), dict(layout=W.TOKEN_MAJOR), dict(fp8_dtype=torch.float8_e4m3fn)):
        w = W.make_config(3, **kw)
        bufs, _ = _run(w, "fp8_loop", schedule=2)
        _check(bufs.out, w, oracle, f"{w.name}/lds/{kw}")


def test_edge_cases(oracle):
    # context lengths 1, 15, 16, 17, 31, 32, 33 and one exactly on a partition boundary
    w = W.make_config(0, num_seqs=8, pool_blocks=256, lens=[1, 15, 16, 17, 31, 32, 33, 256])
    for kernel in ("loop", "reduce"):
        bufs, _ = _run(w, kernel)
        _check(bufs.out, w, oracle, f"edge lens/{kernel}")
    # rows past context_len hold NaN: they must not leak (select, not multiply)
    w2 = W.make_test_shaped(batch_size=2, nheads=8, nheads_k=2, d=128, seqlen_k=300, varlen=True,
                            has_sinks=False, seed=11)
    base_k, base_v = w2.key_cache.clone(), w2.value_cache.clone()
    for s in range(2):
        n = int(w2.context_lens[s])
        for t in range(n, w2.block_tables.shape[1] * w2.block_size):
            blk = int(w2.block_tables[s, t // w2.block_size])
            w2.key_cache[blk, t % w2.block_size] = float("nan")
            w2.value_cache[blk, t % w2.block_size] = float("nan")
    for kernel in ("loop", "reduce"):
        bufs, _ = _run(w2, kernel)
        w2.key_cache, w2.value_cache = base_k, base_v
        _check(bufs.out, w2, oracle, f"nan tail/{kernel}")
        w2.key_cache, w2.value_cache = w2.key_cache.clone(), w2.value_cache.clone()
    # a zero-length sequence leaves its output rows untouched
    w3 = W.make_config(0, lens=[0, 40, 0, 7])
    bufs, _ = _run(w3, "loop")
    out = bufs.out.cpu()
    assert (out[0] == 0).all() and (out[2] == 0).all()
    ref = call_oracle(oracle.attention_ref, w3)
    torch.testing.assert_close(out[[1, 3]].float(), ref[[1, 3]].float(), atol=ATOL, rtol=RTOL)


def test_large_batch_runs_as_sub_batches(oracle):
    """More sequences than the persistent kernels list (256 split, 128 loop): the launchers cut
    the batch into equal sub-batches, one persistent launch each.  The loop launcher gives short rows of
    16-bit caches to the grid form in one launch; in a table of more than 2048 keys it cannot tell."""
    gen = torch.Generator().manual_seed(5)
    lens = torch.randint(1, 700, (300,), generator=gen).tolist()
    w = W.make_config(0, num_seqs=300, pool_blocks=300 * 44, lens=lens)
    w.partition_size = 256
    for kernel in ("reduce", "loop"):
        bufs, _ = _run(w, kernel)
        _check(bufs.out, w, oracle, f"300 sequences/{kernel}")
    w.block_tables = _wide(w.block_tables, 2064 // w.block_size)
    bufs, _ = _run(w, "loop")
    _check(bufs.out, w, oracle, "300 sequences in a wide table/loop")


def test_persistent_split_many_items_per_wavefront(oracle):
    """Enough live partitions that every resident wavefront walks several items, with
    sinks, ragged lengths and empty sequences in between."""
    gen = torch.Generator().manual_seed(9)
    lens = torch.randint(1, 3000, (200,), generator=gen)
    lens[::7] = 0
    w = W.make_config(0, num_seqs=200, pool_blocks=200 * 188, lens=lens.tolist())
    w.partition_size = 256
    w.sinks = torch.linspace(-2, 2, w.num_heads).to(w.query.dtype)
    bufs, _ = _run(w, "reduce")
    out = bufs.out.cpu()
    assert (out[lens == 0] == 0).all()
    ref = call_oracle(oracle.attention_ref, w)
    live = lens > 0
    torch.testing.assert_close(out[live].float(), ref[live].float(), atol=ATOL, rtol=RTOL)


def _segment_mark(word):
    """Segment length in the low byte of a mark, as slot 1 of a row of max_logits holds one behind a segment of
    two or more partitions (None: the word is no mark)."""
    bits = int(word.view(torch.int32).item()) & 0xFFFFFFFF
    return (bits & 0xFF) if (bits & 0xFFFFFF00) == 0x7FD3A600 else None


@pytest.mark.parametrize("batch", ["many_short", "few_long", "one_partition_each"])
def test_segment_kernel_partials_lie_a_segment_apart(oracle, batch):
    """Batches that the split path works in segments of several partitions: the output matches the
    oracle, and the scratch arrays hold one partial per segment, in the slot of the segment's
    first partition -- the partials the kernel model gives for a partition size of one segment --
    and, in slot 1 of max_logits of every row of two or more partitions, a mark (the reduce kernel takes marked
    slots for covered ones; the mark's low byte tells the segment length)."""
    gen = torch.Generator().manual_seed(21)
    if batch == "many_short":     # many sequences per compute unit: most sequences are one segment
        S = 64
        lens = torch.randint(1, 5000, (S,), generator=gen)
        lens[5] = 0
        lens[6] = 4096          # ends exactly on a partition boundary
    elif batch == "few_long":   # whole segments are the work: one per compute unit
        S = 5
        lens = torch.randint(6000, 20000, (S,), generator=gen)
        lens[1] = 300           # a row of one partition: nothing to mark
        lens[3] = 0
    else:                       # no sequence reaches a second partition, though there are slots for two
        S = 200
        lens = torch.randint(1, 512, (S,), generator=gen)
    w = W.make_config(4, num_seqs=S, pool_blocks=int(sum(-(-int(n) // 16) for n in lens)) + 8,
                      lens=lens.tolist())   # bf16 queries, E5M2 pools, G = 8
    w.sinks = torch.linspace(-1, 3, w.num_heads).to(w.query.dtype)
    from flash_attention_factory_amd import runner
    wd = w.to(_dev())
    bufs = runner.alloc_buffers(wd, max_num_partitions=2 if batch == "one_partition_each" else None)
    for t in (bufs.exp_sums, bufs.max_logits, bufs.tmp_out):
        t.fill_(float("nan"))
    runner.run_workload(wd, "fp8_reduce", bufs)
    torch.cuda.synchronize()
    out = bufs.out.cpu()
    ref = call_oracle(oracle.attention_ref, w)
    live = lens > 0
    torch.testing.assert_close(out[live].float(), ref[live].float(), atol=ATOL, rtol=RTOL)
    es = bufs.exp_sums.cpu()
    ml = bufs.max_logits.cpu()
    P = w.partition_size
    if batch == "one_partition_each":
        # one partial per row, in slot 0; slot 1 is nobody's: whatever it holds, nothing reads it
        assert (~torch.isnan(es[live][:, :, 0])).all() and torch.isnan(es[:, :, 1]).all()
        # and every row's only partial is its result: stored into `out`, tmp_out left alone
        assert torch.isnan(bufs.tmp_out).all()
        return
    # which slots were written: 0, m, 2m, ...
    longest = int(lens.argmax())
    written = (~torch.isnan(es[longest, 0])).nonzero().flatten().tolist()
    assert written[0] == 0 and len(written) >= 2
    m = written[1]
    assert m >= 2, "this batch is meant to be cut into multi-partition segments"
    for s in range(S):
        nseg = -(-int(lens[s]) // (m * P))
        want = [j * m for j in range(nseg)]
        assert (~torch.isnan(es[s, 0])).nonzero().flatten().tolist() == want, s
        for h in range(w.num_heads):  # the mark: on every row with a second partition, nowhere else
            mark = _segment_mark(ml[s, h, 1])
            assert mark == (m if int(lens[s]) > P else None), (s, h, mark)
    NP = bufs.exp_sums.shape[2]
    mes, mml, mtmp = call_oracle(oracle.kernel_partition, w, partition_size=m * P, max_num_partitions=NP)
    for s in range(S):
        nseg = -(-int(lens[s]) // (m * P))
        for j in range(nseg):
            torch.testing.assert_close(ml[s, :, j * m], mml[s, :, j], atol=1e-3, rtol=1e-4)
            torch.testing.assert_close(es[s, :, j * m], mes[s, :, j], atol=1e-3, rtol=2e-3)
            if nseg > 1:
                torch.testing.assert_close(bufs.tmp_out[s, :, j * m].cpu(), mtmp[s, :, j], atol=1e-2, rtol=1e-2)
        if nseg == 1:  # the only partial of a row is its result: it went to `out`, tmp_out was left alone
            assert torch.isnan(bufs.tmp_out[s]).all(), s


def _segment_batches(name):
    gen = torch.Generator().manual_seed(33)
    if name == "one_segment_per_unit":      # three long sequences, two work-groups per compute unit
        lens = [21000, 9000, 15000]
        w = W.make_config(2, num_seqs=3, pool_blocks=sum(-(-n // 16) for n in lens) + 4, lens=lens)
        return w, "reduce"
    if name == "three_groups_per_unit":     # head size 64: three work-groups share a compute unit
        w = W.make_test_shaped(batch_size=96, nheads=16, nheads_k=4, d=64, seqlen_k=3000, varlen=True,
                               has_sinks=True, seed=5)
        w.context_lens[::7] = torch.randint(1, 3000, (14,), generator=gen).to(torch.int32)
        return w, "reduce"
    if name == "longest_segment":           # partitions of 64 tokens: the segment length meets its cap
        S = 64
        lens = torch.randint(7000, 8193, (S,), generator=gen).tolist()
        w = W.make_config(4, num_seqs=S, pool_blocks=S * 512 + 8, lens=lens)
        w.partition_size = 64
        return w, "fp8_reduce"
    S = 256                                  # many_sequences: most of them stay whole
    lens = torch.randint(1, 2600, (S,), generator=gen)
    lens[::9] = torch.randint(4000, 9000, (29,), generator=gen)
    w = W.make_config(4, num_seqs=S, pool_blocks=int(sum(-(-int(n) // 16) for n in lens)) + 8, lens=lens.tolist())
    return w, "fp8_reduce"


def _split_plan(wd, kernel):
    """fa_paged_attention_reduce_plan of the call runner.run_workload makes for this workload."""
    import ctypes
    from flash_attention_factory_amd import _cabi, runner
    kc = runner.logical_cache_view(wd, wd.key_cache)
    sh = _cabi.Shape()
    sh.num_seqs, sh.num_heads, sh.head_size = wd.query.shape
    sh.num_kv_heads, sh.block_size = wd.num_kv_heads, wd.block_size
    sh.max_blocks_per_seq, sh.max_num_partitions, sh.partition_size = wd.block_tables.shape[1], wd.max_num_partitions, wd.partition_size
    sh.kv_block_stride, sh.kv_token_stride, sh.kv_head_stride = kc.stride(0), kc.stride(1), kc.stride(2)
    sh.q_dtype = _cabi.FA_DTYPE_BF16 if wd.query.dtype == torch.bfloat16 else _cabi.FA_DTYPE_F16
    sh.num_pool_blocks = kc.size(0)
    plan = _cabi.SplitPlan()
    _cabi.check(_cabi.load().fa_paged_attention_reduce_plan(ctypes.byref(sh), None, 0, int(kernel.startswith("fp8")), 0,
                                                            ctypes.byref(plan)))
    return plan


@pytest.mark.parametrize("name", ["one_segment_per_unit", "three_groups_per_unit", "longest_segment", "many_sequences",
                                  "even_shares"])
def test_segment_length_regimes(oracle, name):
    """One batch for each way the split path arrives at its cuts (one segment per compute unit; half a
    work-group's load where three share a unit; the cap of 64 partitions; a share of a unit's load with
    many sequences; even shares on request): the output matches the oracle, every mark of the launch
    tells the same cut, and exactly the slots that cut names hold partials -- 0, m, 2m, ... of a row's
    live partitions for segments, the starts of the work-groups' shares and of the rows for even shares."""
    import _segment_policy as SP
    forced = 0
    if name == "even_shares":
        name, forced = "many_sequences", -1
    w, kernel = _segment_batches(name)
    from flash_attention_factory_amd import runner
    wd = w.to(_dev())
    bufs = runner.alloc_buffers(wd)
    for t in (bufs.exp_sums, bufs.max_logits, bufs.tmp_out):
        t.fill_(float("nan"))
    runner.run_workload(wd, kernel, bufs, segment_partitions=forced)
    torch.cuda.synchronize()
    _check(bufs.out, w, oracle, f"segment lengths, {name}")
    es = bufs.exp_sums.cpu()
    ml = bufs.max_logits.cpu()
    P = w.partition_size
    lens = [int(n) for n in w.context_lens.tolist()]
    bits = ml.view(torch.int32)
    marks = set((bits[(bits & 0xFFFFFF00) == 0x7FD3A600] & 0xFF).tolist())
    assert len(marks) <= 1, marks
    m = marks.pop() if marks else 1
    print(f"{name}: " + (f"{m} partitions per segment" if m else "even shares"), flush=True)
    if forced:
        assert m == 0
    elif name == "longest_segment":
        assert m == 64
    elif name != "three_groups_per_unit":
        assert m > 1
    group = w.num_heads // w.num_kv_heads
    if m == 0:
        plan = _split_plan(wd, kernel)
        per_item = plan.kv_heads_per_item
        pieces = SP.even_shares_pieces(lens, partition_size=P, max_num_partitions=w.max_num_partitions,
                                       max_ctx=w.block_tables.shape[1] * w.block_size,
                                       num_kv_heads=w.num_kv_heads // per_item, groups=plan.work_groups,
                                       cus=plan.compute_units)
    for s, n in enumerate(lens):
        for h in (0, w.num_heads - 1):
            if m == 0:
                want = [first for first, _, _ in pieces.get((s, h // (group * per_item)), [])]
            else:
                want = [j * m for j in range(-(-n // (m * P)))]
            assert (~torch.isnan(es[s, h])).nonzero().flatten().tolist() == want, (s, h)
            # every slot a piece covers beyond its first holds the mark, in max_logits only
            live = -(-n // P)
            covered = [q for q in range(live) if q not in want]
            assert all(_segment_mark(ml[s, h, q]) == m for q in covered), (s, h)


@pytest.mark.parametrize("shape", ["few_items", "one_group_per_unit", "all_groups", "gqa"])
def test_fp8_loop_two_kv_heads_per_work_group(oracle, shape):
    """FP8 pools in upstream's layout with head size 128: the persistent loop kernel gives a
    work-group two adjacent kv heads of a sequence, a team of two wavefronts each -- fewer pairs
    than compute units (where single heads stay the items), one work-group per unit, all resident
    work-groups, and a grouped-query shape; ragged lengths with empty sequences and sinks."""
    gen = torch.Generator().manual_seed(91)
    if shape == "gqa":   # 8 kv heads of 8 query heads each, bf16 queries
        index, S, hi, fp8_dtype = 4, 80, 2000, torch.float8_e4m3fn
    else:                # 32 kv heads, one query head each, fp16 queries
        index, fp8_dtype = 3, torch.float8_e5m2
        S, hi = {"few_items": (6, 2500), "one_group_per_unit": (32, 1200), "all_groups": (128, 300)}[shape]
    lens = torch.randint(1, hi, (S,), generator=gen)
    lens[1] = 0
    lens[2] = 16
    w = W.make_config(index, num_seqs=S, pool_blocks=int(sum(-(-int(n) // 16) for n in lens)) + 8, lens=lens.tolist(),
                      layout=W.TOKEN_MAJOR, fp8_dtype=fp8_dtype)
    w.sinks = torch.linspace(-2, 2, w.num_heads).to(w.query.dtype)
    bufs, _ = _run(w, "fp8_loop")
    out = bufs.out.cpu()
    assert (out[lens == 0] == 0).all()
    _check(bufs.out, w, oracle, f"loop kernel, two kv heads per work-group, {shape}")


@pytest.mark.parametrize("fp8_dtype", [torch.float8_e5m2, torch.float8_e4m3fn])
def test_fp8_split_two_kv_heads_per_work_group(oracle, fp8_dtype):
    """FP8 pools in upstream's layout with head size 128: the segment kernel gives a work-group two
    adjacent kv heads of a segment, a team of two wavefronts each.  Ragged lengths (empty, one chunk,
    one partition exactly, many segments), sinks: parity with the oracle, partials in the slots
    0, m, 2m, ... of every head of a pair, one mark per row of two or more partitions."""
    gen = torch.Generator().manual_seed(77)
    S = 40
    lens = torch.randint(1, 3000, (S,), generator=gen)
    lens[0], lens[3], lens[4], lens[9], lens[17] = 0, 20, 512, 9000, 6100
    w = W.make_config(4, num_seqs=S, pool_blocks=int(sum(-(-int(n) // 16) for n in lens)) + 8, lens=lens.tolist(),
                      layout=W.TOKEN_MAJOR, fp8_dtype=fp8_dtype)
    w.sinks = torch.linspace(-1, 3, w.num_heads).to(w.query.dtype)
    from flash_attention_factory_amd import runner
    wd = w.to(_dev())
    bufs = runner.alloc_buffers(wd)
    for t in (bufs.exp_sums, bufs.max_logits, bufs.tmp_out):
        t.fill_(float("nan"))
    runner.run_workload(wd, "fp8_reduce", bufs)
    torch.cuda.synchronize()
    _check(bufs.out, w, oracle, f"two kv heads per work-group, {fp8_dtype}")
    es = bufs.exp_sums.cpu()
    ml = bufs.max_logits.cpu()
    P = w.partition_size
    marks = {_segment_mark(ml[s, h, 1]) for s in range(S) for h in range(w.num_heads) if int(lens[s]) > P}
    assert len(marks) == 1, marks
    m = marks.pop() or 1
    for s in range(S):
        want = [j * m for j in range(-(-int(lens[s]) // (m * P)))]
        for h in range(w.num_heads):
            assert (~torch.isnan(es[s, h])).nonzero().flatten().tolist() == want, (s, h)


@pytest.mark.parametrize("batch,heads", [(300, 16), (128, 32)])
def test_reduce_kernel_one_wavefront_form(oracle, batch, heads):
    """From 4096 (sequence, head) pairs on the reduce kernel runs one wavefront per pair;
    lengths up to 9 partitions of 256 tokens exercise its multi-row batches."""
    w = W.make_test_shaped(batch_size=batch, nheads=heads, nheads_k=2, d=64, seqlen_k=4500 if batch == 128 else 600,
                           varlen=True, has_sinks=True, seed=batch)
    assert w.num_seqs * w.num_heads >= 4096
    if batch == 128:  # from 1 to more than 64 partitions per sequence: several row batches and groups
        w.partition_size = 64
        assert w.max_num_partitions > 64
        w.context_lens[::3] = 4500 - torch.arange(0, 43, dtype=torch.int32) * 104
    bufs, _ = _run(w, "reduce")
    _check(bufs.out, w, oracle, f"reduce 1-wave form, {batch} sequences x {heads} heads")


@pytest.mark.parametrize("layout", [W.HEAD_MAJOR, W.TOKEN_MAJOR])
@pytest.mark.parametrize("index", [1, 2, 3, 4])
def test_full_size_configs(oracle, index, layout):
    """The measured configurations at their full sizes, in both pool layouts (in upstream's, the
    FP8 configurations run the instances that give a work-group two kv heads).  The pools are drawn on the GPU
    (a gigabyte of normals takes the host a minute) and copied back for the oracle, so
    both sides see the same bytes.  Also checked at full size: loop == split + reduce,
    and invariance under a permutation of the pool's blocks together with the tables."""
    from flash_attention_factory_amd import runner
    dev = _dev()
    wd = W.make_config(index, device=dev, pools_on_device=True, layout=layout)
    w = wd.to("cpu")
    kernel = W.CONFIG_KERNEL[index]
    bufs = runner.alloc_buffers(wd)
    runner.run_workload(wd, kernel, bufs)
    torch.cuda.synchronize()
    _check(bufs.out, w, oracle, f"full {w.name}, {layout}")
    other = {"loop": "reduce", "reduce": "loop", "fp8_loop": "fp8_reduce", "fp8_reduce": "fp8_loop"}[kernel]
    bufs2 = runner.alloc_buffers(wd)
    runner.run_workload(wd, other, bufs2, schedule=3)  # the split kernels also where the rows are short
    torch.cuda.synchronize()
    a, b = bufs.out.float(), bufs2.out.float()
    ulps = 2.0 ** (-7 if w.query.dtype == torch.bfloat16 else -10)  # two 16-bit roundings apart
    assert (a - b).abs().max().item() <= ulps * a.abs().max().item() + 1e-5
    # permute the pool's blocks and rewrite the tables: same answer, bit for bit
    NB = wd.key_cache.shape[0]
    perm = torch.randperm(NB, device=dev)
    inv = torch.empty_like(perm)
    inv[perm] = torch.arange(NB, device=dev)
    del bufs2
    w2 = W.Workload(**{**wd.__dict__})
    w2.key_cache = wd.key_cache[perm]
    w2.value_cache = wd.value_cache[perm]
    w2.block_tables = inv[wd.block_tables.long()].to(torch.int32)
    bufs3 = runner.alloc_buffers(w2)
    runner.run_workload(w2, kernel, bufs3)
    torch.cuda.synchronize()
    assert torch.equal(bufs3.out, bufs.out)


def test_persistent_kernels_small_batches(oracle):
    """Fewer items than resident work-groups, a single sequence, a batch where most
    wavefronts of a loop work-group have no chunk, and 128 sequences (the limit of the
    persistent loop kernel) next to 129 (one launch of the grid form; in a table of more than
    2048 keys two sub-batches of 65 and 64)."""
    cases = [
        W.make_config(1, num_seqs=1, pool_blocks=200, lens=[1999]),
        W.make_config(0, num_seqs=3, pool_blocks=64, lens=[5, 40, 33]),
        W.make_config(3, num_seqs=2, pool_blocks=300, lens=[17, 2048]),
        W.make_config(0, num_seqs=128, pool_blocks=128 * 8, lens=[(7 * s) % 120 + 1 for s in range(128)]),
        W.make_config(0, num_seqs=129, pool_blocks=129 * 8, lens=[(11 * s) % 120 + 1 for s in range(129)]),
    ]
    for w in cases:
        for kernel in (("fp8_loop", "fp8_reduce") if w.is_fp8 else ("loop", "reduce")):
            bufs, _ = _run(w, kernel)
            _check(bufs.out, w, oracle, f"{w.name} S={w.num_seqs}/{kernel}")
    w.block_tables = _wide(w.block_tables, 2064 // w.block_size)
    bufs, _ = _run(w, "loop")
    _check(bufs.out, w, oracle, f"{w.name} S={w.num_seqs}/loop in a wide table")


def test_table_wider_than_the_persistent_loop_key(oracle):
    """A block table that could hold 2^24 tokens or more per sequence is outside what the
    persistent loop kernel packs into its sort key; the launcher must take the grid form."""
    w = W.make_config(0, num_seqs=2, pool_blocks=64, lens=[40, 33])
    wide = torch.zeros((2, (1 << 24) // w.block_size), dtype=torch.int32)
    wide[:, :w.block_tables.shape[1]] = w.block_tables
    w.block_tables = wide
    for kernel in ("loop", "reduce"):
        bufs, _ = _run(w, kernel, max_context_len=40)
        _check(bufs.out, w, oracle, f"2^24-token table/{kernel}")


def test_grid_forms_on_a_ragged_batch(oracle):
    """The grid forms (one work-group per (kv head[, partition], sequence)) serve what the
    persistent kernels do not take; a table of 2^24 tokens per sequence selects them.  A ragged
    batch with sinks, empty sequences and several partitions, 16-bit and E5M2."""
    gen = torch.Generator().manual_seed(17)
    lens = torch.randint(1, 1400, (6,), generator=gen)
    lens[2] = 0
    for index in (1, 3):
        w = W.make_config(index, num_seqs=6, pool_blocks=600, lens=lens.tolist())
        w.sinks = torch.linspace(-1, 1, w.num_heads).to(w.query.dtype)
        wide = torch.zeros((6, (1 << 24) // w.block_size), dtype=torch.int32)
        wide[:, :w.block_tables.shape[1]] = w.block_tables
        w.block_tables = wide
        for kernel in (("fp8_loop", "fp8_reduce") if w.is_fp8 else ("loop", "reduce")):
            bufs, _ = _run(w, kernel, max_context_len=int(lens.max()))
            out = bufs.out.cpu()
            assert (out[2] == 0).all()
            ref = call_oracle(oracle.attention_ref, w)
            live = lens > 0
            torch.testing.assert_close(out[live].float(), ref[live].float(), atol=ATOL, rtol=RTOL,
                                       msg=lambda m: f"grid {kernel}: {m}")


@pytest.mark.parametrize("qdtype", [torch.float16, torch.bfloat16])
def test_e4m3_caches(oracle, qdtype):
    """FP8 caches in the E4M3 format (torch.float8_e4m3fn pools) through all four FP8 code
    paths: loop and split kernels, head sizes 128 and 64, with sinks and a non-unit scale."""
    cases = [
        W.make_test_shaped(batch_size=3, nheads=8, nheads_k=2, d=128, seqlen_k=1500, varlen=True, has_sinks=True,
                           fp8=True, dtype=qdtype, fp8_dtype=torch.float8_e4m3fn),
        W.make_test_shaped(batch_size=2, nheads=6, nheads_k=6, d=64, seqlen_k=333, varlen=True, has_sinks=False,
                           fp8=True, dtype=qdtype, fp8_dtype=torch.float8_e4m3fn, block_size=16, layout=W.HEAD_MAJOR),
    ]
    cases[1].fp8_scale = 0.5
    if qdtype == torch.float16:
        cases.append(W.make_config(3, num_seqs=6, pool_blocks=800, fp8_dtype=torch.float8_e4m3fn))
    else:
        cases.append(W.make_config(4, num_seqs=5, pool_blocks=8192, fp8_dtype=torch.float8_e4m3fn))
    for w in cases:
        assert w.key_cache.dtype == torch.float8_e4m3fn
        for kernel in ("fp8_loop", "fp8_reduce"):
            bufs, _ = _run(w, kernel)
            _check(bufs.out, w, oracle, f"e4m3 {w.name}/{kernel}")


def test_e4m3_special_bytes(oracle):
    """Every E4M3 byte as a K and a V value (NaN codes kept beyond the context): the decode
    agrees with the oracle's table on all 254 numbers, subnormals included."""
    w = W.make_test_shaped(batch_size=1, nheads=2, nheads_k=1, d=64, seqlen_k=256, varlen=False, has_sinks=False,
                           fp8=True, fp8_dtype=torch.float8_e4m3fn, block_size=64)
    codes = torch.arange(256, dtype=torch.int32).to(torch.uint8)
    numbers = codes[(codes & 0x7f) != 0x7f]                       # all but the two NaN codes
    vals = numbers[torch.randperm(254, generator=torch.Generator().manual_seed(0))]
    kc = w.key_cache.view(torch.uint8).view(-1)
    vc = w.value_cache.view(torch.uint8).view(-1)
    kc.copy_(vals.repeat(kc.numel() // 254 + 1)[:kc.numel()])
    vc.copy_(vals.flip(0).repeat(vc.numel() // 254 + 1)[:vc.numel()])
    w.scale = 1e-4                                                 # keeps the logits of +-448 values finite
    bufs, _ = _run(w, "fp8_loop")
    ref = call_oracle(oracle.attention_ref, w, want_f32=True)[1]
    got = bufs.out.float().cpu()
    assert torch.isfinite(got).all()
    torch.testing.assert_close(got, ref, atol=5e-2, rtol=1e-2)    # values up to 448: the bar scales with them


@pytest.mark.parametrize("qdtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("layout", [W.TOKEN_MAJOR, W.HEAD_MAJOR])
def test_e5m2_special_bytes(oracle, qdtype, layout):
    """Every E5M2 byte through the decode of both FP8 kernels (fp16 queries: the byte-permute decode;
    bf16 queries: the CDNA4 conversion instruction): all 248 finite codes -- both zeros, the
    subnormals, up to +-57344 -- as K and V values inside the contexts, the infinity and NaN codes
    in every row past a context's end."""
    codes = torch.arange(256, dtype=torch.int32).to(torch.uint8)
    finite = codes[(codes & 0x7c) != 0x7c]
    special = codes[(codes & 0x7c) == 0x7c]  # +-inf and the six NaN codes
    assert finite.numel() == 248 and special.numel() == 8
    g = torch.Generator().manual_seed(1)
    w = W.make_test_shaped(batch_size=3, nheads=8, nheads_k=2, d=128, seqlen_k=640, varlen=False, has_sinks=False,
                           fp8=True, block_size=16, dtype=qdtype, layout=layout)
    w.context_lens = torch.tensor([640, 333, 17], dtype=torch.int32)
    n = w.key_cache.numel()
    kb, vb = w.key_cache.view(torch.uint8), w.value_cache.view(torch.uint8)
    kb.view(-1).copy_(finite[torch.randint(0, 248, (n,), generator=g)])
    vb.view(-1).copy_(finite[torch.randint(0, 248, (n,), generator=g)])
    B = w.block_size
    for s_ in range(3):  # rows at and past the end of each context: infinities and NaNs
        ctx = int(w.context_lens[s_])
        for col in range(ctx // B, w.block_tables.shape[1]):
            blk = int(w.block_tables[s_, col])
            first = ctx - col * B if col == ctx // B else 0
            rows = slice(max(first, 0), B)
            for pool in (kb, vb):
                view = pool[blk] if layout == W.TOKEN_MAJOR else pool[blk].permute(1, 0, 2)  # [row, head, d]
                view[rows] = special[torch.randint(0, 8, tuple(view[rows].shape), generator=g)]
    w.scale = 1e-6  # values reach 57344: keeps the logits moderate
    ref = call_oracle(oracle.attention_ref, w, want_f32=True)[1]
    assert torch.isfinite(ref).all()
    unit = ref.abs().max()
    for kernel in ("fp8_loop", "fp8_reduce"):
        for schedule in (0, 1):
            bufs, _ = _run(w, kernel, schedule=schedule)
            got = bufs.out.float().cpu()
            assert torch.isfinite(got).all(), (kernel, schedule)
            torch.testing.assert_close(got / unit, ref / unit, atol=ATOL, rtol=RTOL,
                                       msg=lambda m: f"{kernel} schedule {schedule}: {m}")


@pytest.mark.parametrize("qdtype", [torch.float16, torch.bfloat16])
def test_e5m2_infinities_inside_the_context(oracle, qdtype):
    """+-inf bytes among the values a query sees act as IEEE arithmetic says, in the kernels as in the
    oracle: an infinite V entry under uniform weights makes that output element infinite (NaN where
    both signs meet), an infinite K row makes the rows of its sequence NaN; other sequences are untouched."""
    w = W.make_test_shaped(batch_size=3, nheads=4, nheads_k=2, d=128, seqlen_k=96, varlen=False, has_sinks=False,
                           fp8=True, block_size=16, dtype=qdtype)
    w.query[0] = 0                      # sequence 0: uniform weights
    w.query[1] = w.query[1].abs() + 0.5  # sequence 1: positive queries, so an all-+inf K row scores +inf
    kb, vb = w.key_cache.view(torch.uint8), w.value_cache.view(torch.uint8)
    b0, b1 = int(w.block_tables[0, 2]), int(w.block_tables[1, 1])
    vb[b0, 3, 0, 5] = 0x7c     # +inf: token 35 of sequence 0, kv head 0, d 5
    vb[b0, 4, 0, 9] = 0xfc     # -inf: d 9
    vb[b0, 5, 1, 7] = 0x7c     # kv head 1: +inf and -inf in the same column -> NaN
    vb[b0, 6, 1, 7] = 0xfc
    kb[b1, 2, 0, :] = 0x7c     # sequence 1, token 18, kv head 0: a K row of +inf
    ref = call_oracle(oracle.attention_ref, w, want_f32=True)[1]
    assert torch.isposinf(ref[0, 0, 5]) and torch.isneginf(ref[0, 1, 9]) and torch.isnan(ref[0, 2, 7])
    assert torch.isnan(ref[1, :2]).all() and torch.isfinite(ref[1, 2:]).all() and torch.isfinite(ref[2]).all()
    for kernel in ("fp8_loop", "fp8_reduce"):
        bufs, _ = _run(w, kernel)
        got = bufs.out.float().cpu()
        assert torch.equal(torch.isnan(got), torch.isnan(ref)), kernel
        assert torch.equal(torch.isposinf(got), torch.isposinf(ref)) and torch.equal(torch.isneginf(got), torch.isneginf(ref)), kernel
        fin = torch.isfinite(ref)
        torch.testing.assert_close(got[fin], ref[fin], atol=ATOL, rtol=RTOL)


def test_bf16_and_fp8_scale(oracle):
    # bf16 queries with a bf16 cache, and with an FP8 cache at a non-unit scale
    w = W.make_test_shaped(batch_size=2, nheads=8, nheads_k=2, d=128, seqlen_k=700, varlen=True,
                           has_sinks=True, dtype=torch.bfloat16)
    bufs, _ = _run(w, "loop")
    _check(bufs.out, w, oracle, "bf16 cache/loop")
    w8 = W.make_test_shaped(batch_size=2, nheads=8, nheads_k=2, d=64, seqlen_k=700, varlen=True,
                            has_sinks=False, dtype=torch.bfloat16, fp8=True)
    w8.fp8_scale = 0.5  # parity unpinned upstream (tests only pass 1.0); checked against our reading
    for kernel in ("fp8_loop", "fp8_reduce"):
        bufs, _ = _run(w8, kernel)
        _check(bufs.out, w8, oracle, f"bf16 q, fp8 cache, scale 0.5/{kernel}")


UPSTREAM_HEADS = [(8, 1), (16, 2), (10, 2), (14, 2), (12, 2), (8, 2), (6, 2), (4, 2), (2, 2)]
UPSTREAM_SHORT = [128, 339, 1024, 800, 256, 799, 2048]
UPSTREAM_LONG = [20000, 40000, 50000]


@pytest.mark.parametrize("heads", UPSTREAM_HEADS, ids=lambda h: f"h{h[0]}x{h[1]}")
@pytest.mark.parametrize("fp8", [False, True])
def test_whole_upstream_grid(oracle, heads, fp8):
    """Every case of the upstream test grid (test_paged.py:211-256, test_paged_fp8cache.py:220-264:
    batch 1/2 x sinks x var-len x head size 128/64 x nine head pairs x ten context lengths, block
    64, fp16) through the loop and the split kernel, with upstream's own gate next to the
    absolute one, twice: err <= 3 x err of the rounding-faithful kernel model + 1e-5, and literally,
    err <= 3 x err(out_pt) + 1e-5 with out_pt the reference evaluated without the fp32 upcast
    (test_paged.py:432-447, 603-604).
    All 2 x 1440 cases (two minutes, most of it the oracle on the three long lengths); with
    FA_QUICK_UPSTREAM_GRID=1 the seven lengths up to 2048 in full and of the long ones (20000-50000)
    one combination of the other parameters each, rotating.  (Rows of up to 1024 keys would make the
    split entry run the single-pass kernel, which the loop entry covers: _run asks for the split
    kernels there.)"""
    nheads, nheads_k = heads
    combos = [(b, s, v, d) for b in (1, 2) for s in (True, False) for v in (False, True) for d in (128, 64)]
    n = 0
    for seqlen_k in UPSTREAM_SHORT:
        for b, s, v, d in combos:
            w = W.make_test_shaped(batch_size=b, nheads=nheads, nheads_k=nheads_k, d=d, seqlen_k=seqlen_k, varlen=v,
                                   has_sinks=s, fp8=fp8)
            for kernel in (("fp8_loop", "fp8_reduce") if fp8 else ("loop", "reduce")):
                bufs, times = _run(w, kernel)  # (the split kernels also where rows are short: see _run)
                assert "reduce" not in kernel or times[1] > 0.0
                _check(bufs.out, w, oracle, f"{w.name}/{kernel}", literal_rule=True)
            n += 1
    everything = os.environ.get("FA_QUICK_UPSTREAM_GRID") != "1"   # the long lengths in full too
    for k, seqlen_k in enumerate(UPSTREAM_LONG):
        one = combos[(3 * UPSTREAM_HEADS.index(heads) + k + (8 if fp8 else 0)) % len(combos)]
        for b, s, v, d in (combos if everything else [one]):
            w = W.make_test_shaped(batch_size=b, nheads=nheads, nheads_k=nheads_k, d=d, seqlen_k=seqlen_k, varlen=v,
                                   has_sinks=s, fp8=fp8)
            for kernel in (("fp8_loop", "fp8_reduce") if fp8 else ("loop", "reduce")):
                bufs, _ = _run(w, kernel)
                _check(bufs.out, w, oracle, f"{w.name}/{kernel}", literal_rule=True)
            n += 1
    assert n == len(UPSTREAM_SHORT) * 16 + len(UPSTREAM_LONG) * (16 if everything else 1)


def test_run_rejects_host_tensors_and_mismatched_shapes():
    """Nothing reaches a kernel unless it lives on the query's device and has the shape the kernel
    assumes: a host block table or length array would be a GPU memory fault, not an exception."""
    from flash_attention_factory_amd import _cabi, runner
    from flash_attention_factory_amd.lib import kv_cache_write, paged_attention_reduce
    w = W.make_test_shaped(batch_size=2, nheads=8, nheads_k=2, d=128, seqlen_k=300, varlen=True, has_sinks=True).to(_dev())
    bufs = runner.alloc_buffers(w)
    good = dict(max_logits=bufs.max_logits, exp_sums=bufs.exp_sums, tem_output=bufs.tmp_out, output=bufs.out,
                key_cache=w.key_cache, value_cache=w.value_cache, block_tables=w.block_tables,
                context_lens=w.context_lens, sinks=w.sinks)

    def call(**over):
        a = dict(good, **over)
        return paged_attention_reduce.run(a["max_logits"], a["exp_sums"], a["tem_output"], a["output"], None, w.query,
                                          a["key_cache"], a["value_cache"], a["block_tables"], a["context_lens"], 4,
                                          w.scale, w.block_size, 300, None, a["sinks"], 0.0)
    call()
    for name in good:
        with pytest.raises(_cabi.PagedAttentionError, match=name):
            call(**{name: good[name].cpu()})
    with pytest.raises(_cabi.PagedAttentionError, match="block_tables"):
        call(block_tables=w.block_tables[:1].contiguous())
    with pytest.raises(_cabi.PagedAttentionError, match="context_lens"):
        call(context_lens=w.context_lens[:1].contiguous())
    with pytest.raises(_cabi.PagedAttentionError, match="sinks"):
        call(sinks=w.sinks.float())
    with pytest.raises(_cabi.PagedAttentionError, match="sinks"):
        call(sinks=w.sinks[:4].contiguous())
    with pytest.raises(_cabi.PagedAttentionError, match="rows of 64"):
        call(key_cache=w.key_cache[..., :64], value_cache=w.value_cache[..., :64])
    key = torch.zeros((3, 2, 128), dtype=torch.float16, device=_dev())
    slots = torch.tensor([0, 1, 2], device=_dev())
    kv_cache_write.run(key, key, w.key_cache, w.value_cache, slots)
    for over in (dict(value=key.cpu()), dict(key_cache=w.key_cache.cpu()), dict(value_cache=w.value_cache.cpu()),
                 dict(slot_mapping=slots.cpu())):
        a = dict(dict(value=key, key_cache=w.key_cache, value_cache=w.value_cache, slot_mapping=slots), **over)
        with pytest.raises(_cabi.PagedAttentionError, match=next(iter(over))):
            kv_cache_write.run(key, a["value"], a["key_cache"], a["value_cache"], a["slot_mapping"])


def test_seventy_thousand_sequences(oracle):
    """More sequences than a grid dimension holds (65535): every path cuts the batch into launches."""
    S = 70000
    gen = torch.Generator().manual_seed(5)
    lens = torch.randint(0, 40, (S,), generator=gen)
    for fp8 in (False, True):
        w = W.make_test_shaped(batch_size=S, nheads=2, nheads_k=1, d=64, seqlen_k=48, varlen=False, has_sinks=False,
                               fp8=fp8, block_size=16, seed=9)
        w.context_lens = lens.to(torch.int32)
        w.partition_size = 256
        _, ref32 = call_oracle(oracle.attention_ref, w, want_f32=True)
        live = lens > 0
        for kernel, schedule in (("loop", 0), ("loop", 1), ("reduce", 0), ("reduce", 1)):
            bufs, _ = _run(w, ("fp8_" if fp8 else "") + kernel, schedule=schedule)
            got = bufs.out.float().cpu()
            assert (got[~live] == 0).all()
            torch.testing.assert_close(got[live], ref32[live], atol=ATOL, rtol=RTOL,
                                       msg=lambda m: f"fp8={fp8} {kernel} schedule {schedule}: {m}")


def test_exhausted_spin_limit_is_reported(oracle):
    """A wavefront of a persistent kernel that gives up waiting for its work-group sets a status word
    and lets the grid drain; the timed call returns FA_ERR_RUNTIME.  A negative options->spin_limit
    makes every wait give up at once (the merges go ahead without waiting, so every kernel still ends
    normally): the very first call reports.  An asynchronous call cannot look; its caller asks
    fa_paged_attention_kernel_status at a synchronisation point of its own."""
    from flash_attention_factory_amd import _cabi
    w = W.make_config(1, num_seqs=4, pool_blocks=512)
    for kernel in ("loop", "reduce"):
        with pytest.raises(_cabi.PagedAttentionError, match="gave up waiting") as e:
            _run(w, kernel, spin_limit=-1)
        assert e.value.code == _cabi.FA_ERR_RUNTIME
        _cabi.kernel_status()  # the word was cleared with the report
        _run(w, kernel, spin_limit=-1, timed=False)  # asynchronous: nothing is raised here ...
        with pytest.raises(_cabi.PagedAttentionError, match="gave up waiting"):
            _cabi.kernel_status(clear=False)  # ... the caller finds out when it asks
        with pytest.raises(_cabi.PagedAttentionError, match="gave up waiting"):
            _cabi.kernel_status(clear=True)
        _cabi.kernel_status()
    for kernel in ("loop", "reduce"):
        bufs, _ = _run(w, kernel)
        _check(bufs.out, w, oracle, f"{w.name}/{kernel} after the report")


@pytest.mark.parametrize("heads", [(32, 4), (40, 8), (8, 8), (6, 2), (9, 3)], ids=lambda h: f"h{h[0]}x{h[1]}")
@pytest.mark.parametrize("block_size", [16, 64])
def test_fp8_head_size_64_pairs_of_kv_heads(oracle, heads, block_size):
    """FP8 caches with 64-byte token rows in upstream's token-major layout: two adjacent kv heads share
    every cache line and run as one 128-byte row (several pairs per sequence, groups up to 8, an odd
    number of kv heads that cannot pair, the head-major layout where heads are not adjacent) -- loop
    and split, persistent and grid forms, scratch contents per partition under the grid form."""
    nheads, nheads_k = heads
    for layout in (W.TOKEN_MAJOR, W.HEAD_MAJOR):
        w = W.make_test_shaped(batch_size=5, nheads=nheads, nheads_k=nheads_k, d=64, seqlen_k=900, varlen=False,
                               has_sinks=False, fp8=True, block_size=block_size, layout=layout, seed=nheads)
        w.context_lens = torch.tensor([900, 1, 257, 0, 640], dtype=torch.int32)
        w.sinks = torch.linspace(-2, 2, nheads).to(w.query.dtype)
        live = w.context_lens > 0
        for kernel in ("fp8_loop", "fp8_reduce"):
            for schedule in (0, 1):
                bufs, _ = _run(w, kernel, schedule=schedule)
                assert (bufs.out.cpu()[~live] == 0).all()
                _check(bufs.out, w, oracle, f"{w.name}/{layout}/{kernel}/schedule{schedule}")
                if kernel == "fp8_reduce" and schedule == 1:
                    es, ml, tmp = call_oracle(oracle.kernel_partition, w, partition_size=w.partition_size,
                                              max_num_partitions=w.max_num_partitions)
                    for s in range(w.num_seqs):
                        n = math.ceil(int(w.context_lens[s]) / w.partition_size)
                        torch.testing.assert_close(bufs.max_logits[s, :, :n].cpu(), ml[s, :, :n], atol=1e-4, rtol=1e-5)
                        torch.testing.assert_close(bufs.exp_sums[s, :, :n].cpu(), es[s, :, :n], atol=1e-4, rtol=1e-4)
                        torch.testing.assert_close(bufs.tmp_out[s, :, :n].cpu(), tmp[s, :, :n], atol=2e-3, rtol=1e-2)
                        assert torch.isnan(bufs.tmp_out[s, :, n:]).all()
