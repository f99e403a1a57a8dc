"""Loop path with workspace: rows cut into pieces that several work-groups take, merged inside the launch
(csrc/paged_attention_row_merge.h), against the CPU oracle at the sizes where it can go wrong: rows around the
length from which they are cut, more pieces than a wavefront has lanes, every number of MFMA columns, empty rows,
windows, sinks, several query tokens; workspace of any contents; replays of a HIP graph; two streams at once.

Tolerance: results are rounded to fp16 / bf16 (2^-11, 2^-8 of the value) from probabilities rounded to the same
type before P.V; 1e-2 of the largest value, as in the repository's other comparisons with the oracle."""
import ctypes

import pytest
import torch

from flash_attention_factory_amd import _cabi, runner, workloads as W
from flash_attention_factory_amd.lib import paged_attention_fp8_loop, paged_attention_loop

pytestmark = pytest.mark.gpu


def _workload(lens, hk, group, d, fp8=None, block=16, bf16=False, sinks=False, seed=0):
    w = W.make_test_shaped(batch_size=len(lens), nheads=hk * group, nheads_k=hk, d=d, seqlen_k=max(lens), varlen=False,
                           has_sinks=sinks, fp8=fp8 is not None, block_size=block, seed=seed,
                           dtype=torch.bfloat16 if bf16 else torch.float16, layout=W.HEAD_MAJOR if bf16 else W.TOKEN_MAJOR,
                           **({"fp8_dtype": fp8} if fp8 is not None else {}))
    w.context_lens.copy_(torch.tensor(lens, dtype=torch.int32))
    return w


def _run(w, dev, query=None, out=None, **kw):
    wd = w.to(dev)
    q = wd.query if query is None else query.to(dev)
    out = torch.full_like(q, 7.0) if out is None else out
    head = (None, None, None, out, None, q, runner.logical_cache_view(wd, wd.key_cache),
            runner.logical_cache_view(wd, wd.value_cache), wd.block_tables, wd.context_lens,
            w.num_heads // w.num_kv_heads, w.scale)
    tail = (w.block_size, 0, kw.pop("alibi", None), wd.sinks, kw.pop("softcap", 0.0))
    if w.is_fp8:
        paged_attention_fp8_loop.run(*head, w.fp8_scale, *tail, timed=False, **kw)
    else:
        paged_attention_loop.run(*head, *tail, timed=False, **kw)
    return out


def _needs(w, query_len=1):
    """Bytes the call asks for: > 0 says that it takes the path under test."""
    sh, op = _cabi.Shape(), _cabi.Options()
    sh.num_seqs, sh.num_heads, sh.head_size = w.query.shape[0], w.num_heads, w.query.shape[-1]
    sh.num_kv_heads, sh.block_size, sh.max_blocks_per_seq = w.num_kv_heads, w.block_size, w.block_tables.shape[1]
    sh.max_num_partitions, sh.num_pool_blocks = 1, w.key_cache.shape[0]
    sh.kv_block_stride, sh.kv_token_stride, sh.kv_head_stride = w.kv_strides()
    sh.q_dtype = _cabi.FA_DTYPE_BF16 if w.query.dtype == torch.bfloat16 else _cabi.FA_DTYPE_F16
    op.query_len = query_len
    return _cabi.load().fa_paged_attention_loop_workspace_bytes(ctypes.byref(sh), ctypes.byref(op), int(w.is_fp8))


def _check(oracle, w, out, **kw):
    query = kw.pop("query", w.query)
    ref = oracle.attention_ref(query, w.key_cache, w.value_cache, w.block_tables, w.context_lens, scale=w.scale,
                               block_size=w.block_size, kv_strides=w.kv_strides(), num_kv_heads=w.num_kv_heads, sinks=w.sinks,
                               fp8_scale=w.fp8_scale, want_f32=True, **kw)[1]
    live = w.context_lens > 0
    unit = ref[live].abs().max()
    torch.testing.assert_close(out.float().cpu()[live] / unit, ref[live] / unit, atol=1e-2, rtol=1e-2)
    assert (out.cpu()[~live] == 7.0).all(), "rows without keys are not written"


E5M2, E4M3 = torch.float8_e5m2, torch.float8_e4m3fn


@pytest.mark.parametrize("lens, hk, group, d, fp8, block, bf16", [
    # 5 partitions of 256 keys stay whole; one key more, and rows beside it that do
    ([1281, 1280, 1, 0, 257], 2, 4, 128, None, 16, False),
    ([1536, 1537, 511, 512, 513], 1, 1, 128, None, 64, True),
    # more pieces than lanes; an empty row between
    ([50001, 0, 700], 1, 2, 128, None, 16, True),
    # 16-bit rows of 128 bytes, byte rows of 128 and of 64 bytes (partitions of 256, 512 and 512 keys)
    ([1025, 1024, 0, 300], 2, 4, 64, None, 16, True),
    ([1537, 1536, 40], 3, 2, 64, E5M2, 16, False),
    ([5000, 2561, 2560], 4, 3, 64, None, 32, False),
    ([5121, 2559, 9000], 2, 5, 128, E5M2, 16, False),
    ([2700, 6001], 2, 16, 128, E4M3, 16, True),
    # kv heads in pairs (byte rows of 64 bytes that lie next to each other)
    ([9001, 5121, 40], 2, 4, 64, E5M2, 64, False),
    ([7000, 100], 3, 7, 64, E4M3, 32, True),
    # many short rows and one long
    ([300] * 7 + [12000], 2, 8, 128, None, 16, False),
])
@pytest.mark.parametrize("sinks", [False, True])
def test_against_the_oracle(oracle, lens, hk, group, d, fp8, block, bf16, sinks):
    w = _workload(lens, hk, group, d, fp8, block, bf16, sinks)
    assert _needs(w) > 0
    dev = torch.device("cuda:0")
    out = _run(w, dev)
    again = _run(w, dev)
    torch.cuda.synchronize()
    assert torch.equal(out, again), "the order of arrival shows in the result"
    _check(oracle, w, out)


@pytest.mark.parametrize("window", [0, 1300, 2048, 100000])
@pytest.mark.parametrize("query_len, group", [(1, 4), (3, 4), (2, 8)])
def test_windows_modifiers_and_query_tokens(oracle, window, query_len, group):
    w = _workload([4100, 1500, 2817, 5], 2, group, 128, sinks=True)
    dev = torch.device("cuda:0")
    H = 2 * group
    g = torch.Generator().manual_seed(3)
    query = torch.randn((4, query_len, H, 128), generator=g).to(torch.float16) if query_len > 1 else w.query
    alibi = torch.linspace(0.001, 0.01, H)
    assert _needs(w, query_len) > 0
    out = _run(w, dev, query=query, alibi=alibi.to(dev), softcap=20.0, apply_alibi=True, apply_softcap=True, window_left=window)
    torch.cuda.synchronize()
    _check(oracle, w, out, query=query, alibi_slopes=alibi, softcap=20.0, window_left=window)


@pytest.mark.parametrize("longest, fp8", [(2560, None), (5120, E5M2)])
def test_too_little_workspace_for_short_rows_of_head_size_64(oracle, longest, fp8):
    """Taken, left alone, and the rows stay whole."""
    w = _workload([longest, 900, 0], 3, 4, 64, fp8)
    dev = torch.device("cuda:0")
    assert _needs(w) > 256
    space = torch.full((256,), 0x5A, dtype=torch.uint8, device=dev)
    wd = w.to(dev)
    L, sh, op = _cabi.load(), _cabi.Shape(), _cabi.OptionsWorkspace()
    op.workspace, op.workspace_bytes = space.data_ptr(), 256
    sh.num_seqs, sh.num_heads, sh.head_size, sh.num_kv_heads = 3, 12, 64, 3
    sh.block_size, sh.max_blocks_per_seq, sh.max_num_partitions = w.block_size, w.block_tables.shape[1], 1
    sh.kv_block_stride, sh.kv_token_stride, sh.kv_head_stride = w.kv_strides()
    sh.num_pool_blocks, sh.q_dtype = w.key_cache.shape[0], _cabi.FA_DTYPE_F16
    op.fp8_scale, op.stream, op.kv_fp8_format = 1.0, torch.cuda.current_stream().cuda_stream, _cabi.FA_FP8_E5M2
    out = torch.full_like(wd.query, 7.0)
    fn = L.fa_paged_attention_fp8_loop if fp8 else L.fa_paged_attention_loop
    _cabi.check(fn(out.data_ptr(), wd.query.data_ptr(), wd.key_cache.data_ptr(), wd.value_cache.data_ptr(), wd.block_tables.data_ptr(),
                   wd.context_lens.data_ptr(), w.scale, 0, ctypes.byref(sh), ctypes.byref(op)))
    torch.cuda.synchronize()
    assert (space == 0x5A).all()
    _check(oracle, w, out)


@pytest.mark.parametrize("fill", [0x00, 0xFF, 0x7F])
def test_contents_of_the_workspace_do_not_matter(oracle, fill):
    """Through the C ABI, twice on the same memory, without clearing it in between."""
    w = _workload([6000, 1400, 3000], 2, 4, 128)
    dev = torch.device("cuda:0")
    need = _needs(w)
    space = torch.full((need,), fill, dtype=torch.uint8, device=dev)
    wd = w.to(dev)
    L, sh, op = _cabi.load(), _cabi.Shape(), _cabi.OptionsWorkspace()
    op.workspace, op.workspace_bytes = space.data_ptr(), need
    sh.num_seqs, sh.num_heads, sh.head_size, sh.num_kv_heads = 3, 8, 128, 2
    sh.block_size, sh.max_blocks_per_seq, sh.max_num_partitions = w.block_size, w.block_tables.shape[1], 1
    sh.kv_block_stride, sh.kv_token_stride, sh.kv_head_stride = w.kv_strides()
    sh.num_pool_blocks, sh.q_dtype = w.key_cache.shape[0], _cabi.FA_DTYPE_F16
    op.stream = torch.cuda.current_stream().cuda_stream
    outs = []
    for _ in range(2):
        out = torch.full_like(wd.query, 7.0)
        _cabi.check(L.fa_paged_attention_loop(
            out.data_ptr(), wd.query.data_ptr(), wd.key_cache.data_ptr(), wd.value_cache.data_ptr(), wd.block_tables.data_ptr(),
            wd.context_lens.data_ptr(), w.scale, 0, ctypes.byref(sh), ctypes.byref(op)))
        outs.append(out)
    torch.cuda.synchronize()
    assert torch.equal(*outs)
    _check(oracle, w, outs[0])


def test_graph_replays_and_overlapping_streams(oracle):
    from flash_attention_factory_amd import torch_ops  # noqa: F401
    dev = torch.device("cuda:0")
    w = _workload([6000, 1400, 3000], 4, 4, 128)
    wd = w.to(dev)
    query, lens, out = wd.query.clone(), wd.context_lens.clone(), torch.zeros_like(wd.query)

    def op(o, q, n):
        torch.ops.fa_amd.paged_attention_loop(o, q, wd.key_cache, wd.value_cache, wd.block_tables, n, w.scale)

    eager = torch.zeros_like(out)
    op(eager, query, lens)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        op(out, query, lens)
        op(out, query, lens)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for it in range(4):
        query.copy_(torch.randn_like(query))
        lens.copy_(torch.tensor([6000 - 977 * it, 1400 + 700 * it, 3000 - it], dtype=torch.int32))
        op(eager, query, lens)
        out.zero_()
        torch.randn(1 << 20, device=dev).sum()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), f"replay {it}"
        others = [torch.zeros_like(out) for _ in range(8)]
        torch.cuda.synchronize()
        for k, o in enumerate(others):
            with torch.cuda.stream(streams[k & 1]):
                op(o, query, lens)
        torch.cuda.synchronize()
        assert all(torch.equal(o, eager) for o in others), f"streams {it}"


def test_a_call_that_asks_for_none_leaves_the_workspace_alone(oracle):
    """130 sequences ask for no workspace and run as sub-batches of 65, a number that would ask for some: whatever
    workspace comes with the call, of any size, is not touched.  (The memory behind it is this test's own: 8 MB, more
    than the 2.7 MB that 65 sequences would ask for.)"""
    lens = [1700, 40] * 65
    w = _workload(lens, 2, 2, 128)
    wide = torch.zeros((130, 256), dtype=torch.int32)
    wide[:, :w.block_tables.shape[1]] = w.block_tables
    w.block_tables = wide
    assert _needs(w) == 0
    whole, w.query = w.query, w.query[:65]
    assert _needs(w) > 0
    w.query = whole
    dev = torch.device("cuda:0")
    wd = w.to(dev)
    memory = torch.full((8 << 20,), 0x5A, dtype=torch.uint8, device=dev)
    L, sh, op = _cabi.load(), _cabi.Shape(), _cabi.OptionsWorkspace()
    op.workspace, op.workspace_bytes = memory.data_ptr(), 16
    sh.num_seqs, sh.num_heads, sh.head_size, sh.num_kv_heads = 130, 4, 128, 2
    sh.block_size, sh.max_blocks_per_seq, sh.max_num_partitions = w.block_size, 256, 1
    sh.kv_block_stride, sh.kv_token_stride, sh.kv_head_stride = w.kv_strides()
    sh.num_pool_blocks, sh.q_dtype = w.key_cache.shape[0], _cabi.FA_DTYPE_F16
    op.stream = torch.cuda.current_stream().cuda_stream
    out = torch.full_like(wd.query, 7.0)
    _cabi.check(L.fa_paged_attention_loop(
        out.data_ptr(), wd.query.data_ptr(), wd.key_cache.data_ptr(), wd.value_cache.data_ptr(), wd.block_tables.data_ptr(),
        wd.context_lens.data_ptr(), w.scale, 0, ctypes.byref(sh), ctypes.byref(op)))
    torch.cuda.synchronize()
    assert (memory == 0x5A).all()
    _check(oracle, w, out)


@pytest.mark.parametrize("query_len", [2, 3])
@pytest.mark.parametrize("hk", [2, 12])
@pytest.mark.parametrize("fp8", [None, E5M2])
def test_the_widest_window_is_none(oracle, hk, query_len, fp8):
    """window_left = 2^31 - 1 masks nothing: the bits of the call without a window, also where a context is shorter
    than the query tokens."""
    w = _workload([4100, 1500, 2817, 2], hk, 4, 128, fp8)
    dev = torch.device("cuda:0")
    query = torch.randn((4, query_len, 4 * hk, 128), generator=torch.Generator().manual_seed(4)).to(torch.float16)
    assert _needs(w, query_len) > 0
    out = _run(w, dev, query=query, window_left=2**31 - 1)
    without = _run(w, dev, query=query)
    torch.cuda.synchronize()
    assert torch.equal(out, without)
    _check(oracle, w, out, query=query)


@pytest.mark.parametrize("lens, hk, group, d, fp8, kw", [
    ([200, 900, 5, 0, 1280], 2, 4, 128, None, {}),
    ([300, 1, 64] * 33 + [0], 2, 1, 64, None, {}),             # more than 64 sequences
    ([2560, 7, 700], 8, 4, 128, E5M2, {}),
    ([1500] * 20, 8, 1, 128, None, {}),                        # long enough for cuts, not worth them
    ([2700] * 40, 8, 2, 128, E4M3, {}),                        # the same with more rows than units
    ([1500] * 20, 8, 1, 128, None, dict(softcap=20.0, apply_softcap=True)),
    ([2700, 3000] * 20, 8, 1, 128, E5M2, dict(window_left=2600)),
], ids=str)
def test_rows_that_stay_whole_are_the_persistent_loop_kernels(oracle, monkeypatch, lens, hk, group, d, fp8, kw):
    """Given workspace, rows that the device does not cut give the bits of the call without workspace."""
    w = _workload(lens, hk, group, d, fp8)
    wide = torch.zeros((len(lens), 4096), dtype=torch.int32)
    wide[:, :w.block_tables.shape[1]] = w.block_tables
    w.block_tables = wide
    assert _needs(w) > 0
    dev = torch.device("cuda:0")
    out = _run(w, dev, **dict(kw))
    monkeypatch.setattr(_cabi.load(), "fa_paged_attention_loop_workspace_bytes", lambda *args: 0)
    without = _run(w, dev, **dict(kw))
    torch.cuda.synchronize()
    assert torch.equal(out, without)
    _check(oracle, w, out, **{k: v for k, v in kw.items() if not k.startswith("apply")})


def test_a_full_gpu_leaves_rows_whole(oracle):
    """No memory for the workspace (PyTorch's allocator is held to what it has): the call runs without."""
    from flash_attention_factory_amd import torch_ops  # noqa: F401
    w = _workload([6000, 1400, 3000], 2, 4, 128)
    need = _needs(w)
    dev = torch.device("cuda:0")
    wd = w.to(dev)
    outs = [torch.full_like(wd.query, 7.0) for _ in range(2)]
    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction(1e-9)
    held = []
    try:
        for size in (need, need // 8, need // 64):  # what the allocator has left in blocks of its own
            try:
                while True:
                    held.append(torch.empty(size, dtype=torch.uint8, device=dev))
            except torch.OutOfMemoryError:
                pass
        with pytest.raises(torch.OutOfMemoryError):
            torch.empty(need, dtype=torch.uint8, device=dev)
        _run(wd, dev, out=outs[0])
        torch.ops.fa_amd.paged_attention_loop(outs[1], wd.query, wd.key_cache, wd.value_cache, wd.block_tables, wd.context_lens, w.scale)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
        held.clear()
    torch.cuda.synchronize()
    for out in outs:
        _check(oracle, w, out)


@pytest.mark.parametrize("fp8, d, lens, query_len, window", [
    (E5M2, 128, [6000, 2561, 9001, 30], 1, None),
    (E4M3, 128, [5121, 700, 2600], 2, None),
    (E5M2, 128, [9000, 4000, 41], 1, 3000),
    (E4M3, 64, [5200, 11000, 9], 1, None),
    (E5M2, 64, [12001, 5121], 3, 7000),
])
@pytest.mark.parametrize("per_block", [False, True], ids=["head", "block"])
def test_scales_of_byte_caches_in_cut_rows(oracle, per_block, fp8, d, lens, query_len, window):
    w = _workload(lens, 2, 4, d, fp8, 16, sinks=True)
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(9)
    shape = (w.key_cache.shape[0], 2) if per_block else (2,)
    ks, vs = (torch.exp2(4.0 * torch.rand(shape, generator=g) - 2.0) for _ in range(2))  # 1/4 .. 4
    query = torch.randn((len(lens), query_len, 8, d), generator=g).to(torch.float16) if query_len > 1 else w.query
    assert _needs(w, query_len) > 0
    kw = dict(window_left=window) if window else {}
    out = _run(w, dev, query=query, k_scales=ks.to(dev), v_scales=vs.to(dev), **kw)
    torch.cuda.synchronize()
    _check(oracle, w, out, query=query, k_scales=ks, v_scales=vs, **kw)


def test_calls_go_to_the_current_stream():
    from flash_attention_factory_amd.lib import _run as body
    dev = torch.device("cuda:0")
    w = _workload([6000, 40], 1, 2, 128)
    wd = w.to(dev)
    for stream in (torch.cuda.current_stream(), torch.cuda.Stream(), torch.cuda.Stream()):
        with torch.cuda.stream(stream):
            assert body.current_stream(dev) == stream.cuda_stream == torch.cuda.current_stream().cuda_stream
            out = _run(wd, dev)
            again = torch.empty_like(out).copy_(out)  # ordered behind the call on its stream only
        stream.synchronize()
        assert torch.equal(out, again) and torch.isfinite(again.float()).all()


@pytest.mark.parametrize("lens, hk, group, fp8", [
    ([32768, 300], 1, 4, None),        # 128 partitions in the longest row: a partition a piece
    ([32769, 300], 1, 4, None),        # 129: two
    ([16384, 16128], 2, 2, None),      # 254 pieces of one partition for 256 units
    ([16384, 16385], 2, 2, None),      # 258 would be: two partitions a piece
    ([7000, 0, 513, 4097, 1], 8, 8, E5M2),  # 26 partitions x 8 kv heads, eight wavefronts a work-group
    ([3000] * 9, 4, 1, None),          # 432 partitions, one head a kv head: two partitions a piece
])
def test_pieces_of_one_partition(oracle, lens, hk, group, fp8):
    """Results on both sides of the rule by which a piece is one partition or two (test_the_pieces_are_the_rules looks at the
    pieces), from memory that held another batch's flags."""
    w = _workload(lens, hk, group, 128, fp8, bf16=True, sinks=True)
    assert _needs(w) > 0
    dev = torch.device("cuda:0")
    out, again = _run(w, dev), _run(w, dev)
    torch.cuda.synchronize()
    assert torch.equal(out, again), "the order of arrival shows in the result"
    _check(oracle, w, out)


@pytest.mark.parametrize("lens, hk, group, d, fp8, m, window", [
    # m: partitions a piece; 0: rows stay whole; None: cut, the length follows from the launch's work-groups.  Rows on both sides of
    # what stays whole: five partitions of 256 keys, of 512 in byte caches, also of pairs of kv heads of 64 ...
    ([1280, 300], 2, 4, 128, None, 0, None),
    ([1281, 300], 2, 4, 128, None, 1, None),
    ([2560, 300], 3, 4, 128, E5M2, 0, None),
    ([2561, 300], 3, 4, 128, E5M2, 1, None),
    ([2560, 300], 2, 4, 64, E5M2, 0, None),
    ([2561, 300], 2, 4, 64, E5M2, 1, None),
    # ... four of 256 keys with head size 64, three of 512
    ([1024, 300], 2, 4, 64, None, 0, None),
    ([1025, 300], 2, 4, 64, None, 1, None),
    ([1536, 300], 3, 4, 64, E5M2, 0, None),
    ([1537, 300], 3, 4, 64, E4M3, 1, None),
    # behind a window the keys that are seen count
    ([5000, 300], 2, 4, 64, None, 0, 1023),
    ([5000, 300], 2, 4, 64, None, 1, 1024),
    # the longest row against the others: up to half the units, beyond, more rows than units
    ([1497] * 16, 8, 1, 64, None, None, None),
    ([1497] * 43, 3, 1, 64, None, 0, None),
    ([400 + 1200 * k // 39 for k in range(40)], 8, 1, 64, None, 0, None),
    ([2555] + [700] * 41, 8, 1, 64, None, None, None),
    # a partition a piece or two: partitions x columns up to 512 and beyond, pieces for 256 units and more
    ([32768, 300], 1, 4, 128, None, 1, None),
    ([32769, 300], 1, 4, 128, None, 2, None),
    ([16384, 16128], 2, 2, 128, None, 1, None),
    ([16384, 16385], 2, 2, 128, None, 2, None),
    ([8192, 300], 1, 16, 64, None, 1, None),
    ([8193, 300], 1, 16, 64, None, 2, None),
    # partitions x columns beyond 2048: 256 KiB a piece
    ([32768, 300], 1, 16, 64, None, 2, None),
    ([32769, 300], 1, 16, 64, None, 4, None),
    ([65537, 300], 1, 16, 64, E5M2, 4, None),
    ([65536, 300], 1, 16, 64, E5M2, 2, None),
])
def test_the_pieces_are_the_rules(oracle, lens, hk, group, d, fp8, m, window):
    """The slots of the workspace that a call has written are those of the pieces that the rule gives, in a block table that
    does not tell how long the rows are."""
    dev = torch.device("cuda:0")
    units = torch.cuda.get_device_properties(dev).multi_processor_count
    if units != 256:
        pytest.skip("the batches are made for 256 compute units")
    w = _workload(lens, hk, group, d, fp8)
    wide = torch.zeros((len(lens), max(512, w.block_tables.shape[1])), dtype=torch.int32)
    wide[:, :w.block_tables.shape[1]] = w.block_tables
    w.block_tables = wide
    S, H, fill = len(lens), hk * group, 0x5A5A5A5A
    need = _needs(w)
    assert need > 0
    wd = w.to(dev)
    space = torch.full((need // 4,), fill, dtype=torch.int32, device=dev)
    sh, op = _cabi.Shape(), _cabi.OptionsWorkspace()
    op.workspace, op.workspace_bytes = space.data_ptr(), need
    sh.num_seqs, sh.num_heads, sh.head_size, sh.num_kv_heads = S, H, d, hk
    sh.block_size, sh.max_blocks_per_seq, sh.max_num_partitions = w.block_size, wide.shape[1], 1
    sh.kv_block_stride, sh.kv_token_stride, sh.kv_head_stride = w.kv_strides()
    sh.num_pool_blocks, sh.q_dtype = w.key_cache.shape[0], _cabi.FA_DTYPE_F16
    op.fp8_scale, op.stream = 1.0, torch.cuda.current_stream().cuda_stream
    op.kv_fp8_format = _cabi.FA_FP8_E4M3 if fp8 is E4M3 else _cabi.FA_FP8_E5M2
    if window is not None:
        op.mask_flags, op.window_left = _cabi.FA_MASK_WINDOW, window
    out = torch.full_like(wd.query, 7.0)
    fn = _cabi.load().fa_paged_attention_fp8_loop if fp8 else _cabi.load().fa_paged_attention_loop
    _cabi.check(fn(out.data_ptr(), wd.query.data_ptr(), wd.key_cache.data_ptr(), wd.value_cache.data_ptr(), wd.block_tables.data_ptr(),
                   wd.context_lens.data_ptr(), w.scale, 0, ctypes.byref(sh), ctypes.byref(op)))
    torch.cuda.synchronize()
    _check(oracle, w, out, **({} if window is None else dict(window_left=window)))
    # where the pieces lie: flags for (1024 + rows) pieces x slices, then the slots
    pairs = fp8 is not None and d == 64 and hk % 2 == 0 and 2 * group <= 16 and window is None  # (token-major pools)
    heads, cols, head = (hk // 2, 2 * group, 128) if pairs else (hk, group, d)
    rows = S * heads
    most = 8 if head == 128 else 4                                          # slices that the workspace has room for
    slices = 8 if head == 128 and window is None and 2 * rows <= units else 4  # and the launch uses: its wavefronts
    slot = slices * ((cols * (head // slices + 2) + 3) & ~3)
    slots = space[2 * (1024 + rows) * most:].cpu()
    written = {k for k in range(min(1024 + rows, slots.numel() // slot)) if (slots[k * slot:(k + 1) * slot] != fill).any()}
    if not m:
        assert bool(written) == (m is None), len(written)
        return
    psize = (64 if head == 64 else 128) * 1024 // (2 * head * (1 if fp8 else 2))
    want, before = set(), 0
    base = [0 if window is None else max(0, n - 1 - window) // psize * psize for n in lens]
    full = [(n - b) // (m * psize) for n, b in zip(lens, base)]
    for s, n in enumerate(lens):
        tail = (n - base[s]) % (m * psize) > 0
        if full[s] + tail > 1:  # (a row of a single piece leaves nothing)
            want |= {(before + j) * heads + h for j in range(full[s]) for h in range(heads)}
            want |= {(sum(full) + s) * heads + h for h in range(heads) if tail}
        before += full[s]
    assert written == want, (sorted(written), sorted(want))
