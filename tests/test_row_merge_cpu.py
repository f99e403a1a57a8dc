"""fa_paged_attention_loop_workspace_bytes and the checks of the workspace that goes with the options
(validate_only launches nothing, so no GPU is needed)."""
import ctypes

import pytest

from flash_attention_factory_amd import _cabi


def _call(seqs=3, kv_heads=8, group=4, d=128, blocks=256, block=16, **opts):
    sh, op = _cabi.Shape(), _cabi.Options()
    sh.num_seqs, sh.num_heads, sh.num_kv_heads, sh.head_size = seqs, kv_heads * group, kv_heads, d
    sh.block_size, sh.max_blocks_per_seq, sh.max_num_partitions = block, blocks, 1
    sh.kv_block_stride, sh.kv_token_stride, sh.kv_head_stride = block * kv_heads * d, d, block * d
    sh.num_pool_blocks = 4096
    for k, v in opts.items():
        setattr(op, k, v)
    return sh, op


def _bytes(fp8=0, **kw):
    sh, op = _call(**kw)
    return _cabi.load().fa_paged_attention_loop_workspace_bytes(ctypes.byref(sh), ctypes.byref(op), fp8)


def test_who_asks_for_workspace():
    assert _bytes() > 0
    assert _bytes(seqs=48) > 0 and _bytes(seqs=49) == 0              # 384 rows, 392
    assert _bytes(blocks=80) == 0 and _bytes(blocks=81) > 0          # 1280 keys stay whole
    assert _bytes(fp8=1, blocks=160) == 0 and _bytes(fp8=1, blocks=161) > 0
    assert _bytes(schedule=_cabi.FA_SCHEDULE_GRID) == 0
    assert _bytes(query_len=4) > 0 and _bytes(query_len=5) == 0      # 16 columns, 20
    assert _bytes(mask_flags=_cabi.FA_MASK_WINDOW, window_left=1000) == 0
    assert _bytes(mask_flags=_cabi.FA_MASK_WINDOW, window_left=2000) > 0
    assert _bytes(d=96) == 0                                         # not a valid call
    assert _bytes() <= 16 << 20


@pytest.mark.parametrize("fp8", [0, 1])
def test_argument_checks(fp8):
    L = _cabi.load()
    sh, _ = _call(blocks=1024)
    need = _bytes(fp8=fp8, blocks=1024)
    full = _cabi.OptionsWorkspace()
    assert ctypes.sizeof(full) == full.struct_size == 120 and _cabi.OptionsWorkspace.workspace.offset == 104
    full.validate_only = 1
    room = (ctypes.c_char * 64)()
    p = (ctypes.addressof(room) + 15) // 16 * 16
    entry = L.fa_paged_attention_fp8_loop if fp8 else L.fa_paged_attention_loop

    def call(space, size):
        full.workspace, full.workspace_bytes = space, size
        return entry(p, p, p, p, p, p, 1.0, 0, ctypes.byref(sh), ctypes.byref(full))

    assert call(p, need) == _cabi.FA_OK
    assert call(None, 0) == _cabi.FA_OK
    assert call(p, need - 1) == _cabi.FA_ERR_SCRATCH_TOO_SMALL and b"asks for" in L.fa_last_error()
    assert call(p + 8, need) == _cabi.FA_ERR_BAD_SHAPE
    full.struct_size = 112  # half of the workspace's fields
    assert call(p, need) == _cabi.FA_ERR_BAD_SHAPE and b"options.struct_size" in L.fa_last_error()


@pytest.mark.parametrize("fp8, blocks, refused", [
    # 16-bit rows of head size 64 ask from 1025 keys on, byte caches from 1537; up to 2560 and 5120 they do without
    (0, 64, False), (0, 65, False), (0, 160, False), (0, 161, True),
    (1, 96, False), (1, 97, False), (1, 320, False), (1, 321, True),
])
def test_short_rows_of_head_size_64_take_any_workspace(fp8, blocks, refused):
    L = _cabi.load()
    sh, _ = _call(d=64, blocks=blocks)
    full = _cabi.OptionsWorkspace()
    need = L.fa_paged_attention_loop_workspace_bytes(ctypes.byref(sh), ctypes.byref(_cabi.Options()), fp8)
    assert (need > 0) == (blocks not in (64, 96))
    full.validate_only = 1
    room = (ctypes.c_char * 64)()
    p = (ctypes.addressof(room) + 15) // 16 * 16
    entry = L.fa_paged_attention_fp8_loop if fp8 else L.fa_paged_attention_loop
    for size in (0, 16, max(need - 1, 0)):
        full.workspace, full.workspace_bytes = p, size
        want = _cabi.FA_ERR_SCRATCH_TOO_SMALL if refused else _cabi.FA_OK
        assert entry(p, p, p, p, p, p, 1.0, 0, ctypes.byref(sh), ctypes.byref(full)) == want, size


def test_calls_that_need_not_ask():
    """What lib.*.run rules out without asking, the library answers with 0; the shortest tables for which it asks get some."""
    asked, least = 0, {64: 1 << 40, 128: 1 << 40}
    for fp8, element in ((0, 2), (1, 1)):
        for d in (64, 128):
            for kv_heads in (1, 2, 3, 8, 32):
                for seqs in (1, 12, 24, 25, 48, 49, 96, 97, 128, 129, 384, 385):
                    for blocks in (20, 40, 41, 64, 65, 79, 80, 81, 96, 97, 160, 161, 320, 321, 4096):
                        sh, op = _call(seqs=seqs, kv_heads=kv_heads, group=1, d=d, blocks=blocks)
                        sh.kv_token_stride, sh.kv_head_stride = kv_heads * d, d   # kv heads side by side, as pairs need
                        need = _cabi.load().fa_paged_attention_loop_workspace_bytes(ctypes.byref(sh), ctypes.byref(op), fp8)
                        ruled_out = (seqs > _cabi.LOOP_WORKSPACE_MAX_SEQS or seqs * kv_heads > _cabi.LOOP_WORKSPACE_MAX_ROWS or
                                     blocks * 16 * 2 * d * element <= _cabi.LOOP_WORKSPACE_MIN_HEAD_BYTES[d])
                        assert not (ruled_out and need), (fp8, d, kv_heads, seqs, blocks)
                        asked += need > 0
                        if need:
                            least[d] = min(least[d], (blocks - 1) * 16 * 2 * d * element)
    assert asked > 100 and least == _cabi.LOOP_WORKSPACE_MIN_HEAD_BYTES
