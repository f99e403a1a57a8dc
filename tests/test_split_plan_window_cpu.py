"""A split call with a local window is measured by the keys its query token sees, not by its rows: where they are few
the call is the single-pass kernel (fa_paged_attention_reduce_plan, without a GPU)."""
import pytest

from flash_attention_factory_amd import _cabi
from test_split_plan_cpu import L, LOOP, SEGMENT, _plan  # noqa: F401

WINDOW = _cabi.FA_MASK_WINDOW


@pytest.mark.parametrize("window, seqs, want", [
    (1023, 4, LOOP), (1024, 4, SEGMENT),      # 1024 keys, 1025
    (2047, 32, LOOP), (2048, 32, SEGMENT),    # a row for every compute unit
    (2047, 31, SEGMENT), (0, 1, LOOP)])
def test_form_by_visible_keys(L, window, seqs, want):  # noqa: F811
    args = dict(S=seqs, H=32, Hk=8, D=128, B=16, ctx_bound=20000, mask_flags=WINDOW, window_left=window)
    assert _plan(L, **args) == want
    # rows that the scratch arrays may not hold stay with the split kernels, which cut them to that
    assert _plan(L, NP=3, **args) == SEGMENT
    # several query tokens, and a window that is not asked for: by the rows
    assert _plan(L, query_len=2, **args) == SEGMENT
    assert _plan(L, **dict(args, mask_flags=0)) == SEGMENT
    assert _plan(L, schedule=_cabi.FA_SCHEDULE_SPLIT, **args) == SEGMENT


@pytest.mark.parametrize("fp8, window, seqs, longest, want", [
    # 16-bit, heads of 128: 512 bytes a key
    (False, 767, 1, 1100, LOOP), (False, 768, 1, 1100, SEGMENT),
    (False, 1023, 15, 3000, SEGMENT), (False, 1023, 16, 3000, LOOP),        # half a row per unit
    (False, 1023, 4, 12784, SEGMENT), (False, 1023, 4, 12800, LOOP),        # 1600 keys per unit
    (False, 2047, 32, 6128, SEGMENT), (False, 2047, 32, 6144, LOOP),        # a third of a row
    (False, 2047, 64, 3000, LOOP), (False, 1500, 31, 9000, SEGMENT),
    # byte caches
    (True, 1023, 5, 4080, SEGMENT), (True, 1023, 5, 4096, LOOP), (True, 1023, 6, 1100, LOOP), (True, 1023, 5, 1100, SEGMENT),
    (True, 2047, 32, 2100, LOOP), (True, 2047, 31, 9000, SEGMENT),
])
def test_few_rows_that_see_many_keys(L, fp8, window, seqs, longest, want):  # noqa: F811
    """256 units; 8 kv heads, so 16 sequences are half a row per unit.  The longest is known from the table's width, in
    blocks of 16."""
    args = dict(S=seqs, H=32, Hk=8, D=128, B=16, ctx_bound=longest, mask_flags=WINDOW, window_left=window)
    if fp8:
        args.update(fp8=True, token_major=False)
    assert _plan(L, **args) == want
