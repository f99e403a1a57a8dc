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
