"""torch.ops.fa_amd (native, csrc/torch_ops.cpp) against torch.ops.fa_amd_py (the same operators in Python): over the
forms of a call that the checks tell apart, both give the same bits or raise the same error."""
import pytest
import torch

from flash_attention_factory_amd import torch_ops  # noqa: F401

pytestmark = pytest.mark.gpu

S, H, HK, D, B, NB = 3, 8, 2, 128, 16, 64


def _state(fp8):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(5)
    pool = lambda: torch.randn((NB, HK, B, D), generator=g, device=dev).half()
    k, v = pool(), pool()
    if fp8:
        k, v = k.to(torch.float8_e5m2), v.to(torch.float8_e5m2)
    q = torch.randn((S, H, D), generator=g, device=dev).half()
    parts = 2
    return dict(out=torch.full_like(q, 7.0), query=q, key_cache=k.permute(0, 2, 1, 3), value_cache=v.permute(0, 2, 1, 3),
                block_tables=torch.randperm(NB, generator=g, device=dev)[:S * 20].view(S, 20).int(),
                context_lens=torch.tensor([300, 1, 177], dtype=torch.int32, device=dev), scale=0.09,
                scratch=[torch.zeros((S, H, parts), device=dev), torch.zeros((S, H, parts), device=dev),
                         torch.zeros((S, H, parts, D), device=dev)])


_ORDER = ("query", "key_cache", "value_cache", "block_tables", "context_lens")


def _call(ns, st, fp8, split, **kw):
    name = "paged_attention_" + ("fp8_" if fp8 else "") + ("reduce" if split else "loop")
    args = [st["out"]] + (st["scratch"] if split else []) + [st[k] for k in _ORDER] + [st["scale"]] + ([1.0] if fp8 else [])
    if split:
        kw.setdefault("max_context_len", 300)
    return getattr(getattr(torch.ops, ns), name)(*args, **kw)


def _outcome(ns, fp8, split, change):
    st = _state(fp8)
    kw = change(st) or {}
    try:
        assert _call(ns, st, fp8, split, **kw) is None
    except Exception as e:  # noqa: BLE001
        return type(e), str(e), None
    torch.cuda.synchronize()
    return None, None, st["out"].float().cpu()


def _set(**kw):
    return lambda st: st.update(kw)


def _map(key, f):
    return lambda st: st.update({key: f(st[key])})


def _both_caches(f):
    return lambda st: st.update(key_cache=f(st["key_cache"]), value_cache=f(st["value_cache"]))


_dev = lambda *s, **k: torch.ones(s, device="cuda:0", **k)
CHANGES = {
    "plain": lambda st: None,
    "token-major pools": _both_caches(lambda t: t.contiguous()),
    "sinks": lambda st: dict(sinks=_dev(H, dtype=torch.float16)),
    "sinks of another type": lambda st: dict(sinks=_dev(H)),
    "sinks too short": lambda st: dict(sinks=_dev(H - 1, dtype=torch.float16)),
    "sinks not contiguous": lambda st: dict(sinks=_dev(2 * H, dtype=torch.float16)[::2]),
    "slopes, cap, window": lambda st: dict(alibi_slopes=_dev(H) * 0.01, softcap=20.0, window_left=100),
    "slopes in 16 bits": lambda st: dict(alibi_slopes=_dev(H, dtype=torch.float16)),
    "window 0": lambda st: dict(window_left=0),
    "window beyond 31 bits": lambda st: dict(window_left=1 << 33),
    "negative cap": lambda st: dict(softcap=-1.0),
    "query not contiguous": _map("query", lambda t: torch.cat([t, t], -1)[..., :D]),
    "query in 32 bits": _map("query", lambda t: t.float()),
    "query of two dimensions": _map("query", lambda t: t[0]),
    "several query tokens": lambda st: st.update(query=st["query"][:, None].repeat(1, 2, 1, 1), out=st["out"][:, None].repeat(1, 2, 1, 1),
                                                 scratch=[t.repeat_interleave(2, 0) for t in st["scratch"]]),
    "out of another shape": _map("out", lambda t: t[:, :-1].contiguous()),
    "bf16 out": _map("out", lambda t: t.bfloat16()),
    "tables in 64 bits": _map("block_tables", lambda t: t.long()),
    "tables not contiguous": _map("block_tables", lambda t: torch.cat([t, t], 1)[:, :20]),
    "a row of tables missing": _map("block_tables", lambda t: t[:-1].contiguous()),
    "lengths as a column": _map("context_lens", lambda t: t[:, None]),
    "lengths on the host": _map("context_lens", lambda t: t.cpu()),
    "pools of another head size": _both_caches(lambda t: t[..., :64].contiguous()),
    "pools with a stride in rows": _both_caches(lambda t: t[..., ::2]),
    "pools of three dimensions": _both_caches(lambda t: t[0]),
    "unequal pool strides": _map("value_cache", lambda t: t.contiguous()),
    "unequal pool types": _map("value_cache", lambda t: t.view(torch.uint8) if t.element_size() == 1 else t.bfloat16()),
    "kv heads that do not divide": _both_caches(lambda t: t.repeat(1, 1, 2, 1)[:, :, :3].contiguous()),
    "no kv heads": _both_caches(lambda t: t[:, :, :0]),
    "no sequences": lambda st: st.update({k: st[k][:0] for k in ("out", "query", "block_tables", "context_lens")},
                                         scratch=[t[:0] for t in st["scratch"]]),
    "blocks of 24": _both_caches(lambda t: torch.cat([t, t], 1)[:, :24].contiguous()),
    "misaligned query": _map("query", lambda t: torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape).copy_(t)),
    "scales of no kind": lambda st: dict(k_scales=_dev(5), v_scales=_dev(5)),
    "scales per head": lambda st: dict(k_scales=_dev(HK) * 1.5, v_scales=_dev(HK) * 0.5),
    "scales per block": lambda st: dict(k_scales=_dev(NB, HK) * 1.5, v_scales=_dev(NB, HK) * 0.5),
    "one of the scales": lambda st: dict(k_scales=_dev(HK)),
    "tmp_out in 16 bits": lambda st: st["scratch"].__setitem__(2, st["scratch"][2].half()),
    "scratch of another size": lambda st: st["scratch"].__setitem__(0, st["scratch"][0][:, :-1].contiguous()),
    "scratch too small for the longest": lambda st: dict(max_context_len=5000),
    "longest unknown": lambda st: dict(max_context_len=-1),
    "longest beyond 31 bits": lambda st: dict(max_context_len=1 << 33),
    "partitions of 100": lambda st: dict(partition_size=100),
    "requires grad": _map("query", lambda t: t.requires_grad_()),
}


@pytest.mark.parametrize("split", [False, True], ids=["loop", "reduce"])
@pytest.mark.parametrize("fp8", [False, True], ids=["fp16", "e5m2"])
@pytest.mark.filterwarnings("ignore:the scratch arrays hold")
@pytest.mark.parametrize("change", CHANGES)
def test_attention(change, fp8, split):
    native, python = (_outcome(ns, fp8, split, CHANGES[change]) for ns in ("fa_amd", "fa_amd_py"))
    # (a call that does not fit the schema is refused by the schema, whose text names the operator)
    assert native[0] == python[0], (native, python)
    if native[1] is not None:
        assert native[1].replace("fa_amd_py::", "fa_amd::") == python[1].replace("fa_amd_py::", "fa_amd::")
    else:
        assert torch.equal(native[2], python[2])


@pytest.mark.parametrize("fp8", [None, torch.float8_e5m2, torch.float8_e4m3fn, torch.uint8])
@pytest.mark.parametrize("change", [
    {}, dict(fp8_scale=0.5), dict(key=lambda t: torch.cat([t, t], 1)[:, :HK]), dict(key=lambda t: t.float()),
    dict(slots=lambda t: t.int()), dict(slots=lambda t: t[:-1]), dict(key=lambda t: t[:0], value=lambda t: t[:0], slots=lambda t: t[:0]),
    dict(k_scales=1, v_scales=1), dict(k_scales=1), dict(value=lambda t: t.cpu())], ids=lambda c: "+".join(c) or "plain")
def test_cache_write(change, fp8):
    got = []
    for ns in ("fa_amd", "fa_amd_py"):
        st = _state(False)
        kc, vc = st["key_cache"].contiguous(), st["value_cache"].contiguous()
        if fp8 is not None:
            kc, vc = (t.to(torch.float8_e5m2 if fp8 == torch.uint8 else fp8).view(fp8) for t in (kc, vc))
        t = dict(key=st["query"][:, :HK].contiguous(), value=st["query"][:, HK:2 * HK].contiguous(),
                 slots=torch.tensor([5, -1, 77], device="cuda:0"))
        for k, f in change.items():
            if callable(f):
                t[k] = f(t[k])
                if k == "key" and "value" not in change:
                    t["value"] = f(t["value"])
        kw = {k: _dev(HK) * 1.25 for k in ("k_scales", "v_scales") if k in change}
        try:
            getattr(torch.ops, ns).kv_cache_write(t["key"], t["value"], kc, vc, t["slots"], change.get("fp8_scale", 1.0), **kw)
            torch.cuda.synchronize()
            got.append((None, None, kc.view(torch.uint8).cpu(), vc.view(torch.uint8).cpu()))
        except Exception as e:  # noqa: BLE001
            got.append((type(e), str(e)))
    assert got[0][:2] == got[1][:2]
    if got[0][0] is None:
        assert torch.equal(got[0][2], got[1][2]) and torch.equal(got[0][3], got[1][3])


def test_versions_streams_and_inference_mode():
    st = _state(False)
    for split, written in ((False, [st["out"]]), (True, [st["out"], *st["scratch"]])):
        before = [t._version for t in written]
        _call("fa_amd", st, False, split)
        assert [t._version for t in written] == [v + 1 for v in before]
    want = st["out"].clone()
    side = torch.cuda.Stream()
    st["out"].zero_()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _call("fa_amd", st, False, False)
        copied = st["out"].clone()
    side.synchronize()
    assert torch.equal(copied, want)
    with torch.inference_mode():
        inner = dict(st, out=torch.zeros_like(st["out"]))
        _call("fa_amd", inner, False, False)
        assert torch.equal(inner["out"], want)
    outcomes = []
    for ns in ("fa_amd", "fa_amd_py"):  # an inference tensor written outside of inference mode
        try:
            _call(ns, inner, False, False)
            outcomes.append(None)
        except Exception as e:  # noqa: BLE001
            outcomes.append((type(e), str(e)))
    assert outcomes[0] == outcomes[1]


@pytest.mark.parametrize("ns", ["fa_amd", "fa_amd_py"])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("smaller", [lambda t: t[:-1], lambda t: t[:, :8], lambda t: t[:, :, :1], lambda t: t[..., :64]],
                         ids=["blocks", "block size", "kv heads", "head size"])
def test_a_value_pool_smaller_than_the_key_pool_is_refused(smaller, fp8, ns):
    """Block ids, heads and rows are checked against the key pool, so a smaller value pool would be read, and
    written, beyond its end.  A larger one is as good as an equal one."""
    st = _state(fp8)
    st["value_cache"] = smaller(st["value_cache"])
    for split in (False, True):
        with pytest.raises(RuntimeError, match="smaller than key_cache"):
            _call(ns, st, fp8, split)
    key, slots = st["query"][:, :HK].contiguous(), torch.tensor([5, -1, 77], device="cuda:0")
    with pytest.raises(RuntimeError, match="smaller than key_cache"):
        getattr(torch.ops, ns).kv_cache_write(key, key.clone(), st["key_cache"], st["value_cache"], slots)
    st, fewer = _state(fp8), _state(fp8)
    st["block_tables"].clamp_(max=NB - 2)
    fewer.update(block_tables=st["block_tables"], key_cache=fewer["key_cache"][:-1])
    for t in (st, fewer):
        _call(ns, t, fp8, False)
    torch.cuda.synchronize()
    assert torch.equal(st["out"], fewer["out"])


@pytest.mark.parametrize("fp8", [False, True])
def test_scratch_that_a_wide_table_could_outgrow_is_warned_of_once(fp8, monkeypatch):
    """The default max_context_len with scratch for the rows at hand and a wider table: the Python operator is there
    for the one warning of the process, not for every call."""
    import warnings
    st = _state(fp8)
    st["block_tables"] = torch.cat([st["block_tables"]] * 8, 1)   # 2560 tokens, the scratch arrays hold 1024
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        _call("fa_amd", st, fp8, True, max_context_len=-1)
    torch.cuda.synchronize()
    want = st["out"].clone()

    def never(*args, **kwargs):
        raise AssertionError("the Python operator was called")

    for module in (torch_ops._reduce, torch_ops._fp8_reduce):
        monkeypatch.setattr(module, "run", never)
    st["out"].fill_(7.0)
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        _call("fa_amd", st, fp8, True, max_context_len=-1)
    torch.cuda.synchronize()
    assert torch.equal(st["out"], want)
