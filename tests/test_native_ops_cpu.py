"""The native operators (torch.ops.fa_amd) have the schemas and tags of the Python ones (torch.ops.fa_amd_py)."""
import os
import subprocess
import sys

import pytest
import torch

from flash_attention_factory_amd import torch_ops

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("name", torch_ops._NAMES)
def test_schema_and_tags(name):
    native, python = getattr(torch.ops.fa_amd, name).default, getattr(torch.ops.fa_amd_py, name).default
    assert str(native._schema) == str(python._schema).replace("fa_amd_py::", "fa_amd::")
    assert set(native.tags) == set(python.tags)
    assert getattr(torch_ops, name) is getattr(torch.ops.fa_amd, name)


def _in_a_process(code, **env):
    return subprocess.run([sys.executable, "-c", code], capture_output=True, text=True,
                          env=dict(os.environ, PYTHONPATH=ROOT, **env))


CALL = """
import torch
from flash_attention_factory_amd import torch_ops
q = torch.zeros((1, 2, 64), dtype=torch.float16, device=DEVICE)
pool = torch.zeros((2, 16, 2, 64), dtype=torch.float16, device=DEVICE)
tables, lens = (torch.ones(s, dtype=torch.int32, device=DEVICE) for s in ((1, 2), (1,)))
torch.ops.fa_amd.paged_attention_loop(torch.zeros_like(q), q, pool, pool, tables, lens, 0.125)
"""


def test_importing_the_operators_needs_no_library(tmp_path):
    """A library that is missing, or does not load, is for the calls to report."""
    missing = str(tmp_path / "missing.so")
    torn = tmp_path / "torn.so"
    torn.write_bytes(b"not a library")
    for library in (missing, str(torn)):
        env = dict(FA_PAGED_ATTENTION_LIBRARY=library)
        assert _in_a_process(CALL.replace("DEVICE", "'meta'"), **env).returncode == 0
        patch = f"from flash_attention_factory_amd import _build; _build.TORCH_OPS_LIBRARY = {library!r}\n"
        res = _in_a_process(patch + CALL.replace("DEVICE", "'meta'"))
        assert res.returncode == 0, res.stderr
        res = _in_a_process(patch + CALL.replace("DEVICE", "'cpu'"))
        assert res.returncode != 0 and "does not load" in res.stderr and "g.build()" in res.stderr


def test_schemas_without_the_library(tmp_path):
    code = ("from flash_attention_factory_amd import _build; _build.TORCH_OPS_LIBRARY = '/missing.so'\n"
            "import torch\nfrom flash_attention_factory_amd import torch_ops\n"
            "for n in torch_ops._NAMES: op = getattr(torch.ops.fa_amd, n).default; print(op._schema, sorted(map(str, op.tags)))")
    res = _in_a_process(code)
    assert res.returncode == 0, res.stderr
    here = [f"{op._schema} {sorted(map(str, op.tags))}" for op in (getattr(torch.ops.fa_amd, n).default for n in torch_ops._NAMES)]
    assert res.stdout.splitlines() == here


def test_operators_of_other_sources_say_so(tmp_path):
    """A library that registers operators but does not take the entry points: no call, on whatever path, goes on
    without them."""
    source, library = tmp_path / "other.c", tmp_path / "other.so"
    source.write_text("int nothing(void) { return 0; }")
    subprocess.run(["gcc", "-shared", "-fPIC", str(source), "-o", str(library)], check=True)
    code = ("from flash_attention_factory_amd import _build, _cabi; _build.TORCH_OPS_LIBRARY = %r\n"
            "import flash_attention_factory_amd.torch_ops as ops\n" % str(library))
    # (the stub registers nothing, so the schemas are missing; what matters is that loading the C ABI raises)
    code = code.replace("import flash", "import torch; [torch.library.define('fa_amd::' + n, '(Tensor x) -> ()') for n in "
                        "('paged_attention_loop', 'paged_attention_fp8_loop', 'paged_attention_reduce', "
                        "'paged_attention_fp8_reduce', 'kv_cache_write')]\nimport flash", 1)
    res = _in_a_process(code + "_cabi.load()")
    assert res.returncode != 0 and "built from other sources" in res.stderr, res.stderr
