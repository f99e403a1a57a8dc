"""The native operators (torch.ops.fa_amd) have the schemas and tags of the Python ones (torch.ops.fa_amd_py)."""
import pytest
import torch

from flash_attention_factory_amd import torch_ops


@pytest.mark.parametrize("name", torch_ops._NAMES)
def test_schema_and_tags(name):
    native, python = getattr(torch.ops.fa_amd, name).default, getattr(torch.ops.fa_amd_py, name).default
    assert str(native._schema) == str(python._schema).replace("fa_amd_py::", "fa_amd::")
    assert set(native.tags) == set(python.tags)
    assert getattr(torch_ops, name) is getattr(torch.ops.fa_amd, name)
