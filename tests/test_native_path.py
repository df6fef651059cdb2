"""The operators' native host path on a machine without a GPU."""

import pytest
import torch

from pithtrain_amd.operators.mla_assemble import mla_assemble_qkv
from pithtrain_amd.operators.norm_rope import norm_rope, qk_norm_rope


def _meta(*shape):
    return torch.empty(*shape, dtype=torch.bfloat16, device="meta")


TABLE_CALLS = {
    "norm_rope": (lambda c, s: norm_rope(_meta(1, 4, 2, 128), _meta(128), c, s, 1e-6), 128),
    "norm_rope_no_weight": (lambda c, s: norm_rope(_meta(1, 4, 2, 128), None, c, s, 1e-6), 128),
    "qk_norm_rope": (lambda c, s: qk_norm_rope(_meta(1, 4, 2, 128), _meta(1, 4, 1, 128), _meta(128), _meta(128), c, s, 1e-6), 128),
    "mla_assemble": (lambda c, s: mla_assemble_qkv(_meta(1, 4, 2, 192), _meta(1, 4, 2, 256), _meta(1, 4, 1, 64), c, s), 64),
}


@pytest.mark.parametrize("which", [0, 1])
@pytest.mark.parametrize("name", TABLE_CALLS)
def test_rotary_tables_that_require_grad(name, which):
    """The result requires grad when a rotary table does, and backward() runs without giving the table a gradient."""
    call, dim = TABLE_CALLS[name]
    tables = [_meta(4, dim), _meta(4, dim)]
    tables[which].requires_grad_()
    out = call(*tables)
    outs = [out] if torch.is_tensor(out) else [o for o in out if o.grad_fn is not None]
    assert outs and all(o.requires_grad for o in outs)
    torch.autograd.backward(outs, [torch.empty_like(o) for o in outs])
    assert tables[which].grad is None
