"""The operators have no second derivatives: their backward may run under create_graph, but differentiating through its result
raises (it must not warn and leave the second-order part out). Shapes only, on the meta device."""

import pytest
import torch

from pithtrain_amd.operators.mla.hip import attention_func
from pithtrain_amd.operators.mla_assemble import mla_assemble_qkv
from pithtrain_amd.operators.norm_rope import norm_rope, qk_norm_rope


def _meta(*shape):
    return torch.empty(*shape, dtype=torch.bfloat16, device="meta")


CALLS = {
    "attention": (lambda q, k, v: attention_func(q, k, v, 0.1, True), [(1, 4, 2, 128)] * 3),
    "norm_rope": (lambda x, w: norm_rope(x, w, _meta(4, 128), _meta(4, 128), 1e-6), [(1, 4, 2, 128), (128,)]),
    "norm_rope_no_weight": (lambda x: norm_rope(x, None, _meta(4, 128), _meta(4, 128), 1e-6), [(1, 4, 2, 128)]),
    "qk_norm_rope": (lambda q, k, a, b: qk_norm_rope(q, k, a, b, _meta(4, 128), _meta(4, 128), 1e-6), [(1, 4, 2, 128)] * 2 + [(128,)] * 2),
    "mla_assemble": (lambda q, kv, pe: mla_assemble_qkv(q, kv, pe, _meta(8, 64), _meta(8, 64)), [(1, 4, 2, 192), (1, 4, 2, 256), (1, 4, 1, 64)]),
}


@pytest.mark.parametrize("name", CALLS)
def test_second_derivative_raises(name):
    call, shapes = CALLS[name]
    x = [_meta(*s).requires_grad_() for s in shapes]
    out = call(*x)
    outs = [out] if torch.is_tensor(out) else list(out)
    douts = [torch.empty_like(o).requires_grad_() for o in outs]
    grads = torch.autograd.grad(outs, x, douts, create_graph=True)
    assert [g.shape for g in grads] == [t.shape for t in x]
    with pytest.raises(RuntimeError, match="second derivatives are not implemented"):
        torch.autograd.grad(grads[0].sum(), douts[0])
