"""The native host path: ordinary calls never reach an op's Python body, calls of unusual layout do, and both give the same
bits (they end in the same kernels)."""

import pytest
import torch

from pithtrain_amd._ext import native
from pithtrain_amd.operators.mla.hip import attention_func
from pithtrain_amd.operators.mla_assemble import mla_assemble_qkv
from pithtrain_amd.operators.norm_rope import norm_rope, qk_norm_rope

pytestmark = pytest.mark.gpu


def _attention(mk):
    return lambda q, k, v: attention_func(q, k, v, 0.1, True), [mk(2, 70, 4, 128), mk(2, 70, 2, 128), mk(2, 70, 2, 128)]


def _norm_rope(mk):
    cos, sin = mk(1, 70, 128), mk(1, 70, 128)
    return lambda x, w: norm_rope(x, w, cos, sin, 1e-6), [mk(2, 70, 4, 128), mk(128)]


def _qk_norm_rope(mk):
    cos, sin = mk(70, 128), mk(70, 128)
    return lambda q, k, a, b: qk_norm_rope(q, k, a, b, cos, sin, 1e-6), [mk(2, 70, 4, 128), mk(2, 70, 2, 128), mk(128), mk(128)]


def _mla_assemble(mk):
    cos, sin, pos = mk(80, 64), mk(80, 64), torch.arange(70, device="cuda")[None]
    return lambda q, kv, pe: mla_assemble_qkv(q, kv, pe, cos, sin, pos), [mk(2, 70, 4, 192), mk(2, 70, 4, 256), mk(2, 70, 1, 64)]


@pytest.mark.parametrize("make", [_attention, _norm_rope, _qk_norm_rope, _mla_assemble])
def test_native_and_python_bodies_agree(gpu, make):
    g = torch.Generator().manual_seed(11)
    call, inputs = make(lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(gpu))
    called = []
    import pithtrain_amd.operators.mla.hip as H
    import pithtrain_amd.operators.mla_assemble as A
    import pithtrain_amd.operators.norm_rope as N

    ops = {n: getattr(mod, f"_{n}_body") for mod, names in (
        (H, ("attn_fwd", "attn_bwd")), (A, ("mla_assemble_fwd", "mla_assemble_bwd")),
        (N, ("norm_rope_fwd", "norm_rope_bwd", "qk_norm_rope_fwd", "qk_norm_rope_bwd"))) for n in names}  # fmt: skip

    def spy(name):
        def body(*args):
            called.append(name)
            return ops[name](*args)

        return body

    native.set_bodies({n: spy(n) for n in ops})
    try:
        results = []
        for strided in (False, True):
            leaves = [t.clone().requires_grad_() for t in inputs]
            args = leaves
            if strided:  # every second row of a tensor twice as long: no ordinary layout
                args = [t if t.dim() == 1 else t.repeat_interleave(2, dim=1)[:, ::2] for t in leaves]
            out = call(*args)
            outs = [out] if torch.is_tensor(out) else list(out)
            gg = torch.Generator().manual_seed(5)
            douts = [torch.randn(o.shape, generator=gg).to(torch.bfloat16).to(gpu) for o in outs]
            if strided:
                douts = [d.repeat_interleave(2, dim=1)[:, ::2] for d in douts]
            grads = torch.autograd.grad(outs, leaves, douts)
            results.append([o.detach() for o in outs] + list(grads))
            assert bool(called) == strided, called
        for a, b in zip(*results):
            assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b)
    finally:
        native.set_bodies(ops)
