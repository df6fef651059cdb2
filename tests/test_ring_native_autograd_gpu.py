"""The native node of a ring share (RingFunction) against its Python counterpart: the same kernels, so results are equal bit for
bit, for every form of call that either takes; what only the Python one can see reaches it."""

import pytest
import torch

from pithtrain_amd._ext import native
from pithtrain_amd.operators.ring_attention import local as L

pytestmark = pytest.mark.gpu


def _share(gpu, b, s, hq, hkv, d, cp, rank, layout, split_key=False, seed=0):
    g = torch.Generator(device=gpu).manual_seed(seed)
    t = lambda *shape: torch.randn(*shape, generator=g, device=gpu).to(torch.bfloat16)  # noqa: E731
    visited = sorted({st.kv_rank for st in L.ring_schedule(rank, cp, s, layout)})
    chunks = lambda *shape: [t(*shape) if j in visited else None for j in range(cp)]  # noqa: E731
    ks, vs = chunks(b, s, hkv, d - 64 if split_key else d), chunks(b, s, hkv, min(d, 128))
    return t(b, s, hq, d), ks, vs, chunks(b, s, 64) if split_key else None, t(b, s, hq, min(d, 128)), visited


def _passes(call, q, ks, vs, pes, dout, visited, wanted):
    leaves = [q] + [kind[j] for kind in (ks, vs, pes) if kind is not None for j in visited]
    for i, x in enumerate(leaves):
        x.requires_grad_(wanted(i))
    out = call(q, ks, vs, pes)
    return [out.detach(), *torch.autograd.grad(out, [x for x in leaves if x.requires_grad], dout)]


def _python(scale, rank, cp, layout):
    def call(q, ks, vs, pes):
        fill = lambda kind: [q.new_empty(0) if x is None else x for x in kind]  # noqa: E731
        return L.RingAttentionLocalFunc.apply(q, scale, rank, cp, layout, *fill(ks), *fill(vs), *([] if pes is None else fill(pes)))

    return call


@pytest.mark.parametrize("wanted", [lambda i: True, lambda i: i == 0, lambda i: i == 2], ids=["all", "q", "one chunk"])
@pytest.mark.parametrize(
    "shape",
    [
        (1, 128, 8, 2, 128, 2, 0, "contiguous"),  # one chunk
        (2, 131, 8, 2, 128, 4, 2, "contiguous"),
        (1, 130, 16, 16, 192, 4, 3, "zigzag"),
        (1, 333, 4, 4, 192, 4, 1, "contiguous", True),
        (2, 128, 4, 4, 192, 8, 5, "zigzag", True),
        (1, 8192, 4, 1, 128, 4, 3, "zigzag"),  # forward step by step
        (1, 4096, 32, 4, 128, 2, 1, "zigzag"),  # dS handed over
    ],
    ids=str,
)
def test_equal_to_the_python_node(gpu, shape, wanted):
    q, ks, vs, pes, dout, visited = _share(gpu, *shape)
    cp, rank, layout = shape[5:8]
    assert native.ring_attention(q, ks, vs, pes, 0.1, rank, cp, layout == "zigzag") is not None
    here = _passes(lambda *a: L.ring_attention_local(*a[:3], 0.1, rank, cp, layout, a[3]), q, ks, vs, pes, dout, visited, wanted)
    there = _passes(_python(0.1, rank, cp, layout), q, ks, vs, pes, dout, visited, wanted)
    assert len(here) == len(there) and all(torch.equal(a, b) for a, b in zip(here, there))


def test_hooks_modes_and_refusals(gpu):
    shape = (1, 256, 8, 2, 128, 4, 2, "zigzag")
    q, ks, vs, _, dout, visited = _share(gpu, *shape)
    q.requires_grad_(True)
    call = lambda q=q, ks=ks: L.ring_attention_local(q, ks, vs, 0.1, 2, 4, "zigzag")  # noqa: E731
    out = call()
    assert "CppNode" in type(out.grad_fn).__name__ or "RingFunction" in out.grad_fn.name()
    (want,) = torch.autograd.grad(out, q, dout, retain_graph=True)
    (strided,) = torch.autograd.grad(out, q, dout.transpose(1, 2).contiguous().transpose(1, 2))
    assert torch.equal(want, strided)
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out, q, dout)

    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t.shape) or t.cpu(), lambda t: t.to(gpu)):
        out = call()
    assert len(seen) == 3 + 2 * len(visited)
    assert torch.equal(torch.autograd.grad(out, q, dout)[0], want)

    with torch.no_grad():
        assert torch.equal(call(), out) and call().grad_fn is None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert torch.equal(call(), out)
    with pytest.raises(RuntimeError):  # no batching rule
        torch.vmap(call)(q.detach()[None])
    with torch.autograd.forward_ad.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
        call(torch.autograd.forward_ad.make_dual(q.detach(), torch.ones_like(q)))
    with pytest.raises(AssertionError, match="not contiguous"):
        call(ks=[k.transpose(1, 2).contiguous().transpose(1, 2) for k in ks])
    grads = torch.autograd.grad(call(), q, dout, create_graph=True)
    assert not grads[0].requires_grad  # no second derivative, as before
