"""The first tiles of a workgroup: stationary rows staged through LDS slots that the first tiles take over, with counted waits
that depend on how many tiles follow. Streams of one to five tiles against row counts around 16, 32 and 128."""

import pytest
import torch

from helpers import check_bf16_result
from test_bwd_splits_gpu import test_backward_splits as check_backward
from pithtrain_amd.operators.mla.hip import _mla_fwd

pytestmark = pytest.mark.gpu


def _forward_reference(q, k, v, scale, causal):
    group = q.shape[2] // k.shape[2]
    out = torch.zeros(*q.shape[:3], v.shape[3], device=q.device)
    mask = torch.ones(q.shape[1], k.shape[1], dtype=torch.bool, device=q.device).triu(1) if causal else None
    for b in range(q.shape[0]):
        for h in range(q.shape[2]):
            s = (q[b, :, h].float() @ k[b, :, h // group].float().t().contiguous()) * scale
            if causal:
                s.masked_fill_(mask, float("-inf"))
            out[b, :, h] = torch.softmax(s, -1) @ v[b, :, h // group].float()
    return out


# (rows, keys): equal ones also run under the mask, where every row block has a stream length of its own
SIZES = [(1, 1), (15, 64), (17, 65), (32, 32), (33, 129), (95, 33), (128, 128), (129, 192), (160, 160), (255, 255), (257, 300), (320, 320)]


@pytest.mark.parametrize("D,Hq,Hkv", [(64, 2, 1), (128, 2, 1), (192, 2, 2)])
@pytest.mark.parametrize("Sq,Skv", SIZES)
def test_first_tiles(gpu, D, Hq, Hkv, Sq, Skv):
    g = torch.Generator(device=gpu).manual_seed(5)
    mk = lambda s, h, d: torch.randn(2, s, h, d, generator=g, device=gpu).to(torch.bfloat16)  # noqa: E731
    q, k, v = mk(Sq, Hq, D), mk(Skv, Hkv, D), mk(Skv, Hkv, min(D, 128))
    for causal in [False, True] if Sq == Skv else [False]:
        o, _ = _mla_fwd(q, k, v, D**-0.5, causal)
        check_bf16_result(o, _forward_reference(q, k, v, D**-0.5, causal), "O", otol=1e-3)
        check_backward(gpu, 2, Sq, Skv, Hq, Hkv, D, causal)


@pytest.mark.parametrize("D,H,S", [(128, 130, 512), (128, 130, 545), (192, 20, 700), (192, 66, 513), (64, 150, 545), (128, 20, 700)])
def test_first_tiles_of_larger_grids(gpu, D, H, S):
    """The other work splits: 256-row workgroups, wave pairs splitting keys, two workgroups per unit, 64-row workgroups."""
    g = torch.Generator(device=gpu).manual_seed(6)
    mk = lambda d: torch.randn(1, S, H, d, generator=g, device=gpu).to(torch.bfloat16)  # noqa: E731
    q, k, v = mk(D), mk(D), mk(min(D, 128))
    for causal in [False, True]:
        o, _ = _mla_fwd(q, k, v, D**-0.5, causal)
        check_bf16_result(o, _forward_reference(q, k, v, D**-0.5, causal), "O", otol=1e-3)


@pytest.mark.parametrize("S", [32, 33, 64, 65, 96, 97, 128, 129, 160, 161, 224, 290])
@pytest.mark.parametrize("Hq,Hkv", [(1, 1), (6, 2)])
def test_woven_steps_at_64_features(gpu, S, Hq, Hkv):
    """Gradients of 64 features: streams of one to ten steps of 32 rows, ragged ends, one and several heads to a stream, with
    waves that leave the workgroup's stream early (causal)."""
    for causal in [False, True]:
        check_backward(gpu, 1, S, S, Hq, Hkv, 64, causal)
    check_backward(gpu, 1, S, 290 - S // 2, Hq, Hkv, 64, False)
