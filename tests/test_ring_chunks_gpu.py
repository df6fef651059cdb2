"""A ring share as one launch over all of its chunks: every work split of the kernels, at row counts where a tile or a wave
straddles the first row that sees a chunk, the end of a chunk or the diagonal, against the float64 oracle."""

import pytest
import torch

from helpers import check_bf16_result, check_lse
from oracle import ring_oracle as R
from pithtrain_amd.operators.ring_attention import local as L

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def no_stepwise_path(monkeypatch):
    def used(*args, **kwargs):
        raise AssertionError("the share was not taken by the chunk calls")

    monkeypatch.setattr(L, "RingForward", used)


CASES = [  # B, S_l, Hq, Hkv, D, C, rank, layout, keys in two parts
    (2, 2, 2, 1, 64, 2, 0, "zigzag", False), (1, 66, 4, 2, 64, 3, 1, "zigzag", False), (1, 257, 4, 4, 64, 2, 1, "contiguous", False),
    (1, 1, 2, 1, 128, 2, 1, "contiguous", False), (2, 130, 4, 2, 128, 3, 0, "zigzag", False), (1, 258, 4, 2, 128, 3, 2, "zigzag", False),
    (1, 1100, 32, 4, 128, 2, 1, "zigzag", False), (1, 1026, 30, 2, 128, 2, 0, "zigzag", False), (1, 96, 2, 2, 128, 16, 15, "contiguous", False),
    (1, 34, 2, 2, 192, 4, 1, "zigzag", True), (2, 129, 2, 2, 192, 3, 2, "contiguous", True), (1, 322, 4, 4, 192, 2, 0, "zigzag", False),
    (1, 1022, 36, 36, 192, 2, 1, "contiguous", True),
]  # fmt: skip


@pytest.mark.parametrize("B,S,Hq,Hkv,D,C,rank,layout,two_part", CASES)
def test_share(gpu, B, S, Hq, Hkv, D, C, rank, layout, two_part):
    g = torch.Generator().manual_seed(5)
    mk = lambda h, d: torch.randn(B, S, h, d, generator=g).to(torch.bfloat16)  # noqa: E731
    scale, dv = D**-0.5, min(D, 128)
    q = mk(Hq, D)
    ks = [mk(Hkv, 128 if two_part else D) for _ in range(C)]
    vs = [mk(Hkv, dv) for _ in range(C)]
    pes = [mk(1, 64)[:, :, 0] for _ in range(C)] if two_part else None
    full_ks = [torch.cat([k, pe[:, :, None].expand(-1, -1, Hkv, -1)], -1) for k, pe in zip(ks, pes)] if two_part else ks
    ref_o, ref_lse = R.ring_forward(q, full_ks, vs, scale, rank, C, layout)
    on_gpu = lambda ts: None if ts is None else [t.to(gpu) for t in ts]  # noqa: E731
    out, lse = L.ring_forward_local(q.to(gpu), on_gpu(ks), on_gpu(vs), scale, rank, C, layout, on_gpu(pes))
    check_bf16_result(out, ref_o, "O")
    check_lse(lse, ref_lse, "LSE2")
