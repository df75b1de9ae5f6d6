"""GPU: the soft pointer weights' backward stored into dq and dk equals the
same backward added to zeros, bit for bit, whatever the buffers held, for both
block sizes and head widths and for contiguous and [1,T,H,D]-strided rows."""
from __future__ import annotations

import pytest
import torch

from scope_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("H,NB,bs,D,thd", [(1, 1, 128, 128, False), (3, 17, 128, 128, True), (2, 9, 256, 64, True),
                                           (2, 5, 256, 128, False)])
def test_store_equals_add_to_zero(H, NB, bs, D, thd):
    g = torch.Generator(device=DEV).manual_seed(NB)
    L, T = 4, NB * bs
    num = torch.minimum(torch.arange(1, NB + 1), torch.tensor(L)).to(torch.int32).repeat(H, 1)
    idx = (torch.arange(NB)[:, None] - torch.arange(L)).clamp(min=0).flip(1).to(torch.int32)
    for b in range(min(L - 1, NB)):  # rows of fewer entries: 0 .. b, the tail repeats
        idx[b] = torch.tensor([min(e, b) for e in range(L)], dtype=torch.int32)
    num, idx = num.to(DEV), idx.repeat(H, 1, 1).contiguous().to(DEV)
    q_off, q_list = ops.transpose_blocks(num, idx, NB)
    qbar, kbar = (torch.randn((H, NB, D), generator=g, device=DEV) for _ in range(2))
    pb = -torch.rand(idx.shape, generator=g, device=DEV)
    pb[..., 0] = 0.0  # an entry without a weight
    dpb = torch.randn(idx.shape, generator=g, device=DEV)

    def run(fill, store):
        dq, dk = (torch.full((1, T, H, D) if thd else (1, H, T, D), fill, dtype=torch.bfloat16, device=DEV)
                  for _ in range(2))
        if thd:
            dq, dk = dq.transpose(1, 2), dk.transpose(1, 2)
        ops.pointer_bwd(qbar, kbar, num, idx, q_off, q_list, pb, dpb, dq, dk, bs=bs, logit_scale=11.3, soft_temp=2.0,
                        store=store)
        return dq, dk

    for a, b in zip(run(0.0, False), run(float("nan"), True)):
        assert torch.equal(a, b) and not bool(torch.isnan(b).any())
