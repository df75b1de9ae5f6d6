"""The prefill's steps between its matrix products against the torch ops they
replace: sums and relu² bit for bit (each rounds once, as torch does), the RMS
norm up to its sum order (one bf16 step of a value of RMS 1, on under 1% of
the elements), and the attention glue on rows that are not 16-byte aligned
equal to the aligned ones."""
from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("T,dm", [(1, 8), (5, 256), (130, 520), (129, 1024), (3, 2048), (66, 4096)])
@pytest.mark.parametrize("how", ["plain", "skip", "self"])
def test_add_norm(T, dm, how):
    from scope_amd import ops

    g = torch.Generator().manual_seed(T + dm)
    x, y, k = (torch.randn((T, dm), generator=g).to(torch.bfloat16).to(DEV) for _ in range(3))
    out, xn = ops.decoder_add_norm(x, y, skip=k if how == "skip" else None, skip_self=how == "self")
    ref = x + y
    ref = ref + k if how == "skip" else (ref + ref if how == "self" else ref)
    assert torch.equal(out, ref)
    d = (xn.float() - F.rms_norm(ref, (dm,)).float()).abs()
    assert bool((d <= 2.0 ** -7 * xn.float().abs()).all())
    assert (d > 0).float().mean().item() < 0.01


@pytest.mark.parametrize("n", [8, 2056, 4096 * 130])
def test_relu2(n):
    from scope_amd import ops

    h = (torch.randn(n, generator=torch.Generator().manual_seed(n)) * 3).to(torch.bfloat16).to(DEV)
    h[:4] = torch.tensor([float("inf"), float("-inf"), float("nan"), -0.0], dtype=torch.bfloat16, device=DEV)
    ref = F.relu(h).square()
    got = ops.decoder_relu2(h.clone())
    assert torch.equal(got.nan_to_num(7.0), ref.nan_to_num(7.0))


@pytest.mark.parametrize("T,H", [(1, 1), (7, 3), (33, 8)])
def test_qkv_glue_unaligned_rows(T, H):
    from scope_amd import ops
    from scope_amd.decode import _Rotary

    g = torch.Generator().manual_seed(T)
    D, rows = 128, 64
    qkv = torch.randn((T, 3 * H * D), generator=g).to(torch.bfloat16).to(DEV)
    ve = torch.randn((T, H * D), generator=g).to(torch.bfloat16).to(DEV)
    pos = torch.randperm(rows, generator=g)[:T].to(DEV)
    rot = _Rotary(D, rows, DEV)
    caches = [torch.zeros((H, rows, D), dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    odd = [torch.zeros((H, rows, D + 1), dtype=torch.bfloat16, device=DEV)[..., 1:] for _ in range(2)]
    kw = dict(heads=H, va=0.5, vb=0.25)
    q1, _, _ = ops.decoder_qkv_glue(qkv, ve, pos, rot.cos, rot.sin, k_out=caches[0], v_out=caches[1], **kw)
    q2, _, _ = ops.decoder_qkv_glue(qkv, ve, pos, rot.cos, rot.sin, k_out=odd[0], v_out=odd[1], **kw)
    assert torch.equal(q1, q2) and torch.equal(caches[0], odd[0]) and torch.equal(caches[1], odd[1])
