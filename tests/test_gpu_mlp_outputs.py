"""GPU: the fused MLP's row-wise kernels at output counts whose rows start on
2-byte boundaries (odd O, O below and above the 16-output chunks), at the
smallest row counts and at rows that end inside a workgroup's tile.  With W2,
b2 and the output gradient padded by zeros to 64 outputs the kernels form the
same sums with exact zeros added, so y, dq, x1 and dz1 have the same bits; the
padded gradient itself is a copy."""
from __future__ import annotations

import pytest
import torch

from scope_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("rows", [32, 64, 288, 4128])
@pytest.mark.parametrize("O", [1, 3, 15, 16, 17, 31, 33, 41, 48, 61, 63, 64])
def test_output_counts(O, rows):
    g = torch.Generator(device=DEV).manual_seed(100 * O + rows)
    q = torch.randn((rows, 128), generator=g, device=DEV).to(torch.bfloat16)
    gy = torch.randn((rows, O), generator=g, device=DEV).to(torch.bfloat16)
    w1, w2 = (torch.randn(s, generator=g, device=DEV) * 0.1 for s in ((256, 128), (O, 256)))
    b1, b2 = (torch.randn(n, generator=g, device=DEV) for n in (256, O))
    pad = lambda t: torch.cat([t, t.new_zeros((64 - O,) + t.shape[1:])])  # noqa: E731
    gy64 = torch.cat([gy, gy.new_zeros((rows, 64 - O))], 1)
    y = ops.coeff_mlp_fwd(q, w1, b1, w2, b2)
    y64 = ops.coeff_mlp_fwd(q, w1, b1, pad(w2), pad(b2))
    assert y.shape == (rows, O) and torch.equal(y, y64[:, :O])
    # against fp64 on the bf16 operands: z and x1 rounded to bf16 (2^-9 each, |SiLU'| <= 1.1), then y
    w1d, w2d = w1.bfloat16().double(), w2.bfloat16().double()
    z = q.double() @ w1d.t() + b1.bfloat16().double()
    ref = torch.nn.functional.silu(z) @ w2d.t() + b2.bfloat16().double()
    bound = 2.0 ** -9 * (2.2 * z.abs() @ w2d.abs().t() + ref.abs()) + 1e-5
    assert bool(((y.double() - ref).abs() <= bound).all())
    got, want = ops.coeff_mlp_bwd(q, gy, w1, b1, w2, b2), ops.coeff_mlp_bwd(q, gy64, w1, b1, pad(w2), pad(b2))
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    assert torch.equal(got[3], gy64)
