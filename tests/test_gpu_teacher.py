"""Teacher block mass (scoped_medium.py:1799-1819) on the GPU
(scope_attn_block_mass_ws) against the fp64 oracle: the teacher's dense
document-causal attention with the token-offset band term and slope, a
pointer list with the block-offset bias, and the row-sum invariant at the
training shape.  Bar (written in each comparison): |got - ref| <= 2e-2 +
1e-2·|ref| per (head, q-block, key block) entry."""
from __future__ import annotations

import pytest
import torch

from oracle import attention as OA
from oracle.pointer import doc_start_blocks
from tests.helpers import band_coefficients, docs_with_boundaries, omegas_block, qkv, random_blockscore_mask, tol_check

pytestmark = pytest.mark.gpu
DEV = "cuda"
SCALE, BETA = 0.12, 0.5


def test_teacher_mass_dense_with_token_bias():
    import scope_amd

    H, T, bs, K = 4, 4096, 128, 6
    print(f"teacher mass T={T} H={H}", flush=True)
    docs = docs_with_boundaries(T, 5, seed=21)
    q, k, _ = qkv(H, T, seed=22)
    g = torch.Generator().manual_seed(23)
    cc = torch.randn((1, H, T, K), generator=g) * 0.3
    cs = torch.randn((1, H, T, K), generator=g) * 0.3
    sl = torch.randn((1, H, T), generator=g) * 0.002
    om = OA.omegas_logspaced(K, 1024, 1 << 20)
    sp = scope_amd.SpectralTerms(coeff_cos=cc.to(DEV), coeff_sin=cs.to(DEV), omegas=om.to(DEV), offset="token",
                                 beta=BETA, slope=sl.to(DEV), use_slope=True)
    got = scope_amd.attention.teacher_block_mass(q.to(DEV), k.to(DEV), docs.to(DEV), scale=SCALE, spectral=sp,
                                                 block_size=bs)
    ref = OA.block_mass(q[0].double(), k[0].double(), docs, bs=bs, scale=SCALE, beta=BETA, bias_mode="token",
                        coeff_cos=cc[0].double(), coeff_sin=cs[0].double(), omegas=om.double(),
                        token_kwargs=dict(slope=sl[0].double()))
    ok, worst = tol_check(got.cpu(), ref)
    assert ok, f"teacher mass: worst tolerance ratio {worst:.3f}"


def test_block_mass_pointer_lists_block_bias():
    from scope_amd import ops
    from scope_amd.attention import spectral_table

    H, T, bs = 2, 8192, 256
    print(f"block mass pointer lists T={T} bs={bs}", flush=True)
    docs = docs_with_boundaries(T, 3, seed=31)
    kv_num, kv_idx = random_blockscore_mask(H, T, bs, docs, window=2, n_global=1, budget=4, seed=32)
    q, k, _ = qkv(H, T, seed=33)
    A, B = band_coefficients(q)
    om = omegas_block(8)
    ds_end = torch.from_numpy(doc_start_blocks(docs.numpy(), bs)[2])
    mass, _ = ops.attn_block_mass(q.to(DEV), k.to(DEV), kv_num.to(DEV), kv_idx.to(DEV), docs.to(DEV),
                                  ds_end.to(DEV), bs=bs, scale=SCALE, beta=BETA, bias_mode="block",
                                  table=spectral_table(om.to(DEV), T, bs, "block"), coeff_cos=A.to(DEV),
                                  coeff_sin=B.to(DEV))
    ref = OA.block_mass(q[0].double(), k[0].double(), docs, bs=bs, scale=SCALE, beta=BETA, bias_mode="block",
                        coeff_cos=A[0].double(), coeff_sin=B[0].double(), omegas=om.double(), kv_num=kv_num,
                        kv_idx=kv_idx)
    ok, worst = tol_check(mass.cpu(), ref)
    assert ok, f"pointer-list mass: worst tolerance ratio {worst:.3f}"


def test_teacher_mass_row_sums_at_training_shape():
    """T=65536, H=8, bs=128 (512 blocks): every q-block's mass sums to bs, and
    three sampled q-blocks equal the oracle (no bias)."""
    import scope_amd

    H, T, bs = 8, 65536, 128
    NB = T // bs
    print(f"teacher mass T={T} H={H}", flush=True)
    docs = docs_with_boundaries(T, 8, seed=41)
    q, k, _ = qkv(H, T, seed=42)
    got = scope_amd.attention.teacher_block_mass(q.to(DEV), k.to(DEV), docs.to(DEV), scale=SCALE, block_size=bs)
    torch.cuda.synchronize()
    rs = got.sum(-1).cpu()
    assert (rs - bs).abs().max().item() <= 2e-2 * bs, f"row sums off by {(rs - bs).abs().max().item():.3e}"
    qbs = [0, NB // 3, NB - 1]
    kv_num = torch.zeros((1, NB), dtype=torch.int32)
    kv_idx = torch.zeros((1, NB, NB), dtype=torch.int32)
    for qb in range(NB):
        kv_num[0, qb] = qb + 1
        kv_idx[0, qb, :qb + 1] = torch.arange(qb + 1)
    for h in (0, H - 1):
        for qb in qbs:
            rows = slice(qb * bs, (qb + 1) * bs)
            qq = q[0, h:h + 1].double()
            kk = k[0, h:h + 1].double()
            res = OA.attention_blocksparse(qq, kk, torch.nn.functional.one_hot(torch.arange(T) // bs, NB).double()[None],
                                           kv_num, kv_idx, docs, bs=bs, scale=SCALE, heads=[0], qblocks=[qb])
            want = res[(0, qb)][0].sum(0)
            ok, worst = tol_check(got[h, qb].cpu(), want)
            assert ok, f"head {h} q-block {qb}: worst tolerance ratio {worst:.3f}"


@pytest.mark.parametrize("bs,T,H,mode", [(128, 128, 1, "token"), (128, 2176, 3, "token"), (256, 1280, 2, "block"),
                                         (256, 256, 1, "none"), (128, 4096, 1, "gate")])
def test_block_mass_one_pass_against_two_passes(bs, T, H, mode):
    """The one-pass masses and LSE (scope_attn_block_mass_ws) against the
    two-pass entry point on the same lists: one block, odd block counts, an
    empty row, ragged lists.  Both are fp32 sums of the same probabilities
    (exp2 to 1 ulp, at most bs·2^11 terms added in another order): masses of
    at most bs differ by less than bs·2^-18, the LSE by 2^-18·(1 + |lse|)."""
    import ctypes as C

    from scope_amd import _lib, ops
    from scope_amd.attention import spectral_table

    print(f"block mass one/two passes bs={bs} T={T} H={H} {mode}", flush=True)
    NB = T // bs
    docs = docs_with_boundaries(T, min(3, NB), seed=51)
    kv_num, kv_idx = random_blockscore_mask(H, T, bs, docs, window=2, n_global=1, budget=3, seed=52)
    if NB > 2:
        kv_num[0, 1] = 0
    q, k, _ = qkv(H, T, seed=53)
    A, B = band_coefficients(q)
    bias = {"gate": "token"}.get(mode, mode)
    kw = dict(bs=bs, scale=SCALE, beta=BETA, bias_mode=bias)
    if bias != "none":
        kw.update(table=spectral_table(omegas_block(8).to(DEV), T, bs, bias), coeff_cos=A.to(DEV), coeff_sin=B.to(DEV))
    dm = wd = None
    if mode == "gate":
        g = torch.Generator().manual_seed(54)
        dm, wd = (torch.rand((1, H, T), generator=g) * s for s in (1024.0, 256.0))
        kw.update(delta_main=dm.to(DEV), width=wd.to(DEV), gate_kind="softplus", ramp_lambda=0.2, tau=64.0)
    ds_end = torch.from_numpy(doc_start_blocks(docs.numpy(), bs)[2])
    dev = [t.to(DEV).contiguous() for t in (q, k, kv_num, kv_idx, docs, ds_end)]
    mass, lse = ops.attn_block_mass(*dev, **kw)
    qd, kd, num, idx, dd, de = dev
    prm = ops._attn_params(qd, kd, kd, qd, bs=bs, maxkv=idx.shape[-1], scale=SCALE, beta=BETA,
                           bias_mode=ops.BIAS_MODES[bias], K=0 if bias == "none" else 8, use_slope=False,
                           subtract_b0=False, gate_kind=int(mode == "gate"), ramp_lambda=0.2, tau=64.0)
    m2 = torch.zeros_like(mass)
    l2 = torch.empty_like(lse)
    p = lambda t: None if t is None else C.c_void_p(t.data_ptr())  # noqa: E731
    opt = [kw.get(n) for n in ("table", "coeff_cos", "coeff_sin", "b0", "slope", "delta_main", "width")]
    _lib.call("scope_attn_block_mass", C.byref(prm), p(qd), p(kd), p(num), p(idx), p(dd), p(de), *(p(t) for t in opt),
              p(l2), p(m2), C.c_void_p(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert torch.equal(torch.isinf(lse), torch.isinf(l2))
    fin = torch.isfinite(l2)
    assert ((lse - l2).abs()[fin] <= 2.0 ** -18 * (1 + l2.abs()[fin])).all()
    assert (mass - m2).abs().max().item() <= bs * 2.0 ** -18
    assert torch.equal(mass > 0, m2 > 0)
