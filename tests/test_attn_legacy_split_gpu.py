"""Beta-weighted logits in launches of few workgroups: keys split over pairs of waves in the forward (up to 384 workgroups of 128
queries), 64 own tokens per workgroup in the backward (up to 96 ... 384 workgroups of 128, by length and masks), on both sides of the
two rules and at the edges of the tiles, against the oracles and bars of the other legacy tests."""
import pytest
import torch

import proteusai_amd as pa
from test_attn_dims_gpu import LSE_TOL_BF16, LSE_TOL_F16, check_backward, check_forward, make

pytestmark = pytest.mark.gpu


def _min_rbf(coords, sigma):
    """A lower bound near 0.001 that no pair of the input sits on: the fp32 rbf of a pair is off by up to 10 (its exponent in log2
    units) x 4 roundings x 2^-24 x ln 2 + 1e-7 = 1.8e-6 of itself, and a pair closer to the bound than that is in range for one
    of kernel and oracle only."""
    c = coords.double()
    d2 = ((c[:, :, None] - c[:, None]) ** 2).sum(-1)
    near = [(-d2 / (2 * s * s)).exp().flatten() for s in sigma.double()]
    near = torch.cat([r[(r > 0.0009) & (r < 0.0012)] for r in near])
    return next(lo for lo in (0.001 * (1 + 1e-5 * i) for i in range(1000)) if not ((near / lo - 1).abs() < 3e-6).any())


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("Z,H,N", [(1, 2, 1), (2, 3, 63), (1, 4, 65), (2, 3, 257), (8, 16, 200), (9, 16, 200), (7, 64, 40)])
def test_legacy_logits_in_launches_of_few_workgroups(gpu, Z, H, N, d):
    Q, K, V, dO, coords, sigma, mask = make(40 + N + d, Z, H, N, d, torch.float16, maskfrac=0.2 if N > 60 else 0.0)
    betas = torch.exp(0.3 * torch.randn(H, generator=torch.Generator().manual_seed(N)))
    if Z > 1:
        mask = torch.zeros(Z, N, dtype=torch.bool) if mask is None else mask
        mask[1, N // 3:] = True                       # a wave without a query, a tile without a key
    lo = _min_rbf(coords, sigma)
    O, L = pa.geo_attn(Q.to(gpu), K.to(gpu), V.to(gpu), coords.to(gpu), sigma.to(gpu), None if mask is None else mask.to(gpu),
                       return_lse=True, betas=betas.to(gpu), min_rbf=lo, max_rbf=1.0, operand_dtype=torch.float16)
    check_forward(O, L, Q, K, V, coords, sigma, mask, betas, lo, 1.0, LSE_TOL_F16, f"Z={Z} N={N} d={d}")
    check_backward(gpu, Q, K, V, dO, coords, sigma, mask, betas, lo, 1.0, torch.float16, 2.0 ** -9, f"Z={Z} N={N} d={d}")


@pytest.mark.parametrize("op", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("Z,H,N,padded,pair_mask", [                 # workgroups of 128 own tokens, both passes, and the limit that they meet
    (6, 8, 100, False, False), (7, 7, 100, False, False),            # 96 and 98: 96 for short sequences
    (5, 8, 200, False, True), (6, 7, 200, True, True),               # 160 and 168: 160
    (4, 8, 500, False, True), (3, 11, 500, False, False),            # 256 and 264: 256 without padding
    (4, 10, 500, True, False), (6, 7, 500, True, True),              # 320 and 336: 320 with
    (3, 9, 800, True, False), (4, 7, 800, True, True)])              # 378 and 392: 384 with, from 768 tokens on
def test_legacy_backward_on_both_sides_of_its_rule(gpu, Z, H, N, padded, pair_mask, d, op):
    Q, K, V, dO, coords, sigma, _ = make(60 + N + d, Z, H, N, d, op)
    betas = torch.exp(0.3 * torch.randn(H, generator=torch.Generator().manual_seed(N)))
    mask = torch.arange(N)[None, :] >= torch.linspace(N // 2, N, Z).long()[:, None] if padded else None
    lo = _min_rbf(coords, sigma) if pair_mask else 0.0
    what = f"Z={Z} H={H} N={N} d={d} {op}"
    m = None if mask is None else mask.to(gpu)
    kw = dict(betas=betas.to(gpu), min_rbf=lo, max_rbf=1.0, operand_dtype=op)
    q, k, v, c, s = (t.to(gpu) for t in (Q, K, V, coords, sigma))
    O, L = pa.geo_attn(q, k, v, c, s, m, return_lse=True, **kw)
    check_forward(O, L, Q, K, V, coords, sigma, mask, betas, lo, 1.0, LSE_TOL_F16 if op == torch.float16 else LSE_TOL_BF16, what)
    check_backward(gpu, Q, K, V, dO, coords, sigma, mask, betas, lo, 1.0, op, 2.0 ** -9, what)
    # gradients in the operands' type: the fp32 ones, rounded once
    full = pa.geo_attn_backward(q, k, v, O, L, dO.to(gpu), c, s, m, **kw)
    half = pa.geo_attn_backward(q, k, v, O, L, dO.to(gpu), c, s, m, grad_dtype=op, **kw)
    assert all(torch.equal(a.to(op), b) for a, b in zip(full[:3], half[:3])), what
