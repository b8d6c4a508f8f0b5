"""Beta-weighted logits under a pair mask in launches of few workgroups: keys split over pairs of waves in the forward (up to 384
workgroups of 128 queries), 64 own tokens per workgroup in the backward (up to 512 workgroups of 128), on both sides of
the two rules and at the edges of the tiles, against the oracles and bars of the other legacy tests."""
import pytest
import torch

import proteusai_amd as pa
from test_attn_dims_gpu import LSE_TOL_F16, check_backward, check_forward, make

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
