"""Gradients of the attention backward in the operands' 16-bit type and the launch that prepares it (D = rowsum(O*dO), the
cast of dO, cleared sums): both are roundings of what the fp32 paths give, so everything is compared bit for bit."""
import pytest
import torch

import proteusai_amd as pa
from proteusai_amd import _lib, synth
from proteusai_amd.geometric_attn import _delta, _prepare_backward

pytestmark = pytest.mark.gpu


def _inputs(gpu, Z, H, N, d, op, seed):
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(Z, H, N, d, generator=g).to(op).to(gpu) for _ in range(3))
    coords = torch.stack([synth.random_walk_chain(N, g) for _ in range(Z)]).to(gpu)
    mask = torch.zeros(Z, N, dtype=torch.bool)
    mask[-1, max(1, N - N // 5):] = True
    return q, k, v, coords, synth.log_spaced_sigma(H).to(gpu), mask.to(gpu), torch.randn(Z, H, N, d, generator=g).to(gpu)


@pytest.mark.parametrize("token_major", [False, True])
@pytest.mark.parametrize("legacy", [False, True])
@pytest.mark.parametrize("d", [32, 64, 128])
# (both sides of the 64 / 128 own tokens rule: 288 workgroups of 128 for the README logits, 432 for the beta-weighted ones)
@pytest.mark.parametrize("Z,H,N", [(1, 2, 1), (2, 3, 127), (1, 4, 129), (2, 8, 1030), (3, 8, 1030)])
def test_gradients_in_the_operand_type_are_the_fp32_ones_rounded(gpu, Z, H, N, d, legacy, token_major):
    op = torch.float16 if legacy else torch.bfloat16
    q, k, v, coords, sigma, mask, dO = _inputs(gpu, Z, H, N, d, op, 100 * d + N)
    if token_major:
        q, k, v, dO = (t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3) for t in (q, k, v, dO))
    kw = dict(betas=torch.linspace(0.5, 1.2, H, device=gpu), min_rbf=0.001, operand_dtype=op) if legacy else {}
    O, L = pa.geo_attn(q, k, v, coords, sigma, mask, return_lse=True, token_major_out=token_major, **kw)
    full = pa.geo_attn_backward(q, k, v, O, L, dO, coords, sigma, mask, **kw)
    half = pa.geo_attn_backward(q, k, v, O, L, dO, coords, sigma, mask, grad_dtype=op, **kw)
    for a, b in zip(full[:3], half[:3]):
        assert a.dtype == torch.float32 and b.dtype == op and b.stride() == q.stride()
        assert torch.equal(a.to(op), b)
    for a, b in zip(full[3:], half[3:]):
        assert (a is None and b is None) or torch.allclose(a, b, rtol=1e-4, atol=1e-6)     # (sums in the order of atomics)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("op", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Z,H,N,d", [(1, 1, 1, 32), (2, 3, 333, 64), (1, 300, 5, 128)])
def test_preparation_of_the_backward(gpu, Z, H, N, d, op, dtype):
    g = torch.Generator().manual_seed(N + d)
    O = torch.randn(Z, H, N, d, generator=g).to(gpu)
    dO = torch.randn(Z, H, N, d, generator=g)
    dO[0, 0, 0, :4] = torch.tensor([float("inf"), -1.0e30, 1.0e-30, -0.0])
    dO = dO.to(dtype).to(gpu)
    wide = torch.zeros(Z, H, N, d + 4, dtype=dtype, device=gpu)
    wide[..., :d] = dO
    for what, o_, g_ in (("contiguous", O, dO), ("token-major", O, dO.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)),
                         ("rows of a wider buffer", O, wide[..., :d]), ("one row for all", O, dO[:, :, :1].expand(Z, H, N, d))):
        D, cast, ds, db = _prepare_backward(o_, g_, op, 1 if op == torch.float16 else 0, betas=ds_like(H, gpu))
        assert torch.equal(cast, g_.to(op)) and cast.dtype == op, what
        assert torch.equal(D.nan_to_num(), _delta(o_, g_).nan_to_num()), what
        assert ds.shape == db.shape == (H,) and not ds.any() and not db.any(), what
    assert _prepare_backward(O, dO, op, 1 if op == torch.float16 else 0, betas=None)[3] is None


def ds_like(H, gpu):
    """Leaves memory that is not zero where the next small tensors are likely to go."""
    junk = [torch.full((H,), 7.0, device=gpu) for _ in range(4)]
    del junk
    return torch.ones(H, device=gpu)


def test_tensors_that_do_not_go_together_are_refused(gpu):
    # before anything is launched: their addresses or sizes are not what the kernels take them for
    q, k, v, coords, sigma, mask, dO = _inputs(gpu, 2, 3, 40, 32, torch.bfloat16, 1)
    for t in ((q, k.cpu(), v), (q, k, v.cpu())):
        with pytest.raises(_lib.ProteusError, match="all on one"):
            pa.geo_attn(*t, coords, sigma, mask)
    O, L = pa.geo_attn(q, k, v, coords, sigma, mask, return_lse=True)
    for t in ((q, k.cpu(), v, O, L, dO), (q, k, v, O.cpu(), L, dO), (q, k, v, O, L, dO.cpu())):
        with pytest.raises(_lib.ProteusError, match="all on one"):
            pa.geo_attn_backward(*t, coords, sigma, mask)
    for t in ((q, k[:, :, :39], v, O, L, dO), (q, k, v, O[:, :2], L, dO), (q, k, v, O, L[:1], dO), (q, k, v, O, L, dO[..., :1])):
        with pytest.raises(AssertionError, match="one shape"):
            pa.geo_attn_backward(*t, coords, sigma, mask)
