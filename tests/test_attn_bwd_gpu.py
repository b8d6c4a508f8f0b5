"""GPU parity tests of the geometric attention backward: the HIP kernels, called through the C ABI via the
autograd function, against torch.autograd through the dense fp64 statement of the forward on the same
bf16-rounded inputs.

Bar: the operands of every matrix product are bf16 (Q, K, V, dO, P, dS; the reference uses fp16), so each
gradient tensor is compared in relative L2 norm: <= 1e-2 for dQ, dK, dV (measured: 2.4e-3).

The per-head scalars d_sigma and d_beta are sums over all pairs of P * (dP - D) * dT/d(scalar), terms of both signs,
with D = rowsum(O * dO) from the forward's bf16 output.  dP and D cancel inside a query (exactly, for a query with
one in-range key) and the queries cancel against each other, so the rounding error of the sum scales with what went in
before any cancellation, not with what comes out: the weights of D are the forward's bf16-rounded probabilities, the
backward's P are fp32, and the two differ by up to 2^-8 per pair, which multiplies |dP|, not |dP - D|.  They are held to
  |got - ref| <= 2^-9 * sum over pairs of P * (|dP| + |D|) * |dT/d(scalar)|     always (no term is dropped; half of the
                                                                                worst case 2^-8, measured <= 4.5e-4), and
  relative L2 <= 1e-2                                                          where the result keeps at least a
                                                                                quarter of that pair sum.
The oracle yields the pair sum (geo_attn_scalar_grad_mass) and the per-query contributions (the gradient with respect
to a per-query copy of sigma / beta)."""
import numpy as np
import pytest
import torch

import proteusai_amd as pa
from oracle import torch_oracle
from proteusai_amd import synth

pytestmark = pytest.mark.gpu

REL_L2_TOL = 1e-2
SCALAR_TOL = 2.0 ** -9          # of the pair sum


def rel_l2(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    nb = np.linalg.norm(b)
    return float(np.linalg.norm(a - b) / nb) if nb > 0 else float(np.linalg.norm(a - b))


def make(seed, Z, H, N, maskfrac=0.0, qscale=1.0):
    g = torch.Generator().manual_seed(seed)
    Q = (torch.randn(Z, H, N, 64, generator=g) * qscale).bfloat16()
    K = torch.randn(Z, H, N, 64, generator=g).bfloat16()
    V = torch.randn(Z, H, N, 64, generator=g).bfloat16()
    dO = torch.randn(Z, H, N, 64, generator=g).bfloat16()
    coords = torch.stack([synth.random_walk_chain(N, g) for _ in range(Z)])
    sigma = synth.log_spaced_sigma(H)
    mask = (torch.rand(Z, N, generator=g) < maskfrac) if maskfrac > 0 else None
    return Q, K, V, dO, coords, sigma, mask


def reference_grads(Q, K, V, dO, coords, sigma, mask, betas=None, min_rbf=0.0, max_rbf=1.0):
    """dQ, dK, dV, the per-query contributions [Z,H,N] to d_sigma and d_beta (their sums over Z and N are the
    per-head gradients), and the pair sums [H] that scale the rounding error of the two."""
    Z, H, N, _ = Q.shape
    q, k, v = (t.double().requires_grad_(True) for t in (Q, K, V))
    s = sigma.double()[None, :, None].expand(Z, H, N).clone().requires_grad_(True)
    b = None if betas is None else betas.double()[None, :, None].expand(Z, H, N).clone().requires_grad_(True)
    O = torch_oracle.geo_attn_autograd_torch(q, k, v, coords, s, mask, b, min_rbf, max_rbf)
    O.backward(dO.double())
    mass_s, mass_b, _, _ = torch_oracle.geo_attn_scalar_grad_mass(Q, K, V, dO, coords, sigma, mask, betas, min_rbf, max_rbf)
    return q.grad, k.grad, v.grad, s.grad, None if b is None else b.grad, mass_s, mass_b


def check_head_scalar(got, per_query, pair_mass, what):
    total = per_query.sum(dim=(0, 2))
    err = (got.double() - total).abs()
    assert torch.isfinite(got).all(), f"{what}: non-finite"
    assert (err <= SCALAR_TOL * pair_mass + 1e-30).all(), \
        f"{what}: error / pair mass {(err / pair_mass.clamp_min(1e-300)).max():.3e}"
    if (total.abs() >= 0.25 * pair_mass).all():
        e = rel_l2(got.numpy(), total.numpy())
        assert e <= REL_L2_TOL, f"{what}: rel-L2 {e:.3e}"


def gpu_grads(gpu, Q, K, V, dO, coords, sigma, mask, betas=None, min_rbf=0.0, max_rbf=1.0):
    q, k, v = (t.to(gpu).requires_grad_(True) for t in (Q, K, V))
    s = sigma.to(gpu).requires_grad_(True)
    b = None if betas is None else betas.to(gpu).requires_grad_(True)
    O = pa.geometric_attn(q, k, v, coords.to(gpu), s, b, None if mask is None else mask.to(gpu), min_rbf, max_rbf)
    O.backward(dO.to(gpu).float())
    torch.cuda.synchronize()
    return q.grad.float().cpu(), k.grad.float().cpu(), v.grad.float().cpu(), s.grad.cpu(), None if b is None else b.grad.cpu()


def compare(got, ref, mask, what):
    for g, r, name in zip(got, ref[:5], ("dQ", "dK", "dV", "d_sigma", "d_beta")):
        if r is None:
            continue
        if name in ("d_sigma", "d_beta"):
            check_head_scalar(g, r, ref[5 if name == "d_sigma" else 6], f"{what} {name}")
            continue
        assert torch.isfinite(g).all(), f"{what} {name}: non-finite"
        e = rel_l2(g.numpy(), r.numpy())
        assert e <= REL_L2_TOL, f"{what} {name}: rel-L2 {e:.3e}"
    if mask is not None:
        for g, name in zip(got[:3], ("dQ", "dK", "dV")):
            assert (g[mask[:, None, :].expand(-1, g.shape[1], -1)] == 0).all(), f"{what} {name}: padded tokens must get zeros"


# Launches of at most 256 workgroups of 128 own tokens (both passes together) run workgroups of 64 own tokens instead, two
# waves per own block with half of the streamed tokens each.  The shapes below lie on both sides: FEW (Z, H) keeps the
# launch under the limit at every length tested, MANY takes it over.
FEW, MANY = (2, 3), (9, 16)


@pytest.mark.parametrize("ZH", [FEW, MANY])
@pytest.mark.parametrize("N", [1, 2, 31, 32, 33, 64, 65, 127, 128, 129, 200, 333])
def test_ragged_lengths(gpu, N, ZH):
    if ZH == MANY and N in (2, 31, 32, 64, 65, 128):
        pytest.skip("the larger launch takes a subset of the lengths")
    assert (2 * ZH[0] * ZH[1] * ((N + 127) // 128) <= 256) == (ZH == FEW)
    a = make(300 + N, ZH[0], ZH[1], N)
    if N == 1:
        got = gpu_grads(gpu, *a)
        # a lone token attends to itself with weight 1: O = V, so dV = dO and nothing else moves
        assert rel_l2(got[2].numpy(), a[3].float().numpy()) <= REL_L2_TOL
        assert got[0].abs().max() <= 1e-3 and got[1].abs().max() <= 1e-3
        return
    compare(gpu_grads(gpu, *a), reference_grads(*a), None, f"N={N}")


@pytest.mark.parametrize("H", [2, 32])          # (60 and 960 workgroups of 128 own tokens)
def test_masks(gpu, H):
    N = 300
    Q, K, V, dO, coords, sigma, _ = make(1, 5, H, N)
    g = torch.Generator().manual_seed(1)
    mask = torch.zeros(5, N, dtype=torch.bool)
    mask[0] = torch.rand(N, generator=g) < 0.5
    mask[1, 131:] = True
    mask[2] = True
    mask[3] = True
    mask[3, 77] = False
    mask[4, :64] = True
    a = (Q, K, V, dO, coords, sigma, mask)
    compare(gpu_grads(gpu, *a), reference_grads(*a), mask, "masks")


@pytest.mark.parametrize("H", [2, 4])           # (192 and 384 workgroups of 128 own tokens)
def test_ragged_batch_of_long_sequences(gpu, H):
    # N = 1024 (16 streamed tiles, 8 tiles of own tokens; a mask whose rows are multiples of 16 bytes): whole own tiles
    # of padding, which leave without streaming anything, and sequences whose last unpadded token sits in the first,
    # a middle and the last tile, where the streaming stops; one item padded in the middle only.
    N = 1024
    Q, K, V, dO, coords, sigma, _ = make(7, 6, H, N)
    mask = torch.zeros(6, N, dtype=torch.bool)
    mask[1, 700:] = True
    mask[2, 130:] = True
    mask[3, 64:] = True
    mask[4, 1:] = True
    mask[5, 300:600] = True
    a = (Q, K, V, dO, coords, sigma, mask)
    compare(gpu_grads(gpu, *a), reference_grads(*a), mask, "ragged N=1024")


@pytest.mark.parametrize("H", [3, 10])          # (216 and 720 workgroups of 128 own tokens)
def test_padded_batches_handed_out_longest_first(gpu, H):
    # The workgroups of a padded batch take the own tiles of the longest sequence first (up to 64 batch items): every
    # (item, head, own tile) must still be done exactly once.  Equal lengths, an empty item, lengths on and beside the
    # borders of the own tiles (128 or 64 tokens), a head count that does not divide 8, rows that are not multiples of 16 bytes.
    N = 400
    Q, K, V, dO, coords, sigma, _ = make(11, 9, H, N)
    mask = torch.zeros(9, N, dtype=torch.bool)
    for z, n in enumerate((400, 10, 400, 0, 129, 128, 257, 64, 65)):
        mask[z, n:] = True
    a = (Q, K, V, dO, coords, sigma, mask)
    compare(gpu_grads(gpu, *a), reference_grads(*a), mask, "longest first")
    if H != 3:
        return
    # more items than are ranked: the launch order is kept
    N = 130
    Q, K, V, dO, coords, sigma, _ = make(12, 66, 1, N)
    mask = torch.zeros(66, N, dtype=torch.bool)
    for z in range(66):
        mask[z, (z * 37) % 131:] = True
    a = (Q, K, V, dO, coords, sigma, mask)
    compare(gpu_grads(gpu, *a), reference_grads(*a), mask, "66 items")


# Ranked batches against their sequences one by one (which nothing ranks): lengths off 16, whose pieces of 16 mask bytes lie in two sequences, a mask off 16
# bytes, sequences without a token, with one, of equal length and with holes, as many as are ranked; the second row: too many workgroups of too short sequences, more sequences
# than a single round is ranked for, which are not
@pytest.mark.parametrize("Z,H,N,off", [(9, 2, 517, 0), (9, 2, 517, 3), (50, 6, 530, 0), (64, 1, 1504, 0), (64, 1, 1501, 9), (17, 2, 1507, 0), (2, 3, 1500, 0), (5, 8, 500, 0), (12, 7, 513, 0), (64, 1, 512, 0),
                                         (16, 8, 513, 0), (50, 1, 530, 0)])
def test_ranked_batches_equal_their_sequences(gpu, Z, H, N, off):
    g = torch.Generator(device=gpu).manual_seed(N + Z)
    Q, K, V = (torch.randn(Z, H, N, 32, generator=g, device=gpu).bfloat16() for _ in range(3))
    dO = torch.randn(Z, H, N, 32, generator=g, device=gpu)
    coords = torch.cumsum(torch.randn(Z, N, 3, generator=g, device=gpu) * 2, 1)
    sigma = torch.full((H,), 6.0, device=gpu)
    lens = [(0, 1, N, N, N // 2, 15, 16, 17, N - 1)[z % 9] if z < 9 else (z * 97) % (N + 1) for z in range(Z)]
    mask = torch.empty(Z * N + 16, dtype=torch.bool, device=gpu)[off:off + Z * N].view(Z, N)
    mask.copy_(torch.arange(N, device=gpu)[None] >= torch.tensor(lens, device=gpu)[:, None])
    mask[Z - 1, :N // 3] = True
    one = lambda z: slice(z, z + 1)
    O, L = pa.geo_attn(Q, K, V, coords, sigma, mask, return_lse=True)
    from proteusai_amd.geometric_attn import geo_attn_backward as back
    got = back(Q, K, V, O, L, dO, coords, sigma, mask)
    d_sigma = torch.zeros(H, device=gpu)
    for z in range(Z):
        want = back(Q[one(z)], K[one(z)], V[one(z)], O[one(z)], L[one(z)], dO[one(z)], coords[one(z)], sigma, mask[one(z)].clone())
        d_sigma += want[3]
        for a, b in zip(got[:3], want[:3]):
            # the same pairs and roundings; own tiles of 64 or 128 tokens add up in another order (2^-24 of some N terms)
            assert bool(((a[z] - b[0]).abs() <= 1e-4 * b.abs().max() + 1e-6).all()), (z, lens[z])
    assert float((got[3] - d_sigma).abs().max()) <= 1e-3 * float(d_sigma.abs().max()) + 1e-4


def test_backward_after_a_forward_that_cut_its_items_into_parts(gpu):
    # N > 2048 and few items: the operator's forward splits every item along the keys (parts merged through a
    # workspace) and hands the backward its O and logsumexp; masked as well (the long items of a padded batch)
    from proteusai_amd import _lib
    assert _lib.load().proteus_geo_attn_fwd_workspace_bytes(2, 2, 2304, 64, 0) > 0
    a = make(31, 2, 2, 2304)
    compare(gpu_grads(gpu, *a), reference_grads(*a), None, "unmasked, split forward")
    Q, K, V, dO, coords, sigma, _ = make(32, 3, 2, 2304)
    mask = torch.zeros(3, 2304, dtype=torch.bool)
    mask[0, 2200:] = True
    mask[1, 700:] = True
    mask[2, 1500:] = True
    a = (Q, K, V, dO, coords, sigma, mask)
    assert _lib.load().proteus_geo_attn_fwd_workspace_bytes(3, 2, 2304, 64, 0) > 0
    compare(gpu_grads(gpu, *a), reference_grads(*a), mask, "masked, split forward")


def test_padded_content_cannot_matter(gpu):
    Q, K, V, dO, coords, sigma, mask = make(2, 2, 4, 260, maskfrac=0.3)
    got = gpu_grads(gpu, Q, K, V, dO, coords, sigma, mask)
    Q2, K2, V2, dO2, c2 = Q.clone(), K.clone(), V.clone(), dO.clone(), coords.clone()
    pad = mask[:, None, :].expand(-1, 4, -1)
    for t in (Q2, K2, V2, dO2):
        t[pad] = float("nan")
    c2[mask] = float("nan")
    got2 = gpu_grads(gpu, Q2, K2, V2, dO2, c2, sigma, mask)
    for x, y, name in zip(got[:3], got2[:3], ("dQ", "dK", "dV")):
        assert torch.equal(x, y), name
    assert rel_l2(got2[3].numpy(), got[3].numpy()) <= 1e-5      # (atomic adds: summation order may differ)


def test_padded_keys_beside_queries_with_very_negative_logsumexp(gpu):
    """Every logit of a query around -120 (its logsumexp far below -88) and padded keys in the same key blocks: a
    padded key's score is 0, so exp(0 - L) overflows for it; nothing of that may reach d_sigma or d_beta."""
    Z, H, N = 1, 2, 200
    g = torch.Generator().manual_seed(17)
    Q = 0.05 * torch.randn(Z, H, N, 64, generator=g)
    K = 0.05 * torch.randn(Z, H, N, 64, generator=g)
    Q[..., 0] = 8.0
    K[..., 0] = -120.0
    Q, K = Q.bfloat16(), K.bfloat16()
    V = torch.randn(Z, H, N, 64, generator=g).bfloat16()
    dO = torch.randn(Z, H, N, 64, generator=g).bfloat16()
    coords = synth.random_walk_chain(N, g)[None]
    sigma = torch.tensor([6.0, 15.0])
    mask = torch.zeros(Z, N, dtype=torch.bool)
    mask[0, 150:] = True
    mask[0, 40:47] = True
    a = (Q, K, V, dO, coords, sigma, mask)

    def without_the_cancelling_component(grads):
        # dQ[..., 0] = -15 sum_j dS_ij, and the dS of a query sum to zero: that component is rounding noise times 15
        grads = list(grads)
        grads[0] = grads[0].clone()
        grads[0][..., 0] = 0
        return grads
    compare(without_the_cancelling_component(gpu_grads(gpu, *a)), without_the_cancelling_component(reference_grads(*a)), mask,
            "very negative logsumexp")
    betas = torch.tensor([0.7, -0.4])
    compare(without_the_cancelling_component(gpu_grads(gpu, *a, betas=betas)),
            without_the_cancelling_component(reference_grads(*a, betas=betas)), mask, "very negative logsumexp, beta-weighted logits")


def test_pairs_on_the_rbf_thresholds_are_in_range_in_both_passes_or_in_neither(gpu):
    """Tokens on an integer lattice: every pair at distance 4 has the same rbf, and min_rbf (or max_rbf) is put on it and
    one float above and below.  Whichever way the kernels round, the backward must rebuild the probabilities of exactly
    the pairs the forward's logsumexp counted: with dO = 1 the column sums of P land in dV, and they add up to the
    number of queries.  A pair kept by one pass and dropped by the other would move that sum by its probability."""
    Z, H, N = 1, 2, 96
    g = torch.Generator().manual_seed(23)
    Q = torch.randn(Z, H, N, 64, generator=g).bfloat16()
    K = torch.randn(Z, H, N, 64, generator=g).bfloat16()
    V = torch.randn(Z, H, N, 64, generator=g).bfloat16()
    coords = torch.zeros(Z, N, 3)
    coords[0, :, 0] = torch.arange(N, dtype=torch.float32)
    coords[0, :, 1] = 7.0
    sigma = torch.tensor([3.0, 3.0])
    betas = torch.tensor([0.5, -0.8])
    on_it = np.float32(np.exp(-16.0 / 18.0))
    dO = torch.ones(Z, H, N, 64).bfloat16()
    for kind in ("min", "max"):
        for thr in (np.nextafter(on_it, np.float32(0)), on_it, np.nextafter(on_it, np.float32(1))):
            lo, hi = (float(thr), 1.0) if kind == "min" else (0.0, float(thr))
            O, L = pa.geo_attn(Q.to(gpu), K.to(gpu), V.to(gpu), coords.to(gpu), sigma.to(gpu), None, return_lse=True,
                               betas=betas.to(gpu), min_rbf=lo, max_rbf=hi)
            grads = pa.geo_attn_backward(Q.to(gpu), K.to(gpu), V.to(gpu), O, L, dO.to(gpu), coords.to(gpu), sigma.to(gpu), None,
                                         betas=betas.to(gpu), min_rbf=lo, max_rbf=hi)
            torch.cuda.synchronize()
            rows_with_a_pair = torch.isfinite(L).sum(dim=2).double().cpu()          # [Z,H]
            col_sums = grads[2][..., 0].double().sum(dim=2).cpu()                 # sum_j dV[j][0] = sum_i sum_j P_ij
            assert (rows_with_a_pair > 0).all()
            assert ((col_sums - rows_with_a_pair).abs() <= 1e-2 * rows_with_a_pair).all(), (kind, float(thr), col_sums, rows_with_a_pair)


def test_tiles_skipped_below_min_rbf_hold_no_pair_in_range(gpu):
    """With a lower rbf bound the kernels skip key tiles (forward) and blocks (backward) that lie out of reach of a wave's
    tokens, where every pair is masked.  Here the tokens of the first tile sit in a tight cluster and the others on
    shells around it whose rbf against the cluster is min_rbf times 0.9, 0.99, 0.999, 1.001, 1.01 and 1.1 (shell by
    shell, so whole tiles are just out of or just in range): the logsumexp of the cluster's queries and the dK, dV rows
    of the shell tokens change by far more than the bar if a tile with pairs in range is dropped, or one without is kept."""
    Z, H, N = 1, 2, 64 + 6 * 64
    g = torch.Generator().manual_seed(29)
    Q = torch.randn(Z, H, N, 64, generator=g).bfloat16()
    K = torch.randn(Z, H, N, 64, generator=g).bfloat16()
    V = torch.randn(Z, H, N, 64, generator=g).bfloat16()
    dO = torch.randn(Z, H, N, 64, generator=g).bfloat16()
    sigma = torch.tensor([6.0, 9.0])
    betas = torch.tensor([0.7, -0.4])
    lo, hi = 0.01, 1.0
    coords = torch.zeros(Z, N, 3)
    coords[0, :64] = torch.randn(64, 3, generator=g) * 1e-5 + torch.tensor([4.0, -2.5, 1.0])
    for shell, f in enumerate((0.9, 0.99, 0.999, 1.001, 1.01, 1.1)):
        r = float(np.sqrt(-2.0 * 36.0 * np.log(lo * f)))                    # rbf(r) = lo * f for head 0 (sigma 6)
        d = torch.randn(64, 3, generator=g)
        coords[0, 64 + 64 * shell: 128 + 64 * shell] = coords[0, :64].mean(0) + r * d / d.norm(dim=1, keepdim=True)
    got = gpu_grads(gpu, Q, K, V, dO, coords, sigma, None, betas, lo, hi)
    ref = reference_grads(Q, K, V, dO, coords, sigma, None, betas, lo, hi)
    compare(got, ref, None, "shells around min_rbf")
    # row by row: a dropped or an extra tile changes whole rows of dK and dV
    for gg, rr, name in zip(got[1:3], ref[1:3], ("dK", "dV")):
        err = (gg.double() - rr).norm(dim=-1)
        assert (err <= 2e-2 * rr.norm(dim=-1) + 2e-2 * rr.norm(dim=-1).mean()).all(), f"{name} rows: {(err / rr.norm(dim=-1).mean()).max():.3e}"
    _, L = pa.geo_attn(Q.to(gpu), K.to(gpu), V.to(gpu), coords.to(gpu), sigma.to(gpu), None, return_lse=True,
                       betas=betas.to(gpu), min_rbf=lo, max_rbf=hi)
    _, Lref = torch_oracle.geo_attn_legacy_torch(Q.float(), K.float(), V.float(), coords, sigma, betas, None, lo, hi, dtype=torch.float64)
    assert (L.cpu().double() - Lref).abs().max() <= 4e-3, f"logsumexp {(L.cpu().double() - Lref).abs().max():.3e}"
    # and the cluster's queries do see exactly the three shells in range, beside the cluster itself (head 0)
    n_in = ((torch.cdist(coords[0, :64].double(), coords[0].double()) ** 2 / -72.0).exp() >= lo).sum(dim=1)
    assert (n_in == 64 + 3 * 64).all()


def test_large_logits(gpu):
    a = make(3, 1, 4, 400, qscale=2.5)
    compare(gpu_grads(gpu, *a), reference_grads(*a), None, "large logits")


def test_legacy_logits(gpu):
    Q, K, V, dO, coords, sigma, mask = make(4, 2, 4, 300, maskfrac=0.2)
    betas = torch.tensor([0.5, 1.0, 0.25, 2.0])
    for lo, hi in ((0.0, 1.0), (0.05, 0.9)):
        got = gpu_grads(gpu, Q, K, V, dO, coords, sigma, mask, betas, lo, hi)
        ref = reference_grads(Q, K, V, dO, coords, sigma, mask, betas, lo, hi)
        compare(got, ref, mask, f"legacy [{lo},{hi}]")


def test_gradients_are_deterministic_except_the_atomic_scalars(gpu):
    a = make(5, 1, 2, 500)
    x = gpu_grads(gpu, *a)
    y = gpu_grads(gpu, *a)
    for p, q in zip(x[:3], y[:3]):
        assert torch.equal(p, q)


def test_cfg3_shape_sampled(gpu):
    # Z=4, H=8, N=4096 would need a 4096^2 dense fp64 reference per head: check one batch item and two heads of
    # that shape in full, through the raw operator (heads and batch items are independent)
    Q, K, V, dO, coords, sigma, _ = make(6, 1, 2, 2048)
    compare(gpu_grads(gpu, Q, K, V, dO, coords, sigma, None), reference_grads(Q, K, V, dO, coords, sigma, None), None, "N=2048")


def test_full_length_sequence_every_gradient(gpu):
    # N = 16384 (the benchmark's sequence length: 256 tiles of streamed tokens per workgroup, both stages of the
    # direct-to-LDS staging reused 128 times) on the compacted chain, the narrowest and the widest head of the
    # benchmark's sigma range, against the tiled statement of the gradient formulas (pinned to torch.autograd on the CPU
    # in tests/test_oracle_attn.py; fp32 here, which differs from fp64 by 4e-7 in relative L2 at this size).
    wc, _ = synth.we_inputs(65536, seed=5, compact=True)
    Z, H, N = 1, 2, 16384
    Q, K, V, coords, sigma, _ = synth.attn_inputs(Z, H, N, 64, 5, coords=wc[:, :N].contiguous())
    g = torch.Generator().manual_seed(5)
    dO = (torch.randn(Z, H, N, 64, generator=g) / 8).bfloat16()
    got = gpu_grads(gpu, Q, K, V, dO, coords, sigma, None)
    rQ, rK, rV, rs, mass = torch_oracle.geo_attn_backward_tiled_torch(Q, K, V, dO, coords, sigma, None, row_chunk=1024,
                                                                      dtype=torch.float32)
    for gg, rr, name in zip(got[:3], (rQ, rK, rV), ("dQ", "dK", "dV")):
        assert torch.isfinite(gg).all(), f"N=16384 {name}: non-finite"
        e = rel_l2(gg.numpy(), rr.numpy())
        assert e <= REL_L2_TOL, f"N=16384 {name}: rel-L2 {e:.3e}"
    err = (got[3].double() - rs.double()).abs()
    assert (err <= SCALAR_TOL * mass.double()).all(), f"N=16384 d_sigma: error / pair mass {(err / mass.double()).max():.3e}"


def test_module_trains(gpu):
    torch.manual_seed(0)
    m = pa.GeoAttention(d_model=128, heads=2).to(gpu)
    x = torch.randn(2, 70, 128, device=gpu)
    coords = torch.stack([synth.random_walk_chain(70, torch.Generator().manual_seed(i)) for i in range(2)]).to(gpu)
    mask = torch.zeros(2, 70, dtype=torch.bool, device=gpu)
    mask[1, 50:] = True
    y = m(x, x, x, coords, mask)
    y[~mask].square().mean().backward()
    for name, p in m.named_parameters():
        if name == "beta_weights":
            continue
        assert p.grad is not None and torch.isfinite(p.grad).all(), name
    assert m.spread_weights.grad.abs().sum() > 0 and m.q_proj.grad.abs().sum() > 0


def test_strided_operands_give_the_same_gradients(gpu):
    """Operands as slices of a fused [Z,N,3,H,d] buffer, dO token-major: the strided entry point gives the
    bits of the contiguous one (the per-head scalars are atomic sums: compared to rounding)."""
    Z, H, N = 2, 2, 200
    Q, K, V, dO, coords, sigma, mask = make(41, Z, H, N, maskfrac=0.1)
    dev = lambda t: None if t is None else t.to(gpu)
    O, L = pa.geo_attn(dev(Q), dev(K), dev(V), dev(coords), dev(sigma), dev(mask), return_lse=True)
    ref = pa.geo_attn_backward(dev(Q), dev(K), dev(V), O, L, dev(dO).bfloat16(), dev(coords), dev(sigma), dev(mask))
    fused = torch.stack([t.permute(0, 2, 1, 3) for t in (Q, K, V)], dim=2).contiguous().to(gpu)
    Qs, Ks, Vs = (fused[:, :, i].permute(0, 2, 1, 3) for i in range(3))
    dOs = dev(dO).bfloat16().permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)
    Os = O.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)
    got = pa.geo_attn_backward(Qs, Ks, Vs, Os, L, dOs, dev(coords), dev(sigma), dev(mask))
    torch.cuda.synchronize()
    for name, x, y in zip(("dQ", "dK", "dV"), got[:3], ref[:3]):
        assert torch.equal(x, y), name
    assert torch.allclose(got[3], ref[3], rtol=1e-4, atol=1e-6)
    # a dense head-major operand gets its gradient in the same memory order
    Qh = dev(Q).permute(1, 0, 2, 3).contiguous().permute(1, 0, 2, 3)
    got2 = pa.geo_attn_backward(Qh, dev(K), dev(V), O, L, dev(dO).bfloat16(), dev(coords), dev(sigma), dev(mask))
    assert got2[0].stride() == Qh.stride() and torch.equal(got2[0], ref[0])


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_delta_rowsum_equals_the_torch_expression(gpu, d, dtype):
    """D = rowsum(O * dO) (old/old_scripts/attn/geometric_attn.py:618) from proteus_geo_attn_delta: contiguous tensors,
    token-major O with a differently laid out dO, and a slice of a wider buffer, against the fp64 sum of the same
    products (fp32 products and sums: rel-L2 <= 1e-6, every row within 1e-5 of its sum of absolute products)."""
    from proteusai_amd.geometric_attn import _delta
    Z, H, N = 2, 3, 777
    g = torch.Generator().manual_seed(d)
    O = torch.randn(Z, H, N, d, generator=g)
    dO = torch.randn(Z, H, N, d, generator=g).to(dtype)
    ref = (O.double() * dO.double()).sum(-1)
    scale = (O.double() * dO.double()).abs().sum(-1)

    def check(D, what):
        D = D.double().cpu()
        assert D.shape == (Z, H, N) and torch.isfinite(D).all(), what
        assert float((D - ref).norm() / ref.norm()) <= 1e-6, what
        assert bool(((D - ref).abs() <= 1e-5 * scale).all()), what
    check(_delta(O.to(gpu), dO.to(gpu)), "contiguous")
    # O token-major ([Z,N,H,d] in memory), dO contiguous
    Ot = O.permute(0, 2, 1, 3).contiguous().to(gpu).permute(0, 2, 1, 3)
    assert not Ot.is_contiguous()
    check(_delta(Ot, dO.to(gpu)), "token-major O")
    # both as slices of buffers with room behind every row
    wide_o = torch.zeros(Z, H, N, d + 8)
    wide_o[..., :d] = O
    wide_g = torch.zeros(Z, H, N, 2 * d, dtype=dtype)
    wide_g[..., :d] = dO
    check(_delta(wide_o.to(gpu)[..., :d], wide_g.to(gpu)[..., :d]), "sliced rows")
    # a layout the kernel does not take (rows off the 16-byte grid) falls back to the torch expression
    odd = torch.zeros(Z, H, N, d + 1)
    odd[..., 1:] = O
    check(_delta(odd.to(gpu)[..., 1:], dO.to(gpu)), "unaligned rows")


@pytest.mark.parametrize("legacy", [False, True])
def test_fused_projection_operator_equals_the_sliced_one(gpu, legacy):
    """geometric_attn_qkv on qkv [Z,N,3,H,d] against geometric_attn on its three slices (what autograd then pads
    and adds up): the same O, the same gradient of qkv to the bit (each element is one kernel result rounded once),
    the per-head scalars to the rounding of their atomic sums."""
    Z, H, N, d = 2, 3, 333, 64
    g = torch.Generator().manual_seed(77)
    base = torch.randn(Z, N, 3, H, d, generator=g).bfloat16()
    dO = torch.randn(Z, H, N, d, generator=g).bfloat16().to(gpu)
    coords = torch.stack([synth.random_walk_chain(N, g) for _ in range(Z)]).to(gpu)
    sigma = torch.tensor([3.0, 7.0, 15.0])
    betas = torch.tensor([0.3, 0.6, 1.1]) if legacy else None
    lo, hi = (0.01, 0.98) if legacy else (0.0, 1.0)
    mask = torch.zeros(Z, N, dtype=torch.bool)
    mask[1, 300:] = True
    res = []
    for fused in (True, False):
        qkv = base.clone().to(gpu).requires_grad_(True)
        s = sigma.clone().to(gpu).requires_grad_(True)
        b = None if betas is None else betas.clone().to(gpu).requires_grad_(True)
        if fused:
            O = pa.geometric_attn_qkv(qkv, coords, s, b, mask.to(gpu), lo, hi, out_dtype=torch.bfloat16)
        else:
            q, k, v = (qkv[:, :, i].permute(0, 2, 1, 3) for i in range(3))
            O = pa.geometric_attn(q, k, v, coords, s, b, mask.to(gpu), lo, hi, token_major_out=True, out_dtype=torch.bfloat16)
        assert O.dtype == torch.bfloat16 and O.permute(0, 2, 1, 3).is_contiguous()
        O.backward(dO)
        res.append((O.detach(), qkv.grad, s.grad, None if b is None else b.grad))
    (Oa, ga, sa, ba), (Ob, gb, sb, bb) = res
    assert torch.equal(Oa, Ob)
    assert ga.dtype == torch.bfloat16 and ga.shape == base.shape and torch.equal(ga, gb)
    assert ga.abs().sum() > 0
    assert torch.allclose(sa, sb, rtol=1e-4, atol=1e-7)
    if legacy:
        assert torch.allclose(ba, bb, rtol=1e-4, atol=1e-7)
