"""The fp32 product of the encoder's training step (proteus_gemm_f32) against float64, and what it refuses."""
import ctypes

import pytest
import torch

from proteusai_amd import _lib, train_ops

NN, NT, TN = _lib.GEMM_NN, _lib.GEMM_NT, _lib.GEMM_TN


def _operands(form, M, N, K, gpu):
    g = torch.Generator(device=gpu).manual_seed(M * 7919 + N * 31 + K)
    scale = torch.exp(3 * torch.randn(K, generator=g, device=gpu))             # terms of very different size
    A, B = torch.randn(M, K, generator=g, device=gpu) * scale, torch.randn(K, N, generator=g, device=gpu) / scale.flip(0)[:, None]
    return (A.t().contiguous() if form == TN else A), (B.t().contiguous() if form == NT else B), A.double() @ B.double(), A.double().abs() @ B.double().abs()


# Edges of the 64 x 64 tiles, of the steps of 16 k and of what 1, 2 and 4 groups share out (more than 512 tiles, 257 to 512, fewer);
# gradients of weights: 4, 2 and 8 waves (928 tiles: 2).
@pytest.mark.gpu
@pytest.mark.parametrize("form", [NN, NT, TN])
@pytest.mark.parametrize("M,N,K", [(1, 1, 4), (63, 65, 16), (64, 64, 20), (65, 36, 68), (130, 512, 132), (1, 20, 512), (1100, 1200, 36), (1700, 1600, 52), (2000, 1800, 20)])
def test_product_against_float64(gpu, form, M, N, K):
    if form == TN:
        K -= 3                                                                  # (rows along K need no multiple of 4)
    A, B, want, mass = _operands(form, M, N, K, gpu)
    got = train_ops._product(form, A, B)
    # six instructions per 16 k, each rounding a partial sum (at most the sum of magnitudes) once or, with its inner additions, twice;
    # 16 more for the groups' sums and the dropped pieces (3 x 2^-26 of every term)
    bound = (12 * ((K + 15) // 16) + 16) * 2.0 ** -24 * mass
    assert bool(((got - want).abs() <= bound).all())
    assert torch.equal(got, train_ops._product(form, A, B))


# Tiles of 128 x 128: from 160 of them and K = 512 on with two groups, with one from where those of 64 x 64 are more than 1536; edges of the tiles and of the steps that the groups share out (the last two: half empty, tiles of 64 x 64)
@pytest.mark.gpu
@pytest.mark.parametrize("form", [NN, NT])
@pytest.mark.parametrize("M,N,K", [(1920, 1280, 512), (2047, 1276, 516), (1921, 1284, 532), (257, 10244, 548), (20481, 116, 512), (2945, 2436, 512), (2817, 2492, 540), (129, 10244, 548), (20481, 4, 512)])
def test_wide_tiles_against_float64(gpu, form, M, N, K):
    A, B, want, mass = _operands(form, M, N, K, gpu)
    got = train_ops._product(form, A, B)
    # (as above)
    assert bool(((got - want).abs() <= (12 * ((K + 15) // 16) + 16) * 2.0 ** -24 * mass).all())
    assert torch.equal(got, train_ops._product(form, A, B))
    # ... and not further off than sixty-four columns at a time, which tiles of 64 x 64 do
    narrow = torch.cat([train_ops._product(form, A, (B[n:n + 64] if form == NT else B[:, n:n + 64]).contiguous()) for n in range(0, min(N, 256), 64)], 1)
    near, far = (got[:, :256] - want[:, :256]).norm(), (narrow - want[:, :256]).norm()
    assert float(near) <= 2.0 * float(far)          # (two chains over K for four: rounding errors that add up as sqrt(2), and some room)


# Gradients of weights cut along K: a tile in 7 and in 32 shares, few tiles, 64 of them in four shares, the last in a remainder, 128 in two and the first
# number of tiles that is not cut; nothing is cut where a share spares too little
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,shares", [(1, 4, 1792, 7), (64, 61, 8195, 17), (64, 64, 49150, 32), (64, 64, 50000, 28), (65, 130, 2050, 9), (512, 512, 2048, 4), (300, 320, 1801, 8), (500, 1000, 3072, 2),
                                          (513, 1000, 4096, 1), (64, 64, 1791, 1), (500, 1000, 3071, 1)])
def test_shares(gpu, M, N, K, shares):
    tiles = ((M + 63) // 64) * ((N + 63) // 64)
    assert _lib.load().proteus_gemm_f32_workspace_bytes(M, N, K, TN) == (tiles * shares * 16384 if shares > 1 else 0)
    A, B, want, mass = _operands(TN, M, N, K, gpu)
    got = train_ops._product(TN, A, B)
    # (as above, a rounding more per share)
    assert bool(((got - want).abs() <= (12 * ((K + 15) // 16) + 16 + shares) * 2.0 ** -24 * mass).all())
    assert torch.equal(got, train_ops._product(TN, A, B))


# Operands and results near the ends of fp32's range: pieces that would be smaller than bf16's smallest numbers, subnormal operands, operands and
# sums that leave the enlarged range (from 2^112 and 2^96 on)
@pytest.mark.gpu
@pytest.mark.parametrize("form", [NN, NT, TN])
@pytest.mark.parametrize("ea,eb", [(-112, 0), (-120, 0), (-126, 20), (-140, 60), (0, -120), (-60, -60), (115, -40), (40, 60), (111, -3)])
def test_magnitudes(gpu, form, ea, eb):
    M, N, K = 70, 68, 100
    g = torch.Generator(device=gpu).manual_seed(ea * 1000 + eb + 200000)
    A, B = (torch.randn(s, generator=g, device=gpu).clamp(-4, 4).mul(2.0 ** (e / 2)).mul(2.0 ** (e / 2)) for s, e in (((M, K), ea), ((K, N), eb)))
    want, mass = A.double() @ B.double(), A.double().abs() @ B.double().abs()
    got = train_ops._product(form, A.t().contiguous() if form == TN else A, B.t().contiguous() if form == NT else B)
    # (as in test_product_against_float64; plain sums round once per term; a subnormal result is a multiple of 2^-149)
    assert bool(((got - want).abs() <= (12 * 7 + 16) * 2.0 ** -24 * mass + 2.0 ** -149).all())


def _epilogue(form, epilogue, A, B, bias=None, h=None):
    """The entry point itself, with the matrices' sizes as in _product."""
    M, K = A.shape
    N = B.shape[0] if form == NT else B.shape[1]
    C = torch.empty(M, N, dtype=torch.bfloat16 if epilogue == _lib.GEMM_BF16 else torch.float32, device=A.device)
    train_ops._call("proteus_gemm_f32", A.device, A, B, bias, h, C, None, M, N, K, A.shape[1], B.shape[1], N, form, epilogue)
    return C


@pytest.mark.gpu
@pytest.mark.parametrize("M", [5, 700])
def test_epilogues(gpu, M):
    A, B, want, mass = _operands(NT, M, 132, 72, gpu)
    Bt, bias, h = B.t().contiguous(), torch.randn(132, device=gpu), torch.randn(M, 132, device=gpu)
    bound = 76 * 2.0 ** -24 * mass + 2.0 ** -23 * bias.abs()
    H, C = train_ops._product(NT, A, B, bias, gelu=True)
    assert bool(((H - want - bias).abs() <= bound).all())
    # (erff is good to 2 ulp; gelu of the kernel's own sums)
    exact = torch.nn.functional.gelu(H.double())
    assert bool(((C - exact).abs() <= 2.0 ** -21 * H.abs()).all())
    hd = h.double().requires_grad_(True)
    grad, = torch.autograd.grad(torch.nn.functional.gelu(hd).sum(), hd)
    plain = train_ops._product(NN, A, Bt, bias)
    assert bool(((plain - want - bias).abs() <= bound).all())
    assert bool(((train_ops._product(NN, A, Bt, bias, gelu_grad_of=h) - plain.double() * grad).abs() <= 2.0 ** -20 * plain.abs() * (1 + h.abs())).all())
    assert torch.equal(_epilogue(NN, _lib.GEMM_BF16, A, Bt, bias), plain.to(torch.bfloat16))
    assert torch.equal(_epilogue(NN, _lib.GEMM_ADD, A, Bt, None, h), train_ops._product(NN, A, Bt) + h)
    assert torch.equal(_epilogue(NT, _lib.GEMM_ADD, A, B, bias, h), train_ops._product(NT, A, B, bias) + h)


# (tiles of 128 x 128, with two groups; with one where the epilogue reads no matrix; but with GELU's derivative; with one)
@pytest.mark.gpu
@pytest.mark.parametrize("M,N", [(2049, 1804), (3457, 3204), (3457, 4228), (3969, 4092)])
def test_epilogues_of_wide_tiles(gpu, M, N):
    A, B, want, mass = _operands(NT, M, N, 524, gpu)
    Bt, bias, h = B.t().contiguous(), torch.randn(N, device=gpu), torch.randn(M, N, device=gpu)
    bound = (12 * 33 + 16) * 2.0 ** -24 * mass + 2.0 ** -23 * bias.abs()
    H, C = train_ops._product(NT, A, B, bias, gelu=True)
    assert bool(((H - want - bias).abs() <= bound).all())
    assert bool(((C - torch.nn.functional.gelu(H.double())).abs() <= 2.0 ** -21 * H.abs()).all())
    hd = h.double().requires_grad_(True)
    grad, = torch.autograd.grad(torch.nn.functional.gelu(hd).sum(), hd)
    plain = train_ops._product(NN, A, Bt, bias)
    assert bool(((plain - want - bias).abs() <= bound).all())
    assert bool(((train_ops._product(NN, A, Bt, bias, gelu_grad_of=h) - plain.double() * grad).abs() <= 2.0 ** -20 * plain.abs() * (1 + h.abs())).all())
    assert torch.equal(_epilogue(NN, _lib.GEMM_BF16, A, Bt, bias), plain.to(torch.bfloat16))
    assert torch.equal(_epilogue(NN, _lib.GEMM_ADD, A, Bt, None, h), train_ops._product(NN, A, Bt) + h)
    assert torch.equal(_epilogue(NT, _lib.GEMM_ADD, A, B, bias, h), train_ops._product(NT, A, B, bias) + h)
    A[M - 1, 523] = float("nan")
    B[N - 1, 0] = float("nan")
    hit = torch.zeros_like(plain, dtype=torch.bool)
    hit[M - 1], hit[:, N - 1] = True, True
    got, clean = train_ops._product(NT, A, B), train_ops._product(NN, A, Bt)
    assert torch.equal(got.isnan(), hit) and bool(((got - want).abs()[~hit] <= bound[~hit]).all()) and torch.equal(clean[:M - 1].isnan(), torch.zeros_like(hit[:M - 1]))


@pytest.mark.gpu
@pytest.mark.parametrize("form,K", [(NN, 68), (NT, 68), (TN, 68), (TN, 2100)])
def test_a_diverged_operand(gpu, form, K):
    A, B, want, _ = _operands(form, 130, 132, K, gpu)
    clean = train_ops._product(form, A, B)
    (A if form != TN else A.t())[66, 67] = float("nan")
    (B if form == NT else B.t())[131, 0] = float("nan")
    got = train_ops._product(form, A, B)
    hit = torch.zeros_like(got, dtype=torch.bool)
    hit[66], hit[:, 131] = True, True
    assert torch.equal(got.isnan(), hit) and torch.equal(got[~hit], clean[~hit])


@pytest.mark.gpu
@pytest.mark.parametrize("form,K", [(NN, 4), (NT, 4), (TN, 1), (TN, 2), (TN, 3), (TN, 5), (TN, 16)])
def test_a_diverged_operand_is_read_to_its_end(gpu, form, K):
    # NaN right behind either operand: an element that is infinite must not be taken for one whose row or column holds a NaN
    M, N = 40, 36
    def guarded(rows, cols, seed):
        t = torch.rand(rows + 8, cols, generator=torch.Generator().manual_seed(seed)).to(gpu)
        t[rows:] = float("nan")
        return t[:rows]
    A = guarded(K, M, 1) if form == TN else guarded(M, K, 1)
    B = guarded(N, K, 2) if form == NT else guarded(K, N, 2)
    clean = train_ops._product(form, A, B)
    want = (A.double() if form != TN else A.double().t()) @ (B.double() if form != NT else B.double().t())
    assert bool(((clean - want).abs() <= 28 * 2.0 ** -24 * want).all())                       # (positive terms; as in test_product_against_float64)
    (A if form != TN else A.t())[7, K - 1] = float("inf")
    got = train_ops._product(form, A, B)
    assert bool((got[7] == float("inf")).all())
    rest = torch.arange(M, device=gpu) != 7
    assert torch.equal(got[rest], clean[rest])


# (gradients of weights: 8, 4 and 2 waves per tile, and shares of K)
@pytest.mark.gpu
@pytest.mark.parametrize("form,M,N,K", [(NN, 70, 68, 36), (NT, 70, 68, 36), (NN, 1700, 1600, 36), (NT, 1100, 1200, 36), (NN, 2047, 1276, 516), (NT, 2945, 2436, 512), (TN, 70, 68, 36), (TN, 70, 68, 2100), (TN, 1100, 1000, 37), (TN, 2000, 1800, 38)])
def test_values_that_do_not_split(gpu, form, M, N, K):
    A, B, _, _ = _operands(NN, M, N, K, gpu)
    bad = [(3, 5, float("inf")), (7, 1, float("nan")), (9, 2, 3.4e38), (11, 3, -3.39e38)]      # (bf16 ends at 3.39e38)
    bad += [(M - 1 - m, K - 1 - k, v) for m, k, v in bad] + [(M // 2 + m, K // 2 + k, -v) for m, k, v in bad]
    for m, k, v in bad:
        A[m, k] = v
    got = train_ops._product(form, A.t().contiguous() if form == TN else A, B.t().contiguous() if form == NT else B)
    want, mass = A.double() @ B.double(), A.double().abs() @ B.double().abs()
    # (what fp32 cannot hold: an infinity, or what a plain sum makes of infinities of both signs on its way)
    fits = mass <= torch.finfo(torch.float32).max
    assert torch.equal(got.isnan() & fits, want.isnan() & fits) and bool((got[want.isnan()].isnan()).all())
    infinite = want.isinf()
    assert torch.equal(got[infinite].double(), want[infinite])
    # (plain sums round once per term)
    assert bool(((got - want).abs()[fits] <= (12 * ((K + 15) // 16) + 16 + K) * 2.0 ** -24 * mass[fits]).all())
    assert not bool(got[fits].isinf().any())


def test_what_it_refuses():
    lib = _lib.load()
    at = ctypes.c_void_p(4096)

    def call(A=at, B=at, C=at, h=None, H=None, M=8, N=8, K=8, lda=8, ldb=8, ldc=8, form=NN, epilogue=0):
        return lib.proteus_gemm_f32(A, B, None, h, C, H, M, N, K, lda, ldb, ldc, form, epilogue, None)
    null, unsupported = call(A=None), call(form=3)
    assert null < 0 and unsupported < 0 and null != unsupported
    assert call(C=None) == call(form=NT, epilogue=_lib.GEMM_GELU) == call(epilogue=_lib.GEMM_GELU_GRAD) == call(epilogue=_lib.GEMM_ADD) == null
    # unknown ones, and combinations that the training step does not ask for
    assert call(epilogue=5, h=at, H=at) == call(epilogue=-1, h=at, H=at) == unsupported
    for form, epilogue in ((NN, _lib.GEMM_GELU), (NT, _lib.GEMM_BF16), (NT, _lib.GEMM_GELU_GRAD), (TN, _lib.GEMM_BF16), (TN, _lib.GEMM_GELU), (TN, _lib.GEMM_GELU_GRAD), (TN, _lib.GEMM_ADD)):
        assert call(form=form, epilogue=epilogue, h=at, H=at) == unsupported, (form, epilogue)
    assert call(M=0) < 0 and call(K=6, lda=8) < 0 and call(lda=6) < 0 and call(ldc=4) < 0 and call(form=NT, ldb=10) < 0
    assert call(A=ctypes.c_void_p(4100)) < 0
    assert call(M=1 << 28, lda=8) < 0                                           # (2 GiB and more)
    assert lib.proteus_gemm_f32_ws(at, at, None, None, at, None, 8, 8, 4096, 8, 8, 8, TN, 0, ctypes.c_void_p(4100), 1 << 30, None) < 0      # (the workspace's alignment)
    size = lib.proteus_gemm_f32_workspace_bytes
    assert size(64, 64, 4096, TN) > 0 and size(64, 64, 4096, NN) == size(0, 64, 4096, TN) == size(64, 64, 1 << 30, TN) == 0
