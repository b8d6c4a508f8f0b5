"""Pairs that no cell of the distance grids takes (closer than half a cell; anisotropic: r - c A below half a cell): the workgroups' lists of them
at the sizes where a list is short, nearly full (304 pairs per wave of 16, 608 of 8), over-full, and filled from several waves' sources; and the
units in which the sums are dealt out: 64, 128 and (isotropic) 256 wavenumbers."""
import numpy as np
import pytest
import torch

from oracle import c_oracle
from proteusai_amd import synth
from test_we_grid_gpu import rel_l2, run_aniso, run_grid

pytestmark = pytest.mark.gpu


def _clusters(Z, N, size, shuffled):
    """Tokens in places of `size` tokens, 0.03 angstrom apart; side by side in the sequence, or dealt out over it."""
    anchors, _ = synth.we_inputs((N + size - 1) // size, seed=size + N, batch=Z)
    g = torch.Generator().manual_seed(size)
    a = anchors.repeat_interleave(size, 1)[:, :N] + 0.03 * torch.randn(Z, N, 3, generator=g)
    return a[:, torch.randperm(N, generator=g)] if shuffled else a


# 16 observers of one place find 16 (size - 1) pairs in one wave's sources: 304 are 19 of them and 608 are 38
@pytest.mark.parametrize("shuffled", [False, True])
@pytest.mark.parametrize("size", [2, 20, 21, 39, 40, 300])
@pytest.mark.parametrize("Z,N,K", [(1, 1100, 80), (1, 4100, 80), (8, 1100, 80), (8, 1100, 330), (1, 4100, 250)])
def test_isotropic(gpu, Z, N, K, size, shuffled):
    a, wn = _clusters(Z, N, size, shuffled), synth.wavenumbers(2 * K)
    got = run_grid(gpu, a, wn)
    rows = np.unique(np.concatenate([np.arange(0, N, 97), [15, 16, N - 1]])).astype(np.int32)
    ref = c_oracle.we(a.numpy(), wn.numpy(), None, precision="f64", rows=rows)
    # (the bar of the other sizes: aliasing and fixed point of the grid, a phase rounded to 2^-24 of itself, twice)
    bar = 1.7e-6 + 2 * 2.0 ** -24 * float(wn.max()) * float((a.amax(1) - a.amin(1)).norm(dim=-1).max())
    for x, r, what in zip(got, ref, ("out", "cos_sums", "sin_sums")):
        assert rel_l2(x[:, rows], r) <= bar, (what, rel_l2(x[:, rows], r), bar)
    assert all(np.array_equal(x, y) for x, y in zip(got, run_grid(gpu, a, wn)))


@pytest.mark.parametrize("spread", [0.0, 0.02])
@pytest.mark.parametrize("size,shuffled", [(2, True), (21, False), (40, True), (300, False)])
@pytest.mark.parametrize("Z,N,K", [(1, 1100, 80), (8, 1100, 80), (8, 1100, 200)])
def test_anisotropic(gpu, Z, N, K, size, shuffled, spread):
    a, wn = _clusters(Z, N, size, shuffled), synth.wavenumbers(2 * K)
    g = torch.Generator().manual_seed(N)
    b = torch.randn(Z, N, 3, generator=g)
    b = 1.5 * b / b.norm(dim=-1, keepdim=True)
    cb = 1.0 + spread * torch.randn(K, generator=g)
    rows = np.unique(np.concatenate([np.arange(0, N, 97), [15, 16, N - 1]])).astype(np.int32)
    ref = c_oracle.we_aniso(a.numpy(), b.numpy(), cb.numpy(), wn.numpy(), None, rows=rows)
    # (the isotropic bar and 3e-7 for the terms left out of the expansion)
    bar = 2e-6 + 2 * 2.0 ** -24 * float(wn.max()) * float((a.amax(1) - a.amin(1)).norm(dim=-1).max())
    for partials in (True, False):
        got = run_aniso(gpu, a, b, cb, wn, None, partials=partials)
        for x, r, what in zip(got, ref, ("out", "d_cb", "d_k")):
            assert rel_l2(x[:, rows], r) <= bar, (what, rel_l2(x[:, rows], r), bar)
        assert all(np.array_equal(x, y) for x, y in zip(got, run_aniso(gpu, a, b, cb, wn, None, partials=partials)))
