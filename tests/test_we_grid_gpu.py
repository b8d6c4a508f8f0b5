"""The embedding forward through distance grids (proteus_we_fwd_ws with a workspace) against the float64 oracle, at the
sizes where it can go wrong: tiles of 16 observers, flushes after 2048 sources, octave and window borders of the grid,
pairs closer than half a cell, coordinates that are not finite."""
import numpy as np
import pytest
import torch

from oracle import c_oracle
from proteusai_amd import _lib, synth

pytestmark = pytest.mark.gpu


def run_grid(gpu, coords, wn, mask=None, sums=True, layout=_lib.COORDS_AOS):
    lib = _lib.load()
    Z, N, K = coords.shape[0], coords.shape[1] if layout == _lib.COORDS_AOS else coords.shape[2], wn.numel()
    c, w = coords.to(gpu), wn.to(gpu)
    m = None if mask is None else mask.to(gpu).view(torch.uint8)
    bufs = [torch.full(s, float("nan"), device=gpu) for s in ((Z, N, 2 * K), (Z, N, K), (Z, N, K))]
    nbytes = lib.proteus_we_fwd_workspace_bytes(Z, max(N, 1024), max(K, 64), 0)      # (the size grows with N and K)
    ws = torch.full((nbytes,), 0xA5, dtype=torch.uint8, device=gpu)
    rc = lib.proteus_we_fwd_ws(c.data_ptr(), layout, w.data_ptr(), None if m is None else m.data_ptr(), bufs[0].data_ptr(),
                               bufs[1].data_ptr() if sums else None, bufs[2].data_ptr() if sums else None, ws.data_ptr(), nbytes,
                               Z, N, K, 0, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.proteus_strerror(rc)
    torch.cuda.synchronize()
    return [b.cpu().numpy() for b in bufs[:3 if sums else 1]]


def rel_l2(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    nb = np.linalg.norm(b)
    return float(np.linalg.norm(a - b) / nb) if nb > 0 else float(np.linalg.norm(a - b))


CASES = {                       # N, Z, K, scale of the chain, mask
    "one tile": (16, 1, 16, 1.0, None),
    "tile and a bit, odd K": (17, 3, 37, 1.0, None),
    "two tokens": (2, 2, 5, 1.0, None),
    "half a flush": (1024, 1, 64, 1.0, None),
    "half a flush and a source": (1025, 1, 64, 1.0, None),
    "as many sources as need no flush": (2048, 1, 64, 1.0, None),
    "flushes, one source": (2049, 1, 64, 1.0, None),
    "scattered mask, more than 256 workgroups": (2100, 2, 20, 1.0, "scattered"),
    "flushes, scattered mask": (3600, 1, 20, 1.0, "scattered"),
    "flushes, more than 256 workgroups, an odd number of tiles": (3600, 2, 37, 1.0, "scattered"),
    "tail masks, empty item, lone survivor": (333, 4, 48, 1.0, "tail"),
    "large K": (70, 1, 300, 1.0, None),
    "many pairs closer than half a cell": (200, 1, 64, 0.05, None),
    "all pairs closer than half a cell": (60, 2, 40, 0.005, None),
    "several windows of the grid": (700, 2, 33, 30.0, None),
    "several windows, scattered mask": (1500, 1, 16, 20.0, "scattered"),
    "flushes, windows": (3600, 1, 64, 5.0, None),
    "flushes, windows, more than 256 workgroups": (2500, 2, 64, 5.0, None),
    "beyond the windows": (90, 1, 33, 3000.0, None),
    # sums without the grid: tiles of wavenumbers shared out over workgroups and over the waves of one
    "beyond the windows, 250 wavenumbers, an empty item": (333, 4, 250, 900.0, "tail"),
    "beyond the windows, more than 256 workgroups": (130, 32, 72, 3000.0, "scattered"),
    "windows that cost more than the pairs": (1100, 1, 64, 25.0, "scattered"),
    "windows that cost more than the pairs, more than 256 workgroups": (1100, 4, 112, 25.0, None),
    "everything in a cell or two": (500, 2, 64, 0.002, "scattered"),
    "everything in a cell or two, more than 256 workgroups": (300, 16, 16, 0.002, None),
}


@pytest.mark.parametrize("name", CASES)
def test_grid_matches_the_oracle(gpu, name):
    N, Z, K, scale, kind = CASES[name]
    coords, _ = synth.we_inputs(N, seed=N + K, batch=Z)
    coords = coords * scale
    if N > 50:
        coords[0, 40] = coords[0, 12]                          # a coincident pair is dropped like the observer itself
        coords[0, 20] = coords[0, 30] + torch.tensor([0.01, -0.02, 0.015])      # and one that is merely very close is not
    g = torch.Generator().manual_seed(K)
    wn = synth.wavenumbers(2 * K) * torch.where(torch.rand(K, generator=g) < 0.3, -1.0, 1.0)
    mask = None
    if kind == "scattered":
        mask = torch.rand(Z, N, generator=g) < 0.35
    elif kind == "tail":
        mask = torch.arange(N)[None, :] >= torch.tensor([N, 100, 0, 1])[:, None]
    junk = coords.clone()
    if mask is not None:
        junk[mask] = float("nan")                              # what padded positions hold reaches nothing
    got = run_grid(gpu, junk, wn, mask)
    ref = c_oracle.we(coords.numpy(), wn.numpy(), None if mask is None else mask.numpy(), precision="f64")
    # Bar: 4 x the aliasing error of the grid (2.2e-7) and of its fixed-point sums (2e-7), plus what single precision makes of a
    # phase k r: the distance and (in the direct sums) the phase are each rounded to 2^-24 of themselves, at most k_max times
    # the largest distance.
    c = coords if mask is None else coords.masked_fill(mask[..., None], 0.0)
    far = float((c.amax(1) - c.amin(1)).norm(dim=-1).max())
    bar = 1.7e-6 + 2 * 2.0 ** -24 * float(wn.abs().max()) * far
    sources = N if mask is None else int((~mask).sum(1).max())
    assert ("flushes" in name) == (sources > 2048), sources
    if "flushes, windows" in name:        # 1117 cells of pi / (3.5 k_max) are a window; up to five, which cost less than the pairs
        assert 1117 < 0.5 * far * float(wn.abs().max()) * 3.5 / np.pi and far * float(wn.abs().max()) * 3.5 / np.pi < 5 * 1117, far
    for a, r, what in zip(got, ref, ("out", "cos_sums", "sin_sums")):
        assert np.isfinite(a).all(), f"{name}: {what}"
        if mask is not None:
            assert (a[mask.numpy()] == 0).all(), f"{name}: {what} of padded rows"
        assert rel_l2(a, r) <= bar, f"{name}: {what} {rel_l2(a, r):.3e} (bar {bar:.1e})"
    again = run_grid(gpu, junk, wn, mask)
    lean = run_grid(gpu, junk, wn, mask, sums=False)
    assert all(np.array_equal(a, b) for a, b in zip(got, again)) and np.array_equal(got[0], lean[0])
    soa = run_grid(gpu, junk.transpose(1, 2).contiguous(), wn, mask, layout=_lib.COORDS_SOA)
    assert all(np.array_equal(a, b) for a, b in zip(got, soa))


def test_values_that_are_not_finite_come_through(gpu):
    # as in the direct kernels: an unpadded token at NaN makes every sum of its batch item NaN and touches no other item
    coords, wn = synth.we_inputs(200, seed=5, batch=2, d_model=128)
    coords[1, 77, 1] = float("nan")
    got = run_grid(gpu, coords, wn)
    ref = c_oracle.we(coords[:1].numpy(), wn.numpy(), precision="f64")
    for a, r in zip(got, ref):
        assert np.isnan(a[1]).all() and rel_l2(a[0], r[0]) <= 1e-5
    bad = wn.clone()
    bad[3] = float("nan")
    assert np.isnan(run_grid(gpu, coords[:1], bad)[0][:, :, 6:8]).all()


def test_distances_whose_scaled_squares_overflow(gpu):
    # a token 1e17 away (its square fits in fp32, that of 4096 times it does not) adds next to nothing, as in the direct kernels
    coords, wn = synth.we_inputs(200, seed=5, batch=2, d_model=128)
    near = coords[1:].clone()
    coords[1, 77, 1] = 1e17
    got = run_grid(gpu, coords, wn)
    keep = np.arange(200) != 77
    ref = c_oracle.we(near[:, keep].numpy(), wn.numpy(), precision="f64")[0]
    assert all(np.isfinite(a).all() for a in got) and np.abs(got[0][1, 77]).max() <= 200 * 1.001e-17
    # the bar of the values that are not finite: single-precision phases of a short chain
    assert rel_l2(got[0][1:, keep], ref) <= 1e-5


def run_aniso(gpu, a, b, cb, wn, mask=None, partials=True):
    lib = _lib.load()
    Z, N, K = a.shape[0], a.shape[1], wn.numel()
    a, b, cb, w = a.to(gpu), b.to(gpu), cb.to(gpu), wn.to(gpu)
    m = None if mask is None else mask.to(gpu).view(torch.uint8)
    bufs = [torch.full((Z, N, 2 * K), float("nan"), device=gpu) for _ in range(3)]
    nbytes = lib.proteus_we_aniso_fwd_workspace_bytes(Z, max(N, 4096), max(K, 64), 1, 0, 0)
    ws = torch.full((nbytes,), 0xA5, dtype=torch.uint8, device=gpu)
    rc = lib.proteus_we_aniso_fwd_ws(a.data_ptr(), b.data_ptr(), _lib.COORDS_AOS, cb.data_ptr(), w.data_ptr(), None if m is None else m.data_ptr(),
                                     bufs[0].data_ptr(), bufs[1].data_ptr() if partials else None, bufs[2].data_ptr() if partials else None,
                                     ws.data_ptr(), nbytes, Z, N, K, 0, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.proteus_strerror(rc)
    torch.cuda.synchronize()
    return [t.cpu().numpy() for t in bufs[:3 if partials else 1]]


ANISO = {                       # N, Z, K, scale of the chain, spread of the C-beta scales around 1, mask
    "equal scales": (700, 1, 64, 1.0, 0.0, None),
    "equal scales, scattered mask": (2100, 2, 20, 1.0, 0.0, "scattered"),
    "equal scales, flushes, scattered mask": (3600, 1, 20, 1.0, 0.0, "scattered"),
    "equal scales, several windows": (300, 2, 20, 60.0, 0.0, None),
    "four terms, an empty item, a lone survivor": (1100, 4, 256, 1.0, 0.01, "tail"),
    "ten terms and flushes": (2100, 2, 256, 1.0, 0.2, None),
    "two grids in several windows": (2100, 2, 256, 3.0, 0.02, "scattered"),
    "many pairs too close for a cell": (1300, 3, 256, 0.3, 0.02, None),
    "more terms than pay": (200, 2, 64, 1.0, 1.5, None),
    "more than 256 wavenumbers": (1500, 1, 300, 1.0, 0.02, None),
    "more than 256 items of two boxes": (70, 300, 64, 1.0, 0.0, None),
    "equal scales, more than 256 workgroups": (4200, 1, 64, 1.0, 0.0, None),
    "at most 256 workgroups, flushes, tiles of few terms, a tile in part": (2100, 1, 250, 1.0, 0.1, None),
}


@pytest.mark.parametrize("name", ANISO)
def test_anisotropic_grids_match_the_oracle(gpu, name):
    N, Z, K, scale, spread, kind = ANISO[name]
    a, _ = synth.we_inputs(N, seed=N + K, batch=Z)
    a = a * scale
    a[0, 40] = a[0, 12]
    g = torch.Generator().manual_seed(K + N)
    b = torch.randn(Z, N, 3, generator=g)
    b = 1.5 * b / b.norm(dim=-1, keepdim=True)
    b[:, 0] = 0.0
    cb = 1.0 + spread * torch.randn(K, generator=g)
    wn = synth.wavenumbers(2 * K) * torch.where(torch.rand(K, generator=g) < 0.3, -1.0, 1.0)
    mask = None
    if kind == "scattered":
        mask = torch.rand(Z, N, generator=g) < 0.35
    elif kind == "tail":
        mask = torch.arange(N)[None, :] >= torch.tensor([N, 500, 0, 1])[:, None]
    rows = None if N <= 512 else np.unique(np.concatenate([np.arange(0, N, 41), [15, 16, 1023, 1024, N - 1]]))
    rows = None if rows is None else rows[rows < N].astype(np.int32)
    got = run_aniso(gpu, a, b, cb, wn, mask)
    ref = c_oracle.we_aniso(a.numpy(), b.numpy(), cb.numpy(), wn.numpy(), None if mask is None else mask.numpy(), rows=rows)
    sel = slice(None) if rows is None else rows
    # the bar of the isotropic grids, plus 3e-7 for the terms left out of the expansion
    c = a if mask is None else a.masked_fill(mask[..., None], 0.0)
    far = float((c.amax(1) - c.amin(1)).norm(dim=-1).max())
    bar = 2e-6 + 2 * 2.0 ** -24 * float(wn.abs().max()) * far
    for x, r, what in zip(got, ref, ("out", "d_cb", "d_k")):
        assert np.isfinite(x).all(), f"{name}: {what}"
        if mask is not None:
            assert (x[mask.numpy()] == 0).all(), f"{name}: {what} of padded rows"
        assert rel_l2(x[:, sel], r) <= bar, f"{name}: {what} {rel_l2(x[:, sel], r):.3e} (bar {bar:.1e})"
    if "equal scales, flushes" in name:                     # (a single grid is flushed after 2048 sources, two after 1024)
        assert int((~mask).sum(1).max()) > 2048
    again = run_aniso(gpu, a, b, cb, wn, mask)
    assert all(np.array_equal(x, y) for x, y in zip(got, again))
    lean = run_aniso(gpu, a, b, cb, wn, mask, partials=False)[0]
    assert np.isfinite(lean).all() and rel_l2(lean[:, sel], ref[0]) <= bar


def test_weights_that_fall_below_half_a_unit(gpu):
    # equal C-beta scales: r - cb A may be a small part of r, and with it every fixed-point weight of the pair.  In a ball of three
    # angstrom some hundred thousand pairs lie near the outer edge of the first cell with r four to five times that.
    N, K = 2100, 64
    g = torch.Generator().manual_seed(11)
    a = torch.randn(1, N, 3, generator=g)
    a = 3.0 * a / a.norm(dim=-1, keepdim=True) * torch.rand(1, N, 1, generator=g) ** (1 / 3)
    b = torch.randn(1, N, 3, generator=g)
    b = 1.8154 * b / b.norm(dim=-1, keepdim=True)
    cb, wn = torch.ones(K), synth.wavenumbers(2 * K)
    got = run_aniso(gpu, a, b, cb, wn, partials=False)[0]
    ref = c_oracle.we_aniso(a.numpy(), b.numpy(), cb.numpy(), wn.numpy(), None, rows=np.arange(N, dtype=np.int32))[0]
    # the bar of the anisotropic grids, row by row: one pair's cell that is off by 2^31 units changes a row by 100 times its norm
    err = np.linalg.norm(got - ref, axis=-1) / np.linalg.norm(ref, axis=-1)
    assert err.max() <= 4 * (2e-6 + 2 * 2.0 ** -24 * float(wn.max()) * 6.0), err.max()


def run_aniso_route(gpu, a, b, cb, wn, mask=None, partials=True):
    """The results, and the terms of the expansion that the device chose (0: the direct kernel did the work)."""
    lib = _lib.load()
    Z, N, K = a.shape[0], a.shape[1], wn.numel()
    a, b, cb, w = a.to(gpu), b.to(gpu), cb.to(gpu), wn.to(gpu)
    m = None if mask is None else mask.to(gpu).view(torch.uint8)
    bufs = [torch.full((Z, N, 2 * K), float("nan"), device=gpu) for _ in range(3 if partials else 1)]
    nbytes = lib.proteus_we_aniso_fwd_workspace_bytes(Z, N, K, int(partials), int(mask is not None), 0)
    assert nbytes > 0
    ws = torch.full((nbytes,), 0xA5, dtype=torch.uint8, device=gpu)
    rc = lib.proteus_we_aniso_fwd_ws(a.data_ptr(), b.data_ptr(), _lib.COORDS_AOS, cb.data_ptr(), w.data_ptr(), None if m is None else m.data_ptr(),
                                     bufs[0].data_ptr(), *([t.data_ptr() for t in bufs[1:]] if partials else [None, None]),
                                     ws.data_ptr(), nbytes, Z, N, K, 0, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.proteus_strerror(rc)
    return [t.cpu().numpy() for t in bufs], int(ws[16:20].view(torch.int32).item())


ROUTES = {                      # N, Z, K, scale of the chain, spread of the C-beta scales, partial derivatives, kind, through grids?
    "one grid in several windows": (2000, 1, 64, 10.0, 0.0, False, None, True),
    "one grid in more windows than pay": (2000, 1, 64, 40.0, 0.0, False, None, False),
    "one grid in more windows than pay, more than 256 workgroups": (1000, 8, 64, 40.0, 0.0, False, None, False),
    "more windows than there are": (1000, 1, 256, 3000.0, 0.0, False, None, False),
    "items in frames of their own": (2000, 2, 256, 1.0, 0.02, True, "frames", True),
    "the first item empty": (2000, 3, 256, 1.0, 0.02, True, "first empty", True),
    "a token that is not finite": (1000, 2, 256, 1.0, 0.0, False, "nan", False),
    "more items than lanes of a block share": (300, 40, 256, 1.0, 0.0, False, "scattered", True),
}


@pytest.mark.parametrize("name", ROUTES)
def test_anisotropic_grids_where_they_pay(gpu, name):
    N, Z, K, scale, spread, partials, kind, grids = ROUTES[name]
    a, _ = synth.we_inputs(N, seed=N + K, batch=Z)
    a = a * scale
    g = torch.Generator().manual_seed(K + N)
    b = torch.randn(Z, N, 3, generator=g)
    b = 1.5 * b / b.norm(dim=-1, keepdim=True)
    cb, wn = 1.0 + spread * torch.randn(K, generator=g), synth.wavenumbers(2 * K)
    mask = None
    if kind == "frames":
        a[1] += torch.tensor([8192.0, -4096.0, 4096.0])
    elif kind == "first empty":
        mask = (torch.arange(Z) == 0)[:, None].expand(Z, N)
    elif kind == "scattered":
        mask = torch.rand(Z, N, generator=g) < 0.2
    elif kind == "nan":
        a[1, 77, 1] = float("nan")
    got, terms = run_aniso_route(gpu, a, b, cb, wn, mask, partials)
    assert (terms > 0) == grids, terms
    if kind == "nan":           # an unpadded token at NaN makes every sum of its batch item NaN and touches no other item
        assert np.isnan(got[0][1]).all()
        a, b, got = a[:1], b[:1], [x[:1] for x in got]
    rows = np.unique(np.concatenate([np.arange(0, N, 41), [15, 16, N - 1]])).astype(np.int32)
    ref = c_oracle.we_aniso(a.numpy(), b.numpy(), cb.numpy(), wn.numpy(), None if mask is None else mask.numpy(), rows=rows)
    far = float((a.amax(1) - a.amin(1)).norm(dim=-1).max())         # the bar of the tests above
    bar = 2e-6 + 2 * 2.0 ** -24 * float(wn.abs().max()) * far
    for x, r in zip(got, ref):
        assert np.isfinite(x).all() and rel_l2(x[:, rows], r) <= bar, (name, rel_l2(x[:, rows], r), bar)
