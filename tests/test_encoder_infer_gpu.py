"""The encoder's inference in bf16: its product (proteus_gemm_bf16), the layer in one call (proteus_encoder_infer) against its parts, the sum in front of it."""
import copy

import pytest
import torch
import torch.nn.functional as F

import proteusai_amd as pa
from proteusai_amd import _lib, encoder, synth, train_ops


def _gemm(A, B, bias, gelu, C):
    return _lib.load().proteus_gemm_bf16(A.data_ptr(), B.data_ptr(), None if bias is None else bias.data_ptr(), C.data_ptr(), A.shape[0], B.shape[0], A.shape[1],
                                         A.stride(0), B.stride(0), C.stride(0), gelu, _lib.raw_stream(A.device))


# Every tile of the dispatch at edges of tiles, of the steps of 64 k and of their stages: 64 x 64 (four stages), 128 x 64 (four), 128 x 128 (four, long K),
# 128 x 64 (two), 128 x 128 (two), 256 x 256, and 128 x 64 again where the last round would be empty
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (65, 72, 64), (63, 64, 72), (1000, 1024, 264), (2100, 1032, 136), (2049, 1800, 1032), (1900, 2040, 200), (4000, 1800, 320),
                                   (8190, 1544, 72), (6100, 1536, 64)])
@pytest.mark.parametrize("gelu", [0, 1])
def test_product_against_float64(gpu, M, N, K, gelu):
    g = torch.Generator(device=gpu).manual_seed(M + N + K)
    wide = lambda r, c: torch.randn(r, c + 8, generator=g, device=gpu).bfloat16()[:, :c]                # (rows that are not dense)
    A, B, bias = wide(M, K), wide(N, K) * 0.25, torch.randn(N, generator=g, device=gpu).bfloat16() if N % 16 else None
    C = torch.full((M, N + 16), float("nan"), device=gpu, dtype=torch.bfloat16)
    assert _gemm(A, B, bias, gelu, C[:, :N]) == 0
    want = A.double() @ B.double().t().contiguous() + (0 if bias is None else bias.double())
    mass = A.double().abs() @ B.double().abs().t().contiguous() + (0 if bias is None else bias.double().abs())
    # an fp32 accumulator rounded once or twice per 16 k; GELU's slope is at most 1.13, its erf good to 3e-7 of x; bf16 rounds once
    err = 1.13 * 2 * (K / 16 + 4) * 2.0 ** -24 * mass
    if gelu:
        err, want = err + 3e-7 * want.abs(), F.gelu(want)
    assert bool(((C[:, :N].double() - want).abs() <= err + 2.0 ** -8 * (want.abs() + err)).all())
    assert bool(C[:, N:].isnan().all())                                                                  # nothing beside the tile
    again = torch.empty_like(C)
    assert _gemm(A, B, bias, gelu, again[:, :N]) == 0 and torch.equal(again[:, :N], C[:, :N])


@pytest.mark.gpu
def test_gelu_at_its_ends(gpu):
    x = torch.tensor([0.0, -0.0, 1e-30, 50.0, -50.0, 3e38, -4.0, -9.0, float("inf"), float("nan")], device=gpu)
    x = torch.cat([x, torch.zeros(6, device=gpu)]).bfloat16()
    A, B = torch.zeros(1, 8, device=gpu, dtype=torch.bfloat16), torch.zeros(16, 8, device=gpu, dtype=torch.bfloat16)
    C = torch.empty(1, 16, device=gpu, dtype=torch.bfloat16)
    assert _gemm(A, B, x, 1, C) == 0
    want = F.gelu(x.double())
    got = C[0].double()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    ok = want.isfinite()
    assert bool(((got - want).abs()[ok] <= 2.0 ** -8 * want.abs()[ok] + 1e-12).all())


def test_refusals_come_before_any_launch():
    f = _lib.load().proteus_gemm_bf16
    ok = [4096, 4096, 4096, 4096, 8, 8, 8, 8, 8, 8, 0, None]
    for at, value in ((0, None), (1, None), (3, None), (0, 4104), (3, 4104), (2, 4097), (4, 0), (5, 12), (6, 12), (7, 4), (7, 12), (9, 0)):
        bad = list(ok)
        bad[at] = value
        assert f(*bad) < 0, (at, value)
    assert f(4096, 4096, None, 4096, 8, 8, 8, 1 << 22, 8, 8, 0, None) < 0                                # a tile's rows beyond 31 bits
    lib = _lib.load()
    assert lib.proteus_encoder_infer_bytes(1, 10, 2, 32, 64) > 0
    for bad in ((0, 10, 2, 32, 64), (1, 10, 2, 48, 64), (1, 10, 2, 32, 68), (1, 1 << 21, 8, 64, 64)):
        assert lib.proteus_encoder_infer_bytes(*bad) == 0
    assert lib.proteus_encoder_infer(None, 4096, 4096, None, None, 1e-5, 1e-5, 4096, 4096, 1 << 30, 1, 10, 2, 32, 64, None) < 0
    assert lib.proteus_add_to_bf16(4096, 4096, 4096, 12, None) < 0 and lib.proteus_add_to_bf16(4096, 4100, 4096, 16, None) < 0


def _layer(gpu, Z, N, H, dk, hidden):
    torch.manual_seed(N)
    layer = pa.Encoder(d_model=H * dk, heads=H, d_hidden=hidden, dropout=0.1).to(gpu)
    with torch.no_grad():
        for p in layer.parameters():
            p.add_(0.05 * torch.randn_like(p))
    layer = layer.to(torch.bfloat16).eval()
    coords = torch.stack([synth.random_walk_chain(N, torch.Generator().manual_seed(i)) for i in range(Z)]).to(gpu)
    mask = (torch.arange(N, device=gpu)[None, :] >= torch.linspace(max(1, N // 2), N, Z, device=gpu)[:, None]) if Z > 1 else None
    return layer, torch.randn(Z, N, H * dk, device=gpu).bfloat16(), coords, mask


# one token; odd sizes; wide heads; keys cut over workgroups, with a mask and without; the pipelined kernel (every way that O leaves the attention)
@pytest.mark.gpu
@pytest.mark.parametrize("Z,N,H,dk,hidden", [(1, 1, 1, 32, 8), (2, 70, 2, 32, 104), (3, 129, 2, 128, 264), (1, 2100, 8, 64, 512), (4, 2048, 8, 64, 136), (8, 2048, 8, 64, 64), (13, 2048, 8, 32, 64)])
def test_layer_is_as_near_to_its_weights_as_its_parts(gpu, Z, N, H, dk, hidden, monkeypatch):
    layer, x, coords, mask = _layer(gpu, Z, N, H, dk, hidden)
    with torch.no_grad():
        assert encoder._infer_layer(x, coords, mask, layer) is not None
        got = layer(x, x, x, coords, mask)
        with monkeypatch.context() as m:
            m.setattr(encoder, "_infer_layer", lambda *a: None)
            parts = layer(x, x, x, coords, mask)
            want = copy.deepcopy(layer).float()(*[x.float()] * 3, coords, mask)
        again = layer(x, x, x, coords, mask)
    # Both round to bf16 between the launches, the call at fewer places than its parts: no farther off than they are, but for single roundings
    assert float((got.double() - want).norm()) <= 1.1 * float((parts.double() - want).norm()) + 1e-4 * want.numel() ** 0.5
    assert float((parts.double() - want).norm()) <= 0.03 * float(want.norm())
    pad = mask if mask is not None else torch.zeros_like(x[..., 0], dtype=torch.bool)
    assert bool(got[~pad].isfinite().all()) and torch.equal(got, again)


@pytest.mark.gpu
def test_what_the_call_does_not_take(gpu):
    layer, x, coords, mask = _layer(gpu, 2, 70, 2, 32, 104)
    take = lambda **k: encoder._infer_layer(k.get("x", x), k.get("coords", coords), k.get("mask", mask), layer) is not None
    with pytest.MonkeyPatch.context() as mp:                                                             # gradients are recorded: told before the closer look
        looked = []
        mp.setattr(train_ops, "plain_module", lambda *a: looked.append(a))
        assert not take() and not take(x=x.clone().requires_grad_()) and not looked
        layer.attn_norm.weight.requires_grad_(False)
        assert not take() and looked
    assert not take()
    layer.attn_norm.weight.requires_grad_(True)
    with torch.no_grad():
        assert take() and take(mask=None) and take(x=x.transpose(0, 1).contiguous().transpose(0, 1))
        assert not take(x=x.float()) and not take(mask=mask[:1]) and not take(coords=coords[:, :69]) and not take(x=x[:, :0], coords=coords[:, :0], mask=None)
        with torch.autocast("cuda", dtype=torch.float16):
            assert not take()
        hook = layer.ffn.in_proj.register_forward_hook(lambda *a: None)
        assert not take()
        hook.remove()
        layer.train()
        assert not take()                                                                                # dropout is active
        layer.eval()
        layer.ffn.in_proj.bias = None
        assert not take()
    with torch.no_grad(), pytest.MonkeyPatch.context() as mp:                                             # sigma that the kernel would read past its end, or on the host
        for name, value in (("get_spreads", lambda: torch.full((1,), 5.0, device=gpu)), ("get_spreads", lambda: torch.full((2,), 5.0)), ("min_spread", torch.full((2, 1), 2.0, device=gpu))):
            layer, x, coords, mask = _layer(gpu, 2, 70, 2, 32, 104)
            mp.setattr(layer.attn, name, value)
            assert not take()
            if name == "get_spreads" and value().numel() == 2:
                assert bool(layer(x, x, x, coords, mask)[~mask].isfinite().all())
            else:
                with pytest.raises(AssertionError, match="spreads"):
                    layer(x, x, x, coords, mask)
    wide, y, at, _ = _layer(gpu, 1, 8200, 32, 32, 64)
    with torch.no_grad():                                                                                # products that the library does faster
        assert encoder._infer_layer(y, at, None, wide) is None and encoder._infer_layer(y[:, :8192], at[:, :8192], None, wide) is not None
    with torch.no_grad(), pytest.raises(AssertionError):
        layer(x, x, x, coords[:, :69], mask)                                                             # refused as before


# One head: its output projection is read where it lies, which need not be on 16 bytes (a parameter cut out of a flat buffer)
@pytest.mark.gpu
def test_one_head_with_an_output_projection_off_16_bytes(gpu):
    layer, x, coords, mask = _layer(gpu, 2, 70, 1, 64, 104)
    with torch.no_grad():
        want = layer(x, x, x, coords, mask)
        flat = torch.empty(64 * 64 + 8, dtype=torch.bfloat16, device=gpu)
        w = flat[1:64 * 64 + 1].view(64, 64).copy_(layer.attn.out_proj.weight)
        layer.attn.out_proj.weight = torch.nn.Parameter(w)
        assert layer.attn.out_proj.weight.data_ptr() % 16 == 2 and torch.equal(layer(x, x, x, coords, mask), want)


# new weights, in place and by a state dict, are seen; x as it was
@pytest.mark.gpu
def test_layer_follows_its_weights(gpu):
    layer, x, coords, mask = _layer(gpu, 2, 70, 2, 32, 104)
    other, *_ = _layer(gpu, 1, 71, 2, 32, 104)
    keep = x.clone()
    with torch.no_grad():
        before = layer(x, x, x, coords, mask)
        layer.attn.k_proj.mul_(1.5)
        changed = layer(x, x, x, coords, mask)
        assert not torch.equal(before, changed)
        layer.load_state_dict(other.state_dict())
        assert torch.equal(layer(x, x, x, coords, mask), other(x, x, x, coords, mask)) and torch.equal(x, keep)


# What the module keeps between calls, made on one stream and read on another: the other waits until it is there, and it stays until that read is over; what a capture
# makes is not kept
@pytest.mark.gpu
@pytest.mark.parametrize("one_call", [True, False])
def test_kept_constants_on_other_streams(gpu, monkeypatch, one_call):
    layer, x, coords, mask = _layer(gpu, 2, 70, 2, 32, 104)
    if not one_call:
        monkeypatch.setattr(encoder, "_infer_layer", lambda *a: None)
    run = lambda m: m(x, x, x, coords, mask)
    with torch.no_grad():
        want = run(copy.deepcopy(layer))
        a, b = torch.cuda.Stream(), torch.cuda.Stream()
        torch.cuda.synchronize()
        with torch.cuda.stream(a):
            torch.cuda._sleep(20_000_000)
            first = run(layer)
        kept = [t for k in layer.attn._constants.values() for t in k.tensors]
        with torch.cuda.stream(b):
            second = run(layer)                              # (waits for the sleep of the other stream)
            torch.cuda._sleep(20_000_000)
            third = run(layer)
        at = {t.data_ptr() for t in kept}
        shapes = [(t.shape, t.dtype) for t in kept]
        del kept
        layer.attn.invalidate_caches()
        with torch.cuda.stream(a):                           # (whatever is given back to this stream's memory is written over)
            over = [torch.full(s, float("nan"), dtype=d, device=gpu) for s, d in shapes for _ in range(4)]
        assert not any(t.data_ptr() in at for t in over)
        torch.cuda.synchronize()
        assert torch.equal(first, want) and torch.equal(second, want) and torch.equal(third, want)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            captured = run(layer)
        assert not layer.attn._constants
        for _ in range(3):
            captured.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(captured, want) and torch.equal(run(layer), want)


@pytest.mark.gpu
def test_sum_in_front_of_the_layers(gpu):
    a, b = torch.randn(3, 67, 40, device=gpu), torch.randn(3, 67, 40, device=gpu).bfloat16()
    a[0, 0, :4] = torch.tensor([float("inf"), float("nan"), 3.3e38, 1e-40])
    with torch.no_grad():
        got, want = encoder._add_to_bf16(a, b), (a + b.float()).bfloat16()
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(1.0), want.nan_to_num(1.0))
        assert encoder._add_to_bf16(a[..., :39], b[..., :39]) is None and encoder._add_to_bf16(a, b.float()) is None
    assert encoder._add_to_bf16(a.requires_grad_(), b) is None
