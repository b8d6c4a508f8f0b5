"""The operators' host path in C++ (csrc/ops.cpp) against the Python functions: the same results where it takes a call, the same answers where it does not."""
import contextlib
import threading

import pytest
import torch

import proteusai_amd as pa
from proteusai_amd import _lib, synth


class _General:
    """Takes no call: what remains is the Python path."""
    attention = embedding = aniso = staticmethod(lambda *a: None)


@pytest.fixture
def general(monkeypatch):
    @contextlib.contextmanager
    def use():
        with monkeypatch.context() as m:
            _lib.ops()
            m.setattr(_lib, "_ops", _General)
            yield
    return use


def _attention(gpu, legacy=False, d=32, seed=0, Z=2, N=130, H=3):
    g = torch.Generator(device=gpu).manual_seed(seed)
    op = torch.float16 if legacy else torch.bfloat16
    qkv = [torch.randn(Z, H, N, d, generator=g, device=gpu).to(op).requires_grad_() for _ in range(3)]
    coords = torch.cumsum(torch.randn(Z, N, 3, generator=g, device=gpu) * 2, 1)
    mask = torch.arange(N, device=gpu)[None] >= torch.tensor([N, N // 2], device=gpu)[:, None] if Z == 2 else None
    spreads = torch.linspace(4, 9, H, device=gpu).requires_grad_()
    kw = dict(betas=torch.linspace(0.5, 1.5, H, device=gpu).requires_grad_(), min_rbf=0.001, operand_dtype=op) if legacy else {}
    return qkv, coords, spreads, mask, kw, torch.randn(Z, H, N, d, generator=g, device=gpu)


def _run(qkv, coords, spreads, mask, kw, d, grad=torch.autograd.grad):
    O = pa.geometric_attn(*qkv, coords, spreads, mask=mask, **kw)
    return O, grad(O, [*qkv, spreads] + ([kw["betas"]] if "betas" in kw else []), d)


def _same(a, b, scalars=2):
    """Outputs alike to the bit, but for the gradients per head, which are summed in no order."""
    (Oa, ga), (Ob, gb) = a, b
    assert torch.equal(Oa, Ob) and all(torch.equal(x, y) and x.dtype == y.dtype and x.stride() == y.stride() for x, y in zip(ga[:3], gb[:3]))
    assert all(bool(((x - y).abs() <= 1e-5 * y.abs().max()).all()) for x, y in zip(ga[3:], gb[3:]))


# both logits; every head dimension; a gradient in another type, not dense, expanded; operands as views of a fused projection; O in token order
@pytest.mark.gpu
@pytest.mark.parametrize("legacy,d", [(False, 32), (True, 64), (False, 128)])
@pytest.mark.parametrize("form", ["plain", "bf16 gradient", "strided gradient", "expanded gradient", "token major", "fused", "no mask", "check off"])
def test_attention_equals_the_python_path(gpu, general, legacy, d, form):
    qkv, coords, spreads, mask, kw, dO = _attention(gpu, legacy, d)
    if form == "bf16 gradient":
        dO = dO.to(torch.bfloat16).float()
    if form == "strided gradient":
        dO = dO.transpose(1, 2).contiguous().transpose(1, 2)
    if form == "expanded gradient":
        dO = torch.ones((), device=gpu).expand(dO.shape)
    if form == "token major":
        kw["token_major_out"] = True
    if form == "fused":
        both = torch.stack([t.detach() for t in qkv], 2).permute(0, 3, 2, 1, 4).contiguous()
        qkv = [both[:, :, i].permute(0, 2, 1, 3).requires_grad_() for i in range(3)]
    if form == "no mask":
        mask = None
    if form == "check off":
        kw["check_spreads"] = False
    got = _run(qkv, coords, spreads, mask, kw, dO)
    assert "Attention" in got[0].grad_fn.name()
    with general():
        want = _run(qkv, coords, spreads, mask, kw, dO)
        assert type(want[0].grad_fn).__name__ == "_geometric_attnBackward"
    _same(got, want)
    with torch.no_grad():
        assert torch.equal(pa.geometric_attn(*qkv, coords, spreads, mask=mask, **kw), want[0])


# Contiguous operands with strides of their own along a dimension of size one: a single token (transposed), a single sequence, a single head
@pytest.mark.gpu
@pytest.mark.parametrize("legacy", [False, True])
@pytest.mark.parametrize("token_major", [False, True])
@pytest.mark.parametrize("one", ["token", "sequence", "head"])
@pytest.mark.parametrize("which", [(0, 1, 2), (1,)])
def test_dimensions_of_size_one(gpu, general, legacy, token_major, one, which):
    Z, H, N, d = {"token": (2, 4, 1, 32), "sequence": (1, 4, 40, 32), "head": (2, 1, 40, 32)}[one]
    qkv, coords, spreads, _, kw, dO = _attention(gpu, legacy, d, Z=Z, N=N, H=H)
    strides = {"token": (H * d, d, 1, 1), "sequence": (9, N * d, d, 1), "head": (N * d, 9, d, 1)}[one]
    qkv = [torch.as_strided(t.detach(), t.shape, strides).requires_grad_() if i in which else t for i, t in enumerate(qkv)]
    assert all(t.is_contiguous() for t in qkv) and any(t.stride() == strides for t in qkv)
    kw["token_major_out"] = token_major
    # (what the library holds against an odd stride, beside O in token order or a gradient that is not dense, is refused alike)
    for d_out in (dO, dO.transpose(1, 2).contiguous().transpose(1, 2)):
        with general():
            try:
                want = _run(qkv, coords, spreads, None, kw, d_out)
            except ValueError:
                want = None
        if want is None:
            with pytest.raises(ValueError, match="code -"):
                _run(qkv, coords, spreads, None, kw, d_out)
        else:
            got = _run(qkv, coords, spreads, None, kw, d_out)
            assert "Attention" in got[0].grad_fn.name()
            _same(got, want)


# What has to be converted or refused is the Python functions': not taken, and the same result or error
@pytest.mark.gpu
def test_attention_that_is_not_plain(gpu, general):
    qkv, coords, spreads, mask, kw, dO = _attention(gpu)
    q, k, v = qkv
    def both(*a, **k_):
        with general():
            try:
                want = pa.geometric_attn(*a, **k_)
            except Exception as e:
                with pytest.raises(type(e)):
                    pa.geometric_attn(*a, **k_)
                return
        got = pa.geometric_attn(*a, **k_)
        assert torch.equal(got, want) and type(got.grad_fn) is type(want.grad_fn)
    taken = lambda *a: _lib.ops().attention(*a, 0.0, 1.0, False, False, False) is not None
    assert taken(q, k, v, coords, spreads, None, mask)
    off = torch.empty(q.numel() + 1, dtype=q.dtype, device=gpu)[1:].view(q.shape).copy_(q.detach())
    for a in ((q.detach().float(), k, v, coords, spreads), (off, k, v, coords, spreads), (q, k, v, coords.double(), spreads), (q, k, v, coords, spreads.double()), (q, k, v[:, :, :-1], coords, spreads),
              (q, k, v, coords[:, :-1], spreads), (q, k, v, coords, spreads[:-1]), (q[..., :16], k[..., :16], v[..., :16], coords, spreads), (q.cpu(), k.cpu(), v.cpu(), coords, spreads),
              (q[:0], k[:0], v[:0], coords[:0], spreads)):
        assert not taken(*a, None, None)
        both(*a)
    for m in (mask.to(torch.uint8), mask[:1], mask.t().contiguous().t()):
        assert not taken(q, k, v, coords, spreads, None, m)
        both(q, k, v, coords, spreads, mask=m)
    for s in (torch.tensor([1.0, -1.0, 2.0]), torch.tensor([1.0, 0.0, 2.0]), torch.tensor([1.0, float("nan"), 2.0])):
        with pytest.raises(AssertionError, match="positive"):
            pa.geometric_attn(q, k, v, coords, s.to(gpu))
    both(q, k, v, coords, spreads, operand_dtype=torch.float16)
    both(q, k, v, coords, spreads, out_dtype=torch.bfloat16)
    both(q, k, v, coords, spreads, betas=torch.ones_like(spreads), min_rbf=0.5, max_rbf=0.5 + 1e-12)       # (a range that is empty in fp32)


@pytest.mark.gpu
def test_observers_see_what_they_saw(gpu, general):
    qkv, coords, spreads, mask, kw, dO = _attention(gpu)
    call = lambda q: pa.geometric_attn(q, *qkv[1:], coords, spreads, mask=mask)
    wn = torch.linspace(0.3, 1.7, 64, device=gpu, requires_grad=True)
    embed = lambda w: pa.wf_embedding(coords, w)
    from torch.utils._python_dispatch import TorchDispatchMode

    class Count(TorchDispatchMode):
        def __torch_dispatch__(self, f, types, args=(), kwargs=None):
            return f(*args, **(kwargs or {}))

    class Sub(torch.Tensor):
        pass

    def vmapped(f, x):
        return torch.func.vmap(f)(x[None])

    def tangent(f, x):
        with torch.autograd.forward_ad.dual_level():
            return f(torch.autograd.forward_ad.make_dual(x.detach(), torch.ones_like(x)))

    def in_mode(f, x):
        with Count():
            return f(x)

    def batched(f, x):
        out = f(x)
        return torch.autograd.grad(out, x, torch.stack([torch.ones_like(out)] * 2), is_grads_batched=True)[0]

    for f, x in ((call, qkv[0]), (embed, wn)):
        for way in (vmapped, tangent, in_mode, batched, lambda f, x: f(x.detach().as_subclass(Sub))):
            with general():
                try:
                    want = way(f, x)
                except Exception as e:
                    want = type(e)
            if isinstance(want, type):
                with pytest.raises(want if want is not NotImplementedError else Exception):
                    way(f, x)
            else:
                got = way(f, x)
                assert torch.equal(got, want) and type(got) is type(want)


# Saved tensors in another form (on the host and back, in 64 bits, not dense) go the general way; a tensor changed in place is an error
@pytest.mark.gpu
def test_saved_tensors(gpu, general):
    qkv, coords, spreads, mask, kw, dO = _attention(gpu)
    want = _run(qkv, coords, spreads, mask, kw, dO)
    hooks = torch.autograd.graph.saved_tensors_hooks
    for pack, unpack in ((lambda t: t.cpu(), lambda t: t.to(gpu)), (lambda t: t.double() if t.dtype == torch.float32 else t, lambda t: t),
                         (lambda t: t, lambda t: t.transpose(-1, -2).contiguous().transpose(-1, -2) if t.dim() > 1 else t)):
        with hooks(pack, unpack):
            _same(_run(qkv, coords, spreads, mask, kw, dO), want)
    O = pa.geometric_attn(*qkv, coords, spreads, mask=mask)
    with torch.no_grad():
        spreads.mul_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        O.backward(dO)
    wn = torch.linspace(0.3, 1.7, 64, device=gpu, requires_grad=True)
    out = pa.wf_embedding(coords, wn, mask=mask)
    d = torch.randn_like(out)
    g = torch.autograd.grad(out, wn, d, retain_graph=True)[0]
    assert torch.equal(g, torch.autograd.grad(out, wn, d.transpose(0, 1).contiguous().transpose(0, 1), retain_graph=True)[0])       # (not dense: the general way)
    with hooks(lambda t: t.double(), lambda t: t):
        out2 = pa.wf_embedding(coords, wn, mask=mask)
        assert torch.equal(torch.autograd.grad(out2, wn, d)[0], g)
    assert torch.autograd.grad(out, wn, d, create_graph=True)[0].grad_fn is None


@pytest.mark.gpu
@pytest.mark.parametrize("N,K", [(70, 64), (700, 128)])
def test_embeddings_equal_the_python_path(gpu, general, N, K):
    gen = torch.Generator().manual_seed(N)
    coords = torch.stack([synth.random_walk_chain(N, gen) for _ in range(2)]).to(gpu)
    beta = torch.randn(2, N, 3, generator=gen).to(gpu)
    mask = torch.arange(N, device=gpu)[None] >= torch.tensor([N, N // 3], device=gpu)[:, None]
    wn, cb = torch.linspace(0.3, 1.7, K, device=gpu, requires_grad=True), torch.linspace(0.8, 1.2, K, device=gpu, requires_grad=True)
    d = torch.randn(2, N, 2 * K, device=gpu)
    frozen = cb.detach()
    def results():
        for m in (None, mask):
            out = pa.wf_embedding(coords, wn, mask=m)
            yield from (out, *torch.autograd.grad(out, wn, d))
            out = pa.wf_embedding_learnCB(coords, beta, cb, wn, m)
            yield from (out, *torch.autograd.grad(out, (cb, wn), d))
            out = pa.wf_embedding_learnCB(coords, beta, frozen, wn, m)
            yield from (out, *torch.autograd.grad(out, wn, d))
            with torch.no_grad():
                yield pa.wf_embedding(coords, wn, mask=m)
                yield pa.wf_embedding_learnCB(coords, beta, cb, wn, m)
    got = list(results())
    with general():
        assert all(torch.equal(a, b) for a, b in zip(got, results()))
    # refused and converted as before
    for bad in ((coords[..., :2], wn), (coords, wn[None]), (coords.cpu(), wn)):
        with pytest.raises((ValueError, RuntimeError)):
            pa.wf_embedding(*bad)
    with pytest.raises(ValueError):
        pa.wf_embedding(coords, wn, mask=mask[:, 1:])
    assert torch.equal(pa.wf_embedding(coords.double(), wn), pa.wf_embedding(coords, wn)) and pa.wf_embedding(coords[:, :0], wn).shape == (2, 0, 2 * K)


# On streams and threads of their own
@pytest.mark.gpu
def test_streams_and_threads(gpu):
    qkv, coords, spreads, mask, kw, dO = _attention(gpu)
    kw["check_spreads"] = False
    want = _run(qkv, coords, spreads, mask, kw, dO)
    torch.cuda.synchronize()
    got = []

    def work():
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(3):
                got.append(_run(qkv, coords, spreads, mask, kw, dO))
        s.synchronize()
    threads = [threading.Thread(target=work) for _ in range(2)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert len(got) == 6
    for r in got:
        _same(r, want)


@pytest.mark.gpu
def test_captured(gpu):
    qkv, coords, spreads, mask, kw, dO = _attention(gpu)
    kw["check_spreads"] = False
    O, grads = _run(qkv, coords, spreads, mask, kw, dO)
    want = (O.detach(), grads)
    torch.cuda.synchronize()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        # (leaves of this stream, none of whose earlier graphs is left: a leaf's node keeps the stream on which it was made, and a backward joins it)
        del O
        leaves, at = [t.detach().clone().requires_grad_() for t in qkv], spreads.detach().clone().requires_grad_()
        _run(leaves, coords, at, mask, kw, dO)
        stream.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            O, grads = _run(leaves, coords, at, mask, kw, dO)
            captured = (O.detach(), grads)
            del O
    for _ in range(3):
        for t in (captured[0], *captured[1][:3]):
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        _same(captured, want)
