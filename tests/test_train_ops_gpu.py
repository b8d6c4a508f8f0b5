"""GPU tests of the training step's own kernels (proteusai_amd/train_ops.py) against the torch expressions they stand for,
evaluated in float64 on the CPU from the same inputs.

Bars: results are fp32 with at most a few thousand terms per sum, taken as short chains of partial sums; 2^-24 per operation over
chains of some 50 additions of random sign gives rel-L2 below 1e-6, and products (MLP) of K <= 2048 terms below 3e-6."""
import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

import proteusai_amd as pa
from proteusai_amd import synth, train_ops

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float((a.double().cpu() - b).norm() / b.norm().clamp_min(1e-30))


def double_copy(m):
    import copy
    return copy.deepcopy(m).double().cpu()


@pytest.mark.parametrize("shape", [(1, 4), (3, 64), (2, 5, 260), (130, 512), (1027, 1000), (2049, 2048)])
def test_add_layer_norm(gpu, shape):
    torch.manual_seed(shape[-1])
    norm = nn.LayerNorm(shape[-1])
    with torch.no_grad():
        norm.weight.add_(0.3 * torch.randn(shape[-1]))
        norm.bias.add_(torch.randn(shape[-1]))
    x, r, d = (torch.randn(shape) + 0.5 for _ in range(3))
    x64, r64 = x.double().requires_grad_(), r.double().requires_grad_()
    n64 = double_copy(norm)
    ref = n64(x64 + r64)
    want = torch.autograd.grad(ref, [x64, r64, n64.weight, n64.bias], d.double())
    norm = norm.to(gpu)
    xg, rg = x.to(gpu).requires_grad_(), r.to(gpu).requires_grad_()
    out = train_ops.add_layer_norm(xg, rg, norm)
    got = torch.autograd.grad(out, [xg, rg, norm.weight, norm.bias], d.to(gpu))
    assert rel(out.detach(), ref.detach()) <= 1e-6
    for g, w, name in zip(got, want, ("x", "res", "gamma", "beta")):
        assert rel(g, w) <= 2e-6, (name, rel(g, w))


@pytest.mark.parametrize("rows,d,hidden", [(1, 4, 8), (2, 12, 20), (129, 64, 100), (2048, 128, 256), (4100, 64, 132)])
def test_mlp(gpu, rows, d, hidden):
    torch.manual_seed(rows)
    mlp = pa.MLP(d_in=d, d_out=d, d_hidden=hidden, dropout=0.0)
    x, dout = torch.randn(1, rows, d), torch.randn(1, rows, d)
    m64, x64 = double_copy(mlp), x.double().requires_grad_()
    ref = m64(x64)
    want = torch.autograd.grad(ref, [x64, *m64.parameters()], dout.double())
    mlp, xg = mlp.to(gpu), x.to(gpu).requires_grad_()
    assert train_ops.gelu_mlp(xg, mlp.in_proj, mlp.out_proj) is not None
    out = mlp(xg)
    got = torch.autograd.grad(out, [xg, *mlp.parameters()], dout.to(gpu))
    assert rel(out.detach(), ref.detach()) <= 3e-6
    for g, w in zip(got, want):
        assert rel(g, w) <= 3e-6, (tuple(w.shape), rel(g, w))


@pytest.mark.parametrize("T,V,D", [(1, 1, 4), (127, 33, 64), (129, 64, 100), (2048, 33, 512), (8201, 21, 260), (300, 64, 100)])
def test_embedding_gradient(gpu, T, V, D):
    torch.manual_seed(T)
    emb = nn.Embedding(V, D)
    tokens, d = torch.randint(0, V, (T,)), torch.randn(T, D)
    want = torch.zeros(V, D, dtype=torch.float64).index_add_(0, tokens, d.double())
    emb = emb.to(gpu)
    out = train_ops.embedding(tokens.to(gpu), emb)
    assert torch.equal(out, emb(tokens.to(gpu)))
    got, = torch.autograd.grad(out, [emb.weight], d.to(gpu))
    assert rel(got, want) <= 1e-6


@pytest.mark.parametrize("Z,N,H,dk,frozen", [(1, 1, 1, 32, False), (2, 70, 4, 64, False), (2, 129, 2, 128, True)])
def test_self_attention_module_equals_its_expression(gpu, Z, N, H, dk, frozen, monkeypatch):
    # the same kernels and products on the same bf16 operands: what differs is the order of the bias sums, one rounding in sigma
    # and the products' own choice of order (a flipped bf16 rounding of an operand: 2^-9 of single elements)
    torch.manual_seed(N)
    m = pa.GeoAttention(d_model=H * dk, heads=H).to(gpu)
    with torch.no_grad():
        for p in m.parameters():
            p.add_(0.1 * torch.randn_like(p))
    if frozen:
        m.k_proj.requires_grad_(False)
        m.q_bias.requires_grad_(False)
        m.out_proj.weight.requires_grad_(False)
        m.spread_weights.requires_grad_(False)
    coords = torch.stack([synth.random_walk_chain(N, torch.Generator().manual_seed(i)) for i in range(Z)]).to(gpu)
    mask = torch.arange(N, device=gpu)[None, :] >= torch.tensor([N, max(1, N - 9)][:Z], device=gpu)[:, None]
    x = torch.randn(Z, N, H * dk, device=gpu, requires_grad=True)
    d = torch.randn(Z, N, H * dk, device=gpu)
    leaves = [x] + [p for n, p in m.named_parameters() if p.requires_grad and n != "beta_weights"]
    assert train_ops.self_attention(x, coords, mask, m) is not None
    out = m(x, x, x, coords, mask)
    got = torch.autograd.grad(out, leaves, d)
    monkeypatch.setattr(train_ops, "self_attention", lambda *a: None)
    ref = m(x, x, x, coords, mask)
    want = torch.autograd.grad(ref, leaves, d)
    assert float((out - ref).norm() / ref.norm()) <= 1e-4
    for g, w in zip(got, want):
        # (one token: every softmax is 1, and the gradients of q, k and sigma are rounding errors about zero)
        assert float((g - w).norm()) <= 1e-3 * float(w.norm()) + 1e-4, tuple(w.shape)


def test_recorded_backward_differentiates_the_expression(gpu):
    torch.manual_seed(0)
    mlp, norm = pa.MLP(d_in=16, d_out=16, d_hidden=24, dropout=0.0), nn.LayerNorm(16)
    x = torch.randn(1, 9, 16)

    def second(mlp, norm, x, fused):
        h = mlp(x)
        out = train_ops.add_layer_norm(x, h, norm) if fused else norm(x + h)
        g, = torch.autograd.grad((out ** 3).sum(), [x], create_graph=True)
        return torch.autograd.grad((g ** 2).sum(), [x, norm.weight, mlp.in_proj.weight])
    want = second(double_copy(mlp), double_copy(norm), x.double().requires_grad_(), False)
    got = second(mlp.to(gpu), norm.to(gpu), x.to(gpu).requires_grad_(), True)
    for g, w in zip(got, want):
        assert rel(g, w) <= 1e-5


def test_what_the_general_path_keeps(gpu):
    mlp, norm = pa.MLP(d_in=16, d_out=16, d_hidden=24, dropout=0.0).to(gpu), nn.LayerNorm(16).to(gpu)
    x = torch.randn(1, 9, 16, device=gpu, requires_grad=True)
    lin = (mlp.in_proj, mlp.out_proj)
    assert train_ops.gelu_mlp(x, *lin) is not None
    with torch.no_grad():
        assert train_ops.gelu_mlp(x, *lin) is None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert train_ops.gelu_mlp(x, *lin) is None and train_ops.add_layer_norm(x, x, norm) is None
    assert train_ops.gelu_mlp(x.bfloat16(), *lin) is None
    seen = []
    handle = mlp.in_proj.register_forward_hook(lambda *a: seen.append(1))
    mlp(x)
    handle.remove()
    assert seen == [1]
    tangent = torch.func.jvp(lambda t: norm(t + mlp(t)), (x.detach(),), (torch.ones_like(x),))[1]
    assert torch.isfinite(tangent).all()
    assert torch.func.vmap(mlp)(x.detach()).shape == x.shape


def test_replaced_spreads_keep_the_general_path(gpu):
    m = pa.GeoAttention(d_model=64, heads=2).to(gpu)
    x = torch.randn(1, 9, 64, device=gpu, requires_grad=True)
    coords = synth.random_walk_chain(9, torch.Generator().manual_seed(0)).unsqueeze(0).to(gpu)
    assert train_ops.self_attention(x, coords, None, m) is not None
    m.get_spreads = lambda: torch.full((2,), 5.0, device=gpu)
    assert train_ops.self_attention(x, coords, None, m) is None


def test_batched_gradients_differentiate_the_expressions(gpu):
    # is_grads_batched hands every backward a batch of gradients under vmap: no memory that a kernel could read
    torch.manual_seed(1)
    mlp, norm, emb = pa.MLP(d_in=16, d_out=16, d_hidden=24, dropout=0.0).to(gpu), nn.LayerNorm(16).to(gpu), nn.Embedding(7, 16).to(gpu)
    x = torch.randn(1, 9, 16, device=gpu, requires_grad=True)
    tokens = torch.randint(0, 7, (1, 9), device=gpu)
    out = train_ops.add_layer_norm(train_ops.embedding(tokens, emb), mlp(x), norm)
    leaves = [x, emb.weight, *norm.parameters(), *mlp.parameters()]
    d = torch.randn(3, *out.shape, device=gpu)
    got = torch.autograd.grad(out, leaves, d, is_grads_batched=True, retain_graph=True)
    for i in range(3):
        want = torch.autograd.grad(out, leaves, d[i], retain_graph=True)
        for g, w in zip(got, want):
            assert rel(g[i], w.double().cpu()) <= 6e-6, tuple(w.shape)        # twice the bar of the kernels: two fp32 results
    jac = torch.autograd.functional.jacobian(lambda t: mlp(t), x.detach()[:, :2], vectorize=True)
    assert jac.shape == (1, 2, 16, 1, 2, 16) and torch.isfinite(jac).all()


def test_traced_graphs_hold_the_expressions(gpu):
    # make_fx records torch operators: a graph recorded past a kernel would replay with whatever its output buffer held
    from torch.fx.experimental.proxy_tensor import make_fx
    torch.manual_seed(2)
    layer = pa.Encoder(d_model=64, heads=2, d_hidden=96, dropout=0.0).to(gpu)

    def forward(a, b):
        return layer._residual_norm(a, layer.ffn(b), layer.attn_norm)

    def gradient(a, b):
        # (cubes: the sum of squares of a normalised row is constant, its gradient a rounding error)
        return torch.autograd.grad((forward(a, b) ** 3).sum(), [layer.ffn.in_proj.bias, layer.attn_norm.weight])
    for f in (lambda a, b: (forward(a, b),), gradient):
        graph = make_fx(f)(*(torch.randn(1, 9, 64, device=gpu) for _ in range(2)))
        args = [torch.randn(1, 9, 64, device=gpu) for _ in range(2)]
        for g, w in zip(graph(*args), f(*args)):
            assert rel(g.detach(), w.detach().double().cpu()) <= 6e-6          # twice the bar of the kernels: two fp32 results


def test_tangents_of_gradients_come_through(gpu):
    # a graph recorded outside dual_level, differentiated inside it with a dual gradient: gradients are linear in it
    import torch.autograd.forward_ad as fwad
    torch.manual_seed(3)
    mlp, norm, emb = pa.MLP(d_in=16, d_out=16, d_hidden=24, dropout=0.0).to(gpu), nn.LayerNorm(16).to(gpu), nn.Embedding(7, 16).to(gpu)
    x = torch.randn(1, 9, 16, device=gpu, requires_grad=True)
    out = train_ops.add_layer_norm(train_ops.embedding(torch.randint(0, 7, (1, 9), device=gpu), emb), mlp(x), norm)
    leaves = [x, emb.weight, *norm.parameters(), *mlp.parameters()]
    d, t = torch.randn_like(out), torch.randn_like(out)
    with fwad.dual_level():
        got = [fwad.unpack_dual(g) for g in torch.autograd.grad(out, leaves, fwad.make_dual(d, t), retain_graph=True)]
        got = [(g.primal, g.tangent) for g in got]
    want = [torch.autograd.grad(out, leaves, v, retain_graph=True) for v in (d, t)]
    for (p, q), wp, wt in zip(got, *want):
        assert rel(p, wp.double().cpu()) <= 6e-6 and q is not None and rel(q, wt.double().cpu()) <= 6e-6      # two fp32 results


def test_more_features_than_the_layout_kernel_takes(gpu):
    # proteus_heads_layout takes up to 16384: beyond, the module trains through its expression
    with torch.device(gpu):
        m = pa.GeoAttention(d_model=129 * 128, heads=129)
    x = torch.randn(1, 3, 129 * 128, device=gpu)
    coords = synth.random_walk_chain(3, torch.Generator().manual_seed(0)).unsqueeze(0).to(gpu)
    assert train_ops.self_attention(x, coords, None, m) is None
    g, = torch.autograd.grad(m(x, x, x, coords).sum(), [m.v_bias])
    assert g.shape == m.v_bias.shape and torch.isfinite(g).all()


def test_what_the_kernels_refuse_the_expressions_take(gpu):
    norm = nn.LayerNorm(16, eps=-1e-6).to(gpu)
    x = torch.randn(1, 9, 16, device=gpu, requires_grad=True)
    assert train_ops.add_layer_norm(x, x, norm) is None and torch.isfinite(pa.Encoder._residual_norm(x, x, norm)).all()
    mlp = pa.MLP(d_in=4, d_out=4, d_hidden=4, dropout=0.0).to(gpu)
    rows = torch.zeros(1, 1, 4, device=gpu).expand(1, 65535 * 2048 + 1, 4)
    assert train_ops.gelu_mlp(rows, mlp.in_proj, mlp.out_proj) is None
    # the embedding's gradient keeps a table of all rows in LDS: 64 of them
    tokens = torch.randint(0, 64, (5,), device=gpu)
    assert train_ops.embedding(tokens, nn.Embedding(64, 12).to(gpu)) is not None
    assert train_ops.embedding(tokens, nn.Embedding(65, 12).to(gpu)) is None


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_backward_inside_an_autocast_region(gpu, dtype):
    # a forward outside autocast (or in a region that disables it), differentiated inside: products in 16 bits would be handed
    # to kernels that read fp32
    torch.manual_seed(4)
    layer = pa.Encoder(d_model=128, heads=2, d_hidden=192, dropout=0.0).to(gpu)
    emb = nn.Embedding(7, 128).to(gpu)
    coords = synth.random_walk_chain(65, torch.Generator().manual_seed(0)).unsqueeze(0).to(gpu)
    x = train_ops.embedding(torch.randint(0, 7, (1, 65), device=gpu), emb)
    out = layer(x, x, x, coords)
    leaves = [emb.weight] + [p for n, p in layer.named_parameters() if not n.endswith("beta_weights")]
    d = torch.randn_like(out)
    want = torch.autograd.grad(out, leaves, d, retain_graph=True)
    with torch.autocast("cuda", dtype=dtype):
        got = torch.autograd.grad(out, leaves, d)
    for g, w in zip(got, want):
        # twice the bar of the kernels: two fp32 results (the spreads' gradient: sums in the order of atomics)
        assert rel(g, w.double().cpu()) <= (1e-4 if w.shape == layer.attn.spread_weights.shape else 6e-6), tuple(w.shape)


def _layer_and_inputs(gpu):
    torch.manual_seed(5)
    layer = pa.Encoder(d_model=64, heads=2, d_hidden=96, dropout=0.0).to(gpu)
    coords = synth.random_walk_chain(33, torch.Generator().manual_seed(0)).unsqueeze(0).to(gpu)
    return layer, nn.Embedding(7, 64).to(gpu), torch.randint(0, 7, (1, 33), device=gpu), coords


def test_saved_tensors_that_come_back_lying_differently(gpu):
    # saved-tensor hooks may give back tensors with other strides, at addresses that are multiples of 4 bytes only
    layer, emb, tokens, coords = _layer_and_inputs(gpu)
    leaves = [emb.weight] + [p for n, p in layer.named_parameters() if not n.endswith("beta_weights")]

    def gradients(unpack):
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
            x = train_ops.embedding(tokens, emb)
            out = layer(x, x, x, coords)
        return torch.autograd.grad(out, leaves, torch.ones_like(out).tril())

    def shifted(t):
        return torch.cat((t.new_zeros(1), t.reshape(-1)))[1:].view(t.shape)

    def strided(t):
        return torch.stack((t, t), -1)[..., 0]
    want = gradients(lambda t: t)
    for unpack in (shifted, strided):
        for g, w in zip(gradients(unpack), want):
            # twice the bar of the kernels: two fp32 results (the spreads' gradient: sums in the order of atomics)
            assert rel(g, w.double().cpu()) <= (1e-4 if w.shape == layer.attn.spread_weights.shape else 6e-6), tuple(w.shape)


def test_saved_tensors_of_another_type_are_refused(gpu):
    layer, emb, tokens, coords = _layer_and_inputs(gpu)
    x = torch.randn(1, 33, 64, device=gpu, requires_grad=True)
    for f in (lambda: train_ops.embedding(tokens, emb), lambda: layer.ffn(x), lambda: train_ops.add_layer_norm(x, x, layer.ffn_norm)):
        for unpack in (lambda t: t.to(torch.int32 if t.dtype == torch.int64 else torch.bfloat16), lambda t: t.cpu()):
            with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
                out = f()
            with pytest.raises(RuntimeError):
                out.sum().backward()


def test_outputs_may_be_changed_in_place(gpu):
    layer, emb, tokens, coords = _layer_and_inputs(gpu)
    x = torch.randn(1, 33, 64, device=gpu, requires_grad=True)
    for f in (lambda: train_ops.embedding(tokens, emb), lambda: layer.ffn(x), lambda: layer.attn(x, x, x, coords),
              lambda: train_ops.add_layer_norm(x, x, layer.ffn_norm)):
        out = f()
        assert out is not None and not out._is_view()
        out += 1.0
        out.sum().backward()


def test_parameters_may_change_between_forward_and_backward(gpu):
    # the attention's gradients are those of the parameters that the forward pass used
    layer, _, _, coords = _layer_and_inputs(gpu)
    x, params = torch.randn(1, 33, 64, device=gpu, requires_grad=True), [p for n, p in layer.attn.named_parameters() if n != "beta_weights"]
    out = layer.attn(x, x, x, coords)
    d = torch.randn_like(out)
    want = torch.autograd.grad(out, [x, *params], d, retain_graph=True)
    with torch.no_grad():
        for p in params:
            p.add_(0.1)
    for g, w in zip(torch.autograd.grad(out, [x, *params], d, retain_graph=True), want):
        assert rel(g, w.double().cpu()) <= (1e-4 if w.shape == layer.attn.spread_weights.shape else 6e-6), tuple(w.shape)
    with pytest.raises(RuntimeError, match="changed in place"):
        torch.autograd.grad(out, [x], d, create_graph=True)


def test_frozen_weights_leave_the_input_free(gpu):
    # as with torch's products, whose gradient of the input needs the weights alone
    layer, _, _, coords = _layer_and_inputs(gpu)
    for p in layer.parameters():
        p.requires_grad_(False)
    leaf = torch.randn(1, 33, 64, device=gpu, requires_grad=True)
    for f in (layer.ffn, lambda t: layer.attn(t, t, t, coords)):
        x = leaf * 2.0
        out = f(x)
        x += out
        g, = torch.autograd.grad(x.sum(), [leaf])
        assert torch.isfinite(g).all()


def test_parameters_of_other_shapes_are_the_expressions_to_refuse(gpu):
    # the kernels would read past the end of a smaller parameter; the expressions raise
    layer, _, _, coords = _layer_and_inputs(gpu)
    x = torch.randn(1, 33, 64, device=gpu, requires_grad=True)
    layer.attn.spread_weights = nn.Parameter(torch.zeros(1, device=gpu))
    with pytest.raises(AssertionError):
        layer.attn(x, x, x, coords)
    layer.ffn_norm.bias = nn.Parameter(torch.zeros(4, device=gpu))
    with pytest.raises(RuntimeError):
        layer._residual_norm(x, x, layer.ffn_norm)


def test_minimal_spreads_in_a_tensor_keep_the_general_path(gpu):
    layer, _, _, coords = _layer_and_inputs(gpu)
    x = torch.randn(1, 33, 64, device=gpu, requires_grad=True)
    layer.attn.min_spread = torch.tensor([2.0, 3.0], device=gpu, requires_grad=True)
    g, = torch.autograd.grad(layer.attn(x, x, x, coords).square().sum(), [layer.attn.min_spread])
    assert torch.isfinite(g).all() and g.any()
