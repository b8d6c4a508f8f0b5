"""The encoder's training step between its matrix products, as autograd functions on the HIP kernels of encoder_train.hip.

Each function stands for a torch expression that the modules keep as their general path (fp32 tensors on the GPU take
these; anything else, e.g. other types, autocast, functional transforms, forward-mode differentiation, tracing, dispatch
modes, tensor subclasses, modules with hooks, takes the expression).  A backward that is itself recorded (create_graph) differentiates
the expression.
"""
import ctypes
import functools

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import _lib
from . import geometric_attn as ga

_PLAIN_TYPES = (torch.Tensor, nn.Parameter)


def recording(*tensors):
    """Does plain reverse-mode autograd record an operator on these tensors, all of them ordinary fp32 tensors on one GPU?"""
    if not torch.is_grad_enabled() or torch.is_autocast_enabled("cuda"):
        return False
    needed = False
    dev = tensors[0].get_device()
    if not tensors[0].is_cuda:
        return False
    for t in tensors:
        if type(t) not in _PLAIN_TYPES or t.dtype != torch.float32 or t.get_device() != dev or t.layout != torch.strided:
            return False
        needed = needed or t.requires_grad
    return needed and unobserved()


def unobserved():
    """Does nothing look on that expects torch operators: no functional transform, forward-mode differentiation, tracing or dispatch mode?
    (A dispatch mode, e.g. make_fx's, sees the torch operators only: a graph traced past a kernel would not hold what it writes.)"""
    return (torch.autograd.forward_ad._current_level < 0 and torch._C._functorch.peek_interpreter_stack() is None
            and torch._C._len_torch_dispatch_stack() == 0 and not torch.jit.is_tracing() and not torch.compiler.is_compiling())


def plain_module(m, cls):
    """Is `m` exactly a `cls` whose call is its forward: no hooks, no replaced forward?"""
    g = nn.modules.module
    return (type(m) is cls and "forward" not in m.__dict__
            and not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks
                     or g._global_forward_hooks or g._global_forward_pre_hooks or g._global_backward_hooks or g._global_backward_pre_hooks))


def inactive_dropout(m):
    return plain_module(m, nn.Dropout) and (m.p == 0.0 or not m.training)


def aligned(*tensors):
    return all(t.is_contiguous() and t.data_ptr() % 16 == 0 for t in tensors)


def _call(fn, dev, *args):
    """One entry point on torch's current stream; tensors stand for their addresses."""
    with _lib.on_device(dev):
        rc = getattr(_lib.load(), fn)(*[a.data_ptr() if isinstance(a, torch.Tensor) else a for a in args], _lib.raw_stream(dev))
    _lib.check(rc, fn)


@functools.lru_cache(maxsize=1024)
def _bytes(fn, *sizes):
    """What the library answers for a workspace's size, kept per sizes."""
    return getattr(_lib.load(), fn)(*sizes)


def _workspace(nbytes, dev):
    return torch.empty(nbytes, dtype=torch.uint8, device=dev) if nbytes else None


def _dense(t):
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


def _by_expression(d):
    """Does a backward that is handed the gradient `d` differentiate the expression?  Where it is itself recorded, where `d` has
    no memory of its own for a kernel to read (batched gradients: is_grads_batched, jacobians by vmap), where it may carry a tangent
    (forward-mode differentiation), and under a dispatch mode."""
    return (torch.is_grad_enabled() or type(d) not in _PLAIN_TYPES or not torch._C._has_storage(d) or torch.autograd.forward_ad._current_level >= 0
            or torch._C._functorch.peek_interpreter_stack() is not None or torch._C._len_torch_dispatch_stack() > 0)


def _saved(t, numel, dev, dtype=torch.float32):
    """A saved tensor as a kernel on `dev` may read it.  What saved-tensor hooks give back may lie differently (strides, alignment);
    another type, size or place is an error, as it would be in a torch operator."""
    if t.dtype != dtype or t.numel() != numel or t.device != dev:
        raise RuntimeError(f"a tensor of {numel} {dtype} that was saved on {dev} came back as {tuple(t.shape)} of {t.dtype} on {t.device}")
    return t if t.is_contiguous() and t.data_ptr() % 16 == 0 else _dense(t)


def _saved_sizes(*tensors_and_sizes):
    """Saved tensors of the attention, which takes any type and place of them, hold what the forward saved."""
    for t, numel in tensors_and_sizes:
        if t is not None and t.numel() != numel:
            raise RuntimeError(f"a tensor of {numel} elements that was saved came back as {tuple(t.shape)}")


def _without_autocast(backward):
    """A backward whose products stay in fp32 as its forward's are (`recording`): under autocast, which holds for products of a
    backward called inside its region, they would come out in 16 bits, and the kernels would read past their ends."""
    @functools.wraps(backward)
    def run(ctx, *grads):
        if not torch.is_autocast_enabled("cuda"):
            return backward(ctx, *grads)
        with torch.autocast("cuda", enabled=False):
            return backward(ctx, *grads)
    return run


def _recorded(expr, inputs, needs, grad):
    """Gradients of expr(*inputs) for the inputs that need one, as a graph of their own where gradients are recorded."""
    create_graph = torch.is_grad_enabled()
    with torch.enable_grad():
        wanted = [t for t, n in zip(inputs, needs) if n]
        # (retain_graph: the inputs may be outputs of the very node whose backward this is)
        got = iter(torch.autograd.grad(expr(*inputs), wanted, grad, create_graph=create_graph, retain_graph=True, allow_unused=True))
    return tuple(next(got) if n else None for n in needs)


def column_sums(a):
    """Column sums of a [rows, C]."""
    rows, C = a.shape
    sums = torch.empty(C, dtype=torch.float32, device=a.device)
    n = _bytes("proteus_train_workspace_bytes", rows, C)
    _call("proteus_colsum", a.device, a, sums, _workspace(n, a.device), n, rows, C)
    return sums


# ---------------------------------------------------------------------------------------------------- matrix products

NN, NT, TN = _lib.GEMM_NN, _lib.GEMM_NT, _lib.GEMM_TN


def _product(form, A, B, bias=None, gelu=False, gelu_grad_of=None):
    """A B (NN), A B^T (NT) or A^T B (TN) of dense fp32 matrices, plus `bias` per column: one launch of the library's product, which
    issues in a fifth of the host time of torch's; torch's where rows are not multiples of 16 bytes or a matrix has 2 GiB.
    gelu (NT): returns (sums, gelu(sums)); gelu_grad_of (NN): sums * gelu'(gelu_grad_of)."""
    M, K = A.shape if form != TN else A.shape[::-1]
    N = B.shape[0] if form == NT else B.shape[1]
    if not ((form == TN or K % 4 == 0) and (A.shape[0] + 512) * A.shape[1] < 2 ** 29 and (B.shape[0] + 512) * B.shape[1] < 2 ** 29):
        Am, Bm = A.t() if form == TN else A, B.t() if form == NT else B
        C = Am.mm(Bm) if bias is None else torch.addmm(bias, Am, Bm)
        if gelu:
            return C, F.gelu(C)
        return C if gelu_grad_of is None else torch.ops.aten.gelu_backward(C, gelu_grad_of)
    C = torch.empty(M, N, dtype=torch.float32, device=A.device)
    H = torch.empty_like(C) if gelu else None
    epilogue = _lib.GEMM_GELU if gelu else _lib.GEMM_GELU_GRAD if gelu_grad_of is not None else _lib.GEMM_F32
    n = _bytes("proteus_gemm_f32_workspace_bytes", M, N, K, form) if form == TN else 0
    _call("proteus_gemm_f32_ws", A.device, A, B, bias, gelu_grad_of, C, H, M, N, K, A.shape[1], B.shape[1], N, form, epilogue, _workspace(n, A.device), n)
    return (H, C) if gelu else C


# ---------------------------------------------------------------------------------------------------- add + LayerNorm

class _AddLayerNorm(torch.autograd.Function):
    """(LayerNorm(x + res), x + res): the sum is an output so that a recorded backward stays connected to x and res without
    keeping either."""

    @staticmethod
    def forward(ctx, x, res, w, b, eps):
        D = x.shape[-1]
        rows = x.numel() // D
        xc, rc_ = _dense(x), _dense(res)
        out, ysum = torch.empty_like(xc), torch.empty_like(xc)
        stat = torch.empty(rows, 2, dtype=torch.float32, device=x.device)
        _call("proteus_add_layernorm_train_fwd", x.device, xc, rc_, w, b, out, ysum, stat, rows, D, eps)
        ctx.save_for_backward(ysum, stat, w, b)
        ctx.eps = eps
        ctx.set_materialize_grads(False)
        return out, ysum

    @staticmethod
    @_without_autocast
    def backward(ctx, d, dy):
        ysum, stat, w, b = ctx.saved_tensors
        need = ctx.needs_input_grad
        if d is None:
            return dy if need[0] else None, dy if need[1] else None, None, None, None
        if _by_expression(d):
            dx, dw, db = _recorded(lambda y_, w_, b_: F.layer_norm(y_, (w.numel(),), w_, b_, ctx.eps), (ysum, w, b), (True, need[2], need[3]), d)
        else:
            d, D, dev = _dense(d), d.shape[-1], d.device
            rows = d.numel() // D
            w, ysum, stat = _saved(w, D, dev), _saved(ysum, rows * D, dev), _saved(stat, 2 * rows, dev)
            dx = torch.empty_like(ysum)
            dwb = torch.empty(2, D, dtype=torch.float32, device=d.device)
            n = _bytes("proteus_layernorm_bwd_workspace_bytes", rows, D)
            _call("proteus_layernorm_bwd", d.device, d, ysum, stat, w, dx, dwb, _workspace(n, d.device), n, rows, D)
            dw, db = dwb[0] if need[2] else None, dwb[1] if need[3] else None
        if dy is not None:
            dx = dx + dy
        return dx if need[0] else None, dx if need[1] else None, dw, db, None


def add_layer_norm(x, res, norm):
    """norm(x + res), or None where the kernels do not take it."""
    if not torch.is_grad_enabled():
        return None
    w, b = norm.weight, norm.bias
    if (w is None or b is None or not plain_module(norm, nn.LayerNorm) or x.shape != res.shape or x.dim() < 1 or w.dim() != 1 or b.shape != w.shape
            or w.numel() != x.shape[-1] or x.numel() == 0 or w.numel() % 4 or w.numel() > 2048 or not norm.eps >= 0.0
            or not recording(x, res, w, b) or not aligned(w, b)):
        return None
    return _AddLayerNorm.apply(x, res, w, b, float(norm.eps))[0]


# ---------------------------------------------------------------------------------------------------- feed-forward

class _GeluMLP(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w1, b1, w2, b2):
        x2 = _dense(x).view(-1, x.shape[-1])
        h, a = _product(NT, x2, _dense(w1), _dense(b1), gelu=True)
        ctx.save_for_backward(x, w1, b1, w2, b2, h, a)
        # (resized, not viewed: autograd lets no view that a function returns be changed in place)
        return _product(NT, a, _dense(w2), _dense(b2)).resize_(*x.shape[:-1], w2.shape[0])

    @staticmethod
    @_without_autocast
    def backward(ctx, d):
        x, w1, b1, w2, b2, h, a = ctx.saved_tensors
        need = ctx.needs_input_grad
        if _by_expression(d):
            return _recorded(lambda x_, w1_, b1_, w2_, b2_: F.linear(F.gelu(F.linear(x_, w1_, b1_)), w2_, b2_), (x, w1, b1, w2, b2), need, d)
        d_out, (hidden, d_in), dev = d.shape[-1], w1.shape, d.device
        d2 = _dense(d).view(-1, d_out)
        rows = d2.shape[0]
        x2, a = _saved(x, rows * d_in, dev).view(rows, d_in), _saved(a, rows * hidden, dev).view(rows, hidden)
        w1, w2, h = _saved(w1, hidden * d_in, dev).view(hidden, d_in), _saved(w2, d_out * hidden, dev).view(d_out, hidden), _saved(h, rows * hidden, dev)
        dw2 = _product(TN, d2, a) if need[3] else None
        db2 = column_sums(d2) if need[4] else None
        dx = dw1 = db1 = None
        if need[0] or need[1] or need[2]:
            dh = _product(NN, d2, w2, gelu_grad_of=h)
            db1 = column_sums(dh) if need[2] else None
            dw1 = _product(TN, dh, x2) if need[1] else None
            dx = _product(NN, dh, w1).view(x.shape) if need[0] else None
        return dx, dw1, db1, dw2, db2


def gelu_mlp(x, lin1, lin2):
    """lin2(gelu(lin1(x))), or None where the kernels do not take it."""
    if not torch.is_grad_enabled():
        return None
    if not (plain_module(lin1, nn.Linear) and plain_module(lin2, nn.Linear)) or lin1.bias is None or lin2.bias is None:
        return None
    w1, b1, w2, b2 = lin1.weight, lin1.bias, lin2.weight, lin2.bias
    # (what does not have a linear layer's shapes is the expression's to broadcast or to refuse: the products read biases unseen)
    if w1.dim() != 2 or w2.dim() != 2 or b1.shape != w1.shape[:1] or b2.shape != w2.shape[:1]:
        return None
    # (a frozen first layer keeps the expression, which does not keep x: x may be changed in place behind it)
    if (not w1.requires_grad or x.dim() < 2 or x.shape[-1] != w1.shape[1] or w1.shape[0] != w2.shape[1] or x.numel() == 0 or w1.shape[0] % 4 or w2.shape[0] % 4
            or x.numel() // x.shape[-1] > 65535 * 2048        # (rows of a column sum)
            or not recording(x, w1, b1, w2, b2)):
        return None
    return _GeluMLP.apply(x, w1, b1, w2, b2)


# ---------------------------------------------------------------------------------------------------- self-attention

def _self_attention_expression(x, coords, mask, qw, kw, vw, qb, kb, vb, spread_w, wo, min_spread, operand_dtype):
    H, dm, dk = qw.shape
    Z, N, _ = x.shape
    w = torch.stack((qw, kw, vw)).permute(2, 0, 1, 3).reshape(dm, 3 * H * dk)
    b = torch.stack((qb, kb, vb)).reshape(-1)
    qkv = torch.addmm(b, x.reshape(Z * N, dm), w).view(Z, N, 3, H, dk)
    O = ga.geometric_attn_qkv(qkv, coords, min_spread + torch.exp(spread_w), None, mask=mask, check_spreads=False, out_dtype=x.dtype,
                              operand_dtype=operand_dtype)
    return F.linear(O.permute(0, 2, 1, 3).reshape(Z, N, dm), wo.view(dm, dk, H).permute(0, 2, 1).reshape(dm, dm))


def _layout(tensors, W, b, Wo, sigma, spread_w, dm, H, dk, min_spread, backward):
    ptrs = (ctypes.c_void_p * 8)(*[None if t is None else t.data_ptr() for t in tensors])
    _call("proteus_heads_layout", W.device, ptrs, W, b, Wo, sigma, spread_w, dm, H, dk, float(min_spread), backward)


def _heads(qkv):
    return tuple(qkv[:, :, i].permute(0, 2, 1, 3) for i in range(3))


class _SelfAttention(torch.autograd.Function):
    """Projections, attention and output projection of one self-attention layer.  The heads' weights are laid side by side
    by one launch, the fused projection is cast to the operand type once (kept for the backward in that type), and the
    gradients of the heads' weights and biases leave through one launch."""

    @staticmethod
    def forward(ctx, x, coords, mask, qw, kw, vw, qb, kb, vb, spread_w, wo, min_spread, operand_dtype):
        H, dm, dk = qw.shape
        Z, N, _ = x.shape
        dev = x.device
        W = torch.empty(dm, 3 * dm, dtype=torch.float32, device=dev)
        Wo = torch.empty(dm, dm, dtype=torch.float32, device=dev)
        b = torch.empty(3 * dm, dtype=torch.float32, device=dev)
        sigma, spread = torch.empty(H, dtype=torch.float32, device=dev), torch.empty(H, dtype=torch.float32, device=dev)
        _layout((qw, kw, vw, qb, kb, vb, spread, wo), W, b, Wo, sigma, spread_w, dm, H, dk, min_spread, 0)
        # (torch's product: its sums are rounded to 16 bits next, and the expression's roundings are the ones to make)
        qkv = torch.addmm(b, _dense(x).view(Z * N, dm), W).to(operand_dtype or torch.bfloat16).view(Z, N, 3, H, dk)
        O, L = ga.geo_attn(*_heads(qkv), coords, sigma, mask, return_lse=True, check_sigma=False, token_major_out=True,
                           operand_dtype=operand_dtype)
        ctx.save_for_backward(x, coords, mask, W, Wo, sigma, spread, qkv, O, L)
        # The parameters themselves are wanted by the expression only: what a backward reads of them it has as copies, so that they
        # may be changed (an optimizer's step) between forward and backward.
        ctx.params = (qw, kw, vw, qb, kb, vb, spread_w, wo)
        ctx.versions = [p._version for p in ctx.params]
        ctx.min_spread, ctx.operand_dtype = min_spread, operand_dtype
        return _product(NT, O.permute(0, 2, 1, 3).reshape(Z * N, dm), Wo).resize_(Z, N, dm)       # (as in the feed-forward)

    @staticmethod
    @_without_autocast
    def backward(ctx, d):
        x, coords, mask, W, Wo, sigma, spread, qkv, O, L = ctx.saved_tensors
        need, params = ctx.needs_input_grad, ctx.params
        if _by_expression(d):
            if any(p._version != v for p, v in zip(params, ctx.versions)):
                raise RuntimeError("a parameter of the self-attention was changed in place after the forward pass whose gradient is recorded")
            gx, *gp = _recorded(lambda x_, *p: _self_attention_expression(x_, coords, mask, *p, ctx.min_spread, ctx.operand_dtype),
                                (x, *params), (need[0], *need[3:11]), d)
            return (gx, None, None, *gp, None, None)
        Z, N, dm = d.shape
        H, _, dk = params[0].shape
        dev = d.device
        d2 = _dense(d).view(Z * N, dm)
        W, Wo, x2 = _saved(W, 3 * dm * dm, dev).view(dm, 3 * dm), _saved(Wo, dm * dm, dev).view(dm, dm), _saved(x, Z * N * dm, dev).view(Z * N, dm)
        _saved_sizes((coords, Z * N * 3), (mask, Z * N), (L, Z * H * N), (sigma, H))
        if tuple(qkv.shape) != (Z, N, 3, H, dk) or tuple(O.shape) != (Z, H, N, dk):
            raise RuntimeError(f"the projection and the output of {(Z, N, H, dk)} that were saved came back as {tuple(qkv.shape)} and {tuple(O.shape)}")
        dO = _product(NN, d2, Wo).view(Z, N, H, dk).permute(0, 2, 1, 3)
        g = torch.empty(qkv.shape, dtype=torch.float32, device=dev)
        _, _, _, d_sigma, _ = ga._backward(*_heads(qkv), O, L, dO, coords, sigma, mask, None, 0.0, 1.0, ctx.operand_dtype, grads=_heads(g))
        g2 = g.view(Z * N, 3 * dm)
        dx = _product(NT, g2, W).view(x.shape) if need[0] else None
        grads = [torch.empty_like(p, memory_format=torch.contiguous_format) if n else None for p, n in zip(params, need[3:11])]
        # (what a gradient is not asked of is not looked at: its place in the list is None)
        dW = _product(TN, x2, g2) if any(need[3:6]) else g2
        db = column_sums(g2) if any(need[6:9]) else g2
        dWo = _product(TN, d2, _saved(O.permute(0, 2, 1, 3), Z * N * dm, dev).view(Z * N, dm)) if need[10] else g2
        _layout(grads, dW, db, dWo, d_sigma, _saved(spread, H, dev), dm, H, dk, ctx.min_spread, 1)
        return (dx, None, None, *grads, None, None)


def self_attention(x, coords, mask, m):
    """The output of the GeoAttention module `m` (README logits) on x, x, x, or None where the kernels do not take it."""
    if not torch.is_grad_enabled():
        return None
    H, dk, dm = m.heads, m.d_k, m.d_model
    params = (m.q_proj, m.k_proj, m.v_proj, m.q_bias, m.k_bias, m.v_bias, m.spread_weights, m.out_proj.weight)
    # (whatever does not have the shape it was constructed with is the expression's to judge)
    if not (params[0].shape == params[1].shape == params[2].shape == (H, dm, dk) and params[3].shape == params[4].shape == params[5].shape == (H, dk)
            and params[6].shape == (H,) and params[7].shape == (dm, dm)):
        return None
    # (frozen projections keep the expression, which does not keep x: x may be changed in place behind it)
    if (not (params[0].requires_grad or params[1].requires_grad or params[2].requires_grad) or m.legacy_logits or dk not in (32, 64, 128) or dm > 16384 or x.numel() == 0 or not coords.is_cuda or coords.requires_grad or type(coords) not in _PLAIN_TYPES
            or (mask is not None and type(mask) is not torch.Tensor)
            or x.shape[1] * 3 * dm * 4 >= 2 ** 31 or m.operand_dtype not in (None, torch.bfloat16)
            or type(m).get_spreads is not ga.GeoAttention.get_spreads or "get_spreads" in m.__dict__ or not isinstance(m.min_spread, (int, float))
            or not recording(x, *params) or not aligned(*params)):
        return None
    return _SelfAttention.apply(x, coords, mask, *params, m.min_spread, m.operand_dtype)


# ---------------------------------------------------------------------------------------------------- encoder layer

def _layer_expression(x, coords, mask, qw, kw, vw, qb, kb, vb, spread_w, wo, g1, c1, w1, b1, w2, b2, g2, c2, min_spread, operand_dtype, eps1, eps2):
    x = F.layer_norm(x + _self_attention_expression(x, coords, mask, qw, kw, vw, qb, kb, vb, spread_w, wo, min_spread, operand_dtype), g1.shape, g1, c1, eps1)
    return F.layer_norm(x + F.linear(F.gelu(F.linear(x, w1, b1)), w2, b2), g2.shape, g2, c2, eps2)


def _pointers(tensors):
    return (ctypes.c_void_p * len(tensors))(*[None if t is None else t.data_ptr() for t in tensors])


class _EncoderLayer(torch.autograd.Function):
    """A whole post-LN layer: the launches of the functions above from one call of the library per direction."""

    @staticmethod
    def forward(ctx, x, coords, mask, *args):
        params, (min_spread, operand_dtype, eps1, eps2) = args[:16], args[16:]
        H, dm, dk = params[0].shape
        Z, N, _ = x.shape
        sizes = (Z, N, H, dk, params[10].shape[0])
        dev = x.device
        xc, c, m = _dense(x), ga._f32(coords, dev), None if mask is None else ga._mask_bytes(mask, dev)
        kept = torch.empty(_bytes("proteus_encoder_layer_kept_bytes", *sizes), dtype=torch.uint8, device=dev)
        n = _bytes("proteus_encoder_layer_fwd_bytes", *sizes)
        out = torch.empty(Z, N, dm, dtype=torch.float32, device=dev)
        _call("proteus_encoder_layer_fwd", dev, xc, c, m, _pointers(params), min_spread, eps1, eps2, out, kept, kept.numel(), _workspace(n, dev), n, *sizes)
        # (the attention's parameters may change before the backward, as in its own function: what it reads of them is kept as copies)
        ctx.save_for_backward(x, coords, mask, kept, *params[8:])
        ctx.params = params[:8]
        ctx.versions = [p._version for p in ctx.params]
        ctx.args, ctx.sizes = args[16:], sizes
        return out

    @staticmethod
    @_without_autocast
    def backward(ctx, d):
        x, coords, mask, kept, *rest = ctx.saved_tensors
        need, attn = ctx.needs_input_grad, ctx.params
        min_spread, operand_dtype, eps1, eps2 = ctx.args
        if _by_expression(d):
            if any(p._version != v for p, v in zip(attn, ctx.versions)):
                raise RuntimeError("a parameter of the self-attention was changed in place after the forward pass whose gradient is recorded")
            gx, *gp = _recorded(lambda x_, *p: _layer_expression(x_, coords, mask, *p, *ctx.args), (x, *attn, *rest), (need[0], *need[3:19]), d)
            return (gx, None, None, *gp, None, None, None, None)
        sizes = Z, N, H, dk, hidden = ctx.sizes                 # (the forward's: what the hooks of saved tensors give back is held against them)
        dm, dev = H * dk, d.device
        g1, c1, w1, b1, w2, b2, g2, c2 = rest
        g1, w1, w2, g2 = _saved(g1, dm, dev), _saved(w1, hidden * dm, dev), _saved(w2, dm * hidden, dev), _saved(g2, dm, dev)
        x2, kept = _saved(x, Z * N * dm, dev), _saved(kept, _bytes("proteus_encoder_layer_kept_bytes", *sizes), dev, torch.uint8)
        if kept.data_ptr() % 256:
            kept = kept.clone()
        _saved_sizes((coords, Z * N * 3), (mask, Z * N))
        c, m = ga._f32(coords, dev), None if mask is None else ga._mask_bytes(mask, dev)
        wanted = need[3:19]
        grads = [torch.empty_like(p, memory_format=torch.contiguous_format) if n and not 8 <= i <= 9 and i < 14 else None
                 for i, (p, n) in enumerate(zip((*attn, *rest), wanted))]
        for i in (8, 14):           # gamma's and beta's gradients are one array
            if wanted[i] or wanted[i + 1]:
                grads[i] = torch.empty(2, dm, dtype=torch.float32, device=dev)
        dx = torch.empty(Z, N, dm, dtype=torch.float32, device=dev) if need[0] else None
        n = _bytes("proteus_encoder_layer_bwd_bytes", *sizes)
        _call("proteus_encoder_layer_bwd", dev, x2, c, m, _pointers((None,) * 8 + (g1, None, w1, None, w2, None, g2, None)), _dense(d), dx, _pointers(grads),
              min_spread, kept, kept.numel(), _workspace(n, dev), n, *sizes)
        for i in (8, 14):
            both = grads[i]
            if both is not None:
                grads[i], grads[i + 1] = both[0] if wanted[i] else None, both[1] if wanted[i + 1] else None
        return (dx, None, None, *grads, None, None, None, None)


def encoder_layer(x, coords, mask, m, mlp_class):
    """The output of the Encoder module `m` (self-attention, `mlp_class` its feed-forward) on x, or None where its parts go their own ways."""
    if not torch.is_grad_enabled() or x.dtype != torch.float32 or not x.is_cuda or torch.is_autocast_enabled("cuda"):
        return None                                                         # (what most other calls fail at, before the closer look)
    if not inactive_dropout(m.dropout):
        return None
    a, n1, f, n2 = m.attn, m.attn_norm, m.ffn, m.ffn_norm
    lin1, lin2 = getattr(f, "in_proj", None), getattr(f, "out_proj", None)
    if not (plain_module(a, ga.GeoAttention) and plain_module(n1, nn.LayerNorm) and plain_module(n2, nn.LayerNorm)
            and plain_module(f, mlp_class) and f.act is F.gelu and not f.hidden_proj and inactive_dropout(f.in_dropout)
            and plain_module(lin1, nn.Linear) and plain_module(lin2, nn.Linear) and plain_module(a.out_proj, nn.Linear) and "_residual_norm" not in m.__dict__):
        return None
    H, dk, dm = a.heads, a.d_k, a.d_model
    params = (a.q_proj, a.k_proj, a.v_proj, a.q_bias, a.k_bias, a.v_bias, a.spread_weights, a.out_proj.weight,
              n1.weight, n1.bias, lin1.weight, lin1.bias, lin2.weight, lin2.bias, n2.weight, n2.bias)
    if any(p is None for p in params):
        return None
    hidden = lin1.weight.shape[0]
    w, b = (H, dm, dk), (H, dk)
    if tuple(p.shape for p in params) != (w, w, w, b, b, b, (H,), (dm, dm), (dm,), (dm,), (hidden, dm), (hidden,), (dm, hidden), (dm,), (dm,), (dm,)):
        return None
    # (frozen weights: the parts, which keep of the inputs only what they read again; spreads and what follows a product may be frozen)
    if (not all(params[i].requires_grad for i in (0, 1, 2, 10, 12)) or a.legacy_logits or x.dim() != 3 or x.shape[2] != dm or x.numel() == 0
            or type(coords) is not torch.Tensor or coords.device != x.device or tuple(coords.shape) != (*x.shape[:2], 3) or coords.requires_grad
            or (mask is not None and (type(mask) is not torch.Tensor or tuple(mask.shape) != tuple(x.shape[:2])))
            or a.operand_dtype not in (None, torch.bfloat16) or not isinstance(a.min_spread, (int, float)) or "get_spreads" in a.__dict__
            or a.out_proj.bias is not None or not (n1.eps >= 0.0 and n2.eps >= 0.0)
            or not recording(x, *params) or not aligned(*params)
            or _bytes("proteus_encoder_layer_kept_bytes", *x.shape[:2], H, dk, hidden) == 0):
        return None
    return _EncoderLayer.apply(x, coords, mask, *params, a.min_spread, a.operand_dtype, float(n1.eps), float(n2.eps))


# ---------------------------------------------------------------------------------------------------- token embedding

class _SmallEmbedding(torch.autograd.Function):
    @staticmethod
    def forward(ctx, weight, tokens):
        ctx.save_for_backward(weight, tokens)
        return F.embedding(tokens, weight)

    @staticmethod
    @_without_autocast
    def backward(ctx, d):
        weight, tokens = ctx.saved_tensors
        if _by_expression(d):
            return (*_recorded(lambda w: F.embedding(tokens, w), (weight,), (True,), d), None)
        V, D = weight.shape
        d, t = _dense(d), _saved(tokens, d.numel() // D, d.device, torch.int64)
        dW = torch.empty(V, D, dtype=torch.float32, device=d.device)
        n = _bytes("proteus_embedding_bwd_workspace_bytes", t.numel(), V, D)
        _call("proteus_embedding_bwd", d.device, d, t, dW, _workspace(n, d.device), n, t.numel(), V, D)
        return dW, None


def embedding(tokens, m):
    """m(tokens) for an nn.Embedding of few rows, or None where the kernel does not take its gradient."""
    if not torch.is_grad_enabled():
        return None
    if not (plain_module(m, nn.Embedding) and m.padding_idx is None and m.max_norm is None and not m.scale_grad_by_freq and not m.sparse):
        return None
    V, D = m.weight.shape
    if (V > 64 or D % 4 or D > 16384 or type(tokens) is not torch.Tensor or tokens.dtype != torch.int64 or tokens.device != m.weight.device
            or tokens.numel() == 0 or tokens.numel() > 65535 * 128 or not recording(m.weight)):
        return None
    return _SmallEmbedding.apply(m.weight, tokens)
