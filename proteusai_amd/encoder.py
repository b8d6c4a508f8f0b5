"""Encoder stack around the two kernels.

Follows the legacy transformer architecture the reference's README describes
(README.md:38,48) and its code:
  MLP                          utils/model_utils/base_modules/base_modules.py:6-52
  Encoder (post-LN layer)      old/old_scripts/encoder.py:8-41
  GeoAttention                 old/old_scripts/encoder.py:43-121  (proteusai_amd.geometric_attn.GeoAttention)
The wavefunction embedding is added to an amino-acid embedding table and the
sum runs through the encoder layers and a linear head to 20 amino-acid logits.
Plain PyTorch glue but for the residual add + LayerNorm of a layer; the two O(N^2) operators are the HIP kernels.
"""
import torch
import torch.nn as nn
import torch.nn.functional as F

from . import _lib, train_ops
from .geometric_attn import GeoAttention, _f32, _mask_bytes
from .wf_embedding import WaveFunctionEmbedding


def add_layer_norm(x, res, norm: nn.LayerNorm):
    """norm(x + res) for the post-LN layer (old/old_scripts/encoder.py:36-39).

    Where nothing needs a gradient (inference) and the tensors are fp32 or bf16 on the GPU, one HIP kernel reads x and
    res once and writes the result (proteus_add_layernorm_fwd); otherwise the torch expression, which autograd
    differentiates.  Both evaluate the same thing: the sum in the tensors' type, the statistics in fp32.
    """
    w, b = norm.weight, norm.bias
    D = x.shape[-1]
    needs_grad = torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in (x, res, w, b))
    fused = (not needs_grad and x.is_cuda and x.dtype in (torch.float32, torch.bfloat16) and res.dtype == x.dtype
             and x.shape == res.shape and tuple(norm.normalized_shape) == (D,)
             and all(t is None or t.dtype == x.dtype for t in (w, b))
             and D % (4 if x.dtype == torch.float32 else 8) == 0 and D <= (2048 if x.dtype == torch.float32 else 4096))
    if not fused:
        return norm(x + res)
    lib = _lib.load()
    xc, rc_ = x.contiguous(), res.contiguous()
    out = torch.empty_like(xc)
    rows = xc.numel() // D
    if rows == 0:
        return out
    with _lib.on_device(x.device):
        rc = lib.proteus_add_layernorm_fwd(xc.data_ptr(), rc_.data_ptr(), None if w is None else w.data_ptr(),
                                           None if b is None else b.data_ptr(), out.data_ptr(), rows, D, float(norm.eps),
                                           _lib.DTYPE_F32 if x.dtype == torch.float32 else _lib.DTYPE_BF16,
                                           _lib.raw_stream(x.device))
    _lib.check(rc, "proteus_add_layernorm_fwd")
    return out


class MLP(nn.Module):
    """in_proj -> act -> [hidden -> act]* -> out_proj, dropout after each activation (base_modules.py:6-52)."""

    def __init__(self, d_in=512, d_out=512, d_hidden=1024, hidden_layers=0, dropout=0.1, act="gelu"):
        super().__init__()
        self.in_proj = nn.Linear(d_in, d_hidden)
        self.hidden_proj = nn.ModuleList([nn.Linear(d_hidden, d_hidden) for _ in range(hidden_layers)])
        self.out_proj = nn.Linear(d_hidden, d_out)
        self.in_dropout = nn.Dropout(dropout)
        self.hidden_dropout = nn.ModuleList([nn.Dropout(dropout) for _ in range(hidden_layers)])
        self.act = {"gelu": F.gelu, "silu": F.silu, "relu": F.relu, "sigmoid": torch.sigmoid}.get(act, lambda x: x)
        nn.init.xavier_uniform_(self.in_proj.weight)
        nn.init.zeros_(self.in_proj.bias)
        for layer in self.hidden_proj:
            nn.init.kaiming_uniform_(layer.weight, nonlinearity="relu")
            nn.init.zeros_(layer.bias)
        nn.init.xavier_uniform_(self.out_proj.weight)
        nn.init.zeros_(self.out_proj.bias)

    def forward(self, x):
        if torch.is_grad_enabled() and self.act is F.gelu and not self.hidden_proj and train_ops.inactive_dropout(self.in_dropout):
            out = train_ops.gelu_mlp(x, self.in_proj, self.out_proj)
            if out is not None:
                return out
        x = self.in_dropout(self.act(self.in_proj(x)))
        for hidden, dropout in zip(self.hidden_proj, self.hidden_dropout):
            x = dropout(self.act(hidden(x)))
        return self.out_proj(x)


class Encoder(nn.Module):
    """Post-LN encoder layer: LN(q + attn(q,k,v)), LN(q + ffn(q)) (old/old_scripts/encoder.py:33-41), with the
    geometric attention branch (`bias=True, personal=False` in the reference's constructor)."""

    def __init__(self, d_model=512, heads=8, d_hidden=2048, hidden_layers=0, dropout=0.10, min_spread=2.0, learn_spreads=True):
        super().__init__()
        self.attn = GeoAttention(d_model=d_model, heads=heads, min_spread=min_spread, learn_spreads=learn_spreads)
        self.attn_norm = nn.LayerNorm(d_model)
        self.ffn = MLP(d_in=d_model, d_out=d_model, d_hidden=d_hidden, hidden_layers=hidden_layers, dropout=dropout)
        self.ffn_norm = nn.LayerNorm(d_model)
        self.dropout = nn.Dropout(dropout)

    def forward(self, q, k, v, coords, mask=None):
        if type(self) is Encoder and q is k and k is v:
            out = train_ops.encoder_layer(q, coords, mask, self, MLP)   # fp32 training
            if out is None:
                out = _infer_layer(q, coords, mask, self)               # bf16 inference
            if out is not None:
                return out
        q = self._residual_norm(q, self.dropout(self.attn(q, k, v, coords, mask=mask)), self.attn_norm)
        q = self._residual_norm(q, self.dropout(self.ffn(q)), self.ffn_norm)
        return q

    @staticmethod
    def _residual_norm(q, branch, norm):
        out = train_ops.add_layer_norm(q, branch, norm)
        return add_layer_norm(q, branch, norm) if out is None else out


def _infer_layer(x, coords, mask, m):
    """The output of the Encoder module `m` (self-attention) on a bf16 x where nothing needs a gradient, all launches of the layer from one call of the
    library, or None where its parts go their own ways."""
    if x.dtype != torch.bfloat16 or not x.is_cuda or type(x) is not torch.Tensor or torch.is_autocast_enabled("cuda"):
        return None
    if torch.is_grad_enabled() and (x.requires_grad or getattr(getattr(m.attn_norm, "weight", None), "requires_grad", False)):
        return None                                                         # (training, before the closer look, which takes 15 us of host time)
    a, n1, f, n2 = m.attn, m.attn_norm, m.ffn, m.ffn_norm
    plain = train_ops.plain_module
    if not (plain(a, GeoAttention) and plain(n1, nn.LayerNorm) and plain(n2, nn.LayerNorm) and plain(f, MLP) and f.act is F.gelu and not f.hidden_proj
            and train_ops.inactive_dropout(m.dropout) and train_ops.inactive_dropout(f.in_dropout) and plain(f.in_proj, nn.Linear) and plain(f.out_proj, nn.Linear)
            and plain(a.out_proj, nn.Linear) and "_residual_norm" not in m.__dict__ and a.out_proj.bias is None
            and "get_spreads" not in a.__dict__ and isinstance(a.min_spread, (int, float))):       # (a sigma of another shape is the operator's to refuse)
        return None
    H, dk, dm, l1, l2 = a.heads, a.d_k, a.d_model, f.in_proj, f.out_proj
    rest = (n1.weight, n1.bias, l1.weight, l1.bias, l2.weight, l2.bias, n2.weight, n2.bias)
    attn = (a.q_proj, a.k_proj, a.v_proj, a.q_bias, a.k_bias, a.v_bias, a.out_proj.weight)
    if any(type(p) not in train_ops._PLAIN_TYPES or p.dtype != torch.bfloat16 or p.get_device() != x.get_device() for p in rest + attn):
        return None
    if torch.is_grad_enabled() and (x.requires_grad or a.spread_weights.requires_grad or any(p.requires_grad for p in rest + attn)):
        return None
    hidden = l1.weight.shape[0]
    w, b = (H, dm, dk), (H, dk)
    if (tuple(p.shape for p in rest + attn) != ((dm,), (dm,), (hidden, dm), (hidden,), (dm, hidden), (dm,), (dm,), (dm,), w, w, w, b, b, b, (dm, dm))
            or a.legacy_logits or a.operand_dtype not in (None, torch.bfloat16) or x.dim() != 3 or x.shape[2] != dm or x.numel() == 0
            or type(a.spread_weights) not in train_ops._PLAIN_TYPES or a.spread_weights.shape != (H,) or a.spread_weights.device != x.device or not (n1.eps >= 0.0 and n2.eps >= 0.0)
            or tuple(coords.shape) != (*x.shape[:2], 3) or (mask is not None and tuple(mask.shape) != tuple(x.shape[:2]))
            or not train_ops.unobserved() or not train_ops.aligned(*rest)):
        return None
    # Products beyond 512 features: the library's are the faster ones from about 2^33 rows x features^2 on.  Layers in parts / in one call, us: features 512, 8192 tokens
    # (padded: 210 / 148 a layer), 65536 933 / 886; 768 12288 398 / 383, 32768 846 / 851; 1024 8192 339 / 326, 16384 581 / 625; 2048 2048 277 / 294
    if dm > 512 and (dm > 1024 or x.shape[0] * x.shape[1] * dm * dm > 2 ** 33):
        return None
    sizes = (*x.shape[:2], H, dk, hidden)
    nbytes = train_ops._bytes("proteus_encoder_infer_bytes", *sizes)
    if nbytes == 0:
        return None
    dev = x.device
    wqkv, bqkv, wo, sigma = a._infer_constants()
    params = (wqkv, bqkv, wo, *rest)
    x, c = train_ops._dense(x), _f32(coords, dev)
    pad = None if mask is None else _mask_bytes(mask, dev)
    out = torch.empty_like(x)
    train_ops._call("proteus_encoder_infer", dev, x, c, sigma, pad, train_ops._pointers(params), float(n1.eps), float(n2.eps), out,
                    train_ops._workspace(nbytes, dev), nbytes, *sizes)
    return out


def _add_to_bf16(a, b):
    """(a + b.to(a.dtype)).to(torch.bfloat16) of an fp32 and a bf16 tensor in one pass, or None where a gradient is needed or the kernel does not take them."""
    if not (type(a) is type(b) is torch.Tensor and a.is_cuda and a.dtype == torch.float32 and b.dtype == torch.bfloat16 and a.device == b.device
            and a.shape == b.shape and a.numel() % 8 == 0 and a.numel() > 0 and not (torch.is_grad_enabled() and (a.requires_grad or b.requires_grad))
            and train_ops.unobserved() and train_ops.aligned(a, b)):
        return None
    out = torch.empty_like(b)
    train_ops._call("proteus_add_to_bf16", a.device, a, b, out, a.numel())
    return out


class ProteusEncoder(nn.Module):
    """WE(coords) + Embedding[tokens] -> `layers` encoder layers -> Linear(d_model, 20).

    sigma per head is log-spaced from `sigma_min` to `sigma_max` at initialisation
    (sigma = min_spread + exp(w), old/old_scripts/encoder.py:88-89).  The embedding runs in
    fp32; the encoder layers run in the dtype of their weights (e.g. after `.to(torch.bfloat16)`
    applied to `layers`, `aa_embedding` and `head`).
    """

    def __init__(self, d_model=512, heads=8, layers=4, d_hidden=2048, vocab=33, n_out=20,
                 min_wl=3.7, max_wl=20.0, base_wl=20.0, sigma_min=3.0, sigma_max=25.0, min_spread=2.0, dropout=0.0):
        super().__init__()
        self.wf_embedding = WaveFunctionEmbedding(d_wf=d_model, min_wl=min_wl, max_wl=max_wl, base_wl=base_wl, anisotropic=False)
        self.aa_embedding = nn.Embedding(vocab, d_model)
        self.layers = nn.ModuleList([Encoder(d_model=d_model, heads=heads, d_hidden=d_hidden, dropout=dropout, min_spread=min_spread)
                                     for _ in range(layers)])
        self.head = nn.Linear(d_model, n_out)
        if heads > 1:
            sig = sigma_min * (sigma_max / sigma_min) ** (torch.arange(heads, dtype=torch.float64) / (heads - 1))
        else:
            sig = torch.tensor([sigma_min], dtype=torch.float64)
        w = torch.log(sig - min_spread).to(torch.float32)
        with torch.no_grad():
            for layer in self.layers:
                layer.attn.spread_weights.copy_(w)

    def forward(self, coords, tokens, key_padding_mask=None):
        wf = self.wf_embedding(coords, None, key_padding_mask=key_padding_mask)           # fp32 [Z,N,d_model]
        aa = train_ops.embedding(tokens, self.aa_embedding)
        aa = self.aa_embedding(tokens) if aa is None else aa
        x = _add_to_bf16(wf, aa) if self.head.weight.dtype == torch.bfloat16 else None
        if x is None:
            x = (wf + aa.to(wf.dtype)).to(self.head.weight.dtype)
        for layer in self.layers:
            x = layer(x, x, x, coords, mask=key_padding_mask)
        return self.head(x)
