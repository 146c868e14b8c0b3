"""Hilbert-order gather and scatter of the node features, fused with the layer norms next to them.

The reference's patched transformer permutes the mesh nodes into Hilbert order before its
layers and back after them (``patch.py:274-276, 288-292``):

    node_features = jnp.take(node_features, perm, axis=1)      # before the layer loop
    ...                                                         # block 0 starts with st.layernorm
    x = st.layernorm(x, create_scale=False, create_offset=False)
    x = LinearNormConditioning(...)(x, norm_conditioning=...)   # per-member scale and offset
    x = jnp.take(x, argsort(perm), axis=1)                      # after the layer loop

``gather_layer_norm`` does the first gather together with block 0's layer norm, and
``layer_norm_scatter`` the final layer norm, its per-member affine and the scatter, each as one
HIP pass over [batch, n, channels] (``include/fwn_rows.h``). ``layer_norm_affine`` is the same
pass without a permutation: each block's conditioned layer norm in front of the attention and
the feed-forward (``patch.py:240-244, 250-251``), and ``add_layer_norm_affine`` adds the
residual in front of it in the same pass. The affine's scale and offset come
from the conditioning vector through LinearNormConditioning's own projections, which the caller
evaluates: pass ``mul`` (its multiplier of the normalised features) and ``add``.

The forward passes and their gradients run on the GPU only. Each gradient is one HIP pass as well
(``fwn_rows_norm_bwd_launch``: the layer norm's analytic backward, with the permutation and the
gradient that bypassed the norm in the same pass), plus a small reduction for mul and add. A
backward that has to be differentiated again (create_graph) or whose gradients are batched
(is_grads_batched) runs as torch operations instead.
"""
import ctypes

import torch

from . import _native as nat

_DTYPES = {torch.float32: nat.F32, torch.bfloat16: nat.BF16}


def _desc(x, eps):
  if not isinstance(x, torch.Tensor) or not x.is_cuda:
    raise ValueError("x must be a CUDA tensor")
  if x.dim() != 3:
    raise ValueError(f"x must be [batch, n, channels], got shape {tuple(x.shape)}")
  if x.dtype not in _DTYPES:
    raise TypeError(f"x must be float32 or bfloat16, got {x.dtype}")
  if not x.is_contiguous():
    raise ValueError("x must be contiguous")
  b, n, c = x.shape
  return nat.RowsDesc(b, n, c, _DTYPES[x.dtype], float(eps))


def _perm(perm, x):
  if not isinstance(perm, torch.Tensor) or perm.device != x.device or perm.dtype != torch.int64:
    raise ValueError("perm must be an int64 tensor on the device of x")
  if perm.shape != (x.shape[1],) or not perm.is_contiguous():
    raise ValueError(f"perm must be contiguous with shape ({x.shape[1]},), got {tuple(perm.shape)}")
  return perm


def _affine(t, x, name):
  if t is None:
    return None
  if not isinstance(t, torch.Tensor) or t.device != x.device or t.dtype != torch.float32:
    raise ValueError(f"{name} must be a float32 tensor on the device of x")
  if t.shape != (x.shape[0], x.shape[2]) or not t.is_contiguous():
    raise ValueError(f"{name} must be contiguous [batch, channels] = {(x.shape[0], x.shape[2])}")
  return t


def _stream(x):
  return torch.cuda.current_stream(x.device).cuda_stream


def _addr(t):
  return t.data_ptr() if t is not None and t.numel() else None


def gather_layer_norm_forward(x, perm, eps=1e-5, norm=True):
  """(x[:, perm], layer_norm(x[:, perm]) or None), computed by one HIP pass (no autograd)."""
  d = _desc(x, eps)
  perm = _perm(perm, x)
  x_out = torch.empty_like(x)
  n_out = torch.empty_like(x) if norm else None
  with torch.cuda.device(x.device):
    nat.check(nat.lib().fwn_rows_gather_norm_launch(d, _addr(x), _addr(perm), _addr(x_out), _addr(n_out),
                                                    _stream(x)))
  return x_out, n_out


def layer_norm_scatter_forward(x, perm, mul=None, add=None, eps=1e-5):
  """out with out[:, perm] = layer_norm(x) * mul[:, None] + add[:, None], one HIP pass (no autograd)."""
  d = _desc(x, eps)
  perm = _perm(perm, x)
  mul = _affine(mul, x, "mul")
  add = _affine(add, x, "add")
  out = torch.empty_like(x)
  with torch.cuda.device(x.device):
    nat.check(nat.lib().fwn_rows_norm_scatter_launch(d, _addr(x), _addr(perm), _addr(mul), _addr(add), _addr(out),
                                                     _stream(x)))
  return out


def layer_norm_affine_forward(x, mul=None, add=None, eps=1e-5):
  """layer_norm(x) * mul[:, None] + add[:, None], one HIP pass (no autograd)."""
  d = _desc(x, eps)
  mul = _affine(mul, x, "mul")
  add = _affine(add, x, "add")
  out = torch.empty_like(x)
  with torch.cuda.device(x.device):
    nat.check(nat.lib().fwn_rows_norm_affine_launch(d, _addr(x), _addr(mul), _addr(add), _addr(out), _stream(x)))
  return out


def add_layer_norm_affine(x, y, *, mul=None, add=None, eps=1e-5, inplace=False):
  """(x + y, layer_norm(x + y) * mul[:, None] + add[:, None]) in one HIP pass: a block's residual
  add fused with the conditioned layer norm that reads it (``patch.py:240-253``). The sum is
  added in float32 and rounded once to x's dtype, as ``x + y`` stores it, and the norm is the
  sum's. With ``inplace`` the sum is written into x. mul and add are float32 [batch, channels]
  (None: 1 and 0). Forward only: it refuses inputs that autograd would need to differentiate."""
  if torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in (x, y, mul, add)):
    raise RuntimeError("add_layer_norm_affine has no derivative; use x + y and layer_norm_affine under autograd")
  d = _desc(x, eps)
  if not isinstance(y, torch.Tensor) or y.shape != x.shape or y.dtype != x.dtype or y.device != x.device:
    raise ValueError("y must be a tensor of x's shape, dtype and device")
  if not y.is_contiguous():
    raise ValueError("y must be contiguous")
  mul = _affine(mul, x, "mul")
  add = _affine(add, x, "add")
  s = x if inplace else torch.empty_like(x)
  out = torch.empty_like(x)
  with torch.cuda.device(x.device):
    nat.check(nat.lib().fwn_rows_add_norm_affine_launch(d, _addr(x), _addr(y), _addr(mul), _addr(add), _addr(s),
                                                        _addr(out), _stream(x)))
  return s, out


def _dense(t):
  """t as the kernels read it: contiguous and 16-byte aligned (None stays None)."""
  if t is None:
    return None
  t = t.contiguous()
  return t if t.data_ptr() % 16 == 0 else t.clone()


def _norm_backward_pass(x, eps, g_norm, g_res=None, mul=None, perm=None, perm_rows=0, sums=False):
  """(gradient of the rows, g_mul or None, g_add or None): one HIP pass (fwn_rows_norm_bwd_launch)."""
  x, g_norm, g_res, mul, perm = (_dense(t) for t in (x, g_norm, g_res, mul, perm))
  d = _desc(x, eps)
  L = nat.lib()
  gx = torch.empty_like(x)
  g_mul = g_add = ws = None
  if sums:
    g_mul, g_add = (torch.empty((x.shape[0], x.shape[2]), dtype=torch.float32, device=x.device) for _ in range(2))
    size = ctypes.c_uint64(0)
    nat.check(L.fwn_rows_norm_bwd_workspace_size(d, ctypes.byref(size)))
    ws = torch.empty(int(size.value), dtype=torch.uint8, device=x.device)
  with torch.cuda.device(x.device):
    nat.check(L.fwn_rows_norm_bwd_launch(d, _addr(x), _addr(perm), perm_rows, _addr(g_norm), _addr(g_res), _addr(mul),
                                         _addr(gx), _addr(g_mul), _addr(g_add), _addr(ws),
                                         0 if ws is None else ws.numel(), _stream(x)))
  return gx, g_mul, g_add


# The same gradients as torch operations, for backwards under create_graph or of batched gradients.


def as_torch(*grads):
  """Whether a backward with these gradients has to run as torch operations: it is differentiated
  again (create_graph), or they are vmap's batched tensors (is_grads_batched), which have no memory."""
  return torch.is_grad_enabled() or any(
      g is not None and (torch._C._functorch.is_legacy_batchedtensor(g) or
                         torch._C._functorch.is_functorch_wrapped_tensor(g)) for g in grads)


def _norm_stats(x, eps):
  xf = x.float()
  mean = xf.mean(-1, keepdim=True)
  var = (xf - mean).square().mean(-1, keepdim=True)
  rstd = torch.rsqrt(var + eps)
  return (xf - mean) * rstd, rstd


def _norm_backward(xhat, rstd, g):
  """Gradient of layer_norm (no affine) at normalised values xhat for upstream gradient g."""
  g = g.float()
  return rstd * (g - g.mean(-1, keepdim=True) - xhat * (g * xhat).mean(-1, keepdim=True))


def _inverse(perm):
  inv = torch.empty_like(perm)
  inv[perm] = torch.arange(perm.numel(), device=perm.device)
  return inv


def _affine_norm_backward(x, eps, g_y, mul, need_mul, need_add):
  """(gradient of x in float32, g_mul, g_add) of layer_norm(x) * mul + add for the gradient g_y."""
  g_y = g_y.float()
  xhat, rstd = _norm_stats(x, eps)
  g_mul = (g_y * xhat).sum(1) if need_mul else None
  g_add = g_y.sum(1) if need_add else None
  return _norm_backward(xhat, rstd, g_y * mul[:, None, :] if mul is not None else g_y), g_mul, g_add


class _GatherNorm(torch.autograd.Function):
  @staticmethod
  def forward(ctx, x, perm, eps):
    x_out, n_out = gather_layer_norm_forward(x, perm, eps)
    ctx.save_for_backward(x_out, perm)
    ctx.set_materialize_grads(False)
    ctx.eps = eps
    return x_out, n_out

  @staticmethod
  def backward(ctx, g_x, g_n):
    x_out, perm = ctx.saved_tensors
    if not as_torch(g_x, g_n):
      return _norm_backward_pass(x_out, ctx.eps, g_n, g_x, perm=perm, perm_rows=nat.ROWS_PERM_OUT)[0], None, None
    g = torch.zeros(x_out.shape, device=x_out.device, dtype=torch.float32)
    if g_x is not None:
      g = g + g_x.float()
    if g_n is not None:
      xhat, rstd = _norm_stats(x_out, ctx.eps)
      g = g + _norm_backward(xhat, rstd, g_n)
    return g[:, _inverse(perm)].to(x_out.dtype), None, None


class _NormScatter(torch.autograd.Function):
  @staticmethod
  def forward(ctx, x, perm, mul, add, eps):
    if perm is None:
      out = layer_norm_affine_forward(x, mul, add, eps)
    else:
      out = layer_norm_scatter_forward(x, perm, mul, add, eps)
    ctx.save_for_backward(x, perm, mul)
    ctx.eps = eps
    ctx.has_add = add is not None
    return out

  @staticmethod
  def backward(ctx, g_out):
    x, perm, mul = ctx.saved_tensors
    need_mul, need_add = mul is not None and ctx.needs_input_grad[2], ctx.has_add and ctx.needs_input_grad[3]
    if as_torch(g_out):
      g_y = g_out if perm is None else g_out[:, perm]  # gradient of the un-scattered rows
      g_x, g_mul, g_add = _affine_norm_backward(x, ctx.eps, g_y, mul, need_mul, need_add)
      return g_x.to(x.dtype), None, g_mul, g_add, None
    g_x, g_mul, g_add = _norm_backward_pass(x, ctx.eps, g_out, mul=mul, perm=perm,
                                            perm_rows=0 if perm is None else nat.ROWS_PERM_GRAD,
                                            sums=need_mul or need_add)
    return g_x, None, g_mul if need_mul else None, g_add if need_add else None, None


class _AddNorm(torch.autograd.Function):
  """(x + y, layer_norm(x + y) * mul + add): the gradient of the sum adds to the norm's in the
  norm's backward pass."""

  @staticmethod
  def forward(ctx, x, y, mul, add, eps):
    s, out = add_layer_norm_affine(x, y, mul=mul, add=add, eps=eps)
    ctx.save_for_backward(s, mul)
    ctx.set_materialize_grads(False)
    ctx.eps = eps
    return s, out

  @staticmethod
  def backward(ctx, g_s, g_out):
    s, mul = ctx.saved_tensors
    if g_out is None:
      return g_s, g_s, None, None, None
    need_mul, need_add = ctx.needs_input_grad[2], ctx.needs_input_grad[3]
    if as_torch(g_s, g_out):
      g, g_mul, g_add = _affine_norm_backward(s, ctx.eps, g_out, mul, need_mul, need_add)
      g = (g if g_s is None else g + g_s.float()).to(s.dtype)
    else:
      g, g_mul, g_add = _norm_backward_pass(s, ctx.eps, g_out, g_s, mul, sums=need_mul or need_add)
    return g, g, g_mul if need_mul else None, g_add if need_add else None, None


def residual_norm(x, y, *, mul, add, eps=1e-5):
  """(x + y, layer_norm_affine(x + y)) with gradients: one pass forward and one backward where x and
  y are contiguous, aligned and of one dtype, else torch's add and the norm's own pass."""
  same = (x.dtype == y.dtype and x.shape == y.shape and x.is_contiguous() and y.is_contiguous() and
          x.data_ptr() % 16 == 0 and y.data_ptr() % 16 == 0)
  if same and x.is_cuda and x.dim() == 3 and x.dtype in _DTYPES:
    return _AddNorm.apply(x, y, mul, add, float(eps))
  s = (x + y).contiguous()  # torch's add keeps a dense operand's strides
  return s, layer_norm_affine(s, mul=mul, add=add, eps=eps)


def cond_affine(cond, weights, biases):
  """[(mul, add)] of each norm, float32 [batch, channels]: 1 + scale and offset from its weight
  [2 * channels, cond_size] and bias, as ``LinearNormConditioning`` projects them, in one HIP launch
  for up to COND_MAX norms (no autograd). cond is [batch, cond_size] in the weights' dtype."""
  batch, size = cond.shape
  channels = weights[0].shape[0] // 2
  out = torch.empty((2, len(weights), batch, channels), dtype=torch.float32, device=cond.device)
  with torch.cuda.device(cond.device):
    for lo in range(0, len(weights), nat.COND_MAX):
      hi = min(lo + nat.COND_MAX, len(weights))
      table = lambda ts: (ctypes.c_void_p * (hi - lo))(*(t.data_ptr() for t in ts[lo:hi]))
      nat.check(nat.lib().fwn_cond_affine_launch(hi - lo, batch, channels, size, _DTYPES[cond.dtype], _addr(cond),
                                                 table(weights), table(biases), _addr(out[0, lo]), _addr(out[1, lo]),
                                                 _stream(cond)))
  return list(zip(out[0].unbind(0), out[1].unbind(0)))


def gather_layer_norm(x, perm, *, eps=1e-5):
  """x [batch, n, channels] -> (x[:, perm], layer_norm(x[:, perm])): the Hilbert gather before
  the layer loop (``patch.py:274-276``) and block 0's ``st.layernorm(x, create_scale=False,
  create_offset=False)`` (``patch.py:244``) in one pass. Differentiable in x."""
  return _GatherNorm.apply(x, perm, float(eps))


def layer_norm_scatter(x, perm, *, mul=None, add=None, eps=1e-5):
  """x [batch, n, channels] -> out with out[:, perm] = layer_norm(x) * mul[:, None] + add[:, None]:
  the final layer norm, LinearNormConditioning's per-member affine and the scatter back to mesh
  order (``patch.py:288-292``) in one pass. mul and add are float32 [batch, channels] (None: 1
  and 0). Differentiable in x, mul and add."""
  return _NormScatter.apply(x, perm, mul, add, float(eps))


def layer_norm_affine(x, *, mul=None, add=None, eps=1e-5):
  """x [batch, n, channels] -> layer_norm(x) * mul[:, None] + add[:, None] in one pass: a block's
  ``norm_conditioning_layer(st.layernorm(x, create_scale=False, create_offset=False))``
  (``patch.py:240-244, 250-251``). mul and add are float32 [batch, channels] (None: 1 and 0).
  Differentiable in x, mul and add."""
  return _NormScatter.apply(x, None, mul, add, float(eps))
