"""The mesh transformer's attention block on the HIP kernels, with no layout copies.

Mirrors the caller of the reference's kernel, ``tiled_mha`` (``patch.py:165-177``): q, k, v
projections of the node features, masked attention over the k-hop mesh neighbourhood with
scale key_size**-0.5, reshape to [batch, n, heads * key_size] and the ``mha_final`` projection.
In the reference each projection writes [batch, n, heads, key_size], the Pallas op transposes
them to head-major and pads them (``pallas_attn.py:334-335``), and transposes the output back
(``pallas_attn.py:354``).

Here one fused projection writes q, k, v node-major into one [batch, n, 3, heads, key_size]
buffer. The kernels read the three views where they lie and write dq, dk, dv into one packed
gradient. The output [batch, n, heads, key_size] is already the [batch, n, heads * key_size]
input of the final projection. The parameters are plain torch Linear layers initialised by
torch; official WeatherNext checkpoints are Haiku parameters of the JAX model, which this
package does not load.
"""
import ctypes

import torch

from . import _native as nat
from . import patch
from .hip_attn import TileList, tiled_flash_attention, tiled_flash_attention_qkv
from .rows import as_torch

# hipBLASLt's bf16 GEMMs on MI355X run much faster when the row count is a multiple of 512: for
# the block's four GEMMs at n = 40,962 nodes, 680 us per block against 519 us at 40,960 rows.
ROW_QUANTUM = 512


def linear_rows(x, weight, bias=None, gelu=False):
  """x [M, K] @ weight[N, K]^T (+ bias) (then tanh GELU when `gelu`), without autograd.

  Runs as two GEMMs into one output: the largest multiple of ROW_QUANTUM rows, then the rest,
  so most rows get the fast kernels (for M = 40,962: 556 us per block instead of 680). The
  bias and GELU run in the GEMM epilogue. Row results do not depend on the split beyond the
  GEMM kernels' own accumulation order.
  """
  m_all = x.shape[0]
  out = torch.empty((m_all, weight.shape[0]), device=x.device, dtype=x.dtype)
  m = m_all - m_all % ROW_QUANTUM
  for lo, hi in ((0, m), (m, m_all)) if 0 < m < m_all else ((0, m_all),):
    xs, o = x[lo:hi], out[lo:hi]
    if gelu:
      torch._addmm_activation(bias, xs, weight.t(), use_gelu=True, out=o)
    elif bias is not None:
      torch.addmm(bias, xs, weight.t(), out=o)
    else:
      torch.mm(xs, weight.t(), out=o)
  return out


def needs_grad(x, module):
  """True when autograd has to see this module's computation on x."""
  return torch.is_grad_enabled() and (x.requires_grad or any(p.requires_grad for p in module.parameters()))


def linear_wgrad(g, x, bias):
  """(g^T x, g's column sums or None) of contiguous bfloat16 g [M, N] and x [M, K], N and K multiples
  of 64: the gradients of a Linear's weight and bias in two HIP launches (``fwn_linear_wgrad_launch``)."""
  (m, outs), ins = g.shape, x.shape[1]
  dw = torch.empty((outs, ins), dtype=g.dtype, device=g.device)
  db = torch.empty(outs, dtype=g.dtype, device=g.device) if bias else None
  size = ctypes.c_uint64()
  nat.check(nat.lib().fwn_linear_wgrad_workspace_size(m, outs, ins, ctypes.byref(size)))
  with torch.cuda.device(g.device):
    work = torch.empty(size.value, dtype=torch.uint8, device=g.device)
    nat.check(nat.lib().fwn_linear_wgrad_launch(m, outs, ins, g.data_ptr(), x.data_ptr(), dw.data_ptr(),
                                                db.data_ptr() if bias else None, work.data_ptr(), size.value,
                                                torch.cuda.current_stream(g.device).cuda_stream))
  return dw, db


class _Linear(torch.autograd.Function):
  """F.linear of x [M, K] with the faster row split, and with ``linear_wgrad`` for the weight's and
  bias's gradients. Its output is a tensor of its own, not a view: a program may write into it."""

  @staticmethod
  def forward(ctx, x, weight, bias):
    # Each is kept only for the gradient that reads it, as F.linear does: a frozen weight holds no x, and
    # may be written where x needs no gradient.
    need_x, need_w, _ = ctx.needs_input_grad
    ctx.save_for_backward(x if need_w else None, weight if need_x else None)
    ctx.has_bias = bias is not None
    return linear_rows(x, weight, bias)

  @staticmethod
  def backward(ctx, g):
    x, weight = ctx.saved_tensors
    need_x, need_w, need_b = ctx.needs_input_grad
    need_b = need_b and ctx.has_bias
    dx = dw = db = None
    if as_torch(g):
      return (torch.mm(g, weight) if need_x else None, torch.mm(g.t(), x) if need_w else None,
              g.sum(0) if need_b else None)
    if need_x:
      dx = linear_rows(g, weight.t())
    if need_w:
      g, x = g.contiguous(), x.contiguous()
      if (g.data_ptr() | x.data_ptr()) & 15:
        dw, db = torch.mm(g.t(), x), g.sum(0) if need_b else None
      else:
        dw, db = linear_wgrad(g, x, need_b)
    elif need_b:
      db = g.sum(0)
    return dx, dw, db


# Rows from which a Linear's training pass runs as ``_Linear``, where the smaller side of its weight is 800
# wide; with a narrower weight as many entries on that side, or 8 times as many rows. Its two gradients are
# always quicker on the GPU (8,192 rows, GEMM and column sum against ``linear_wgrad``: 57 and 16 us at 64 x
# 64, 67 and 24 at 384 x 384, 77 and 39 at 2,048 x 512), but the Function costs about 60 us of host time a
# layer, and a training pass of a MeshBlock launched from Python is bound by the host below the line. Whole
# passes, us, modules against ``_Linear`` (rows x d_model, ffw_hidden = 4 d_model): below, 10,242 x 256 1222
# and 1457, x 512 1171 and 1429, 20,484 x 256 1182 and 1417, 30,726 x 192 1217 and 1445, 40,962 x 128 1184 and
# 1405; about the line and with the host's pace, 10,242 x 768 1307 to 1363 and 1231 to 1449, 20,484 x 384 1257 to
# 1285 and 1191 to 1449, 81,924 x 64 1374 to 1396 and 1165 to 1482; above, 10,242 x 1,024 1598 and 1443, 20,484 x
# 512 1582 and 1370, 30,726 x 384 1690 and 1372, 40,962 x 192 1507 and 1218, x 768 4156 and 3185.
WGRAD_ROWS = 8192
# Largest weight whose gradient is ``linear_wgrad``: half of the 256 CUs' 256 x 256 tiles. Above it a
# GEMM's own tiles fill the chip (20,484 rows: 4,096 x 1,024 299 and 175 us, 8,192 x 2,048 645 and
# 594, for 64 MB of partials).
WGRAD_ENTRIES = 128 * 256 * 256


def is_plain(module, kind):
  """Whether calling `module` is calling kind.forward: no subclass, hook, parametrization, wrapper or
  compiled call (``Module.compile``)."""
  return (type(module) is kind and "forward" not in module.__dict__ and module._compiled_call_impl is None and
          not (module._forward_hooks or module._forward_pre_hooks or module._backward_hooks or
               module._backward_pre_hooks) and not torch.nn.modules.module._has_any_global_hook())


def rows_enough(rows, outs, ins):
  """Whether a Linear of that weight over `rows` rows is past the line of WGRAD_ROWS."""
  return rows >= WGRAD_ROWS and (rows * min(outs, ins) >= 800 * WGRAD_ROWS or rows >= 8 * WGRAD_ROWS)


def linear(lin, x):
  """lin(x) with gradients: as ``_Linear`` where x and lin's parameters are plain bfloat16 tensors on one
  GPU, sizes are whole 64s and there are rows enough; else the module as it is."""
  if (x.dtype == torch.bfloat16 and x.is_cuda and x.numel() > 0 and is_plain(lin, torch.nn.Linear) and
      rows_enough(x.numel() // x.shape[-1], *lin.weight.shape) and
      type(x) in (torch.Tensor, torch.nn.Parameter) and type(lin.weight) is torch.nn.Parameter and
      lin.weight.dtype == x.dtype and lin.weight.device == x.device and lin.weight.is_contiguous() and
      x.shape[-1] == lin.weight.shape[1] and
      all(s % 64 == 0 and 0 < s <= 16384 for s in lin.weight.shape) and lin.weight.numel() <= WGRAD_ENTRIES and
      (lin.bias is None or (type(lin.bias) is torch.nn.Parameter and lin.bias.dtype == x.dtype and
                            lin.bias.device == x.device)) and
      not torch.is_autocast_enabled("cuda") and not torch.compiler.is_compiling() and
      not torch._C._are_functorch_transforms_active() and torch.autograd.forward_ad._current_level < 0):
    y = _Linear.apply(x.reshape(-1, x.shape[-1]), lin.weight, lin.bias)
    return y.view(*x.shape[:-1], y.shape[-1])
  return lin(x)


class TiledMHA(torch.nn.Module):
  """x [batch, n, d_model] -> x's attention update [batch, n, d_model].

  ``tiles`` is the mesh's TileList (or the array triple of ``build_tile_mask``), built once and
  shared by every layer; ``tiles_t`` is the transposed mask's list for non-symmetric masks.
  ``dtype`` None takes the enable() option (bfloat16 when ``bf16``, else float32), ``precision``
  None the precision ``patch.resolve_precision`` picks from the enable() options ``precision``
  and ``strict_fp32`` and torch's float32 matmul precision (float32 only: "native" or "bf16x3").
  """

  def __init__(self, d_model, num_heads, key_size, tiles, tiles_t=None, *, device=None, dtype=None, precision=None):
    super().__init__()
    dtype = patch.default_dtype(dtype)
    self.precision = patch.default_precision(precision, dtype)
    self.num_heads, self.key_size = num_heads, key_size
    self.tiles, self.tiles_t = tiles, tiles_t
    self.qkv = torch.nn.Linear(d_model, 3 * num_heads * key_size, bias=False, device=device, dtype=dtype)
    self.final = torch.nn.Linear(num_heads * key_size, d_model, device=device, dtype=dtype)

  def forward(self, x):
    b, n, d = x.shape
    hd = self.num_heads * self.key_size
    if needs_grad(x, self):
      qkv = linear(self.qkv, x).view(b, n, 3, self.num_heads, self.key_size)
      out = tiled_flash_attention_qkv(qkv, self.tiles, scale=self.key_size ** -0.5, tiles_t=self.tiles_t,
                                      precision=self.precision)
      return linear(self.final, out.view(b, n, hd))
    # Without autograd the projections run through linear_rows (the faster GEMM row split).
    qkv = linear_rows(x.reshape(b * n, d), self.qkv.weight).view(b, n, 3, self.num_heads, self.key_size)
    out = tiled_flash_attention_qkv(qkv, self.tiles, scale=self.key_size ** -0.5, tiles_t=self.tiles_t,
                                      precision=self.precision)
    return linear_rows(out.reshape(b * n, hd), self.final.weight, self.final.bias).view(b, n, -1)

  def forward_unfused(self, x):
    """The same block with separate q, k, v tensors copied to contiguous [batch, n, heads,
    key_size] layouts, as three separate projections would leave them (comparison path)."""
    b, n, _ = x.shape
    q, k, v = (t.contiguous() for t in self.qkv(x).view(b, n, 3, self.num_heads, self.key_size).unbind(2))
    tiles = self.tiles if isinstance(self.tiles, TileList) else tuple(self.tiles)
    if isinstance(tiles, tuple):
      out = tiled_flash_attention(q, k, v, *tiles, scale=self.key_size ** -0.5, tiles_t=self.tiles_t,
                                  precision=self.precision)
    else:
      out = tiled_flash_attention(q, k, v, tiles, scale=self.key_size ** -0.5, tiles_t=self.tiles_t,
                                  precision=self.precision)
    return self.final(out.reshape(b, n, self.num_heads * self.key_size))
