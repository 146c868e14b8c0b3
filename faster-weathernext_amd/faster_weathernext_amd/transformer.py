"""The mesh transformer around the attention kernels: the reference's patched
``ChunkedTransformer`` / ``ChunkedBlock`` (``patch.py:193-293``) in PyTorch.

Structure, as the reference wires it:

* at construction, the k-hop mask of the refined icosahedral mesh, the optional Hilbert
  permutation and the live-tile list, built once and shared by every layer
  (``_transformer_init``, ``patch.py:193-226``; ``optimization_barrier``, ``:263-266``);
* before the layers, the gather of the node features into Hilbert order (``:274-276``), here
  fused with block 0's first layer norm (``rows.gather_layer_norm``);
* per block (``ChunkedBlock.__call__``, ``:233-253``):
  ``x = x + mha(cond_norm(layernorm(x)))`` then ``x = x + ffw(cond_norm(layernorm(x)))``, with the
  attention ``TiledMHA`` (``tiled_mha``, ``:165-177``) on the HIP kernels;
* after the layers, the final layer norm, its conditioning and the scatter back to mesh order
  (``:288-292``), fused into one pass (``rows.layer_norm_scatter``).

Two parts live in weathernext, which is not vendored, so their exact form is not pinned here:
``LinearNormConditioning`` is implemented as published with GenCast (a linear map of the
conditioning vector, zero-initialised, giving a per-channel scale-minus-one and offset:
``x * (1 + scale) + offset``), and ``st.ffw`` as a two-layer GELU MLP of width ``ffw_hidden``
with the tanh form of GELU (``jax.nn.gelu``'s default). Without autograd, the first layer's bias
and GELU run in the epilogue of its GEMM (``torch._addmm_activation``, which has no derivative),
so the [n, ffw_hidden] activations make one trip to HBM instead of three, every block GEMM
splits its rows at a multiple of 512 (``mha.linear_rows``), and each residual add runs in one
pass with the conditioned layer norm after it (``rows.add_layer_norm_affine``); with autograd the
same functions run as Linear (``mha.linear``), GELU, Linear and adds, the attention's add fused with
the feed-forward's conditioned norm (``rows.residual_norm``).
Parameters are random-initialised torch parameters; official checkpoints are Haiku parameters of
the JAX model, which this package does not load.
"""
import numpy as np
import torch
import torch.nn.functional as F
from scipy import sparse

from . import patch
from .hip_attn import TileList
from .mesh import hilbert_order, khop_mask, mesh_mask
from .mha import TiledMHA, is_plain, linear, linear_rows, needs_grad
from .rows import (add_layer_norm_affine, cond_affine, gather_layer_norm, layer_norm_affine, layer_norm_scatter,
                   residual_norm)


class NormConditioning(torch.nn.Module):
  """x * (1 + scale(cond)) + offset(cond) per channel; the linear map starts at zero."""

  def __init__(self, d_model, cond_size, device=None, dtype=None):
    super().__init__()
    self.linear = torch.nn.Linear(cond_size, 2 * d_model, device=device, dtype=dtype)
    torch.nn.init.zeros_(self.linear.weight)
    torch.nn.init.zeros_(self.linear.bias)

  def affine(self, cond):
    """(multiplier, offset), each [batch, d_model]."""
    scale_m1, offset = self.linear(cond).chunk(2, dim=-1)
    return 1 + scale_m1, offset

  def forward(self, x, cond):
    mul, add = self.affine(cond)
    return x * mul[:, None, :] + add[:, None, :]

  def affine_f32(self, cond):
    """affine(cond) as the norm passes take it: contiguous float32."""
    mul, add = self.affine(cond)
    return mul.float().contiguous(), add.float().contiguous()

  def norm(self, x, cond, eps):
    """forward(layer_norm(x), cond) as one HIP pass (statistics and affine in float32)."""
    mul, add = self.affine_f32(cond)
    return layer_norm_affine(x, mul=mul, add=add, eps=eps)

  def residual_norm(self, x, y, cond, eps):
    """(x + y, norm(x + y)) with gradients, in one HIP pass where x and y allow it."""
    mul, add = self.affine_f32(cond)
    return residual_norm(x, y, mul=mul, add=add, eps=eps)

  def add_norm(self, x, y, cond, eps, affine=None):
    """(x + y, forward(layer_norm(x + y), cond)) as one HIP pass, without autograd; `affine` is
    ``affine_f32(cond)`` where the caller has it."""
    mul, add = affine or self.affine_f32(cond)
    return add_layer_norm_affine(x, y, mul=mul, add=add, eps=eps)

  def plain(self, cond):
    """Whether ``affine`` is the linear map as built, on parameters the conditioning kernel reads: no
    replaced method, hook, parametrization or autocast that would see or change the call. Asked of
    norms of this very class only (``affines_f32``)."""
    lin = self.linear
    return (not vars(self).keys() & {"affine", "add_norm"} and not torch.is_autocast_enabled("cuda")
            and is_plain(lin, torch.nn.Linear) and cond.dim() == 2 and cond.is_cuda
            and cond.dtype in (torch.float32, torch.bfloat16) and cond.is_contiguous() and cond.numel() > 0
            and all(type(t) is torch.nn.Parameter and t.dtype == cond.dtype and t.device == cond.device and
                    t.is_contiguous() for t in (lin.weight, lin.bias))
            and lin.weight.shape[1] == cond.shape[1])


# Batch members times conditioning features up to which one conditioning launch for all norms beats
# their projections one by one. Its threads read a weight row each, so its time grows with the
# product where a GEMM's hardly does; at 4,096 (8 x 512) it is ahead in every shape measured (5 to 49
# norms of 256 to 2,048 channels: 46 to 329 us against 150 to 1,700), at 32,768 (64 x 512) behind in
# most (309 to 2,360 against 150 to 1,690).
COND_WORK = 1 << 12


def affines_f32(norms, cond):
  """``affine_f32(cond)`` of each norm, without autograd, in one launch; None for each where a norm is
  not a ``plain`` one or the projections are large enough for a GEMM each."""
  if (cond.numel() <= COND_WORK and all(type(norm) is NormConditioning and norm.plain(cond) for norm in norms) and
      len({norm.linear.weight.shape for norm in norms}) == 1):
    return cond_affine(cond, [norm.linear.weight for norm in norms], [norm.linear.bias for norm in norms])
  return [None] * len(norms)


def _is_own(obj, cls, name):
  """Whether obj.name is cls's method: of a class or object of the program's own, its methods are called
  as they have always been."""
  return getattr(type(obj), name, None) is getattr(cls, name) and name not in vars(obj)


def _add_norm(norm, x, y, cond, eps, affine):
  return norm.add_norm(x, y, cond, eps) if affine is None else norm.add_norm(x, y, cond, eps, affine)


class MeshBlock(torch.nn.Module):
  """One transformer block (``ChunkedBlock``, ``patch.py:229-253``)."""

  def __init__(self, d_model, num_heads, key_size, ffw_hidden, cond_size, tiles, tiles_t=None, *, device=None,
               dtype=None, eps=1e-5, precision=None):
    super().__init__()
    self.eps = eps
    kw = dict(device=device, dtype=dtype)
    self.norm_mha = NormConditioning(d_model, cond_size, **kw)
    self.mha = TiledMHA(d_model, num_heads, key_size, tiles, tiles_t, precision=precision, **kw)
    self.norm_ffw = NormConditioning(d_model, cond_size, **kw)
    self.ffw = torch.nn.Sequential(torch.nn.Linear(d_model, ffw_hidden, **kw), torch.nn.GELU(approximate="tanh"),
                                   torch.nn.Linear(ffw_hidden, d_model, **kw))

  def feed_forward(self, h):
    """self.ffw(h); without autograd, the first layer's bias and GELU are fused into its GEMM and
    both GEMMs use the faster row split (``linear_rows``)."""
    l1, l2 = self.ffw[0], self.ffw[2]
    if needs_grad(h, self.ffw):
      if is_plain(self.ffw, torch.nn.Sequential) and len(self.ffw) == 3:
        return linear(l2, self.ffw[1](linear(l1, h)))
      return self.ffw(h)
    lead = h.shape[:-1]
    y = linear_rows(h.reshape(-1, h.shape[-1]), l1.weight, l1.bias, gelu=True)
    return linear_rows(y, l2.weight, l2.bias).view(*lead, l2.out_features)

  def forward(self, x, cond, normed=None):
    """`normed` is layernorm(x) when the caller has it already (block 0 gets it from the fused
    gather). Otherwise each conditioned layer norm is one fused pass (``layer_norm_affine``)."""
    h = self.norm_mha(normed, cond) if normed is not None else self.norm_mha.norm(x, cond, self.eps)
    y = self.mha(h)
    if _is_own(self.norm_ffw, NormConditioning, "norm"):
      x, h = self.norm_ffw.residual_norm(x, y, cond, self.eps)
    else:
      x = x + y
      h = self.norm_ffw.norm(x, cond, self.eps)
    return x + self.feed_forward(h)

  def forward_fused(self, x, h, cond, next_norm=None, affines=(None, None)):
    """The block without autograd, from h = norm_mha(layernorm(x)) already computed: each residual
    add runs in one pass with the conditioned layer norm that reads it (``add_layer_norm_affine``),
    the feed-forward's own and, when `next_norm` is given, the next block's. `affines` are the two
    norms' ``affine_f32(cond)`` where the caller has them. Returns (x, the next block's h or None)."""
    x, h = _add_norm(self.norm_ffw, x, self.mha(h), cond, self.eps, affines[0])
    f = self.feed_forward(h)
    if next_norm is None:
      return x + f, None
    return _add_norm(next_norm, x, f, cond, self.eps, affines[1])


class MeshTransformer(torch.nn.Module):
  """The 24-layer mesh transformer of WeatherNext 2's processor, node features [batch, n, d_model]
  in mesh (subdivision) order in and out; the attention runs in Hilbert order when `reorder`.

  The mask is the k-hop neighbourhood of the refined icosahedral mesh, or of ``adjacency`` (a
  boolean [n, n] sparse matrix, with the nodes' ``latlon`` in degrees for the Hilbert order) when
  one is given, as the reference builds it from the model's own adjacency (``patch.py:193-219``).
  A non-symmetric adjacency gives a non-symmetric mask, whose transposed tile list the backward
  walks. ``reorder``, ``dtype`` and ``precision`` None take the enable() options (``reorder``,
  ``bf16``, ``precision``).
  """

  def __init__(self, refinement=6, k_hop=32, num_layers=24, d_model=768, num_heads=6, key_size=128,
               ffw_hidden=3072, cond_size=32, reorder=None, *, device="cuda", dtype=None, tiles=None,
               tiles_t=None, adjacency=None, latlon=None, eps=1e-5, precision=None):
    super().__init__()
    reorder = patch.default_reorder(reorder)
    dtype = patch.default_dtype(dtype)
    if adjacency is None:
      mask, lat, lon, perm = mesh_mask(refinement, k_hop, reorder=reorder)
      symmetric = True  # powers of the mesh's symmetric adjacency
    else:
      adjacency = sparse.csr_matrix(adjacency).astype(bool)
      mask = khop_mask(adjacency, k_hop)
      perm = hilbert_order(*latlon) if reorder and latlon is not None else None
      symmetric = (adjacency != adjacency.T).nnz == 0
    self.n = mask.shape[0]
    self.eps = eps
    # One tile list for every layer (patch.py:214); the backward walks the transposed mask's list,
    # built only when the adjacency is not symmetric (patch.py:215-218).
    if tiles is None:
      tiles = TileList.from_mask(mask, perm, device=device)
      if not symmetric and tiles_t is None:
        permuted = mask if perm is None else mask[perm][:, perm]
        tiles_t = TileList.from_mask(permuted.T.tocsr(), device=device)
    elif not symmetric and tiles_t is None:
      # The backward would walk the forward list as its own transpose: wrong dK/dV.
      raise ValueError("a non-symmetric adjacency with caller-built tiles needs tiles_t, the transposed mask's "
                       "tile list")
    self.tiles, self.tiles_t = tiles, tiles_t
    self.register_buffer("perm", None if perm is None else torch.from_numpy(np.asarray(perm, np.int64)).to(device),
                         persistent=False)
    self.blocks = torch.nn.ModuleList(
        MeshBlock(d_model, num_heads, key_size, ffw_hidden, cond_size, self.tiles, self.tiles_t, device=device,
                  dtype=dtype, eps=eps, precision=precision)
        for _ in range(num_layers))
    self.final_norm = NormConditioning(d_model, cond_size, device=device, dtype=dtype)

  def forward(self, x, cond):
    d = x.shape[-1]
    normed = final = None
    if self.perm is not None:
      x, normed = gather_layer_norm(x, self.perm, eps=self.eps)
    elif len(self.blocks):
      normed = F.layer_norm(x, (d,), eps=self.eps)
    if len(self.blocks) and not needs_grad(x, self):
      # Without autograd the residual adds are fused into the conditioned layer norms after them, and
      # the conditioning of all norms that HIP passes apply (all but block 0's first and, without the
      # scatter, the final one) is evaluated up front in one launch.
      nexts = [block.norm_mha for block in self.blocks[1:]]
      affines = [None]
      if all(_is_own(block, MeshBlock, "forward_fused") for block in self.blocks):
        norms = [block.norm_ffw for block in self.blocks] + nexts
        affines = affines_f32(norms if self.perm is None else norms + [self.final_norm], cond)
      h = self.blocks[0].norm_mha(normed, cond)
      if affines[0] is None:
        for block, after in zip(self.blocks, nexts + [None]):
          x, h = block.forward_fused(x, h, cond, after)
      else:
        ffw, mha = affines[:len(self.blocks)], affines[len(self.blocks):]
        final = None if self.perm is None else mha.pop()
        for block, after, own, other in zip(self.blocks, nexts + [None], ffw, mha + [None]):
          x, h = block.forward_fused(x, h, cond, after, (own, other))
    else:
      for i, block in enumerate(self.blocks):
        x = block(x, cond, normed if i == 0 else None)
    if self.perm is not None:
      mul, add = final or self.final_norm.affine(cond)
      return layer_norm_scatter(x, self.perm, mul=mul.float().contiguous(), add=add.float().contiguous(), eps=self.eps)
    mul, add = self.final_norm.affine(cond)
    return F.layer_norm(x, (d,), eps=self.eps) * mul[:, None, :] + add[:, None, :]
