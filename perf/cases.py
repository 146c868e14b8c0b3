"""Workloads of the mesh-attention framework, for timing and for comparing one build with another.

Each case is a call that a program around the WeatherNext 2 mesh transformer makes: one layer's
masked attention (forward, or forward and backward), the permutation and layer-norm passes around
the layers, one transformer block's training pass, or a whole forward of the transformer. All run
on the icosahedral meshes the package generates (n = 10 * 4**refinement + 2 nodes, never a
multiple of the kernels' 128-row blocks), in the mesh's own node order or in Hilbert order.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "faster-weathernext_amd"))

import faster_weathernext_amd as fwn  # noqa: E402

DEV = "cuda"
EPS = 1e-5


def _attention(name, refinement, k_hop, reorder, heads, head_dim, dtype, precision="native", backward=True, batch=1,
               sigma=1.0):
  return dict(name=name, kind="attention", refinement=refinement, k_hop=k_hop, reorder=reorder, batch=batch,
              heads=heads, head_dim=head_dim, dtype=dtype, precision=precision, backward=backward, sigma=sigma)


def listed():
  return [
      # The smallest configuration the benchmark has: a coarse mesh as used while developing a
      # model, where a training step's attention is a handful of launches.
      _attention("attn_r3_2hop_f32_train", 3, 2, False, 2, 32, "f32"),
      # Inference of a small ensemble on a coarse mesh: latency of one layer's forward.
      _attention("attn_r4_8hop_b2_bf16_infer", 4, 8, True, 4, 64, "bf16", backward=False, batch=2),
      # One layer's training step on the mesh of a 1-degree model.
      _attention("attn_r5_16hop_bf16_train", 5, 16, True, 4, 128, "bf16"),
      # One layer's full-precision inference at 0.25 degrees, short-range mask, mesh order.
      _attention("attn_r6_8hop_f32_infer", 6, 8, False, 4, 128, "f32", backward=False, sigma=128 ** -0.5),
      # The benchmark's default: one layer's training step at 0.25 degrees, 16-hop mask, mesh order.
      _attention("attn_r6_16hop_bf16_train", 6, 16, False, 4, 128, "bf16"),
      # Ensemble training: 8 members at 0.25 degrees.
      _attention("attn_r6_8hop_b8_bf16_train", 6, 8, False, 4, 128, "bf16", batch=8),
      # One WeatherNext 2 layer (6 heads x 128, 32-hop, Hilbert order), training, in the three
      # product precisions the op offers: bf16 tensors, float32 tensors with split products
      # (torch's "high" matmul precision), float32 tensors with IEEE products (strict_fp32).
      _attention("attn_r6_32hop_bf16_train", 6, 32, True, 6, 128, "bf16"),
      _attention("attn_r6_32hop_x3_train", 6, 32, True, 6, 128, "f32", precision="bf16x3"),
      _attention("attn_r6_32hop_f32_train", 6, 32, True, 6, 128, "f32"),
      # The passes around the layer loop (Hilbert gather with the first layer norm, final
      # conditioned layer norm with the scatter back), float32 features, in training.
      dict(name="rows_r6_f32_train", kind="rows", n=40962, batch=1, channels=768, dtype="f32", backward=True),
      # One transformer block's training pass at WeatherNext 2 sizes.
      dict(name="block_r6_bf16_train", kind="block", refinement=6, k_hop=32, reorder=True, batch=1, d_model=768,
           heads=6, head_dim=128, ffw_hidden=3072, cond_size=32, dtype="bf16"),
      # The whole 24-layer mesh transformer, forecast inference.
      dict(name="model_r6_24l_bf16_infer", kind="model", refinement=6, k_hop=32, reorder=True, batch=1, layers=24,
           d_model=768, heads=6, head_dim=128, ffw_hidden=3072, cond_size=32, dtype="bf16"),
  ]


def _nodes(refinement):
  return 10 * 4 ** refinement + 2


def _entries(refinement, k_hop):
  """About how many entries the k-hop mask has: a disc of k hops holds 3k(k + 1) + 1 nodes."""
  n = _nodes(refinement)
  return n * min(n, 3 * k_hop * (k_hop + 1) + 1)


def _draw_attention(rng):
  while True:
    refinement = rng.randint(2, 6)
    k_hop = round(math.exp(rng.uniform(math.log(1.5), math.log(2.0 ** (refinement - 1) + 0.49))))
    dtype, precision = rng.choice([("bf16", "native"), ("bf16", "native"), ("f32", "bf16x3"), ("f32", "native")])
    c = _attention("", refinement, k_hop, rng.random() < 0.6, rng.randint(1, 8), rng.choice([32, 64, 128, 128]),
                   dtype, precision, rng.random() < 0.6, rng.choice([1, 1, 1, 2, 3, 4, 8]),
                   rng.choice([1.0, 128 ** -0.5]))
    del c["name"]
    cost = _entries(refinement, k_hop) * c["heads"] * c["head_dim"] * c["batch"] * (14 if c["backward"] else 4)
    cost *= {"bf16": 1, "f32": 3 if precision == "bf16x3" else 8}[dtype]
    # Within the largest listed layer (float32 IEEE, 32-hop, 6 x 128).
    if cost <= _entries(6, 32) * 6 * 128 * 14 * 8:
      return c


def draw(rng):
  kind = rng.choice(["attention"] * 5 + ["rows", "rows", "block", "model"])
  if kind == "attention":
    return _draw_attention(rng)
  if kind == "rows":
    return dict(kind="rows", n=round(math.exp(rng.uniform(math.log(600), math.log(41000)))), batch=rng.choice([1, 1, 2, 4]),
                channels=8 * rng.randint(32, 160), dtype=rng.choice(["f32", "bf16"]), backward=rng.random() < 0.5)
  heads = rng.choice([2, 4, 6])
  head_dim = rng.choice([32, 64, 128])
  c = dict(kind=kind, refinement=rng.randint(3, 5), k_hop=rng.randint(2, 16), reorder=rng.random() < 0.8,
           batch=rng.choice([1, 2, 3]), d_model=heads * head_dim, heads=heads, head_dim=head_dim,
           ffw_hidden=4 * heads * head_dim, cond_size=rng.choice([16, 32]), dtype=rng.choice(["bf16", "bf16", "f32"]))
  if kind == "model":
    c["layers"] = rng.randint(2, 8)
  return c


# ------------------------------------------------------------------------------------------------
# What a program has in hand: the mesh's mask and its tile list (built once per mesh, shared by
# every layer and call), the weights, and the inputs.


@functools.lru_cache(maxsize=4)
def _mesh(refinement, k_hop, reorder):
  mask, _, _, perm = fwn.mesh_mask(refinement, k_hop, reorder=reorder)
  return mask, perm, fwn.TileList.from_mask(mask, perm, device=DEV)


@functools.lru_cache(maxsize=4)
def _nnz(refinement, k_hop):
  return int(fwn.mesh_mask(refinement, k_hop)[0].nnz)


def _dtype(case):
  return {"bf16": torch.bfloat16, "f32": torch.float32}[case["dtype"]]


def _generator(seed):
  return torch.Generator(device=DEV).manual_seed(int(seed))


def _normal(gen, *shape, dtype=torch.float32, sigma=1.0):
  return torch.randn(*shape, device=DEV, generator=gen).mul_(sigma).to(dtype)


def _attention_inputs(case, seed):
  g = _generator(seed)
  shape = (case["batch"], _nodes(case["refinement"]), case["heads"], case["head_dim"])
  # Projections of normalised features: q and k such that the scaled logits have deviation sigma^2
  # * sqrt(head_dim) * head_dim**-0.5 = sigma^2.
  q, k, v = (_normal(g, *shape, dtype=_dtype(case), sigma=s) for s in (case["sigma"], case["sigma"], 1.0))
  do = _normal(g, *shape, dtype=_dtype(case)) if case["backward"] else None
  return q, k, v, do


def _rows_inputs(case, seed):
  g = _generator(seed)
  b, n, c = case["batch"], case["n"], case["channels"]
  x = _normal(g, b, n, c, dtype=_dtype(case)) + 0.5 * _normal(g, b, 1, c, dtype=_dtype(case))
  perm = torch.randperm(n, device=DEV, generator=g)
  mul = 1 + _normal(g, b, c, sigma=0.1)
  add = _normal(g, b, c, sigma=0.1)
  grads = [_normal(g, b, n, c, dtype=_dtype(case)) for _ in range(3)] if case["backward"] else None
  return x, perm, mul, add, grads


def _weights(module, case, seed):
  """Random weights of the given seed, the conditioning (which starts at zero) included."""
  g = _generator(seed + 1)
  with torch.no_grad():
    for name, p in sorted(module.named_parameters()):
      if "norm" in name:
        p.copy_(_normal(g, *p.shape, sigma=0.1))
      else:
        p.copy_(_normal(g, *p.shape, sigma=p.shape[-1] ** -0.5 if p.dim() > 1 else 0.02))
  return module


def _layer_args(case):
  return case["d_model"], case["heads"], case["head_dim"], case["ffw_hidden"], case["cond_size"]


def _block(case, seed):
  _, _, tiles = _mesh(case["refinement"], case["k_hop"], case["reorder"])
  block = fwn.MeshBlock(*_layer_args(case), tiles, device=DEV, dtype=_dtype(case), precision="native")
  return _weights(block, case, seed)


def _model(case, seed):
  _, _, tiles = _mesh(case["refinement"], case["k_hop"], case["reorder"])
  model = fwn.MeshTransformer(case["refinement"], case["k_hop"], case["layers"], *_layer_args(case), case["reorder"],
                              device=DEV, dtype=_dtype(case), tiles=tiles, precision="native")
  return _weights(model, case, seed)


def _features(case, seed, grad):
  g = _generator(seed)
  x = _normal(g, case["batch"], _nodes(case["refinement"]), case["d_model"], dtype=_dtype(case))
  cond = _normal(g, case["batch"], case["cond_size"], dtype=_dtype(case))
  return x, cond, _normal(g, *x.shape, dtype=_dtype(case)) if grad else None


def prepare(case, seed):
  if case["kind"] == "attention":
    q, k, v, do = _attention_inputs(case, seed)
    tiles = _mesh(case["refinement"], case["k_hop"], case["reorder"])[2]
    for t in (q, k, v):
      t.requires_grad_(case["backward"])
    return dict(case=case, q=q, k=k, v=v, do=do, tiles=tiles)
  if case["kind"] == "rows":
    x, perm, mul, add, grads = _rows_inputs(case, seed)
    for t in (x, mul, add):
      t.requires_grad_(case["backward"])
    return dict(case=case, x=x, perm=perm, mul=mul, add=add, grads=grads)
  if case["kind"] == "block":
    x, cond, g = _features(case, seed, True)
    return dict(case=case, module=_block(case, seed), x=x.requires_grad_(True), cond=cond, g=g)
  x, cond, _ = _features(case, seed, False)
  return dict(case=case, module=_model(case, seed), x=x, cond=cond)


def run(state):
  case = state["case"]
  if case["kind"] == "attention":
    q, k, v = state["q"], state["k"], state["v"]
    out = fwn.tiled_flash_attention(q, k, v, state["tiles"], scale=case["head_dim"] ** -0.5,
                                    precision=case["precision"])
    if not case["backward"]:
      return [out]
    return [out.detach(), *torch.autograd.grad(out, (q, k, v), state["do"])]
  if case["kind"] == "rows":
    x, mul, add = state["x"], state["mul"], state["add"]
    # The layers run between the two passes; here the first pass's features go straight on.
    gathered, normed = fwn.gather_layer_norm(x, state["perm"], eps=EPS)
    out = fwn.layer_norm_scatter(gathered, state["perm"], mul=mul, add=add, eps=EPS)
    if not case["backward"]:
      return [gathered, normed, out]
    grads = torch.autograd.grad((gathered, normed, out), (x, mul, add), state["grads"])
    return [gathered.detach(), normed.detach(), out.detach(), *grads]
  if case["kind"] == "block":
    x, block = state["x"], state["module"]
    out = block(x, state["cond"])
    return [out.detach(), *torch.autograd.grad(out, (x, *block.parameters()), state["g"])]
  with torch.no_grad():
    return [state["module"](state["x"], state["cond"])]


# ------------------------------------------------------------------------------------------------
# What a pass cannot do without: the mask's valid entries (2 * head_dim operations for each product
# of a pair of rows, five products in the backward, two in the forward), each tensor once.


def _attention_flops(case, products):
  return 2.0 * products * _nnz(case["refinement"], case["k_hop"]) * case["heads"] * case["head_dim"] * case["batch"]


def _gemm_flops(case):
  m = case["batch"] * _nodes(case["refinement"])
  hd, d, f = case["heads"] * case["head_dim"], case["d_model"], case["ffw_hidden"]
  return 2.0 * m * d * (4 * hd + 2 * f)


def work(case):
  item = 2 if case["dtype"] == "bf16" else 4
  if case["kind"] == "attention":
    tensor = case["batch"] * _nodes(case["refinement"]) * case["heads"] * case["head_dim"] * item
    mask = _nnz(case["refinement"], case["k_hop"]) / 8
    # q, k, v read and out written; with the backward dout read and dq, dk, dv written.
    return {"bytes": (8 if case["backward"] else 4) * tensor + mask,
            "flops": _attention_flops(case, 7 if case["backward"] else 2)}
  if case["kind"] == "rows":
    tensor = case["batch"] * case["n"] * case["channels"] * item
    elements = case["batch"] * case["n"] * case["channels"]
    # x read; gathered, normed, out written; three gradients read and one written.
    return {"bytes": (8 if case["backward"] else 4) * tensor, "flops": (40 if case["backward"] else 12) * elements}
  x = case["batch"] * _nodes(case["refinement"]) * case["d_model"] * item
  hd, d, f = case["heads"] * case["head_dim"], case["d_model"], case["ffw_hidden"]
  weights = (4 * hd * d + 2 * d * f) * item
  if case["kind"] == "block":
    # x, g read, out and dx written; weights read, their gradients written.
    return {"bytes": 4 * x + 2 * weights, "flops": _attention_flops(case, 7) + 3 * _gemm_flops(case)}
  return {"bytes": 2 * x + case["layers"] * weights,
          "flops": case["layers"] * (_attention_flops(case, 2) + _gemm_flops(case))}


def tolerance(case):
  # About four times the error against 64 bits that the paths show: 2.3e-3 (attention) to 6e-3 (a
  # block's gradients) and 9e-3 (24 layers) in bf16, 8e-6 with split products, 2.5e-6 (a saved
  # log-sum-exp under the backward's exponentials) with IEEE float32 products.
  if case["dtype"] == "bf16":
    return {"rel": 2e-2 if case["kind"] in ("block", "model") else 1e-2}
  if case["kind"] == "rows":
    return {"rel": 2e-6}
  return {"rel": 4e-5 if case.get("precision") == "bf16x3" else 1e-5}


# ------------------------------------------------------------------------------------------------
# The same results from plain torch in 64 bits.


@functools.lru_cache(maxsize=1)
def _columns(refinement, k_hop, reorder):
  """(row pointer, column indices) of the mask in the call's node order, on the GPU."""
  mask, perm, _ = _mesh(refinement, k_hop, reorder)
  m = mask if perm is None else mask[perm][:, perm]
  return (torch.from_numpy(np.asarray(m.indptr, np.int64)).to(DEV),
          torch.from_numpy(np.asarray(m.indices, np.int64)).to(DEV))


class _Dense:
  """Masked softmax attention of one [n, heads * ...] problem in float64, by chunks of rows."""

  def __init__(self, case, chunk=2048):
    self.ptr, self.idx = _columns(case["refinement"], case["k_hop"], case["reorder"])
    self.n, self.chunk = len(self.ptr) - 1, chunk

  def masks(self):
    """(first row, last row, mask of entries that take no part) of every chunk."""
    for lo in range(0, self.n, self.chunk):
      hi = min(lo + self.chunk, self.n)
      off = torch.ones(hi - lo, self.n, dtype=torch.bool, device=DEV)
      counts = self.ptr[lo + 1:hi + 1] - self.ptr[lo:hi]
      rows = torch.repeat_interleave(torch.arange(hi - lo, device=DEV), counts)
      off[rows, self.idx[self.ptr[lo]:self.ptr[hi]]] = False
      yield lo, hi, off

  def run(self, q, k, v, do, scale):
    """q, k, v, do float64 [batch, n, heads, head_dim] -> out (, dq, dk, dv)."""
    outs = [torch.zeros_like(q) for _ in range(1 if do is None else 4)]
    pairs = [(b, h) for b in range(q.shape[0]) for h in range(q.shape[2])]
    for lo, hi, off in self.masks():
      for b, h in pairs:
        qs, ks, vs = q[b, lo:hi, h].contiguous(), k[b, :, h].contiguous(), v[b, :, h].contiguous()
        p = torch.mm(qs * scale, ks.t()).masked_fill_(off, float("-inf"))
        p = torch.softmax(p, dim=1)
        o = torch.mm(p, vs)
        outs[0][b, lo:hi, h] = o
        if do is None:
          continue
        g = do[b, lo:hi, h].contiguous()
        ds = torch.mm(g, vs.t()).sub_((g * o).sum(1, keepdim=True)).mul_(p)
        outs[1][b, lo:hi, h] = torch.mm(ds, ks) * scale
        outs[2][b, :, h] += torch.mm(ds.t(), qs) * scale
        outs[3][b, :, h] += torch.mm(p.t(), g)
    return outs


class _DenseAttention(torch.autograd.Function):
  @staticmethod
  def forward(ctx, q, k, v, dense, scale):
    ctx.save_for_backward(q, k, v)
    ctx.dense, ctx.scale = dense, scale
    return dense.run(q, k, v, None, scale)[0]

  @staticmethod
  def backward(ctx, do):
    _, dq, dk, dv = ctx.dense.run(*ctx.saved_tensors, do, ctx.scale)
    return dq, dk, dv, None, None


def _norm(x):
  xc = x - x.mean(-1, keepdim=True)
  return xc * torch.rsqrt(xc.square().mean(-1, keepdim=True) + EPS)


def _exact_conditioned(norm, x, cond, p, prefix):
  scale, offset = (cond @ p[prefix + "linear.weight"].t() + p[prefix + "linear.bias"]).chunk(2, dim=-1)
  return norm * (1 + scale[:, None]) + offset[:, None]


def _exact_block(case, dense, x, cond, p, prefix=""):
  b, n, _ = x.shape
  h = _exact_conditioned(_norm(x), x, cond, p, prefix + "norm_mha.")
  q, k, v = (h @ p[prefix + "mha.qkv.weight"].t()).view(b, n, 3, case["heads"], case["head_dim"]).unbind(2)
  o = _DenseAttention.apply(q, k, v, dense, case["head_dim"] ** -0.5).reshape(b, n, -1)
  x = x + o @ p[prefix + "mha.final.weight"].t() + p[prefix + "mha.final.bias"]
  h = _exact_conditioned(_norm(x), x, cond, p, prefix + "norm_ffw.")
  y = torch.nn.functional.gelu(h @ p[prefix + "ffw.0.weight"].t() + p[prefix + "ffw.0.bias"], approximate="tanh")
  return x + y @ p[prefix + "ffw.2.weight"].t() + p[prefix + "ffw.2.bias"]


def exact(case, seed):
  if case["kind"] == "attention":
    q, k, v, do = (None if t is None else t.double() for t in _attention_inputs(case, seed))
    return _Dense(case).run(q, k, v, do, case["head_dim"] ** -0.5)
  if case["kind"] == "rows":
    x, perm, mul, add, grads = _rows_inputs(case, seed)
    x, mul, add = (t.double().requires_grad_(case["backward"]) for t in (x, mul, add))
    gathered = x[:, perm]
    normed = _norm(gathered)
    out = (normed * mul[:, None] + add[:, None])[:, torch.argsort(perm)]
    outs = [gathered, normed, out]
    if not case["backward"]:
      return outs
    return [t.detach() for t in outs] + list(torch.autograd.grad(outs, (x, mul, add), [g.double() for g in grads]))
  dense = _Dense(case)
  if case["kind"] == "block":
    x, cond, g = (t.double() for t in _features(case, seed, True))
    x.requires_grad_(True)
    p = {name: t.detach().double().requires_grad_(True) for name, t in _block(case, seed).named_parameters()}
    out = _exact_block(case, dense, x, cond, p)
    return [out.detach(), *torch.autograd.grad(out, (x, *p.values()), g.double())]
  with torch.no_grad():
    x, cond, _ = _features(case, seed, False)
    x, cond = x.double(), cond.double()
    model = _model(case, seed)
    p = {name: t.detach().double() for name, t in model.named_parameters()}
    perm = model.perm
    x = x if perm is None else x[:, perm]
    for i in range(case["layers"]):
      x = _exact_block(case, dense, x, cond, p, f"blocks.{i}.")
    y = _exact_conditioned(_norm(x), x, cond, p, "final_norm.")
    return [y if perm is None else y[:, torch.argsort(perm)]]
