"""Blocks and norms of a program's own classes in the mesh transformer: the transformer calls the methods
they have with the arguments it has always passed (CPU; the attention is replaced by a scaling)."""
import pytest
import torch
import torch.nn.functional as F

import faster_weathernext_amd as fwn
from faster_weathernext_amd import transformer

D, COND = 16, 4


class OwnNorm(torch.nn.Module):
  """A conditioned norm with the methods the blocks call, and no more."""

  def __init__(self):
    super().__init__()
    self.scale = torch.nn.Linear(COND, D)

  def forward(self, x, cond):
    return x * self.scale(cond)[:, None]

  def norm(self, x, cond, eps):
    return self(F.layer_norm(x, (D,), eps=eps), cond)

  def add_norm(self, x, y, cond, eps):
    return x + y, self.norm(x + y, cond, eps)


class OwnSubclass(transformer.NormConditioning):
  """NormConditioning with an affine-free norm of its own."""

  def norm(self, x, cond, eps):
    return 2 * F.layer_norm(x, (D,), eps=eps)

  def add_norm(self, x, y, cond, eps):
    return x + y, self.norm(x + y, cond, eps)


class OwnAffine(torch.nn.Module):
  """A final norm with what the transformer reads of it."""

  def affine(self, cond):
    return cond[:, :1].double() * torch.ones(D), cond[:, 1:2].expand(-1, D)


class Scaled(torch.nn.Module):
  def forward(self, h):
    return 0.5 * h


class OwnBlock(torch.nn.Module):
  """A block that has what the transformer uses: norm_mha, forward and forward_fused."""

  def __init__(self):
    super().__init__()
    self.norm_mha = OwnNorm()

  def forward(self, x, cond, normed=None):
    return x + self.norm_mha.norm(x, cond, 1e-5)

  def forward_fused(self, x, h, cond, next_norm=None):
    x = x + h
    return (x, None) if next_norm is None else (x, next_norm.norm(x, cond, 1e-5))


def _model(blocks):
  torch.manual_seed(0)
  model = fwn.MeshTransformer(refinement=1, k_hop=1, num_layers=2, d_model=D, num_heads=1, key_size=32, ffw_hidden=32,
                              cond_size=COND, reorder=False, device="cpu", dtype=torch.float32)
  for i, block in enumerate(model.blocks):
    if blocks is OwnBlock:
      model.blocks[i] = OwnBlock()
    else:
      block.norm_mha, block.norm_ffw, block.mha = blocks(), blocks(), Scaled()
      block.ffw[1] = torch.nn.ReLU()
  torch.nn.init.normal_(model.final_norm.linear.weight, std=0.2)
  return model


def _expected(model, x, cond):
  d = F.layer_norm(x, (D,), eps=model.eps)
  for i, block in enumerate(model.blocks):
    if isinstance(block, OwnBlock):
      x = x + block.norm_mha.norm(x, cond, 1e-5)
      continue
    h = block.norm_mha(d, cond) if i == 0 else block.norm_mha.norm(x, cond, model.eps)
    x = x + 0.5 * h
    x = x + block.ffw(block.norm_ffw.norm(x, cond, model.eps))
  mul, add = model.final_norm.affine(cond)
  return F.layer_norm(x, (D,), eps=model.eps) * mul[:, None] + add[:, None]


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("blocks", [OwnNorm, lambda: OwnSubclass(D, COND), OwnBlock])
def test_own_norms_and_blocks(monkeypatch, blocks, grad):
  model = _model(blocks)
  monkeypatch.setattr(transformer.MeshBlock, "feed_forward", lambda self, h: self.ffw(h))
  x, cond = torch.randn(2, model.n, D), torch.randn(2, COND)
  with torch.set_grad_enabled(grad):
    got = model(x, cond)
  assert got.requires_grad == grad
  torch.testing.assert_close(got, _expected(model, x, cond), rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("reorder", [True, False])
def test_own_final_norm(monkeypatch, reorder, grad):
  model = _model(OwnNorm)
  model.final_norm = OwnAffine()
  monkeypatch.setattr(transformer.MeshBlock, "feed_forward", lambda self, h: self.ffw(h))
  norm = lambda x, eps: F.layer_norm(x, (D,), eps=eps)
  if reorder:  # the two passes in torch
    model.perm = torch.randperm(model.n)
    monkeypatch.setattr(transformer, "gather_layer_norm", lambda x, perm, eps: (x[:, perm], norm(x[:, perm], eps)))

    def scatter(x, perm, mul, add, eps):
      assert mul.dtype == add.dtype == torch.float32 and mul.is_contiguous() and add.is_contiguous()
      return (norm(x, eps) * mul[:, None] + add[:, None])[:, torch.argsort(perm)]

    monkeypatch.setattr(transformer, "layer_norm_scatter", scatter)
  x, cond = torch.randn(2, model.n, D), torch.randn(2, COND)
  with torch.set_grad_enabled(grad):
    got = model(x, cond)
  torch.testing.assert_close(got.float(), _expected(model, x, cond).float(), rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("taken", [True, False])
@pytest.mark.parametrize("reorder", [True, False])
def test_conditioning_launch_holds_the_norms_that_use_it(monkeypatch, reorder, taken):
  """All norms but block 0's first and, where no scatter pass applies it, the final one; each gets its
  own affine."""
  torch.manual_seed(1)
  model = fwn.MeshTransformer(refinement=1, k_hop=1, num_layers=3, d_model=D, num_heads=1, key_size=32, ffw_hidden=32,
                              cond_size=COND, reorder=False, device="cpu", dtype=torch.float32).requires_grad_(False)
  for mod in model.modules():
    if isinstance(mod, transformer.NormConditioning):
      torch.nn.init.normal_(mod.linear.weight, std=0.3)
  for block in model.blocks:
    block.mha, block.ffw[1] = Scaled(), torch.nn.ReLU()
  seen = []
  monkeypatch.setattr(transformer, "affines_f32", lambda norms, cond: seen.extend(norms) or
                      [norm.affine_f32(cond) if taken else None for norm in norms])
  monkeypatch.setattr(transformer.MeshBlock, "feed_forward", lambda self, h: self.ffw(h))
  norm = lambda x, mul, add, eps: F.layer_norm(x, (D,), eps=eps) * mul[:, None] + add[:, None]
  monkeypatch.setattr(transformer, "add_layer_norm_affine",
                      lambda x, y, mul, add, eps: (x + y, norm(x + y, mul, add, eps)))
  monkeypatch.setattr(transformer, "layer_norm_affine", lambda x, mul, add, eps: norm(x, mul, add, eps))
  if reorder:
    model.perm = torch.arange(model.n)
    monkeypatch.setattr(transformer, "gather_layer_norm", lambda x, perm, eps: (x, F.layer_norm(x, (D,), eps=eps)))
    monkeypatch.setattr(transformer, "layer_norm_scatter", lambda x, perm, mul, add, eps: norm(x, mul, add, eps))
  x, cond = torch.randn(2, model.n, D), torch.randn(2, COND)
  got = model(x, cond)
  want = [b.norm_ffw for b in model.blocks] + [b.norm_mha for b in model.blocks[1:]] + [model.final_norm] * reorder
  assert len(seen) == len(want) and all(a is b for a, b in zip(seen, want))
  torch.testing.assert_close(got, _expected(model, x, cond), rtol=1e-5, atol=1e-5)
