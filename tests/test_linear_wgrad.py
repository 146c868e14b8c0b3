"""A Linear's weight and bias gradients over many rows (``fwn_linear_wgrad_launch``) against float64 at
the edges of its split (32-row stages, 256 x 256 tiles with ragged columns, one row range to many),
and ``mha.linear`` against the module it stands for."""
import ctypes

import pytest
import torch
import torch.nn.functional as F

from faster_weathernext_amd import _native as nat
from faster_weathernext_amd import mha

DEV = "cuda"


SIZES = [(1, 64, 64), (31, 64, 256), (32, 256, 64), (33, 256, 256), (127, 192, 320), (128, 320, 192), (129, 512, 256),
         (257, 768, 2304), (1000, 128, 384), (4097, 256, 256), (70001, 64, 128), (9001, 1536, 384)]


def _framed(t):
  """A copy of t [rows, cols] on the GPU inside NaNs: a read outside it shows."""
  rows, cols = t.shape
  buf = torch.full(((rows + 8) * cols,), float("nan"), device=DEV, dtype=torch.bfloat16)
  return buf[4 * cols:(rows + 4) * cols].view(rows, cols).copy_(t)


def _random(rows, outs, ins):
  gen = torch.Generator().manual_seed(rows + outs)
  return [torch.randn(rows, cols, generator=gen).to(torch.bfloat16) for cols in (outs, ins)]


def _integers(rows, outs, ins):
  gen = torch.Generator().manual_seed(rows + ins)
  return [torch.randint(-2, 3, (rows, cols), generator=gen).to(torch.bfloat16) for cols in (outs, ins)]


def _gradients(g, x):
  """(weight gradient, bias gradient) in float64."""
  return g.double().t() @ x.double(), g.double().sum(0)


def _bounds(g, x, dw, db):
  """How far a float32 sum of the rows in any order, rounded to bf16 once, is from the float64 sums. The
  rounding: half an ulp of 8 significant bits, at most 2^-8 of the value. The sum: each of `rows`
  additions rounds by 2^-24 of a partial sum, and the partial sums of k random terms grow as sqrt(k)
  times a term's deviation, together at most (2 / 3) sqrt(rows) 2^-24 |g| |x| (norms over the rows);
  twelve times that for partial sums several deviations large."""
  rows, gn, xn = g.shape[0], g.double().norm(dim=0), x.double().norm(dim=0)
  sums = 8 * rows ** 0.5 * 2.0 ** -24
  return 2.0 ** -8 * dw.abs() + sums * gn[:, None] * xn, 2.0 ** -8 * db.abs() + sums * gn * rows ** 0.5


@pytest.mark.gpu
@pytest.mark.parametrize("rows,outs,ins", SIZES)
@pytest.mark.parametrize("bias", [True, False])
def test_wgrad_matches_float64(rows, outs, ins, bias):
  g, x = _random(rows, outs, ins)
  dw, db = mha.linear_wgrad(_framed(g), _framed(x), bias)
  want = _gradients(g, x)
  assert (db is None) == (not bias)
  for got, ref, bound in zip((dw, db), want, _bounds(g, x, *want)):
    if got is not None:
      assert bool(((got.double().cpu() - ref).abs() <= bound).all())
      # One rounding to bf16 leaves 1.7e-3 of the norm.
      assert float((got.double().cpu() - ref).norm() / ref.norm()) <= 3e-3


@pytest.mark.gpu
@pytest.mark.parametrize("rows,outs,ins", SIZES)
def test_wgrad_of_integers_is_exact(rows, outs, ins):
  """Entries from -2 to 2: every partial sum is a whole number below 2^24, so the float32 sums are exact
  in any order and the results are the true sums rounded to bf16, to the bit."""
  g, x = _integers(rows, outs, ins)
  for got, ref in zip(mha.linear_wgrad(_framed(g), _framed(x), True), _gradients(g, x)):
    assert torch.equal(got.cpu(), ref.to(torch.bfloat16))


@pytest.mark.parametrize("rows,outs,ins", [s for s in SIZES if s[0] > 32])
def test_a_left_out_stage_would_show(rows, outs, ins):
  """The two tests above fail for results that miss rows (on the CPU, the rows taken out of the sums):
  any one 32-row stage for both, and with whole numbers a single row."""
  for make, spans in ((_random, (32,)), (_integers, (1, 32))):
    g, x = make(rows, outs, ins)
    want = _gradients(g, x)
    bounds = _bounds(g, x, *want)
    for span in spans:
      for lo in {0, rows // 2 // 32 * 32, (rows - 1) // 32 * 32 if span == 1 else rows - span}:
        part = _gradients(g[lo:lo + span], x[lo:lo + span])
        for ref, miss, bound in zip(want, part, bounds):
          off = ref - miss
          if make is _integers:
            assert not torch.equal(off.to(torch.bfloat16), ref.to(torch.bfloat16))
          else:
            assert bool(((off - ref).abs() > bound).any()) or float((off - ref).norm() / ref.norm()) > 3e-3


def test_invalid_arguments_are_refused():
  lib, size = nat.lib(), ctypes.c_uint64()
  for bad in ((0, 64, 64), (5, 63, 64), (5, 64, 96), (5, 64, 0), (5, 1 << 15, 64)):
    assert lib.fwn_linear_wgrad_workspace_size(*bad, ctypes.byref(size)) != 0
    assert lib.fwn_linear_wgrad_launch(*bad, 16, 16, 16, 16, 16, 1 << 40, None) != 0
  assert lib.fwn_linear_wgrad_workspace_size(40962, 768, 768, None) != 0
  assert lib.fwn_linear_wgrad_workspace_size(40962, 768, 768, ctypes.byref(size)) == 0 and size.value > 0
  for bad in ((None, 16, 16, 16, 16), (16, None, 16, 16, 16), (16, 16, None, 16, 16), (16, 16, 16, 16, None),
              (24, 16, 16, 16, 16), (16, 24, 16, 16, 16), (16, 16, 24, 16, 16), (16, 16, 16, 24, 16), (16, 16, 16, 16, 24)):
    assert lib.fwn_linear_wgrad_launch(40962, 768, 768, *bad, size.value, None) != 0
  assert lib.fwn_linear_wgrad_launch(40962, 768, 768, 16, 16, 16, 16, 16, size.value - 1, None) != 0


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["plain", "no_bias", "3d", "strided", "frozen_weight", "frozen_input", "frozen_bias",
                                  "odd_size", "hooked", "graph", "saved_hooks", "batched"])
def test_linear_matches_the_module(monkeypatch, form):
  monkeypatch.setattr(mha, "WGRAD_ROWS", 1)
  torch.manual_seed(1)
  lin = torch.nn.Linear(96 if form == "odd_size" else 128, 192, bias=form != "no_bias", device=DEV, dtype=torch.bfloat16)
  x = torch.randn(2, 350, 96 if form == "odd_size" else 256, device=DEV).to(torch.bfloat16)
  if form == "strided":
    x = x[..., ::2]
  elif form != "odd_size":
    x = x[..., :128].contiguous()
  x = x.requires_grad_(form != "frozen_input")
  lin.weight.requires_grad_(form != "frozen_weight")
  if lin.bias is not None:
    lin.bias.requires_grad_(form != "frozen_bias")
  if form == "hooked":
    lin.register_forward_hook(lambda mod, args, out: out * 2)
  g = torch.randn(2, 350, 192, device=DEV).to(torch.bfloat16)
  leaves = [t for t in (x, *lin.parameters()) if t.requires_grad]
  calls = []
  monkeypatch.setattr(mha._Linear, "forward", staticmethod(lambda ctx, *a, f=mha._Linear.forward: calls.append(1) or f(ctx, *a)))

  def run(f, graph):
    packs = []
    if form == "saved_hooks":
      with torch.autograd.graph.saved_tensors_hooks(lambda t: packs.append(1) or t.cpu(), lambda t: t.to(DEV)):
        out = f(x)
      assert packs
    else:
      out = f(x)
    if form == "batched":
      return [out, *torch.autograd.grad(out, leaves, torch.stack([g, -g.flip(1)]), is_grads_batched=True)]
    return [out, *torch.autograd.grad(out, leaves, g, create_graph=graph)]

  got, want = run(lambda t: mha.linear(lin, t), form == "graph"), run(lin, form == "graph")
  assert len(calls) == (form not in ("odd_size", "hooked"))
  if form == "graph":  # second derivatives through the first ones
    second = lambda grads: torch.autograd.grad(sum((t.float() ** 2).sum() for t in grads[1:]), [x, lin.weight])
    got, want = got + list(second(got)), want + list(second(want))
  # Each side rounds float32 sums to bf16 (2^-9) at most twice along the way.
  for a, b in zip(got, want):
    assert a.shape == b.shape and a.dtype == b.dtype
    assert float((a.double() - b.double()).norm() / b.double().norm()) <= 2.0 ** -7


def test_output_may_be_written_in_place():
  """A Linear's output is its caller's: an in-place activation or residual add after it works as after
  the module, on the output and on a view of it."""
  torch.manual_seed(4)
  lin = torch.nn.Linear(64, 128, dtype=torch.bfloat16)
  x = torch.randn(6, 64).to(torch.bfloat16).requires_grad_(True)
  for shape in ((6, 128), (2, 3, 128)):
    y = mha._Linear.apply(x, lin.weight, lin.bias).view(shape)
    want = lin(x).view(shape)
    assert torch.equal(torch.nn.functional.silu(y, inplace=True), torch.nn.functional.silu(want, inplace=True))
    (y.add_(1.0) * 2).sum()


@pytest.mark.gpu
@pytest.mark.parametrize("act", [torch.nn.SiLU(inplace=True), torch.nn.ReLU(inplace=True)])
def test_in_place_activation_after_linear(monkeypatch, act):
  monkeypatch.setattr(mha, "WGRAD_ROWS", 1)
  torch.manual_seed(5)
  lin = torch.nn.Linear(64, 128, device=DEV, dtype=torch.bfloat16)
  x = torch.randn(3, 100, 64, device=DEV).to(torch.bfloat16).requires_grad_(True)
  g = torch.randn(3, 100, 128, device=DEV).to(torch.bfloat16)
  leaves = [x, *lin.parameters()]
  run = lambda f: [out := act(f(x)), *torch.autograd.grad(out, leaves, g)]
  # Each side rounds float32 sums to bf16 (2^-9) at most twice along the way.
  for a, b in zip(run(lambda t: mha.linear(lin, t)), run(lin)):
    assert a.shape == b.shape and float((a.double() - b.double()).norm() / b.double().norm()) <= 2.0 ** -7


@pytest.mark.parametrize("need_x,need_w", [(True, True), (True, False), (False, True), (False, False)])
def test_saves_what_its_gradients_read(need_x, need_w):
  """x is kept for the weight's gradient and the weight for x's, as the module keeps them: not a frozen
  weight's input, and a weight whose input needs no gradient may be written before the backward."""
  lin = torch.nn.Linear(64, 128, dtype=torch.bfloat16)
  lin.weight.requires_grad_(need_w)
  x = torch.randn(6, 64).to(torch.bfloat16).requires_grad_(need_x)
  kept = []
  with torch.autograd.graph.saved_tensors_hooks(lambda t: kept.append(t.data_ptr()) or t, lambda t: t):
    mha._Linear.apply(x, lin.weight, lin.bias)
    own, kept = kept, []
    lin(x)
  assert sorted(own) == sorted(kept) == sorted([x.data_ptr()] * need_w + [lin.weight.data_ptr()] * need_x)
