"""The conditioning of several norms in one launch (``fwn_cond_affine_launch``) against float64, at
the edges of its split (256 columns a workgroup, 4 batch members a pass, 64 norms a launch), and the
transformer's calls that take it against the same calls with each norm projected by itself."""
import pytest
import torch

import faster_weathernext_amd as fwn
from faster_weathernext_amd import _native as nat
from faster_weathernext_amd import rows, transformer

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("count,batch,channels,size", [(1, 1, 8, 1), (3, 2, 128, 32), (2, 4, 136, 7), (65, 5, 64, 16),
                                                       (2, 9, 768, 512), (1, 3, 4096, 33)])
def test_cond_affine_matches_float64(dtype, count, batch, channels, size):
  g = torch.Generator(device=DEV).manual_seed(count + size)
  rand = lambda *shape: torch.randn(*shape, device=DEV, generator=g).to(dtype)
  cond, ws, bs = rand(batch, size), [rand(2 * channels, size) for _ in range(count)], \
      [rand(2 * channels) for _ in range(count)]
  got = rows.cond_affine(cond, ws, bs)
  assert len(got) == count
  for (mul, add), w, b in zip(got, ws, bs):
    want = cond.double() @ w.double().t() + b.double()
    # size + 2 roundings to float32 (2^-24 each), relative to the sum of the terms' magnitudes.
    bound = (size + 2) * 2.0 ** -24 * (cond.double().abs() @ w.double().abs().t() + b.double().abs() + 1)
    bound_mul, bound_add = bound.chunk(2, dim=-1)
    assert mul.shape == add.shape == (batch, channels) and mul.dtype == torch.float32
    assert bool(((mul.double() - want[:, :channels] - 1).abs() <= bound_mul).all())
    assert bool(((add.double() - want[:, channels:]).abs() <= bound_add).all())


def test_invalid_arguments_are_refused():
  w = torch.randn(16, 4, device=DEV)
  table = (nat.ctypes.c_void_p * 1)(w.data_ptr())
  call = lambda count, batch, channels, size, dtype=nat.F32, weight=table: nat.lib().fwn_cond_affine_launch(
      count, batch, channels, size, dtype, w.data_ptr(), weight, table, w.data_ptr(), w.data_ptr(), None)
  null = (nat.ctypes.c_void_p * 1)(None)
  for bad in (call(0, 1, 8, 4), call(nat.COND_MAX + 1, 1, 8, 4), call(1, 0, 8, 4), call(1, 1, 0, 4), call(1, 1, 8, 0),
              call(1, 1, 1 << 20, 4), call(1, 1, 8, 4, 7), call(1, 1, 8, 4, weight=null)):
    assert bad != 0


@pytest.mark.parametrize("reorder", [True, False])
@pytest.mark.parametrize("form", ["plain", "expanded", "strided", "hooked", "unconditioned"])
def test_model_forward_with_and_without_the_one_launch(monkeypatch, reorder, form):
  """Forms the launch takes ("plain", "unconditioned": frozen parameters with gradients enabled) and
  forms left to each norm's own projection give the results of the latter."""
  torch.manual_seed(3)
  model = fwn.MeshTransformer(refinement=2, k_hop=3, num_layers=3, d_model=64, num_heads=2, key_size=32, ffw_hidden=64,
                              cond_size=8, reorder=reorder, device=DEV, dtype=torch.float32)
  for mod in model.modules():
    if isinstance(mod, fwn.transformer.NormConditioning):
      torch.nn.init.normal_(mod.linear.weight, std=0.2)
      torch.nn.init.normal_(mod.linear.bias, std=0.2)
  x, cond = torch.randn(2, model.n, 64, device=DEV), torch.randn(2, 8, device=DEV)
  seen = []
  if form == "expanded":
    cond = cond[:1].expand(2, 8)
  elif form == "strided":
    cond = torch.randn(2, 16, device=DEV)[:, ::2]
  elif form == "hooked":
    model.blocks[1].norm_ffw.linear.register_forward_hook(lambda *a: seen.append(1))
  elif form == "unconditioned":
    model.requires_grad_(False)
  calls = []
  monkeypatch.setattr(transformer, "cond_affine", lambda *a: calls.append(1) or rows.cond_affine(*a))
  with torch.set_grad_enabled(form == "unconditioned"):
    got = model(x, cond)
    assert len(calls) == (form in ("plain", "unconditioned")) and len(seen) == (form == "hooked")
    monkeypatch.setattr(transformer, "COND_WORK", -1)
    want = model(x, cond)
  # float32 sums of 8 terms in another order, through three layers.
  assert float((got - want).norm() / want.norm()) <= 2e-6
