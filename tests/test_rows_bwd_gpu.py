"""Gradients of the row passes as one HIP pass (``fwn_rows_norm_bwd_launch``): against float64 torch at
the sizes where the kernel's split changes (one vector per lane to sixteen, ragged channel counts,
rows fewer than a workgroup's, several batch members), with each gradient missing or strided, and
under create_graph or with batched gradients, where the torch composite runs."""
import numpy as np
import pytest
import torch

from faster_weathernext_amd import _native as nat
from faster_weathernext_amd import rows

pytestmark = pytest.mark.gpu
DEV = "cuda"
EPS = 1e-5
# Against float64 on the same (rounded) inputs: float32 sums of up to 4,096 terms, one bf16 rounding
# (2^-9, rel RMS 1.7e-3) of each bf16 result.
TOL = {torch.float32: 2e-6, torch.bfloat16: 3e-3}


def _rel(got, want):
  want = want.double()
  return float((got.double() - want).norm() / want.norm().clamp_min(1e-30))


def _norm(x):
  c = x - x.mean(-1, keepdim=True)
  return c * torch.rsqrt(c.square().mean(-1, keepdim=True) + EPS)


def _data(b, n, c, dtype, seed):
  g = torch.Generator(device=DEV).manual_seed(seed)
  t = [torch.randn(b, n, c, device=DEV, generator=g).to(dtype) for _ in range(4)]
  x = (t[0] * 1.5 + 0.3).to(dtype)
  mul, add = 1 + 0.2 * torch.randn(b, c, device=DEV, generator=g), torch.randn(b, c, device=DEV, generator=g)
  return x, t[1], t[2], t[3], mul, add, torch.randperm(n, device=DEV, generator=g)


SHAPES = [(1, 1, 8), (2, 5, 256), (1, 33, 264), (3, 17, 512), (1, 700, 768), (2, 300, 1000), (1, 9, 2056), (1, 21, 4096),
          (1, 5000, 64), (1100, 2, 16)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("b,n,c", SHAPES)
def test_gradients_match_float64(dtype, b, n, c):
  print(f"row gradients {dtype} {b} {n} {c}", flush=True)
  x, g1, g2, y, mul, add, perm = _data(b, n, c, dtype, n + c)
  leaf = lambda *ts: [t.detach().clone().requires_grad_(True) for t in ts]
  wide = lambda *ts: [t.detach().double().requires_grad_(True) for t in ts]
  tol = TOL[dtype]

  (xa,), (xr,) = leaf(x), wide(x)
  got = torch.autograd.grad(rows.gather_layer_norm(xa, perm, eps=EPS), xa, (g1, g2))
  p = xr[:, perm]
  want = torch.autograd.grad((p, _norm(p)), xr, (g1.double(), g2.double()))
  assert _rel(got[0], want[0]) <= tol

  for perm_, fn in ((perm, lambda *a: rows.layer_norm_scatter(a[0], perm, mul=a[1], add=a[2], eps=EPS)),
                    (None, lambda *a: rows.layer_norm_affine(a[0], mul=a[1], add=a[2], eps=EPS))):
    la, lr = leaf(x, mul, add), wide(x, mul, add)
    got = torch.autograd.grad(fn(*la), la, g1)
    z = _norm(lr[0]) * lr[1][:, None] + lr[2][:, None]
    z = z if perm_ is None else z[:, torch.argsort(perm_)]
    for k, (a, r) in enumerate(zip(got, torch.autograd.grad(z, lr, g1.double()))):
      # a single row's mul gradient with eight channels has terms that cancel: 1e-5 of it
      assert _rel(a, r) <= (tol if k == 0 else 1e-5), (perm_ is None, k)

  la = leaf(x, y, mul, add)
  s, out = rows.residual_norm(la[0], la[1], mul=la[2], add=la[3], eps=EPS)
  assert torch.equal(s, x + y)
  got = torch.autograd.grad((s, out), la, (g1, g2))
  sr, mr, ar = wide(x + y, mul, add)
  want = torch.autograd.grad((sr * 1, _norm(sr) * mr[:, None] + ar[:, None]), (sr, mr, ar), (g1.double(), g2.double()))
  assert torch.equal(got[0], got[1])
  for k, (a, r) in enumerate(zip((got[0], got[2], got[3]), want)):
    assert _rel(a, r) <= (tol if k == 0 else 1e-5), k


def test_missing_strided_and_offset_gradients():
  """One output unused (its gradient is zero), an expanded gradient, a gradient and an input whose
  base is not 16-byte aligned: the same results as from dense gradients."""
  b, n, c = 2, 40, 72
  x, g1, g2, y, mul, add, perm = _data(b, n, c, torch.float32, 3)
  xa = x.clone().requires_grad_(True)
  zero = torch.zeros_like(g1)
  pair = lambda: rows.gather_layer_norm(xa, perm, eps=EPS)
  grad = lambda o, g: torch.autograd.grad(o, xa, g)[0]
  assert torch.equal(grad(pair()[0], g1), grad(pair(), (g1, zero)))
  assert _rel(grad(pair()[1], g2), grad(pair(), (zero, g2))) <= 1e-6
  one = torch.ones((), device=DEV).expand(b, n, c)
  affine = lambda: rows.layer_norm_affine(xa, mul=mul, add=add, eps=EPS)
  assert torch.equal(grad(affine(), one), grad(affine(), one.contiguous()))
  store = torch.empty(b * n * c + 1, device=DEV)
  off = store[1:].view(b, n, c).copy_(g1)
  assert off.data_ptr() % 16 != 0
  assert torch.equal(grad(affine(), off), grad(affine(), g1))
  # residual_norm takes any layout and mixed dtypes, as torch's add does
  s0, o0 = rows.residual_norm(x, y, mul=mul, add=add)
  flipped = x.transpose(0, 1).contiguous().transpose(0, 1)
  assert not flipped.is_contiguous() and not (flipped + y).is_contiguous()
  for xx in (off.copy_(x), flipped, x.permute(2, 0, 1).contiguous().permute(1, 2, 0)):
    s, o = rows.residual_norm(xx, y, mul=mul, add=add)
    assert torch.equal(s, s0) and torch.equal(o, o0)
  same = y[:, :1].expand(b, n, c)
  s, o = rows.residual_norm(x, same, mul=mul, add=add)
  s1, o1 = rows.residual_norm(x, same.contiguous(), mul=mul, add=add)
  assert torch.equal(s, s1) and torch.equal(o, o1)
  s, o = rows.residual_norm(x, y.to(torch.bfloat16), mul=mul, add=add)
  assert s.dtype == torch.float32 and torch.equal(s, x + y.to(torch.bfloat16))


def test_second_derivatives():
  """A backward that is itself differentiated (create_graph) runs as torch operations: gradients of
  a gradient's norm against the float64 composite."""
  b, n, c = 1, 12, 24
  x, g1, g2, y, mul, add, perm = _data(b, n, c, torch.float32, 5)

  def penalty(norm_fn, xs, ms, as_, g):
    z = norm_fn(xs, ms, as_)
    (gx,) = torch.autograd.grad(z, xs, g, create_graph=True)
    return torch.autograd.grad(gx.square().sum(), (xs, ms))

  leaf = lambda t: t.detach().clone().requires_grad_(True)
  got = penalty(lambda a, m, d: rows.layer_norm_scatter(a, perm, mul=m, add=d, eps=EPS), leaf(x), leaf(mul), leaf(add), g1)
  want = penalty(lambda a, m, d: (_norm(a) * m[:, None] + d[:, None])[:, torch.argsort(perm)], leaf(x.double()),
                 leaf(mul.double()), leaf(add.double()), g1.double())
  for a, r in zip(got, want):
    assert _rel(a, r) <= 1e-5


def test_batched_gradients():
  """is_grads_batched hands the backward vmap's batched tensors: each member's gradients as by itself."""
  b, n, c = 2, 12, 24
  x, g1, g2, y, mul, add, perm = _data(b, n, c, torch.float32, 7)
  leaves = [t.clone().requires_grad_(True) for t in (x, mul, add)]
  xa, ma, da = leaves
  grads = torch.stack([g1, g2, y])
  outs = {"scatter": (rows.layer_norm_scatter(xa, perm, mul=ma, add=da), leaves),
          "affine": (rows.layer_norm_affine(xa, mul=ma, add=da), leaves),
          "gather": (rows.gather_layer_norm(xa, perm)[1], [xa]),
          "residual": (rows.residual_norm(xa, y, mul=ma, add=da)[1], leaves)}
  for name, (out, wrt) in outs.items():
    got = torch.autograd.grad(out, wrt, grads, is_grads_batched=True, retain_graph=True)
    for i, g in enumerate(grads):
      for a, r in zip(got, torch.autograd.grad(out, wrt, g, retain_graph=True)):
        assert _rel(a[i], r) <= 1e-5, name


def test_bad_arguments_are_refused():
  x, g1, _, _, mul, _, perm = _data(1, 8, 16, torch.float32, 0)
  gx, gm = torch.empty_like(x), torch.empty(1, 16, device=DEV)
  L, d = nat.lib(), nat.RowsDesc(1, 8, 16, nat.F32, EPS)
  st = torch.cuda.current_stream().cuda_stream
  call = lambda perm_=None, how=0, gx_=gx.data_ptr(), m=None, a=None, ws=None, size=0, d_=d: L.fwn_rows_norm_bwd_launch(
      d_, x.data_ptr(), perm_, how, g1.data_ptr(), None, mul.data_ptr(), gx_, m, a, ws, size, st)
  assert call() == nat.OK
  torch.cuda.synchronize()
  bad = nat.ERR_INVALID_ARG
  assert call(how=1) == bad and call(perm_=perm.data_ptr()) == bad and call(perm_=perm.data_ptr(), how=3) == bad
  assert call(gx_=None) == bad and call(gx_=x.data_ptr()) == bad and call(gx_=gx.data_ptr() + 4) == bad
  assert call(m=gm.data_ptr()) == bad and call(m=gm.data_ptr(), a=gm.data_ptr()) == bad
  assert call(m=gm.data_ptr(), a=gm.data_ptr(), ws=gx.data_ptr(), size=4) == bad
  assert call(d_=nat.RowsDesc(1, 8, 12, nat.F32, EPS)) == bad
