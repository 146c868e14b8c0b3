"""The row passes' kernels for large tensors, whose outputs bypass the caches: the built code has the
hint in them and in no other (a run-time choice between two stores loses it), and their results are
those of the kernels for small tensors, to the bit."""
import collections
import os
import re
import shutil
import subprocess

import pytest
import torch

from faster_weathernext_amd import _native as nat
from faster_weathernext_amd import rows

DEV = "cuda"
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_stores_of_the_built_kernels(tmp_path):
  lib = shutil.copy(nat.LIB_PATH, tmp_path / "lib.so")
  subprocess.run([OBJDUMP, "--offloading", lib], cwd=tmp_path, check=True, capture_output=True)
  seen = collections.Counter()
  for obj in sorted(tmp_path.glob("lib.so.*gfx950")):
    if b"norm_scatter_kernel" not in obj.read_bytes():
      continue
    text = subprocess.run([OBJDUMP, "-d", str(obj)], check=True, capture_output=True, text=True).stdout
    for part in re.split(r"\n[0-9a-f]+ <", text)[1:]:
      name = re.match(r"_ZN3fwn\S*?(gather_norm|norm_scatter|norm_bwd)_kernelI\S*Lb([01])EEEv", part)
      if name is None:
        continue
      stores = [line for line in part.splitlines() if "global_store_dwordx4" in line]
      hinted = [line for line in stores if re.search(r"\bnt\b", line.split("//")[0])]
      assert stores and len(hinted) == (len(stores) if name[2] == "1" else 0), name[0]
      seen[name[1], name[2]] += 1
  assert set(seen) == {(k, nt) for k in ("gather_norm", "norm_scatter", "norm_bwd") for nt in "01"}


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_large_tensors_match_their_parts(dtype):
  """Rows are independent: a pass over a tensor past the line and over eight parts of it, far below,
  give the same rows."""
  c, parts = 768, 8
  n = parts * (11300 if dtype == torch.float32 else 22600)  # 278 MB
  g = torch.Generator(device=DEV).manual_seed(1)
  rand = lambda: torch.randn(1, n, c, device=DEV, generator=g).to(dtype)
  x, y = rand(), rand()
  assert x.numel() * x.element_size() >= 256 << 20
  mul, add = 1 + 0.1 * torch.randn(1, c, device=DEV, generator=g), torch.randn(1, c, device=DEV, generator=g)
  # A permutation that keeps to the parts, so that they can be permuted by themselves.
  perm = torch.cat([k * (n // parts) + torch.randperm(n // parts, device=DEV, generator=g) for k in range(parts)])
  passes = {
      "gather": lambda x, y, p: rows.gather_layer_norm_forward(x, p),
      "scatter": lambda x, y, p: [rows.layer_norm_scatter_forward(x, p, mul, add)],
      "affine": lambda x, y, p: [rows.layer_norm_affine_forward(x, mul, add)],
      "add": lambda x, y, p: rows.add_layer_norm_affine(x, y, mul=mul, add=add),
      "gather gradient": lambda x, y, p: rows._norm_backward_pass(x, 1e-5, y, x, perm=p, perm_rows=nat.ROWS_PERM_OUT)[:1],
      "scatter gradient": lambda x, y, p: rows._norm_backward_pass(x, 1e-5, y, None, mul, p, nat.ROWS_PERM_GRAD)[:1],
  }
  for name, run in passes.items():
    whole = run(x, y, perm)
    for k in range(parts):
      lo, hi = k * (n // parts), (k + 1) * (n // parts)
      for a, b in zip(whole, run(x[:, lo:hi].contiguous(), y[:, lo:hi].contiguous(), perm[lo:hi] - lo)):
        assert torch.equal(a[:, lo:hi], b), (name, k)
  whole = rows._norm_backward_pass(x, 1e-5, y, None, mul, sums=True)
  xf, yf = x.double(), y.double()
  xhat = (xf - xf.mean(-1, keepdim=True)) * torch.rsqrt(xf.var(-1, unbiased=False, keepdim=True) + 1e-5)
  # float32 sums of n terms: the additions of random terms leave at most about sqrt(n) 2^-24 of the
  # terms' norm, here taken four times (0.02 of sums whose terms are of order 1: a row left out shows).
  for got, terms in zip(whole[1:], (yf * xhat, yf)):
    assert bool(((got - terms.sum(1)).abs() <= 4 * n ** 0.5 * 2.0 ** -24 * terms.norm(dim=1)).all())
