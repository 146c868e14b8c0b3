"""mha.linear_rows (the GEMM row split used by the mesh transformer without autograd) against a
plain torch linear layer: the split at a multiple of 512 rows, with and without bias. CPU,
float32 and float64. The GELU epilogue is checked on the GPU (test_transformer_gpu's inference
path), where it is hipBLASLt's tanh GELU; torch's CPU kernel for it uses another GELU form."""
import pytest
import torch
import torch.nn.functional as F

from faster_weathernext_amd.mha import ROW_QUANTUM, linear_rows


@pytest.mark.parametrize("rows", [300, ROW_QUANTUM, 2 * ROW_QUANTUM + 6])
@pytest.mark.parametrize("bias,gelu", [(False, False), (True, False)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_linear_rows_matches_linear(rows, bias, gelu, dtype):
  g = torch.Generator().manual_seed(rows)
  x = torch.randn(rows, 24, generator=g, dtype=dtype)
  w = torch.randn(40, 24, generator=g, dtype=dtype)
  b = torch.randn(40, generator=g, dtype=dtype) if bias else None
  ref = F.linear(x, w, b)
  if gelu:
    ref = F.gelu(ref, approximate="tanh")
  got = linear_rows(x, w, b, gelu=gelu)
  assert got.shape == ref.shape and got.dtype == dtype
  tol = 1e-5 if dtype == torch.float32 else 1e-12
  torch.testing.assert_close(got, ref, rtol=tol, atol=tol)


def test_linear_rows_split_rows_are_the_unsplit_rows():
  # Every row of the split result equals the same row computed on its own (float64: the GEMM
  # order cannot move a row's value beyond rounding).
  g = torch.Generator().manual_seed(1)
  x = torch.randn(ROW_QUANTUM + 3, 8, generator=g, dtype=torch.float64)
  w = torch.randn(5, 8, generator=g, dtype=torch.float64)
  got = linear_rows(x, w)
  for r in (0, ROW_QUANTUM - 1, ROW_QUANTUM, ROW_QUANTUM + 2):
    torch.testing.assert_close(got[r], x[r] @ w.t(), rtol=1e-12, atol=1e-12)


def test_residual_norm_hands_a_contiguous_sum_to_the_norm(monkeypatch):
  """torch's add keeps a dense operand's strides; the norm's pass takes contiguous rows only."""
  from faster_weathernext_amd import rows
  seen = []
  monkeypatch.setattr(rows, "layer_norm_affine", lambda s, **kw: seen.append(s) or s)
  x, y = torch.randn(2, 5, 8), torch.randn(2, 5, 8)
  for xx in (x, x.transpose(0, 1).contiguous().transpose(0, 1), x.permute(2, 0, 1).contiguous().permute(1, 2, 0)):
    s, _ = rows.residual_norm(xx, y, mul=None, add=None)
    assert s.is_contiguous() and seen[-1] is s and torch.equal(s, x + y)


def test_plain_modules_are_those_whose_call_is_their_forward():
  from faster_weathernext_amd.mha import is_plain
  make = lambda: torch.nn.Linear(4, 4)
  assert is_plain(make(), torch.nn.Linear) and not is_plain(make(), torch.nn.Sequential)
  hooked, replaced, compiled = make(), make(), make()
  hooked.register_forward_pre_hook(lambda mod, args: None)
  replaced.forward = lambda x: x
  compiled._compiled_call_impl = lambda x: x  # what Module.compile() sets and a call then runs
  assert torch.equal(compiled(torch.ones(4)), torch.ones(4))
  for lin in (hooked, replaced, compiled, torch.nn.utils.parametrizations.weight_norm(make())):
    assert not is_plain(lin, torch.nn.Linear)


def test_rows_from_which_training_takes_the_split_gradients():
  """As many entries as WGRAD_ROWS rows have at 800 wide, whichever side of the weight is the smaller;
  always from eight times as many rows, never below them."""
  from faster_weathernext_amd.mha import rows_enough
  for rows, d, past in ((10242, 512, False), (20484, 256, False), (40962, 128, False), (8191, 4096, False), (65535, 64, False),
                        (8192, 832, True), (10242, 768, True), (20484, 384, True), (30726, 256, True), (40962, 192, True),
                        (65536, 64, True), (40962, 768, True)):
    for outs, ins in ((d, d), (3 * d, d), (d, 4 * d)):
      assert rows_enough(rows, outs, ins) == past
