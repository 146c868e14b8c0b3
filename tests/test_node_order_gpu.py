"""Tile lists laid out for the kernels (``TileList.launch_list``, ``exchange_lists``: a node order of
their own, packed columns): the kernels gather and scatter the rows through the node tables, so the op's results are those of the mask in the
caller's order. Against the float64 dense oracle at block edges, every head size, split work items,
non-symmetric masks, packed tensors and both backwards."""
import numpy as np
import pytest
import torch
from scipy import sparse

import faster_weathernext_amd as fwn
from faster_weathernext_amd import hip_attn
from gpu_helpers import DEV, MAXTOL, TOL, dev, host, rounded
from oracle import attention as A

pytestmark = pytest.mark.gpu


def _shuffled_mesh(n, k_hop, seed, directed=False):
  """The first n nodes of a shuffled refinement-3 mesh (642 nodes)."""
  mask = fwn.mesh_mask(3, k_hop)[0]
  rng = np.random.default_rng(seed)
  p = rng.permutation(mask.shape[0])[:n]
  m = mask[p][:, p].toarray()
  if directed:
    drop = rng.random((n, n)) < 0.3
    np.fill_diagonal(drop, False)
    m &= ~drop
  return sparse.csr_matrix(m)


CASES = {"bf16": (torch.bfloat16, "native"), "f32": (torch.float32, "native"), "bf16x3": (torch.float32, "bf16x3")}


def _check(got, ref, case, what):
  """The bars of the other parity tests: 1e-5 (float32), 5e-3 (bf16) and, with split products
  (16 bits per operand, at most six of them in a chain of two contractions), 3e-5."""
  dtype = CASES[case][0]
  rr, mr = A.rel_rms(got, ref), A.max_rel_err(got, ref)
  assert rr <= (3e-5 if case == "bf16x3" else TOL[dtype]), (what, rr)
  assert mr <= (1e-4 if case == "bf16x3" else MAXTOL[dtype]), (what, mr)


def _run(case, q, k, v, do, tiles, tiles_t, scale, packed=False):
  dtype, precision = CASES[case]
  if packed:
    qkv = dev(np.stack([q, k, v], 2), dtype, True)
    out = fwn.tiled_flash_attention_qkv(qkv, tiles, scale=scale, tiles_t=tiles_t, precision=precision)
    grads = torch.autograd.grad(out, qkv, dev(do, dtype))[0].unbind(2)
  else:
    x = [dev(t, dtype, True) for t in (q, k, v)]
    out = fwn.tiled_flash_attention(*x, tiles, scale=scale, tiles_t=tiles_t, precision=precision)
    grads = torch.autograd.grad(out, x, dev(do, dtype))
  return [host(t) for t in (out, *grads)]


@pytest.mark.parametrize("case", sorted(CASES))
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("n,directed,cap,exchange,packed", [
    (642, False, None, True, False), (257, False, None, True, True), (384, True, None, True, False),
    (515, False, 1, True, False), (642, True, 2, False, True), (130, False, None, False, False)])
def test_matches_dense_reference(case, d, n, directed, cap, exchange, packed, monkeypatch):
  print(f"node order {case} d={d} n={n} directed={directed} cap={cap} exchange={exchange} packed={packed}", flush=True)
  monkeypatch.setattr(hip_attn, "DS_EXCHANGE", exchange)
  monkeypatch.setattr(hip_attn, "LAID_OUT_GAIN", 10.0)  # the layout applies whatever it saves
  mask = _shuffled_mesh(n, 3, n + d, directed)
  tiles = fwn.TileList.from_mask(mask, device=DEV, max_item_tiles=cap)
  tiles_t = fwn.TileList.from_mask(mask.T.tocsr(), device=DEV, max_item_tiles=cap) if directed else None
  assert tiles._layout is not None
  rng = np.random.default_rng(n)
  b, h = 2, 2
  q, k, v, do = (rounded(rng.standard_normal((b, n, h, d)), CASES[case][0]) for _ in range(4))
  scale = d ** -0.5
  got = _run(case, q, k, v, do, tiles, tiles_t, scale, packed)
  dense = mask.toarray()
  refs = [A.dense_attention(q, k, v, dense, scale), *A.dense_grads(q, k, v, do, dense, scale)]
  for name, g, r in zip(("out", "dq", "dk", "dv"), got, refs):
    _check(g, r, case, name)


@pytest.mark.parametrize("case", sorted(CASES))
def test_lse_and_empty_rows(case):
  """The saved log-sum-exp is in node order, and rows without a valid key give zeros (their lse
  stays the empty row's) wherever the order puts them."""
  dtype, precision = CASES[case]
  n, h, d = 515, 1, 64
  mask = _shuffled_mesh(n, 2, 7).tolil()
  empty = [0, 127, 128, 300, 514]
  for r in empty:
    mask[r, :] = False
    mask[:, r] = False
  mask = mask.tocsr()
  tiles = fwn.TileList.from_mask(mask, device=DEV)
  assert tiles._layout is not None
  rng = np.random.default_rng(3)
  q, k, v = (dev(rounded(rng.standard_normal((1, n, h, d)), dtype), dtype) for _ in range(3))
  out, lse = fwn.attention_forward(q, k, v, tiles, d ** -0.5, precision=precision)
  plain = tiles._layout
  tiles._layout = None
  out0, lse0 = fwn.attention_forward(q, k, v, tiles, d ** -0.5, precision=precision)
  tiles._layout = plain
  assert not host(out)[0, empty].any()
  _check(host(out), host(out0), case, "out")
  keep = np.setdiff1d(np.arange(n), empty)
  # One list's statistics against the other's: sums of the same float32 terms in another order.
  np.testing.assert_allclose(host(lse)[..., keep], host(lse0)[..., keep], rtol=0, atol=1e-5)
  assert np.array_equal(host(lse)[..., empty], host(lse0)[..., empty])


def test_order_is_kept_only_where_it_pays():
  """A mesh in mesh order takes an order of its own; a mask without locality, a single block and a
  list whose order saves nothing keep the given one."""
  assert fwn.TileList.from_mask(fwn.mesh_mask(4, 4)[0], device=DEV)._layout is not None
  rng = np.random.default_rng(0)
  m = fwn.mesh_mask(2, 2)[0]
  assert fwn.TileList.from_mask(m[:128][:, :128].tocsr(), device=DEV)._layout is None
  dense = sparse.csr_matrix(np.ones((300, 300), bool))
  assert fwn.TileList.from_mask(dense, device=DEV)._layout is None
  noise = (sparse.random(600, 600, 0.2, random_state=1) + sparse.identity(600)).astype(bool).tocsr()
  assert fwn.TileList.from_mask(noise, device=DEV)._layout is None


@pytest.mark.parametrize("case", sorted(CASES))
@pytest.mark.parametrize("directed,exchange", [(False, True), (True, True), (False, False)])
def test_given_exchange_under_a_laid_out_forward(case, directed, exchange, monkeypatch):
  """A few rows and columns that reach everywhere spoil the order for whole groups: the forward walks the
  list laid out for it and the backward the given pair, on the same statistics."""
  print(f"mixed lists {case} directed={directed} exchange={exchange}", flush=True)
  monkeypatch.setattr(hip_attn, "DS_EXCHANGE", exchange)
  mesh, _, _, perm = fwn.mesh_mask(3, 1, reorder=True)
  mask, n = mesh[perm][:, perm].tolil(), mesh.shape[0]
  for r in np.random.default_rng(0).choice(n, 6 if directed else 3, replace=False):
    mask[r, :] = True
    mask[:, r] = True
  mask = mask.tocoo()
  keep = (mask.row >= mask.col) | ((mask.row + mask.col) % 3 > 0) | (not directed)
  mask = sparse.csr_matrix((mask.data[keep], (mask.row[keep], mask.col[keep])), shape=(n, n))
  assert ((mask != mask.T).nnz > n) == directed
  tiles = fwn.TileList.from_mask(mask, device=DEV)
  tiles_t = fwn.TileList.from_mask(mask.T.tocsr(), device=DEV) if directed else None
  assert tiles.launch_list() is not tiles
  assert tiles.exchange_lists(tiles_t or tiles, case)[:2] == (tiles, tiles_t or tiles)
  rng = np.random.default_rng(n)
  b, h, d = 2, 2, 64
  q, k, v, do = (rounded(rng.standard_normal((b, n, h, d)), CASES[case][0]) for _ in range(4))
  got = _run(case, q, k, v, do, tiles, tiles_t, d ** -0.5)
  dense = mask.toarray()
  refs = [A.dense_attention(q, k, v, dense, d ** -0.5), *A.dense_grads(q, k, v, do, dense, d ** -0.5)]
  for name, g, r in zip(("out", "dq", "dk", "dv"), got, refs):
    _check(g, r, case, name)
