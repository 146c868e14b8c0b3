"""The locality order of a tile list's nodes and the permuted list (``fwn_tiles_node_order``,
``fwn_tiles_permute_count``, ``fwn_tiles_permute_fill``): the order is a permutation for any mask, the
permuted list is the one built from the permuted mask, and the order shrinks a mesh's list."""
import numpy as np
import pytest
from scipy import sparse

import faster_weathernext_amd as fwn
from faster_weathernext_amd import _native as nat


def _arrays(mask, perm=None):
  return fwn.build_tile_mask(mask, perm=perm)


def _order(n, tp, kb, bits):
  perm = np.full(n, -1, np.int64)
  nat.check(nat.lib().fwn_tiles_node_order(n, nat.ptr(tp), nat.ptr(kb), nat.ptr(bits), nat.ptr(perm)))
  return perm


def _permuted(n, tp, kb, bits, perm):
  new_ptr = np.zeros_like(tp)
  args = (n, nat.ptr(tp), nat.ptr(kb), nat.ptr(bits), nat.ptr(perm))
  nat.check(nat.lib().fwn_tiles_permute_count(*args, nat.ptr(new_ptr)))
  new_kb = np.zeros(new_ptr[-1], np.int32)
  new_bits = np.full((new_ptr[-1], 128, 4), 0xFFFFFFFF, np.uint32)
  nat.check(nat.lib().fwn_tiles_permute_fill(*args, nat.ptr(new_ptr), nat.ptr(new_kb), nat.ptr(new_bits)))
  return new_ptr, new_kb, new_bits


def _masks():
  rng = np.random.default_rng(0)
  shuffle = lambda m: m[rng.permutation(m.shape[0])][:, rng.permutation(m.shape[0])]
  yield "mesh", fwn.mesh_mask(3, 3)[0]
  yield "directed", shuffle(fwn.mesh_mask(2, 2)[0])
  yield "empty rows", sparse.csr_matrix(sparse.random(300, 300, 0.002, random_state=1).astype(bool))
  yield "no entries", sparse.csr_matrix((130, 130), dtype=bool)
  yield "dense", sparse.csr_matrix(np.ones((257, 257), bool))
  yield "identity", sparse.identity(513, dtype=bool, format="csr")
  yield "one node", sparse.identity(1, dtype=bool, format="csr")
  yield "two components", sparse.block_diag([np.ones((200, 200)), np.ones((184, 184))]).astype(bool).tocsr()


@pytest.mark.parametrize("name", [n for n, _ in _masks()])
def test_order_is_a_permutation_and_permuted_list_matches(name):
  mask = dict(_masks())[name].tocsr()
  n = mask.shape[0]
  tp, kb, bits = _arrays(mask)
  perm = _order(n, tp, kb, bits)
  assert np.array_equal(np.sort(perm), np.arange(n))
  for p in (perm, np.random.default_rng(1).permutation(n), np.arange(n)):
    p = np.asarray(p, np.int64)
    for got, want in zip(_permuted(n, tp, kb, bits, p), _arrays(mask, p)):
      assert np.array_equal(got, want)


def test_order_is_deterministic_and_compact_on_a_shuffled_mesh():
  """The order recovers a shuffled mesh's locality: no more tiles than Hilbert order of the nodes'
  positions needs, and the same order whenever it is computed."""
  mask, _, _, hilbert = fwn.mesh_mask(4, 4, reorder=True)
  n = mask.shape[0]
  p = np.random.default_rng(2).permutation(n)
  tp, kb, bits = _arrays(mask[p][:, p].tocsr())
  perm = _order(n, tp, kb, bits)
  assert np.array_equal(perm, _order(n, tp, kb, bits))
  tiles = _permuted(n, tp, kb, bits, perm)[0][-1]
  assert tiles <= _arrays(mask, hilbert)[0][-1] < tp[-1]


def test_bad_arguments_are_refused():
  tp, kb, bits = _arrays(fwn.mesh_mask(2, 1)[0])
  n, L = 162, nat.lib()
  perm, ptr = np.arange(n), np.zeros_like(tp)
  good = (n, nat.ptr(tp), nat.ptr(kb), nat.ptr(bits))
  assert L.fwn_tiles_node_order(0, *good[1:], nat.ptr(perm)) == nat.ERR_INVALID_ARG
  assert L.fwn_tiles_node_order(*good, None) == nat.ERR_INVALID_ARG
  assert L.fwn_tiles_node_order(n, nat.ptr(tp), None, nat.ptr(bits), nat.ptr(perm)) == nat.ERR_INVALID_ARG
  twice = perm.copy()
  twice[3] = twice[4]
  for bad in (twice, perm + 1, perm - 1):
    assert L.fwn_tiles_permute_count(*good, nat.ptr(bad), nat.ptr(ptr)) == nat.ERR_INVALID_ARG
  col = kb.copy()
  col[0] = 99
  assert L.fwn_tiles_node_order(n, nat.ptr(tp), nat.ptr(col), nat.ptr(bits), nat.ptr(perm)) == nat.ERR_TILES
  # a pointer array of another order's list
  assert L.fwn_tiles_permute_fill(*good, nat.ptr(perm), nat.ptr(np.array([0, 1, 2], np.int32)), nat.ptr(np.zeros(2, np.int32)),
                                  nat.ptr(np.zeros((2, 128, 4), np.uint32))) == nat.ERR_INVALID_ARG


def test_launchers_check_the_node_table():
  """Refused on the host, before any launch: unknown flags, a null table, too many rows."""
  F = 1 << 20
  size = np.zeros(1, np.uint64)
  desc = nat.AttnDesc(1, 256, 1, 32, nat.F32, 1.0, 32 * 256, 32, 32)
  def status(flags, node, d=desc, blocks=2):
    t = nat.Tiles(blocks, 1, F, F, F, F, blocks, 0, 0, 0, F, None, None, None, 0, flags, node)
    return nat.lib().fwn_attn_workspace_size(d, t, nat.ptr(size))
  assert status(0, None) == nat.OK and status(nat.TILES_NODES, F) == nat.OK
  assert status(2, F) == nat.ERR_INVALID_ARG
  assert status(nat.TILES_NODES, None) == nat.ERR_TILES
  n = 1 << 24
  big = nat.AttnDesc(1, n, 1, 32, nat.BF16, 1.0, 32 * n, 32, 32)
  assert status(0, None, big, n // 128) == nat.OK
  assert status(nat.TILES_NODES, F, big, n // 128) == nat.ERR_INVALID_ARG
