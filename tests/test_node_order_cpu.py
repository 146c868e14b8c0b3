"""The locality order of a tile list's nodes, the permuted and the packed lists and the dS unit
numbering of packed pairs (``fwn_tiles_node_order``, ``fwn_tiles_permute_*``, ``fwn_tiles_compact_*``,
``fwn_tiles_unit_map``): the order is a permutation for any mask, the permuted list is the one built
from the permuted mask, a packed list holds the mask's entries, and every dS unit has one number."""
import collections
import ctypes
import gc
import threading
import time
import weakref

import numpy as np
import pytest
import torch
from scipy import sparse

import faster_weathernext_amd as fwn
from faster_weathernext_amd import _native as nat
from faster_weathernext_amd import hip_attn


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


def _band(n, width):
  off = range(-width, width + 1)
  return sparse.diags([np.ones(n - abs(k)) for k in off], list(off)).astype(bool).tocsr()


@pytest.mark.parametrize("n,width,own", [(40962, 1, True), (40962, 16, True), (100000, 1, False)])
def test_order_of_a_long_path_takes_seconds(n, width, own):
  """A mask of long paths has tens of thousands of breadth-first levels: the searches cost what their
  fronts do (a scan of the list, or a start of threads, per level took 70 s and more for the first
  of these; 0.7 s now), and one that takes too many steps leaves the nodes in their own order."""
  lists = _arrays(_band(n, width))
  start = time.perf_counter()
  perm = _order(n, *lists)
  assert time.perf_counter() - start < 15
  assert np.array_equal(np.sort(perm), np.arange(n))
  assert np.array_equal(perm, np.arange(n)) == (not own)


def _compact(n, tp, kb, bits, group, parts=0, window=0):
  new_ptr = np.zeros_like(tp)
  args = (n, nat.ptr(tp), nat.ptr(kb), nat.ptr(bits), group)
  nat.check(nat.lib().fwn_tiles_compact_count(*args, nat.ptr(new_ptr)))
  args = (*args, parts, window)
  cols = np.full((new_ptr[-1], 128), -7, np.int32)
  new_bits = np.full((new_ptr[-1], 128, 4), 0xFFFFFFFF, np.uint32)
  nat.check(nat.lib().fwn_tiles_compact_fill(*args, nat.ptr(new_ptr), nat.ptr(cols), nat.ptr(new_bits)))
  return new_ptr, cols, new_bits


def _bools(bits):
  return np.unpackbits(bits.view(np.uint8), axis=-1, bitorder="little").reshape(len(bits), 128, 128).astype(bool)


@pytest.mark.parametrize("group,parts,window", [(1, 0, 0), (16, 0, 0), (16, 0, 2), (32, 0, 1), (32, 1, 0)])
@pytest.mark.parametrize("name", [n for n, _ in _masks()])
def test_packed_list_holds_the_mask(name, group, parts, window):
  """Unpacked through its columns, a packed list is the mask; every column group it holds is live
  in the block, whole and once, in as few tiles as hold them."""
  mask = dict(_masks())[name].tocsr()
  n = mask.shape[0]
  ptr, cols, bits = _compact(n, *_arrays(mask), group, parts, window)
  dense, got = mask.toarray(), np.zeros((n, n + 1), bool)
  b = _bools(bits)
  for blk in range(len(ptr) - 1):
    r0, r1 = 128 * blk, min(n, 128 * blk + 128)
    c = cols[ptr[blk]:ptr[blk + 1]].reshape(-1, group)
    c = c[c[:, 0] < n]
    assert np.all(c[:, 0] % group == 0) and np.array_equal(c, np.minimum(c[:, :1] + np.arange(group), n))
    want = np.unique(np.nonzero(dense[r0:r1].any(0))[0] // group)
    assert np.array_equal(np.sort(c[:, 0] // group), want)
    assert ptr[blk + 1] - ptr[blk] == -(-len(want) * group // 128)
    for t in range(ptr[blk], ptr[blk + 1]):
      assert not b[t][:, cols[t] == n].any() and not b[t][r1 - r0:].any()
      got[r0:r1, cols[t]] |= b[t][:r1 - r0]
  assert np.array_equal(got[:, :n], dense)


def test_packed_list_balances_the_waves():
  """Per tile, the part of a workgroup with the most live runs has at most 15% more than the mean of
  its four parts, over a mesh's blocks (36 to 70% more when the runs are packed in ascending order)."""
  mask, _, _, _ = fwn.mesh_mask(5, 8)
  n = mask.shape[0]
  tp, kb, bits = _arrays(mask)
  arrays = _permuted(n, tp, kb, bits, _order(n, tp, kb, bits))
  for group, parts in ((16, 0), (32, 1)):
    b = _bools(_compact(n, *arrays, group, parts)[2])
    rows = 32 if parts == 0 else 16
    live = b.reshape(len(b), 128 // rows, rows, 128 // group, group).any((2, 4)).sum(2)
    load = live if parts == 0 else live[:, :4] + live[:, 4:]
    assert load.max(1).sum() <= 1.15 * load.mean(1).sum(), (group, load.max(1).sum() / load.mean(1).sum())


def _unit_map(n, f, t, unit_keys):
  (ptr, cols, bits), (ptr_t, cols_t, bits_t) = f, t
  ubase, tmap, units = np.zeros(max(len(cols), 1), np.int32), np.full((max(len(cols_t), 1), 9, 4), -9, np.int32), np.zeros(1, np.int64)
  status = nat.lib().fwn_tiles_unit_map(n, nat.ptr(ptr), nat.ptr(bits), nat.ptr(cols), nat.ptr(ptr_t), nat.ptr(bits_t),
                                        nat.ptr(cols_t), unit_keys, nat.ptr(ubase), nat.ptr(tmap), nat.ptr(units))
  return status, ubase, tmap, int(units[0])


@pytest.mark.parametrize("unit_keys", [16, 32])
@pytest.mark.parametrize("name", [n for n, _ in _masks()])
def test_unit_map_numbers_every_unit_once(name, unit_keys):
  """The number dQ gives a unit (its tile's first plus the rank of its bit) is the one dK/dV's table
  holds for the same 32 queries and keys; the numbers are 0 .. n_units - 1."""
  mask = dict(_masks())[name].tocsr()
  n = mask.shape[0]
  f, t = _compact(n, *_arrays(mask), unit_keys), _compact(n, *_arrays(mask.T.tocsr()), 32)
  status, ubase, tmap, units = _unit_map(n, f, t, unit_keys)
  assert status == nat.OK
  want = {}
  (ptr, cols, bits), (ptr_t, cols_t, bits_t) = f, t
  b = _bools(bits)
  for blk in range(len(ptr) - 1):
    for tile in range(ptr[blk], ptr[blk + 1]):
      u = ubase[tile]
      for g in range(4):
        for c0 in range(0, 128, unit_keys):
          if b[tile, 32 * g:32 * g + 32, c0:c0 + unit_keys].any():
            want[4 * blk + g, cols[tile, c0] // unit_keys] = u
            u += 1
  assert sorted(want.values()) == list(range(units))
  b, seen = _bools(bits_t), set()
  for blk in range(len(ptr_t) - 1):
    for tile in range(ptr_t[blk], ptr_t[blk + 1]):
      for kg in range(8):
        for c in range(4):
          r0 = 16 * kg // unit_keys * unit_keys
          live = b[tile, r0:r0 + unit_keys, 32 * c:32 * c + 32].any()
          own = b[tile, 16 * kg:16 * kg + 16, 32 * c:32 * c + 32].any()
          assert bool(tmap[tile, 8, 0] >> (8 * c + kg) & 1) == own
          unit = tmap[tile, kg, c]
          assert (unit >= 0) == live
          if live:
            assert unit == want[cols_t[tile, 32 * c] // 32, (128 * blk + r0) // unit_keys]
            seen.add(int(unit))
  assert seen == set(range(units))


def test_unit_map_refuses_lists_that_are_not_transposes():
  m = sparse.identity(300, dtype=bool, format="lil")
  m[3, 290] = True
  m = m.tocsr()
  n = m.shape[0]
  f, wrong = _compact(n, *_arrays(m), 16), _compact(n, *_arrays(m), 32)
  assert _unit_map(n, f, wrong, 16)[0] == nat.ERR_TILES
  assert _unit_map(n, f, _compact(n, *_arrays(m.T.tocsr()), 32), 16)[0] == nat.OK
  assert _unit_map(n, _compact(n, *_arrays(m), 1), _compact(n, *_arrays(m.T.tocsr()), 32), 16)[0] == nat.ERR_TILES


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
  for group in (0, 2, 64):
    assert L.fwn_tiles_compact_count(*good, group, nat.ptr(ptr)) == nat.ERR_INVALID_ARG
  assert L.fwn_tiles_compact_fill(*good, 1, 0, 0, nat.ptr(np.array([0, 1, 1], np.int32)), nat.ptr(np.zeros(128, np.int32)),
                                  nat.ptr(np.zeros((1, 128, 4), np.uint32))) == nat.ERR_INVALID_ARG
  # a pointer array of another order's list
  assert L.fwn_tiles_permute_fill(*good, nat.ptr(perm), nat.ptr(np.array([0, 1, 2], np.int32)), nat.ptr(np.zeros(2, np.int32)),
                                  nat.ptr(np.zeros((2, 128, 4), np.uint32))) == nat.ERR_INVALID_ARG


def test_launchers_check_the_node_table():
  """Refused on the host, before any launch: unknown flags, a null table, too many rows."""
  F = 1 << 20
  size = np.zeros(1, np.uint64)
  desc = nat.AttnDesc(1, 256, 1, 32, nat.F32, 1.0, 32 * 256, 32, 32)
  def status(flags, node, d=desc, blocks=2):
    t = nat.Tiles(blocks, 1, F, F, F, F, blocks, 0, 0, 0, F, None, None, None, 0, flags, node, node)
    return nat.lib().fwn_attn_workspace_size(d, t, nat.ptr(size))
  assert status(0, None) == nat.OK and status(nat.TILES_NODES, F) == nat.OK
  assert status(2, F) == nat.ERR_INVALID_ARG
  assert status(nat.TILES_NODES, None) == nat.ERR_TILES
  n = 1 << 24
  big = nat.AttnDesc(1, n, 1, 32, nat.BF16, 1.0, 32 * n, 32, 32)
  assert status(0, None, big, n // 128) == nat.OK
  assert status(nat.TILES_NODES, F, big, n // 128) == nat.ERR_INVALID_ARG


def test_an_exchange_keeps_no_list_alive():
  """The exchange kept by a list refers to the program's lists weakly: a transposed list goes when the
  program drops it, though the list it was used with lives on."""
  mask = sparse.random(300, 300, 0.05, format="csr", random_state=np.random.RandomState(1)).astype(bool)
  tl, tlt = (fwn.TileList.from_mask(m, device="cpu") for m in (mask, mask.T.tocsr()))
  sym = fwn.TileList.from_mask((mask + mask.T).tocsr(), device="cpu")
  for products in ("bf16", "f32", "bf16x3"):
    assert tl.exchange_lists(tlt, products)[:2] == (tl, tlt)
    assert sym.exchange_lists(sym, products)[:2] == (sym, sym)
  refs = [weakref.ref(t) for t in (tl, tlt, sym)]
  del tlt
  gc.collect()
  assert refs[1]() is None and not len(tl._exchanges)
  del tl, sym
  gc.collect()
  assert refs[0]() is None and refs[2]() is None


@pytest.mark.parametrize("name", ["mesh", "hilbert", "global rows", "directed global rows", "random", "coarse"])
def test_exchange_lists_are_no_costlier_than_the_given_ones(name):
  """The lists of the dS exchange are weighed by themselves: where a few rows and columns that reach
  everywhere spoil the order, or the mask has no locality, the forward's list pays and the given two are
  walked in the backward; in any case neither their tiles, nor their cost, nor the dS buffer grow."""
  coarse, wide = name == "coarse", "global" in name
  mask, _, _, perm = fwn.mesh_mask(2 if coarse else 4, 2 if coarse else 4, reorder=name not in ("mesh", "random"))
  n = mask.shape[0]
  if wide:
    mask = mask.tolil()
    for r in np.random.default_rng(0).choice(n, 6, replace=False):
      mask[r, :] = True
      mask[:, r] = True
    if name != "global rows":
      mask[5, 2000] = True
      mask[2000, 5] = False
    mask = mask.tocsr()
  elif name == "random":
    mask = (sparse.random(n, n, 0.01, random_state=1) + sparse.identity(n)).astype(bool).tocsr()
    mask = (mask + mask.T).tocsr()
  tl = fwn.TileList.from_mask(mask, perm, device="cpu")
  tlt = fwn.TileList.from_mask(mask.T.tocsr(), perm, device="cpu") if "directed" in name else tl
  tl._layout = hip_attn._Layout.choose(tl)  # as a list on the GPU has it
  assert tl._layout is not None
  kept = {}
  for products, unit_keys in hip_attn.DS_UNIT_KEYS.items():
    dq, kv, dmap = tl.exchange_lists(tlt, products)
    given = tl.ds_map(tlt, unit_keys)
    kept[products] = (dq, kv, dmap) == (tl, tlt, given)
    assert kept[products] or (dq is not tl and kv is not tlt and dmap is not given)
    gain = 0.95 if products == "bf16" else 1.0
    for laid_out, own in ((dq.n_tiles, tl.n_tiles), (dq.cost, tl.cost), (kv.n_tiles, tlt.n_tiles), (kv.cost, tlt.cost),
                          (dmap.n_units, given.n_units)):
      assert laid_out == own if kept[products] else laid_out <= gain * own
    assert dmap.struct.table == dq.struct.flags == kv.struct.flags == (0 if kept[products] else 1)
  assert kept["bf16"] == (name not in ("mesh", "hilbert"))
  assert kept["f32"] == kept["bf16x3"] == wide


def test_a_list_in_the_making_holds_up_no_other_call(monkeypatch):
  """Lists of array triples are built outside the cache's lock: while one is being made, calls with
  other arrays go on, and two threads that make the same one use the same."""
  monkeypatch.setattr(hip_attn, "_cache", collections.OrderedDict())
  first, second = (_arrays(fwn.mesh_mask(2, k)[0]) for k in (1, 2))
  cpu = torch.device("cpu")
  ready = hip_attn._as_tiles(second, 162, cpu)
  started, go = threading.Semaphore(0), threading.Event()

  def make(*args):
    started.release()
    assert go.wait(30)
    return fwn.TileList(*args)

  monkeypatch.setattr(hip_attn, "TileList", type("Slow", (), {"__new__": staticmethod(lambda cls, *a: make(*a))}))
  made = []
  threads = [threading.Thread(target=lambda: made.append(hip_attn._as_tiles(first, 162, cpu))) for _ in range(2)]
  for t in threads:
    t.start()
  try:
    assert started.acquire(timeout=30)
    other = threading.Thread(target=lambda: made.append(hip_attn._as_tiles(second, 162, cpu)))
    other.start()
    other.join(30)
    assert made == [ready]
    assert started.acquire(timeout=30)
  finally:
    go.set()
    for t in threads:
      t.join()
  assert len(made) == 3 and made[1] is made[2] is hip_attn._as_tiles(first, 162, cpu)


def test_an_order_that_spreads_the_mask_is_not_laid_out(monkeypatch):
  """A list in its own node order takes 2 KB of host memory a tile: where it has more than PERMUTED_TILES
  times the given list's, its tiles are never filled and the given order is packed, or kept."""
  mask, _, _, perm = fwn.mesh_mask(4, 4, reorder=True)
  tl = fwn.TileList.from_mask(mask, perm, device="cpu")
  n, given = mask.shape[0], hip_attn._Arrays(tl.n_cols, tl._tile_ptr, tl._tile_col, tl._tile_bits)
  shuffle = np.random.default_rng(0).permutation(n)
  assert _arrays(mask[perm][:, perm][shuffle][:, shuffle].tocsr())[0][-1] > 2 * tl.n_tiles

  def spread(n, ptr, col, bits, out):
    np.ctypeslib.as_array((ctypes.c_int64 * n).from_address(out))[:] = shuffle
    return nat.OK

  class Lib:
    fwn_tiles_node_order = staticmethod(spread)

    def __getattr__(self, name):
      assert name != "fwn_tiles_permute_fill"
      return getattr(real, name)

  real = nat.lib()
  monkeypatch.setattr(nat, "lib", Lib)
  assert given.permuted(shuffle) is None
  layout = hip_attn._Layout.choose(tl)
  assert np.array_equal(layout.perm, np.arange(n)) and layout.forward.cost <= 0.95 * tl.cost


def test_lists_past_the_node_table_keep_the_given_ones(monkeypatch):
  """The launchers refuse lists with node tables of 2^22 tiles and more, so a mask that would have
  them is walked as given, and so is the exchange where only its lists would."""
  F = 1 << 20
  size, desc = np.zeros(1, np.uint64), nat.AttnDesc(1, 256, 1, 32, nat.F32, 1.0, 32 * 256, 32, 32)
  status = lambda tiles: nat.lib().fwn_attn_workspace_size(
      desc, nat.Tiles(2, tiles, F, F, F, F, 2, 0, 0, 0, F, None, None, None, 0, nat.TILES_NODES, F, F), nat.ptr(size))
  assert status((1 << 22) - 1) == nat.OK and status(1 << 22) == nat.ERR_INVALID_ARG
  mask, _, _, perm = fwn.mesh_mask(4, 4, reorder=True)
  tl = fwn.TileList.from_mask(mask, perm, device="cpu")
  layout = hip_attn._Layout.choose(tl)
  tiles = [layout.forward.n_tiles, *(hip_attn._Packed(layout.arrays, g, p).n_tiles for g, p in ((16, 0), (32, 1)))]
  assert tiles == sorted(tiles) and tiles[0] < tiles[1]
  for most, forward in ((tiles[0], False), (tiles[0] + 1, True)):
    monkeypatch.setattr(nat, "TILES_NODES_MAX", most)
    tl._layout = hip_attn._Layout.choose(tl)
    assert (tl._layout is not None) == forward
    assert tl.exchange_lists(tl, "bf16")[:2] == tl.exchange_lists(tl, "f32")[:2] == (tl, tl)


def test_launchers_check_the_unit_table():
  """Refused on the host: a unit table that the kernels' 16-byte copies cannot read, or one that does not
  go with the list. (The tensors are null, so that no call gets further than their check.)"""
  F = 1 << 20
  desc = nat.AttnDesc(1, 256, 1, 32, nat.BF16, 1.0, 32 * 256, 32, 32)
  def message(flags, table, tmap):
    t = nat.Tiles(2, 1, F, F, F, F, 2, 0, 0, 0, F, None, None, None, 0, flags, F, F)
    m = nat.DsMap(4, F, tmap, 16, table)
    assert nat.lib().fwn_attn_bwd_dkv_ds_launch(desc, *[None] * 6, t, m, None, None, F, 1 << 20, None, 0, None) == nat.ERR_INVALID_ARG
    return nat.lib().fwn_last_error().decode()
  assert "q is null" in message(nat.TILES_NODES, 1, F) and "q is null" in message(0, 0, F + 8)
  for offset in (4, 8, 12):
    assert "tmap" in message(nat.TILES_NODES, 1, F + offset)
  assert "table" in message(nat.TILES_NODES, 0, F) and "table" in message(0, 1, F)
