"""dK/dV schedules of calls with few jobs: blocks cut into runs of tiles so that the last round fills
the chip (``_PackedList._filled``)."""
import ctypes

import numpy as np
import pytest
import torch

import faster_weathernext_amd as fwn
from faster_weathernext_amd import _native as nat
from faster_weathernext_amd import hip_attn


def _list(refinement, k_hop, device):
  mask, _, _, perm = fwn.mesh_mask(refinement, k_hop, reorder=True)
  return fwn.TileList.from_mask(mask, perm, device=device)


def _desc(pairs, head_dim=128, dtype=nat.F32, precision=nat.PREC_NATIVE, n=2562):
  return nat.AttnDesc(1, n, pairs, head_dim, dtype, 0.1, n * pairs * head_dim, pairs * head_dim, head_dim, 0, 0, 0, precision, 0)


@pytest.mark.parametrize("refinement,k_hop", [(4, 4), (4, 8), (5, 8), (5, 16)])
def test_filled_schedule_covers_every_tile_once(refinement, k_hop):
  layout = hip_attn._Layout.choose(_list(refinement, k_hop, "cpu"))
  tl = layout.packed(layout.arrays, 32, nat.PARTS_PAIRS16)
  n, taken = layout.arrays.n, 0
  for pairs in (1, 2, 3, 4, 5, 8, 12, 13, 24, 50):
    desc = _desc(pairs, n=n)
    plan = hip_attn.order_plan(desc, "kv")
    whole, sch = tl.schedule_for(1, pairs, "kv"), tl._filled(desc)
    for other in (_desc(pairs, dtype=nat.BF16, n=n), _desc(pairs, 64, n=n) if whole.n_items * pairs >= 256 else None):
      if other is not None:
        assert tl._filled(other) is None
        assert tl.struct_for_desc(other, "kv").n_parts == whole.n_parts
    st = tl.struct_for_desc(desc, "kv")
    if sch is None:
      assert st.n_items == whole.n_items
      continue
    taken += 1
    assert st.n_items == sch.n_items and tl.struct_for_desc(desc, "kv") is st and st.n_work >= sch.n_items * pairs
    size = ctypes.c_uint64(0)
    nat.check(nat.lib().fwn_attn_workspace_size(desc, st, ctypes.byref(size)))
    assert tl.workspace_bytes(desc) >= size.value == sch.n_parts * pairs * 128 * (2 * 128 + 2) * 4
    assert sch.makespan(pairs, *plan) < hip_attn.FILL_GAIN * whole.makespan(pairs, *plan)
    items, at = sch.items_host, 0
    for b in range(tl.n_blocks):
      runs = items[items[:, 0] == b]
      edges = [int(tl._tile_ptr[b])] + runs[:, 2].tolist()
      assert runs[:, 1].tolist() == edges[:-1] and edges[-1] == tl._tile_ptr[b + 1]
      assert 1 <= len(runs) <= hip_attn.FILL_PIECES
      if len(runs) == 1:
        assert runs[0, 3] == -1
      else:
        assert np.diff(edges).min() >= 2
        assert runs[:, 3].tolist() == list(range(at, at + len(runs)))
        assert [b, at, len(runs)] in sch.split_host.tolist()
        at += len(runs)
    assert at == sch.n_parts and np.all(np.diff(items[:, 0]) >= 0)
  assert taken
  assert tl._filled(_desc(-(-hip_attn.FILL_ROUNDS * 256 // tl.n_blocks), n=n)) is None


def test_cut_items_match_the_native_schedule():
  ptr = np.array([0, 3, 3, 20, 21, 29], np.int32)
  for cap in (1, 2, 5, 7, 30):
    counts = np.zeros(3, np.int32)
    lib = nat.lib()
    nat.check(lib.fwn_tiles_schedule_count(5, nat.ptr(ptr), cap, *(nat.ptr(counts[i:]) for i in range(3))))
    items, split = np.zeros((counts[0], 4), np.int32), np.zeros((max(counts[2], 1), 3), np.int32)
    nat.check(lib.fwn_tiles_schedule_fill(5, nat.ptr(ptr), cap, nat.ptr(items), nat.ptr(split)))
    got = hip_attn._cut_items(ptr, np.maximum(-(-np.diff(ptr) // cap), 1))
    assert np.array_equal(got[0], items) and np.array_equal(got[1], split) and got[2] == tuple(counts)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["native", "bf16x3"])
@pytest.mark.parametrize("head_dim", [32, 64, 128])
@pytest.mark.parametrize("exchange", [True, False])
def test_filled_gradients_match_whole_ones(monkeypatch, precision, head_dim, exchange):
  """The same products, float32 sums in another order (up to 20 tiles of 128 terms: a few 2^-24)."""
  if precision == "bf16x3" and not exchange:
    pytest.skip("bf16x3 gradients need the exchange")
  monkeypatch.setattr(hip_attn, "DS_EXCHANGE", exchange)
  tl = _list(4, 8, "cuda")
  b, h, n = 1, 2, tl.n_cols
  g = torch.Generator(device="cuda").manual_seed(head_dim)
  q, k, v, do = (torch.randn(b, n, h, head_dim, device="cuda", generator=g) for _ in range(4))
  grads, parts = [], []
  for rounds in (hip_attn.FILL_ROUNDS, 0):
    monkeypatch.setattr(hip_attn, "FILL_ROUNDS", rounds)
    lst = tl if not grads else _list(4, 8, "cuda")
    leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
    out = fwn.tiled_flash_attention(*leaves, lst, scale=head_dim ** -0.5, precision=precision)
    grads.append(torch.autograd.grad(out, leaves, do))
    kv = lst.exchange_lists(lst, "f32" if precision == "native" else precision)[1]
    prec = nat.PREC_BF16X3 if precision == "bf16x3" else nat.PREC_NATIVE
    parts.append(kv.struct_for_desc(_desc(h, head_dim, precision=prec, n=n), "kv").n_parts)
  assert parts[0] > 0 and parts[1] == 0
  for got, want in zip(*grads):
    assert float((got.double() - want.double()).norm() / want.double().norm()) <= 2e-6
