// A locality order of a tile list's nodes, computed from its mask alone, the list of the permuted
// mask, the same with each block's live columns packed together, and the dS unit numbering of such
// lists.
//
// The kernels compute whole 32 x 32 groups of a live tile, so their work depends on how compactly
// each node's neighbourhood lies in the node numbering. The mask is the only description of the
// geometry the op gets (the reference orders nodes along a Hilbert curve from their latitudes and
// longitudes before building its list, patch.py:208-214), so the order is built from it: breadth-first
// distances to a few far-apart landmark nodes, averaged over each node's neighbourhood (which
// turns the coarse hop counts into smooth coordinates), then recursive bisection along the
// principal axis of the coordinates, in runs of whole 128-row blocks. On the refinement-6
// icosahedral mesh this leaves (live 32 x 32 groups / 16) 1,676 of 4,341 with the 8-hop mask in mesh
// order (Hilbert order: 2,151), 3,955 of 7,576 with 16 hops (4,764) and 11,190 of 16,545 with 32
// (12,528), within 1% of bisecting the nodes' true positions.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <new>
#include <vector>

#include "fwn_attn.h"
#include "fwn_internal.h"
#include "host_parallel.h"

namespace {

using fwn::parallel_for;

constexpr int32_t kWords = FWN_BLOCK / 32;
constexpr int64_t kTileWords = (int64_t)FWN_BLOCK * kWords;
constexpr int kLandmarks = 6;
constexpr int kSmooth = 3;      // neighbourhood averages of the distances
constexpr int kDims = 8;        // coordinates per node (kLandmarks, padded for the vector units)
constexpr int32_t kLeaf = 16;   // nodes of a bisection leaf: the finest width the kernels skip
constexpr int kAxisSamples = 512;
constexpr int64_t kSerialVisits = 1 << 14;
// Rows looked at over all searches of a list: meshes take 2 to 17 per row of a tile. A list that takes
// more than these (a path of 10^5 nodes, a shuffled band) is left in its own order: 40,962 nodes in a
// row take 0.7 s, the searches stop after about 2 s (5 s for lists of 10^5 tiles).
constexpr int64_t kVisitsPerRow = 24, kVisits = INT64_C(1) << 25;

struct List {
  int32_t n, n_blocks;
  const int32_t* ptr;
  const int32_t* col;
  const uint32_t* bits;
};

// The list's tiles by column block, and the rows of each tile that hold an entry.
struct Columns {
  std::vector<int32_t> ptr, tile;  // tiles of column block kb: tile[ptr[kb]] .. tile[ptr[kb + 1]]
  std::vector<int32_t> blk;        // row block of each tile
  std::vector<uint32_t> rows;      // [n_tiles][kWords], rows past the last node clear

  explicit Columns(const List& m) : ptr(m.n_blocks + 1, 0), tile(m.ptr[m.n_blocks]), blk(tile.size()), rows(tile.size() * kWords) {
    for (size_t t = 0; t < tile.size(); ++t) ++ptr[m.col[t] + 1];
    for (int32_t k = 0; k < m.n_blocks; ++k) ptr[k + 1] += ptr[k];
    std::vector<int32_t> at(ptr.begin(), ptr.end() - 1);
    for (int32_t b = 0; b < m.n_blocks; ++b)
      for (int32_t t = m.ptr[b]; t < m.ptr[b + 1]; ++t) {
        tile[at[m.col[t]]++] = t;
        blk[t] = b;
      }
    parallel_for((int64_t)tile.size(), 256, [&](int64_t begin, int64_t end) {
      for (int64_t t = begin; t < end; ++t) {
        const uint32_t* w = m.bits + t * kTileWords;
        const int32_t last = std::min(FWN_BLOCK, m.n - blk[t] * FWN_BLOCK);
        for (int32_t r = 0; r < last; ++r, w += kWords)
          if (w[0] | w[1] | w[2] | w[3]) rows[t * kWords + r / 32] |= 1u << (r % 32);
      }
    });
  }
};

// Breadth-first distances from `src`: a node is one step further than the nearest node its row
// of the mask holds. Nodes not reached get the largest distance plus one. Each level reads the
// tiles whose column block has a node of the last level, and of those the rows with an entry that
// are not reached yet: its cost follows the front, not the list, as a mask of long paths has
// thousands of levels. `visits` counts the rows and tiles looked at; false when it passes `most`.
bool distances(const List& m, const Columns& cols, int32_t src, int64_t most, int64_t& visits, std::vector<int32_t>& dist) {
  struct Rows {
    uint32_t w[kWords] = {};
    bool any() const { return w[0] | w[1] | w[2] | w[3]; }
    void set(int32_t r) { w[r / 32] |= 1u << (r % 32); }
  };
  std::vector<Rows> front(m.n_blocks), next(m.n_blocks), left(m.n_blocks);  // left: rows not reached
  std::vector<std::vector<int32_t>> todo(m.n_blocks);                       // tiles of a level by row block
  std::vector<int32_t> active{src / FWN_BLOCK}, blocks;
  for (int32_t i = 0; i < m.n; ++i) left[i / FWN_BLOCK].set(i % FWN_BLOCK);
  dist.assign(m.n, -1);
  dist[src] = 0;
  front[active[0]].set(src % FWN_BLOCK);
  left[active[0]].w[src % FWN_BLOCK / 32] &= ~(1u << (src % 32));
  int32_t level = 0;
  while (!active.empty()) {
    ++level;
    int64_t count = 0;
    blocks.clear();
    for (int32_t kb : active)
      for (int32_t k = cols.ptr[kb]; k < cols.ptr[kb + 1]; ++k) {
        const int32_t t = cols.tile[k], blk = cols.blk[t];
        int32_t rows = 0;
        for (int32_t q = 0; q < kWords; ++q) rows += __builtin_popcount(cols.rows[(int64_t)t * kWords + q] & left[blk].w[q]);
        count += 1 + rows;
        if (!rows) continue;
        if (todo[blk].empty()) blocks.push_back(blk);
        todo[blk].push_back(t);
      }
    visits += count;
    if (visits > most) return false;
    // Small levels in this thread: starting the others takes longer.
    const int64_t grain = count < kSerialVisits ? std::max<int64_t>(1, (int64_t)blocks.size()) : 4;
    parallel_for((int64_t)blocks.size(), grain, [&](int64_t b, int64_t e) {
      for (int64_t i = b; i < e; ++i) {
        const int32_t blk = blocks[i];
        Rows out;
        for (int32_t t : todo[blk]) {
          const uint32_t* f = front[m.col[t]].w;
          for (int32_t q = 0; q < kWords; ++q)
            for (uint32_t v = cols.rows[(int64_t)t * kWords + q] & left[blk].w[q] & ~out.w[q]; v; v &= v - 1) {
              const int32_t r = 32 * q + __builtin_ctz(v);
              const uint32_t* w = m.bits + t * kTileWords + r * kWords;
              if (!((w[0] & f[0]) | (w[1] & f[1]) | (w[2] & f[2]) | (w[3] & f[3]))) continue;
              dist[blk * FWN_BLOCK + r] = level;
              out.set(r);
            }
        }
        next[blk] = out;
        todo[blk].clear();
      }
    });
    for (int32_t kb : active) front[kb] = Rows();
    active.clear();
    for (int32_t blk : blocks) {
      if (!next[blk].any()) continue;
      front[blk] = next[blk];
      for (int32_t q = 0; q < kWords; ++q) left[blk].w[q] &= ~next[blk].w[q];
      active.push_back(blk);
    }
  }
  for (int32_t i = 0; i < m.n; ++i)
    if (dist[i] < 0) dist[i] = level;
  return true;
}

// One neighbourhood average of the coordinates: each node's are replaced by the mean over the
// nodes its row holds (its own are kept when the row is empty).
void average(const List& m, const std::vector<float>& x, std::vector<float>& y) {
  parallel_for(m.n_blocks, 2, [&](int64_t b, int64_t e) {
    for (int64_t blk = b; blk < e; ++blk) {
      const int32_t r0 = (int32_t)blk * FWN_BLOCK, rows = std::min(FWN_BLOCK, m.n - r0);
      for (int32_t r = 0; r < rows; ++r) {
        float sum[kDims] = {};
        int32_t count = 0;
        for (int32_t t = m.ptr[blk]; t < m.ptr[blk + 1]; ++t) {
          const uint32_t* w = m.bits + t * kTileWords + r * kWords;
          for (int32_t q = 0; q < kWords; ++q) {
            const float* base = &x[((int64_t)m.col[t] * FWN_BLOCK + 32 * q) * kDims];
            for (uint32_t v = w[q]; v; v &= v - 1) {
              const float* p = base + __builtin_ctz(v) * kDims;
              for (int d = 0; d < kDims; ++d) sum[d] += p[d];
              ++count;
            }
          }
        }
        float* o = &y[(int64_t)(r0 + r) * kDims];
        if (count == 0) {
          std::memcpy(o, &x[(int64_t)(r0 + r) * kDims], sizeof(sum));
          continue;
        }
        const float inv = 1.f / (float)count;
        for (int d = 0; d < kDims; ++d) o[d] = sum[d] * inv;
      }
    }
  });
}

// Where a run of m nodes is cut: near its middle, at a whole number of blocks while it spans more
// than one, then at a power of two of leaves (so that 64-, 32- and 16-row groups are compact too).
int32_t cut(int32_t m) {
  int32_t unit = FWN_BLOCK;
  if (m <= FWN_BLOCK)
    for (unit = kLeaf; unit * 4 <= m;) unit *= 2;
  const int32_t k = std::max(unit, (m / 2 + unit / 2) / unit * unit);
  return k < m ? k : unit;
}

struct Key {
  float v;
  int32_t node;
  bool operator<(const Key& o) const { return v < o.v || (v == o.v && node < o.node); }
};

// Recursive bisection of keys[0, m) by their projection on the run's principal axis (power
// iteration on the covariance of a sample, from its axis of largest variance).
void bisect(const std::vector<float>& x, Key* keys, int32_t m) {
  while (m > kLeaf) {
    double mean[kDims] = {}, cov[kDims][kDims] = {};
    const int32_t step = std::max(1, m / kAxisSamples);
    int32_t count = 0;
    for (int32_t i = 0; i < m; i += step, ++count)
      for (int d = 0; d < kDims; ++d) mean[d] += x[(int64_t)keys[i].node * kDims + d];
    for (int d = 0; d < kDims; ++d) mean[d] /= count;
    for (int32_t i = 0; i < m; i += step) {
      double c[kDims];
      for (int d = 0; d < kDims; ++d) c[d] = x[(int64_t)keys[i].node * kDims + d] - mean[d];
      for (int d = 0; d < kDims; ++d)
        for (int f = 0; f < kDims; ++f) cov[d][f] += c[d] * c[f];
    }
    int top = 0;
    for (int d = 1; d < kDims; ++d)
      if (cov[d][d] > cov[top][top]) top = d;
    double axis[kDims];
    for (int d = 0; d < kDims; ++d) axis[d] = cov[top][d];
    for (int it = 0; it < 24; ++it) {
      double big = 0.0, y[kDims] = {};
      for (int d = 0; d < kDims; ++d) big = std::max(big, std::fabs(axis[d]));
      if (big == 0.0) break;  // every sampled node at one point: any cut will do
      for (int d = 0; d < kDims; ++d)
        for (int f = 0; f < kDims; ++f) y[d] += cov[d][f] * (axis[f] / big);
      std::memcpy(axis, y, sizeof(y));
    }
    double norm = 0.0;
    for (int d = 0; d < kDims; ++d) norm += axis[d] * axis[d];
    norm = norm > 0.0 ? 1.0 / std::sqrt(norm) : 0.0;
    for (int32_t i = 0; i < m; ++i) {
      double v = 0.0;
      for (int d = 0; d < kDims; ++d) v += axis[d] * norm * x[(int64_t)keys[i].node * kDims + d];
      keys[i].v = (float)v;
    }
    const int32_t k = cut(m);
    std::nth_element(keys, keys + k, keys + m);
    bisect(x, keys, k);
    keys += k;
    m -= k;
  }
  std::sort(keys, keys + m, [](const Key& a, const Key& b) { return a.node < b.node; });
}

int make_list(List& m, const char* what, int32_t n, const int32_t* tile_ptr, const int32_t* tile_col,
              const uint32_t* tile_bits) {
  if (n <= 0 || !tile_ptr) return fwn::fail(FWN_ERR_INVALID_ARG, "%s: null or empty argument", what);
  m = List{n, (n + FWN_BLOCK - 1) / FWN_BLOCK, tile_ptr, tile_col, tile_bits};
  const int32_t n_tiles = tile_ptr[m.n_blocks];
  if (n_tiles > 0 && (!tile_col || !tile_bits)) return fwn::fail(FWN_ERR_INVALID_ARG, "%s: null tile arrays", what);
  return fwn::check_tile_list(m.n_blocks, n_tiles, n, tile_ptr, tile_col);
}

// Calls fn(row within the new block, new column) for every entry of rows [128 blk, + 128) of the
// permuted mask. Bits past the last row or column are not part of the mask.
template <typename Fn>
void for_entries(const List& m, const int64_t* perm, const std::vector<int32_t>& inv, int64_t blk, Fn fn) {
  const int32_t r0 = (int32_t)blk * FWN_BLOCK, rows = std::min(FWN_BLOCK, m.n - r0);
  for (int32_t r = 0; r < rows; ++r) {
    const int32_t o = (int32_t)perm[r0 + r], ob = o / FWN_BLOCK;
    for (int32_t t = m.ptr[ob]; t < m.ptr[ob + 1]; ++t) {
      const uint32_t* w = m.bits + t * kTileWords + (int64_t)(o % FWN_BLOCK) * kWords;
      for (int32_t q = 0; q < kWords; ++q) {
        const int32_t c0 = m.col[t] * FWN_BLOCK + 32 * q;
        for (uint32_t v = w[q]; v; v &= v - 1) {
          const int32_t c = c0 + __builtin_ctz(v);
          if (c < m.n) fn(r, inv[c]);
        }
      }
    }
  }
}

// One run of columns that a packed list keeps together, with the load it gives each of the four
// parts of a workgroup that meet at the tile barriers.
struct Run {
  int32_t first;    // index of its first column in the block's column order
  uint8_t load[4];
};

// The columns of block blk in the order they are packed, and their runs of `width` columns.
// group 1: the columns some row has an element in, sorted by the 32-row groups they are live in, then by
// those all of whose rows have the element, so that a 32-column run is live (or needs no mask) for
// all of a wave's rows or none; runs of 32. group 16 or 32: the live aligned groups, one run each.
// Loads: the 32-row groups a run is live in (`pairs` false), or the count of live 16-row groups s and
// s + 4 (`pairs`: dK/dV's waves by SIMD).
void block_runs(const List& m, int64_t blk, int32_t group, bool pairs, std::vector<int32_t>& cols,
                std::vector<Run>& runs) {
  cols.clear();
  runs.clear();
  const int32_t rows = std::min(FWN_BLOCK, m.n - (int32_t)blk * FWN_BLOCK);
  struct Column {
    int32_t col;
    uint8_t live16, full32;
  };
  std::vector<Column> all;
  for (int32_t t = m.ptr[blk]; t < m.ptr[blk + 1]; ++t) {
    // any[g]: columns with an element in rows 16 g ..; every[g]: in all of rows 32 g .. + 31.
    uint32_t any[8][kWords] = {}, every[4][kWords];
    std::memset(every, 0xff, sizeof(every));
    const uint32_t* w = m.bits + t * kTileWords;
    for (int32_t r = 0; r < FWN_BLOCK; ++r)
      for (int32_t q = 0; q < kWords; ++q) {
        const uint32_t v = r < rows ? w[r * kWords + q] : 0u;
        any[r / 16][q] |= v;
        every[r / 32][q] &= v;
      }
    for (int32_t c = 0; c < FWN_BLOCK; ++c) {
      const int32_t col = m.col[t] * FWN_BLOCK + c;
      Column x{col, 0, 0};
      for (int32_t g = 0; g < 8; ++g) x.live16 |= (any[g][c / 32] >> (c % 32) & 1u) << g;
      for (int32_t g = 0; g < 4; ++g) x.full32 |= (every[g][c / 32] >> (c % 32) & 1u) << g;
      if (x.live16 && col < m.n) all.push_back(x);
    }
  }
  auto live32 = [](uint8_t l) {
    return (uint8_t)((l & 3 ? 1 : 0) | (l & 12 ? 2 : 0) | (l & 48 ? 4 : 0) | (l & 192 ? 8 : 0));
  };
  std::vector<uint8_t> live;  // of each packed column
  if (group == 1) {
    std::stable_sort(all.begin(), all.end(), [&](const Column& a, const Column& b) {
      const uint8_t la = live32(a.live16), lb = live32(b.live16);
      const int pa = __builtin_popcount(la), pb = __builtin_popcount(lb);
      if (pa != pb) return pa > pb;
      if (la != lb) return la < lb;
      return a.full32 < b.full32;
    });
    for (const Column& x : all) {
      cols.push_back(x.col);
      live.push_back(x.live16);
    }
  } else {
    for (size_t k = 0; k < all.size();) {
      const int32_t g = all[k].col / group;
      const size_t at = cols.size();
      for (int32_t c = 0; c < group; ++c) cols.push_back(std::min(g * group + c, m.n));
      live.resize(at + group, 0);
      for (; k < all.size() && all[k].col / group == g; ++k) live[at + all[k].col % group] = all[k].live16;
    }
  }
  const int32_t width = group == 1 ? 32 : group;
  for (int32_t i = 0; i < (int32_t)cols.size(); i += width) {
    uint8_t l = 0;
    for (int32_t c = i; c < std::min((int32_t)cols.size(), i + width); ++c) l |= live[c];
    Run r{i, {}};
    for (int32_t p = 0; p < 4; ++p)
      r.load[p] = (uint8_t)(pairs ? (l >> p & 1) + (l >> (p + 4) & 1) : live32(l) >> p & 1);
    runs.push_back(r);
  }
}

// Distributes the runs over tiles of `cap` runs so that the four parts of the workgroup have about
// the same load in each tile, which is what the tile barriers cost: minimises the sum over the tiles
// of the largest part's load (weighted 64, against the sum of squares that leads there), by dealing
// the runs out heaviest first and then exchanging pairs while that helps, within a fixed number of
// trials. slot[k] is the place (tile * cap + position) of run k; runs of a tile keep their order.
void balance(const std::vector<Run>& runs, int32_t cap, std::vector<int32_t>& slot) {
  const int32_t n = (int32_t)runs.size(), tiles = (n + cap - 1) / cap, places = tiles * cap;
  std::vector<Run> item(runs);
  item.resize(places, Run{-1, {0, 0, 0, 0}});  // empty places have no load
  std::vector<int32_t> order(places);
  for (int32_t i = 0; i < places; ++i) order[i] = i;
  auto total = [&](int32_t i) { return item[i].load[0] + item[i].load[1] + item[i].load[2] + item[i].load[3]; };
  std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) { return total(a) > total(b); });
  struct Tile {
    int32_t load[4] = {}, count = 0;
  };
  std::vector<Tile> tile(tiles);
  auto value = [](const int32_t (&l)[4]) {
    const int32_t top = std::max(std::max(l[0], l[1]), std::max(l[2], l[3]));
    return 64 * top + l[0] * l[0] + l[1] * l[1] + l[2] * l[2] + l[3] * l[3];
  };
  std::vector<int32_t> at(places);  // tile of each item
  int32_t start = 0;
  for (int32_t i : order) {
    int32_t best = -1, best_cost = 0;
    for (int32_t k = 0; k < tiles; ++k) {
      const int32_t t = (start + k) % tiles;
      if (tile[t].count == cap) continue;
      int32_t l[4];
      for (int p = 0; p < 4; ++p) l[p] = tile[t].load[p] + item[i].load[p];
      const int32_t cost = value(l) - value(tile[t].load);
      if (best < 0 || cost < best_cost) best = t, best_cost = cost;
    }
    for (int p = 0; p < 4; ++p) tile[best].load[p] += item[i].load[p];
    ++tile[best].count;
    at[i] = best;
    start = (best + 1) % tiles;
  }
  int64_t trials = 400000;
  for (bool more = true; more && trials > 0;) {
    more = false;
    for (int32_t a = 0; a < places && trials > 0; ++a)
      for (int32_t b = a + 1; b < places; ++b) {
        if (at[a] == at[b] || !std::memcmp(item[a].load, item[b].load, 4)) continue;
        --trials;
        Tile &x = tile[at[a]], &y = tile[at[b]];
        int32_t lx[4], ly[4];
        for (int p = 0; p < 4; ++p) {
          const int32_t d = item[b].load[p] - item[a].load[p];
          lx[p] = x.load[p] + d;
          ly[p] = y.load[p] - d;
        }
        if (value(lx) + value(ly) >= value(x.load) + value(y.load)) continue;
        std::memcpy(x.load, lx, sizeof(lx));
        std::memcpy(y.load, ly, sizeof(ly));
        std::swap(at[a], at[b]);
        more = true;
      }
  }
  slot.assign(n, 0);
  std::vector<int32_t> used(tiles, 0);
  for (int32_t k = 0; k < n; ++k) slot[k] = at[k] * cap + used[at[k]]++;
}

bool good_group(int32_t group) { return group == 1 || group == 16 || group == 32; }

// One unit of a dS numbering: the 16- or 32-column group it covers and its number.
struct Unit {
  int32_t col, unit;
  bool operator<(const Unit& o) const { return col < o.col; }
};

int inverse(const char* what, int32_t n, const int64_t* perm, std::vector<int32_t>& inv) {
  if (!perm) return fwn::fail(FWN_ERR_INVALID_ARG, "%s: null perm", what);
  inv.assign(n, -1);
  for (int32_t i = 0; i < n; ++i) {
    if (perm[i] < 0 || perm[i] >= n || inv[perm[i]] >= 0)
      return fwn::fail(FWN_ERR_INVALID_ARG, "%s: perm is not a permutation", what);
    inv[perm[i]] = i;
  }
  return FWN_OK;
}

}  // namespace

extern "C" {

int fwn_tiles_node_order(int32_t n, const int32_t* tile_ptr, const int32_t* tile_col, const uint32_t* tile_bits,
                         int64_t* perm) {
  fwn::clear_error();
  List m;
  if (int rc = make_list(m, "fwn_tiles_node_order", n, tile_ptr, tile_col, tile_bits)) return rc;
  if (!perm) return fwn::fail(FWN_ERR_INVALID_ARG, "fwn_tiles_node_order: null perm");
  try {
    // Landmarks: the node furthest from node 0, then each time the node furthest from all so far.
    std::vector<int32_t> dist, nearest;
    std::vector<float> x((size_t)m.n_blocks * FWN_BLOCK * kDims, 0.f), y(x.size(), 0.f);
    const Columns cols(m);
    const int64_t most = std::max(kVisits, kVisitsPerRow * FWN_BLOCK * tile_ptr[m.n_blocks]);
    int64_t visits = 0;
    bool near = distances(m, cols, 0, most, visits, dist);
    int32_t src = (int32_t)(std::max_element(dist.begin(), dist.end()) - dist.begin());
    for (int l = 0; near && l < kLandmarks; ++l) {
      near = distances(m, cols, src, most, visits, dist);
      for (int32_t i = 0; i < n; ++i) x[(int64_t)i * kDims + l] = (float)dist[i];
      if (l == 0) nearest = dist;
      for (int32_t i = 0; i < n; ++i) nearest[i] = std::min(nearest[i], dist[i]);
      src = (int32_t)(std::max_element(nearest.begin(), nearest.end()) - nearest.begin());
    }
    if (!near) {
      for (int32_t i = 0; i < n; ++i) perm[i] = i;
      return FWN_OK;
    }
    for (int s = 0; s < kSmooth; ++s) {
      average(m, x, y);
      x.swap(y);
    }
    std::vector<Key> keys(n);
    for (int32_t i = 0; i < n; ++i) keys[i] = Key{0.f, i};
    bisect(x, keys.data(), n);
    for (int32_t i = 0; i < n; ++i) perm[i] = keys[i].node;
  } catch (const std::exception& e) {
    return fwn::fail(FWN_ERR_INVALID_ARG, "fwn_tiles_node_order: %s", e.what());
  }
  return FWN_OK;
}

int fwn_tiles_permute_count(int32_t n, const int32_t* tile_ptr, const int32_t* tile_col, const uint32_t* tile_bits,
                            const int64_t* perm, int32_t* new_ptr) {
  fwn::clear_error();
  List m;
  if (int rc = make_list(m, "fwn_tiles_permute_count", n, tile_ptr, tile_col, tile_bits)) return rc;
  if (!new_ptr) return fwn::fail(FWN_ERR_INVALID_ARG, "fwn_tiles_permute_count: null output");
  try {
    std::vector<int32_t> inv;
    if (int rc = inverse("fwn_tiles_permute_count", n, perm, inv)) return rc;
    std::vector<int32_t> count(m.n_blocks);
    parallel_for(m.n_blocks, 2, [&](int64_t b, int64_t e) {
      std::vector<uint8_t> seen(m.n_blocks);
      for (int64_t blk = b; blk < e; ++blk) {
        std::fill(seen.begin(), seen.end(), (uint8_t)0);
        for_entries(m, perm, inv, blk, [&](int32_t, int32_t c) { seen[c / FWN_BLOCK] = 1; });
        count[blk] = (int32_t)std::count(seen.begin(), seen.end(), (uint8_t)1);
      }
    });
    int64_t total = 0;
    new_ptr[0] = 0;
    for (int32_t blk = 0; blk < m.n_blocks; ++blk) {
      total += count[blk];
      if (total > INT32_MAX) return fwn::fail(FWN_ERR_INVALID_ARG, "fwn_tiles_permute_count: too many tiles");
      new_ptr[blk + 1] = (int32_t)total;
    }
  } catch (const std::exception& e) {
    return fwn::fail(FWN_ERR_INVALID_ARG, "fwn_tiles_permute_count: %s", e.what());
  }
  return FWN_OK;
}

int fwn_tiles_permute_fill(int32_t n, const int32_t* tile_ptr, const int32_t* tile_col, const uint32_t* tile_bits,
                           const int64_t* perm, const int32_t* new_ptr, int32_t* new_col, uint32_t* new_bits) {
  fwn::clear_error();
  List m;
  if (int rc = make_list(m, "fwn_tiles_permute_fill", n, tile_ptr, tile_col, tile_bits)) return rc;
  if (!new_ptr || (new_ptr[m.n_blocks] > 0 && (!new_col || !new_bits)))
    return fwn::fail(FWN_ERR_INVALID_ARG, "fwn_tiles_permute_fill: null output");
  std::atomic<bool> bad(false);
  try {
    std::vector<int32_t> inv;
    if (int rc = inverse("fwn_tiles_permute_fill", n, perm, inv)) return rc;
    parallel_for(m.n_blocks, 2, [&](int64_t b, int64_t e) {
      // One block's rows as a dense bitmap by column block, then its blocks with a bit in order.
      std::vector<uint32_t> dense((size_t)m.n_blocks * kTileWords);
      std::vector<uint8_t> seen(m.n_blocks);
      for (int64_t blk = b; blk < e; ++blk) {
        std::fill(seen.begin(), seen.end(), (uint8_t)0);
        for_entries(m, perm, inv, blk, [&](int32_t r, int32_t c) {
          const int32_t kb = c / FWN_BLOCK, within = c % FWN_BLOCK;
          uint32_t* tile = &dense[kb * kTileWords];
          if (!seen[kb]) {
            seen[kb] = 1;
            std::memset(tile, 0, kTileWords * sizeof(uint32_t));
          }
          tile[r * kWords + within / 32] |= 1u << (within % 32);
        });
        int64_t t = new_ptr[blk];
        if (std::count(seen.begin(), seen.end(), (uint8_t)1) != new_ptr[blk + 1] - t) {
          bad = true;
          return;
        }
        for (int32_t kb = 0; kb < m.n_blocks; ++kb) {
          if (!seen[kb]) continue;
          new_col[t] = kb;
          std::memcpy(new_bits + t * kTileWords, &dense[kb * kTileWords], kTileWords * sizeof(uint32_t));
          ++t;
        }
      }
    });
  } catch (const std::exception& e) {
    return fwn::fail(FWN_ERR_INVALID_ARG, "fwn_tiles_permute_fill: %s", e.what());
  }
  if (bad) return fwn::fail(FWN_ERR_INVALID_ARG, "fwn_tiles_permute_fill: new_ptr does not match the mask");
  return FWN_OK;
}

int fwn_tiles_compact_count(int32_t n, const int32_t* tile_ptr, const int32_t* tile_col, const uint32_t* tile_bits,
                            int32_t group, int32_t* new_ptr) {
  fwn::clear_error();
  List m;
  if (int rc = make_list(m, "fwn_tiles_compact_count", n, tile_ptr, tile_col, tile_bits)) return rc;
  if (!new_ptr || !good_group(group))
    return fwn::fail(FWN_ERR_INVALID_ARG, "fwn_tiles_compact_count: null output or group %d (1, 16 or 32)", group);
  try {
    std::vector<int32_t> count(m.n_blocks);
    parallel_for(m.n_blocks, 4, [&](int64_t b, int64_t e) {
      std::vector<int32_t> cols;
      std::vector<Run> runs;
      for (int64_t blk = b; blk < e; ++blk) {
        block_runs(m, blk, group, false, cols, runs);
        count[blk] = (int32_t)((cols.size() + FWN_BLOCK - 1) / FWN_BLOCK);
      }
    });
    new_ptr[0] = 0;
    for (int32_t blk = 0; blk < m.n_blocks; ++blk) new_ptr[blk + 1] = new_ptr[blk] + count[blk];  // at most n_tiles
  } catch (const std::exception& e) {
    return fwn::fail(FWN_ERR_INVALID_ARG, "fwn_tiles_compact_count: %s", e.what());
  }
  return FWN_OK;
}

int fwn_tiles_compact_fill(int32_t n, const int32_t* tile_ptr, const int32_t* tile_col, const uint32_t* tile_bits,
                           int32_t group, int32_t parts, int32_t window, const int32_t* new_ptr, int32_t* cols,
                           uint32_t* new_bits) {
  fwn::clear_error();
  List m;
  if (int rc = make_list(m, "fwn_tiles_compact_fill", n, tile_ptr, tile_col, tile_bits)) return rc;
  if (!new_ptr || !good_group(group) || (new_ptr[m.n_blocks] > 0 && (!cols || !new_bits)) || parts < 0 ||
      parts > FWN_PARTS_PAIRS16 || window < 0)
    return fwn::fail(FWN_ERR_INVALID_ARG,
                     "fwn_tiles_compact_fill: null output, group %d (1, 16 or 32), parts %d or window %d", group, parts,
                     window);
  std::atomic<bool> bad(false);
  try {
    parallel_for(m.n_blocks, 4, [&](int64_t b, int64_t e) {
      const int32_t width = group == 1 ? 32 : group;
      std::vector<int32_t> packed, slot, place, at((size_t)m.n_blocks * FWN_BLOCK, -1);
      std::vector<Run> runs, part;
      for (int64_t blk = b; blk < e; ++blk) {
        block_runs(m, blk, group, parts == FWN_PARTS_PAIRS16, packed, runs);
        const int64_t t0 = new_ptr[blk], tiles = new_ptr[blk + 1] - t0;
        if (tiles != (int64_t)(packed.size() + FWN_BLOCK - 1) / FWN_BLOCK) {
          bad = true;
          return;
        }
        if (tiles == 0) continue;
        slot.clear();
        const size_t cap = FWN_BLOCK / width, step = window ? window * cap : runs.size();
        for (size_t k = 0; k < runs.size(); k += step) {
          part.assign(runs.begin() + k, runs.begin() + std::min(runs.size(), k + step));
          balance(part, (int32_t)cap, place);
          for (int32_t x : place) slot.push_back((int32_t)k + x);
        }
        std::memset(new_bits + t0 * kTileWords, 0, tiles * kTileWords * sizeof(uint32_t));
        std::fill(cols + t0 * FWN_BLOCK, cols + (t0 + tiles) * FWN_BLOCK, n);
        for (size_t k = 0; k < runs.size(); ++k)
          for (int32_t c = 0; c < width && runs[k].first + c < (int32_t)packed.size(); ++c) {
            const int32_t col = packed[runs[k].first + c], to = slot[k] * width + c;
            cols[t0 * FWN_BLOCK + to] = col;
            if (col < n) at[col] = to;
          }
        const int32_t rows = std::min(FWN_BLOCK, n - (int32_t)blk * FWN_BLOCK);
        for (int32_t t = m.ptr[blk]; t < m.ptr[blk + 1]; ++t)
          for (int32_t r = 0; r < rows; ++r)
            for (int32_t q = 0; q < kWords; ++q)
              for (uint32_t v = m.bits[t * kTileWords + r * kWords + q]; v; v &= v - 1) {
                const int32_t c = m.col[t] * FWN_BLOCK + 32 * q + __builtin_ctz(v);
                if (c >= n) continue;
                const int32_t to = at[c];
                new_bits[(t0 + to / FWN_BLOCK) * kTileWords + r * kWords + to % FWN_BLOCK / 32] |= 1u << (to % 32);
              }
      }
    });
  } catch (const std::exception& e) {
    return fwn::fail(FWN_ERR_INVALID_ARG, "fwn_tiles_compact_fill: %s", e.what());
  }
  if (bad) return fwn::fail(FWN_ERR_INVALID_ARG, "fwn_tiles_compact_fill: new_ptr does not match the mask");
  return FWN_OK;
}

int fwn_tiles_unit_map(int32_t n, const int32_t* tile_ptr, const uint32_t* bits, const int32_t* cols,
                       const int32_t* tile_ptr_t, const uint32_t* bits_t, const int32_t* cols_t, int32_t unit_keys,
                       int32_t* ubase, int32_t* tmap, int64_t* n_units) {
  fwn::clear_error();
  if (n <= 0 || !tile_ptr || !tile_ptr_t || !n_units || (unit_keys != 16 && unit_keys != 32))
    return fwn::fail(FWN_ERR_INVALID_ARG, "fwn_tiles_unit_map: null argument or unit_keys %d (16 or 32)", unit_keys);
  const int32_t n_blocks = (n + FWN_BLOCK - 1) / FWN_BLOCK;
  const int32_t n_tiles = tile_ptr[n_blocks], n_tiles_t = tile_ptr_t[n_blocks];
  if ((n_tiles > 0 && (!bits || !cols || !ubase)) || (n_tiles_t > 0 && (!bits_t || !cols_t || !tmap)))
    return fwn::fail(FWN_ERR_INVALID_ARG, "fwn_tiles_unit_map: null tile arrays");
  try {
    // The units of each 32-row group, in the order of their columns.
    std::vector<std::vector<Unit>> units((size_t)n_blocks * 4);
    int64_t total = 0;
    const int32_t per = FWN_BLOCK / unit_keys;  // units of a 32-row group in one tile
    for (int32_t blk = 0; blk < n_blocks; ++blk)
      for (int32_t t = tile_ptr[blk]; t < tile_ptr[blk + 1]; ++t) {
        ubase[t] = (int32_t)total;
        const uint32_t* w = bits + t * kTileWords;
        for (int32_t g = 0; g < 4; ++g)
          for (int32_t x = 0; x < per; ++x) {
            const int32_t c0 = x * unit_keys;
            const uint32_t mask = unit_keys == 32 ? 0xffffffffu : 0xffffu << (c0 % 32);
            uint32_t any = 0;
            for (int32_t r = 32 * g; r < 32 * g + 32; ++r) any |= w[r * kWords + c0 / 32] & mask;
            if (!any) continue;
            const int32_t c = cols[(int64_t)t * FWN_BLOCK + c0];
            if (c < 0 || c >= n || c % unit_keys)
              return fwn::fail(FWN_ERR_TILES, "fwn_tiles_unit_map: tile %d is not compacted in groups of %d", t, unit_keys);
            units[4 * blk + g].push_back(Unit{c / unit_keys, (int32_t)total++});
            if (total > INT32_MAX) return fwn::fail(FWN_ERR_INVALID_ARG, "fwn_tiles_unit_map: more than 2^31 units");
          }
      }
    for (auto& u : units) std::sort(u.begin(), u.end());
    std::atomic<int64_t> found(0);
    std::atomic<bool> bad(false);
    parallel_for(n_blocks, 4, [&](int64_t b, int64_t e) {
      int64_t mine = 0;
      for (int64_t blk = b; blk < e; ++blk)
        for (int32_t t = tile_ptr_t[blk]; t < tile_ptr_t[blk + 1]; ++t) {
          int32_t* m = tmap + (int64_t)t * 36;
          const uint32_t* w = bits_t + t * kTileWords;
          uint32_t live = 0;
          for (int32_t kg = 0; kg < 8; ++kg)
            for (int32_t c = 0; c < 4; ++c) {
              m[4 * kg + c] = -1;
              uint32_t own = 0, any = 0;
              const int32_t r0 = unit_keys == 32 ? 32 * (kg / 2) : 16 * kg;
              for (int32_t r = r0; r < r0 + unit_keys; ++r) any |= w[r * kWords + c];
              for (int32_t r = 16 * kg; r < 16 * kg + 16; ++r) own |= w[r * kWords + c];
              if (own) live |= 1u << (8 * c + kg);
              if (!any) continue;
              const int32_t q = cols_t[(int64_t)t * FWN_BLOCK + 32 * c], key = ((int32_t)blk * FWN_BLOCK + r0) / unit_keys;
              if (q < 0 || q >= n || q % 32) {
                bad = true;
                return;
              }
              const auto& u = units[q / 32];
              const auto it = std::lower_bound(u.begin(), u.end(), Unit{key, 0});
              if (it == u.end() || it->col != key) {
                bad = true;
                return;
              }
              m[4 * kg + c] = it->unit;
              if (unit_keys == 16 || kg % 2 == 0) ++mine;
            }
          m[32] = (int32_t)live;
          m[33] = m[34] = m[35] = 0;
        }
      found += mine;
    });
    // Each unit of one list is one of the other's, and as many: none is written twice or never.
    if (bad || found != total)
      return fwn::fail(FWN_ERR_TILES, "fwn_tiles_unit_map: the lists have different units (not transposes)");
    *n_units = total;
  } catch (const std::exception& e) {
    return fwn::fail(FWN_ERR_INVALID_ARG, "fwn_tiles_unit_map: %s", e.what());
  }
  return FWN_OK;
}

}  // extern "C"
