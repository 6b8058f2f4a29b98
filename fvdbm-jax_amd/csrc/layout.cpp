// Host-side device-layout construction (see layout.h).
#include "layout.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <numeric>
#include <system_error>
#include <thread>
#include <utility>

namespace fvdbm {

namespace {

// BFS over the unvisited component of `s`; returns the last level and the
// eccentricity of s. `stamp`/`mark` avoid clearing a per-call array.
int bfs_last_level(int s, const std::vector<int32_t> &xadj,
                   const std::vector<int32_t> &adj, const std::vector<char> &placed,
                   std::vector<int32_t> &mark, int32_t stamp,
                   std::vector<int32_t> &queue, std::vector<int32_t> &last) {
  queue.clear();
  queue.push_back(s);
  mark[s] = stamp;
  int depth = 0;
  size_t level_start = 0, level_end = 1;
  for (;;) {
    for (size_t h = level_start; h < level_end; ++h) {
      int v = queue[h];
      for (int e = xadj[v]; e < xadj[v + 1]; ++e) {
        int u = adj[e];
        if (placed[u] || mark[u] == stamp) continue;
        mark[u] = stamp;
        queue.push_back(u);
      }
    }
    if (queue.size() == level_end) break;
    level_start = level_end;
    level_end = queue.size();
    ++depth;
  }
  last.assign(queue.begin() + level_start, queue.begin() + level_end);
  return depth;
}

// Index of (x, y) along a Hilbert curve over a 2^order x 2^order grid.
uint64_t hilbert_index(uint32_t x, uint32_t y, int order) {
  uint64_t d = 0;
  for (uint32_t s = 1u << (order - 1); s > 0; s >>= 1) {
    const uint32_t rx = (x & s) ? 1u : 0u, ry = (y & s) ? 1u : 0u;
    d += (uint64_t)s * s * ((3u * rx) ^ ry);
    if (ry == 0) {  // rotate the quadrant
      if (rx == 1) {
        x = s - 1 - (x & (s - 1)) + (x & ~(s - 1));
        y = s - 1 - (y & (s - 1)) + (y & ~(s - 1));
      }
      const uint32_t t = x;
      x = y;
      y = t;
    }
  }
  return d;
}

}  // namespace

std::vector<int32_t> hilbert_order(int n, const double *xy) {
  double x0 = xy[0], x1 = xy[0], y0 = xy[1], y1 = xy[1];
  for (int i = 0; i < n; ++i) {
    x0 = std::min(x0, xy[2 * i]);
    x1 = std::max(x1, xy[2 * i]);
    y0 = std::min(y0, xy[2 * i + 1]);
    y1 = std::max(y1, xy[2 * i + 1]);
  }
  const int order = 20;
  const double span = std::max(x1 - x0, y1 - y0);
  const double scale = span > 0 ? ((1u << order) - 1) / span : 0.0;
  std::vector<std::pair<uint64_t, int32_t>> key(n);
  for (int i = 0; i < n; ++i) {
    const uint32_t gx = (uint32_t)((xy[2 * i] - x0) * scale);
    const uint32_t gy = (uint32_t)((xy[2 * i + 1] - y0) * scale);
    key[i] = {hilbert_index(gx, gy, order), i};
  }
  std::sort(key.begin(), key.end());
  std::vector<int32_t> perm(n);
  for (int i = 0; i < n; ++i) perm[i] = key[i].second;
  return perm;
}

std::vector<int32_t> reverse_cuthill_mckee(int n, const std::vector<int32_t> &xadj,
                                           const std::vector<int32_t> &adj) {
  std::vector<int32_t> deg(n);
  for (int i = 0; i < n; ++i) deg[i] = xadj[i + 1] - xadj[i];
  std::vector<char> placed(n, 0);
  std::vector<int32_t> mark(n, -1), queue, last, order, nbrs;
  order.reserve(n);
  int32_t stamp = 0;
  for (int s0 = 0; s0 < n; ++s0) {
    if (placed[s0]) continue;
    // George-Liu pseudo-peripheral node: restart from the lowest-degree node
    // of the last BFS level while the eccentricity grows.
    int root = s0;
    int ecc = bfs_last_level(root, xadj, adj, placed, mark, stamp++, queue, last);
    for (int it = 0; it < 16; ++it) {
      int best = last[0];
      for (int v : last)
        if (deg[v] < deg[best] || (deg[v] == deg[best] && v < best)) best = v;
      int e2 = bfs_last_level(best, xadj, adj, placed, mark, stamp++, queue, last);
      if (e2 <= ecc) break;
      ecc = e2;
      root = best;
    }
    // Cuthill-McKee: BFS, unplaced neighbours in increasing (degree, id).
    size_t head = order.size();
    order.push_back(root);
    placed[root] = 1;
    while (head < order.size()) {
      int v = order[head++];
      nbrs.clear();
      for (int e = xadj[v]; e < xadj[v + 1]; ++e) {
        int u = adj[e];
        if (!placed[u]) {
          placed[u] = 1;
          nbrs.push_back(u);
        }
      }
      std::sort(nbrs.begin(), nbrs.end(), [&](int a, int b) {
        return deg[a] < deg[b] || (deg[a] == deg[b] && a < b);
      });
      order.insert(order.end(), nbrs.begin(), nbrs.end());
    }
  }
  std::reverse(order.begin(), order.end());
  return order;
}

// The rings of the tiles roots[first, last), as (first cell, cells), into R, whose
// offsets start at 0; code and fan_own ([3][Cp], [Cp]) get the own cells' entries.
template <typename T>
static void build_ring_part(const fvdbm_mesh_desc &m, const HostLayout<T> &L,
                            const std::vector<int32_t> &node_an, int tile, int depth,
                            const std::function<bool(const int32_t *)> &fits,
                            const std::vector<std::pair<int, int>> &roots, int first, int last,
                            std::atomic<int> &left, HostRings<T> &R, int32_t *code, int32_t *fan_own) {
  const T *fd = static_cast<const T *>(m.face_dists);
  const int K = L.K;
  const size_t Cp = (size_t)L.Cp;
  const int block = L.Cp / L.ntiles;
  std::vector<int32_t> stage_of(Cp, -1);  // device cell -> stage slot in the current tile
  std::vector<int32_t> entry_of(L.N, -1); // node -> table entry of the current tile
  std::vector<int32_t> fan_of(Cp, -1);    // device cell -> fan record of the current tile
  std::vector<int32_t> ring, next, nodes, fans;
  auto cell_id = [](int32_t cj) { return cj >= 0 ? cj : -2 - cj; };
  // a ghost face (device cell i, face k) names its two nodes by mesh face
  auto face_of = [&](int i, int k) { return m.cell_faces[3 * (size_t)L.new_to_old[i] + k]; };
  // the tile of cells [lo, lo + n_own); false, and nothing added, when it
  // does not fit
  auto build_tile = [&](int lo, int n_own) {
    const int t = (int)(R.meta.size() / kRingMeta);
    R.meta.resize(R.meta.size() + kRingMeta, 0);
    int32_t *meta = R.meta.data() + (size_t)t * kRingMeta;
    meta[kMetaRing] = (int32_t)R.ring_cells.size();
    meta[kMetaFaces] = (int32_t)(R.rg_code.size() / 3);
    meta[kMetaEntry] = (int32_t)R.entries.size();
    meta[kMetaPair] = (int32_t)R.pair_fan.size();
    meta[kMetaGhost] = (int32_t)R.gh_s0.size();
    meta[kMetaCount] = n_own;
    meta[kMetaCase] = L.tile_case[lo / block];
    meta[kMetaTile] = t;
    meta[kMetaFirst] = lo;
    for (int i = 0; i < n_own; ++i) stage_of[lo + i] = i;
    ring.clear();
    nodes.clear();
    auto add_entry = [&](int node) {
      if (entry_of[node] >= 0) return;
      entry_of[node] = (int32_t)nodes.size();
      nodes.push_back(node);
    };
    // level by level: the table entries of the level's ghost faces, then
    // the next level = neighbours and node cells not staged yet
    size_t lev0 = 0;  // first ring cell of the level being closed
    for (int k = 0; k < depth; ++k) {
      const size_t nodes0 = nodes.size();
      const size_t nc = k == 0 ? (size_t)n_own : ring.size() - lev0;
      next.clear();
      for (size_t j = 0; j < nc; ++j) {
        const int i = k == 0 ? lo + (int)j : ring[lev0 + j];
        for (int f = 0; f < 3; ++f) {
          const int32_t code = L.nb[(size_t)f * Cp + i];
          if (code >= 0) {
            const int o = code & kIndexMask;
            if (stage_of[o] < 0) next.push_back(o);
          } else {
            const int fid = face_of(i, f);
            add_entry(m.face_nodes[2 * (size_t)fid]);
            add_entry(m.face_nodes[2 * (size_t)fid + 1]);
          }
        }
      }
      meta[kMetaEntries + k] = (int32_t)nodes.size();
      for (size_t e = nodes0; e < nodes.size(); ++e) {
        const int an = node_an[nodes[e]];
        if (an < 0) continue;
        for (int c = 0; c < K; ++c) {
          const int32_t cj = L.an_cells[(size_t)an * K + c];
          if (cj < 0 && L.an_w[(size_t)an * K + c] == T(0)) continue;
          if (stage_of[cell_id(cj)] < 0) next.push_back(cell_id(cj));
        }
      }
      std::sort(next.begin(), next.end());
      next.erase(std::unique(next.begin(), next.end()), next.end());
      lev0 = ring.size();
      for (int c : next) {
        stage_of[c] = tile + (int)ring.size();
        ring.push_back(c);
      }
      meta[kMetaCells + k + 1] = (int32_t)ring.size();
    }
    meta[kMetaSlot] = tile + (int32_t)ring.size();
    // table entries, their pairs and the fan records; S_k's extra fan cells
    meta[kMetaExtra] = (int32_t)(R.extra.size() / 2);
    fans.clear();
    int np = 0;
    size_t e = 0;
    for (int k = 0; k < depth; ++k) {
      for (; e < (size_t)meta[kMetaEntries + k]; ++e) {
        const int an = node_an[nodes[e]];
        R.entries.push_back(an >= 0 ? an : -1 - nodes[e]);
        R.entry_pair.push_back(np);
        for (int c = 0; an >= 0 && c < K; ++c) {
          const int32_t cj = L.an_cells[(size_t)an * K + c];
          const T w = L.an_w[(size_t)an * K + c];
          if (cj < 0 && w == T(0)) continue;
          int32_t &fan = fan_of[cell_id(cj)];
          if (fan < 0) {
            fan = (int32_t)fans.size();
            fans.push_back(cell_id(cj));
          }
          R.pair_fan.push_back(fan | (cj < 0 ? kGhostBit : 0));
          R.pair_w.push_back(w);
          ++np;
        }
      }
      meta[kMetaPairs + k] = np;
      int extra = 0;
      for (size_t i = 0; i < fans.size(); ++i)
        if (stage_of[fans[i]] >= tile + meta[kMetaCells + k]) {
          R.extra.push_back(stage_of[fans[i]]);
          R.extra.push_back((int32_t)i);
          ++extra;
        }
      meta[kMetaExtras + k + 1] = meta[kMetaExtras + k] + extra;
      meta[kMetaThreads] = std::max(meta[kMetaThreads], tile + meta[kMetaCells + k] + extra);
    }
    R.entry_pair.push_back(np);
    auto clear = [&] {
      for (int i = 0; i < n_own; ++i) stage_of[lo + i] = -1;
      for (int c : ring) stage_of[c] = -1;
      for (int nd : nodes) entry_of[nd] = -1;
      for (int c : fans) fan_of[c] = -1;
    };
    meta[kMetaFan] = (int32_t)fans.size();
    for (int i = -n_own; i < meta[kMetaCells + depth - 1]; ++i)
      for (int f = 0; f < 3; ++f)
        meta[kMetaGhosts + depth - 1] += L.nb[(size_t)f * Cp + (i < 0 ? lo + n_own + i : ring[i])] < 0;
    if (n_own > 1 && !fits(meta)) {
      clear();
      R.entries.resize(meta[kMetaEntry]);
      R.entry_pair.resize((size_t)meta[kMetaEntry] + t);
      R.pair_fan.resize(meta[kMetaPair]);
      R.pair_w.resize(meta[kMetaPair]);
      R.extra.resize(2 * (size_t)meta[kMetaExtra]);
      R.meta.resize((size_t)t * kRingMeta);
      return false;
    }
    R.ring_cells.insert(R.ring_cells.end(), ring.begin(), ring.end());
    for (int i = lo; i < lo + n_own; ++i) fan_own[i] = fan_of[i];
    for (int r = 0; r < meta[kMetaCells + depth - 1]; ++r) R.rg_fan.push_back(fan_of[ring[r]]);
    // face records: own cells, then the updated ring cells, ghosts in that order
    int ng = 0;
    auto face_code = [&](int i, int f, int self) {
      const int32_t nb = L.nb[(size_t)f * Cp + i];
      if (nb >= 0) return stage_of[nb & kIndexMask] | (nb & kSlot1Bit);
      const int fid = face_of(i, f);
      const bool slot1 = (nb & kSlot1Bit) != 0;
      const T d0 = fd[2 * (size_t)fid], d1 = fd[2 * (size_t)fid + 1];
      R.gh_s0.push_back(entry_of[m.face_nodes[2 * (size_t)fid]]);
      R.gh_s1.push_back(entry_of[m.face_nodes[2 * (size_t)fid + 1]]);
      R.gh_self.push_back(self);
      R.gh_ratio.push_back(slot1 ? d0 / d1 : d1 / d0);
      return (meta[kMetaSlot] + ng++) | (nb & kSlot1Bit);
    };
    for (int i = 0; i < n_own; ++i)
      for (int f = 0; f < 3; ++f) code[(size_t)f * Cp + lo + i] = face_code(lo + i, f, i);
    meta[kMetaGhosts] = ng;
    for (int k = 1; k < depth; ++k) {
      for (int r = meta[kMetaCells + k - 1]; r < meta[kMetaCells + k]; ++r)
        for (int f = 0; f < 3; ++f) R.rg_code.push_back(face_code(ring[r], f, tile + r));
      meta[kMetaGhosts + k] = ng;
    }
    clear();
    return true;
  };
  std::vector<std::pair<int, int>> todo;
  for (int r = first; r < last; ++r) {
    todo.assign(1, roots[r]);
    while (!todo.empty()) {
      const auto [at, n] = todo.back();
      todo.pop_back();
      if (build_tile(at, n)) {
        if (--left < 0) return;
        continue;
      }
      todo.push_back({at + n / 2, n - n / 2});
      todo.push_back({at, n / 2});
    }
  }
}

template <typename T>
void build_rings(const fvdbm_mesh_desc &m, const HostLayout<T> &L, int tile, int depth,
                 const std::function<bool(const int32_t *)> &fits, double most, HostRings<T> &R) {
  R = HostRings<T>();
  if (depth < 2 || depth > kMaxDepth) return;
  R.depth = depth;
  R.tile = tile;
  R.code.assign(3 * (size_t)L.Cp, 0);
  R.fan_own.assign(L.Cp, -1);
  std::vector<int32_t> node_an(L.N, -1);
  for (int a = 0; a < L.nan; ++a) node_an[L.an_gid[a]] = a;
  // the tiles: each case's cells, which are consecutive (only the last of its tiles
  // in the layout has empty slots), in parts of `tile`
  const int block = L.Cp / L.ntiles;
  std::vector<std::pair<int, int>> roots;
  for (int b = 0, last; b < L.ntiles; b = last + 1) {
    for (last = b; last + 1 < L.ntiles && L.tile_count[last] == block && L.tile_case[last + 1] == L.tile_case[b];)
      ++last;
    const int end = last * block + L.tile_count[last];
    for (int lo = b * block; lo < end; lo += tile) roots.push_back({lo, std::min(tile, end - lo)});
  }
  // tiles are independent: ranges of them on threads, then one after the
  // other in the lists (the result does not depend on the thread count). A
  // thread per 16 tiles from 64 on: 200 tiles of 64 cells 4.4 ms with a thread per
  // 64, 1.8 so; 32 tiles take 0.7 ms on one, 3.3 on two.
  const int hw = (int)std::thread::hardware_concurrency(), tiles = (int)roots.size();
  const int n = tiles < 64 ? 1 : std::max(1, std::min({8, hw, tiles / 16}));
  std::vector<HostRings<T>> part(n);
  std::atomic<int> left((int)std::min<double>(most * tiles, INT32_MAX));  // tiles that may yet be built
  auto on_threads = [&](auto &&work) {
    std::vector<std::thread> pool;
    pool.reserve(n);
    std::atomic<int> next(0);
    std::exception_ptr error;
    std::mutex mu;
    auto run = [&] {
      for (int i = next++; i < n; i = next++) try {
          work(i);
        } catch (...) {
          std::lock_guard<std::mutex> lock(mu);
          error = std::current_exception();
        }
    };
    for (int i = 1; i < n; ++i) try {
        pool.emplace_back(run);
      } catch (const std::system_error &) {
        break;  // no more threads: the others take its share
      }
    run();
    for (std::thread &t : pool) t.join();
    if (error) std::rethrow_exception(error);
  };
  on_threads([&](int i) {
    build_ring_part(m, L, node_an, tile, depth, fits, roots, (int)((int64_t)tiles * i / n),
                    (int)((int64_t)tiles * (i + 1) / n), left, part[i], R.code.data(), R.fan_own.data());
  });
  if (left < 0) return;
  // where each part goes in the lists
  struct At {
    size_t tiles = 0, ring = 0, faces = 0, entries = 0, pairs = 0, ghosts = 0, extra = 0;
  };
  std::vector<At> at(n + 1);
  for (int i = 0; i < n; ++i) {
    const HostRings<T> &p = part[i];
    at[i + 1] = {at[i].tiles + p.meta.size() / kRingMeta, at[i].ring + p.ring_cells.size(),
                 at[i].faces + p.rg_fan.size(), at[i].entries + p.entries.size(),
                 at[i].pairs + p.pair_fan.size(), at[i].ghosts + p.gh_s0.size(),
                 at[i].extra + p.extra.size() / 2};
  }
  R.ntiles = (int)at[n].tiles;
  R.meta.resize(at[n].tiles * kRingMeta);
  R.ring_cells.resize(at[n].ring);
  R.rg_code.resize(3 * at[n].faces);
  R.rg_fan.resize(at[n].faces);
  R.entries.resize(at[n].entries);
  R.entry_pair.resize(at[n].entries + at[n].tiles);
  R.pair_fan.resize(at[n].pairs);
  R.pair_w.resize(at[n].pairs);
  R.gh_s0.resize(at[n].ghosts);
  R.gh_s1.resize(at[n].ghosts);
  R.gh_self.resize(at[n].ghosts);
  R.gh_ratio.resize(at[n].ghosts);
  R.extra.resize(2 * at[n].extra);
  on_threads([&](int i) {
    HostRings<T> &p = part[i];
    const At &o = at[i];
    for (size_t t = 0; t < p.meta.size(); t += kRingMeta) {
      int32_t *meta = p.meta.data() + t;
      meta[kMetaRing] += (int32_t)o.ring;
      meta[kMetaFaces] += (int32_t)o.faces;
      meta[kMetaEntry] += (int32_t)o.entries;
      meta[kMetaPair] += (int32_t)o.pairs;
      meta[kMetaGhost] += (int32_t)o.ghosts;
      meta[kMetaExtra] += (int32_t)o.extra;
      meta[kMetaTile] += (int32_t)o.tiles;
    }
    auto put = [](auto &dst, const auto &src, size_t to) {
      std::copy(src.begin(), src.end(), dst.begin() + to);
    };
    put(R.meta, p.meta, o.tiles * kRingMeta);
    put(R.ring_cells, p.ring_cells, o.ring);
    put(R.rg_code, p.rg_code, 3 * o.faces);
    put(R.rg_fan, p.rg_fan, o.faces);
    put(R.entries, p.entries, o.entries);
    put(R.entry_pair, p.entry_pair, o.entries + o.tiles);
    put(R.pair_fan, p.pair_fan, o.pairs);
    put(R.pair_w, p.pair_w, o.pairs);
    put(R.gh_s0, p.gh_s0, o.ghosts);
    put(R.gh_s1, p.gh_s1, o.ghosts);
    put(R.gh_self, p.gh_self, o.ghosts);
    put(R.gh_ratio, p.gh_ratio, o.ghosts);
    put(R.extra, p.extra, 2 * o.extra);
    p = HostRings<T>();
  });
  // every index the kernel uses stays within its tile's stage and table
  for (int t = 0; t < R.ntiles; ++t) {
    const int32_t *meta = R.meta.data() + (size_t)t * kRingMeta;
    const int ng = meta[kMetaGhosts + depth - 1], ne = meta[kMetaEntries + depth - 1];
    const int slots = meta[kMetaSlot] + ng;
    auto bad = [&](int32_t code) { return code < 0 || (code & kIndexMask) >= slots; };
    for (int i = meta[kMetaFirst]; i < meta[kMetaFirst] + meta[kMetaCount]; ++i)
      for (int f = 0; f < 3; ++f)
        if (bad(R.code[(size_t)f * L.Cp + i])) return;
    for (int r = 0; r < 3 * meta[kMetaCells + depth - 1]; ++r)
      if (bad(R.rg_code[3 * (size_t)meta[kMetaFaces] + r])) return;
    for (int p = meta[kMetaPair]; p < meta[kMetaPair] + meta[kMetaPairs + depth - 1]; ++p)
      if ((R.pair_fan[p] & kIndexMask) >= meta[kMetaFan]) return;
    for (int x = meta[kMetaExtra]; x < meta[kMetaExtra] + meta[kMetaExtras + depth]; ++x)
      if (R.extra[2 * (size_t)x] >= meta[kMetaSlot] || R.extra[2 * (size_t)x + 1] >= meta[kMetaFan]) return;
    for (int g = meta[kMetaGhost]; g < meta[kMetaGhost] + ng; ++g)
      if (R.gh_s0[g] < 0 || R.gh_s0[g] >= ne || R.gh_s1[g] < 0 || R.gh_s1[g] >= ne) return;
  }
  R.ok = true;
}

template void build_rings<float>(const fvdbm_mesh_desc &, const HostLayout<float> &, int, int,
                                 const std::function<bool(const int32_t *)> &, double, HostRings<float> &);
template void build_rings<double>(const fvdbm_mesh_desc &, const HostLayout<double> &, int, int,
                                  const std::function<bool(const int32_t *)> &, double, HostRings<double> &);

template <typename T>
bool build_layout(const fvdbm_mesh_desc &m, int reorder, int tile,
                  HostLayout<T> &L, std::string &err, const int32_t *cell_case, int ncases) {
  const int C = m.n_cells, F = m.n_faces, N = m.n_nodes, K = m.k_max;
  if (C <= 0 || F <= 0 || N <= 0 || K < 0) {
    err = "mesh must have cells, faces and nodes";
    return false;
  }
  if (!m.cell_faces || !m.cell_signs || !m.face_cells || !m.face_dists ||
      !m.face_nodes || !m.face_n || !m.face_L || !m.node_type ||
      (K > 0 && (!m.node_cells || !m.node_dists)) || !m.node_rho || !m.node_vel) {
    err = "mesh descriptor has a null array";
    return false;
  }
  if (C > kIndexMask || F > kIndexMask || N > kIndexMask) {
    err = "mesh too large for 30-bit indices";
    return false;
  }
  const T *fd = static_cast<const T *>(m.face_dists);
  const T *fn = static_cast<const T *>(m.face_n);
  const T *fL = static_cast<const T *>(m.face_L);
  const T *nd = static_cast<const T *>(m.node_dists);
  const T *nrho = static_cast<const T *>(m.node_rho);
  const T *nvel = static_cast<const T *>(m.node_vel);

  L.C = C;
  L.F = F;
  L.N = N;
  L.K = K;

  // --- per cell-face: slot of the cell in the face stencil and the other side
  std::vector<int32_t> other(3 * (size_t)C), slot(3 * (size_t)C);
  std::vector<char> has_ghost(C, 0);
  for (int c = 0; c < C; ++c) {
    for (int k = 0; k < 3; ++k) {
      int fid = m.cell_faces[3 * c + k];
      if (fid < 0 || fid >= F) {
        err = "cells.face_indices out of range at cell " + std::to_string(c);
        return false;
      }
      int s = m.cell_signs[3 * c + k];
      if (s < -1 || s > 1) {
        err = "cells.face_normals must hold signs in {-1,0,1}";
        return false;
      }
      int a = m.face_cells[2 * fid], b = m.face_cells[2 * fid + 1];
      if (a < -1 || a >= C || b < -1 || b >= C) {
        err = "faces.stencil_cells_index out of range at face " + std::to_string(fid);
        return false;
      }
      int sl, o;
      if (a == c && b != c) {
        sl = 0;
        o = b;
      } else if (b == c && a != c) {
        sl = 1;
        o = a;
      } else {
        err = "cell " + std::to_string(c) + " is not in the stencil of its face " +
              std::to_string(fid);
        return false;
      }
      slot[3 * c + k] = sl;
      other[3 * c + k] = o;
      if (o == -1) {
        has_ghost[c] = 1;
        int p = m.face_nodes[2 * fid], r = m.face_nodes[2 * fid + 1];
        if (p < 0 || p >= N || r < 0 || r >= N) {
          err = "faces.nodes_index out of range at face " + std::to_string(fid);
          return false;
        }
      }
    }
  }

  // --- cell order
  std::vector<int32_t> perm(C);
  if (reorder < 0 || reorder > 4) {
    err = "reorder must be 0, 1, 2, 3 or 4";
    return false;
  }
  if (reorder >= 3 && !m.cell_xy) {
    err = "reorder 3/4 (Hilbert order) needs cell centroids (cell_xy)";
    return false;
  }
  if (reorder == 0) {
    std::iota(perm.begin(), perm.end(), 0);
  } else if (reorder >= 3) {
    perm = hilbert_order(C, m.cell_xy);
    if (reorder == 3)
      std::stable_partition(perm.begin(), perm.end(),
                            [&](int32_t c) { return has_ghost[c] != 0; });
  } else {
    std::vector<int32_t> xadj(C + 1, 0), adj;
    adj.reserve(3 * (size_t)C);
    for (int c = 0; c < C; ++c) {
      for (int k = 0; k < 3; ++k)
        if (other[3 * c + k] >= 0) adj.push_back(other[3 * c + k]);
      xadj[c + 1] = (int32_t)adj.size();
    }
    perm = reverse_cuthill_mckee(C, xadj, adj);
    if (reorder == 1) {
      std::stable_partition(perm.begin(), perm.end(),
                            [&](int32_t c) { return has_ghost[c] != 0; });
    }
  }
  const int pad = tile > 0 ? tile : 1;
  // device slots: cases (if any) grouped and tile-aligned, holes = -1
  if (cell_case) {
    if (ncases < 1) {
      err = "ncases must be >= 1";
      return false;
    }
    for (int c = 0; c < C; ++c)
      if (cell_case[c] < 0 || cell_case[c] >= ncases) {
        err = "cell case id out of range at cell " + std::to_string(c);
        return false;
      }
    for (int c = 0; c < C; ++c)
      for (int k = 0; k < 3; ++k)
        if (other[3 * c + k] >= 0 && cell_case[other[3 * c + k]] != cell_case[c]) {
          err = "a face joins cells of different cases";
          return false;
        }
    std::stable_sort(perm.begin(), perm.end(),
                     [&](int32_t a, int32_t b) { return cell_case[a] < cell_case[b]; });
  }
  L.ncases = cell_case ? ncases : 1;
  L.new_to_old.clear();
  L.case_tile_off.assign(L.ncases + 1, 0);
  {
    size_t i = 0;
    for (int k = 0; k < L.ncases; ++k) {
      L.case_tile_off[k] = (int32_t)(L.new_to_old.size() / pad);
      while (i < perm.size() && (!cell_case || cell_case[perm[i]] == k))
        L.new_to_old.push_back(perm[i++]);
      while (L.new_to_old.size() % pad) L.new_to_old.push_back(-1);
    }
    L.case_tile_off[L.ncases] = (int32_t)(L.new_to_old.size() / pad);
  }
  L.Cp = (int)L.new_to_old.size();
  const size_t Cp = (size_t)L.Cp;
  L.old_to_new.assign(C, 0);
  for (size_t i = 0; i < Cp; ++i)
    if (L.new_to_old[i] >= 0) L.old_to_new[L.new_to_old[i]] = (int32_t)i;
  L.n_bcells = 0;
  for (int c = 0; c < C; ++c) L.n_bcells += has_ghost[c];
  L.last_cell_new = L.old_to_new[C - 1];
  L.tile_count.assign(Cp / pad, 0);
  L.tile_case.assign(Cp / pad, 0);
  for (size_t i = 0; i < Cp; ++i)
    if (L.new_to_old[i] >= 0) ++L.tile_count[i / pad];
  for (int k = 0; k < L.ncases; ++k)
    for (int t = L.case_tile_off[k]; t < L.case_tile_off[k + 1]; ++t) L.tile_case[t] = k;

  // --- active nodes
  std::vector<int32_t> node_an(N, -1);
  for (int i = 0; i < N; ++i) {
    int t = m.node_type[i];
    if (t == 1 || t == 2) {
      node_an[i] = (int32_t)L.an_gid.size();
      L.an_gid.push_back(i);
      L.an_type.push_back(t);
    } else if (t != 0) {
      err = "nodes.type must be 0, 1 or 2";
      return false;
    }
  }
  L.nan = (int)L.an_gid.size();
  L.an_cells.assign((size_t)L.nan * K, 0);
  L.an_w.assign((size_t)L.nan * K, T(0));
  L.an_wsum.assign(L.nan, T(0));
  L.an_rho.resize(L.nan);
  L.an_ux.resize(L.nan);
  L.an_uy.resize(L.nan);
  for (int a = 0; a < L.nan; ++a) {
    int i = L.an_gid[a];
    T wsum = T(0);
    for (int k = 0; k < K; ++k) {
      int ci = m.node_cells[(size_t)i * K + k];
      T d = nd[(size_t)i * K + k];
      // utils.extrapolate: w = 1/d, negative weights -> 0 (utils/utils.py:58-59)
      T w = T(1) / d;
      if (w < T(0)) w = T(0);
      if (ci < -1 || ci >= C) {
        err = "nodes.cells_index out of range at node " + std::to_string(i);
        return false;
      }
      L.an_cells[(size_t)a * K + k] = ci >= 0 ? L.old_to_new[ci] : -2 - L.last_cell_new;
      L.an_w[(size_t)a * K + k] = w;
      wsum += w;
    }
    L.an_wsum[a] = wsum;
    L.an_rho[a] = nrho[i];
    L.an_ux[a] = nvel[2 * (size_t)i];
    L.an_uy[a] = nvel[2 * (size_t)i + 1];
  }

  // --- per cell-face arrays in device order
  L.nb.assign(3 * Cp, 0);
  L.nx.assign(3 * Cp, T(0));
  L.ny.assign(3 * Cp, T(0));
  L.sL.assign(3 * Cp, T(0));
  L.lwa.assign(3 * Cp, T(0));
  L.lwden2.assign(3 * Cp, T(1));
  L.bf_ratio.clear();
  std::vector<int32_t> bf0, bf1, bs0, bs1;
  L.ntiles = L.Cp / pad;
  L.tile_node_off.assign(L.ntiles + 1, 0);
  L.tile_nodes.clear();
  std::vector<int32_t> slot_of(N, -1);  // node -> slot in the current tile table
  std::vector<int32_t> touched;
  int cur_tile = -1;
  auto tile_slot = [&](int node) {
    if (slot_of[node] < 0) {
      slot_of[node] = (int32_t)(L.tile_nodes.size() - L.tile_node_off[cur_tile]);
      L.tile_nodes.push_back(node_an[node] >= 0 ? node_an[node] : -1 - node);
      touched.push_back(node);
    }
    return slot_of[node];
  };
  int bw = 0;
  for (int i = 0; i < (int)Cp; ++i) {
    const int t = i / pad;
    while (cur_tile < t) {  // close the previous tile's node table
      for (int nd_ : touched) slot_of[nd_] = -1;
      touched.clear();
      ++cur_tile;
      L.tile_node_off[cur_tile] = (int32_t)L.tile_nodes.size();
    }
    const int c = L.new_to_old[i];
    if (c < 0) continue;  // hole
    for (int k = 0; k < 3; ++k) {
      int fid = m.cell_faces[3 * c + k];
      int sl = slot[3 * c + k], o = other[3 * c + k];
      size_t at = (size_t)k * Cp + i;
      T d0 = fd[2 * (size_t)fid], d1 = fd[2 * (size_t)fid + 1];
      L.nx[at] = fn[2 * (size_t)fid];
      L.ny[at] = fn[2 * (size_t)fid + 1];
      L.sL[at] = T(m.cell_signs[3 * c + k]) * fL[fid];
      T s = d0 + d1;
      L.lwa[at] = d0 / s;
      L.lwden2[at] = T(2) * s;
      int32_t code;
      if (o >= 0) {
        int j = L.old_to_new[o];
        code = j;
        bw = std::max(bw, std::abs(j - i));
      } else {
        int bf = (int)L.bf_ratio.size();
        // ghost distance / known distance: (d1/d0) when the cell is slot 0
        L.bf_ratio.push_back(sl == 0 ? d1 / d0 : d0 / d1);
        int p = m.face_nodes[2 * (size_t)fid], r = m.face_nodes[2 * (size_t)fid + 1];
        bf0.push_back(p);
        bf1.push_back(r);
        bs0.push_back(tile_slot(p));
        bs1.push_back(tile_slot(r));
        code = kGhostBit | bf;
      }
      if (sl == 1) code |= kSlot1Bit;
      L.nb[at] = code;
    }
  }
  while (cur_tile < L.ntiles - 1) {
    ++cur_tile;
    L.tile_node_off[cur_tile] = (int32_t)L.tile_nodes.size();
  }
  L.tile_node_off[L.ntiles] = (int32_t)L.tile_nodes.size();
  L.max_tile_nodes = 0;
  for (int t = 0; t < L.ntiles; ++t)
    L.max_tile_nodes = std::max(L.max_tile_nodes, L.tile_node_off[t + 1] - L.tile_node_off[t]);
  // (node, cell) pairs per tile table entry
  L.tile_pair_off.assign(L.ntiles + 1, 0);
  L.entry_pair_off.assign(L.tile_nodes.size() + 1, 0);
  L.pair_cell.clear();
  L.pair_w.clear();
  L.max_tile_pairs = 0;
  for (int t = 0; t < L.ntiles; ++t) {
    L.tile_pair_off[t] = (int32_t)L.pair_cell.size();
    for (int e = L.tile_node_off[t]; e < L.tile_node_off[t + 1]; ++e) {
      L.entry_pair_off[e] = (int32_t)L.pair_cell.size();
      const int an = L.tile_nodes[e];
      if (an < 0) continue;
      for (int k = 0; k < K; ++k) {
        const int32_t cj = L.an_cells[(size_t)an * K + k];
        const T w = L.an_w[(size_t)an * K + k];
        if (cj < 0 && w == T(0)) continue;
        L.pair_cell.push_back(cj);
        L.pair_w.push_back(w);
      }
    }
    L.max_tile_pairs =
        std::max(L.max_tile_pairs, (int)L.pair_cell.size() - L.tile_pair_off[t]);
  }
  L.tile_pair_off[L.ntiles] = (int32_t)L.pair_cell.size();
  L.entry_pair_off[L.tile_nodes.size()] = (int32_t)L.pair_cell.size();
  // halos and LDS-slot codes
  L.halo_off.assign(L.ntiles + 1, 0);
  L.halo_cells.clear();
  L.nb_slot = L.nb;
  L.max_halo = 0;
  {
    std::vector<int32_t> h;
    for (int t = 0; t < L.ntiles; ++t) {
      L.halo_off[t] = (int32_t)L.halo_cells.size();
      const int lo = t * pad, hi = t * pad + L.tile_count[t];
      h.clear();
      for (int k = 0; k < 3; ++k)
        for (int i = lo; i < hi; ++i) {
          const int32_t code = L.nb[(size_t)k * Cp + i];
          if (code < 0) continue;
          const int j = code & kIndexMask;
          if (j < lo || j >= t * pad + pad) h.push_back(j);
        }
      std::sort(h.begin(), h.end());
      h.erase(std::unique(h.begin(), h.end()), h.end());
      L.halo_cells.insert(L.halo_cells.end(), h.begin(), h.end());
      L.max_halo = std::max(L.max_halo, (int)h.size());
      for (int k = 0; k < 3; ++k)
        for (int i = lo; i < hi; ++i) {
          int32_t &code = L.nb_slot[(size_t)k * Cp + i];
          if (code < 0) continue;
          const int j = code & kIndexMask;
          int slot;
          if (j >= t * pad && j < t * pad + pad) {
            slot = j - t * pad;
          } else {
            slot = pad + (int)(std::lower_bound(h.begin(), h.end(), j) - h.begin());
          }
          code = (code & ~kIndexMask) | slot;
        }
    }
    L.halo_off[L.ntiles] = (int32_t)L.halo_cells.size();
  }
  L.nbf = (int)L.bf_ratio.size();
  L.bf_gnode.resize(2 * (size_t)L.nbf);
  L.bf_slot.resize(2 * (size_t)L.nbf);
  std::copy(bf0.begin(), bf0.end(), L.bf_gnode.begin());
  std::copy(bf1.begin(), bf1.end(), L.bf_gnode.begin() + L.nbf);
  std::copy(bs0.begin(), bs0.end(), L.bf_slot.begin());
  std::copy(bs1.begin(), bs1.end(), L.bf_slot.begin() + L.nbf);
  L.bandwidth = bw;

  // --- faces in reference order (for the flux observable)
  L.fc0.resize(F);
  L.fc1.resize(F);
  L.fn0.resize(F);
  L.fn1.resize(F);
  L.fd0.resize(F);
  L.fd1.resize(F);
  L.fnx.resize(F);
  L.fny.resize(F);
  L.fL.resize(F);
  for (int j = 0; j < F; ++j) {
    int a = m.face_cells[2 * j], b = m.face_cells[2 * j + 1];
    if (a < -1 || a >= C || b < -1 || b >= C) {
      err = "faces.stencil_cells_index out of range at face " + std::to_string(j);
      return false;
    }
    int p = m.face_nodes[2 * j], r = m.face_nodes[2 * j + 1];
    if (p < 0 || p >= N || r < 0 || r >= N) {
      err = "faces.nodes_index out of range at face " + std::to_string(j);
      return false;
    }
    L.fc0[j] = a >= 0 ? L.old_to_new[a] : -1;
    L.fc1[j] = b >= 0 ? L.old_to_new[b] : -1;
    L.fn0[j] = p;
    L.fn1[j] = r;
    L.fd0[j] = fd[2 * (size_t)j];
    L.fd1[j] = fd[2 * (size_t)j + 1];
    L.fnx[j] = fn[2 * (size_t)j];
    L.fny[j] = fn[2 * (size_t)j + 1];
    L.fL[j] = fL[j];
  }
  return true;
}

template bool build_layout<float>(const fvdbm_mesh_desc &, int, int, HostLayout<float> &,
                                  std::string &, const int32_t *, int);
template bool build_layout<double>(const fvdbm_mesh_desc &, int, int, HostLayout<double> &,
                                   std::string &, const int32_t *, int);

}  // namespace fvdbm

// Host-only entry point (no device needed): the device cell order and layout
// statistics the library would use for this mesh.
extern "C" int fvdbm_layout_order(const fvdbm_mesh_desc *mesh, int32_t precision,
                                  int32_t reorder, int32_t *new_to_old, int32_t *stats) {
  if (!mesh || !new_to_old || !stats) return FVDBM_ERR_INVALID;
  std::string err;
  if (precision == FVDBM_FP64) {
    fvdbm::HostLayout<double> L;
    if (!fvdbm::build_layout<double>(*mesh, reorder, 1, L, err)) return FVDBM_ERR_INVALID;
    std::copy(L.new_to_old.begin(), L.new_to_old.end(), new_to_old);
    stats[0] = L.n_bcells; stats[1] = L.nbf; stats[2] = L.nan; stats[3] = L.bandwidth;
  } else {
    fvdbm::HostLayout<float> L;
    if (!fvdbm::build_layout<float>(*mesh, reorder, 1, L, err)) return FVDBM_ERR_INVALID;
    std::copy(L.new_to_old.begin(), L.new_to_old.end(), new_to_old);
    stats[0] = L.n_bcells; stats[1] = L.nbf; stats[2] = L.nan; stats[3] = L.bandwidth;
  }
  return FVDBM_OK;
}
