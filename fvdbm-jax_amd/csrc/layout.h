// Host-side construction of the device layout: cell renumbering (reverse
// Cuthill-McKee, cells with a ghost face first), per cell-face structure of
// arrays, boundary-face and active-node records. Pure C++ (no HIP calls), so
// it is also exercised by the CPU tests through fvdbm_layout_* helpers.
#pragma once

#include <cstdint>
#include <functional>
#include <string>
#include <vector>

#include "fvdbm.h"

namespace fvdbm {

// Bits of a cell-face code (nb array):
//   bit 31 set      : ghost face; bits 0..29 = boundary-face record index
//   bit 31 clear    : interior face; bits 0..29 = neighbour cell (device id)
//   bit 30 set      : this cell sits in stencil slot 1 of the face
constexpr int32_t kGhostBit = int32_t(0x80000000u);
constexpr int32_t kSlot1Bit = 0x40000000;
constexpr int32_t kIndexMask = 0x3fffffff;

template <typename T>
struct HostLayout {
  // C cells occupy Cp device slots; a slot whose new_to_old is -1 is a hole
  // (batched layouts start every case on a tile boundary). The live cells of
  // a tile are its first tile_count[t] slots.
  int C = 0, Cp = 0, F = 0, N = 0, K = 0;
  int ncases = 1;
  std::vector<int32_t> tile_count, tile_case, case_tile_off;
  int n_bcells = 0;   // cells with >= 1 ghost face, stored first when reorder==1
  int nbf = 0;        // boundary-face records
  int nan = 0;        // active (type 1 / 2) nodes
  int bandwidth = 0;
  int last_cell_new = 0;  // device id of reference cell C-1 (JAX's index -1)
  std::vector<int32_t> new_to_old, old_to_new;

  // per cell-face, [3][Cp]
  std::vector<int32_t> nb;
  // same codes with the neighbour given as its slot in the tile's LDS stage
  // (own cells 0..tile-1, then the tile's halo cells)
  std::vector<int32_t> nb_slot;
  // halo of each tile: distinct out-of-tile neighbour cells, ascending
  int max_halo = 0;
  std::vector<int32_t> halo_off, halo_cells;

  std::vector<T> nx, ny, sL;      // face normal, sign * L
  std::vector<T> lwa, lwden2;     // Lax-Wendroff: d0/(d0+d1), 2*(d0+d1)

  // boundary-face records: [2][nbf] endpoint slots in the owning tile's
  // node table, [2][nbf] endpoint node ids, [nbf] ghost/known distance ratio
  std::vector<int32_t> bf_slot, bf_gnode;
  std::vector<T> bf_ratio;

  // per-tile node tables (tile = `block` consecutive device cells): the
  // distinct face nodes the tile's ghost faces read, CSR over tiles.
  // entry >= 0: active-node index; < 0: -1 - node id (stored pdf)
  int ntiles = 0, max_tile_nodes = 0;
  std::vector<int32_t> tile_node_off, tile_nodes;

  // (node, cell) pairs of the active nodes in each tile table, in table
  // order and, per node, in nodes.cells_index order; padding entries with
  // weight 0 are left out (they add +0). pair_cell: device cell id, or
  // -2 - (wrapped id) for a padding entry with a non-zero weight.
  int max_tile_pairs = 0;
  std::vector<int32_t> tile_pair_off;   // [ntiles+1]
  std::vector<int32_t> entry_pair_off;  // [tile_nodes.size()+1], absolute
  std::vector<int32_t> pair_cell;
  std::vector<T> pair_w;

  // active nodes
  std::vector<int32_t> an_gid, an_type;
  std::vector<int32_t> an_cells;  // [nan][K]: device id, or -2 - (wrapped id) for padding
  std::vector<T> an_w;            // [nan][K]  1/d, negatives -> 0
  std::vector<T> an_wsum;         // [nan]     0-initialised ordered sum of an_w
  std::vector<T> an_rho, an_ux, an_uy;

  // faces in reference order (flux observable)
  std::vector<int32_t> fc0, fc1, fn0, fn1;
  std::vector<T> fd0, fd1, fnx, fny, fL;
};

// Multi-step tiles: one launch advances a tile by up to `depth` steps. With
// S_0 = the tile's cells, S_{k+1} = S_k, the face neighbours of S_k and every
// cell that a node of an S_k ghost face reads; ring level k = S_k \ S_{k-1}.
// An m-step launch reads S_m, then updates S_{m-1}, .., S_0, one step each,
// from the previous step's values of the cells one level further out: every
// operand of a step is in the tile's LDS stage. Lists are level-sorted, so
// the cells, table entries, pairs and ghosts of S_k are a prefix.
//
// Stage slots: own cells 0 .. tile-1, ring cells from `tile` (level 1 first),
// then one ghost record per ghost face of S_{depth-1} (S_0's first).
constexpr int kMaxDepth = 8;
constexpr int kRingMeta = 64;  // int32 words per tile, see below

// words of a tile's record in HostRings::meta
enum RingMeta {
  kMetaRing = 0,     // first ring cell (ring_cells)
  kMetaFaces = 1,    // first updated ring cell (rg_code, rg_fan)
  kMetaEntry = 2,    // first node-table entry
  kMetaPair = 3,     // first (node, cell) pair
  kMetaGhost = 4,    // first ghost record
  kMetaCount = 5,    // live cells of the tile
  kMetaCase = 6,     // case of the tile
  kMetaSlot = 7,     // stage slot of the first ghost record
  kMetaCells = 8,    // [k]: ring cells of levels 1 .. k, k = 0 .. kMaxDepth
  kMetaTile = 17,    // the tile
  kMetaFirst = 19,   // its first cell
  kMetaThreads = 18, // most cells (updated, or extra fan cells) that the tile works on in a step
  kMetaEntries = 20, // [k]: node-table entries of S_k, k = 0 .. kMaxDepth-1
  kMetaPairs = 28,   // [k]: pairs of those entries
  kMetaGhosts = 36,  // [k]: ghost faces of S_k
  kMetaFan = 44,     // distinct node cells (fan records) of the tile
  kMetaExtra = 45,   // first extra fan cell
  kMetaExtras = 46,  // [k]: start of S_k's extra fan cells after the first, k = 0 .. kMaxDepth
};

template <typename T>
struct HostRings {
  bool ok = false;
  int depth = 0, tile = 0, ntiles = 0;
  std::vector<int32_t> meta;        // [ntiles][kRingMeta]
  std::vector<int32_t> ring_cells;  // device ids, per tile and level
  // face codes of the cells updated with a ring (levels 1 .. depth-1),
  // [3 per cell]: stage slot of the neighbour or ghost record | slot-1 bit;
  // the faces' geometry is that of the cell's own record
  std::vector<int32_t> rg_code;
  std::vector<int32_t> code;        // [3][Cp] the own cells' codes, as rg_code
  // node table: entries (active-node index, or -1 - node id) with the pair
  // offset of each relative to the tile's first pair (one more per tile:
  // entry i of a tile has pairs [entry_pair[e], entry_pair[e + 1]) with
  // e = first entry + tile + i). A pair names its cell by the cell's fan
  // record (one per distinct cell that a table node reads).
  std::vector<int32_t> entries, entry_pair;
  std::vector<int32_t> pair_fan;    // fan record, bit 31: padding (no non-equilibrium part)
  std::vector<T> pair_w;
  std::vector<int32_t> fan_own;     // [Cp] fan record of each own cell, -1 = none
  std::vector<int32_t> rg_fan;      // the same per updated ring cell
  // fan cells that S_k's entries read outside S_k: (stage slot, fan record)
  std::vector<int32_t> extra;
  // ghost records: table slots of the face's nodes, stage slot of the
  // owning cell, ghost / known distance
  std::vector<int32_t> gh_s0, gh_s1, gh_self;
  std::vector<T> gh_ratio;
};

// Rings of the mesh laid out as L, in tiles of `tile` cells of one case (smaller or
// larger than the layout's), for at most `depth` steps per launch. A tile whose record
// does not fit is built as two halves, down to one cell; `fits` sees the record
// with all its counts at the full depth. Given up (not ok) where the parts make more
// than `most` times the tiles.
template <typename T>
void build_rings(const fvdbm_mesh_desc &m, const HostLayout<T> &L, int tile, int depth,
                 const std::function<bool(const int32_t *)> &fits, double most, HostRings<T> &out);

// `tile` is the number of cells per thread block; the cell count is padded
// to a multiple of it. With cell_case (case id of every cell, ncases cases)
// the cells are grouped by case and each case starts on a tile boundary.
template <typename T>
bool build_layout(const fvdbm_mesh_desc &m, int reorder, int tile,
                  HostLayout<T> &out, std::string &err,
                  const int32_t *cell_case = nullptr, int ncases = 1);

// Cells sorted by the Hilbert index of their centroids ([n][2]).
std::vector<int32_t> hilbert_order(int n, const double *xy);

// Reverse Cuthill-McKee over an undirected graph in CSR form.
// Returns perm with perm[new] = old.
std::vector<int32_t> reverse_cuthill_mckee(int n, const std::vector<int32_t> &xadj,
                                           const std::vector<int32_t> &adj);

}  // namespace fvdbm
