// Multi-step tiles (k_multi): one launch advances a tile of cells by up to
// eight steps, for any lattice, with the host code that chooses the rings,
// groups the tiles into launches and runs them. Used by the D2Q9 handles
// (fvdbm_step.hip) and the any-lattice handles (fvdbm_lattice.hip); also the
// LDS cell records and face records that their one-step kernels share.
//
// A lattice is a type `Lat` with
//   Value, Q            working precision, velocities
//   Consts              lattice constants, with invtau and dt
//   threads, waves<SCHEME>()  most threads per block, and waves per SIMD that
//                       k_multi's registers are bounded for (see WIDE)
//   state(k, f, rho, ux, uy, feq)        moments and equilibrium of a cell
//   equilibrium_lane(k, q, rho, ux, uy)  component q of equilibrium, for a
//                       lane that holds one q, bit for bit the same
//   normal_speeds(nx, ny, phi)           ksi.n
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <utility>
#include <vector>

#include "errors.h"
#include "fvdbm.h"
#include "layout.h"

namespace fvdbm {

#define MULTI_TRY(expr)                                                                           \
  do {                                                                                            \
    hipError_t e_ = (expr);                                                                       \
    if (e_ != hipSuccess)                                                                         \
      return set_error(FVDBM_ERR_HIP, std::string(#expr ": ") + hipGetErrorString(e_));           \
  } while (0)

// ----------------------------------------------------------------------------
// raw buffer access: 32-bit per-lane byte offsets plus a uniform (SGPR)
// offset; loads past num_records return 0 and stores past it are dropped
// ----------------------------------------------------------------------------
constexpr int32_t kRsrcWord3 = 0x00020000;  // gfx9-family raw buffer descriptor

struct Buf {
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ Buf(const void *p, uint32_t bytes)
      : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes,
                                            kRsrcWord3)) {}
  template <typename T>
  __device__ __forceinline__ T ld(uint32_t voff, uint32_t soff) const;
  template <typename T>
  __device__ __forceinline__ void st(T v, uint32_t voff, uint32_t soff) const;
  __device__ __forceinline__ uint4 ld128(uint32_t voff, uint32_t soff) const {
    auto v = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
    return make_uint4(v[0], v[1], v[2], v[3]);
  }
};
template <>
__device__ __forceinline__ float Buf::ld<float>(uint32_t voff, uint32_t soff) const {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}
template <>
__device__ __forceinline__ double Buf::ld<double>(uint32_t voff, uint32_t soff) const {
  auto v = __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0);
  return __builtin_bit_cast(double, v);
}
template <>
__device__ __forceinline__ int32_t Buf::ld<int32_t>(uint32_t voff, uint32_t soff) const {
  return (int32_t)__builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0);
}
template <>
__device__ __forceinline__ void Buf::st<float>(float v, uint32_t voff, uint32_t soff) const {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, voff, soff, 0);
}
template <>
__device__ __forceinline__ void Buf::st<double>(double v, uint32_t voff, uint32_t soff) const {
  using v2u = decltype(__builtin_amdgcn_raw_buffer_load_b64(r, 0, 0, 0));
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, v), r, voff, soff, 0);
}

// LDS cell records: a cell's Q pdfs, read and written one value at a time, of
// Q values with an odd stride in 32-bit words (9 or 13 for FP32; FP64 records
// are 18 or 26 words whose even start banks, with each value's second word,
// cover all 32 banks), so the records that 32 lanes read at scattered slots
// spread over all LDS banks. A 12-word stride (16-byte aligned records) used
// only a quarter of the banks: 4-way conflicts.
template <typename T, int Q = 9>
struct LdsCell {
  static constexpr int W = Q;  // values per cell record
  __device__ static __forceinline__ void put(T *base, int slot, const T (&f)[Q]) {
    T *d = base + slot * W;
#pragma unroll
    for (int q = 0; q < Q; ++q) d[q] = f[q];
  }
  __device__ static __forceinline__ void get(const T *base, int slot, T (&f)[Q]) {
    const T *d = base + slot * W;
#pragma unroll
    for (int q = 0; q < Q; ++q) f[q] = d[q];
  }
};

// The value `bytes` after p, which is the same for all lanes: the access adds a
// 32-bit offset to a scalar address, and takes no vector instruction for it
// (the empty asm keeps the compiler from forming the sums per lane).
template <typename V>
using Global = __attribute__((address_space(1))) V;
template <typename V>
__device__ __forceinline__ Global<V> *at(V *p, uint32_t bytes) {
  Global<char> *g = (Global<char> *)p;
  asm("" : "+s"(g));
  return (Global<V> *)(g + bytes);
}
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// One face of one cell: neighbour code, face normal, sign * length.
// FP32: one 16-byte record; FP64: two 16-byte records (code, pad, nx | ny, sL).
template <typename T>
struct FaceRec {
  int32_t code;
  T nx, ny, sL;
};
template <typename T>
struct GeoLayout;
template <>
struct GeoLayout<float> {
  static constexpr uint32_t bytes = 16;
  __device__ static __forceinline__ FaceRec<float> load(const Buf &b, uint32_t vo, uint32_t so) {
    const uint4 v = b.ld128(vo, so);
    return {(int32_t)v.x, __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w)};
  }
  __device__ static __forceinline__ FaceRec<float> load(const uint4 *g, uint32_t i) {
    const u32x4 v = *at(reinterpret_cast<const u32x4 *>(g), i * bytes);
    return {(int32_t)v[0], __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3])};
  }
};
template <>
struct GeoLayout<double> {
  static constexpr uint32_t bytes = 32;
  __device__ static __forceinline__ FaceRec<double> load(const Buf &b, uint32_t vo, uint32_t so) {
    const uint4 v0 = b.ld128(vo, so), v1 = b.ld128(vo + 16, so);
    auto d = [](uint32_t lo, uint32_t hi) {
      return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
    };
    return {(int32_t)v0.x, d(v0.z, v0.w), d(v1.x, v1.y), d(v1.z, v1.w)};
  }
  __device__ static __forceinline__ FaceRec<double> load(const uint4 *g, uint32_t i) {
    const auto *r = at(reinterpret_cast<const u32x4 *>(g), i * bytes);
    const u32x4 v0 = r[0], v1 = r[1];
    auto d = [](uint32_t lo, uint32_t hi) {
      return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
    };
    return {(int32_t)v0[0], d(v0[2], v0[3]), d(v1[0], v1[1]), d(v1[2], v1[3])};
  }
};

// Padded cells up to which single handles take multi-step tiles of 64 (see
// choose_rings): a tile per CU.
constexpr int kSmallTileCells = 16384;

// Multi-step tiles (k_multi): the tables of HostRings (layout.h). Every face
// record names its neighbour by a stage slot: own cells 0 .. tile-1, the
// tile's ring from `tile`, then one ghost record per ghost face.
template <typename Lat>
struct MultiArgs {
  using T = typename Lat::Value;
  const T *fsrc;  // [Q][Cp]
  T *fdst;        // [Q][Cp]
  // batched solves: the two pdf buffers and per-case parity, mask, parameters
  T *f0, *f1;
  const int32_t *__restrict__ case_active, *__restrict__ case_cur;
  const T *__restrict__ case_invtau, *__restrict__ case_dt;
  const int32_t *__restrict__ meta;        // [grid][kRingMeta] of each block's tile, tile -1 = none
  const int32_t *__restrict__ slots;       // [grid][threads] device cell of each thread's stage slot, -1 = none
  const int32_t *__restrict__ ring_cells;
  const uint4 *geo;                        // [3][Cp] face records, codes for the cell's own tile
  const int32_t *__restrict__ rg_code;     // [3][nrg] codes of the updated ring cells
  const T *__restrict__ lwa, *__restrict__ lwden2;        // [3][Cp] (Lax-Wendroff)
  const int32_t *__restrict__ fan_own, *__restrict__ rg_fan;  // [Cp], [nrg]
  const int32_t *__restrict__ extra;       // (stage slot, fan record) pairs
  const int32_t *__restrict__ entries, *__restrict__ entry_pair;
  const int32_t *__restrict__ pair_fan;
  const T *__restrict__ pair_w;
  const int32_t *__restrict__ an_type;
  const T *__restrict__ an_wsum, *__restrict__ an_rho, *__restrict__ an_ux, *__restrict__ an_uy;
  const T *__restrict__ node_pdf;          // [Q][N]
  const int32_t *__restrict__ gh_s0, *__restrict__ gh_s1, *__restrict__ gh_self;
  const T *__restrict__ gh_ratio;
  int batch, bstep;                        // launch index within the batch interval
  int Cp, N;
  int nrg;                                 // updated ring cells of all tiles
  int tile;                                // cells per tile (threads per block: at least as many)
  int rows, pairs, fans, ghosts, extras;   // LDS partition
  typename Lat::Consts k;
};

// The Q pdfs of cell c from a q-major [Q][Cp] buffer, for cells whose index is
// known to lie in [0, Cp): a multi-step tile's own cells and its ring cells (ids
// the layout builder made). On the 1M-cell channel a two-step form of k_multi
// ran 1-2% faster this way than with buffer loads at nine per-plane scalar
// offsets (same results bit for bit).
template <typename T, int Q>
__device__ __forceinline__ void load_cell_at(const T *__restrict__ f, size_t Cp, int c, T (&out)[Q]) {
#pragma unroll
  for (int q = 0; q < Q; ++q) out[q] = *at(f + (size_t)q * Cp, (uint32_t)c * (uint32_t)sizeof(T));
}

// x / y for a lattice constant y with r = RN(1/y) and l = RN(1/y - r): RN(x r
// + RN(x l)), two operations. It is the IEEE quotient for each constant of D2Q9
// and of D2Q13 (tests/test_constant_division.py: in FP32 by trial of every
// significand, in FP64 by trial of those that come near a rounding boundary) and
// every x whose biased exponent lies in [51, 251] in FP32, [128, 2000] in FP64,
// and +0 for x = +0.
__device__ __forceinline__ float fast_div(float x, float r, float l) { return __builtin_fmaf(x, r, x * l); }
__device__ __forceinline__ double fast_div(double x, double r, double l) { return __builtin_fma(x, r, x * l); }

// r and l of a constant
template <typename T>
void reciprocal_of(T y, T &r, T &l) {
  r = T(1) / y;
  l = std::fma(-r, y, T(1)) / y;  // the FMA is exact
}

// a / r and b / r of one divisor: its reciprocal by the hardware estimate and
// Newton steps (one, FP64 two), then FMA corrections per quotient (two, FP64
// one; Markstein). These are the operations of the compiler's IEEE division but
// for its scaling of operands near the ends of the exponent range: the same
// quotients for r in [2^-32, 2^32] and a, b zero or of at least 2^-70.
__device__ __forceinline__ void fast_quotients(float r, float &a, float &b) {
  const float y0 = __builtin_amdgcn_rcpf(r);
  const float y = __builtin_fmaf(__builtin_fmaf(-r, y0, 1.0f), y0, y0);
  auto quotient = [&](float x) {
    float q = x * y;
    q = __builtin_fmaf(__builtin_fmaf(-r, q, x), y, q);
    return __builtin_fmaf(__builtin_fmaf(-r, q, x), y, q);
  };
  a = quotient(a);
  b = quotient(b);
}
__device__ __forceinline__ void fast_quotients(double r, double &a, double &b) {
  double y = __builtin_amdgcn_rcp(r);
  y = __builtin_fma(y, __builtin_fma(-r, y, 1.0), y);
  y = __builtin_fma(y, __builtin_fma(-r, y, 1.0), y);
  auto quotient = [&](double x) {
    const double q = x * y;
    return __builtin_fma(__builtin_fma(-r, q, x), y, q);
  };
  a = quotient(a);
  b = quotient(b);
}

// r in [2^-32, 2^32]
__device__ __forceinline__ bool plain_divisor(float r) {
  return __float_as_uint(r) - 0x2f800000u <= 0x20000000u;
}
__device__ __forceinline__ bool plain_divisor(double r) {
  return (uint32_t)__double2hiint(r) - 0x3df00000u < 0x04000000u;
}

// x / y for a lattice constant y: `fast` = uu < 1/2
template <typename T>
__device__ __forceinline__ T div_const(T x, T y, T r, T l, bool fast) {
  return fast ? fast_div(x, r, l) : x / y;
}

// Adds one face's Lax-Wendroff flux (Faces.calc_lax_wendroff_flux,
// src/containers.py:242-278) to acc: the value at the face is fu + (fd - fu) *
// interp with interp = la - (phi * dt) / den2, upstream the cell in slot 0.
// phi holds ksi.n. Opposite velocities have exactly opposite phi, so their
// quotients are exact negatives: one division per pair (q, q + 2) instead of
// one per q (ksi = 0 has phi = +0, whose quotient is +0), in k_multi loop
// invariants: 12 registers instead of 27. FP32 80k-cell cavity 4.15 -> 3.95 us
// per step; FP64 40k / 100k cells, which spilled, 11.4 / 25.2 -> 5.2 / 8.2.
template <typename T, int Q>
__device__ __forceinline__ void lax_wendroff_flux(const T (&f)[Q], const T (&o)[Q], bool slot1,
                                                  const T (&phi)[Q], T sL, T la, T den2, T dt,
                                                  T (&acc)[Q]) {
  auto add = [&](int q, T interp) {
    const T fu = slot1 ? o[q] : f[q];
    const T fd = slot1 ? f[q] : o[q];
    acc[q] += ((fu + (fd - fu) * interp) * phi[q]) * sL;
  };
  add(0, la);
#pragma unroll
  for (int q = 1; q < Q; ++q) {
    if ((q - 1) & 2) continue;  // 3, 4, 7, 8, 11, 12: the second of a pair
    const T c = (phi[q] * dt) / den2;
    add(q, la - c);
    add(q + 2, la + c);
  }
}

// Has these values computed here. Without it the one-step kernels in FP64, whose
// equilibrium branches, leave all fluxes behind the last face's gather, with three
// faces' neighbours in registers, and spill 2 to 201 of them. us per step at 260k
// cells before the branch, with it, and so: D2Q9 15.6, 15.6, 15.1, Lax-Wendroff
// 20.3, 22.1, 16.8; D2Q13 28.5, 53.9, 28.3, Lax-Wendroff 37.9, 62.3, 30.6.
template <typename T, int Q>
__device__ __forceinline__ void hold(T (&v)[Q]) {
#pragma unroll
  for (int q = 0; q < Q; ++q) asm volatile("" : "+v"(v[q]));
}

// LDS partition of k_multi, in values of the working precision: node table
// [Q][rows], fan records, then the tile's static lists (table entries, pairs,
// ghosts, extra fan cells), copied there once per launch, then the stage.
// Odd strides spread the records over the LDS banks.
constexpr int fan_words(int q) { return (q + 3) | 1; }  // rho, ux, uy, Q non-equilibrium parts
constexpr int kEntryW = 9;   // wsum, boundary rho, ux, uy, node, type, first and last pair
constexpr int kPairW2 = 2;   // weight, fan record
constexpr int kGhostW = 5;   // ratio, two table slots, stage slot of the owner
constexpr int kExtraW = 2;   // stage slot, fan record

template <int Q>
struct MultiLds {
  static constexpr int kFanW = fan_words(Q);
  int fan, entry, pair, ghost, extra, stage;
  __host__ __device__ MultiLds(int rows, int pairs, int fans, int ghosts, int extras) {
    fan = Q * rows;
    entry = fan + kFanW * fans;
    pair = entry + kEntryW * rows;
    ghost = pair + kPairW2 * pairs;
    extra = ghost + kGhostW * ghosts;
    stage = (extra + kExtraW * extras + 7) & ~7;
  }
};

// integers kept among values of the working precision
template <typename T>
__device__ __forceinline__ T from_int(int v);
template <>
__device__ __forceinline__ float from_int<float>(int v) { return __int_as_float(v); }
template <>
__device__ __forceinline__ double from_int<double>(int v) { return __hiloint2double(0, v); }
__device__ __forceinline__ int to_int(float v) { return __float_as_int(v); }
__device__ __forceinline__ int to_int(double v) { return __double2loint(v); }

// m steps of one tile (m at most the rings' depth). One thread holds one
// cell, own (thread = slot below `tile`) or ring, in registers with its face
// records; the pdfs of S_m go to the LDS stage once, then each step updates
// S_{m-1}, .., S_0 from the stage and writes them back to it, and the last
// step's own cells go to fdst: the intermediate states never go to HBM. Per
// step:
//   a. moments and equilibrium of the thread's cell; the cells that a
//      boundary node of the tile's table reads (fan cells) leave rho, u and
//      f - feq in their fan record. Fan cells outside the updated set are
//      taken by the threads after it.
//   b. node table, 16 lanes per node: lane q sums the weighted f_q - feq_q of
//      the node's cells in list order, two more lanes the moments; one
//      division per lane, then lane q forms feq_q(rho, u) + IDW(f_q - feq_q)
//      (Nodes.calc_dirichlet_pdf, src/containers.py:343-390).
//   c. ghost records, 16 lanes per ghost face (Faces.calc_ghost +
//      utils.extrap_pdf, src/containers.py:280-287, utils/utils.py:153-154):
//      fbar = mean of the two node pdfs, g = fbar + (fbar - f_owner) * ratio.
//   d. face fluxes and the cell update (phase 2 of k_step).
// a to c end with a barrier, only in tiles with boundary nodes. Every
// operation is the one k_step performs on the same operands, so the result
// equals m launches of k_step bit for bit. Batched handles: a.bstep is the
// launch index within the interval, and a frozen case's tiles return at once.
// WIDE bounds the registers only by the largest block, for launches whose tiles
// are all resident at once all the same: there a wave's own chain is the time
// (D2Q9 FP32, 2k / 60k cells: 2.80 / 3.50 -> 2.65 / 3.29 us per step), beyond
// it the waves in flight count (1M cells: 14.1 us, 17.3 with WIDE).
template <typename Lat, int SCHEME, bool WIDE>
__global__ void __launch_bounds__(Lat::template threads<SCHEME>(),
                                  WIDE ? Lat::template threads<SCHEME>() / 256 : Lat::template waves<SCHEME>()) k_multi(MultiArgs<Lat> a, int m) {
  using T = typename Lat::Value;
  constexpr int Q = Lat::Q, kFanW = fan_words(Q);
  using Cell = LdsCell<T, Q>;
  static_assert(Q + 2 <= 16, "a node's 16 lanes: Q pdfs and two moments");
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *sh = reinterpret_cast<T *>(smem_raw);
  const int32_t *__restrict__ meta = a.meta + (size_t)blockIdx.x * kRingMeta;
  const int tile = meta[kMetaTile];
  if (tile < 0) return;  // uniform per block
  const T *fsrc = a.fsrc;
  T *fdst = a.fdst;
  T invtau = a.k.invtau, dt = a.k.dt;
  if (a.batch) {  // every ring cell belongs to the tile's case
    const int cs = meta[kMetaCase];
    if (!a.case_active[cs]) return;  // uniform per block
    const int cur = (a.case_cur[cs] + a.bstep) & 1;
    fsrc = cur ? a.f1 : a.f0;
    fdst = cur ? a.f0 : a.f1;
    invtau = a.case_invtau[cs];
    dt = a.case_dt[cs];
  }
  const int bs = blockDim.x, tid = threadIdx.x;
  const MultiLds<Q> off(a.rows, a.pairs, a.fans, a.ghosts, a.extras);
  T *shf = static_cast<T *>(__builtin_assume_aligned(sh + off.stage, 16));
  const int c = a.slots[(size_t)blockIdx.x * bs + tid];  // this thread's cell
  const int ri = tid - a.tile;
  const bool own = ri < 0, live = own && c >= 0;
  T f[Q];
  if (c >= 0) load_cell_at(fsrc, (size_t)a.Cp, c, f);
  const int r0 = meta[kMetaRing], nload = meta[kMetaCells + m];
  const int nrow = meta[kMetaEntries + m - 1];
  // its face records and fan record
  const bool ring = !own && ri < meta[kMetaCells + m - 1];
  const int rf = meta[kMetaFaces] + ri;
  FaceRec<T> fr[3] = {};
  T la[3] = {}, den2[3] = {T(1), T(1), T(1)};
  int fan = -1;
  if (live || ring) {
#pragma unroll
    for (int kf = 0; kf < 3; ++kf) {
      const size_t plane = (size_t)kf * a.Cp;
      const uint32_t vo = (uint32_t)c * (uint32_t)sizeof(T);
      fr[kf] = GeoLayout<T>::load(a.geo + plane * (GeoLayout<T>::bytes / 16), (uint32_t)c);
      if (ring) fr[kf].code = *at(a.rg_code + (size_t)kf * a.nrg, 4u * (uint32_t)rf);
      if constexpr (SCHEME == 1) {
        la[kf] = *at(a.lwa + plane, vo);
        den2[kf] = *at(a.lwden2 + plane, vo);
      }
    }
    if (nrow > 0) fan = live ? a.fan_own[c] : a.rg_fan[rf];
  }
  if (c >= 0) Cell::put(shf, tid, f);  // after the requests for the face records
  for (int i = tid + bs - a.tile; i < nload; i += bs) {  // ring cells past the threads
    T g[Q];
    load_cell_at(fsrc, (size_t)a.Cp, a.ring_cells[r0 + i], g);
    Cell::put(shf, a.tile + i, g);
  }
  if (nrow > 0) {  // the tile's static lists (uniform per block)
    const int e0 = meta[kMetaEntry], p0 = meta[kMetaPair], np = meta[kMetaPairs + m - 1];
    for (int i = tid; i < nrow; i += bs) {
      T *st = sh + off.entry + kEntryW * i;
      const int e = a.entries[e0 + i];
      st[4] = from_int<T>(e);
      st[6] = from_int<T>(a.entry_pair[e0 + tile + i]);
      st[7] = from_int<T>(a.entry_pair[e0 + tile + i + 1]);
      if (e >= 0) {
        st[0] = a.an_wsum[e];
        st[1] = a.an_rho[e];
        st[2] = a.an_ux[e];
        st[3] = a.an_uy[e];
        st[5] = from_int<T>(a.an_type[e]);
      }
    }
    for (int i = tid; i < np; i += bs) {
      T *st = sh + off.pair + kPairW2 * i;
      st[0] = a.pair_w[p0 + i];
      st[1] = from_int<T>(a.pair_fan[p0 + i]);
    }
    const int g0 = meta[kMetaGhost], ng = meta[kMetaGhosts + m - 1];
    for (int i = tid; i < ng; i += bs) {
      T *st = sh + off.ghost + kGhostW * i;
      st[0] = a.gh_ratio[g0 + i];
      st[1] = from_int<T>(a.gh_s0[g0 + i]);
      st[2] = from_int<T>(a.gh_s1[g0 + i]);
      st[3] = from_int<T>(a.gh_self[g0 + i]);
    }
    const int x0 = meta[kMetaExtra], nx = meta[kMetaExtras + m];
    for (int i = tid; i < nx; i += bs) {
      T *st = sh + off.extra + kExtraW * i;
      st[0] = from_int<T>(a.extra[2 * (size_t)(x0 + i)]);
      st[1] = from_int<T>(a.extra[2 * (size_t)(x0 + i) + 1]);
    }
  }
  __syncthreads();
  const int gslot = meta[kMetaSlot];
  for (int k = m - 1;; --k) {  // this step updates S_k
    const int end = a.tile + meta[kMetaCells + k], nent = meta[kMetaEntries + k];
    const bool upd = live || (!own && tid < end);
    // a. moments, equilibrium, fan records
    bool work = upd;
    if (nent > 0) {
      const int x = meta[kMetaExtras + k], j = tid - end;
      if (!own && j >= 0 && x + j < meta[kMetaExtras + k + 1]) {
        // this thread's ring cell is not updated any more: take a fan cell
        const T *st = sh + off.extra + kExtraW * (x + j);
        Cell::get(shf, to_int(st[0]), f);
        fan = to_int(st[1]);
        work = true;
      }
    }
    T feq[Q];
    if (work) {
      T rho, ux, uy;
      Lat::state(a.k, f, rho, ux, uy, feq);
      if (nent > 0 && fan >= 0) {
        T *o = sh + off.fan + kFanW * fan;
        o[0] = rho;
        o[1] = ux;
        o[2] = uy;
#pragma unroll
        for (int q = 0; q < Q; ++q) o[3 + q] = f[q] - feq[q];
      }
    }
    if (nent > 0) {
      __syncthreads();
      // b. node table
      const int l = tid & 15;
      for (int i = tid >> 4; i < nent; i += bs >> 4) {
        const T *st = sh + off.entry + kEntryW * i;
        const int e = to_int(st[4]);
        if (e < 0) {
          if (l < Q) sh[l * nrow + i] = a.node_pdf[(size_t)l * a.N + (-1 - e)];
          continue;
        }
        const int type = to_int(st[5]), p0 = to_int(st[6]), p1 = to_int(st[7]);
        // lanes 0 .. Q-1: f_q - feq_q; Q, Q + 1: rho (type 1) or ux, uy (type 2)
        const int comp = l < Q ? 3 + l : (type == 1 ? 0 : (l == Q ? 1 : 2));
        T s = T(0);
        for (int p = p0; p < p1; p += 4) {  // four pairs' reads in flight
          T v[4], w[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const T *pr = sh + off.pair + kPairW2 * min(p + j, p1 - 1);
            const int fc = to_int(pr[1]);
            w[j] = pr[0];
            v[j] = sh[off.fan + kFanW * (fc & kIndexMask) + comp];
            if (l < Q && fc < 0) v[j] = T(0);
          }
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (p + j < p1) s += v[j] * w[j];
        }
        s = s / st[0];
        const int g = (tid & 48) + Q;
        const T s0 = __shfl(s, g, 64), s1 = __shfl(s, g + 1, 64);
        const T rho = type == 1 ? s0 : st[1], ux = type == 1 ? st[2] : s0,
                uy = type == 1 ? st[3] : s1;
        if (l < Q) sh[l * nrow + i] = Lat::equilibrium_lane(a.k, l, rho, ux, uy) + s;
      }
      __syncthreads();
      // c. ghost records
      const int ng = meta[kMetaGhosts + k];
      for (int i = tid >> 4; i < ng; i += bs >> 4) {
        if (l < Q) {
          const T *st = sh + off.ghost + kGhostW * i;
          const T *tab = sh + l * nrow;
          const T fbar = (tab[to_int(st[1])] + tab[to_int(st[2])]) / T(2);
          const T fs = shf[to_int(st[3]) * Cell::W + l];
          shf[(gslot + i) * Cell::W + l] = fbar + (fbar - fs) * st[0];
        }
      }
      __syncthreads();
    }
    // d. fluxes and update
    if (upd) {
      T acc[Q];
#pragma unroll
      for (int q = 0; q < Q; ++q) acc[q] = T(0);
#pragma unroll
      for (int kf = 0; kf < 3; ++kf) {
        const int32_t code = fr[kf].code;
        T nx = fr[kf].nx, ny = fr[kf].ny;
        const T sL = fr[kf].sL;
        // keeps the sums and doubles of a D2Q13 cell's normals out of registers
        // (100 -> 90), where they would stay over all steps: 250k cells 8.9 ->
        // 8.4 us per step. The side masks stay, in scalar registers.
        if constexpr (Q > 9) asm volatile("" : "+v"(nx), "+v"(ny));
        const bool slot1 = (code & kSlot1Bit) != 0;
        T o[Q];
        Cell::get(shf, code & kIndexMask, o);
        T phi[Q], side[Q];
        Lat::normal_speeds(nx, ny, phi);
        Lat::normal_speeds(fr[kf].nx, fr[kf].ny, side);
        if constexpr (SCHEME == 0) {
#pragma unroll
          for (int q = 1; q < Q; ++q) {
            // (+-2, 0), (0, +-2) have the signs of (+-1, 0), (0, +-1): fewer masks
            const bool take_slot0 = side[q < 9 ? q : q - 8] >= T(0);
            const T up = (take_slot0 != slot1) ? f[q] : o[q];
            const T flux = (up * phi[q]) * sL;
            acc[q] = kf == 0 ? flux : acc[q] + flux;  // 0 + x is x (but for -0, as good)
          }
        } else {
          lax_wendroff_flux(f, o, slot1, phi, sL, la[kf], den2[kf], dt, acc);
        }
      }
#pragma unroll
      for (int q = 0; q < Q; ++q) f[q] = f[q] + dt * (invtau * (feq[q] - f[q]) - acc[q]);
    }
    if (k == 0) break;
    __syncthreads();  // every input of this step has been read
    if (upd) Cell::put(shf, tid, f);
    __syncthreads();
  }
  if (live) {
#pragma unroll
    for (int q = 0; q < Q; ++q)
      *at(fdst + (size_t)q * a.Cp, (uint32_t)c * (uint32_t)sizeof(T)) = f[q];
  }
}

// LDS of a multi-step launch over a set of tiles: the kernel partitions it
// (MultiLds) with the set's largest of each list and of the stage (own, ring
// and ghost cell records).
struct PairLds {
  int rows = 0, pairs = 0, fans = 0, ghosts = 0, extras = 0, stage = 0;
  void add(const int32_t *m, int tile, int depth) {  // a tile's record, used to `depth`
    const int k = depth - 1;
    rows = std::max(rows, m[kMetaEntries + k]);
    pairs = std::max(pairs, m[kMetaPairs + k]);
    fans = std::max(fans, m[kMetaFan]);
    ghosts = std::max(ghosts, m[kMetaGhosts + k]);
    extras = std::max(extras, m[kMetaExtras + k + 1]);
    stage = std::max(stage, tile + m[kMetaCells + depth] + m[kMetaGhosts + k]);
  }
  bool covers(const PairLds &o) const {
    return rows >= o.rows && pairs >= o.pairs && fans >= o.fans && ghosts >= o.ghosts && extras >= o.extras &&
           stage >= o.stage;
  }
  template <typename T, int Q>
  size_t bytes() const {
    return ((size_t)MultiLds<Q>(rows, pairs, fans, ghosts, extras).stage + (size_t)Q * stage) * sizeof(T);
  }
};

// A handle's multi-step tiles on the device.
struct MultiTiles {
  int depth = 0, tile = 0;  // steps per launch (at most), cells per tile; 0 = none
  // launches that make up a multi-step launch (see build_classes)
  struct Class {
    int grid = 0, threads = 0;
    PairLds set;
    void *meta = nullptr, *slots = nullptr;
  };
  int nclass = 0;
  Class cls[2];
  int nrg = 0;
  bool wide = false;  // the kernel's WIDE
  bool single = false;  // takes single steps too (else the one-step kernel does, which is faster there)
  void *ring_cells = nullptr, *geo = nullptr, *rg_code = nullptr, *entries = nullptr,
       *entry_pair = nullptr, *pair_fan = nullptr, *pair_w = nullptr, *fan_own = nullptr,
       *rg_fan = nullptr, *extra = nullptr, *gh_s0 = nullptr, *gh_s1 = nullptr, *gh_self = nullptr,
       *gh_ratio = nullptr;
};

// The kernel of a lattice and scheme; one where both bounds are the same.
template <typename Lat, int SCHEME>
auto multi_kernel(bool wide) {
  constexpr bool both = Lat::template waves<SCHEME>() != Lat::template threads<SCHEME>() / 256;
  return both && !wide ? k_multi<Lat, SCHEME, !both> : k_multi<Lat, SCHEME, true>;
}

// m steps of every tile, f[src] to f[src ^ 1] (or dst). `extra` sets what the
// handle adds to the arguments.
template <typename Lat, typename H, typename Extra>
int launch_multi(const H &h, const typename Lat::Consts &k, int src, int m, void *dst, Extra extra) {
  using T = typename Lat::Value;
  const MultiTiles &M = h.multi;
  auto I = [](void *p) { return static_cast<const int32_t *>(p); };
  auto F = [](void *p) { return static_cast<const T *>(p); };
  MultiArgs<Lat> a{};
  a.fsrc = F(h.f[src]);
  a.fdst = static_cast<T *>(dst ? dst : h.f[src ^ 1]);
  a.ring_cells = I(M.ring_cells);
  a.geo = static_cast<const uint4 *>(M.geo);
  a.rg_code = I(M.rg_code);
  a.lwa = F(h.lwa);
  a.lwden2 = F(h.lwden2);
  a.fan_own = I(M.fan_own);
  a.rg_fan = I(M.rg_fan);
  a.extra = I(M.extra);
  a.entries = I(M.entries);
  a.entry_pair = I(M.entry_pair);
  a.pair_fan = I(M.pair_fan);
  a.pair_w = F(M.pair_w);
  a.an_type = I(h.an_type);
  a.an_wsum = F(h.an_wsum);
  a.an_rho = F(h.an_rho);
  a.an_ux = F(h.an_ux);
  a.an_uy = F(h.an_uy);
  a.node_pdf = F(h.node_pdf);
  a.gh_s0 = I(M.gh_s0);
  a.gh_s1 = I(M.gh_s1);
  a.gh_self = I(M.gh_self);
  a.gh_ratio = F(M.gh_ratio);
  a.Cp = h.Cp;
  a.N = h.N;
  a.nrg = M.nrg;
  a.tile = M.tile;
  a.k = k;
  extra(a);
  // the classes partition the tiles, and a tile reads only fsrc and writes
  // only its own cells of fdst: two launches are one multi-step launch
  for (int i = M.nclass - 1; i >= 0; --i) {
    const MultiTiles::Class &c = M.cls[i];
    a.meta = I(c.meta);
    a.slots = I(c.slots);
    a.rows = c.set.rows;
    a.pairs = c.set.pairs;
    a.fans = c.set.fans;
    a.ghosts = c.set.ghosts;
    a.extras = c.set.extras;
    const size_t lds = c.set.template bytes<T, Lat::Q>();
    auto fn = h.scheme == FVDBM_UPWIND ? multi_kernel<Lat, 0>(M.wide) : multi_kernel<Lat, 1>(M.wide);
    hipLaunchKernelGGL(fn, dim3(c.grid), dim3(c.threads), lds, h.stream, a, m);
    MULTI_TRY(hipGetLastError());
  }
  return FVDBM_OK;
}

// Runs of a handle with multi-step tiles; launch(src, m) makes one launch of m
// steps from f[src]. A captured run of `launches` full-depth launches from
// `parity` (cached per (parity, launches)); *out is its executable graph.
template <typename H, typename Launch>
int ensure_graph2(H &h, int parity, int launches, hipGraphExec_t *out, Launch launch) {
  const auto key = std::make_pair(parity, launches);
  auto it = h.graphs2.find(key);
  if (it != h.graphs2.end()) {
    *out = it->second.second;
    return FVDBM_OK;
  }
  MULTI_TRY(hipStreamBeginCapture(h.stream, hipStreamCaptureModeThreadLocal));
  int src = parity;
  int rc = FVDBM_OK;
  for (int s = 0; s < launches && rc == FVDBM_OK; ++s) {
    rc = launch(src, h.multi.depth);
    src ^= 1;
  }
  hipGraph_t g = nullptr;
  hipError_t e = hipStreamEndCapture(h.stream, &g);
  if (rc) {
    if (g) (void)hipGraphDestroy(g);
    return rc;
  }
  if (e != hipSuccess) return set_error(FVDBM_ERR_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
  hipGraphExec_t x = nullptr;
  e = hipGraphInstantiate(&x, g, nullptr, nullptr, 0);
  if (e != hipSuccess) {
    (void)hipGraphDestroy(g);
    return set_error(FVDBM_ERR_HIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
  }
  h.graphs2[key] = std::make_pair(g, x);
  *out = x;
  return FVDBM_OK;
}

// `launches` full-depth launches from f[h.cur]: captured runs of
// graph_steps / 2 launches, then one captured run for the rest (a single launch
// goes direct). With dry, nothing is launched and only the graphs such a run
// would replay are built (so a timed run captures nothing).
template <typename H, typename Launch>
int run_multi_launches(H &h, int64_t launches, bool dry, Launch launch) {
  int cur = h.cur;
  const int per = h.graph_steps >= 2 ? h.graph_steps / 2 : 0;
  hipGraphExec_t x = nullptr;
  while (per > 0 && launches > 0) {
    const int nl = (int)std::min<int64_t>(launches, per);
    if (nl < 2) break;
    int rc = ensure_graph2(h, cur, nl, &x, launch);
    if (rc) return rc;
    if (!dry) {
      MULTI_TRY(hipGraphLaunch(x, h.stream));
      h.steps += (int64_t)h.multi.depth * nl;
    }
    cur ^= nl & 1;
    launches -= nl;
  }
  for (; launches > 0; --launches) {
    if (!dry) {
      int rc = launch(cur, h.multi.depth);
      if (rc) return rc;
      h.steps += h.multi.depth;
    }
    cur ^= 1;
  }
  if (!dry) h.cur = cur;
  return FVDBM_OK;
}

// n steps as multi-step launches, the shorter one (n % depth steps) first.
template <typename H, typename Launch>
int run_multi(H &h, int64_t n, bool dry, Launch launch) {
  const int cur0 = h.cur, first = (int)(n % h.multi.depth);
  if (first > 0) {
    if (!dry) {
      const int rc = launch(h.cur, first);
      if (rc) return rc;
      h.steps += first;
    }
    h.cur ^= 1;
  }
  const int rc = run_multi_launches(h, n / h.multi.depth, dry, launch);
  if (dry) {
    h.cur = cur0;
    return rc;
  }
  if (rc) return rc;
  h.back = n >= h.multi.depth ? h.multi.depth : first;
  h.mid_ready = false;
  return FVDBM_OK;
}

// Threads of a block that works on n cells: whole rounds of one wave per
// SIMD. A block of 5-7 waves leaves SIMDs unevenly filled: 448 threads took
// 16.7 us per step where 512 took 15.3 (1M-cell channel, 3 steps per launch).
inline int round_threads(int n) { return n <= 64 ? 64 : n <= 128 ? 128 : (n + 255) & ~255; }

// Resident blocks per CU of k_multi with these threads and LDS; 0 = unknown.
template <typename Lat>
int resident_blocks(int scheme, bool wide, int threads, size_t lds) {
  const void *fn = scheme == FVDBM_UPWIND ? reinterpret_cast<const void *>(multi_kernel<Lat, 0>(wide))
                                          : reinterpret_cast<const void *>(multi_kernel<Lat, 1>(wide));
  int nb = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, threads, lds) == hipSuccess) return nb;
  (void)hipGetLastError();  // leave no error for the next launch check to report
  return 0;
}

inline int device_attribute(hipDeviceAttribute_t what) {
  int dev = 0, v = 0;
  if (hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&v, what, dev) == hipSuccess) return v;
  (void)hipGetLastError();
  return 0;
}

// One launch over the tiles of `order` (block b: order[b], -1 = none).
template <typename T, typename H>
int add_class(H &h, const HostRings<T> &R, const std::vector<int32_t> &order) {
  MultiTiles::Class &k = h.multi.cls[h.multi.nclass++];
  k.grid = (int)order.size();
  int threads = 0;
  for (int t : order)
    if (t >= 0) {
      k.set.add(R.meta.data() + (size_t)t * kRingMeta, R.tile, R.depth);
      threads = std::max(threads, R.meta[(size_t)t * kRingMeta + kMetaThreads]);
    }
  k.threads = round_threads(threads);
  std::vector<int32_t> meta(order.size() * kRingMeta, -1), slots(order.size() * k.threads, -1);
  for (size_t b = 0; b < order.size(); ++b) {
    const int t = order[b];
    if (t < 0) continue;
    const int32_t *m = R.meta.data() + (size_t)t * kRingMeta;
    std::copy(m, m + kRingMeta, meta.data() + b * kRingMeta);
    int32_t *s = slots.data() + b * k.threads;
    for (int i = 0; i < m[kMetaCount]; ++i) s[i] = m[kMetaFirst] + i;
    const int n = std::min(m[kMetaCells + R.depth], k.threads - R.tile);
    std::copy(R.ring_cells.begin() + m[kMetaRing], R.ring_cells.begin() + m[kMetaRing] + n, s + R.tile);
  }
  const int rc = h.upload(&k.meta, meta);
  return rc ? rc : h.upload(&k.slots, slots);
}

// Blocks in XCD-aware order: block b runs on XCD b % 8 and takes the
// (b / 8)-th tile of that XCD's list, tiles with boundary nodes first; only
// tiles with pick[t] set. The list is a contiguous eighth of all tiles or, with
// per_case, of every case's, so that the cases still active when the others
// have stopped run on all XCDs; which eighth turns with the case, as the same
// eighth of every channel is its inlet. us per step, 64 porous cases with 64 /
// 16 / 2 active, without and with per_case: FP32 158 / 145 / 41 -> 154 / 46 / 12,
// FP64 369 / 350 / 95 -> 360 / 118 / 29. Batches whose tiles are all resident at
// once go without: 3 cases of 33k cells 5.2, 5.4.
template <typename T>
std::vector<int32_t> xcd_order(const HostRings<T> &R, const std::vector<char> &pick, bool per_case) {
  auto word = [&](int t, int w) { return R.meta[(size_t)t * kRingMeta + w]; };
  std::vector<int> xcd(R.ntiles);
  for (int first = 0, last; first < R.ntiles; first = last) {
    const int cs = per_case ? word(first, kMetaCase) : 0;
    last = per_case ? first + 1 : R.ntiles;
    while (last < R.ntiles && word(last, kMetaCase) == cs) ++last;
    for (int t = first; t < last; ++t) xcd[t] = (int)((8 * (int64_t)(t - first) / (last - first) + cs) % 8);
  }
  std::vector<int32_t> order[8];
  for (int pass = 0; pass < 2; ++pass)
    for (int t = 0; t < R.ntiles; ++t)
      if (pick[t] && (word(t, kMetaEntries) > 0) == (pass == 0)) order[xcd[t]].push_back(t);
  size_t longest = 0;
  for (const auto &o : order) longest = std::max(longest, o.size());
  std::vector<int32_t> bt(8 * longest, -1);
  for (int x = 0; x < 8; ++x)
    for (size_t i = 0; i < order[x].size(); ++i) bt[i * 8 + x] = order[x][i];
  return bt;
}

// The launches of a multi-step launch: one over all tiles, or, where some
// tiles need a larger block than `threads` (see choose_rings), one over those
// that fit it and one over the others. One after the other on the handle's
// stream: two streams joined by events cost 20 us per launch.
template <typename T, typename H>
int build_classes(H &h, const HostRings<T> &R, int threads, bool plain_order, bool per_case) {
  if (plain_order) {  // plain tile order
    std::vector<int32_t> order(R.ntiles);
    for (int t = 0; t < R.ntiles; ++t) order[t] = t;
    return add_class(h, R, order);
  }
  std::vector<char> light(R.ntiles), heavy(R.ntiles);
  int n_heavy = 0;
  for (int t = 0; t < R.ntiles; ++t) {
    heavy[t] = R.meta[(size_t)t * kRingMeta + kMetaThreads] > threads;
    light[t] = !heavy[t];
    n_heavy += heavy[t];
  }
  int rc = n_heavy < R.ntiles ? add_class(h, R, xcd_order(R, light, per_case)) : FVDBM_OK;
  if (!rc && n_heavy > 0) rc = add_class(h, R, xcd_order(R, heavy, per_case));
  return rc;
}

// LDS of a CU, in the granules it is allocated by, and the most a block asks for.
constexpr int kLdsGranule = 1280, kCuLdsGranules = 128;
constexpr size_t kBlockLds = 65536;

// The lists that a batch's tiles may have without being split: a launch gives
// every block the largest of each, so that a few large tiles can keep the others
// from being resident, or from fitting a block. The lists of the smallest tiles,
// 9 in 10 at least, with which the most blocks are resident, up to what the
// registers allow; those of all tiles where these are resident at once. Tiles that
// work on more than `threads` cells are split whatever their lists. Empty if 9 in
// 10 do not fit a block.
template <typename Lat, typename T>
PairLds split_lists(const HostRings<T> &R, const std::vector<int32_t> &need, int scheme, int depth, int threads,
                    int cus) {
  std::vector<std::pair<size_t, int>> own;  // LDS of each tile alone
  auto add = [&](PairLds &lds, int t) {
    lds.add(R.meta.data() + (size_t)t * kRingMeta, R.tile, depth);
    return lds.template bytes<T, Lat::Q>();
  };
  for (int t = 0; t < R.ntiles; ++t)
    if (need[t] <= threads) {
      PairLds lds;
      own.push_back({add(lds, t), t});
    }
  std::sort(own.begin(), own.end());
  std::vector<size_t> joint;  // [n]: LDS of a launch of the n + 1 smallest
  PairLds lds;
  for (const auto &o : own) joint.push_back(add(lds, o.second));
  auto resident = [](size_t b) { return kCuLdsGranules / (int)((b + kLdsGranule - 1) / kLdsGranule); };
  if (!joint.empty() && joint.back() <= kBlockLds && R.ntiles <= cus * resident(joint.back())) return lds;
  const int rounds = (R.ntiles + cus - 1) / std::max(cus, 1);  // more blocks than tiles gain nothing
  for (int r = std::min(rounds, resident_blocks<Lat>(scheme, false, threads, 0)); r > 0; --r) {
    const size_t most = std::min<size_t>(kBlockLds, (size_t)(kCuLdsGranules / r) * kLdsGranule);
    const size_t n = std::upper_bound(joint.begin(), joint.end(), most) - joint.begin();
    if (n < 0.9 * R.ntiles) continue;
    PairLds set;
    for (size_t i = 0; i < n; ++i) add(set, own[i].second);
    return set;
  }
  return PairLds();
}

// Rings in tiles of `tile` cells, for blocks of at most `most` threads, with
// by_lists split by split_lists too; see choose_rings.
template <typename Lat, typename T>
int rings_of(const fvdbm_mesh_desc &m, const HostLayout<T> &L, int scheme, int tile, int most, int cus,
             bool batch, bool by_lists, HostRings<T> &R) {
  const int tiles = L.Cp / tile;
  const bool deep = !batch && tiles <= 3 * cus;
  auto record = [&](int t) { return R.meta.data() + (size_t)t * kRingMeta; };
  auto whole_tiles = [](const int32_t *q) { return q[kMetaThreads] <= 1024; };
  // the deepest rings for which the parts of tiles are few, or that two blocks per CU
  // hold: with cells in reverse Cuthill-McKee or the mesh's order rings are far larger
  // than the tiles, and 60k cells in parts took 20.9 us per step where one step per
  // launch took 9.4 (now, at the depth that fits, 4.1)
  const double parts = deep ? std::max(1.1, 2.0 * cus / tiles) : 1.1;
  for (int depth = deep ? kMaxDepth : 4; depth >= 2 && !R.ok; depth = depth > 4 ? 4 : depth - 1)
    build_rings<T>(m, L, tile, depth, whole_tiles, parts, R);
  while (R.ok) {
    // the blocks and LDS that fewer steps of these rings need
    int best = 0, threads = 0, block2 = 0;
    bool split = false, two = false;  // large tiles are split, or take a second launch
    PairLds lists;                    // of the best
    std::vector<int32_t> need(R.ntiles, 0), chosen;
    for (int d = 2; d <= R.depth; ++d) {
      PairLds lds;
      int small = 0;  // tiles that fit a block's LDS
      for (int t = 0; t < R.ntiles; ++t) {
        const int32_t *q = record(t);
        for (int k = d == 2 ? 0 : d - 1; k < d; ++k)
          need[t] = std::max(need[t], R.tile + q[kMetaCells + k] + q[kMetaExtras + k + 1] - q[kMetaExtras + k]);
        lds.add(q, tile, d);
        PairLds own;
        own.add(q, tile, d);
        small += own.template bytes<T, Lat::Q>() <= kBlockLds;
      }
      std::vector<int32_t> order(need);
      std::sort(order.begin(), order.end());
      auto block_of = [&](double share) {  // that this share of the tiles fits
        return round_threads(order[std::min<size_t>((size_t)(share * R.ntiles), R.ntiles - 1)]);
      };
      const int whole = block_of(1.0);
      const size_t all = lds.template bytes<T, Lat::Q>();
      if (d == 2) block2 = block_of(0.9);
      if (block2 > most || (all > kBlockLds && !(by_lists && small >= 0.9 * R.ntiles))) break;
      if (all <= kBlockLds &&
          (whole <= block2 ||
           (deep && whole <= most && tiles <= cus * resident_blocks<Lat>(scheme, false, whole, all)))) {
        threads = whole;
        split = two = false;
      } else if (block_of(0.9) <= block2) {
        threads = block2;
        split = true;
        two = false;
      } else if (batch && tile == 64 && all <= kBlockLds && whole <= most && block_of(0.75) <= block2) {
        threads = block2;
        split = false;
        two = true;
      } else {
        continue;
      }
      best = d;
      lists = lds;
      chosen = need;
    }
    if (best < 2) break;
    if (by_lists && !two) {
      const PairLds set = split_lists<Lat>(R, chosen, scheme, best, threads, cus);
      if (set.stage == 0) break;
      split = split || !set.covers(lists);
      lists = set;
    }
    if (best == R.depth && !split) return threads;
    if (!split) {
      build_rings<T>(m, L, tile, best, whole_tiles, parts, R);
      continue;
    }
    // split tiles (to 32 cells at least for their lists): done, if they fit
    build_rings<T>(m, L, tile, best, [&](const int32_t *q) {
      PairLds own;
      own.add(q, tile, best);
      return q[kMetaThreads] <= threads && (q[kMetaCount] <= 32 || lists.covers(own));
    }, 1.25, R);
    PairLds lds;
    for (int t = 0; t < R.ntiles && R.ok; ++t) {
      lds.add(record(t), tile, best);
      R.ok = record(t)[kMetaThreads] <= threads;
    }
    if (lds.template bytes<T, Lat::Q>() > kBlockLds) R.ok = false;
    return threads;
  }
  R.ok = false;
  return 0;
}

// Rings of the handle's multi-step tiles: cells per tile and steps per
// launch; returns the threads of its (first) launch. Not ok where not even
// two steps fit a block.
//
// More steps per launch share one read of pdfs and face records and one
// launch, and cost a wider ring: more threads, and redundant updates. With
// every tile of a mesh resident at once a step is bound by latency and the
// deepest rings win: 60k-cell channel 4.5 (3 steps), 4.2 (4), 3.7 us per step
// (8). With several rounds of tiles, and for batches, it is the cells in
// flight that count, so the block stays at the size B that two steps need:
// the deepest rings that fit B for 9 tiles in 10, the others split in halves
// (1M-cell channel, tiles of 256, B = 512: 18.3 (2 steps), 15.3 (3), 13.8 us
// per step (4), and 20 (5) in blocks of 768; 16 porous cases 20.3 with a
// second launch for the largest tiles, 17.4 with those split).
//
// A launch gives every block the LDS of its largest tile, and a few tiles of a
// porous batch hold twice what the others do. With these split too, as many
// blocks are resident as the registers allow, and FP64 tiles fit a block at all;
// where they still do not, tiles of half the size do. All cases active, us per
// step: 64 cases of 5-40 discs, 7.4M cells, FP64 in tiles of 128 487 -> 367
// (59046 tiles for 57763), of 256 (one step per launch before, now of 128) 565 ->
// 369, FP32 in tiles of 128 184 -> 163 (57959 tiles, 5 -> 6 blocks per CU); 16
// cases of 3-8 discs, 1.8M cells, FP64 86 -> 65; 6 cases of 4k-16k cells, FP64
// 7.2 -> 5.6.
//
// Large batches take no smaller tiles than 256 cells (FP64 128), whose rings are a
// smaller part of the work, whatever the layout's: the 64 cases in FP32 with a
// layout in tiles of 64 / 128 204 / 163 -> 154; 256 cases 851 / 644 -> 616 (763 /
// 660 before multi-step tiles).
//
// A small batch in tiles of 64 takes a second launch for up to a quarter of its
// tiles instead. It is the one configuration with two launches, and no faster for
// it: splitting took the 6 cases 5.4 us per step, this takes 10.5 (the two-step
// tiles before took 16.7).
template <typename Lat, typename T>
int choose_rings(const fvdbm_mesh_desc &m, const HostLayout<T> &L, int scheme, int block, bool batch,
                 HostRings<T> &R) {
  const int most = scheme == FVDBM_UPWIND ? Lat::template threads<0>() : Lat::template threads<1>();
  // the layout's tile, or a part of it that leaves room for a ring. Small
  // meshes take tiles of 64, so that more CUs share them: 2048-cell cavity
  // 3.17 -> 2.90 us per step.
  int tile = block;
  while (tile > most / 2 && tile % 128 == 0) tile /= 2;
  // a record of 13 doubles: two blocks of 256 threads per CU run better than one
  // of 512, by registers and LDS (100k / 300k cells: 12.6 / 27.6 us per step
  // with tiles of 256, 10.7 / 23.7 with 128)
  if (Lat::Q * sizeof(T) > 72 && tile > 128) tile = tile % 128 == 0 ? 128 : 64;
  if (!batch && L.Cp <= kSmallTileCells) tile = 64;
  const int cus = device_attribute(hipDeviceAttributeMultiprocessorCount);
  // large batches: those that the GPU does not hold at once, at about 768 cells a CU
  if (batch && L.Cp > 768 * cus) tile = std::max(tile, sizeof(T) == 8 ? 128 : 256);
  if (!batch) return rings_of<Lat>(m, L, scheme, tile, most, cus, false, false, R);
  for (int part = tile;; part /= 2) {
    const int threads = rings_of<Lat>(m, L, scheme, part, most, cus, true, true, R);
    if (R.ok) return threads;
    if (part % 128 != 0) break;
  }
  return rings_of<Lat>(m, L, scheme, tile, most, cus, true, false, R);
}

// The multi-step tiles of a handle, if its rings fit. The handle uploads. They
// take single steps of meshes of up to single_cells padded cells, and of batches
// whose tiles are all resident at once.
template <typename Lat, typename H>
int build_multi(H &h, const fvdbm_mesh_desc &m, const HostLayout<typename Lat::Value> &L, bool batch,
                bool plain_order, int single_cells) {
  using T = typename Lat::Value;
  HostRings<T> R;
  const int threads = choose_rings<Lat>(m, L, h.scheme, h.block, batch, R);
  if (!R.ok) return FVDBM_OK;
  // the kernel's 32-bit offsets into a plane of face records, and of ring codes
  if ((uint64_t)L.Cp * GeoLayout<T>::bytes >= (1ull << 32) || R.rg_code.size() / 3 >= (1ull << 30)) return FVDBM_OK;
  MultiTiles &M = h.multi;
  const size_t nrg = R.rg_code.size() / 3, n3 = 3 * (size_t)L.Cp;
  std::vector<int32_t> rgc(R.rg_code.size());
  for (size_t r = 0; r < nrg; ++r)
    for (int k = 0; k < 3; ++k) rgc[(size_t)k * nrg + r] = R.rg_code[3 * r + k];
  // the codes wait in a pdf buffer for finish_multi
  MULTI_TRY(hipMemcpy(h.f[1], R.code.data(), n3 * sizeof(int32_t), hipMemcpyHostToDevice));
  int rc = h.alloc(&M.geo, n3 * GeoLayout<T>::bytes);
  if (!rc) rc = h.upload(&M.rg_code, rgc);
  if (!rc) rc = h.upload(&M.ring_cells, R.ring_cells);
  if (!rc) rc = h.upload(&M.entries, R.entries);
  if (!rc) rc = h.upload(&M.entry_pair, R.entry_pair);
  if (!rc) rc = h.upload(&M.pair_fan, R.pair_fan);
  if (!rc) rc = h.upload(&M.fan_own, R.fan_own);
  if (!rc) rc = h.upload(&M.rg_fan, R.rg_fan);
  if (!rc) rc = h.upload(&M.extra, R.extra);
  if (!rc) rc = h.upload(&M.pair_w, R.pair_w);
  if (!rc) rc = h.upload(&M.gh_s0, R.gh_s0);
  if (!rc) rc = h.upload(&M.gh_s1, R.gh_s1);
  if (!rc) rc = h.upload(&M.gh_self, R.gh_self);
  if (!rc) rc = h.upload(&M.gh_ratio, R.gh_ratio);
  if (!rc && !batch) rc = h.alloc(&h.fmid, (size_t)Lat::Q * L.Cp * sizeof(T));
  if (!rc) {
    M.depth = R.depth;
    M.tile = R.tile;
    M.nrg = (int)nrg;
    PairLds lds;
    for (int t = 0; t < R.ntiles; ++t) lds.add(R.meta.data() + (size_t)t * kRingMeta, R.tile, R.depth);
    const int at_once = device_attribute(hipDeviceAttributeMultiprocessorCount) *
                        resident_blocks<Lat>(h.scheme, false, threads, lds.template bytes<T, Lat::Q>());
    const bool waits = R.ntiles > at_once;
    M.single = batch ? !waits : L.Cp <= single_cells;
    rc = build_classes<T>(h, R, threads, plain_order, batch && waits);
    const MultiTiles::Class &c = M.cls[0];
    M.wide = M.nclass == 1 && c.grid <= device_attribute(hipDeviceAttributeMultiprocessorCount) *
                                            resident_blocks<Lat>(h.scheme, true, c.threads,
                                                                 c.set.template bytes<T, Lat::Q>());
  }
  return rc;
}

// The face records of the multi-step tiles, from their codes and from the face
// normals and lengths that the one-step kernels read: records of the same form
// (`geo`) or planes. Formed on the host and sent, they made the set-up of 80k /
// 260k cells in FP64 22.1 / 66.5 ms, so 20.8 / 63.4.
template <typename T>
__global__ void k_face_records(const int32_t *__restrict__ code, const uint4 *__restrict__ geo,
                               const T *__restrict__ nx, const T *__restrict__ ny, const T *__restrict__ sL,
                               size_t n, unsigned char *__restrict__ out) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  constexpr size_t o = sizeof(T) == 4 ? 4 : 8;
  unsigned char *d = out + i * GeoLayout<T>::bytes;
  const unsigned char *g = reinterpret_cast<const unsigned char *>(geo) + i * GeoLayout<T>::bytes;
  T v[3];
  if (geo)
    for (int k = 0; k < 3; ++k) v[k] = *reinterpret_cast<const T *>(g + o + k * sizeof(T));
  else
    v[0] = nx[i], v[1] = ny[i], v[2] = sL[i];
  *reinterpret_cast<int32_t *>(d) = code[i];
  if (o == 8) *reinterpret_cast<int32_t *>(d + 4) = 0;
  for (int k = 0; k < 3; ++k) *reinterpret_cast<T *>(d + o + k * sizeof(T)) = v[k];
}

// After build_multi, once the handle's tables are on the device.
template <typename T, typename H>
int finish_multi(H &h, const void *geo, const void *nx, const void *ny, const void *sL) {
  if (h.multi.depth == 0) return FVDBM_OK;
  const size_t n = 3 * (size_t)h.Cp;
  auto F = [](const void *p) { return static_cast<const T *>(p); };
  hipLaunchKernelGGL((k_face_records<T>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, h.stream,
                     static_cast<const int32_t *>(h.f[1]), static_cast<const uint4 *>(geo), F(nx), F(ny), F(sL), n,
                     static_cast<unsigned char *>(h.multi.geo));
  MULTI_TRY(hipGetLastError());  // the buffer's first state is written after it, on the same stream
  return FVDBM_OK;
}

#undef MULTI_TRY

}  // namespace fvdbm
