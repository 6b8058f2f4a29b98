// Inputs of the warm-start surrogate for a group of porous cases, built on the
// device: the node features and one CSR graph over all cases, as nn_inputs.cpp
// builds them for one case on the host (its header states the construction:
// mesh nodes, grid nodes and the global node of a case in consecutive rows,
// rows sorted by target). No reference counterpart; the C ABI is declared in
// include/fvdbm.h (fvdbm_nn_device_inputs). Double precision with the host
// code's operations (no contraction), so the float32 arrays are its own but
// where hypot, pow or log round differently, once in about 1e8 values.
//
// What a prediction needs of the graph is built: the lists of the forward
// pass. On the host this took 10.5 ms for 12 cases of 20k-90k cells on 16
// threads, and 5.4 ms more to join the cases and to copy 67 MB; now the
// meshes are copied (15 MB) and the kernels take 0.3 ms, most of it atomics on
// the degrees and the lists of the grid nodes.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

#include "errors.h"
#include "fvdbm.h"

namespace fvdbm_nn_graph {

constexpr int kMeta = 7;  // per case: first row, first mesh node, mesh nodes, first edge, edges, first disc, discs
constexpr int kParams = 3;  // per case: u_in, tau, column 15
constexpr int kScan = 2048;  // rows a block scans
constexpr int kMaxSection = 2048;

struct Args {
  const int32_t *meta;
  const double *params;
  const double *xy, *discs;
  const int32_t *markers, *edges;
  int ncases, rows, mesh_nodes, n_edges;
  int gx, gy, section;
  double height;
  int32_t codes[4];
  float shift[9], scale[9], sshift[4], sscale[4];
  int32_t *count, *cursor, *cell, *sums;
  float *tables;  // [ncases][3 * section + 1]: scaled columns 11-13, then column 14
  unsigned long long *error;  // least (case, kind, index) refused
  float *x;
  int32_t *off, *col;
  float *w, *ex, *ey;
};

// The case of item i by a word of the meta records (ascending firsts).
__device__ __forceinline__ int case_of(const Args &a, int word, int i) {
  int lo = 0, hi = a.ncases;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (a.meta[mid * kMeta + word] <= i) lo = mid;
    else hi = mid;
  }
  return lo;
}

__device__ __forceinline__ void refuse(const Args &a, int cs, int kind, int index) {
  atomicMin(a.error, ((unsigned long long)cs << 33) | ((unsigned long long)kind << 32) | (unsigned)index);
}

__global__ void k_clear(Args a) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < a.rows) a.count[i] = a.cursor[i] = 0;
  if (i == 0) *a.error = ~0ull;
}

// Cross-section of a case's channel on a grid of x: open fraction, hydraulic
// resistance and the share of it downstream. One block per case; the two sums
// run in index order, as on the host, each on one lane of its own wave.
__global__ __launch_bounds__(256) void k_sections(Args a) {
  __shared__ double r3[kMaxSection], run[kMaxSection];
  __shared__ double sum;
  const int32_t *m = a.meta + blockIdx.x * kMeta;
  const double *d = a.discs + 3 * (size_t)m[5];
  const int G = a.section, nd = m[6];
  float *t = a.tables + (size_t)blockIdx.x * (3 * G + 1);
  for (int i = threadIdx.x; i < G; i += blockDim.x) {
    const double xs = (i + 0.5) / G;
    double blocked = 0.0;
    for (int k = 0; k < nd; ++k) {
      const double dxs = xs - d[3 * k], r = d[3 * k + 2];
      const double d2 = r * r - dxs * dxs;
      blocked += d2 > 0.0 ? 2.0 * sqrt(d2) : 0.0;
    }
    const double v = fmin(fmax(1.0 - blocked / a.height, 0.05), 1.0);
    t[i] = ((float)v - a.sshift[0]) / a.sscale[0];
    t[G + i] = ((float)(1.0 / v) - a.sshift[1]) / a.sscale[1];
    r3[i] = 1.0 / pow(v, 3.0);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
#pragma unroll 8
    for (int i = 0; i < G; ++i) s += r3[i];
    sum = s;
  } else if (threadIdx.x == 64) {
    double s = 0.0;
#pragma unroll 8
    for (int i = G - 1; i >= 0; --i) {
      s += r3[i];
      run[i] = s;
    }
  }
  __syncthreads();
  const double total = sum / G;
  for (int i = threadIdx.x; i < G; i += blockDim.x)
    t[2 * G + i] = ((float)(run[i] / G / total) - a.sshift[2]) / a.sscale[2];
  if (threadIdx.x == 0) t[3 * G] = ((float)log(total) - a.sshift[3]) / a.sscale[3];
}

// Degrees of the mesh edges; an edge that names no two nodes of its mesh is
// refused and left out here and in k_fill.
__device__ __forceinline__ bool edge_rows(const Args &a, int e, int &u, int &v, int &cs) {
  cs = case_of(a, 3, e);
  const int32_t *m = a.meta + cs * kMeta;
  u = a.edges[2 * (size_t)e];
  v = a.edges[2 * (size_t)e + 1];
  const bool ok = u >= 0 && v >= 0 && u < m[2] && v < m[2] && u != v;
  u += m[0];
  v += m[0];
  return ok;
}

__global__ __launch_bounds__(256) void k_count(Args a) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= a.n_edges) return;
  int u, v, cs;
  if (!edge_rows(a, e, u, v, cs)) {
    refuse(a, cs, 0, e - a.meta[cs * kMeta + 3]);
    return;
  }
  atomicAdd(a.count + u, 1);
  atomicAdd(a.count + v, 1);
}

// The grid column (or row) of coordinate t = x * cells: truncated, at most
// cells - 1; -1 below the grid or beyond any integer.
__device__ __forceinline__ int grid_index(double t, int cells) {
  if (!(t > -1.0) || !(t < 9.2e18)) return -1;
  return t < cells ? (int)t : cells - 1;
}

__device__ double distance(const double *d, int nd, double px, double py) {
  double best = INFINITY;
  for (int k = 0; k < nd; ++k) best = fmin(best, hypot(px - d[3 * k], py - d[3 * k + 1]) - d[3 * k + 2]);
  return best;
}

// One thread per row: its 16 features, and the degrees of the links to grid
// nodes and the global node.
__global__ __launch_bounds__(256) void k_nodes(Args a) {
  const int row = blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= a.rows) return;
  const int cs = case_of(a, 0, row);
  const int32_t *m = a.meta + cs * kMeta;
  const double *p = a.params + cs * kParams, *discs = a.discs + 3 * (size_t)m[5];
  const int local = row - m[0], S = a.gx * a.gy, s = local - m[2];
  double px = 0.5, py = 0.25, dist = a.shift[2];
  float flags[4] = {0.f, 0.f, 0.f, 0.f}, virt = 0.f, global = 0.f;
  if (s < 0) {
    const int node = m[1] + local;
    px = a.xy[2 * (size_t)node];
    py = a.xy[2 * (size_t)node + 1];
    dist = distance(discs, m[6], px, py);
    const int mark = a.markers[node];
#pragma unroll
    for (int j = 0; j < 4; ++j) flags[j] = mark == a.codes[j] ? 1.f : 0.f;
    const int ci = grid_index(px * a.gx, a.gx), cj = grid_index(py / a.height * a.gy, a.gy);
    const int c = ci < 0 || cj < 0 ? -1 : cj * a.gx + ci;
    a.cell[node] = c;
    if (c < 0) {
      refuse(a, cs, 1, local);
    } else {
      atomicAdd(a.count + row, 1);
      atomicAdd(a.count + m[0] + m[2] + c, 1);
    }
  } else if (s < S) {
    const int i = s % a.gx, j = s / a.gx;
    px = (i + 0.5) / a.gx;
    if (a.gy > 1) {
      py = (j + 0.5) / a.gy * a.height;
      dist = distance(discs, m[6], px, py);
    }
    virt = 1.f;
    const int wide = 1 + (i > 0) + (i < a.gx - 1), high = 1 + (j > 0) + (j < a.gy - 1);
    atomicAdd(a.count + row, wide * high - 1 + 1);  // neighbours and the global node
  } else {
    global = 1.f;
    a.count[row] = S;
  }
  long long at = (long long)(px * a.section);
  at = at < 0 ? 0 : (at > a.section - 1 ? a.section - 1 : at);
  const float *t = a.tables + (size_t)cs * (3 * a.section + 1);
  auto scaled = [&](double v, int k) { return ((float)v - a.shift[k]) / a.scale[k]; };
  float4 *o = reinterpret_cast<float4 *>(a.x + 16 * (size_t)row);
  o[0] = make_float4(scaled(px, 0), scaled(py, 1), scaled(dist, 2), scaled(flags[0], 3));
  o[1] = make_float4(scaled(flags[1], 4), scaled(flags[2], 5), scaled(flags[3], 6), scaled(p[0], 7));
  o[2] = make_float4(scaled(p[1], 8), virt, global, t[at]);
  o[3] = make_float4(t[a.section + at], t[2 * a.section + at], t[3 * a.section], (float)p[2]);
}

// off = exclusive sums of count: block sums, their sums in one block, then
// each block's own rows.
__device__ __forceinline__ int block_scan(int v, int &total) {  // exclusive, 256 threads
  __shared__ int wave_sum[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int s = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int up = __shfl_up(s, d, 64);
    if (lane >= d) s += up;
  }
  if (lane == 63) wave_sum[wave] = s;
  __syncthreads();
  int before = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    if (w < wave) before += wave_sum[w];
    total += wave_sum[w];
  }
  __syncthreads();
  return before + s - v;
}

__global__ __launch_bounds__(256) void k_block_sums(Args a) {
  int v = 0, total;
  for (int i = 0; i < kScan / 256; ++i) {
    const int row = blockIdx.x * kScan + i * 256 + threadIdx.x;
    if (row < a.rows) v += a.count[row];
  }
  block_scan(v, total);
  if (threadIdx.x == 0) a.sums[blockIdx.x] = total;
}

__global__ __launch_bounds__(256) void k_scan_sums(Args a, int blocks) {
  int base = 0;
  for (int i0 = 0; i0 < blocks; i0 += 256) {  // uniform
    const int i = i0 + threadIdx.x;
    int total;
    const int before = block_scan(i < blocks ? a.sums[i] : 0, total);
    if (i < blocks) a.sums[i] = base + before;
    base += total;
  }
  if (threadIdx.x == 0) a.off[a.rows] = base;
}

__global__ __launch_bounds__(256) void k_offsets(Args a) {
  const int row0 = blockIdx.x * kScan + threadIdx.x * (kScan / 256);
  int v[kScan / 256], s = 0, total;
#pragma unroll
  for (int i = 0; i < kScan / 256; ++i) {
    v[i] = row0 + i < a.rows ? a.count[row0 + i] : 0;
    s += v[i];
  }
  int at = a.sums[blockIdx.x] + block_scan(s, total);
#pragma unroll
  for (int i = 0; i < kScan / 256; ++i) {
    if (row0 + i < a.rows) a.off[row0 + i] = at;
    at += v[i];
  }
}

// Mesh neighbours into their rows, in any order (k_mesh_rows sorts them).
__global__ __launch_bounds__(256) void k_fill(Args a) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= a.n_edges) return;
  int u, v, cs;
  if (!edge_rows(a, e, u, v, cs)) return;
  a.col[a.off[u] + atomicAdd(a.cursor + u, 1)] = v;
  a.col[a.off[v] + atomicAdd(a.cursor + v, 1)] = u;
}

// One thread per mesh node: its neighbours sorted, their directions, and its
// grid node last (the largest of the row's targets).
__global__ __launch_bounds__(256) void k_mesh_rows(Args a) {
  const int node = blockIdx.x * blockDim.x + threadIdx.x;
  if (node >= a.mesh_nodes) return;
  const int cs = case_of(a, 1, node);
  const int32_t *m = a.meta + cs * kMeta;
  const int row = m[0] + node - m[1], p0 = a.off[row], p1 = p0 + a.cursor[row];
  for (int p = p0 + 1; p < p1; ++p) {
    const int v = a.col[p];
    int q = p;
    for (; q > p0 && a.col[q - 1] > v; --q) a.col[q] = a.col[q - 1];
    a.col[q] = v;
  }
  const float w = (float)(1.0 / (double)a.count[row]);
  const double px = a.xy[2 * (size_t)node], py = a.xy[2 * (size_t)node + 1];
  for (int p = p0; p < p1; ++p) {
    const size_t to = (size_t)(a.col[p] - m[0] + m[1]);
    const double dx = a.xy[2 * to] - px, dy = a.xy[2 * to + 1] - py, L = hypot(dx, dy);
    a.w[p] = w;
    a.ex[p] = (float)(dx / L);
    a.ey[p] = (float)(dy / L);
  }
  if (a.cell[node] >= 0) {
    a.col[p1] = m[0] + m[2] + a.cell[node];
    a.w[p1] = w;
    a.ex[p1] = a.ey[p1] = 0.f;
  }
}

// One wave per virtual node. A grid node lists the mesh nodes of its cell,
// found by passing over the case's cell numbers in order, then its neighbours
// and the global node; the global node lists the grid nodes.
__global__ __launch_bounds__(256) void k_virtual_rows(Args a) {
  const int S = a.gx * a.gy, lane = threadIdx.x & 63;
  const int v = blockIdx.x * 4 + (threadIdx.x >> 6);  // uniform per wave
  if (v >= a.ncases * (S + 1)) return;
  const int cs = v / (S + 1), s = v % (S + 1);
  const int32_t *m = a.meta + cs * kMeta;
  const int first = m[0] + m[2], row = first + s;
  const float w = (float)(1.0 / (double)a.count[row]);
  int p = a.off[row];
  if (s == S) {
    for (int i = lane; i < S; i += 64) {
      a.col[p + i] = first + i;
      a.w[p + i] = w;
      a.ex[p + i] = a.ey[p + i] = -0.f;
    }
    return;
  }
  constexpr int U = 8;  // loads in flight
  for (int i0 = 0; i0 < m[2]; i0 += 64 * U) {
    int c[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + 64 * u + lane;
      c[u] = i < m[2] ? a.cell[m[1] + i] : -1;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const unsigned long long hit = __ballot(c[u] == s);
      if (c[u] == s) {
        const int at = p + __popcll(hit & ((1ull << lane) - 1));
        a.col[at] = m[0] + i0 + 64 * u + lane;
        a.w[at] = w;
        a.ex[at] = a.ey[at] = -0.f;
      }
      p += __popcll(hit);
    }
  }
  if (lane == 0) {
    const int i = s % a.gx, j = s / a.gx;
    for (int dj = -1; dj <= 1; ++dj)
      for (int di = -1; di <= 1; ++di) {
        if ((di == 0 && dj == 0) || i + di < 0 || i + di >= a.gx || j + dj < 0 || j + dj >= a.gy) continue;
        const bool back = dj < 0 || (dj == 0 && di < 0);  // the reverse of a listed direction
        const int d0 = back ? -di : di, d1 = back ? -dj : dj;
        const double ox = (double)d0 / a.gx, oy = (double)d1 / a.gy * a.height, L = hypot(ox, oy);
        const float fx = (float)(ox / L), fy = (float)(oy / L);
        a.col[p] = first + (j + dj) * a.gx + i + di;
        a.w[p] = w;
        a.ex[p] = back ? -fx : fx;
        a.ey[p] = back ? -fy : fy;
        ++p;
      }
    a.col[p] = first + S;
    a.w[p] = w;
    a.ex[p] = a.ey[p] = 0.f;
  }
}

// ---------------------------------------------------------------------------
// a prediction's fields
// ---------------------------------------------------------------------------
// Node rho = 1 + y0 s0 u_in and u = (y1 s1, y2 s2) u_in of the mesh nodes, in
// double, stored float32, and what the calibration reads of them per case:
// sums of rho - 1 over all and over the inlet nodes, the inlet count, the
// largest velocity component (NaN if any), and the extent of the points. One
// block per case; sums in a fixed order. On the host this and the rescaling
// took 3.7 ms for 12 cases (prediction 8.7 ms), here 0.1 ms (4.0).
constexpr int kStats = 8;  // sum, inlet sum, inlet count, largest |u|, x and y: least, largest

struct Fields {
  const int32_t *meta;
  const float *y;
  int64_t stride;
  double s0, s1, s2;
  const double *params, *xy;
  const int32_t *markers;
  int inlet;
  float *rho, *vel;
  double *stats;
};

__device__ __forceinline__ double larger(double a, double b) { return b > a || b != b ? b : a; }  // NaN stays

__global__ __launch_bounds__(1024) void k_fields(Fields a) {
  const int32_t *m = a.meta + blockIdx.x * kMeta;
  const double u_in = a.params[blockIdx.x * kParams];
  double v[kStats] = {0.0, 0.0, 0.0, 0.0, INFINITY, -INFINITY, INFINITY, -INFINITY};
  for (int i = threadIdx.x; i < m[2]; i += blockDim.x) {
    const float *y = a.y + (m[0] + i) * a.stride;
    const size_t node = (size_t)m[1] + i;
    const float r = (float)(1.0 + ((double)y[0] * a.s0) * u_in);
    const float ux = (float)(((double)y[1] * a.s1) * u_in), uy = (float)(((double)y[2] * a.s2) * u_in);
    a.rho[node] = r;
    a.vel[2 * node] = ux;
    a.vel[2 * node + 1] = uy;
    const double p = (double)r - 1.0, px = a.xy[2 * node], py = a.xy[2 * node + 1];
    v[0] += p;
    if (a.markers[node] == a.inlet) {
      v[1] += p;
      v[2] += 1.0;
    }
    v[3] = larger(larger(v[3], fabs((double)ux)), fabs((double)uy));
    v[4] = fmin(v[4], px);
    v[5] = fmax(v[5], px);
    v[6] = fmin(v[6], py);
    v[7] = fmax(v[7], py);
  }
  auto join = [](double (&x)[kStats], const double (&o)[kStats]) {
    for (int k = 0; k < 3; ++k) x[k] += o[k];
    x[3] = larger(x[3], o[3]);
    x[4] = fmin(x[4], o[4]);
    x[5] = fmax(x[5], o[5]);
    x[6] = fmin(x[6], o[6]);
    x[7] = fmax(x[7], o[7]);
  };
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    double o[kStats];
#pragma unroll
    for (int k = 0; k < kStats; ++k) o[k] = __shfl_down(v[k], d, 64);
    join(v, o);
  }
  __shared__ double sh[16][kStats];
  if ((threadIdx.x & 63) == 0)
    for (int k = 0; k < kStats; ++k) sh[threadIdx.x >> 6][k] = v[k];
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) join(v, sh[w]);
    for (int k = 0; k < kStats; ++k) a.stats[blockIdx.x * kStats + k] = v[k];
  }
}

// rho = 1 + f0 (rho - 1), u = f1 u with the factors of each case.
__global__ __launch_bounds__(256) void k_rescale(const int32_t *meta, int ncases, const double *factors,
                                                 int nodes, float *rho, float *vel) {
  const int node = blockIdx.x * blockDim.x + threadIdx.x;
  if (node >= nodes) return;
  Args a{};
  a.meta = meta;
  a.ncases = ncases;
  const double *f = factors + 2 * case_of(a, 1, node);
  rho[node] = (float)(1.0 + f[0] * ((double)rho[node] - 1.0));
  vel[2 * (size_t)node] = (float)(f[1] * (double)vel[2 * (size_t)node]);
  vel[2 * (size_t)node + 1] = (float)(f[1] * (double)vel[2 * (size_t)node + 1]);
}

}  // namespace fvdbm_nn_graph

extern "C" {

int64_t fvdbm_nn_device_inputs_ints(int64_t rows, int64_t mesh_nodes, int32_t ncases, int32_t section) {
  using namespace fvdbm_nn_graph;
  if (rows < 0 || mesh_nodes < 0 || ncases < 0 || section < 1) return -1;
  return 2 + 2 * rows + mesh_nodes + (rows + kScan - 1) / kScan + (int64_t)ncases * (3 * section + 1);
}

int fvdbm_nn_device_inputs(int32_t ncases, int64_t rows, int64_t mesh_nodes, int64_t n_edges,
                           const int32_t *meta, const double *params, const double *xy,
                           const int32_t *markers, const int32_t *edges, const double *discs,
                           int32_t gx, int32_t gy, double height, int32_t section,
                           const int32_t *marker_codes, const float *shift, const float *scale,
                           const float *sshift, const float *sscale, int32_t *work, float *x,
                           int32_t *off, int32_t *col, float *w, float *ex, float *ey, void *stream) {
  using namespace fvdbm_nn_graph;
  auto bad = [](const char *what) { return fvdbm::set_error(FVDBM_ERR_INVALID, what); };
  if (ncases < 1 || gx < 1 || gy < 1 || section < 1 || section > kMaxSection || mesh_nodes < 0 ||
      n_edges < 0 || !(height > 0.0))
    return bad("bad sizes");
  const int64_t S = (int64_t)gx * gy;
  if (rows != mesh_nodes + ncases * (S + 1)) return bad("rows do not match the nodes");
  if (2 * (n_edges + mesh_nodes + 4 * S * ncases + S * ncases) > INT32_MAX || rows > INT32_MAX - 2048)
    return bad("graph too large");
  if (!meta || !params || (mesh_nodes > 0 && (!xy || !markers)) || (n_edges > 0 && !edges) || !discs ||
      !marker_codes || !shift || !scale || !sshift || !sscale || !work || !x || !off || !col || !w ||
      !ex || !ey)
    return bad("null pointer");
  if ((reinterpret_cast<uintptr_t>(x) & 15) || (reinterpret_cast<uintptr_t>(work) & 7))
    return bad("x must be 16-byte aligned, work 8-byte aligned");
  Args a{};
  a.meta = meta;
  a.params = params;
  a.xy = xy;
  a.discs = discs;
  a.markers = markers;
  a.edges = edges;
  a.ncases = ncases;
  a.rows = (int)rows;
  a.mesh_nodes = (int)mesh_nodes;
  a.n_edges = (int)n_edges;
  a.gx = gx;
  a.gy = gy;
  a.section = section;
  a.height = height;
  for (int i = 0; i < 4; ++i) {
    a.codes[i] = marker_codes[i];
    a.sshift[i] = sshift[i];
    a.sscale[i] = sscale[i];
  }
  for (int i = 0; i < 9; ++i) {
    a.shift[i] = shift[i];
    a.scale[i] = scale[i];
  }
  const int blocks = (a.rows + kScan - 1) / kScan;
  a.error = reinterpret_cast<unsigned long long *>(work);
  a.count = work + 2;
  a.cursor = a.count + rows;
  a.cell = a.cursor + rows;
  a.sums = a.cell + mesh_nodes;
  a.tables = reinterpret_cast<float *>(a.sums + blocks);
  a.x = x;
  a.off = off;
  a.col = col;
  a.w = w;
  a.ex = ex;
  a.ey = ey;
  const hipStream_t st = static_cast<hipStream_t>(stream);
  auto grid = [](int64_t n, int per) { return dim3((unsigned)((n + per - 1) / per)); };
  hipLaunchKernelGGL(k_clear, grid(a.rows, 256), dim3(256), 0, st, a);
  hipLaunchKernelGGL(k_sections, dim3(ncases), dim3(256), 0, st, a);
  if (n_edges > 0) hipLaunchKernelGGL(k_count, grid(n_edges, 256), dim3(256), 0, st, a);
  hipLaunchKernelGGL(k_nodes, grid(a.rows, 256), dim3(256), 0, st, a);
  hipLaunchKernelGGL(k_block_sums, dim3(blocks), dim3(256), 0, st, a);
  hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(256), 0, st, a, blocks);
  hipLaunchKernelGGL(k_offsets, dim3(blocks), dim3(256), 0, st, a);
  if (n_edges > 0) hipLaunchKernelGGL(k_fill, grid(n_edges, 256), dim3(256), 0, st, a);
  if (mesh_nodes > 0) hipLaunchKernelGGL(k_mesh_rows, grid(mesh_nodes, 256), dim3(256), 0, st, a);
  hipLaunchKernelGGL(k_virtual_rows, grid(ncases * (S + 1), 4), dim3(256), 0, st, a);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? FVDBM_OK : fvdbm::set_error(FVDBM_ERR_HIP, hipGetErrorString(e));
}

int fvdbm_nn_fields(int32_t ncases, const int32_t *meta, const float *y, int64_t stride,
                    const double *target_scale, const double *params, const double *xy,
                    const int32_t *markers, int32_t inlet, float *rho, float *vel, double *stats,
                    void *stream) {
  using namespace fvdbm_nn_graph;
  if (ncases < 1 || stride < 3) return fvdbm::set_error(FVDBM_ERR_INVALID, "bad sizes");
  if (!meta || !y || !target_scale || !params || !xy || !markers || !rho || !vel || !stats)
    return fvdbm::set_error(FVDBM_ERR_INVALID, "null pointer");
  const Fields a{meta,   y,  stride,  target_scale[0], target_scale[1], target_scale[2],
                 params, xy, markers, inlet,           rho,             vel,
                 stats};
  hipLaunchKernelGGL(k_fields, dim3(ncases), dim3(1024), 0, static_cast<hipStream_t>(stream), a);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? FVDBM_OK : fvdbm::set_error(FVDBM_ERR_HIP, hipGetErrorString(e));
}

int fvdbm_nn_rescale(int32_t ncases, const int32_t *meta, const double *factors, int64_t nodes, float *rho,
                     float *vel, void *stream) {
  using namespace fvdbm_nn_graph;
  if (ncases < 1 || nodes < 0 || nodes > INT32_MAX - 256)
    return fvdbm::set_error(FVDBM_ERR_INVALID, "bad sizes");
  if (!meta || !factors || !rho || !vel) return fvdbm::set_error(FVDBM_ERR_INVALID, "null pointer");
  if (nodes == 0) return FVDBM_OK;
  hipLaunchKernelGGL(k_rescale, dim3((unsigned)((nodes + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), meta, ncases, factors, (int)nodes, rho, vel);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? FVDBM_OK : fvdbm::set_error(FVDBM_ERR_HIP, hipGetErrorString(e));
}

}  // extern "C"
