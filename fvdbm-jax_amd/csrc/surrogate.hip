// Kernels of the warm-start surrogate: a mesh message-passing network whose
// dense layers run on BF16 MFMA with FP32 accumulation, and the mesh
// aggregation that couples the nodes. No reference counterpart (the
// reference has no learned component); the C ABI is declared in
// include/fvdbm.h (fvdbm_nn_*).
//
// Building blocks (all row-major float32 in HBM; weights are float32 master
// copies, rounded to bf16 when staged in LDS):
//   mlp2   y = silu(x W1 + b1) W2 + b2, x [M,K], W1 [K,64], W2 [64,NO]
//   mlp2 backward (data part): recomputes z = x W1 + b1, then
//          dz = (dy W2^T) * silu'(z), dx = dz W1^T; writes dz and h = silu(z)
//   mlp2 gradients: dx and all weight gradients in one pass over the rows
//   wgrad  out = A^T B over the rows (A [M,KA], B [M,NB]) as per-chunk
//          partial products plus a fixed-order reduction (deterministic)
//   colsum out = sum over rows, same chunking
//   aggregate: z = [h | sum_e w h_j | sum_e w ex h_j | sum_e w ey h_j]
//          over each node's CSR edge list, and its transpose for dh.
//
// MFMA use: fragments follow the 16x16x16 bf16 layout. For one 64-lane
// wave with i = lane % 16 and g = lane / 16:
//   A (16x16, MxK): lane holds A[i][4g .. 4g+3]
//   B (16x16, KxN): lane holds B[4g .. 4g+3][i]
//   D (16x16, MxN): lane holds D[4g + r][i], r = 0..3
// K is consumed 32 at a time by gfx950's 16x16x32 bf16 MFMA (mfma2: two
// such fragments per operand), 16 at a time only for a 16-wide input.
// The dense layers are computed transposed (hidden units as MFMA rows, data
// rows as MFMA columns): then the D fragment of one layer is, lane by lane,
// exactly the B fragment the next layer needs, so the hidden activations
// never leave registers.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <mutex>
#include <string>

#include "fvdbm.h"

#pragma clang fp contract(fast)

namespace fvdbm_nn {

constexpr int HID = 64;
constexpr int CHUNK = 1024;  // rows per partial product in wgrad / colsum
constexpr int RGROUP = 32;   // partials summed per thread in the first reduction pass

typedef short s4 __attribute__((ext_vector_type(4)));
typedef short s8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

// float -> bf16 bits, round to nearest even (finite inputs)
__device__ __forceinline__ unsigned short f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}

__device__ __forceinline__ f4 mfma(s4 a, s4 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// Two consecutive K = 16 steps, c + A0 B0 + A1 B1, as one gfx950
// 16x16x32 MFMA. Each lane gives that instruction eight k values of A
// and the same eight k positions of B: here its four of (a0, b0) and its
// four of (a1, b1). A and B use one assignment of the 32 k indices to
// (lane group, slot), so the product sums exactly the 32 products of the
// two 16-blocks, in the instruction's own order (FP32 accumulation).
__device__ __forceinline__ f4 mfma2(s4 a0, s4 a1, s4 b0, s4 b1, f4 c) {
  const s8 a = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
  const s8 b = __builtin_shufflevector(b0, b1, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), c,
                                                  0, 0, 0);
}

__device__ __forceinline__ float silu(float z) { return z / (1.0f + __expf(-z)); }
__device__ __forceinline__ float dsilu(float z) {
  const float s = 1.0f / (1.0f + __expf(-z));
  return s * (1.0f + z * (1.0f - s));
}

__device__ __forceinline__ s4 lds4(const unsigned short *p) {
  return s4{(short)p[0], (short)p[1], (short)p[2], (short)p[3]};
}

__device__ __forceinline__ s4 bf4(float4 v) {
  return s4{(short)f2bf(v.x), (short)f2bf(v.y), (short)f2bf(v.z), (short)f2bf(v.w)};
}

// as bf4, by gfx950's packed conversion (the same bits for every number)
typedef __bf16 b4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ s4 cvt4(f4 v) {
  return __builtin_bit_cast(s4, __builtin_convertvector(v, b4));
}

// s[0 .. 3], 8-byte aligned
__device__ __forceinline__ s4 lds8(const unsigned short *p) { return *reinterpret_cast<const s4 *>(p); }

// The fragment (column c0 + i, rows r0 + 4g .. + 3) of a row-major LDS array
// with row stride S, by the transposing read: lane q of a group of 16 points
// at four consecutive columns of one of the group's four rows and receives
// column q of them.
template <int S>
__device__ __forceinline__ s4 lds_columns(const unsigned short *s, int r0, int c0) {
  const int i = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
  const unsigned short *p = s + (r0 + 4 * g + (i >> 2)) * S + c0 + 4 * (i & 3);
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s4 *)const_cast<unsigned short *>(p));
}

// ---------------------------------------------------------------------------
// mlp2 forward, with RES plus a residual: y = res + mlp2(x)
// ---------------------------------------------------------------------------
// A block of four waves takes 32 rows at a time: wave w owns hidden units
// 16 w .. 16 w + 15 and the same outputs, with its shares of W1 and W2 in
// registers over all its rows. Rows and hidden values pass through LDS as
// bf16; the next rows are loaded while the current are computed. Bound by
// memory: x is read and y written once (K = 256, 540k rows: 691 MB, 140 us at
// 5 TB/s). A wave per 16 rows with all weights read from LDS for each took
// 245 us at 540k rows and 61 at 46k, this takes 148 and 27. Four blocks per CU
// instead of three (K = 256) spill 22 registers.
constexpr int GR = 32;  // rows per tile

__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The four floats e, e + 1, .. of rows [row0, row0 + GR) of X [M][K], zero
// from row M on; e = 4 (thread + 256 u).
template <int K>
struct RowLoad {
  static constexpr int N4 = GR * K / 4, N = (N4 + 255) / 256;
  f4 v[N];
  __device__ __forceinline__ void load(const float *__restrict__ X, int64_t row0, int M) {
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const int e = threadIdx.x + 256 * u;
      const int64_t row = row0 + e / (K / 4);
      v[u] = e < N4 && row < M ? *reinterpret_cast<const f4 *>(X + row * K + 4 * (e % (K / 4)))
                               : f4{0.f, 0.f, 0.f, 0.f};
    }
  }
  template <int S>
  __device__ __forceinline__ void store(unsigned short *s) const {
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const int e = threadIdx.x + 256 * u;
      if (N4 % 256 == 0 || e < N4)
        *reinterpret_cast<s4 *>(s + (e / (K / 4)) * S + 4 * (e % (K / 4))) = cvt4(v[u]);
    }
  }
};

template <int K, int NO, bool RES>
__global__ __launch_bounds__(256, K == 256 ? 3 : 4) void k_mlp_fwd(const float *__restrict__ x, int M,
                                                    const float *__restrict__ w1,
                                                    const float *__restrict__ b1,
                                                    const float *__restrict__ w2,
                                                    const float *__restrict__ b2,
                                                    const float *__restrict__ res,
                                                    float *__restrict__ y) {
  constexpr int KB = K / 16, XS = K + 8, HS = HID + 8;
  constexpr int J = NO == 64 ? 2 : 1;  // 16-row halves of a tile this wave writes
  __shared__ __align__(16) unsigned short sX[GR * XS], sH[GR * HS];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, i = lane & 15, g = lane >> 4;
  const int ob = NO == 64 ? w : 0, j0 = NO == 64 ? 0 : w;  // 16 outputs: wave w < 2 takes half w
  s4 w1z[KB], w2f[4];
  float bias1[4], bias2[4];
#pragma unroll
  for (int ks = 0; ks < KB; ++ks) {
    const float *p = w1 + (size_t)(ks * 16 + 4 * g) * HID + w * 16 + i;
    w1z[ks] = cvt4(f4{p[0], p[HID], p[2 * HID], p[3 * HID]});
  }
#pragma unroll
  for (int hs = 0; hs < 4; ++hs) {
    const float *p = w2 + (size_t)(hs * 16 + 4 * g) * NO + ob * 16 + i;
    w2f[hs] = cvt4(f4{p[0], p[NO], p[2 * NO], p[3 * NO]});
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    bias1[r] = b1[w * 16 + 4 * g + r];
    bias2[r] = b2[ob * 16 + 4 * g + r];
  }
  const int tiles = (M - 1) / GR + 1;
  RowLoad<K> xr;
  int t = blockIdx.x;
  if (t < tiles) xr.load(x, (int64_t)t * GR, M);
  for (; t < tiles; t += gridDim.x) {
    const int64_t row0 = (int64_t)t * GR;
    xr.template store<XS>(sX);
    f4 base[J];
    if constexpr (RES) {
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const int64_t row = row0 + (j0 + j) * 16 + i;
        if (row < M) base[j] = *reinterpret_cast<const f4 *>(res + row * NO + ob * 16 + 4 * g);
      }
    }
    if (t + (int64_t)gridDim.x < tiles) xr.load(x, row0 + (int64_t)gridDim.x * GR, M);
    lds_barrier();
    f4 z[2] = {f4{0.f, 0.f, 0.f, 0.f}, f4{0.f, 0.f, 0.f, 0.f}};
    const unsigned short *px = sX + i * XS + 4 * g;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if constexpr (KB % 2 == 0) {
#pragma unroll
        for (int kp = 0; kp < KB / 2; ++kp)
          z[j] = mfma2(w1z[2 * kp], w1z[2 * kp + 1], lds8(px + j * 16 * XS + 32 * kp),
                       lds8(px + j * 16 * XS + 32 * kp + 16), z[j]);
      } else {
        z[j] = mfma(w1z[0], lds8(px + j * 16 * XS), z[j]);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) z[j][r] = silu(z[j][r] + bias1[r]);
      *reinterpret_cast<s4 *>(sH + (j * 16 + i) * HS + w * 16 + 4 * g) = cvt4(z[j]);
    }
    lds_barrier();
    if (NO == 64 || w < 2) {
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const unsigned short *ph = sH + ((j0 + j) * 16 + i) * HS + 4 * g;
        f4 acc = f4{0.f, 0.f, 0.f, 0.f};
        acc = mfma2(w2f[0], w2f[1], lds8(ph), lds8(ph + 16), acc);
        acc = mfma2(w2f[2], w2f[3], lds8(ph + 32), lds8(ph + 48), acc);
        const int64_t row = row0 + (j0 + j) * 16 + i;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          acc[r] += bias2[r];
          if constexpr (RES) acc[r] = base[j][r] + acc[r];
        }
        if (row < M) *reinterpret_cast<f4 *>(y + row * NO + ob * 16 + 4 * g) = acc;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// mlp2 backward, data part: dz [M,64], h [M,64] and (optionally) dx [M,K]
// ---------------------------------------------------------------------------
template <int K, int NO>
__global__ __launch_bounds__(256) void k_mlp_bwd(const float *__restrict__ x, int M,
                                                 const float *__restrict__ w1,
                                                 const float *__restrict__ b1,
                                                 const float *__restrict__ w2,
                                                 const float *__restrict__ dy,
                                                 float *__restrict__ dx, float *__restrict__ dz,
                                                 float *__restrict__ hout) {
  constexpr int HP = HID + 4, NP = NO + 4;
  __shared__ unsigned short sW1[K * HP];    // [k][hidden]: z (strided reads) and dx
  __shared__ unsigned short sW2[HID * NP];  // [hidden][out]: dh = dy W2^T
  __shared__ float sb1[HID];
  for (int e = threadIdx.x; e < K * HID; e += blockDim.x) sW1[(e / HID) * HP + e % HID] = f2bf(w1[e]);
  for (int e = threadIdx.x; e < HID * NO; e += blockDim.x) sW2[(e / NO) * NP + e % NO] = f2bf(w2[e]);
  if (threadIdx.x < HID) sb1[threadIdx.x] = b1[threadIdx.x];
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i = lane & 15, g = lane >> 4;
  const int ntiles = (M + 15) / 16;
  for (int t = blockIdx.x * 4 + wave; t < ntiles; t += gridDim.x * 4) {
    const int row = t * 16 + i;
    const bool ok = row < M;
    f4 z[4], dh[4];
#pragma unroll
    for (int hb = 0; hb < 4; ++hb) {
      z[hb] = f4{0.f, 0.f, 0.f, 0.f};
      dh[hb] = f4{0.f, 0.f, 0.f, 0.f};
    }
    // B fragments of x's and dy's 16-column block ks, and the A fragment
    // W1^T[hidden block hb][k block ks] read down sW1's columns
    auto xfrag = [&](int ks) {
      const float4 xv = ok ? *reinterpret_cast<const float4 *>(x + (size_t)row * K + ks * 16 + 4 * g)
                           : make_float4(0.f, 0.f, 0.f, 0.f);
      return bf4(xv);
    };
    auto dyfrag = [&](int os) {
      const float4 dv = ok ? *reinterpret_cast<const float4 *>(dy + (size_t)row * NO + os * 16 + 4 * g)
                           : make_float4(0.f, 0.f, 0.f, 0.f);
      return bf4(dv);
    };
    auto w1t = [&](int ks, int hb) {
      const unsigned short *p = sW1 + (ks * 16 + 4 * g) * HP + hb * 16 + i;
      return s4{(short)p[0], (short)p[HP], (short)p[2 * HP], (short)p[3 * HP]};
    };
    if constexpr (K % 32 == 0) {
#pragma unroll
      for (int kp = 0; kp < K / 32; ++kp) {
        const s4 b0 = xfrag(2 * kp), b1 = xfrag(2 * kp + 1);
#pragma unroll
        for (int hb = 0; hb < 4; ++hb) z[hb] = mfma2(w1t(2 * kp, hb), w1t(2 * kp + 1, hb), b0, b1, z[hb]);
      }
    } else {
#pragma unroll
      for (int ks = 0; ks < K / 16; ++ks) {
        const s4 b = xfrag(ks);
#pragma unroll
        for (int hb = 0; hb < 4; ++hb) z[hb] = mfma(w1t(ks, hb), b, z[hb]);
      }
    }
    // dh^T [hidden][rows] = W2 [hidden][out] . dy^T [out][rows]
    if constexpr (NO % 32 == 0) {
#pragma unroll
      for (int op = 0; op < NO / 32; ++op) {
        const s4 b0 = dyfrag(2 * op), b1 = dyfrag(2 * op + 1);
#pragma unroll
        for (int hb = 0; hb < 4; ++hb) {
          const unsigned short *w = sW2 + (hb * 16 + i) * NP + op * 32 + 4 * g;
          dh[hb] = mfma2(lds4(w), lds4(w + 16), b0, b1, dh[hb]);
        }
      }
    } else {
#pragma unroll
      for (int os = 0; os < NO / 16; ++os) {
        const s4 b = dyfrag(os);
#pragma unroll
        for (int hb = 0; hb < 4; ++hb)
          dh[hb] = mfma(lds4(sW2 + (hb * 16 + i) * NP + os * 16 + 4 * g), b, dh[hb]);
      }
    }
    s4 dzfrag[4];
#pragma unroll
    for (int hb = 0; hb < 4; ++hb) {
      float d4[4], h4[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float zz = z[hb][r] + sb1[hb * 16 + 4 * g + r];
        h4[r] = silu(zz);
        d4[r] = dh[hb][r] * dsilu(zz);
      }
      if (ok) {
        const size_t o = (size_t)row * HID + hb * 16 + 4 * g;
        *reinterpret_cast<float4 *>(dz + o) = make_float4(d4[0], d4[1], d4[2], d4[3]);
        *reinterpret_cast<float4 *>(hout + o) = make_float4(h4[0], h4[1], h4[2], h4[3]);
      }
      dzfrag[hb] = bf4(make_float4(d4[0], d4[1], d4[2], d4[3]));
    }
    if (dx) {
      // dx^T [k][rows] = W1 [k][hidden] . dz^T [hidden][rows]
#pragma unroll
      for (int kb = 0; kb < K / 16; ++kb) {
        f4 acc = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kp = 0; kp < 2; ++kp) {
          const unsigned short *w = sW1 + (kb * 16 + i) * HP + kp * 32 + 4 * g;
          acc = mfma2(lds4(w), lds4(w + 16), dzfrag[2 * kp], dzfrag[2 * kp + 1], acc);
        }
        if (ok)
          *reinterpret_cast<float4 *>(dx + (size_t)row * K + kb * 16 + 4 * g) =
              make_float4(acc[0], acc[1], acc[2], acc[3]);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// mlp2 backward, all of it: dx and the four weight gradients in one pass
// ---------------------------------------------------------------------------
// A block of four waves takes 32 rows at a time. Wave w owns hidden units
// 16 w .. 16 w + 15 of z and dy W2^T, a quarter of dx's columns and the same
// quarter of dW1's rows, so its shares of W1 and W2 and of the gradients stay
// in registers over all its rows. Rows, dz and h pass through LDS as bf16,
// row-major; the weight gradients contract over rows and read them by the
// transposing read. The next rows are loaded while the current are computed.
// Bound by memory: x and dy are read and dx is written once (K = 256, 540k
// rows: 1.25 GB, 250 us at 5 TB/s), where separate kernels for dx and the four
// sums read x twice, dy three times and passed dz and h through memory. All
// gradients at 540k / 46k rows: 990 / 390 -> 343 / 122 us. W1 sits in LDS
// when dx is asked for: in registers as well, 22 spilled and every reload
// waited for the rows in flight.
// GR rows a tile, as the forward kernel.
constexpr int GRAD_BLOCKS = 512;  // two blocks per CU

constexpr int grad_floats(int K, int NO) { return K * HID + HID * NO + HID + NO; }

template <int K, int NO, bool DX>
__global__ __launch_bounds__(256, 2) void k_mlp_grad(const float *__restrict__ x, int M,
                                                     const float *__restrict__ w1,
                                                     const float *__restrict__ b1,
                                                     const float *__restrict__ w2,
                                                     const float *__restrict__ dy,
                                                     float *__restrict__ dx,
                                                     float *__restrict__ partial) {
  constexpr int KB = K / 16, OB = NO / 16, PER = KB >= 4 ? KB / 4 : 1;
  constexpr int XS = K + 8, YS = NO + 8, HS = HID + 8;
  __shared__ __align__(16) unsigned short sX[GR * XS], sY[GR * YS], sD[GR * HS], sH[GR * HS];
  __shared__ __align__(16) unsigned short sW[DX ? K * HS : 4];  // W1, for dx
  __shared__ __align__(16) float red[256 * 4];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, i = lane & 15, g = lane >> 4;
  // this wave's shares: W1^T (hidden 16 w + i; all k), W2 (hidden 16 w + i;
  // all outputs)
  s4 w1z[DX ? 1 : KB], w2f[OB];  // with dx, W1^T comes from sW
  float bias[4];
#pragma unroll
  for (int ks = 0; !DX && ks < KB; ++ks) {
    const float *p = w1 + (size_t)(ks * 16 + 4 * g) * HID + w * 16 + i;
    w1z[ks] = cvt4(f4{p[0], p[HID], p[2 * HID], p[3 * HID]});
  }
#pragma unroll
  for (int os = 0; os < OB; ++os) {
    const float *p = w2 + (size_t)(w * 16 + i) * NO + os * 16 + 4 * g;
    w2f[os] = cvt4(f4{p[0], p[1], p[2], p[3]});
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) bias[r] = b1[w * 16 + 4 * g + r];
  const int kb0 = KB >= 4 ? w * PER : 0;  // a 16-wide input has one block: wave 0's dx
  if constexpr (DX)
    for (int e = threadIdx.x; e < K * HID / 4; e += 256)
      *reinterpret_cast<s4 *>(sW + (e / 16) * HS + 4 * (e % 16)) =
          cvt4(f4{w1[4 * e], w1[4 * e + 1], w1[4 * e + 2], w1[4 * e + 3]});
  constexpr int HB1 = KB >= 4 ? 4 : 1;  // dW1's hidden blocks of this wave: all, or block w
  f4 g1[PER][HB1], g2[OB], gb1 = f4{0.f, 0.f, 0.f, 0.f}, gb2 = gb1;
#pragma unroll
  for (int p = 0; p < PER; ++p)
#pragma unroll
    for (int hb = 0; hb < HB1; ++hb) g1[p][hb] = gb1;
#pragma unroll
  for (int ob = 0; ob < OB; ++ob) g2[ob] = gb1;

  const int tiles = (M - 1) / GR + 1;
  RowLoad<K> xr;
  RowLoad<NO> yr;
  int t = blockIdx.x;
  if (t < tiles) {
    xr.load(x, (int64_t)t * GR, M);
    yr.load(dy, (int64_t)t * GR, M);
  }
  for (; t < tiles; t += gridDim.x) {
    const int64_t row0 = (int64_t)t * GR;
    xr.template store<XS>(sX);
    yr.template store<YS>(sY);
#pragma unroll
    for (int u = 0; u < RowLoad<NO>::N; ++u) gb2 += yr.v[u];
    if (t + (int64_t)gridDim.x < tiles) {
      xr.load(x, row0 + (int64_t)gridDim.x * GR, M);
      yr.load(dy, row0 + (int64_t)gridDim.x * GR, M);
    }
    lds_barrier();
    f4 zj[2] = {f4{0.f, 0.f, 0.f, 0.f}, f4{0.f, 0.f, 0.f, 0.f}};
    auto w1t = [&](int ks) {
      if constexpr (DX) return lds_columns<HS>(sW, ks * 16, w * 16);
      else return w1z[ks];
    };
    const unsigned short *px = sX + i * XS + 4 * g;
    if constexpr (KB % 2 == 0) {
#pragma unroll
      for (int kp = 0; kp < KB / 2; ++kp) {
        const s4 a0 = w1t(2 * kp), a1 = w1t(2 * kp + 1);
#pragma unroll
        for (int j = 0; j < 2; ++j)
          zj[j] = mfma2(a0, a1, lds8(px + j * 16 * XS + 32 * kp), lds8(px + j * 16 * XS + 32 * kp + 16), zj[j]);
      }
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j) zj[j] = mfma(w1t(0), lds8(px + j * 16 * XS), zj[j]);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const f4 z = zj[j];
      f4 dh = f4{0.f, 0.f, 0.f, 0.f};
      const unsigned short *py = sY + (j * 16 + i) * YS + 4 * g;
      if constexpr (OB % 2 == 0) {
#pragma unroll
        for (int op = 0; op < OB / 2; ++op)
          dh = mfma2(w2f[2 * op], w2f[2 * op + 1], lds8(py + 32 * op), lds8(py + 32 * op + 16), dh);
      } else {
        dh = mfma(w2f[0], lds8(py), dh);
      }
      const bool ok = row0 + j * 16 + i < M;
      f4 d, h;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float zz = z[r] + bias[r];
        h[r] = ok ? silu(zz) : 0.f;
        d[r] = ok ? dh[r] * dsilu(zz) : 0.f;
      }
      gb1 += d;
      const int o = (j * 16 + i) * HS + w * 16 + 4 * g;
      *reinterpret_cast<s4 *>(sD + o) = cvt4(d);
      *reinterpret_cast<s4 *>(sH + o) = cvt4(h);
    }
    lds_barrier();
    if constexpr (DX) {
      if (KB >= 4 || w == 0) {
        s4 df[2][4];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int hs = 0; hs < 4; ++hs) df[j][hs] = lds8(sD + (j * 16 + i) * HS + hs * 16 + 4 * g);
#pragma unroll
        for (int p = 0; p < PER; ++p) {
          const unsigned short *pw = sW + ((kb0 + p) * 16 + i) * HS + 4 * g;
          const s4 a0 = lds8(pw), a1 = lds8(pw + 16), a2 = lds8(pw + 32), a3 = lds8(pw + 48);
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const int64_t row = row0 + j * 16 + i;
            f4 acc = f4{0.f, 0.f, 0.f, 0.f};
            acc = mfma2(a0, a1, df[j][0], df[j][1], acc);
            acc = mfma2(a2, a3, df[j][2], df[j][3], acc);
            if (row < M) *reinterpret_cast<f4 *>(dx + row * K + (kb0 + p) * 16 + 4 * g) = acc;
          }
        }
      }
    }
    s4 dT[HB1][2];
#pragma unroll
    for (int hb = 0; hb < HB1; ++hb)
#pragma unroll
      for (int j = 0; j < 2; ++j) dT[hb][j] = lds_columns<HS>(sD, j * 16, (KB >= 4 ? hb : w) * 16);
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const s4 x0 = lds_columns<XS>(sX, 0, (kb0 + p) * 16), x1 = lds_columns<XS>(sX, 16, (kb0 + p) * 16);
#pragma unroll
      for (int hb = 0; hb < HB1; ++hb) g1[p][hb] = mfma2(x0, x1, dT[hb][0], dT[hb][1], g1[p][hb]);
    }
    const s4 h0 = lds_columns<HS>(sH, 0, w * 16), h1 = lds_columns<HS>(sH, 16, w * 16);
#pragma unroll
    for (int ob = 0; ob < OB; ++ob)
      g2[ob] = mfma2(h0, h1, lds_columns<YS>(sY, 0, ob * 16), lds_columns<YS>(sY, 16, ob * 16), g2[ob]);
    lds_barrier();
  }

  // this block's sums: [dW1 | dW2 | db1 | db2]
  float *out = partial + (size_t)blockIdx.x * grad_floats(K, NO);
#pragma unroll
  for (int p = 0; p < PER; ++p)
#pragma unroll
    for (int hb = 0; hb < HB1; ++hb)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        out[((kb0 + p) * 16 + 4 * g + r) * HID + (KB >= 4 ? hb : w) * 16 + i] = g1[p][hb][r];
  out += K * HID;
#pragma unroll
  for (int ob = 0; ob < OB; ++ob)
#pragma unroll
    for (int r = 0; r < 4; ++r) out[(w * 16 + 4 * g + r) * NO + ob * 16 + i] = g2[ob][r];
  out += HID * NO;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float v = gb1[r];
    for (int m = 1; m < 16; m <<= 1) v += __shfl_xor(v, m);
    if (i == 0) out[w * 16 + 4 * g + r] = v;
  }
  out += HID;
  *reinterpret_cast<f4 *>(red + 4 * threadIdx.x) = gb2;  // columns 4 (thread % (NO / 4)) ..
  __syncthreads();
  if (threadIdx.x < NO) {
    float v = 0.f;
    for (int e = threadIdx.x; e < 256 * 4; e += NO) v += red[e];
    out[threadIdx.x] = v;
  }
}

// ---------------------------------------------------------------------------
// wgrad: partial[c] = A[rows of chunk c]^T B[rows of chunk c]  ([KA][NB])
// One block per chunk of CHUNK rows, staged 64 rows at a time in LDS as
// bf16, transposed (feature-major, [feature][row]): an MFMA operand
// fragment (one feature, four consecutive rows) is then one 8-byte LDS
// read. The output 16x16 blocks are dealt round-robin to the four waves;
// each wave's accumulators live in registers across the chunk.
// ---------------------------------------------------------------------------
// Stage rows [base, base + R) of X [rows][K] (rows from r1 on read as 0)
// into s as bf16, feature-major ([K][RS]). Work item e takes the 4x4 block
// of features 4c .. 4c+3 and rows 4q .. 4q+3 (q = e % (R/4) fastest, so
// neighbouring lanes write neighbouring 8-byte words of one feature row):
// four 16-byte loads, one per row, and four 8-byte LDS stores, one per
// feature. X rows must be 16-byte aligned (K a multiple of 4).
template <int K, int R, int RS>
__device__ __forceinline__ void stage_transposed(const float *__restrict__ X, int base, int r1,
                                                 unsigned short *__restrict__ s) {
  static_assert(K % 4 == 0 && R % 4 == 0, "4x4 blocks");
  for (int e = threadIdx.x; e < (K / 4) * (R / 4); e += blockDim.x) {
    const int q = e % (R / 4), c = e / (R / 4);
    float4 v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int row = base + 4 * q + j;
      v[j] = row < r1 ? *reinterpret_cast<const float4 *>(X + (size_t)row * K + 4 * c)
                      : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    const float col[4][4] = {{v[0].x, v[1].x, v[2].x, v[3].x},
                             {v[0].y, v[1].y, v[2].y, v[3].y},
                             {v[0].z, v[1].z, v[2].z, v[3].z},
                             {v[0].w, v[1].w, v[2].w, v[3].w}};
#pragma unroll
    for (int f = 0; f < 4; ++f)
      *reinterpret_cast<uint2 *>(s + (4 * c + f) * RS + 4 * q) =
          make_uint2((uint32_t)f2bf(col[f][0]) | ((uint32_t)f2bf(col[f][1]) << 16),
                     (uint32_t)f2bf(col[f][2]) | ((uint32_t)f2bf(col[f][3]) << 16));
  }
}

template <int KA, int NB>
__global__ __launch_bounds__(256) void k_wgrad(const float *__restrict__ A,
                                               const float *__restrict__ B, int M,
                                               float *__restrict__ partial) {
  constexpr int R = 64;          // rows per LDS stage
  constexpr int RP = R + 4;      // row stride of a feature, in bf16 (8-byte aligned, odd in 8-byte units)
  constexpr int NBLK = (KA / 16) * (NB / 16);
  constexpr int PER = (NBLK + 3) / 4;
  __shared__ __align__(16) unsigned short sA[KA * RP];
  __shared__ __align__(16) unsigned short sB[NB * RP];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i = lane & 15, g = lane >> 4;
  const int r0 = blockIdx.x * CHUNK, r1 = min(M, r0 + CHUNK);
  f4 acc[PER];
#pragma unroll
  for (int p = 0; p < PER; ++p) acc[p] = f4{0.f, 0.f, 0.f, 0.f};
  for (int base = r0; base < r1; base += R) {
    __syncthreads();
    stage_transposed<KA, R, RP>(A, base, r1, sA);
    stage_transposed<NB, R, RP>(B, base, r1, sB);
    __syncthreads();
#pragma unroll
    for (int mp = 0; mp < R / 32; ++mp) {
      const int m = mp * 32 + 4 * g;  // this lane's four rows of each 16-row slab of the pair
#pragma unroll
      for (int p = 0; p < PER; ++p) {
        const int blk = wave + 4 * p;
        if (blk < NBLK) {
          const int kb = blk / (NB / 16), nb = blk % (NB / 16);
          // A fragments: feature kb*16+i, rows m..m+3 and m+16..m+19; B: feature nb*16+i, same rows
          const unsigned short *pa = sA + (kb * 16 + i) * RP + m;
          const unsigned short *pb = sB + (nb * 16 + i) * RP + m;
          acc[p] = mfma2(*reinterpret_cast<const s4 *>(pa), *reinterpret_cast<const s4 *>(pa + 16),
                         *reinterpret_cast<const s4 *>(pb), *reinterpret_cast<const s4 *>(pb + 16), acc[p]);
        }
      }
    }
  }
  float *out = partial + (size_t)blockIdx.x * KA * NB;
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int blk = wave + 4 * p;
    if (blk < NBLK) {
      const int kb = blk / (NB / 16), nb = blk % (NB / 16);
#pragma unroll
      for (int r = 0; r < 4; ++r) out[(size_t)(kb * 16 + 4 * g + r) * NB + nb * 16 + i] = acc[p][r];
    }
  }
}

// partial[c][n] = sum of column n over the rows of chunk c: 256 / N row
// groups per column each sum their rows in order, then the groups are added
// in group order (fixed order, deterministic)
__global__ __launch_bounds__(256) void k_colsum(const float *__restrict__ A, int M, int N,
                                                float *__restrict__ partial) {
  __shared__ float red[256];
  const int groups = 256 / N;
  const int n = threadIdx.x % N, grp = threadIdx.x / N;
  const int r0 = blockIdx.x * CHUNK, r1 = min(M, r0 + CHUNK);
  float s = 0.f;
  if (grp < groups)
    for (int r = r0 + grp; r < r1; r += groups) s += A[(size_t)r * N + n];
  red[threadIdx.x] = s;
  __syncthreads();
  if (threadIdx.x < N) {
    float t = 0.f;
    for (int g = 0; g < groups; ++g) t += red[g * N + threadIdx.x];
    partial[(size_t)blockIdx.x * N + threadIdx.x] = t;
  }
}

__global__ void k_zero(float *__restrict__ p, int n) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e < n) p[e] = 0.f;
}

// First pass of the chunk reduction, in place: for group q (blockIdx.y),
// partial[q * RGROUP][e] <- the sum, in chunk order, of partial[c][e] over
// the group's chunks c = q*RGROUP .. Each thread reads only its group's
// chunks and writes its group's first slot, so the pass is race-free.
__global__ void k_reduce_groups(float *__restrict__ partial, int nchunks, int n) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const int c0 = blockIdx.y * RGROUP, c1 = min(nchunks, c0 + RGROUP);
  float s = 0.f;
  for (int c = c0; c < c1; ++c) s += partial[(size_t)c * n + e];
  partial[(size_t)c0 * n + e] = s;
}

// The second pass of the gradient kernel's reduction, for its four parts.
__global__ void k_reduce_grads(const float *__restrict__ partial, int nparts, int n1, int n2, int n3,
                               int n4, float *__restrict__ o1, float *__restrict__ o2,
                               float *__restrict__ o3, float *__restrict__ o4) {
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  const int n = n1 + n2 + n3 + n4;
  if (e >= n) return;
  float s = 0.f;
  for (int c = 0; c < nparts; c += RGROUP) s += partial[(size_t)c * n + e];
  if (e < n1) o1[e] = s;
  else if ((e -= n1) < n2) o2[e] = s;
  else if ((e -= n2) < n3) o3[e] = s;
  else o4[e - n3] = s;
}

// Second pass: out[e] = the sum, in group order, of the group sums.
__global__ void k_reduce_final(const float *__restrict__ partial, int nchunks, int n,
                               float *__restrict__ out) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  float s = 0.f;
  for (int c = 0; c < nchunks; c += RGROUP) s += partial[(size_t)c * n + e];
  out[e] = s;
}

// ---------------------------------------------------------------------------
// aggregation: lane = feature, one wave per R consecutive nodes
// ---------------------------------------------------------------------------
// Bound by the gathers of 256-byte rows (z and h alone: 691 MB, 140 us at 5
// TB/s, for 540k nodes). One wave per node, one edge at a time, waited a
// memory round trip per edge, and the global node (one edge per grid node) 512
// of them. Here a wave walks the edges of its nodes as one list: 64 edges'
// lists are read by one coalesced load, and the rows of the next 16 edges are
// requested while the current 16 are summed, across node borders. Each sum
// takes its edges in list order, so the results are those of the plain loop.
// Forward / backward, 46k nodes: 171 / 187 -> 39 / 70 us; 540k nodes: 704 /
// 684 -> 243 / 340 us. Groups of 8 edges: 286 / 410 us at 540k.
constexpr int kEdgeGroup = 16;

__device__ __forceinline__ int lane_int(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ float lane_float(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// Walks the edges of nodes [r0, r1) (r1 - r0 < 64). `request(col, u)` asks
// for the row of node `col` into slot u (0 .. 2 * kEdgeGroup - 1), `add(u, w,
// ex, ey)` adds the row in slot u, `finish(r)` ends node r. Slots alternate
// between two halves: the one requested and the one summed.
template <typename Request, typename Add, typename Finish>
__device__ __forceinline__ void walk_edges(int r0, int r1, const int32_t *__restrict__ off,
                                           const int32_t *__restrict__ col,
                                           const float *__restrict__ w, const float *__restrict__ ex,
                                           const float *__restrict__ ey, Request request, Add add,
                                           Finish finish) {
  const int lane = threadIdx.x & 63;
  const int ends = off[min(r0 + lane, r1)];  // lane k: first edge of node r0 + k
  const int e0 = lane_int(ends, 0), e1 = lane_int(ends, r1 - r0);
  int r = r0, end = lane_int(ends, 1);
  int c = 0;
  float cw = 0.f, cx = 0.f, cy = 0.f;
  auto list_at = [&](int e) {  // the lists of edges e .. e + 63, one per lane
    const int i = min(e + lane, e1 - 1);
    c = col[i];
    cw = w[i];
    cx = ex[i];
    cy = ey[i];
  };
  if (e0 < e1) {
    list_at(e0);
#pragma unroll
    for (int u = 0; u < kEdgeGroup; ++u) request(lane_int(c, u), u);
  }
  for (int base = e0; base < e1; base += 64) {
    const int pc = c;
    const float pw = cw, px = cx, py = cy;
    if (base + 64 < e1) list_at(base + 64);
#pragma unroll
    for (int g = 0; g < 64 / kEdgeGroup; ++g) {
      const int from = base + g * kEdgeGroup;
      if (from >= e1) break;
      // request the next group
      if (from + kEdgeGroup < e1) {
#pragma unroll
        for (int u = 0; u < kEdgeGroup; ++u) {
          const int k = (g + 1) * kEdgeGroup + u;
          request(k < 64 ? lane_int(pc, k & 63) : lane_int(c, k & 63),
                  ((g + 1) & 1) * kEdgeGroup + u);
        }
      }
#pragma unroll
      for (int u = 0; u < kEdgeGroup; ++u) {
        if (from + u < e1) {
          while (from + u == end) {  // also nodes without edges
            finish(r);
            ++r;
            end = lane_int(ends, r - r0 + 1);
          }
          const int k = g * kEdgeGroup + u;
          add((g & 1) * kEdgeGroup + u, lane_float(pw, k), lane_float(px, k), lane_float(py, k));
        }
      }
    }
  }
  for (; r < r1; ++r) finish(r);
}

// Nodes per wave. Up to kAggSmallNodes the long lists of the last nodes set
// the time, and a wave each spreads them best (46k nodes, forward: 39 us with
// 1, 45 with 2, 58 with 4); beyond, short lists cost more than they spread
// (540k nodes: 267 us with 2, 243 with 4, 253 with 8, 309 with 16).
constexpr int kAggRows = 4, kAggRowsSmall = 1, kAggSmallNodes = 131072;

// First node of this wave; the last nodes (a graph's virtual nodes, whose
// lists are long) first.
__device__ __forceinline__ int agg_first(int n, int rows) {
  const int waves = (n + rows - 1) / rows;
  const int wave = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
  return (waves - 1 - wave) * rows;  // negative: none
}

__global__ __launch_bounds__(256) void k_aggregate(const float *__restrict__ h, int n, int rows,
                                                   const int32_t *__restrict__ off,
                                                   const int32_t *__restrict__ col,
                                                   const float *__restrict__ w,
                                                   const float *__restrict__ ex,
                                                   const float *__restrict__ ey,
                                                   float *__restrict__ z) {
  const int f = threadIdx.x & 63, r0 = agg_first(n, rows);
  if (r0 < 0) return;
  float v[2 * kEdgeGroup], a0 = 0.f, ax = 0.f, ay = 0.f;
  float own = h[(size_t)r0 * HID + f];  // loaded one node ahead: no wait at a node's end
  walk_edges(
      r0, min(r0 + rows, n), off, col, w, ex, ey,
      [&](int c, int u) { v[u] = h[(size_t)c * HID + f]; },
      [&](int u, float we, float xe, float ye) {
        const float t = v[u] * we;
        a0 = __builtin_fmaf(v[u], we, a0);
        ax = __builtin_fmaf(t, xe, ax);
        ay = __builtin_fmaf(t, ye, ay);
      },
      [&](int r) {
        float *zr = z + (size_t)r * 4 * HID;
        zr[f] = own;
        own = h[(size_t)min(r + 1, n - 1) * HID + f];
        zr[HID + f] = a0;
        zr[2 * HID + f] = ax;
        zr[3 * HID + f] = ay;
        a0 = ax = ay = 0.f;
      });
}

// dh[i] = dz[i][0:64] + sum over i's edges e = (i, j) of the transpose
// weights (wt = weight of edge j -> i, (ext, eyt) its direction) times
// dz[j][64:256], plus plus[i] where given
__global__ __launch_bounds__(256) void k_aggregate_bwd(const float *__restrict__ dz, int n, int rows,
                                                       const int32_t *__restrict__ off,
                                                       const int32_t *__restrict__ col,
                                                       const float *__restrict__ wt,
                                                       const float *__restrict__ ext,
                                                       const float *__restrict__ eyt,
                                                       const float *__restrict__ plus,
                                                       float *__restrict__ dh) {
  const int f = threadIdx.x & 63, r0 = agg_first(n, rows);
  if (r0 < 0) return;
  float v0[2 * kEdgeGroup], v1[2 * kEdgeGroup], v2[2 * kEdgeGroup];
  float s = dz[(size_t)r0 * 4 * HID + f];
  float own = dz[(size_t)min(r0 + 1, n - 1) * 4 * HID + f];  // the next node's, as above
  walk_edges(
      r0, min(r0 + rows, n), off, col, wt, ext, eyt,
      [&](int c, int u) {
        const float *dj = dz + (size_t)c * 4 * HID + f;
        v0[u] = dj[HID];
        v1[u] = dj[2 * HID];
        v2[u] = dj[3 * HID];
      },
      [&](int u, float we, float xe, float ye) {
        s = __builtin_fmaf(we, __builtin_fmaf(ye, v2[u], __builtin_fmaf(xe, v1[u], v0[u])), s);
      },
      [&](int r) {
        dh[(size_t)r * HID + f] = plus ? s + plus[(size_t)r * HID + f] : s;
        s = own;
        own = dz[(size_t)min(r + 2, n - 1) * 4 * HID + f];
      });
}

static thread_local std::string g_err;

static int nn_fail(const std::string &m) {
  g_err = m;
  return FVDBM_ERR_INVALID;
}

static int hip_status(const char *what) {
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) return FVDBM_OK;
  g_err = std::string(what) + ": " + hipGetErrorString(e);
  return FVDBM_ERR_HIP;
}

static int grid_for(int64_t m) {
  const int64_t tiles = (m + 15) / 16;
  const int64_t blocks = (tiles + 3) / 4;
  return (int)(blocks < 2048 ? (blocks > 0 ? blocks : 1) : 2048);
}

// blocks of the forward kernel: as many as are resident, at least two tiles
// each so that the weights of a block pay for more than one
static int fwd_blocks(int64_t m, int k) {
  const int64_t tiles = (m + GR - 1) / GR;
  return (int)std::min<int64_t>(256 * (k == 256 ? 3 : 4), (tiles + 1) / 2);
}

template <int K, int NO>
static void launch_fwd(const float *x, int m, const float *w1, const float *b1, const float *w2,
                       const float *b2, float *y, hipStream_t s) {
  hipLaunchKernelGGL((k_mlp_fwd<K, NO, false>), dim3(fwd_blocks(m, K)), dim3(256), 0, s, x, m, w1, b1, w2, b2,
                     nullptr, y);
}

template <int K, int NO>
static void launch_bwd(const float *x, int m, const float *w1, const float *b1, const float *w2,
                       const float *dy, float *dx, float *dz, float *h, hipStream_t s) {
  hipLaunchKernelGGL((k_mlp_bwd<K, NO>), dim3(grid_for(m)), dim3(256), 0, s, x, m, w1, b1, w2, dy,
                     dx, dz, h);
}

// Blocks of the gradient kernel: two per CU, what LDS and registers hold; for
// few rows at least four tiles each, so that a block's partial sums (82 KB at
// K = 256) stay small beside its rows (164 KB).
static int grad_blocks(int64_t m) {
  const int64_t tiles = (m + GR - 1) / GR;
  return (int)std::min<int64_t>(GRAD_BLOCKS, std::max<int64_t>(1, (tiles + 3) / 4));
}

template <int K, int NO>
static void launch_grad(const float *x, int m, const float *w1, const float *b1, const float *w2,
                        const float *dy, float *dx, float *ws, float *dw1, float *db1, float *dw2,
                        float *db2, hipStream_t s) {
  const int blocks = grad_blocks(m), n = grad_floats(K, NO);
  if (dx)
    hipLaunchKernelGGL((k_mlp_grad<K, NO, true>), dim3(blocks), dim3(256), 0, s, x, m, w1, b1, w2, dy, dx, ws);
  else
    hipLaunchKernelGGL((k_mlp_grad<K, NO, false>), dim3(blocks), dim3(256), 0, s, x, m, w1, b1, w2, dy, dx, ws);
  const int bx = (n + 255) / 256;
  hipLaunchKernelGGL(k_reduce_groups, dim3(bx, (blocks + RGROUP - 1) / RGROUP), dim3(256), 0, s, ws, blocks, n);
  hipLaunchKernelGGL(k_reduce_grads, dim3(bx), dim3(256), 0, s, ws, blocks, K * HID, HID * NO, HID, NO,
                     dw1, dw2, db1, db2);
}

template <int KA, int NB>
static void launch_wgrad(const float *a, const float *b, int m, float *partial, hipStream_t s) {
  const int nch = (m + CHUNK - 1) / CHUNK;
  hipLaunchKernelGGL((k_wgrad<KA, NB>), dim3(nch), dim3(256), 0, s, a, b, m, partial);
}

// out [n] = sum over the nch chunk partials [nch][n] in a fixed order (in
// groups of RGROUP chunks, then the groups); overwrites the partials
static void launch_reduce(float *partial, int nch, int n, float *out, hipStream_t s) {
  const int bx = (n + 255) / 256;
  hipLaunchKernelGGL(k_reduce_groups, dim3(bx, (nch + RGROUP - 1) / RGROUP), dim3(256), 0, s,
                     partial, nch, n);
  hipLaunchKernelGGL(k_reduce_final, dim3(bx), dim3(256), 0, s, partial, nch, n, out);
}

// ---------------------------------------------------------------------------
// Allocation-free weight gradient (fvdbm_nn_wgrad_noalloc): the per-chunk
// partial products live in this file-scope device array instead of a
// caller workspace. Each GPU holds its own copy for the life of the
// process. Its host-side name is not a device address: the address on the
// current device comes from hipGetSymbolAddress, looked up once per device
// and kept in scratch_dev. k_wgrad writes every word of the partials it
// reduces, so nothing needs clearing between calls; calls that overlap on
// one GPU share the array and race.
// ---------------------------------------------------------------------------
constexpr size_t kScratchFloats = size_t(4) << 20;  // 16 MiB
static __device__ __align__(256) float scratch[kScratchFloats];

constexpr int kMaxDevices = 64;
static std::mutex scratch_mu;
static float *scratch_dev[kMaxDevices] = {};

// The scratch array's address on the current device (looked up on a
// device's first call).
static int scratch_on_current_device(float **out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    g_err = std::string("hipGetDevice: ") + hipGetErrorString(e);
    return FVDBM_ERR_HIP;
  }
  if (dev < 0 || dev >= kMaxDevices) return nn_fail("device ordinal out of range");
  std::lock_guard<std::mutex> lock(scratch_mu);
  if (!scratch_dev[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      g_err = std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e);
      return FVDBM_ERR_HIP;
    }
    scratch_dev[dev] = static_cast<float *>(p);
  }
  *out = scratch_dev[dev];
  return FVDBM_OK;
}

}  // namespace fvdbm_nn

using namespace fvdbm_nn;

extern "C" {

const char *fvdbm_nn_last_error(void) { return g_err.c_str(); }

int fvdbm_nn_chunk_rows(void) { return CHUNK; }

// the dense kernels move four floats per lane: their row arrays must be
// 16-byte aligned
static bool aligned16(const void *p) { return p == nullptr || ((uintptr_t)p & 15u) == 0; }

#define NN_DISPATCH_K_NO(K_, NO_, CALL) \
  if (k == K_ && n_out == NO_) {        \
    CALL(K_, NO_);                      \
    return hip_status("mlp launch");    \
  }

int fvdbm_nn_mlp_forward(const float *x, int64_t m, int32_t k, const float *w1, const float *b1,
                         const float *w2, const float *b2, int32_t n_out, float *y, void *stream) {
  if (m < 0 || m > INT32_MAX) return nn_fail("row count out of range");
  if (m == 0) return FVDBM_OK;
  if (!x || !w1 || !b1 || !w2 || !b2 || !y) return nn_fail("null pointer");
  if (!aligned16(x) || !aligned16(y)) return nn_fail("x and y must be 16-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int mi = (int)m;
#define CALL_FWD(K_, NO_) launch_fwd<K_, NO_>(x, mi, w1, b1, w2, b2, y, s)
  NN_DISPATCH_K_NO(16, 64, CALL_FWD)
  NN_DISPATCH_K_NO(64, 64, CALL_FWD)
  NN_DISPATCH_K_NO(256, 64, CALL_FWD)
  NN_DISPATCH_K_NO(64, 16, CALL_FWD)
#undef CALL_FWD
  return nn_fail("unsupported (in, out) widths: (16|64|256, 64) or (64, 16)");
}

int fvdbm_nn_mlp_backward(const float *x, int64_t m, int32_t k, const float *w1, const float *b1,
                          const float *w2, int32_t n_out, const float *dy, float *dx, float *dz,
                          float *h, void *stream) {
  if (m < 0 || m > INT32_MAX) return nn_fail("row count out of range");
  if (m == 0) return FVDBM_OK;
  if (!x || !w1 || !b1 || !w2 || !dy || !dz || !h) return nn_fail("null pointer");
  if (!aligned16(x) || !aligned16(dy) || !aligned16(dx) || !aligned16(dz) || !aligned16(h))
    return nn_fail("x, dy, dx, dz and h must be 16-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int mi = (int)m;
#define CALL_BWD(K_, NO_) launch_bwd<K_, NO_>(x, mi, w1, b1, w2, dy, dx, dz, h, s)
  NN_DISPATCH_K_NO(16, 64, CALL_BWD)
  NN_DISPATCH_K_NO(64, 64, CALL_BWD)
  NN_DISPATCH_K_NO(256, 64, CALL_BWD)
  NN_DISPATCH_K_NO(64, 16, CALL_BWD)
#undef CALL_BWD
  return nn_fail("unsupported (in, out) widths: (16|64|256, 64) or (64, 16)");
}

int64_t fvdbm_nn_mlp_gradients_floats(int64_t m, int32_t k, int32_t n_out) {
  if (m < 0 || m > INT32_MAX || k < 0 || k > 256 || n_out < 0 || n_out > 64) return 0;
  return (int64_t)grad_blocks(m) * grad_floats(k, n_out);
}

int fvdbm_nn_mlp_gradients(const float *x, int64_t m, int32_t k, const float *w1, const float *b1,
                           const float *w2, int32_t n_out, const float *dy, float *dx, float *dw1,
                           float *db1, float *dw2, float *db2, float *workspace, void *stream) {
  if (m < 0 || m > INT32_MAX) return nn_fail("row count out of range");
  if (!dw1 || !db1 || !dw2 || !db2) return nn_fail("null pointer");
  if (m > 0 && (!x || !w1 || !b1 || !w2 || !dy || !workspace)) return nn_fail("null pointer");
  if (!aligned16(x) || !aligned16(dy) || !aligned16(dx)) return nn_fail("x, dy and dx must be 16-byte aligned");
  if (!((n_out == 64 && (k == 16 || k == 64 || k == 256)) || (n_out == 16 && k == 64)))
    return nn_fail("unsupported (in, out) widths: (16|64|256, 64) or (64, 16)");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int mi = (int)m;
  if (mi == 0) {
    auto zero = [&](float *p, int n) {
      hipLaunchKernelGGL(k_zero, dim3((n + 255) / 256), dim3(256), 0, s, p, n);
    };
    zero(dw1, k * HID);
    zero(db1, HID);
    zero(dw2, HID * n_out);
    zero(db2, n_out);
    return hip_status("zero launch");
  }
#define CALL_GRAD(K_, NO_) \
  launch_grad<K_, NO_>(x, mi, w1, b1, w2, dy, dx, workspace, dw1, db1, dw2, db2, s)
  NN_DISPATCH_K_NO(16, 64, CALL_GRAD)
  NN_DISPATCH_K_NO(64, 64, CALL_GRAD)
  NN_DISPATCH_K_NO(256, 64, CALL_GRAD)
  NN_DISPATCH_K_NO(64, 16, CALL_GRAD)
#undef CALL_GRAD
  return nn_fail("unsupported (in, out) widths: (16|64|256, 64) or (64, 16)");
}

int fvdbm_nn_wgrad(const float *a, const float *b, int64_t m, int32_t ka, int32_t nb, float *partial,
                   float *out, void *stream) {
  if (m < 0 || m > INT32_MAX) return nn_fail("row count out of range");
  if (!a || !b || !partial || !out) return nn_fail("null pointer");
  if (!aligned16(a) || !aligned16(b)) return nn_fail("a and b must be 16-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int mi = (int)m;
  const int nch = (mi + CHUNK - 1) / CHUNK;
  if (mi == 0) {
    hipLaunchKernelGGL(k_zero, dim3((ka * nb + 255) / 256), dim3(256), 0, s, out, ka * nb);
    return hip_status("zero launch");
  }
  if (ka == 16 && nb == 64) launch_wgrad<16, 64>(a, b, mi, partial, s);
  else if (ka == 64 && nb == 64) launch_wgrad<64, 64>(a, b, mi, partial, s);
  else if (ka == 256 && nb == 64) launch_wgrad<256, 64>(a, b, mi, partial, s);
  else if (ka == 64 && nb == 16) launch_wgrad<64, 16>(a, b, mi, partial, s);
  else return nn_fail("unsupported wgrad widths");
  launch_reduce(partial, nch, ka * nb, out, s);
  return hip_status("wgrad launch");
}

int fvdbm_nn_wgrad_noalloc(const float *a, const float *b, int64_t m, int32_t ka, int32_t nb,
                           float *out, void *stream) {
  if (m < 0 || m > INT32_MAX) return nn_fail("row count out of range");
  if (!a || !b || !out) return nn_fail("null pointer");
  if (!aligned16(a) || !aligned16(b)) return nn_fail("a and b must be 16-byte aligned");
  if (!((ka == 16 && nb == 64) || (ka == 64 && nb == 64) || (ka == 256 && nb == 64) ||
        (ka == 64 && nb == 16)))
    return nn_fail("unsupported wgrad widths");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int mi = (int)m;
  const int n = ka * nb;
  const int64_t nch = (m + CHUNK - 1) / CHUNK;
  if ((uint64_t)nch * (uint64_t)n > kScratchFloats)
    return nn_fail("fvdbm_nn_wgrad_noalloc: " + std::to_string(m) + " rows need " +
                   std::to_string(nch * n) + " partial floats, more than the " +
                   std::to_string(kScratchFloats) + " of the static scratch (at most " +
                   std::to_string((int64_t)(kScratchFloats / n) * CHUNK) + " rows for widths (" +
                   std::to_string(ka) + ", " + std::to_string(nb) + "))");
  if (mi == 0) {
    hipLaunchKernelGGL(k_zero, dim3((n + 255) / 256), dim3(256), 0, s, out, n);
    return hip_status("zero launch");
  }
  float *partial = nullptr;
  const int rc = scratch_on_current_device(&partial);
  if (rc) return rc;
  if (ka == 16) launch_wgrad<16, 64>(a, b, mi, partial, s);
  else if (ka == 256) launch_wgrad<256, 64>(a, b, mi, partial, s);
  else if (nb == 64) launch_wgrad<64, 64>(a, b, mi, partial, s);
  else launch_wgrad<64, 16>(a, b, mi, partial, s);
  launch_reduce(partial, (int)nch, n, out, s);
  return hip_status("wgrad launch");
}

int fvdbm_nn_colsum(const float *a, int64_t m, int32_t n, float *partial, float *out, void *stream) {
  if (m < 0 || m > INT32_MAX) return nn_fail("row count out of range");
  if (!a || !partial || !out) return nn_fail("null pointer");
  if (n < 1 || n > 256) return nn_fail("column count must be in [1, 256]");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int mi = (int)m;
  const int nch = (mi + CHUNK - 1) / CHUNK;
  if (mi == 0) {
    hipLaunchKernelGGL(k_zero, dim3(1), dim3(256), 0, s, out, n);
    return hip_status("zero launch");
  }
  hipLaunchKernelGGL(k_colsum, dim3(nch), dim3(256), 0, s, a, mi, n, partial);
  launch_reduce(partial, nch, n, out, s);
  return hip_status("colsum launch");
}

int fvdbm_nn_aggregate(const float *h, int64_t n_nodes, const int32_t *row_off, const int32_t *col,
                       const float *w, const float *ex, const float *ey, float *z, void *stream) {
  if (n_nodes < 0 || n_nodes > INT32_MAX) return nn_fail("node count out of range");
  if (n_nodes == 0) return FVDBM_OK;
  if (!h || !row_off || !col || !w || !ex || !ey || !z) return nn_fail("null pointer");
  const int n = (int)n_nodes;
  const int rows = n < kAggSmallNodes ? kAggRowsSmall : kAggRows;
  hipLaunchKernelGGL(k_aggregate, dim3((n + 4 * rows - 1) / (4 * rows)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), h, n, rows, row_off, col, w, ex, ey, z);
  return hip_status("aggregate launch");
}

int fvdbm_nn_aggregate_backward(const float *dz, int64_t n_nodes, const int32_t *row_off,
                                const int32_t *col, const float *wt, const float *ext,
                                const float *eyt, float *dh, void *stream) {
  if (n_nodes < 0 || n_nodes > INT32_MAX) return nn_fail("node count out of range");
  if (n_nodes == 0) return FVDBM_OK;
  if (!dz || !row_off || !col || !wt || !ext || !eyt || !dh) return nn_fail("null pointer");
  const int n = (int)n_nodes;
  const int rows = n < kAggSmallNodes ? kAggRowsSmall : kAggRows;
  hipLaunchKernelGGL(k_aggregate_bwd, dim3((n + 4 * rows - 1) / (4 * rows)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), dz, n, rows, row_off, col, wt, ext, eyt, nullptr, dh);
  return hip_status("aggregate backward launch");
}

int fvdbm_nn_layer_forward(const float *h, int64_t n_nodes, const int32_t *row_off, const int32_t *col,
                           const float *w, const float *ex, const float *ey, const float *w1,
                           const float *b1, const float *w2, const float *b2, float *z, float *y,
                           void *stream) {
  if (n_nodes < 0 || n_nodes > INT32_MAX) return nn_fail("node count out of range");
  if (n_nodes == 0) return FVDBM_OK;
  if (!w1 || !b1 || !w2 || !b2 || !y) return nn_fail("null pointer");
  if (!aligned16(h) || !aligned16(z) || !aligned16(y)) return nn_fail("h, z and y must be 16-byte aligned");
  const int rc = fvdbm_nn_aggregate(h, n_nodes, row_off, col, w, ex, ey, z, stream);
  if (rc) return rc;
  hipLaunchKernelGGL((k_mlp_fwd<256, 64, true>), dim3(fwd_blocks(n_nodes, 4 * HID)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), z, (int)n_nodes, w1, b1, w2, b2, h, y);
  return hip_status("layer launch");
}

int fvdbm_nn_layer_backward(const float *z, int64_t n_nodes, const int32_t *row_off, const int32_t *col,
                            const float *wt, const float *ext, const float *eyt, const float *w1,
                            const float *b1, const float *w2, const float *dy, float *dz, float *dh,
                            float *dw1, float *db1, float *dw2, float *db2, float *workspace,
                            void *stream) {
  if (dh && !dz) return nn_fail("null pointer");
  if (dh && n_nodes > 0 && (!row_off || !col || !wt || !ext || !eyt)) return nn_fail("null pointer");
  const int rc = fvdbm_nn_mlp_gradients(z, n_nodes, 4 * HID, w1, b1, w2, HID, dy, dh ? dz : nullptr, dw1, db1,
                                        dw2, db2, workspace, stream);
  if (rc || !dh || n_nodes == 0) return rc;
  const int n = (int)n_nodes;
  const int rows = n < kAggSmallNodes ? kAggRowsSmall : kAggRows;
  hipLaunchKernelGGL(k_aggregate_bwd, dim3((n + 4 * rows - 1) / (4 * rows)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), dz, n, rows, row_off, col, wt, ext, eyt, dy, dh);
  return hip_status("layer backward launch");
}

}  // extern "C"
