// Conversion between the device layout (one plane per component, device cell
// order) and host arrays (one row per cell or node, reference order) on the
// device, so that a field crosses the bus as the caller's rows in one copy.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>

namespace fvdbm {

// Where plane slot i of a field lives: row map[i] (-1 = none; null map:
// row i) and, for batched handles, which of two buffers holds it (slot i
// belongs to case tile_case[i / block], whose buffer is case_cur).
struct RowMap {
  const int32_t *map = nullptr;
  const int32_t *tile_case = nullptr, *case_cur = nullptr;
  int block = 1;
  __device__ __forceinline__ int row(int i) const { return map ? map[i] : i; }
  __device__ __forceinline__ bool second(int i) const {
    return tile_case && case_cur[tile_case[i / block]] != 0;
  }
};

// rows[row(i) - first][q] = planes[q][i] for the n slots whose row is one of the
// `count` from `first`, COMPS components, planes `stride` apart. Bound by the bus
// copy that follows: 36 MB of pdf rows (1M cells) take 0.05 ms here; the same
// reordering on the host took 12 ms.
template <typename T, int COMPS>
__global__ void k_planes_to_rows(const T *__restrict__ p0, const T *__restrict__ p1, size_t stride,
                                 int n, RowMap m, int first, int count, T *__restrict__ rows) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int o = m.row(i) - first;
  if (o < 0 || o >= count) return;
  const T *p = m.second(i) ? p1 : p0;
#pragma unroll
  for (int q = 0; q < COMPS; ++q) rows[(size_t)o * COMPS + q] = p[(size_t)q * stride + i];
}

// The reverse; slots without a row become 0.
template <typename T, int COMPS>
__global__ void k_rows_to_planes(const T *__restrict__ rows, int n, RowMap m, int first, int count,
                                 T *__restrict__ p0, T *__restrict__ p1, size_t stride) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int row = m.row(i), o = row - first;
  if (row >= 0 && (o < 0 || o >= count)) return;
  T *p = m.second(i) ? p1 : p0;
#pragma unroll
  for (int q = 0; q < COMPS; ++q)
    p[(size_t)q * stride + i] = row < 0 ? T(0) : rows[(size_t)o * COMPS + q];
}

// A handle's row buffers, kept between calls: device memory for large fields,
// pinned host memory for small ones (the kernels write and read it directly,
// which spares the copy engine's start and a pageable copy's page locking:
// reading 74 KB takes 20 us against 54, 2 MB 130 against 156, and from there
// there is no difference; writing pays up to 1 MB). A larger field than
// kDeviceRows passes in parts, one pass over the slots each, and where the device
// has no memory left through the pinned buffer. Used on the handle's stream,
// which is idle when a call returns.
class RowIO {
 public:
  RowIO() = default;
  RowIO(const RowIO &) = delete;
  RowIO &operator=(const RowIO &) = delete;
  ~RowIO() {
    if (dev_) (void)hipFree(dev_);
    if (pinned_) (void)hipHostFree(pinned_);
  }
  int64_t device_bytes() const { return (int64_t)dev_bytes_; }

  // `rows` rows of COMPS values to dst, from planes of n slots.
  template <typename T, int COMPS>
  hipError_t out(hipStream_t s, const void *p0, const void *p1, int n, RowMap m, size_t rows,
                 void *dst) {
    return parts(s, rows, COMPS * sizeof(T), kPinnedOut, [&](bool small, int first, int count) {
      const size_t at = (size_t)first * COMPS * sizeof(T), bytes = (size_t)count * COMPS * sizeof(T);
      hipLaunchKernelGGL((k_planes_to_rows<T, COMPS>), dim3((n + 255) / 256), dim3(256), 0, s,
                         static_cast<const T *>(p0), static_cast<const T *>(p1), (size_t)n, n, m, first,
                         count, static_cast<T *>(small ? pinned_ : dev_));
      hipError_t e = hipGetLastError();
      char *to = static_cast<char *>(dst) + at;
      if (e == hipSuccess && !small) e = hipMemcpyAsync(to, dev_, bytes, hipMemcpyDeviceToHost, s);
      if (e == hipSuccess) e = hipStreamSynchronize(s);
      if (e == hipSuccess && small) std::memcpy(to, pinned_, bytes);
      return e;
    });
  }

  // The reverse, from src.
  template <typename T, int COMPS>
  hipError_t in(hipStream_t s, void *p0, void *p1, int n, RowMap m, size_t rows, const void *src) {
    return parts(s, rows, COMPS * sizeof(T), kPinnedIn, [&](bool small, int first, int count) {
      const size_t at = (size_t)first * COMPS * sizeof(T), bytes = (size_t)count * COMPS * sizeof(T);
      const char *from = static_cast<const char *>(src) + at;
      hipError_t e = hipSuccess;
      if (small)
        std::memcpy(pinned_, from, bytes);
      else
        e = hipMemcpyAsync(dev_, from, bytes, hipMemcpyHostToDevice, s);
      if (e != hipSuccess) return e;
      hipLaunchKernelGGL((k_rows_to_planes<T, COMPS>), dim3((n + 255) / 256), dim3(256), 0, s,
                         static_cast<const T *>(small ? pinned_ : dev_), n, m, first, count,
                         static_cast<T *>(p0), static_cast<T *>(p1), (size_t)n);
      e = hipGetLastError();
      return e == hipSuccess ? hipStreamSynchronize(s) : e;
    });
  }

 private:
  static constexpr size_t kPinnedOut = 2u << 20, kPinnedIn = 1u << 20, kDeviceRows = 64u << 20;
  void *dev_ = nullptr, *pinned_ = nullptr;
  size_t dev_bytes_ = 0, pinned_bytes_ = 0;

  // pass(small, first row, rows) for as many rows of `row` bytes at a time as
  // the buffer holds: the pinned one for up to `pinned` bytes in all.
  template <typename Pass>
  hipError_t parts(hipStream_t s, size_t rows, size_t row, size_t pinned, Pass pass) {
    const size_t bytes = rows * row;
    bool small = bytes <= pinned;
    hipError_t e = reserve(s, small, small ? bytes : std::min(bytes, kDeviceRows));
    if (e == hipErrorOutOfMemory && !small) {
      (void)hipGetLastError();  // leave no error for the next launch check to report
      small = true;
      e = reserve(s, small, pinned);
    }
    if (e != hipSuccess) return e;
    const size_t most = std::max<size_t>((small ? pinned : kDeviceRows) / row, 1);
    for (size_t first = 0; first < rows && e == hipSuccess; first += most)
      e = pass(small, (int)first, (int)std::min(most, rows - first));
    return e;
  }

  hipError_t reserve(hipStream_t s, bool small, size_t bytes) {
    void *&p = small ? pinned_ : dev_;
    size_t &have = small ? pinned_bytes_ : dev_bytes_;
    if (have >= bytes) return hipSuccess;
    hipError_t e = hipStreamSynchronize(s);
    if (e != hipSuccess) return e;
    if (p) (void)(small ? hipHostFree(p) : hipFree(p));
    p = nullptr;
    have = 0;
    e = small ? hipHostMalloc(&p, bytes, hipHostMallocDefault) : hipMalloc(&p, bytes);
    if (e == hipSuccess) have = bytes;
    return e;
  }
};

}  // namespace fvdbm
