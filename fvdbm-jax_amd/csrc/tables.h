// Small tables of a handle share one allocation and one copy: to set up the
// 2048-cell cavity takes 0.8 ms so, with D2Q13 1.3 ms by an allocation and a copy
// for each table.
#pragma once

#include <cstddef>
#include <cstring>
#include <utility>
#include <vector>

namespace fvdbm {

class SmallTables {
 public:
  static constexpr size_t kMost = 65536;  // bytes of a table taken

  // Keeps v for flush, which sets *out.
  template <typename V>
  void add(void **out, const std::vector<V> &v) {
    const size_t n = v.size() * sizeof(V);
    at_.push_back({out, bytes_.size()});
    bytes_.resize(bytes_.size() + ((n + 255) & ~(size_t)255) + (n == 0 ? 256 : 0));
    if (n) std::memcpy(bytes_.data() + at_.back().second, v.data(), n);
  }
  const std::vector<unsigned char> &bytes() const { return bytes_; }
  // The tables are at `base` on the device.
  void placed(void *base) {
    for (auto &t : at_) *t.first = static_cast<unsigned char *>(base) + t.second;
    bytes_ = {};
    at_ = {};
  }

 private:
  std::vector<unsigned char> bytes_;
  std::vector<std::pair<void **, size_t>> at_;
};

}  // namespace fvdbm
