// Tables of a population laid out one after the other in one device
// allocation, the small ones in one copy, and space behind them.  A population
// has a dozen and a half of them, and an allocation with its copy takes 15-20 us
// each (1024 olive cells' CN engine: 0.85 -> 0.63 ms to create).
#pragma once
#include <hip/hip_runtime.h>

#include <cstring>
#include <functional>
#include <memory>
#include <vector>

#include "engine.hpp"

namespace cbrkc {

class TablePack {
 public:
  // dst points to a device copy of h after upload()
  template <class P, class T>
  void put(P *&dst, std::vector<T> &&h) {
    auto own = std::make_shared<std::vector<T>>(std::move(h));
    keep_.push_back(own);
    put_static(dst, *own);
  }
  // the same for a table that outlives upload()
  template <class P, class T>
  void put_static(P *&dst, const std::vector<T> &h) {
    static_assert(sizeof(P) == sizeof(T), "the table's element");
    tables_.push_back({(const void *)h.data(), sizeof(T) * h.size(), [&dst](char *at) { dst = (P *)at; }});
  }
  // dst points to n doubles behind the tables after upload(), one such space after the other
  void space(double *&dst, size_t n) {
    const size_t at = space_;
    space_ += n;
    spaces_.push_back([&dst, at](double *base) { dst = base + at; });
  }
  size_t spaces() const { return space_; }   // doubles in all
  // the allocation; its spaces begin at *space
  void *upload(double **space = nullptr) {
    size_t bytes = 0;
    std::vector<char> small;
    for (int large = 0; large < 2; large++)
      for (Table &t : tables_)
        if ((t.n > SMALL) == (large != 0)) {
          t.at = bytes;
          bytes += (t.n + 255) & ~(size_t)255;
          if (large) continue;
          small.resize(bytes);
          if (t.n) std::memcpy(&small[t.at], t.h, t.n);
        }
    char *base = nullptr;
    CB_HIP(hipMalloc((void **)&base, bytes + sizeof(double) * space_ + 1));
    hipError_t e = hipMemcpy(base, small.data(), small.size(), hipMemcpyHostToDevice);
    for (const Table &t : tables_) {
      if (t.n > SMALL && e == hipSuccess) e = hipMemcpy(base + t.at, t.h, t.n, hipMemcpyHostToDevice);
      t.fix(base + t.at);
    }
    if (e != hipSuccess) {
      (void)hipFree(base);
      CB_HIP(e);
    }
    for (auto &f : spaces_) f((double *)(base + bytes));
    if (space) *space = (double *)(base + bytes);
    return base;
  }

 private:
  static constexpr size_t SMALL = 1 << 14;
  struct Table {
    const void *h;
    size_t n;
    std::function<void(char *)> fix;
    size_t at = 0;
  };
  std::vector<Table> tables_;
  std::vector<std::shared_ptr<void>> keep_;
  std::vector<std::function<void(double *)>> spaces_;
  size_t space_ = 0;
};

}  // namespace cbrkc
