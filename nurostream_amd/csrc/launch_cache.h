// What the runtime answered once about a kernel, kept for the launches after it (host only, no HIP: the callers ask).
#pragma once

#include <cstddef>
#include <map>
#include <mutex>
#include <tuple>

// An answer per (kernel, LDS bytes, threads, device). The keys are a process's kernels times the LDS sizes that its
// shapes take, so the table grows to that and holds all of them: one that stopped growing would ask the runtime at every
// later launch of what came too late.
class NsxLaunchCache {
 public:
  template <typename Ask>
  int get(const void* kernel, size_t lds, int threads, int dev, Ask&& ask) {
    const std::lock_guard<std::mutex> lock(mu_);
    const Key key{kernel, lds, threads, dev};
    const auto it = table_.find(key);
    if (it != table_.end()) return it->second;
    const int v = ask();
    try {
      table_.emplace(key, v);
    } catch (...) {  // out of memory: asked again next time
    }
    return v;
  }

 private:
  using Key = std::tuple<const void*, size_t, int, int>;
  std::mutex mu_;
  std::map<Key, int> table_;
};

// The dynamic LDS size each kernel was allowed, per device: raised when a launch needs more, never lowered (a smaller
// launch in between would take it from a larger one).
class NsxLdsLimits {
 public:
  // set(lds) -> 0 or an error, which is returned and not remembered
  template <typename Set>
  int allow(const void* kernel, int dev, size_t lds, Set&& set) {
    const std::lock_guard<std::mutex> lock(mu_);
    const auto key = std::make_pair(kernel, dev);
    const auto it = limit_.find(key);
    if (it != limit_.end() && it->second >= lds) return 0;
    if (const int rc = set(lds)) return rc;
    try {
      limit_[key] = lds;
    } catch (...) {  // out of memory: set again next time
    }
    return 0;
  }

 private:
  std::mutex mu_;
  std::map<std::pair<const void*, int>, size_t> limit_;
};
