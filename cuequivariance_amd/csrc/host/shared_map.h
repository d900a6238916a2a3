// A small map that threads add to and look up in at the same time: PyTorch runs a backward on threads of its own, without the
// interpreter's lock, while another thread's call may be adding an entry.  Entries are handed out as copies.
#pragma once

#include <mutex>
#include <optional>
#include <unordered_map>

namespace cueq_host {

template <typename T>
class SharedMap {
 public:
  std::optional<T> find(int key) const {
    std::lock_guard<std::mutex> lock(mutex_);
    const auto it = map_.find(key);
    return it == map_.end() ? std::nullopt : std::optional<T>(it->second);
  }
  void set(int key, T value) {
    std::lock_guard<std::mutex> lock(mutex_);
    map_[key] = std::move(value);
  }

 private:
  mutable std::mutex mutex_;
  std::unordered_map<int, T> map_;
};

}  // namespace cueq_host
