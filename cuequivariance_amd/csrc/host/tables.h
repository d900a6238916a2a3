// Tables of a call that the kernels read from device memory: packed one after the other, uploaded to a device in one piece at the
// first call that needs them (an inference never uploads those of the gradients).
#pragma once

#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

#include "host.h"

namespace cueq_host {

class DeviceTables {
 public:
  // (before the first use) the number of the table
  int add(const void* data, size_t bytes) {
    bytes_.resize((bytes_.size() + 15) / 16 * 16);
    at_.push_back(bytes_.size());
    size_.push_back(bytes);
    bytes_.append(static_cast<const char*>(data), bytes);
    return static_cast<int>(at_.size()) - 1;
  }
  int add(const std::string& s) { return add(s.data(), s.size()); }
  int add(const std::vector<int64_t>& v) { return add(v.data(), v.size() * sizeof(int64_t)); }

  bool empty() const { return at_.empty(); }
  int count(int table, int entry_bytes) const { return static_cast<int>(size_[table] / entry_bytes); }
  template <typename T = void>
  const T* on(at::Device device, int table) {
    std::lock_guard<std::mutex> lock(mutex_);
    auto it = devices_.find(device.index());
    if (it == devices_.end())
      it = devices_.emplace(device.index(), at::from_blob(bytes_.data(), {static_cast<int64_t>(bytes_.size())}, at::kByte).to(device)).first;
    return reinterpret_cast<const T*>(static_cast<const char*>(it->second.data_ptr()) + at_[table]);
  }
  // Whether they are there or may be uploaded now: a first call that is captured into a HIP graph has to do without.
  bool at_hand(at::Device device) {
    std::lock_guard<std::mutex> lock(mutex_);
    return devices_.count(device.index()) || !capturing();
  }

 private:
  std::string bytes_;
  std::vector<size_t> at_, size_;
  std::mutex mutex_;
  std::unordered_map<int, at::Tensor> devices_;
};

// contiguous, 16-byte aligned, of that type
inline at::Tensor rows_of(const at::Tensor& t, at::ScalarType dtype) {
  at::Tensor r = t.to(dtype).contiguous();
  return reinterpret_cast<uintptr_t>(r.data_ptr()) % 16 ? r.clone() : r;
}

}  // namespace cueq_host
