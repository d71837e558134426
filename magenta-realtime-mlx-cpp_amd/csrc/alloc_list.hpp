// The allocations that an object frees with itself.
#pragma once

#include <mutex>
#include <vector>

namespace mrt {

// Additions come from any thread: the parts of a model that are built on first
// use (q/k/v tables, laid-out weights, staging) have a lock each, which does not
// exclude the others.
class AllocList {
 public:
  void add(void* p) {
    std::lock_guard<std::mutex> lock(mu_);
    p_.push_back(p);
  }
  void add(const std::vector<void*>& ps) {
    std::lock_guard<std::mutex> lock(mu_);
    p_.insert(p_.end(), ps.begin(), ps.end());
  }
  // free_one(p) of every allocation, once; no additions meanwhile.
  template <class F>
  void drain(F&& free_one) {
    std::lock_guard<std::mutex> lock(mu_);
    for (void* p : p_) free_one(p);
    p_.clear();
  }

 private:
  std::mutex mu_;
  std::vector<void*> p_;
};

}  // namespace mrt
