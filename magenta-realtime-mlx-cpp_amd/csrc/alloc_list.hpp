// The allocations that an object frees with itself.
#pragma once

#include <cstddef>
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

// Allocations that are of use together only: kept as a whole or given back.
// Dev: bool alloc(void** p, size_t bytes), false when there is no memory (other
// errors throw), free(void* p) and sync(), which waits for the work that writes
// them.
template <class Dev>
class AllocGroup {
 public:
  explicit AllocGroup(Dev dev) : dev_(dev) {}
  AllocGroup(const AllocGroup&) = delete;
  AllocGroup& operator=(const AllocGroup&) = delete;
  ~AllocGroup() {
    if (ps_.empty()) return;
    try {
      dev_.sync();
    } catch (...) {  // freed all the same
    }
    for (void* p : ps_) dev_.free(p);
  }
  // nullptr once there was no memory.
  void* alloc(size_t bytes) {
    void* p = nullptr;
    if (full_ || !dev_.alloc(&p, bytes)) {
      full_ = true;
      return nullptr;
    }
    ps_.push_back(p);
    return p;
  }
  // Waits and hands all to the list; false, with everything given back, where an
  // allocation was refused.
  bool keep(AllocList& list) {
    dev_.sync();
    if (!full_) list.add(ps_);
    if (full_)
      for (void* p : ps_) dev_.free(p);
    ps_.clear();
    return !full_;
  }

 private:
  Dev dev_;
  std::vector<void*> ps_;
  bool full_ = false;
};

}  // namespace mrt
