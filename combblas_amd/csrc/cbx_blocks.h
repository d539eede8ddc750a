// The caching allocator's block sizes and lists, free of HIP so that the host
// can test them.
#pragma once

#include <cstddef>
#include <map>
#include <unordered_map>
#include <vector>

namespace cbx {

// The size of a new block for `bytes`: rounded up to an eighth of its leading
// power of two, so that products whose sizes differ by a few percent (the
// column phases of an MCL expansion) find each other's blocks, but by less than
// kBlockStep, so that the largest products keep the card's memory (unbounded,
// ir and val of R-MAT s20 took 16 GB more than their 156).  Twelve MCL
// expansions of new matrices of 480 to 535 K columns (blocks of 20 to 30 GB):
// 82 to 92 ms each with this bound and without one; with 256 MB two of them took
// 0.4 and 1.6 s to give blocks back, with 16 MB one 3 s.
constexpr size_t kBlockStep = (size_t)1 << 30;
inline size_t block_bytes(size_t bytes) {
  size_t step = 256;
  while (step < kBlockStep && step * 16 <= bytes) step *= 2;
  return (bytes + step - 1) / step * step;
}

// Blocks in use and idle ones, by device (not thread-safe).
class BlockLists {
  struct Block {
    int device;
    size_t bytes;
  };
  struct Idle {
    std::multimap<size_t, void*> blocks;
    size_t bytes = 0;
  };
  std::unordered_map<void*, Block> live_;
  std::vector<Idle> idle_;  // by device

 public:
  // An idle block of the device for `bytes`, not much larger; null if there is none.
  void* take(int device, size_t bytes) {
    if ((size_t)device >= idle_.size()) return nullptr;
    Idle& d = idle_[(size_t)device];
    const auto it = d.blocks.lower_bound(bytes);
    if (it == d.blocks.end() || it->first > bytes + bytes / 4 + (1u << 20)) return nullptr;
    void* p = it->second;
    live_[p] = Block{device, it->first};
    d.bytes -= it->first;
    d.blocks.erase(it);
    return p;
  }
  // A block newly allocated on the device.
  void add(void* p, int device, size_t bytes) {
    if ((size_t)device >= idle_.size()) idle_.resize((size_t)device + 1);
    live_[p] = Block{device, bytes};
  }
  // A block in use becomes idle; false if p is none.
  bool give_back(void* p) {
    const auto it = live_.find(p);
    if (it == live_.end()) return false;
    Idle& d = idle_[(size_t)it->second.device];
    d.blocks.emplace(it->second.bytes, p);
    d.bytes += it->second.bytes;
    live_.erase(it);
    return true;
  }
  size_t idle_bytes(int device) const { return (size_t)device < idle_.size() ? idle_[(size_t)device].bytes : 0; }
  // Every idle block to f, and off the lists.
  template <class F>
  void release(F&& f) {
    for (Idle& d : idle_) {
      for (auto& b : d.blocks) f(b.second);
      d = Idle{};
    }
  }
};

}  // namespace cbx
