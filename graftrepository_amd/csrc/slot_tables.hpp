// slot_tables.hpp -- host tables of a bank: which slot holds a node id, and
// which slots are free.
//
// A bank update looks up, drops and adds an entry per node while the route
// that follows waits for it; flat tables take a cache line or two per entry
// where node-based maps and trees take an allocation and a chain of misses.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <vector>

namespace grm {

// Node id -> slot, open addressing with linear probing.  Any id may be a
// key; slots are below UINT64_MAX, which marks an empty cell.
class IdTable {
 public:
  size_t size() const { return size_; }

  // Room for n entries at most half full.
  void reserve(size_t n) {
    size_t want = 16;
    while (want < 2 * n) want *= 2;
    if (want > cells_.size()) rehash(want);
  }

  uint64_t* find(uint64_t id) {
    if (cells_.empty()) return nullptr;
    Cell& c = cells_[place(id)];
    return c.slot == kEmpty ? nullptr : &c.slot;
  }

  // False (and no change) when the id is there already.
  bool emplace(uint64_t id, uint64_t slot) {
    reserve(size_ + 1);
    Cell& c = cells_[place(id)];
    if (c.slot != kEmpty) return false;
    c.id = id;
    c.slot = slot;
    ++size_;
    return true;
  }

  void erase(uint64_t id) {
    if (cells_.empty()) return;
    size_t hole = place(id);
    if (cells_[hole].slot == kEmpty) return;
    --size_;
    // entries of the run behind the hole move up unless that would put
    // them before their own first cell
    const size_t mask = cells_.size() - 1;
    for (size_t i = (hole + 1) & mask; cells_[i].slot != kEmpty; i = (i + 1) & mask) {
      const size_t home = first(cells_[i].id);
      if (((i - home) & mask) >= ((i - hole) & mask)) {
        cells_[hole] = cells_[i];
        hole = i;
      }
    }
    cells_[hole].slot = kEmpty;
  }

 private:
  static constexpr uint64_t kEmpty = ~0ull;
  struct Cell {
    uint64_t id = 0;
    uint64_t slot = kEmpty;
  };

  // The id's first cell: the high bits of an odd multiple (2^64 over the
  // golden ratio), which spread runs of neighbouring ids.
  size_t first(uint64_t id) const {
    return static_cast<size_t>((id * 0x9e3779b97f4a7c15ull) >> shift_);
  }

  // The id's cell, or the empty one where it would go.
  size_t place(uint64_t id) const {
    const size_t mask = cells_.size() - 1;
    size_t i = first(id);
    while (cells_[i].slot != kEmpty && cells_[i].id != id) i = (i + 1) & mask;
    return i;
  }

  void rehash(size_t n) {
    std::vector<Cell> old(n);
    old.swap(cells_);
    shift_ = 64;
    for (size_t m = n; m > 1; m /= 2) --shift_;
    for (const Cell& c : old) {
      if (c.slot != kEmpty) cells_[place(c.id)] = c;
    }
  }

  std::vector<Cell> cells_;
  size_t size_ = 0;
  int shift_ = 64;
};

// A set of slots as a bit each, with the lowest member at hand.
class FreeSlots {
 public:
  void resize(uint64_t slots) { words_.assign((slots + 63) / 64, 0); }
  uint64_t size() const { return count_; }

  // False when the slot is a member already.
  bool insert(uint64_t slot) {
    uint64_t& w = words_[slot / 64];
    const uint64_t bit = 1ull << (slot % 64);
    if (w & bit) return false;
    w |= bit;
    ++count_;
    lowest_ = std::min<uint64_t>(lowest_, slot / 64);
    return true;
  }

  void erase(uint64_t slot) {
    uint64_t& w = words_[slot / 64];
    const uint64_t bit = 1ull << (slot % 64);
    if (!(w & bit)) return;
    w &= ~bit;
    --count_;
  }

  // Take the lowest member out; UINT64_MAX when there is none.
  uint64_t pop_lowest() {
    if (count_ == 0) return ~0ull;
    while (words_[lowest_] == 0) ++lowest_;
    const uint64_t slot = lowest_ * 64 + static_cast<uint64_t>(__builtin_ctzll(words_[lowest_]));
    erase(slot);
    return slot;
  }

 private:
  std::vector<uint64_t> words_;
  uint64_t count_ = 0;
  uint64_t lowest_ = 0;  // no member lies in an earlier word
};

}  // namespace grm
