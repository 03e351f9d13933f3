"""The banks' host tables against the standard containers, over random
updates with ids that collide and runs that wrap around the table's end."""

import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "graftrepository_amd" / "csrc"

PROGRAM = r"""
#include "slot_tables.hpp"
#include <cassert>
#include <map>
#include <random>
#include <set>
#undef NDEBUG
#include <assert.h>
int main() {
  std::mt19937_64 rng(7);
  for (int round = 0; round < 40; ++round) {
    grm::IdTable t;
    std::map<uint64_t, uint64_t> want;
    grm::FreeSlots f;
    std::set<uint64_t> free_want;
    f.resize(300);
    // few distinct ids; in half of the rounds all with one first cell or the last
    const uint64_t inverse = 0xf1de83e19937733dull;  // of the table's multiplier
    assert(inverse * 0x9e3779b97f4a7c15ull == 1);
    auto id = [&]() -> uint64_t {
      const uint64_t x = rng() % 200;
      if (round % 2) return x == 0 ? ~0ull : x;
      return ((x % 3 == 0 ? 0xffffffull << 40 : 0) + x) * inverse;
    };
    for (int i = 0; i < 5000; ++i) {
      const uint64_t x = id(), s = rng() % 300;
      switch (rng() % 5) {
        case 0: case 1: assert(t.emplace(x, i) == want.emplace(x, i).second); break;
        case 2: t.erase(x); want.erase(x); break;
        case 3: assert(f.insert(s) == free_want.insert(s).second); break;
        default:
          if (rng() % 2) { f.erase(s); free_want.erase(s); }
          else {
            const uint64_t low = f.pop_lowest();
            assert(low == (free_want.empty() ? ~0ull : *free_want.begin()));
            free_want.erase(low);
          }
      }
      assert(t.size() == want.size() && f.size() == free_want.size());
      const uint64_t y = id();
      const uint64_t* got = t.find(y);
      const auto it = want.find(y);
      assert((got != nullptr) == (it != want.end()) && (!got || *got == it->second));
    }
    for (const auto& kv : want) assert(t.find(kv.first) && *t.find(kv.first) == kv.second);
  }
  return 0;
}
"""


def test_tables_against_standard_containers(tmp_path):
    src, exe = tmp_path / "tables.cpp", tmp_path / "tables"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{CSRC}", str(src), "-o", str(exe)],
                   check=True)
    subprocess.run([str(exe)], check=True, timeout=120)
