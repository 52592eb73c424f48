// Checks of BlockPool over a counted memory of a fixed size; exits with the line that failed.
#include <cstdlib>
#include <map>
#include <thread>
#include <vector>

#include "block_pool.hpp"

#define CHECK(x)                   \
  do {                             \
    if (!(x)) std::_Exit(__LINE__ > 255 ? 255 : __LINE__); \
  } while (0)

struct Memory {
  static inline std::mutex mu;
  static inline std::map<void*, size_t> live;
  static inline size_t used = 0, size = 0;
  static inline char* next = reinterpret_cast<char*>(4096);
  static bool alloc(void** p, size_t bytes) {
    std::lock_guard<std::mutex> g(mu);
    if (used + bytes > size) return false;
    *p = next;
    next += bytes + 4096;
    live[*p] = bytes;
    used += bytes;
    return true;
  }
  static void release(void* p) noexcept {
    std::lock_guard<std::mutex> g(mu);
    auto it = live.find(p);
    if (it == live.end()) std::_Exit(254);
    used -= it->second;
    live.erase(it);
  }
};
using Pool = gj::BlockPool<Memory>;

int main() {
  constexpr size_t MiB = 1 << 20;
  Memory::size = 1024 * MiB;
  Pool pool;
  size_t cap = 0;
  // a kept block is handed out again for its size and device only
  void* a = pool.take(100 * MiB + 1, cap, 0);
  CHECK(a && cap == 104 * MiB);
  CHECK(pool.keep(a, cap, 0));
  CHECK(pool.take(104 * MiB, cap, 1) != a);
  CHECK(pool.take(101 * MiB, cap, 0) == a);
  CHECK(pool.keep(a, cap, 0));
  // what is kept goes back before memory from outside the pool is refused
  CHECK(Memory::used == 208 * MiB);
  void* big = pool.alloc(900 * MiB);
  CHECK(big && Memory::used == 1004 * MiB);
  CHECK(!pool.alloc(21 * MiB));
  Memory::release(big);
  // the exact size where the rounded one does not fit; such a block is not kept
  Memory::size = Memory::used + 100 * MiB + 4096;
  void* odd = pool.take(100 * MiB + 4096, cap, 0);
  CHECK(odd && cap == 100 * MiB + 4096);
  CHECK(!pool.keep(odd, cap, 0));
  Memory::release(odd);
  // bounds: total, blocks, largest; the oldest go first
  Memory::size = 8192 * MiB;
  const size_t before = Memory::used;
  std::vector<void*> v;
  for (int i = 0; i < 6; ++i) v.push_back(pool.take(128 * MiB, cap, 0));
  for (void* p : v) CHECK(pool.keep(p, cap, 0));
  CHECK(Memory::used == before + 512 * MiB && !Memory::live.count(v[0]) && Memory::live.count(v[5]));
  void* huge = pool.take(256 * MiB + 1, cap, 0);
  CHECK(cap == 256 * MiB + 1 && !pool.keep(huge, cap, 0));
  Memory::release(huge);
  v.clear();
  for (int i = 0; i < 80; ++i) v.push_back(pool.take(4096, cap, 0));
  for (void* p : v) CHECK(pool.keep(p, cap, 0));
  pool.trim(0, 0);
  CHECK(Memory::used == before);
  // threads that share it
  std::vector<std::thread> t;
  for (int k = 0; k < 8; ++k)
    t.emplace_back([&, k] {
      for (int i = 0; i < 3000; ++i) {
        size_t c = 0;
        void* p = pool.take(4096u << ((i + k) % 12), c, k % 2);
        if (!p) std::_Exit(253);
        if (!pool.keep(p, c, k % 2)) Memory::release(p);
        if (i % 500 == 0) pool.trim(0, 0);
      }
    });
  for (auto& x : t) x.join();
  pool.trim(0, 0);
  CHECK(Memory::used == before);
  return 0;
}
