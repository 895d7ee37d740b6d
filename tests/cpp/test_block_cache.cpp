// The block cache's rules (raptr_amd/csrc/blockcache.hpp) over a model of the
// driver: what is handed out is always the driver's, large enough, of the right
// device, cleared and handed out once.
#include <cstdint>
#include <cstdio>
#include <map>
#include <mutex>
#include <new>
#include <set>
#include <thread>
#include <vector>

#include "blockcache.hpp"

static int failures = 0;
#define CHECK(c)                                                      \
  do {                                                                \
    if (!(c)) {                                                       \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c);             \
      ++failures;                                                     \
    }                                                                 \
  } while (0)

struct Model {
  enum Error { kOk, kNoMemory, kInvalid, kNoWait };
  struct Mem {
    size_t bytes;
    int dev;
    bool cleared;
  };
  std::map<uintptr_t, Mem> mem;
  uintptr_t next = 0x1000;
  size_t used = 0, room = size_t(64) << 30;
  int dev = 0, allocs = 0, releases = 0, waits = 0, clears = 0;
  bool can_wait = true, can_release = true, throws = false;
  Error device(int* d) {
    *d = dev;
    return kOk;
  }
  Error place(uintptr_t at, size_t bytes) {
    mem[at] = Mem{bytes, dev, true};
    used += bytes;
    return kOk;
  }
  Error alloc(void** p, size_t bytes) {
    if (throws) throw std::bad_alloc();
    if (used + bytes > room) return kNoMemory;
    ++allocs;
    *p = reinterpret_cast<void*>(next);
    place(next, bytes);
    next += (bytes + 0xfff) / 0x1000 * 0x1000;
    return kOk;
  }
  Error release(void* p) {
    auto it = mem.find(uintptr_t(p));
    if (it == mem.end() || !can_release) return kInvalid;
    ++releases;
    used -= it->second.bytes;
    mem.erase(it);
    return kOk;
  }
  size_t extent(void* p) {
    auto it = mem.find(uintptr_t(p));
    return it == mem.end() ? 0 : it->second.bytes;
  }
  Error wait() {
    ++waits;
    return can_wait ? kOk : kNoWait;
  }
  Error clear(void* p, size_t bytes, int) {
    if (throws) throw std::bad_alloc();
    auto it = mem.find(uintptr_t(p));
    CHECK(it != mem.end() && bytes <= it->second.bytes);  // inside the driver's block
    if (it != mem.end()) it->second.cleared = true;
    ++clears;
    return kOk;
  }
  Error wait_clear(int) { return kOk; }
  void forget_error() {}
};
using Cache = raptr::BlockCache<Model>;
constexpr size_t MB = size_t(1) << 20;

static void* get(Cache& c, size_t bytes) {
  void* p = nullptr;
  CHECK(c.malloc(&p, bytes) == Model::kOk);
  auto it = c.driver().mem.find(uintptr_t(p));
  CHECK(it != c.driver().mem.end() && it->second.bytes >= bytes &&
        it->second.dev == c.driver().dev && it->second.cleared);
  if (it != c.driver().mem.end()) it->second.cleared = false;  // the owner writes it
  return p;
}

static void test_reuse() {
  Cache c;
  void* a = get(c, 9 * MB);
  CHECK(c.free(a, false) == Model::kOk && c.driver().waits == 1 && c.driver().clears == 1);
  CHECK(c.kept_bytes() == Cache::rounded(9 * MB));
  CHECK(get(c, 9 * MB - 5) == a && c.kept_bytes() == 0);
  CHECK(c.free(a, true) == Model::kOk && c.driver().waits == 1);
  void* b = get(c, 5 * MB);  // less than four fifths of it: a block of its own
  CHECK(b != a);
  c.driver().dev = 1;  // the other device's
  CHECK(get(c, 9 * MB) != a);
  c.driver().dev = 0;
  CHECK(get(c, 9 * MB) == a);
  CHECK(c.free(nullptr, false) == Model::kOk);
}

static void test_freed_twice() {
  Cache c;
  void* a = get(c, 9 * MB);
  CHECK(c.free(a, false) == Model::kOk);
  CHECK(c.free(a, false) == Model::kInvalid);
  void* b = get(c, 9 * MB);
  CHECK(get(c, 9 * MB) != b);  // once only
  CHECK(c.free(b, false) == Model::kOk && c.free(b, true) == Model::kInvalid);
  int foreign = 0;
  CHECK(c.free(&foreign, false) == Model::kInvalid);
}

// A block released with the driver's own call: whatever comes to its address
// later is not the cache's.
static void test_released_elsewhere() {
  Cache c;
  void* a = get(c, 9 * MB);
  CHECK(c.driver().release(a) == Model::kOk);
  c.driver().place(uintptr_t(a), 4096);
  CHECK(c.free(a, false) == Model::kOk && c.driver().extent(a) == 0);  // the driver's free
  CHECK(c.driver().clears == 0 && c.kept_bytes() == 0);
  void* b = get(c, 9 * MB);
  CHECK(c.free(b, false) == Model::kOk && c.driver().release(b) == Model::kOk);
  CHECK(get(c, 9 * MB) != b && c.kept_bytes() == 0);  // a kept block that is gone
  void* d = get(c, 9 * MB);
  CHECK(c.free(d, false) == Model::kOk && c.driver().release(d) == Model::kOk);
  c.driver().place(uintptr_t(d), 4096);
  CHECK(c.free(d, false) == Model::kOk && c.driver().extent(d) == 0 && c.kept_bytes() == 0);
}

// The bound, the oldest first, and everything given back to find memory.
static void test_bounds() {
  Cache c;
  std::vector<void*> p;
  const size_t one = 512 * MB;
  for (int k = 0; k < 12; ++k) p.push_back(get(c, one));
  for (void* q : p) CHECK(c.free(q, false) == Model::kOk);
  CHECK(c.kept_bytes() == Cache::kBytes && c.driver().releases == 4);
  for (int k = 0; k < 4; ++k) CHECK(c.driver().extent(p[k]) == 0);
  CHECK(c.driver().extent(p[4]) >= one);
  c.driver().room = c.driver().used;  // no memory but the kept blocks'
  void* big = get(c, 700 * MB);
  CHECK(big && c.kept_bytes() == 0);
  c.driver().room = c.driver().used;
  c.driver().room += 9 * MB - 17;  // room for the block but not for its rounding
  void* tight = get(c, 9 * MB - 17);
  CHECK(c.free(tight, false) == Model::kOk && c.kept_bytes() == 9 * MB - 17);
  CHECK(c.give_back(0, 0) == 9 * MB - 17 && c.kept_bytes() == 0);
  c.driver().room = c.driver().used;
  void* none = &c;
  CHECK(c.malloc(&none, 700 * MB) == Model::kNoMemory && !none);
  CHECK(c.malloc(&none, Cache::kBlock + 1) == Model::kNoMemory && !none);
  // smaller and larger blocks are the driver's alone
  Cache d;
  for (size_t bytes : {size_t(1), Cache::kLeast - 1, Cache::kBlock + 1}) {
    void* l = get(d, bytes);
    CHECK(d.driver().used == bytes);
    CHECK(d.free(l, false) == Model::kOk && d.kept_bytes() == 0 && d.driver().used == 0);
    CHECK(d.free(l, false) == Model::kInvalid);
  }
  CHECK(d.driver().waits == 0 && d.driver().clears == 0);
  for (size_t bytes : {Cache::kLeast, Cache::kLeast + 1, Cache::kBlock - 1, Cache::kBlock})
    CHECK(d.free(get(d, bytes), false) == Model::kOk && d.kept_bytes() >= bytes);
  c.driver().room = c.driver().used;  // a small one finds the kept blocks' memory too
  CHECK(c.free(big, false) == Model::kOk && c.kept_bytes() > 0);
  CHECK(get(c, 4096) && c.kept_bytes() == 0);
}

// A device that cannot be waited for and one that is not current: the driver's
// free, nothing kept.
static void test_no_wait() {
  Cache c;
  void* a = get(c, 9 * MB);
  c.driver().can_wait = false;
  CHECK(c.free(a, false) == Model::kOk && c.kept_bytes() == 0 && c.driver().used == 0);
  void* b = get(c, 9 * MB);
  c.driver().can_wait = true;
  c.driver().dev = 1;
  CHECK(c.free(b, false) == Model::kOk && c.kept_bytes() == 0 && c.driver().used == 0);
}

// Everything given back on request, of one device; what the driver refuses to
// release stays.
static void test_give_back() {
  Cache c;
  void* a = get(c, 9 * MB);
  void* b = get(c, 30 * MB);
  c.driver().dev = 1;
  void* other = get(c, 9 * MB);
  CHECK(c.free(other, false) == Model::kOk);
  c.driver().dev = 0;
  CHECK(c.free(a, false) == Model::kOk && c.free(b, false) == Model::kOk);
  c.driver().can_release = false;
  CHECK(c.give_back(0, 0) == 0 && c.kept_bytes() >= 39 * MB);
  c.driver().can_release = true;
  CHECK(c.give_back(0, 0) >= 39 * MB && c.kept_bytes() == 0 && c.give_back(0, 0) == 0);
  CHECK(c.free(a, false) == Model::kInvalid);
  CHECK(c.driver().extent(other) && c.driver().mem.size() == 1);
}

// An exception below (no host memory) is an error of the call, and the lock is
// free again.
static void test_exceptions() {
  Cache c;
  void* a = get(c, 9 * MB);
  c.driver().throws = true;
  void* b = &c;
  CHECK(c.malloc(&b, 30 * MB) == Model::kNoMemory && !b);
  CHECK(c.malloc(&b, 100) == Model::kNoMemory && !b);
  CHECK(c.free(a, false) == Model::kNoMemory);
  c.driver().throws = false;
  CHECK(c.free(get(c, 30 * MB), false) == Model::kOk && c.kept_bytes() >= 30 * MB);
}

// Four threads allocate, write and free blocks of a few sizes.
static void test_threads() {
  struct Locked : Model {
    std::mutex mu;
    Error alloc(void** p, size_t n) { std::lock_guard<std::mutex> l(mu); return Model::alloc(p, n); }
    Error release(void* p) { std::lock_guard<std::mutex> l(mu); return Model::release(p); }
    size_t extent(void* p) { std::lock_guard<std::mutex> l(mu); return Model::extent(p); }
    Error wait() { std::lock_guard<std::mutex> l(mu); return Model::wait(); }
    Error clear(void* p, size_t n, int d) { std::lock_guard<std::mutex> l(mu); return Model::clear(p, n, d); }
  };
  raptr::BlockCache<Locked> c;
  c.driver().room = size_t(3) << 30;
  std::mutex mu;
  std::set<void*> out;
  std::vector<std::thread> threads;
  for (int t = 0; t < 4; ++t)
    threads.emplace_back([&, t] {
      for (int k = 0; k < 3000; ++k) {
        void* p = nullptr;
        const size_t n = (3 + (t * 7 + k * 13) % 11 * 40) * MB;
        if (c.malloc(&p, n) != Model::kOk) continue;
        {
          std::lock_guard<std::mutex> l(mu);
          CHECK(out.insert(p).second);  // nobody else's
        }
        std::this_thread::yield();
        {
          std::lock_guard<std::mutex> l(mu);
          out.erase(p);
        }
        CHECK(c.free(p, k % 2) == Model::kOk);
        if (k % 500 == 0) (void)c.give_back(0, 0);
      }
    });
  for (auto& t : threads) t.join();
  (void)c.give_back(0, 0);
  CHECK(c.driver().used == 0 && c.kept_bytes() == 0);
}

int main() {
  test_reuse();
  test_freed_twice();
  test_released_elsewhere();
  test_bounds();
  test_no_wait();
  test_give_back();
  test_exceptions();
  test_threads();
  std::printf("%d failure(s)\n", failures);
  return failures != 0;
}
