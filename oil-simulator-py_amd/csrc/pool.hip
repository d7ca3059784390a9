// Device memory of hierarchy builds: slab sub-allocation and deferred release
// (SetupPool, PoolScope; declared in common.h) over a bounded cache of idle blocks.
// Host code only.
#include <map>
#include <mutex>
#include <vector>

#include "common.h"

namespace impes {

namespace {

// Idle device blocks kept for the next build on the same device (a build of a
// 500,000-cell hierarchy took 5 ms in 120 hipMalloc calls and its destruction 26 ms
// in as many hipFree calls). At most kBlockCacheBytes per device; more is freed at
// once. An allocation of the library that runs out of memory gives the whole cache back
// and tries again (device_malloc), and trim() does so on request. Blocks enter only once the device has finished with
// them (the callers below), so any stream may take them.
constexpr size_t kBlockCacheBytes = size_t(4) << 30;
struct BlockCache {
  std::mutex m;
  std::map<int, std::multimap<size_t, void*>> idle;  // by device, then size
  std::map<int, size_t> bytes;

  void* take(int dev, size_t want, size_t* got) {
    {
      std::lock_guard<std::mutex> g(m);
      auto& blocks = idle[dev];
      auto it = blocks.lower_bound(want);
      if (it != blocks.end() && it->first <= want + want / 2) {
        void* p = it->second;
        *got = it->first;
        bytes[dev] -= it->first;
        blocks.erase(it);
        return p;
      }
    }
    *got = want;
    return device_malloc(want);
  }
  void give(int dev, void* p, size_t size) {
    {
      std::lock_guard<std::mutex> g(m);
      if (bytes[dev] + size <= kBlockCacheBytes) {
        idle[dev].emplace(size, p);
        bytes[dev] += size;
        return;
      }
    }
    (void)hipFree(p);
  }
  void trim() {
    std::vector<void*> all;
    {
      std::lock_guard<std::mutex> g(m);
      for (auto& d : idle)
        for (auto& b : d.second) all.push_back(b.second);
      idle.clear();
      bytes.clear();
    }
    for (void* p : all) (void)hipFree(p);
  }
};
// never destroyed: its blocks go with the process, after the HIP runtime may be gone
BlockCache& block_cache() {
  static BlockCache* c = new BlockCache();
  return *c;
}

// Waits for a device; false when that fails (its blocks are then freed, not kept). By
// hipFree, which waits for all of the device's work: hipDeviceSynchronize would end every
// capture in progress, those of other threads included.
bool device_idle(int dev) {
  int cur = 0;
  if (hipGetDevice(&cur) != hipSuccess) return false;
  if (cur != dev && hipSetDevice(dev) != hipSuccess) return false;
  void* p = nullptr;
  const bool ok = hipMalloc(&p, 256) == hipSuccess && hipFree(p) == hipSuccess;
  if (!ok) (void)hipGetLastError();
  if (cur != dev) (void)hipSetDevice(cur);
  return ok;
}

}  // namespace

void release_cached_memory() { block_cache().trim(); }

void* device_malloc(size_t bytes) {
  void* p = nullptr;
  hipError_t rc = hipMalloc(&p, bytes);
  if (rc == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    release_cached_memory();
    rc = hipMalloc(&p, bytes);
  }
  IMPES_HIP_CHECK(rc);
  return p;
}

struct SetupPool::Impl {
  struct Slab {
    size_t size = 0, used = 0;
    long live = 0;
  };
  std::mutex m;
  std::map<char*, Slab> slabs;  // by base address
  char* cur = nullptr;          // slab that new small blocks are carved from
  std::map<void*, size_t> large;        // live large blocks and their sizes
  std::multimap<size_t, void*> spare;   // large blocks released under the scope
  int open = 0;
  int dev = 0;        // the device of the pool's blocks (the current one when a scope opens)
  bool idle = false;  // the device has finished with every block of the pool
  bool mixed = false; // blocks of several devices: none is cached

  void drop(void* p, size_t size) {
    if (idle && !mixed) block_cache().give(dev, p, size);
    else (void)hipFree(p);
  }

  std::map<char*, Slab>::iterator slab_of(void* p) {
    auto it = slabs.upper_bound(static_cast<char*>(p));
    if (it == slabs.begin()) return slabs.end();
    --it;
    if (static_cast<char*>(p) >= it->first + it->second.size) return slabs.end();
    return it;
  }
  void free_slab(std::map<char*, Slab>::iterator it) {
    if (it->first == cur) cur = nullptr;
    drop(it->first, it->second.size);
    slabs.erase(it);
  }
};

SetupPool::SetupPool() = default;

SetupPool::Impl* SetupPool::impl() {
  if (!impl_) impl_.reset(new Impl());
  return impl_.get();
}

SetupPool::~SetupPool() {
  if (!impl_) return;
  for (auto& b : impl_->spare) impl_->drop(b.second, b.first);
  for (auto& b : impl_->large) impl_->drop(b.first, b.second);
  for (auto& s : impl_->slabs) impl_->drop(s.first, s.second.size);
}

void SetupPool::retire() {
  if (!impl_) return;
  std::lock_guard<std::mutex> g(impl_->m);
  impl_->idle = device_idle(impl_->dev);
}

void* SetupPool::alloc(size_t bytes) {
  Impl* I = impl();
  std::lock_guard<std::mutex> g(I->m);
  IMPES_REQUIRE(I->open > 0, "setup pool: allocation outside a scope");
  if (bytes > kPoolSmall) {
    auto it = I->spare.lower_bound(bytes);
    if (it != I->spare.end() && it->first <= 2 * bytes) {
      void* p = it->second;
      I->large[p] = it->first;
      I->spare.erase(it);
      return p;
    }
    size_t got = 0;
    void* p = block_cache().take(I->dev, bytes, &got);
    I->large[p] = got;
    return p;
  }
  const size_t r = (bytes + 255) & ~size_t(255);
  if (!I->cur || I->slabs[I->cur].used + r > I->slabs[I->cur].size) {
    size_t got = 0;
    char* base = static_cast<char*>(block_cache().take(I->dev, kSlab, &got));
    I->slabs[base] = Impl::Slab{got, 0, 0};
    I->cur = base;
  }
  Impl::Slab& s = I->slabs[I->cur];
  char* p = I->cur + s.used;
  s.used += r;
  ++s.live;
  return p;
}

void SetupPool::release(void* p) {
  Impl* I = impl();
  std::lock_guard<std::mutex> g(I->m);
  auto lit = I->large.find(p);
  if (lit != I->large.end()) {
    if (I->open > 0) I->spare.emplace(lit->second, p);
    else I->drop(p, lit->second);
    I->large.erase(lit);
    return;
  }
  auto it = I->slab_of(p);
  if (it == I->slabs.end()) return;  // not a block of this pool
  --it->second.live;
  if (I->open == 0 && it->second.live == 0) I->free_slab(it);
}

void SetupPool::open() {
  Impl* I = impl();
  std::lock_guard<std::mutex> g(I->m);
  I->idle = false;  // new work will use the pool's blocks
  if (I->open == 0) {
    int dev = 0;
    IMPES_HIP_CHECK(hipGetDevice(&dev));
    if (dev != I->dev && !(I->large.empty() && I->spare.empty() && I->slabs.empty())) I->mixed = true;
    I->dev = dev;
  }
  ++I->open;
}

void SetupPool::close() {
  Impl* I = impl();
  std::lock_guard<std::mutex> g(I->m);
  if (--I->open > 0) return;
  // the blocks released under the scope: kept once the device has finished with them
  // (as hipFree would wait; the scope's own work has been waited for already, unless
  // an error ends it)
  I->idle = device_idle(I->dev);
  for (auto& b : I->spare) I->drop(b.second, b.first);
  I->spare.clear();
  for (auto it = I->slabs.begin(); it != I->slabs.end();) {
    auto next = std::next(it);
    if (it->second.live == 0) I->free_slab(it);
    it = next;
  }
  I->cur = nullptr;  // slab space is not reused across scopes either
  I->idle = false;   // the live blocks are about to be used
}

size_t SetupPool::slab_bytes() const {
  if (!impl_) return 0;
  std::lock_guard<std::mutex> g(impl_->m);
  size_t b = 0;
  for (auto& s : impl_->slabs) b += s.second.size;
  return b;
}

namespace {
thread_local std::shared_ptr<SetupPool> t_pool;
}

std::shared_ptr<SetupPool> current_setup_pool() { return t_pool; }

PoolScope::PoolScope(std::shared_ptr<SetupPool> pool) : pool_(std::move(pool)), prev_(t_pool) {
  pool_->open();
  t_pool = pool_;
}

PoolScope::~PoolScope() {
  t_pool = prev_;
  pool_->close();
}

}  // namespace impes
