// Context, device memory, event timing and host<->device helpers.
#include "jues_internal.h"

#include <atomic>

namespace jues {

static std::atomic<size_t> g_bytes{0};
size_t device_bytes_in_use() { return g_bytes.load(); }

static thread_local bool tl_no_alloc = false;
NoAllocScope::NoAllocScope() : prev(tl_no_alloc) { tl_no_alloc = true; }
NoAllocScope::~NoAllocScope() { tl_no_alloc = prev; }
bool no_alloc_active() { return tl_no_alloc; }

// ---- kept blocks ----------------------------------------------------------------------
namespace {
constexpr size_t kMaxBlocks = 256;

void device_free(void* p, size_t bytes) {
  (void)hipFree(p);
  g_bytes -= bytes;
}

// every open pool of the process
std::mutex g_pools_mu;
std::list<BlockPool*>& all_pools() {
  static std::list<BlockPool*> l;
  return l;
}
thread_local std::shared_ptr<BlockPool> tl_pool;
}  // namespace

BlockPool::BlockPool(int device) : device_(device) {
  size_t free_b = 0, total_b = 0;
  if (hipMemGetInfo(&free_b, &total_b) == hipSuccess) limit_ = total_b / 16;
  std::lock_guard<std::mutex> l(g_pools_mu);
  all_pools().push_back(this);
}

BlockPool::~BlockPool() {
  {
    std::lock_guard<std::mutex> l(g_pools_mu);
    all_pools().remove(this);
  }
  trim();
}

// The smallest kept block that holds `bytes` with at most an eighth (and 256 bytes) to spare, so that a
// pool serves the same sizes again without tying up large blocks under small buffers.
void* BlockPool::take(size_t bytes, size_t& capacity) {
  std::lock_guard<std::mutex> l(mu_);
  auto best = blocks_.end();
  for (auto it = blocks_.begin(); it != blocks_.end(); ++it)
    if (it->capacity >= bytes && it->capacity <= bytes + bytes / 8 + 256 &&
        (best == blocks_.end() || it->capacity < best->capacity))
      best = it;
  if (best == blocks_.end()) return nullptr;
  void* p = best->p;
  capacity = best->capacity;
  kept_ -= capacity;
  blocks_.erase(best);
  return p;
}

void BlockPool::give(void* p, size_t capacity) {
  std::list<Block> out;  // freed outside the lock (hipFree waits for the device)
  {
    std::lock_guard<std::mutex> l(mu_);
    bool keep = open_ && capacity <= limit_;
    if (keep) {
      try {
        blocks_.push_back({p, capacity});
      } catch (...) {  // no host memory for the list node: called from destructors, so nothing may leave
        keep = false;
      }
    }
    if (keep) {
      p = nullptr;
      kept_ += capacity;
      while (kept_ > limit_ || blocks_.size() > kMaxBlocks) {
        kept_ -= blocks_.front().capacity;
        out.splice(out.end(), blocks_, blocks_.begin());
      }
    }
  }
  if (p) device_free(p, capacity);
  for (const Block& b : out) device_free(b.p, b.capacity);
}

void BlockPool::trim() {
  std::list<Block> out;
  {
    std::lock_guard<std::mutex> l(mu_);
    out.swap(blocks_);
    kept_ = 0;
  }
  for (const Block& b : out) device_free(b.p, b.capacity);
}

void BlockPool::close() {
  {
    std::lock_guard<std::mutex> l(mu_);
    open_ = false;
  }
  trim();
}

size_t BlockPool::kept() {
  std::lock_guard<std::mutex> l(mu_);
  return kept_;
}

PoolScope::PoolScope(const std::shared_ptr<BlockPool>& pool) : prev(std::move(tl_pool)) { tl_pool = pool; }
PoolScope::~PoolScope() { tl_pool = std::move(prev); }

void DevBuf::alloc(size_t nbytes) {
  release();
  if (nbytes == 0) return;
  if (tl_no_alloc) throw Error(JUES_BAD_ARG, "device allocation inside an allocation-free entry point");
  void* q = tl_pool ? tl_pool->take(nbytes, capacity) : nullptr;
  if (!q) {
    hipError_t e = hipMalloc(&q, nbytes);
    if (e == hipErrorOutOfMemory) {
      (void)hipGetLastError();
      {
        std::lock_guard<std::mutex> l(g_pools_mu);
        for (BlockPool* b : all_pools()) b->trim();
      }
      e = hipMalloc(&q, nbytes);
    }
    if (e != hipSuccess) {
      (void)hipGetLastError();
      throw Error(e == hipErrorOutOfMemory ? JUES_OOM : JUES_HIP_ERROR,
                  "hipMalloc(" + std::to_string(nbytes) + " bytes): " + hipGetErrorString(e));
    }
    capacity = nbytes;
    g_bytes += nbytes;
  }
  p = q;
  bytes = nbytes;
  pool = tl_pool;
}

void DevBuf::release() {
  if (p) {
    if (pool) pool->give(p, capacity);
    else device_free(p, capacity);
  }
  p = nullptr;
  bytes = capacity = 0;
  pool.reset();
}

void device_memory(jues_ctx* ctx, size_t* free_bytes, size_t* total_bytes) {
  JUES_HIP(hipMemGetInfo(free_bytes, total_bytes));
  std::lock_guard<std::mutex> l(g_pools_mu);
  for (BlockPool* b : all_pools())
    if (b->device() == ctx->device) *free_bytes += b->kept();
}

void* scratch(jues_ctx* ctx, int slot, size_t bytes) {
  if (tl_no_alloc) throw Error(JUES_BAD_ARG, "context scratch inside an allocation-free entry point");
  DevBuf& b = ctx->scratch[slot];
  if (b.bytes < bytes) {
    if (b.p) JUES_HIP(hipStreamSynchronize(ctx->stream));
    b.alloc(bytes + bytes / 8 + 256);
  }
  return b.p;
}

void release_scratch(jues_ctx* ctx) {
  for (DevBuf& b : ctx->scratch) b.release();
}

void h2d(jues_ctx* ctx, void* dst, const void* src, size_t bytes) {
  if (bytes == 0) return;
  JUES_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->stream));
  JUES_HIP(hipStreamSynchronize(ctx->stream));
}

void d2h(jues_ctx* ctx, void* dst, const void* src, size_t bytes) {
  if (bytes == 0) return;
  JUES_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
  JUES_HIP(hipStreamSynchronize(ctx->stream));
}

void sync(jues_ctx* ctx) { JUES_HIP(hipStreamSynchronize(ctx->stream)); }

KTimer::KTimer(jues_ctx* c, const char* name, double flops, double bytes) : ctx(c), on(c->timing) {
  if (!on) return;
  hipEvent_t a, b;
  if (ctx->event_pool.size() >= 2) {
    a = ctx->event_pool.back(); ctx->event_pool.pop_back();
    b = ctx->event_pool.back(); ctx->event_pool.pop_back();
  } else {
    JUES_HIP(hipEventCreate(&a));
    JUES_HIP(hipEventCreate(&b));
  }
  JUES_HIP(hipEventRecord(a, ctx->stream));
  slot = ctx->pending.size();
  ctx->pending.push_back({name, a, b, flops, bytes});
}

KTimer::~KTimer() {
  if (!on) return;
  (void)hipEventRecord(ctx->pending[slot].b, ctx->stream);
  if (ctx->pending.size() > 4096) {
    try { flush_timers(ctx); } catch (...) {}
  }
}

void flush_timers(jues_ctx* ctx) {
  if (ctx->pending.empty()) return;
  JUES_HIP(hipStreamSynchronize(ctx->stream));
  for (auto& p : ctx->pending) {
    float ms = 0.f;
    JUES_HIP(hipEventElapsedTime(&ms, p.a, p.b));
    KStat& s = ctx->kstats[p.name];
    s.ms += ms;
    s.calls += 1;
    s.flops += p.flops;
    s.bytes += p.bytes;
    ctx->event_pool.push_back(p.a);
    ctx->event_pool.push_back(p.b);
  }
  ctx->pending.clear();
}

}  // namespace jues

jues_ctx::jues_ctx() {}
jues_ctx::~jues_ctx() {}
