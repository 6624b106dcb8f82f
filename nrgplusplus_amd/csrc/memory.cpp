// Device memory of chains, observables and recorders: growing buffers charged to the context's capacity,
// handed back to its pool once the streams that used them have drained.  Host code without kernels, so
// that tests/host_memory.cpp can run it against stand-ins for the HIP calls.
#include "common.hpp"

namespace nrgk {

// A quarter of headroom; from a pool, as much of it as its size at or below that leaves (9 to 25 %).
void DevBuf::ensure(size_t bytes) {
  if (bytes <= cap) return;
  release();
  const size_t want = bytes + bytes / 4 + 256, size = retired ? MemPool::size_below(want) : want;
  if (ctx) ctx->charge(size);
  if (ctx && retired) p = ctx->pool.take(size);
  if (!p) {
    if (ctx) ctx->make_room();
    hipError_t e = handled(hipMalloc(&p, size));
    if (e != hipSuccess && ctx) {  // everything idle is freed
      ctx->drain();
      ctx->pool.trim();
      e = handled(hipMalloc(&p, size));
    }
    if (e != hipSuccess) {
      if (ctx) ctx->refund(size);
      p = nullptr;
      throw Error(NRGK_ERR_NOMEM, std::string("hipMalloc(") + std::to_string(size) + "): " + hipGetErrorString(e));
    }
  }
  cap = size;
}
void DevBuf::release() {
  if (p) {
    if (retired) {
      retired->add(p, cap);
    } else {
      (void)hipFree(p);
      if (ctx) ctx->refund(cap);
    }
  }
  p = nullptr;
  cap = 0;
}

void Retired::attach(Ctx* c, hipStream_t s) {
  ctx = c;
  st = s;
  std::lock_guard<std::mutex> lk(c->lists_m);
  c->lists.push_back(this);
}
Retired::~Retired() {
  if (!ctx) return;
  {
    std::lock_guard<std::mutex> lk(ctx->lists_m);
    ctx->lists.erase(std::find(ctx->lists.begin(), ctx->lists.end(), this));
  }
  if (!bufs.empty() && st) (void)hipStreamSynchronize(st);
  give_all();
}
void Retired::give_all() {
  List b;
  take(b);
  for (auto& [p, size] : b) {
    ctx->pool.give(p, size);
    ctx->refund(size);
  }
}
void Ctx::drain() {
  Retired::List b;
  {
    std::lock_guard<std::mutex> lk(lists_m);
    for (Retired* r : lists) r->take(b);
  }
  if (b.empty()) return;
  const bool idle = hipDeviceSynchronize() == hipSuccess;
  for (auto& [p, size] : b) {
    if (idle) pool.give(p, size);
    else (void)hipFree(p);
    refund(size);
  }
}

}  // namespace nrgk
