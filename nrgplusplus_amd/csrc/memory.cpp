// Device memory of chains, observables and recorders: growing buffers charged to the context's capacity,
// handed back to its pool once the streams that used them have drained.  Host code without kernels, so
// that tests/host_memory.cpp can run it against stand-ins for the HIP calls.
#include "common.hpp"

namespace nrgk {

void DevBuf::ensure(size_t bytes) {
  if (bytes <= cap) return;
  release();
  const size_t want = bytes + bytes / 4 + 256;
  size = retired ? MemPool::size_class(want) : want;
  if (ctx) ctx->charge(want);
  if (ctx && retired) p = ctx->pool.take(size);
  if (!p) {
    if (ctx && ctx->capacity && ctx->used + ctx->pool.held() > ctx->capacity) ctx->pool.trim();
    hipError_t e = handled(hipMalloc(&p, size));
    if (e != hipSuccess && ctx) {
      // the device waits, as hipFree made it, and everything idle is freed
      if (retired && hipDeviceSynchronize() == hipSuccess) retired->give_all();
      ctx->pool.trim();
      size = want;
      e = handled(hipMalloc(&p, size));
    }
    if (e != hipSuccess) {
      if (ctx) ctx->refund(want);
      p = nullptr;
      throw Error(NRGK_ERR_NOMEM, std::string("hipMalloc(") + std::to_string(want) + "): " + hipGetErrorString(e));
    }
  }
  cap = want;
}
void DevBuf::release() {
  if (p) {
    if (retired) retired->add(p, size);
    else (void)hipFree(p);
    if (ctx) ctx->refund(cap);
  }
  p = nullptr;
  cap = 0;
}
void Retired::give_all() {
  std::vector<std::pair<void*, size_t>> b;
  {
    std::lock_guard<std::mutex> lk(m);
    b.swap(bufs);
  }
  for (auto& [p, size] : b) {
    if (ctx) ctx->pool.give(p, size);
    else (void)hipFree(p);
  }
}

}  // namespace nrgk
