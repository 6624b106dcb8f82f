// Host-side checks of the library's memory layer (csrc/common.hpp, csrc/memory.cpp), compiled with the host
// compiler and stand-ins for the HIP calls it makes: "device" memory is malloc'ed, so nothing here needs a GPU.
// Usage: host_memory <check>; prints one line and exits with 0 if the check holds.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <random>
#include <string>
#include <thread>
#include <vector>

#include "../nrgplusplus_amd/csrc/memory.cpp"

static int failures = 0;
#define CHECK(c)                                                \
  do {                                                          \
    if (!(c)) {                                                 \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c);       \
      failures++;                                               \
    }                                                           \
  } while (0)

extern "C" {
// (freed memory is overwritten and kept, so that a later read of it shows)
static std::map<void*, size_t> live;
static size_t live_bytes = 0, live_peak = 0;  // of device memory
static std::mutex hip_m;
static int fail_next = 0;  // allocations to refuse
static hipError_t last_error = hipSuccess;
hipError_t hipMalloc(void** p, size_t n) {
  if (fail_next > 0) {
    fail_next--;
    return last_error = hipErrorOutOfMemory;
  }
  std::lock_guard<std::mutex> lk(hip_m);
  live[*p = std::malloc(n)] = n;
  live_bytes += n;
  live_peak = std::max(live_peak, live_bytes);
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = last_error;
  last_error = hipSuccess;
  return e;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> lk(hip_m);
  CHECK(!p || live.count(p));
  if (!p) return hipSuccess;
  std::memset(p, 0xA5, live[p]);
  live_bytes -= live[p];
  live.erase(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = std::malloc(n);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "stand-in"; }
}

using namespace nrgk;

// What get() read back stays readable after reset() until the staging's owner takes new regions, and a chunk
// that a launch made after reset() may still read goes to nobody else before the owner's next synchronisation,
// also where the interval needed several chunks and another owner's staging takes some at once.
static void staging_readback() {
  Ctx ctx;
  ctx.set_capacity(size_t(1) << 30);
  Staging a, b;
  a.ctx = b.ctx = &ctx;
  std::vector<double> dev(1000), big(200000, 1.0);
  for (size_t i = 0; i < dev.size(); i++) dev[i] = (double)i;
  for (int round = 0; round < 3; round++) {
    double* first = a.put(big, nullptr);
    a.put(big, nullptr);  // a second chunk, and a third
    a.put(big, nullptr);
    const double* r = a.get(dev.data(), dev.size(), nullptr);
    if (round == 0) CHECK(a.chunks.size() > 1);
    a.reset();
    std::vector<double> other(200000, -1.0);
    for (int k = 0; k < 3; k++) b.put(other, nullptr);  // (chunks of the same sizes)
    b.get(other.data(), dev.size(), nullptr);
    CHECK(std::memcmp(r, dev.data(), dev.size() * sizeof(double)) == 0);
    CHECK(first[0] == 1.0 && first[199999] == 1.0);
    b.reset();
  }
  // the regions are filled again from the front: an owner's memory settles
  const size_t used = ctx.used;
  for (int round = 0; round < 5; round++) {
    for (int k = 0; k < 3; k++) a.put(big, nullptr);
    a.reset();
  }
  CHECK(ctx.used == used);
  b.release();
  a.release();
  CHECK(ctx.used == 0);
}

// An allocation that fails, is retried after idle memory was freed and succeeds leaves no error behind (the next
// launch's check would report it), nor does one that fails for good with NRGK_ERR_NOMEM; the account stands.
static void failed_allocation() {
  Ctx ctx;
  ctx.set_capacity(size_t(1) << 30);
  Retired ret;
  ret.attach(&ctx, nullptr);
  {
    DevBuf old(&ctx, &ret);
    old.ensure(1 << 20);
  }
  ret.give_all();
  CHECK(ctx.pool.held() > 0);
  DevBuf b(&ctx, &ret);
  fail_next = 1;
  b.ensure(3 << 20);
  CHECK(b.p && last_error == hipSuccess);
  CHECK(ctx.pool.held() == 0);
  Staging st;
  st.ctx = &ctx;
  fail_next = 1;
  st.take(100);
  CHECK(st.chunks.size() == 1 && last_error == hipSuccess);
  const size_t used = ctx.used;
  DevBuf c(&ctx, &ret);
  for (int k = 0; k < 2; k++) {
    fail_next = 4;
    int status = 0;
    try {
      if (k == 0) c.ensure(1 << 20);
      else st.take(4 << 20);
    } catch (const Error& e) {
      status = e.status;
    }
    CHECK(status == NRGK_ERR_NOMEM && last_error == hipSuccess);
    CHECK(ctx.used == used && !c.p);
  }
  fail_next = 0;
  c.ensure(1 << 20);
  CHECK(c.p);
}

// Owners that grow, drop and replace buffers: what lies on the device never passes the capacity, whether used,
// retired or idle, what fits beside the buffers in use is not refused, and the account is what the buffers hold.
static void capacity_bounds(unsigned seed, Ctx& ctx, bool alone) {
  std::mt19937 rng(seed);
  auto owner = [&] {
    auto r = std::make_unique<Retired>();
    r->attach(&ctx, nullptr);
    return r;
  };
  struct Own {
    std::unique_ptr<Retired> r;
    std::vector<DevBuf> b;
  };
  std::vector<Own> own(3);
  size_t refused = 0;
  for (auto& o : own) o.r = owner();
  auto held = [&] {
    size_t n = 0;
    for (auto& o : own)
      for (auto& b : o.b) n += b.cap;
    return n;
  };
  for (int k = 0; k < 4000; k++) {
    Own& o = own[rng() % own.size()];
    const int what = rng() % 40;
    if (what == 0) {
      o.b.clear();
    } else if (what == 1) {
      o.r->give_all();  // (a synchronisation)
    } else if (what == 2) {
      o.b.clear();
      o.r = owner();
    } else {
      if (o.b.size() < 6) o.b.emplace_back(&ctx, o.r.get());
      DevBuf& b = o.b[rng() % o.b.size()];
      const size_t bytes = size_t(1) << (8 + rng() % 15), n = bytes + rng() % bytes;
      const size_t others = held() - (n > b.cap ? b.cap : 0), old = b.cap;
      try {
        b.ensure(n);
        CHECK(b.cap >= n && b.cap <= std::max(old, n + n / 4 + 256));
        static_cast<char*>(b.p)[0] = static_cast<char*>(b.p)[n - 1] = 1;
      } catch (const Error& e) {
        refused++;
        CHECK(e.status == NRGK_ERR_NOMEM && !b.p);
        if (alone) CHECK(others + MemPool::size_below(n + n / 4 + 256) > ctx.capacity);
      }
    }
  }
  if (alone) {
    for (auto& o : own) o.r->give_all();
    CHECK(ctx.used == held());
    CHECK(refused > 0);
  }
}
static void capacity() {
  Ctx ctx;
  ctx.set_capacity(size_t(20) << 20);
  for (unsigned s = 0; s < 5; s++) {
    live_peak = 0;
    capacity_bounds(s, ctx, true);
    CHECK(live_peak <= ctx.capacity && live_peak > ctx.capacity / 2);
    CHECK(ctx.used == 0 && live_bytes == ctx.pool.held());
  }
  std::vector<std::thread> ts;
  for (unsigned s = 0; s < 4; s++) ts.emplace_back([&, s] { capacity_bounds(100 + s, ctx, false); });
  for (auto& t : ts) t.join();
  CHECK(live_peak <= ctx.capacity);
  CHECK(ctx.used == 0 && live_bytes == ctx.pool.held());
}

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "staging_readback") staging_readback();
  else if (what == "failed_allocation") failed_allocation();
  else if (what == "capacity") capacity();
  else return 2;
  std::printf("%s: %s\n", what.c_str(), failures ? "failed" : "ok");
  return failures != 0;
}
