// The device memory kept for reuse (host/hip_runtime.cpp) over a stub of the HIP
// library, with host allocations that fail on demand.  Exits with the number of
// failed checks.
#include "gaffa/gpu_memory.h"

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>

namespace {

int failures = 0;
void expect(bool ok, const char* what, int k) {
  if (ok) return;
  ++failures;
  std::printf("failed: %s (host allocation %d)\n", what, k);
}

long fail_at = -1;  // the host allocation to refuse, counted down

constexpr int kMaxLive = 256;
struct {
  void* p;
  int device;
  uint64_t bytes;
} live[kMaxLive];
int current = 0;
uint64_t used = 0;
constexpr uint64_t kMemory = 1 << 20;  // per device; the sum of all is bounded here

int live_count() {
  int n = 0;
  for (const auto& l : live) n += l.p != nullptr;
  return n;
}
bool is_live(const void* p) {
  for (const auto& l : live)
    if (l.p == p) return p != nullptr;
  return false;
}

}  // namespace

void* operator new(std::size_t n) {
  if (fail_at >= 0 && fail_at-- == 0) throw std::bad_alloc();
  if (void* p = std::malloc(n != 0 ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

extern "C" {
const char* gaffa_hip_last_error(void) { return "stub"; }
int gaffa_hip_device_count(int32_t* n) { return *n = 64, 0; }
int gaffa_hip_get_device(int32_t* d) { return *d = current, 0; }
int gaffa_hip_set_device(int32_t d) { return current = d, 0; }
int gaffa_hip_device_info_get(int32_t, gaffa_hip_device_info* out) {
  std::memset(out, 0, sizeof(*out));
  out->total_memory = kMemory;
  return 0;
}
gaffa_hip_reclaim_fn reclaim = nullptr;
int gaffa_hip_set_reclaim(gaffa_hip_reclaim_fn f) { return reclaim = f, 0; }
int waits = 0;  // one-byte allocations
int gaffa_hip_malloc(void** p, uint64_t bytes) {
  *p = nullptr;
  waits += bytes == 1;
  if (used + bytes > kMemory && reclaim != nullptr) (void)reclaim(current);
  if (used + bytes > kMemory) return GAFFA_HIP_RUNTIME;
  for (auto& l : live)
    if (l.p == nullptr) {
      l.p = *p = std::malloc(bytes);
      l.device = current;
      l.bytes = bytes;
      used += bytes;
      return 0;
    }
  return GAFFA_HIP_RUNTIME;
}
int gaffa_hip_free(void* p) {
  if (p == nullptr) return 0;
  for (auto& l : live)
    if (l.p == p) {
      // not returned to the host: no later allocation has this address by chance
      l.p = nullptr;
      used -= l.bytes;
      return 0;
    }
  expect(false, "freed memory is freed again", -1);
  return GAFFA_HIP_RUNTIME;
}
int gaffa_hip_memcpy(void*, const void*, uint64_t, gaffa_hip_stream) { return 0; }
int gaffa_hip_stream_create(gaffa_hip_stream*) { return 0; }
int gaffa_hip_stream_destroy(gaffa_hip_stream) { return 0; }
int gaffa_hip_stream_synchronize(gaffa_hip_stream) { return 0; }
int gaffa_hip_stream_wait_event(gaffa_hip_stream, gaffa_hip_event) { return 0; }
int gaffa_hip_host_malloc(void**, uint64_t) { return 0; }
int gaffa_hip_host_free(void*) { return 0; }
int gaffa_hip_event_create(gaffa_hip_event*) { return 0; }
int gaffa_hip_event_destroy(gaffa_hip_event) { return 0; }
int gaffa_hip_event_record(gaffa_hip_event, gaffa_hip_stream) { return 0; }
int gaffa_hip_event_synchronize(gaffa_hip_event) { return 0; }
}

int main() {
  // The first releases on a device, one host allocation refused in each: the
  // memory is kept or freed, and never both.
  for (int reset = 0; reset < 2; ++reset)
    for (int k = 0; k < 12; ++k) {
      current = 12 * reset + k;
      gaffa::GpuDeviceMemory first(1000);
      fail_at = k;
      try {
        if (reset != 0) first.reset();
        else first = gaffa::GpuDeviceMemory();
      } catch (const std::bad_alloc&) {
        expect(false, "a release throws", k);
      }
      fail_at = -1;
      {
        gaffa::GpuDeviceMemory again(1000), more(1000);
        expect(is_live(again.data()) && is_live(more.data()), "freed memory handed out", k);
        expect(again.data() != more.data(), "memory handed out twice", k);
      }
      gaffa::release_device_cache();
      expect(live_count() == 0, "memory lost", k);
    }
  // the bound (1/32 of the device), oldest first
  current = 30;
  { gaffa::GpuDeviceMemory a(kMemory / 64), b(kMemory / 48), c(kMemory / 40); }
  expect(used <= kMemory / 32 && used > 0, "more kept than the bound, or nothing", 0);
  gaffa::release_device_cache();
  expect(live_count() == 0, "memory lost", 0);
  // one wait for several; each is kept or freed
  {
    gaffa::GpuDeviceMemory a(5000), b(kMemory / 8), c(7000), d(300);
    a.reset();
    waits = 0;
    gaffa::GpuDeviceMemory::release_together({&a, &b, &c, &d});
    expect(waits == 0 && b.data() == nullptr && d.data() == nullptr, "wait after a free", 0);
    gaffa::GpuDeviceMemory e(5000), f(7000), g(300);
    gaffa::GpuDeviceMemory::release_together({&e, &f, &g});
    expect(waits == 1, "not one wait", waits);
  }
  gaffa::release_device_cache();
  expect(live_count() == 0, "memory lost", 0);
  // an allocation that needs what is kept gets it
  current = 31;
  { gaffa::GpuDeviceMemory kept(kMemory / 40); }
  { gaffa::GpuDeviceMemory all(kMemory); }
  expect(used == 0, "more kept than the bound", 0);
  std::printf("%d failures\n", failures);
  return failures < 100 ? failures : 100;
}
