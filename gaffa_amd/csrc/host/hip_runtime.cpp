// RAII device memory / streams over the C ABI, and the mapping of C-ABI
// status codes onto the exception classes gaffa throws.
#include "gaffa/gpu_memory.h"

#include <iterator>
#include <list>
#include <map>
#include <mutex>
#include <stdexcept>
#include <string>

namespace gaffa {

namespace {

// Released device memory kept for reuse (see GpuDeviceMemory).  Every call is made
// with the block's device current.
class DeviceCache {
 public:
  // Never destroyed: the runtime may be gone before static destructors run.
  static DeviceCache& get() {
    static DeviceCache* cache = [] {
      auto* c = new DeviceCache;
      (void)gaffa_hip_set_reclaim([](int32_t device) -> int { return get().release(device); });
      return c;
    }();
    return *cache;
  }

  // An allocation of at least `bytes`; `block` becomes its size.
  void* take(int device, std::size_t bytes, std::size_t& block) {
    {
      std::lock_guard<std::mutex> lock(mutex_);
      auto best = blocks_.end();
      for (auto it = blocks_.begin(); it != blocks_.end(); ++it)
        if (it->device == device && it->bytes >= bytes && it->bytes - bytes <= bytes / 4 &&
            (best == blocks_.end() || it->bytes < best->bytes))
          best = it;
      if (best != blocks_.end()) {
        void* p = best->data;
        block = best->bytes;
        devices_.find(device)->second.bytes -= block;
        blocks_.erase(best);
        return p;
      }
    }
    void* p = nullptr;
    block = bytes;
    hip_ok(gaffa_hip_malloc(&p, bytes), "hipMalloc");
    return p;
  }

  // `idle`: the device is known to be done with the block.
  int give(int device, void* data, std::size_t bytes, bool idle = false) noexcept {
    std::list<Block> own, out;
    Device* held = nullptr;
    try {  // all that can fail for want of host memory comes before the block is listed
      own.push_back(Block{device, data, bytes});
      held = &state(device);
    } catch (...) {
      return gaffa_hip_free(data);
    }
    if (bytes > held->limit) return gaffa_hip_free(data);
    // no kernel of any stream uses the block after this, as with hipFree
    const int status = idle ? GAFFA_HIP_OK : wait_for_device();
    if (status != GAFFA_HIP_OK) {
      (void)gaffa_hip_free(data);
      return status;
    }
    {
      std::lock_guard<std::mutex> lock(mutex_);
      blocks_.splice(blocks_.end(), own);
      held->bytes += bytes;
      for (auto it = blocks_.begin(); held->bytes > held->limit;) {
        const auto next = std::next(it);
        if (it->device == device) {
          held->bytes -= it->bytes;
          out.splice(out.end(), blocks_, it);
        }
        it = next;
      }
    }
    int freed = GAFFA_HIP_OK;
    for (const Block& b : out) {
      const int st = gaffa_hip_free(b.data);
      if (freed == GAFFA_HIP_OK) freed = st;
    }
    return freed;
  }

  // Frees what is kept on `device`; whether there was anything.
  bool release(int device) {
    std::list<Block> out;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      for (auto it = blocks_.begin(); it != blocks_.end();) {
        const auto next = std::next(it);
        if (it->device == device) {
          devices_.find(device)->second.bytes -= it->bytes;
          out.splice(out.end(), blocks_, it);
        }
        it = next;
      }
    }
    for (const Block& b : out) (void)gaffa_hip_free(b.data);
    return !out.empty();
  }

 private:
  struct Block {
    int device;
    void* data;
    std::size_t bytes;
  };
  struct Device {
    std::size_t bytes = 0;  // kept
    std::size_t limit = 0;
  };

  // Waits until the device is idle by freeing an allocation of a byte (under 1 us
  // on an idle device): hipFree waits as hipDeviceSynchronize does, but a device
  // synchronisation is refused while another thread captures a graph, and ends
  // that capture with an error.
  static int wait_for_device() {
    void* token = nullptr;
    const int status = gaffa_hip_malloc(&token, 1);
    return status == GAFFA_HIP_OK ? gaffa_hip_free(token) : status;
  }

  // A device's entry, made at its first release (a map's entries never move).
  Device& state(int device) {
    std::lock_guard<std::mutex> lock(mutex_);
    const auto [it, fresh] = devices_.try_emplace(device);
    if (fresh) {
      gaffa_hip_device_info info{};
      const bool ok = gaffa_hip_device_info_get(device, &info) == GAFFA_HIP_OK;
      it->second.limit = ok ? static_cast<std::size_t>(info.total_memory) / 32 : 0;
    }
    return it->second;
  }

  std::mutex mutex_;
  std::list<Block> blocks_;  // oldest first
  std::map<int, Device> devices_;
};

}  // namespace

void release_device_cache() {
  for (int d = 0; d < gpu_device_count(); ++d) {
    GpuDeviceScope scope(d);
    (void)DeviceCache::get().release(d);
  }
}

void throw_hip_status(int status, const char* what) {
  const std::string msg = gaffa_hip_last_error();
  const std::string full = msg.empty() ? std::string(what) : msg;
  switch (status) {
    case GAFFA_HIP_INVALID_ARGUMENT:
      throw std::invalid_argument(full);
    case GAFFA_HIP_OVERFLOW:
      throw std::overflow_error(full);
    case GAFFA_HIP_OUT_OF_RANGE:
      throw std::out_of_range(full);
    case GAFFA_HIP_LOGIC:
      throw std::logic_error(full);
    default:
      throw std::runtime_error(std::string(what) + ": " + full);
  }
}

GpuDeviceScope::GpuDeviceScope(int device_id) {
  int32_t cur = 0;
  hip_ok(gaffa_hip_get_device(&cur), "hipGetDevice");
  previous_ = cur;
  if (cur != device_id) {
    hip_ok(gaffa_hip_set_device(device_id), "hipSetDevice");
    restore_ = true;
  }
}

GpuDeviceScope::~GpuDeviceScope() {
  if (restore_) (void)gaffa_hip_set_device(previous_);
}

GpuDeviceMemory::GpuDeviceMemory(std::size_t bytes) {
  int32_t dev = 0;
  hip_ok(gaffa_hip_get_device(&dev), "hipGetDevice");
  if (bytes != 0) data_ = DeviceCache::get().take(dev, bytes, block_);
  bytes_ = bytes;
  device_id_ = dev;
}

GpuDeviceMemory::GpuDeviceMemory(GpuDeviceMemory&& o) noexcept
    : data_(std::exchange(o.data_, nullptr)),
      bytes_(std::exchange(o.bytes_, 0)),
      block_(std::exchange(o.block_, 0)),
      device_id_(std::exchange(o.device_id_, -1)) {}

GpuDeviceMemory& GpuDeviceMemory::operator=(GpuDeviceMemory&& o) noexcept {
  if (this != &o) {
    release_noexcept();
    data_ = std::exchange(o.data_, nullptr);
    bytes_ = std::exchange(o.bytes_, 0);
    block_ = std::exchange(o.block_, 0);
    device_id_ = std::exchange(o.device_id_, -1);
  }
  return *this;
}

GpuDeviceMemory::~GpuDeviceMemory() { release_noexcept(); }

void GpuDeviceMemory::reset() {
  if (data_ != nullptr) {
    GpuDeviceScope scope(device_id_);
    bytes_ = 0;
    hip_ok(DeviceCache::get().give(device_id_, std::exchange(data_, nullptr),
                                   std::exchange(block_, 0)),
           "hipFree");
  }
  bytes_ = 0;
}

void GpuDeviceMemory::release_together(std::initializer_list<GpuDeviceMemory*> blocks) noexcept {
  bool idle = false;
  for (GpuDeviceMemory* m : blocks) idle = m->release_noexcept(idle);
}

bool GpuDeviceMemory::release_noexcept(bool idle) noexcept {
  if (data_ == nullptr) return idle;
  int32_t cur = 0;
  const bool switch_dev = gaffa_hip_get_device(&cur) == 0 && cur != device_id_;
  if (switch_dev) (void)gaffa_hip_set_device(device_id_);
  idle = DeviceCache::get().give(device_id_, data_, block_, idle) == GAFFA_HIP_OK;
  if (switch_dev) (void)gaffa_hip_set_device(cur);
  data_ = nullptr;
  bytes_ = 0;
  block_ = 0;
  return idle;
}

GpuStream GpuStream::create() {
  GpuStream s;
  hip_ok(gaffa_hip_stream_create(&s.s_), "hipStreamCreate");
  return s;
}

void GpuStream::synchronize() const {
  hip_ok(gaffa_hip_stream_synchronize(s_), "hipStreamSynchronize");
}

void GpuStream::destroy() noexcept {
  if (s_ != nullptr) (void)gaffa_hip_stream_destroy(s_);
  s_ = nullptr;
}

GpuPinnedBuffer::GpuPinnedBuffer(std::size_t bytes) : bytes_(bytes) {
  hip_ok(gaffa_hip_host_malloc(&p_, bytes), "hipHostMalloc");
}

void GpuPinnedBuffer::release() noexcept {
  if (p_ != nullptr) (void)gaffa_hip_host_free(p_);
  p_ = nullptr;
  bytes_ = 0;
}

GpuEvent::GpuEvent() { hip_ok(gaffa_hip_event_create(&e_), "hipEventCreate"); }

GpuEvent::~GpuEvent() {
  if (e_ != nullptr) (void)gaffa_hip_event_destroy(e_);
}

void GpuEvent::record(gaffa_hip_stream stream) {
  hip_ok(gaffa_hip_event_record(e_, stream), "hipEventRecord");
}

void GpuEvent::wait(gaffa_hip_stream stream) {
  hip_ok(gaffa_hip_stream_wait_event(stream, e_), "hipStreamWaitEvent");
}

void GpuEvent::synchronize() { hip_ok(gaffa_hip_event_synchronize(e_), "hipEventSynchronize"); }

void copy_to_device(void* dst, const void* src, std::size_t bytes, gaffa_hip_stream stream) {
  hip_ok(gaffa_hip_memcpy(dst, src, bytes, stream), "hipMemcpy host-to-device");
}

void copy_to_host(void* dst, const void* src, std::size_t bytes, gaffa_hip_stream stream) {
  hip_ok(gaffa_hip_memcpy(dst, src, bytes, stream), "hipMemcpy device-to-host");
  if (stream != nullptr) hip_ok(gaffa_hip_stream_synchronize(stream), "hipStreamSynchronize");
}

int gpu_device_count() {
  int32_t n = 0;
  hip_ok(gaffa_hip_device_count(&n), "hipGetDeviceCount");
  return n;
}

int gpu_runtime_version() {
  gaffa_hip_device_info info{};
  if (gpu_device_count() == 0) return 0;
  hip_ok(gaffa_hip_device_info_get(0, &info), "hipGetDeviceProperties");
  return info.runtime_version;
}

}  // namespace gaffa
