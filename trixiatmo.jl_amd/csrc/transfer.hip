// Copies from the device to caller memory.  A copy into pageable memory runs at
// the rate of one host thread, which also meets the pages of a fresh destination
// one by one (the system clears each as it is first written): 74 MB of state took
// 7.2 ms where the link moves them in 1.3 ms.  A large copy goes through pinned
// slots instead, each emptied by a thread of its own while the others are on the
// link: 2.2 ms (38 MB 3.9 -> 1.7, 16 MB 0.94 -> 0.55).  The other direction gains
// little that way (74 MB 2.5 -> 2.1 ms, 16 MB 0.48 -> 0.57) and stays plain.
//
// The slots belong to the process (pinning them costs milliseconds): taken by
// one copy at a time, a copy that finds them taken goes the plain way; they are
// given back when the last handle is destroyed.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstring>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

#include "handle.hpp"

namespace atmo {

namespace {

constexpr int kSlots = 8;
constexpr size_t kSlotBytes = (size_t)2 << 20;
// below this the threads cost what they save (5 MB: 0.29 ms either way)
constexpr size_t kStagedBytes = (size_t)8 << 20;

struct Slots {
  std::mutex mutex;       // held by the copy that uses the slots
  char* memory = nullptr;  // kSlots * kSlotBytes, pinned for every device
};
Slots g_slots;
std::atomic<int> g_handles{0};

// one copy: its chunks are taken in order by whichever thread is free
struct Copy {
  atmo_handle* h;
  char* dst;
  const char* src;
  size_t bytes;
  std::atomic<size_t> next{0};
  std::atomic<int> error{(int)hipSuccess};

  void fail(hipError_t e) {
    int none = (int)hipSuccess;
    error.compare_exchange_strong(none, (int)e);
  }

  // on a thread whose current device is the handle's
  void work(char* slot) {
    hipEvent_t ev = nullptr;
    hipError_t e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
    while (e == hipSuccess && error.load() == (int)hipSuccess) {
      const size_t at = next.fetch_add(1) * kSlotBytes;
      if (at >= bytes) break;
      const size_t len = bytes - at < kSlotBytes ? bytes - at : kSlotBytes;
      e = hipMemcpyAsync(slot, src + at, len, hipMemcpyDeviceToHost, h->stream);
      if (e == hipSuccess) e = hipEventRecord(ev, h->stream);
      if (e == hipSuccess) e = hipEventSynchronize(ev);
      if (e == hipSuccess) std::memcpy(dst + at, slot, len);
    }
    if (e != hipSuccess) fail(e);
    if (ev) (void)hipEventDestroy(ev);
  }

  void work_on_device(char* slot) {
    const hipError_t e = hipSetDevice(h->device);
    if (e == hipSuccess) work(slot);
    else fail(e);
  }
};

// whether p is memory that HIP does not know: the system's own, pageable
bool pageable(const void* p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return true;
}

}  // namespace

hipError_t copy_to_host(atmo_handle* h, void* dst, const void* src, size_t bytes) {
  if (bytes >= kStagedBytes && pageable(dst)) {
    std::unique_lock<std::mutex> lock(g_slots.mutex, std::try_to_lock);
    if (lock.owns_lock() &&
        (g_slots.memory || hipHostMalloc(reinterpret_cast<void**>(&g_slots.memory),
                                         kSlots * kSlotBytes, hipHostMallocPortable) == hipSuccess)) {
      Copy c{h, static_cast<char*>(dst), static_cast<const char*>(src), bytes};
      std::vector<std::thread> threads;
      try {  // with fewer threads than slots the others take the chunks
        threads.reserve(kSlots - 1);
        for (int t = 1; t < kSlots; ++t)
          threads.emplace_back(&Copy::work_on_device, &c, g_slots.memory + t * kSlotBytes);
      } catch (const std::system_error&) {
      } catch (const std::bad_alloc&) {
      }
      int device = h->device;  // the caller's, given back to it
      (void)hipGetDevice(&device);
      c.work_on_device(g_slots.memory);
      if (device != h->device) (void)hipSetDevice(device);
      for (auto& t : threads) t.join();
      // a copy may still be on its way into a slot if another failed
      const hipError_t e = hipStreamSynchronize(h->stream);
      return c.error.load() != (int)hipSuccess ? (hipError_t)c.error.load() : e;
    }
    if (lock.owns_lock()) {
      g_slots.memory = nullptr;
      (void)hipGetLastError();  // no pinned memory: the plain copy below
    }
  }
  const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, h->stream);
  return e == hipSuccess ? hipStreamSynchronize(h->stream) : e;
}

HandleCount::HandleCount() { g_handles.fetch_add(1); }

HandleCount::~HandleCount() {
  if (g_handles.fetch_sub(1) != 1) return;
  std::lock_guard<std::mutex> lock(g_slots.mutex);
  // a handle created meanwhile keeps them
  if (g_handles.load() != 0 || !g_slots.memory) return;
  (void)hipHostFree(g_slots.memory);
  g_slots.memory = nullptr;
}

}  // namespace atmo
