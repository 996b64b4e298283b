// transfer.cpp -- large copies between device and host memory.
//
// Copies from and to ordinary (pageable) host memory.  The runtime's own
// copy of such memory runs at 30 GB/s up and 18 GB/s down of the 57 GB/s that
// pinned memory reaches, one host thread copying at a time.  Here the caller
// and one helper thread take every other chunk, each through two pinned slots:
// one is on the bus while the other is filled or emptied.  75 MB up 2530 -> 1800
// us (chunks of 4 MB; 1 MB 2440, 8 MB 1810; one thread 2640, four 1810), 25 MB
// up 673 -> 650, down 1416 -> 742 (chunks of 2 MB; 4 MB 771; one thread 970).
// The shortest that gain, us: up 8.8 MB 271 -> 310, 9.8 300 -> 350, 11.8 378 -> 387,
// 13.8 495 -> 433; down 8.8 MB 519 -> 364.
// The slots (16 MB) are kept and given back by qcd_hip_release_cache.  All calls
// hold state_mutex.  The calling thread's current device need not be the library's
// (streams name their device; memory and events take the current one), and is left
// as it is.
#include "internal.h"

#include <thread>

namespace qcdhip {

constexpr size_t kSlotBytes = (size_t)4 << 20, kDownChunk = (size_t)2 << 20;
constexpr size_t kUpMin = (size_t)12 << 20, kDownMin = (size_t)8 << 20;
struct HostSlots {
  char *mem = nullptr;   // four slots: two of the caller, two of the helper
  hipEvent_t ev[4] = {};
  bool used[4] = {};     // ev holds the last copy through the slot
};
static HostSlots g_slots;

void host_slots_free() {
  for (int i = 0; i < 4; i++) {
    if (g_slots.used[i]) (void)hipEventSynchronize(g_slots.ev[i]);
    if (g_slots.ev[i]) (void)hipEventDestroy(g_slots.ev[i]);
  }
  if (g_slots.mem) (void)hipHostFree(g_slots.mem);
  g_slots = HostSlots{};
}

static bool slots_ready() {
  if (g_slots.mem) return true;
  int current = 0;
  if (hipGetDevice(&current) != hipSuccess || hipSetDevice(ctx()->device) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  bool ok = hipHostMalloc((void **)&g_slots.mem, 4 * kSlotBytes, hipHostMallocDefault) == hipSuccess;
  if (!ok) g_slots.mem = nullptr;
  for (int i = 0; ok && i < 4; i++)
    ok = hipEventCreateWithFlags(&g_slots.ev[i], hipEventDisableTiming) == hipSuccess;
  if (!ok) {
    (void)hipGetLastError();
    host_slots_free();
  }
  (void)hipSetDevice(current);
  return ok;
}

// whether p is memory that the runtime does not know (no pinned, managed or
// device allocation, which its own copy handles best)
static bool pageable(const void *p) {
  hipPointerAttribute_t at;
  if (hipPointerGetAttributes(&at, p) == hipSuccess) return at.type == hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return true;
}

// chunks first, first + step, .. through slots s0 and s0 + 1
static hipError_t copy_chunks(char *dev, char *host, size_t bytes, size_t chunk, size_t first, size_t step, int s0,
                              bool up, hipStream_t st) {
  size_t at[2] = {}, len[2] = {};   // of the chunk on its way down through a slot
  auto drain = [&](int i) -> hipError_t {
    const int s = s0 + i;
    if (!g_slots.used[s]) return hipSuccess;
    const hipError_t e = hipEventSynchronize(g_slots.ev[s]);
    if (e == hipSuccess && !up && len[i]) std::memcpy(host + at[i], g_slots.mem + s * kSlotBytes, len[i]);
    len[i] = 0;
    return e;
  };
  int i = 0;
  for (size_t o = first * chunk; o < bytes; o += step * chunk, i ^= 1) {
    char *slot = g_slots.mem + (s0 + i) * kSlotBytes;
    const size_t n = std::min(chunk, bytes - o);
    hipError_t e = drain(i);
    if (e != hipSuccess) return e;
    if (up) std::memcpy(slot, host + o, n);
    e = up ? hipMemcpyAsync(dev + o, slot, n, hipMemcpyHostToDevice, st)
           : hipMemcpyAsync(slot, dev + o, n, hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipEventRecord(g_slots.ev[s0 + i], st);
    if (e != hipSuccess) return e;
    g_slots.used[s0 + i] = true;
    at[i] = o;
    len[i] = n;
  }
  for (int k = 0; k < 2 && !up; k++, i ^= 1) {
    const hipError_t e = drain(i);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// Copy between device and host on st.  The caller holds state_mutex and waits
// for st before it touches or frees either side.
hipError_t host_copy(void *dev, void *host, size_t bytes, bool up, hipStream_t st) {
  if (bytes < (up ? kUpMin : kDownMin) || !pageable(host) || !slots_ready())
    return up ? hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, st)
              : hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st);
  const size_t chunk = up ? kSlotBytes : kDownChunk;
  const int device = ctx()->device;
  hipError_t e1 = hipSuccess;
  std::thread helper;
  try {
    helper = std::thread([&, device] {
      e1 = hipSetDevice(device);
      if (e1 == hipSuccess) e1 = copy_chunks((char *)dev, (char *)host, bytes, chunk, 1, 2, 2, up, st);
    });
  } catch (...) {   // no thread to be had: the caller takes all chunks
    return copy_chunks((char *)dev, (char *)host, bytes, chunk, 0, 1, 0, up, st);
  }
  const hipError_t e0 = copy_chunks((char *)dev, (char *)host, bytes, chunk, 0, 2, 0, up, st);
  helper.join();
  return e0 != hipSuccess ? e0 : e1;
}

}  // namespace qcdhip
