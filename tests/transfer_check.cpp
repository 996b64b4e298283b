// The library's host transfers (qcd_amd/csrc/transfer.cpp) on two devices that
// are host memory: the HIP calls they make, with the rule that an event is
// recorded on streams of its own device only.  The library's device is 1, the
// calling thread's 0.  Prints "ok".
#include "internal.h"

struct ihipStream_t { int device; };
struct ihipEvent_t { int device; };

static thread_local int current = 0;
static int allocations = 0, events = 0, copies = 0;
static bool no_memory = false;
static ihipStream_t stream{1};
static qcdhip::Context context;

extern "C" {
hipError_t hipGetDevice(int *d) { *d = current; return hipSuccess; }
hipError_t hipSetDevice(int d) { current = d; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *) {
  a->type = hipMemoryTypeUnregistered;
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  if (no_memory || !(*p = malloc(n))) return hipErrorOutOfMemory;
  allocations++;
  return hipSuccess;
}
hipError_t hipHostFree(void *p) { free(p); allocations--; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = new ihipEvent_t{current}; events++; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { delete e; events--; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  return e->device == s->device ? hipSuccess : hipErrorInvalidHandle;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  memcpy(d, s, n);
  __atomic_add_fetch(&copies, 1, __ATOMIC_RELAXED);
  return hipSuccess;
}
}
namespace qcdhip {
Context *ctx() { return &context; }
}

#define CHECK(x) do { if (!(x)) { printf("failed: %s (line %d)\n", #x, __LINE__); return 1; } } while (0)

int main() {
  context.device = 1;
  for (int pass = 0; pass < 3; pass++) {
    no_memory = pass == 2;   // the runtime's copy
    const size_t MB = (size_t)1 << 20;
    for (size_t n : {(size_t)1000, 8 * MB - 24, 8 * MB, 12 * MB - 24, 12 * MB, 12 * MB + 24, (size_t)20971528}) {
      std::vector<char> host(n), dev(n, 0), back(n, 0);
      for (size_t i = 0; i < n; i++) host[i] = (char)(i * 2654435761u >> 13);
      copies = 0;
      CHECK(qcdhip::host_copy(dev.data(), host.data(), n, true, &stream) == hipSuccess);
      CHECK(dev == host);
      CHECK((copies > 1) == (n >= 12 * MB && !no_memory));
      copies = 0;
      CHECK(qcdhip::host_copy(dev.data(), back.data(), n, false, &stream) == hipSuccess);
      CHECK(back == host);
      CHECK(current == 0);
      CHECK((copies > 1) == (n >= 8 * MB && !no_memory));
    }
    CHECK(allocations == (no_memory ? 0 : 1) && events == (no_memory ? 0 : 4));
    qcdhip::host_slots_free();
    CHECK(allocations == 0 && events == 0);
  }
  puts("ok");
  return 0;
}
