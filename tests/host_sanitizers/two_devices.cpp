// What a small vector's device blocks owe a caller, on two devices that exist only here: the runtime's calls that
// vector.cpp makes and the transfers of transfer.cpp are stand-ins that write down what was asked of which device.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "sarek_hip.h"
#include "transfer.hpp"

static int g_device = 0;
static int g_queued[2] = {0, 0};   // uploads left to the order of a device's default stream, not waited for
static int g_waits[2] = {0, 0};

extern "C" {
hipError_t hipGetDevice(int *d) { *d = g_device; return hipSuccess; }
hipError_t hipSetDevice(int d) { g_device = d; return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { *p = std::malloc(n); return hipSuccess; }
hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
  ++g_waits[g_device];
  g_queued[g_device] = 0;
  return hipSuccess;
}
int sarek_hip_memcpy_htod(void *dst, const void *src, size_t n) { std::memcpy(dst, src, n); return SAREK_HIP_OK; }
int sarek_hip_memcpy_dtoh(void *dst, const void *src, size_t n) { std::memcpy(dst, src, n); return SAREK_HIP_OK; }
int sarek_hip_host_alloc(void **p, size_t n) { *p = std::malloc(n ? n : 1); return SAREK_HIP_OK; }
int sarek_hip_host_free(void *p) { std::free(p); return SAREK_HIP_OK; }
int sarek_hip_mem_alloc_zero_copy(void *, size_t, void **, int *supported) { *supported = 0; return SAREK_HIP_OK; }
}
namespace sarek_hip {
int put_small(void *dst, const void *src, size_t n) {
  std::memcpy(dst, src, n);
  ++g_queued[g_device];
  return SAREK_HIP_OK;
}
int get_small(void *dst, const void *src, size_t n, int) { std::memcpy(dst, src, n); return SAREK_HIP_OK; }
}  // namespace sarek_hip

#define CHECK(c)                                              \
  do {                                                        \
    if (!(c)) {                                               \
      std::printf("line %d: %s\n", __LINE__, #c);             \
      return 1;                                               \
    }                                                         \
  } while (0)

int main() {
  sarek_hip_vector v;
  void *p = nullptr, *q = nullptr;
  const float x = 1.f, y = 2.f;
  CHECK(sarek_hip_vector_create(SAREK_HIP_KIND_FLOAT32, 256, 0, 0, &v) == 0);
  CHECK(sarek_hip_vector_fill(v, &x) == 0);
  // an upload on each device, then the address on the second: it waits for that device's stream alone
  CHECK(sarek_hip_transfer_to_device(v) == 0 && g_queued[0] == 1);
  hipSetDevice(1);
  CHECK(sarek_hip_vector_fill(v, &y) == 0 && sarek_hip_transfer_to_device(v) == 0 && g_queued[1] == 1);
  CHECK(sarek_hip_vector_device_ptr(v, &q) == 0 && q && g_waits[1] == 1 && g_waits[0] == 0);
  // the first device's upload is still queued: its address waits for it
  hipSetDevice(0);
  CHECK(sarek_hip_vector_device_ptr(v, &p) == 0 && p && p != q && g_waits[0] == 1 && g_queued[0] == 0);
  CHECK(sarek_hip_vector_device_ptr(v, &p) == 0 && g_waits[0] == 1);
  // blocks whose address is known get uploads that are complete
  CHECK(sarek_hip_vector_fill(v, &x) == 0 && sarek_hip_transfer_to_device(v) == 0 && g_queued[0] == 0);
  CHECK(static_cast<float *>(p)[255] == 1.f && static_cast<float *>(q)[255] == 2.f);
  CHECK(sarek_hip_vector_destroy(v) == 0);
  // an address on one device says nothing about the block on the other
  CHECK(sarek_hip_vector_create(SAREK_HIP_KIND_FLOAT32, 256, 0, 0, &v) == 0 && sarek_hip_vector_fill(v, &x) == 0);
  CHECK(sarek_hip_transfer_to_device(v) == 0 && sarek_hip_vector_device_ptr(v, &p) == 0);
  hipSetDevice(1);
  g_queued[1] = 0;
  CHECK(sarek_hip_vector_fill(v, &y) == 0 && sarek_hip_transfer_to_device(v) == 0 && g_queued[1] == 1);
  // new blocks after the old ones were given back
  CHECK(sarek_hip_vector_device_ptr(v, &q) == 0 && sarek_hip_transfer_free_buffers(v) == 0);
  CHECK(sarek_hip_vector_device_ptr(v, &q) == 0 && q == nullptr);
  g_queued[1] = 0;
  CHECK(sarek_hip_transfer_to_device(v) == 0 && g_queued[1] == 1);
  CHECK(sarek_hip_vector_destroy(v) == 0);
  std::printf("two devices ok\n");
  return 0;
}
