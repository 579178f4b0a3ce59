// Runs GEMM launches of libtriton_int_hip.so on the CPU: the HIP calls that a launch makes are the ones below, which count
// launches and give or refuse memory.  Arguments: `capturing` or `none`, bytes that hipMalloc gives in all, then launches of
// "M,N,K" (fp32 out), each on the same stream.  Prints a line per launch: status, configuration, K splits, launches, bytes held.
#include <hip/hip_runtime_api.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <map>

#include "../../include/triton_int_hip.h"

static bool capturing;
static size_t room, held;
static int launches;
static hipError_t last = hipSuccess;
static std::map<void*, size_t> blocks;
static dim3 grid, block;
static size_t lds;
static hipStream_t queue;

extern "C" {
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
  if (held + n > room) return last = hipErrorOutOfMemory;
  *p = aligned_alloc(256, 256);  // never read: nothing runs
  blocks[*p] = n;
  held += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  held -= blocks[p];
  blocks.erase(p);
  free(p);
  return hipSuccess;
}
hipError_t hipGetLastError(void) {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
  *s = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t l, hipStream_t s) {
  grid = g, block = b, lds = l, queue = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* l, hipStream_t* s) {
  *g = grid, *b = block, *l = lds, *s = queue;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) {
  ++launches;
  return hipSuccess;
}
}

int main(int argc, char** argv) {
  capturing = !strcmp(argv[1], "capturing");
  room = strtoull(argv[2], nullptr, 0);
  for (int i = 3; i < argc; ++i) {
    int M, N, K;
    if (sscanf(argv[i], "%d,%d,%d", &M, &N, &K) != 3) return 2;
    const auto at = [](size_t a) { return (void*)(a << 32); };  // 16-byte aligned, never read
    launches = 0;
    const int rc = ti_bmm_i8((const int8_t*)at(1), 0, K, 1, (const int8_t*)at(2), 0, K, 1, at(3), 0, N, 1, 1, M, N, K, nullptr, TI_BIAS_NONE, (const float*)at(4),
                             nullptr, TI_EPI_SCALE_F, TI_F32, TI_ROUND_RNE_CLAMP, (void*)16);
    printf("%d %s %d %d %zu\n", rc, ti_gemm_config_name(ti_gemm_last_config()), ti_gemm_last_splits(), launches, held);
  }
  return 0;
}
