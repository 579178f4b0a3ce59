// The HIP calls that a launch of libtriton_int_hip.so makes, for programs that run its host code on the CPU: they count launches and
// give or refuse memory.  Linked into the program itself (-rdynamic), they come before the runtime's.
#pragma once
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

static void* fake_address(size_t a) { return (void*)(a << 32); }  // 16-byte aligned, never read
