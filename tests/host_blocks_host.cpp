// Runs the runtime's device-block pool (zml_amd/csrc/runtime.cpp) on the CPU over a HIP
// that only counts: reads commands ("call BYTES.." one host-memory call with these
// blocks, "ws SLOT BYTES" a workspace, "room BYTES" the device's memory) and prints after
// each: allocations and frees of it, bytes held, and whether it failed.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <iostream>
#include <map>
#include <sstream>
#include <string>
#include <vector>

#include "../zml_amd/csrc/zmlhip_internal.hpp"

static std::map<void*, size_t> blocks;
static size_t held = 0, room = size_t(1) << 40;
static int mallocs = 0, frees = 0;

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  if (held + n > room) return hipErrorOutOfMemory;
  *p = malloc(1);
  blocks[*p] = n;
  held += n;
  ++mallocs;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (!blocks.count(p)) { printf("free of an unknown block\n"); exit(3); }
  held -= blocks[p];
  blocks.erase(p);
  free(p);
  ++frees;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) { *s = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t*, unsigned) { return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipExtStreamCreateWithCUMask(hipStream_t*, uint32_t, const uint32_t*) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t*) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t*, unsigned) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float*, hipEvent_t, hipEvent_t) { return hipSuccess; }
}

int main() {
  std::string line;
  while (std::getline(std::cin, line)) {
    std::istringstream in(line);
    std::string what;
    in >> what;
    mallocs = frees = 0;
    int failed = 0;
    try {
      if (what == "call") {
        std::vector<std::pair<void*, size_t>> mine;
        size_t n;
        try {
          while (in >> n) {
            size_t got = 0;
            void* const p = zmlhip::host_block(n, &got);
            if (got < n || blocks.at(p) != got) { printf("block of a wrong size\n"); return 3; }
            mine.emplace_back(p, got);
          }
        } catch (const zmlhip::HipError&) {
          failed = 1;
        }
        for (auto& b : mine) zmlhip::host_block_done(b.first, b.second, true);
      } else if (what == "ws") {
        size_t slot, n;
        in >> slot >> n;
        zmlhip::workspace(n, (int)slot);
      } else if (what == "room") {
        in >> room;
      }
    } catch (const zmlhip::HipError&) {
      failed = 1;
    }
    printf("%d %d %zu %d\n", mallocs, frees, held, failed);
  }
  return 0;
}
