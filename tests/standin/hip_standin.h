// A stand-in for the HIP runtime, for tests of the library's host code on a machine without a
// GPU: the library's objects, their device code left out, are linked with it instead of
// libamdhip64.  Device memory is host memory, copies are copies, and a kernel launch is recorded
// and leaves what the kernel tells the host (its completion words), but no sums.
#pragma once

#include <cstdint>
#include <string>
#include <vector>

namespace standin {

struct Launch {
  std::string kernel;               // the device function's mangled name
  uint32_t grid, block;
  void* stream;
  bool captured;                    // recorded into a graph, not run
  std::vector<char> scan_args;      // scan kernels: their ScanArgs
  void* workspace = nullptr;        // scan_fast: its workspace argument
  std::vector<char> fetch_args;     // fetch_columns: its FetchArgs
  bool is(const char* part) const { return kernel.find(part) != std::string::npos; }
};

struct Copy {
  const void* src;
  uint64_t bytes;
  bool to_device;
};

struct State {
  std::vector<Launch> launches;
  std::vector<Copy> copies;
  uint64_t device_bytes = 0;        // allocated by hipMalloc
  uint64_t budget = UINT64_MAX;     // hipMalloc fails beyond it
  uint64_t stream_waits = 0;        // calls of hipStreamSynchronize
  uint64_t device_waits = 0;        // calls of hipDeviceSynchronize
  uint64_t frees = 0;               // calls of hipFree
  void* capturing = nullptr;        // a stream that is being captured
  bool silent = false;              // kernels end without telling the host
  unsigned device_flags = 0;        // what hipGetDeviceFlags says
  void* late_stream = nullptr;      // stream whose kernels tell the host only `late_us` later
  int late_us = 0;
};
State& state();

// Makes [base, base + bytes) pinned host memory, one range, as hipHostMalloc does.
void pin(const void* base, uint64_t bytes);

}  // namespace standin
