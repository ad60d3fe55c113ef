// Scratch memory of the entry point that allocates nothing (q1_enqueue_noalloc): a static
// per-device array, so that a caller that cannot allocate device memory (code under HIP
// graph capture, serving loops that forbid hipMalloc) can still run the scan kernels that
// need scratch -- the merge set of grids of kSpreadMinBlocks blocks or more, and the global
// placement's per-block tables.
//
// Every GPU the library runs on holds its own copy of `scratch` until the process ends.
// In host code `scratch` names a host-side stand-in, not a device address: q1_init looks up
// each device's address once (hipGetSymbolAddress, with that device current) and every use
// goes through that address.  All calls on one GPU share the array, which keeps the last
// call's contents: the merge set is cleared before every launch that uses it, and the global
// placement's per-block tables are cleared by the kernel itself.  Calls that overlap on one GPU race:
// their own results are wrong, those of later calls are not.
#include <hip/hip_runtime.h>

#include <mutex>

#include "q1_internal.h"

namespace {

constexpr uint64_t kScratchBytes = sizeof(q1::MergeSet) + q1::kNoallocWorkspaceBytes;
constexpr int kMaxDevices = 64;

static __device__ __align__(256) uint64_t scratch[kScratchBytes / 8];

std::mutex g_lock;
void* g_scratch[kMaxDevices];   // device address of `scratch` on each device

}  // namespace

namespace q1 {

q1_status noalloc_setup(int device, void* stream) {
  if (device < 0 || device >= kMaxDevices) return Q1_EINVAL;
  std::lock_guard<std::mutex> g(g_lock);
  if (g_scratch[device]) return Q1_OK;
  void* p = nullptr;
  if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return Q1_EDEVICE;
  // the merge set starts at zero (a fill kernel, no memset node)
  q1_status s = launch_zero(p, sizeof(MergeSet), stream);
  if (s == Q1_OK && hipStreamSynchronize((hipStream_t)stream) != hipSuccess) s = Q1_EDEVICE;
  if (s != Q1_OK) return s;
  g_scratch[device] = p;
  return Q1_OK;
}

q1_status noalloc_launch_scan(int device, q1_placement placement, q1_layout layout, bool fast, const ScanArgs& a,
                              const LaunchShape& shape, void* stream, const char** why) {
  if (device < 0 || device >= kMaxDevices) {
    *why = "device out of range";
    return Q1_EINVAL;
  }
  void* base = nullptr;
  {
    std::lock_guard<std::mutex> g(g_lock);
    base = g_scratch[device];
  }
  if (!base) {
    *why = "the scratch array of this device is not set up (q1_init does it)";
    return Q1_EDEVICE;
  }
  if (scan_workspace_bytes(placement, fast, shape) > kNoallocWorkspaceBytes) {
    *why = kNoallocRefused;
    return Q1_EINVAL;
  }
  void* workspace = static_cast<char*>(base) + sizeof(MergeSet);
  MergeSet* const set = static_cast<MergeSet*>(base);
  // A launch leaves the set clear if it had it to itself; block counts that two overlapping grids
  // left would make every later one fold its tables too early.  The fill kernel is recorded into a
  // caller's graph with the scan.  It costs 1.5 us of queued launches (512 blocks of 4,096 rows 13.1
  // -> 14.6 us) and 2.8 of a lone one.
  if (shape.blocks >= kSpreadMinBlocks && launch_zero(set, sizeof(MergeSet), stream) != Q1_OK) {
    *why = "clearing the merge tables failed";
    return Q1_EDEVICE;
  }
  const q1_status s = launch_scan(placement, layout, fast, a, shape, workspace, stream, set);
  if (s != Q1_OK) *why = "scan kernel launch failed";
  return s;
}

}  // namespace q1
