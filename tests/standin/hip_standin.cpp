#include "hip_standin.h"

#include <hip/hip_runtime.h>

#include <chrono>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>

#include "../../tpchq01_gpu_amd/csrc/q1_kernels.h"

namespace {

std::recursive_mutex& lock() {
  static std::recursive_mutex m;
  return m;
}
#define GUARD std::lock_guard<std::recursive_mutex> guard(lock())

std::map<const void*, std::string>& kernels() {
  static std::map<const void*, std::string> m;
  return m;
}
std::map<const void*, std::pair<void*, size_t>>& variables() {
  static std::map<const void*, std::pair<void*, size_t>> m;
  return m;
}
std::map<const char*, uint64_t>& pinned() {
  static std::map<const char*, uint64_t> m;
  return m;
}
std::map<void*, uint64_t>& device() {
  static std::map<void*, uint64_t> m;
  return m;
}
// The pinned range that holds p, or end().
std::map<const char*, uint64_t>::iterator range_of(const void* p) {
  auto it = pinned().upper_bound((const char*)p);
  if (it == pinned().begin()) return pinned().end();
  --it;
  return (const char*)p < it->first + it->second ? it : pinned().end();
}

void tell(void* stream, uint64_t* word, uint64_t value) {
  const standin::State& s = standin::state();
  if (s.silent) return;
  if (s.late_stream == stream && s.late_us) {
    std::thread([word, value, us = s.late_us] {
      std::this_thread::sleep_for(std::chrono::microseconds(us));
      __atomic_store_n(word, value, __ATOMIC_RELEASE);
    }).detach();
    return;
  }
  __atomic_store_n(word, value, __ATOMIC_RELEASE);
}

thread_local struct {
  dim3 grid, block;
  size_t lds = 0;
  hipStream_t stream = nullptr;
} pushed;

}  // namespace

namespace standin {
State& state() {
  static State s;
  return s;
}
void pin(const void* base, uint64_t bytes) {
  GUARD;
  pinned()[(const char*)base] = bytes;
}
}  // namespace standin

extern "C" {

void** __hipRegisterFatBinary(const void*) {
  static void* handle = nullptr;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  kernels()[host] = name;
}
void __hipRegisterVar(void**, void* var, char*, char*, int, size_t size, int, int) {
  variables()[var] = {std::calloc(1, size), size};
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream) {
  pushed = {grid, block, lds, stream};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream) {
  *grid = pushed.grid;
  *block = pushed.block;
  *lds = pushed.lds;
  *stream = pushed.stream;
  return hipSuccess;
}

hipError_t hipLaunchKernel(const void* fn, dim3 grid, dim3 block, void** args, size_t, hipStream_t stream) {
  GUARD;
  standin::State& s = standin::state();
  standin::Launch l;
  l.kernel = kernels().at(fn);
  l.grid = grid.x;
  l.block = block.x;
  l.stream = (void*)stream;
  l.captured = s.capturing && s.capturing == (void*)stream;
  const bool scan = l.is("scan_fast") || l.is("scan_any") || l.is("scan_direct");
  if (scan) l.scan_args.assign((char*)args[0], (char*)args[0] + sizeof(q1::ScanArgs));
  if (l.is("scan_fast")) l.workspace = *(void**)args[2];
  if (l.is("fetch_columns")) l.fetch_args.assign((char*)args[0], (char*)args[0] + sizeof(q1::FetchArgs));
  s.launches.push_back(l);
  if (l.captured) return hipSuccess;
  if (scan) {
    const q1::ScanArgs& a = *(const q1::ScanArgs*)args[0];
    if (a.host)
      for (uint32_t b = 0; b < (l.is("scan_direct") ? grid.x : 1); b++) tell(stream, &a.host[b].sequence, a.sequence);
    else if (a.done)
      tell(stream, a.done, a.sequence);
  } else if (l.is("zero_words")) {
    std::memset(*(void**)args[0], 0, *(uint64_t*)args[1] * 8);
  } else if (l.is("domain_check")) {
    const q1::Completion& c = *(const q1::Completion*)args[2];
    tell(stream, &c.host->sequence, c.sequence);
  } else if (l.is("report_end")) {
    tell(stream, &(*(q1::HostResult**)args[0])->sequence, *(uint64_t*)args[1]);
  } else if (l.is("batch_scan")) {
    tell(stream, &(*(q1::BatchDone**)args[5])->sequence, (*(const q1::BatchHeader**)args[0])->sequence);
  }
  return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t bytes) {
  GUARD;
  standin::State& s = standin::state();
  *p = nullptr;
  if (s.device_bytes + bytes > s.budget) return hipErrorOutOfMemory;
  *p = std::calloc(1, bytes ? bytes : 1);
  device()[*p] = bytes;
  s.device_bytes += bytes;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  GUARD;
  if (!p) return hipSuccess;
  standin::State& s = standin::state();
  s.frees++;
  s.device_bytes -= device().at(p);
  device().erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  GUARD;
  *p = std::calloc(1, bytes ? bytes : 1);
  pinned()[(const char*)*p] = bytes;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  GUARD;
  pinned().erase((const char*)p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) {
  *d = h;
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  GUARD;
  std::memset((void*)a, 0, sizeof(*a));
  if (range_of(p) == pinned().end()) return hipErrorInvalidValue;
  a->type = hipMemoryTypeHost;
  a->devicePointer = a->hostPointer = (void*)p;
  return hipSuccess;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t* base, size_t* size, hipDeviceptr_t p) {
  GUARD;
  auto it = range_of(p);
  if (it == pinned().end()) return hipErrorNotFound;
  *base = (hipDeviceptr_t)it->first;
  *size = it->second;
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* free_bytes, size_t* total) {
  *free_bytes = *total = 288ull << 30;
  return hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n) {
  std::memset(p, v, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind kind, hipStream_t) {
  GUARD;
  standin::state().copies.push_back({src, n, kind == hipMemcpyHostToDevice});
  std::memcpy(dst, src, n);
  return hipSuccess;
}
hipError_t hipMemcpy(void* dst, const void* src, size_t n, hipMemcpyKind kind) {
  return hipMemcpyAsync(dst, src, n, kind, nullptr);
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = (hipStream_t)std::malloc(16);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  std::free((void*)s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t stream) {
  int late = 0;
  {
    GUARD;
    standin::State& s = standin::state();
    s.stream_waits++;
    if (s.late_stream == (void*)stream) late = s.late_us;
  }
  if (late) std::this_thread::sleep_for(std::chrono::microseconds(2 * late));
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
  GUARD;
  standin::state().device_waits++;
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* status) {
  GUARD;
  const void* c = standin::state().capturing;
  *status = c && c == (void*)s ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = (hipEvent_t)std::malloc(16);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) {
  std::free((void*)e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 0;
  return hipSuccess;
}

hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceFlags(unsigned* flags) {
  *flags = standin::state().device_flags;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset((void*)p, 0, sizeof(*p));
  std::strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  p->warpSize = 64;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  *v = 100000;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 4;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* symbol) {
  *p = variables().at(symbol).first;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }

}  // extern "C"
