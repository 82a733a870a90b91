// fake_hip.hpp - the HIP runtime calls of libmtg.so on host memory, for tests of its
// host code without a GPU. A test program that includes this (once) defines the symbols
// itself, so the library's references resolve to them: device memory is host memory,
// copies and fills happen at the call, streams and events order nothing, and a kernel
// launch is recorded by name and runs nothing. A failure that a test asks for leaves a
// last error as the runtime does.
#pragma once

#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <vector>

namespace fake {

enum { kOk = 0, kInvalid = 1, kOutOfMemory = 2 };
struct Dim3 {
  uint32_t x, y, z;
};
struct Launch {
  std::string kernel;
  Dim3 grid;
  size_t lds;
  void* stream;
};
struct Copy {
  void* dst;
  const void* src;
  size_t bytes;
  int kind;  // 1 host to device, 2 device to host
  void* stream;
};
struct State {
  std::map<const void*, std::string> kernels;   // host stub -> mangled name
  std::map<const void*, int> lds_limit;         // hipFuncSetAttribute
  std::vector<Launch> launches;
  std::vector<Copy> copies;
  std::function<bool(size_t)> malloc_fails;     // by size
  std::function<bool(const std::string&)> launch_fails, attribute_fails;
  std::function<void()> attribute_set;          // after an attribute is set
  int waits = 0, stream_syncs = 0;              // hipStreamWaitEvent, hipStreamSynchronize
  int last_error = kOk;
  uintptr_t handles = 0;
};
inline State& state() {  // the library registers its kernels before main()
  static State s;
  return s;
}
inline int fail(int e) { return state().last_error = e; }
inline void* handle() { return (void*)(++state().handles * 16); }
inline std::string name_of(const void* f) {
  auto it = state().kernels.find(f);
  return it == state().kernels.end() ? "?" : it->second;
}
// launches of kernels whose mangled name contains `part`
inline int count(const char* part) {
  int n = 0;
  for (const Launch& l : state().launches) n += l.kernel.find(part) != std::string::npos;
  return n;
}

}  // namespace fake

extern "C" {
void** __hipRegisterFatBinary(const void*) { return (void**)fake::handle(); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* stub, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  fake::state().kernels[stub] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
static fake::Dim3 g_grid, g_block;
static size_t g_lds;
static void* g_stream;
int __hipPushCallConfiguration(fake::Dim3 grid, fake::Dim3 block, size_t lds, void* stream) {
  g_grid = grid, g_block = block, g_lds = lds, g_stream = stream;
  return fake::kOk;
}
int __hipPopCallConfiguration(fake::Dim3* grid, fake::Dim3* block, size_t* lds, void** stream) {
  *grid = g_grid, *block = g_block, *lds = g_lds, *stream = g_stream;
  return fake::kOk;
}
int hipLaunchKernel(const void* f, fake::Dim3 grid, fake::Dim3, void**, size_t lds, void* stream) {
  fake::State& s = fake::state();
  const std::string name = fake::name_of(f);
  const int limit = s.lds_limit.count(f) ? s.lds_limit[f] : 64 * 1024;
  if ((int)lds > limit || (s.launch_fails && s.launch_fails(name))) return fake::fail(fake::kInvalid);
  s.launches.push_back({name, grid, lds, stream});
  return fake::kOk;
}
int hipFuncSetAttribute(const void* f, int, int value) {
  fake::State& s = fake::state();
  if (s.attribute_fails && s.attribute_fails(fake::name_of(f))) return fake::fail(fake::kInvalid);
  s.lds_limit[f] = value;
  if (s.attribute_set) s.attribute_set();
  return fake::kOk;
}
int hipGetLastError() {
  const int e = fake::state().last_error;
  fake::state().last_error = fake::kOk;
  return e;
}
const char* hipGetErrorString(int) { return "fake error"; }
int hipGetDevice(int* d) { return *d = 0; }
int hipDeviceGetAttribute(int* v, int, int) {
  *v = 256;
  return fake::kOk;
}
int hipDeviceSynchronize() { return fake::kOk; }

int hipMalloc(void** p, size_t bytes) {
  *p = nullptr;
  if (fake::state().malloc_fails && fake::state().malloc_fails(bytes)) return fake::fail(fake::kOutOfMemory);
  *p = std::aligned_alloc(256, (bytes + 255) / 256 * 256);
  return *p ? fake::kOk : fake::fail(fake::kOutOfMemory);
}
int hipFree(void* p) {
  std::free(p);
  return fake::kOk;
}
int hipHostMalloc(void** p, size_t bytes, unsigned) { return hipMalloc(p, bytes); }
int hipHostFree(void* p) { return hipFree(p); }
int hipHostGetDevicePointer(void** d, void* h, unsigned) {
  *d = h;
  return fake::kOk;
}
int hipGetSymbolAddress(void**, const void*) { return fake::fail(fake::kInvalid); }
int hipMemset(void* p, int v, size_t n) {
  std::memset(p, v, n);
  return fake::kOk;
}
int hipMemsetAsync(void* p, int v, size_t n, void*) { return hipMemset(p, v, n); }
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* stream) {
  fake::state().copies.push_back({d, s, n, kind, stream});
  std::memmove(d, s, n);
  return fake::kOk;
}
int hipMemcpy(void* d, const void* s, size_t n, int kind) { return hipMemcpyAsync(d, s, n, kind, nullptr); }

int hipStreamCreateWithFlags(void** s, unsigned) {
  *s = fake::handle();
  return fake::kOk;
}
int hipStreamDestroy(void*) { return fake::kOk; }
int hipStreamSynchronize(void*) {
  ++fake::state().stream_syncs;
  return fake::kOk;
}
int hipStreamWaitEvent(void*, void*, unsigned) {
  ++fake::state().waits;
  return fake::kOk;
}
int hipEventCreateWithFlags(void** e, unsigned) {
  *e = fake::handle();
  return fake::kOk;
}
int hipEventCreate(void** e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void*) { return fake::kOk; }
int hipEventRecord(void*, void*) { return fake::kOk; }
int hipEventSynchronize(void*) { return fake::kOk; }
int hipEventElapsedTime(float* ms, void*, void*) {
  *ms = 0.0f;
  return fake::kOk;
}
}
