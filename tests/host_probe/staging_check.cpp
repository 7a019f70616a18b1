// The staging of the host-pointer entry points over a stand-in for the HIP
// runtime's memory calls, as a library of checks (see the Makefile).  Device
// memory is host memory; an error stays until hipGetLastError takes it, as in
// the runtime.
#include <stdint.h>
#include <stdlib.h>

#include <map>
#include <vector>

#include "staging.hpp"

namespace {
std::map<void*, size_t> g_device, g_pinned;
bool g_no_pinned = false;
hipError_t g_last = hipSuccess;

size_t total(const std::map<void*, size_t>& m) {
  size_t t = 0;
  for (const auto& kv : m) t += kv.second;
  return t;
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t b) {
  *p = malloc(b);
  g_device[*p] = b;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  g_device.erase(p);
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t b, unsigned) {
  if (g_no_pinned) return g_last = hipErrorOutOfMemory;
  *p = malloc(b);
  g_pinned[*p] = b;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  g_pinned.erase(p);
  free(p);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t b, hipMemcpyKind, hipStream_t) {
  memcpy(d, s, b);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError(void) {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}

// One staged call: an input, one that is also an output, an output and scratch,
// of `bytes` each; the "kernel" adds the input to both outputs.  0 when the
// arrays come back right.
static int call(pysa::DevBuf& stage, pysa::HostBuf& pin, size_t bytes) {
  std::vector<uint8_t> in(bytes), io(bytes), out(bytes, 9), want_io(bytes), want_out(bytes);
  for (size_t i = 0; i < bytes; ++i) {
    in[i] = (uint8_t)(i * 7 + 1), io[i] = (uint8_t)(i * 3);
    want_io[i] = (uint8_t)(in[i] + io[i]), want_out[i] = in[i];
  }
  pysa::Arena ar(stage, pin);
  const int a = ar.add(in.data(), nullptr, bytes), b = ar.add(io.data(), io.data(), bytes);
  const int c = ar.add(nullptr, out.data(), bytes);
  ar.add(nullptr, nullptr, bytes);
  if (ar.up(nullptr) != hipSuccess) return 1;
  for (size_t i = 0; i < bytes; ++i) {
    ar.at<uint8_t>(b)[i] += ar.at<uint8_t>(a)[i];
    ar.at<uint8_t>(c)[i] = ar.at<uint8_t>(a)[i];
  }
  if (ar.down(nullptr) != hipSuccess) return 2;
  return io == want_io && out == want_out ? 0 : 3;
}

// A call whose pinned memory is refused: copied without it, and no error left
// behind for the launch checks that follow.
int staging_without_pinned(size_t bytes) {
  pysa::DevBuf stage;
  pysa::HostBuf pin;
  g_no_pinned = true;
  g_last = hipSuccess;
  const int rc = call(stage, pin, bytes);
  g_no_pinned = false;
  return rc ? rc : hipGetLastError() != hipSuccess ? 4 : 0;
}

// Calls of these sizes one after another on one problem's buffers; returns the
// device bytes kept behind them, or minus a code.
long long staging_kept(const size_t* bytes, int count) {
  pysa::DevBuf stage;
  pysa::HostBuf pin;
  for (int k = 0; k < count; ++k)
    if (const int rc = call(stage, pin, bytes[k])) return -rc;
  return (long long)total(g_device);
}

// Bytes alive after the buffers of the calls above are gone.
long long staging_alive(void) { return (long long)(total(g_device) + total(g_pinned)); }
}
