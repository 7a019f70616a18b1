// Buffers that a problem keeps between calls, and the staging of the
// host-pointer entry points.
#pragma once
#include <hip/hip_runtime.h>
#include <string.h>

#include <vector>

namespace pysa {

struct DevBuf {
  void* p = nullptr;
  size_t bytes = 0;
  hipError_t ensure(size_t b) {
    if (b <= bytes) return hipSuccess;
    if (p) (void)hipFree(p);
    p = nullptr;
    bytes = 0;
    hipError_t e = hipMalloc(&p, b ? b : 1);
    if (e == hipSuccess) bytes = b;
    return e;
  }
  ~DevBuf() {
    if (p) (void)hipFree(p);
  }
};

// Pinned host memory.
struct HostBuf {
  void* p = nullptr;
  size_t bytes = 0;
  hipError_t ensure(size_t b) {
    if (b <= bytes) return hipSuccess;
    if (p) (void)hipHostFree(p);
    p = nullptr;
    bytes = 0;
    hipError_t e = hipHostMalloc(&p, b, hipHostMallocDefault);
    if (e == hipSuccess) bytes = b;
    return e;
  }
  ~HostBuf() {
    if (p) (void)hipHostFree(p);
  }
};

// The device arrays of one host-pointer call in one block of memory that the
// problem keeps for the next call (up to kKeep bytes; a larger block lives for
// the call).  Arrays are added in the order inputs, inputs that are also
// outputs, outputs, scratch, so the copies in and out cover one range each:
// below kPin bytes each is a single copy through pinned memory.  (Before, a call
// made and freed a buffer per array and copied each by itself: about 1 ms a
// call, of which a short run of a small problem is a fraction.)
struct Arena {
  // kKeep: a program with many problems pays it for each.  Above it the copies
  // of ordinary memory take milliseconds, beside which one allocation is little
  // (energies of 50 MB of states 11.0 ms either way, of 215 MB 46.5 -> 46.9).
  static constexpr size_t kKeep = size_t(32) << 20, kPin = size_t(1) << 20;
  struct Item {
    const void* src;
    void* dst;
    size_t bytes, off;
  };
  std::vector<Item> items;
  size_t total = 0;
  DevBuf& stage;
  HostBuf& pin;
  DevBuf own;
  char* base = nullptr;
  Arena(DevBuf& stage_, HostBuf& pin_) : stage(stage_), pin(pin_) { items.reserve(16); }
  int add(const void* src, void* dst, size_t bytes) {
    items.push_back({src, dst, bytes, total});
    total += (bytes + 255) & ~size_t(255);
    return (int)items.size() - 1;
  }
  template <typename T>
  T* at(int i) const {
    return reinterpret_cast<T*>(base + items[i].off);
  }
  // Whether pinned memory is there for this call's copies.  A refused
  // allocation is no error of the call, so it leaves none behind for the launch
  // checks to find.
  bool pinned() {
    if (pin.ensure(kPin) == hipSuccess) return true;
    (void)hipGetLastError();
    return false;
  }
  // Allocates and copies the inputs in.
  hipError_t up(hipStream_t st) {
    DevBuf& b = total <= kKeep ? stage : own;
    hipError_t e = b.ensure(total ? total : 1);
    if (e != hipSuccess) return e;
    base = (char*)b.p;
    size_t end = 0;
    for (const Item& it : items)
      if (it.src) end = it.off + it.bytes;
    if (end == 0) return hipSuccess;
    if (end <= kPin && pinned()) {
      for (const Item& it : items)
        if (it.src) memcpy((char*)pin.p + it.off, it.src, it.bytes);
      return hipMemcpyAsync(base, pin.p, end, hipMemcpyHostToDevice, st);
    }
    for (const Item& it : items)
      if (it.src && it.bytes) {
        e = hipMemcpyAsync(base + it.off, it.src, it.bytes, hipMemcpyHostToDevice, st);
        if (e != hipSuccess) return e;
      }
    return hipSuccess;
  }
  // Copies the outputs back and waits for them.
  hipError_t down(hipStream_t st) {
    size_t lo = total, hi = 0;
    for (const Item& it : items)
      if (it.dst) {
        lo = it.off < lo ? it.off : lo;
        hi = it.off + it.bytes;
      }
    if (hi <= lo) return hipStreamSynchronize(st);
    hipError_t e;
    if (hi - lo <= kPin && pinned()) {
      e = hipMemcpyAsync(pin.p, base + lo, hi - lo, hipMemcpyDeviceToHost, st);
      if (e == hipSuccess) e = hipStreamSynchronize(st);
      if (e != hipSuccess) return e;
      for (const Item& it : items)
        if (it.dst) memcpy(it.dst, (const char*)pin.p + (it.off - lo), it.bytes);
      return hipSuccess;
    }
    for (const Item& it : items)
      if (it.dst && it.bytes) {
        e = hipMemcpyAsync(it.dst, base + it.off, it.bytes, hipMemcpyDeviceToHost, st);
        if (e != hipSuccess) return e;
      }
    return hipStreamSynchronize(st);
  }
};

}  // namespace pysa
