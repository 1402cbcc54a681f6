// Kernel launches by the function's own handle.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <tuple>

#include "common.hpp"

namespace LLMHIP_NS {

// The handle of a kernel on the stream's device, or null where that is not the current one (handles are asked for on the current
// device).  A small table per thread; an entry that another kernel needs is asked for again.
inline hipFunction_t function_of(const void *kern, hipStream_t stream) {
  struct Entry {
    const void *kern;
    int dev;
    hipFunction_t function;
  };
  constexpr unsigned kEntries = 256;
  static thread_local Entry table[kEntries] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return nullptr;
  hipDevice_t of_stream = dev;
  if (stream != nullptr && hipStreamGetDevice(stream, &of_stream) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  if (of_stream != dev) return nullptr;
  Entry &e = table[((unsigned)(reinterpret_cast<uintptr_t>(kern) >> 3) * 0x9E3779B1u >> 24) % kEntries];
  if (e.kern == kern && e.dev == dev) return e.function;
  hipFunction_t f;
  if (hipGetFuncBySymbol(&f, kern) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  e = {kern, dev, f};
  return f;
}

// hipLaunchKernelGGL looks the kernel up behind a lock, passes the launch's shape through a stack of its own, and tells how it went in
// hipGetLastError only: 2.91 us of the host a launch, 2.70 so.
template <typename... P, typename... A>
inline hipError_t launch(void (*kern)(P...), dim3 grid, unsigned threads, size_t lds_bytes, hipStream_t stream, const A &...given) {
  std::tuple<P...> args(given...);
  return std::apply(
      [&](P &...p) {
        void *at[] = {const_cast<void *>(static_cast<const void *>(&p))...};
        const void *const host = reinterpret_cast<const void *>(kern);
        const hipFunction_t f = function_of(host, stream);
        const hipError_t e = f ? hipModuleLaunchKernel(f, grid.x, grid.y, grid.z, threads, 1, 1, (unsigned)lds_bytes, stream, at, nullptr)
                               : hipLaunchKernel(host, grid, dim3(threads), at, lds_bytes, stream);
        if (e != hipSuccess) (void)hipGetLastError();  // told here: not for the next call to report
        return e;
      },
      args);
}

}  // namespace LLMHIP_NS
