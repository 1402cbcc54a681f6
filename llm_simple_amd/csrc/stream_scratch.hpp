// Scratch that the library keeps for a stream between calls.  Host code without HIP, so that the host tests can run it on devices of their own.
#pragma once
#include <stddef.h>

#include <map>
#include <utility>
#include <vector>

#include "../../include/llmhip.h"

namespace llmhip {

// A buffer that only grows.  One that has become too small is not freed when a larger one replaces it: launches already
// queued, and HIP graphs captured earlier, keep their pointer valid.  Retired buffers go with the stream's others.
struct StreamScratch {
  void *ptr = nullptr;
  size_t bytes = 0;
  std::vector<void *> retired;
};

// One buffer per stream and device: the null stream is the same handle on every device.
// Runtime, with status 0 for success: device_of(stream); allocate(device, &ptr, bytes), also while another stream is captured; release(ptr);
// capturing(stream); wait_stream(device, stream); wait_device(device).  The caller holds a lock over each call, and over the launches that use the buffer.
template <typename Runtime> class ScratchTable {
 public:
  // The stream's scratch for a call whose fastest form takes `need` bytes and that is to run with no less than least().
  // Where the buffer cannot grow -- its stream is under capture, which must not allocate, or the device is full -- the
  // call gets what there is; only if that is less than least() is it refused (LLMHIP_ERR_WORKSPACE under capture:
  // warm the stream up with its largest shape first).  Sizes are powers of two from 4 MiB on (the exact size where the
  // device has no room for that), so that the replaced buffers together are smaller than the one in use.
  template <typename Least> int get(void *stream, size_t need, Least least, StreamScratch **out) {
    const int device = Runtime::device_of(stream);
    StreamScratch &s = table_[{device, stream}];
    *out = &s;
    if (s.bytes >= need) return LLMHIP_OK;
    const size_t fewest = least();
    int refused = LLMHIP_ERR_WORKSPACE;
    if (!Runtime::capturing(stream)) {
      size_t grown = (size_t)4 << 20;
      while (grown < need) grown *= 2;
      const size_t wanted[] = {grown, need, fewest};
      for (size_t want : wanted) {
        if (want <= s.bytes) continue;
        void *fresh = nullptr;
        const int e = Runtime::allocate(device, &fresh, want);
        if (e != 0) {
          refused = e;
          continue;
        }
        if (s.ptr) s.retired.push_back(s.ptr);
        s.ptr = fresh;
        s.bytes = want;
        return LLMHIP_OK;
      }
    }
    return s.bytes >= fewest ? LLMHIP_OK : refused;
  }

  // All buffers of a stream that is about to be destroyed
  void drop(void *stream) {
    for (auto it = table_.begin(); it != table_.end();) {
      if (it->first.second != stream) {
        ++it;
        continue;
      }
      if (it->second.ptr) Runtime::wait_stream(it->first.first, stream);
      (void)free_all(it->second);
      it = table_.erase(it);
    }
  }

  // All buffers there are; the last error (queued launches may still use them: each device is waited for)
  int release() {
    int rc = 0, waited = -1;
    for (auto &entry : table_) {  // (in the order of devices)
      if (entry.first.first == waited) continue;
      waited = entry.first.first;
      if (const int e = Runtime::wait_device(waited)) rc = e;
    }
    for (auto &entry : table_)
      if (const int e = free_all(entry.second)) rc = e;
    table_.clear();
    return rc;
  }

 private:
  static int free_all(StreamScratch &s) {
    const int rc = s.ptr ? Runtime::release(s.ptr) : 0;
    for (void *old : s.retired) (void)Runtime::release(old);
    return rc;
  }
  std::map<std::pair<int, void *>, StreamScratch> table_;
};

}  // namespace llmhip
