// Host-to-device copies out of pageable memory through a pinned staging area (left to the runtime, such a
// copy runs at a fraction of the link's rate: 4 against 27 GB/s measured for the 158 MB batch of the
// AlexNet shape, and the call waits for it).  Used by the ArrayLoader operator (reference
// cuda.cpp:592-598), by the batch prefetch and for reading tensors back.
#pragma once
#include <cstddef>
#include <cstring>
#include <mutex>

#include "mnv_hip.h"

namespace minerva {

// The pinned staging area of one worker stream, in two halves.  Copies of up to half of it are laid
// one behind the other into the active half and left in flight; when it is full the other half becomes the
// active one, once the copies that it held have left.  `mutex` guards everything.
struct StagingArea {
  static constexpr size_t kAlign = 256;
  std::mutex mutex;
  char* base = nullptr;
  size_t half = 0;
  size_t used = 0;             // of the active half
  int active = 0;
  void* left[2] = {};          // events behind a half's last copy
  bool in_flight[2] = {};      // the event is recorded and not yet waited for
  ~StagingArea() {
    for (void* e : left)
      if (e) mnv_event_destroy(e);
  }
  // `bytes` <= half of it that no copy in flight touches; the caller's copy goes to `stream`, in order.
  int Take(size_t bytes, void* stream, char** at) {
    if (used + bytes > half) {
      int rc = MNV_OK;
      if (!left[active]) rc = mnv_event_create_ordering(&left[active]);
      if (rc == MNV_OK) rc = mnv_event_record(left[active], stream);
      if (rc != MNV_OK) return rc;
      in_flight[active] = true;
      active ^= 1;
      if (in_flight[active]) rc = mnv_event_sync(left[active]);
      if (rc != MNV_OK) return rc;
      in_flight[active] = false;
      used = 0;
    }
    *at = base + active * half + used;
    used += (bytes + kAlign - 1) / kAlign * kAlign;
    return MNV_OK;
  }
  // The stream has been synchronised: nothing is in flight.
  void Drained() {
    used = 0;
    in_flight[0] = in_flight[1] = false;
  }
};

// The host buffer may go away when this returns.  Up to half of the staging area: the copy is left in flight
// on `stream`, and the caller queues the step behind it (four minibatches of 256 through the MLP of 784-256-10 and its
// parameters read back: 967 -> 625 us without the waits, through the MNIST CNN 1437 -> 1069).  Larger ones go through the two halves in
// turn, the CPU filling one while the DMA engine drains the other, and are complete on return.
inline int StagedHostToDevice(void* dst_device, const void* src_host, size_t bytes, void* stream, StagingArea* area) {
  const char* src = static_cast<const char*>(src_host);
  char* dst = static_cast<char*>(dst_device);
  if (!area || !area->half) {
    int rc = mnv_memcpy_h2d(dst, src, bytes, stream);
    const int rs = mnv_stream_sync(stream);
    return rc != MNV_OK ? rc : rs;
  }
  std::lock_guard<std::mutex> lock(area->mutex);
  const size_t half = area->half;
  if (bytes <= half) {
    char* at = nullptr;
    int rc = area->Take(bytes, stream, &at);
    if (rc != MNV_OK) return rc;
    std::memcpy(at, src, bytes);
    return mnv_memcpy_h2d(dst, at, bytes, stream);
  }
  int rc = mnv_stream_sync(stream);  // what the area still held
  area->Drained();
  void* drained[2] = {nullptr, nullptr};
  if (rc == MNV_OK) rc = mnv_event_create_ordering(&drained[0]);
  if (rc == MNV_OK) rc = mnv_event_create_ordering(&drained[1]);
  size_t off = 0;
  for (int i = 0; off < bytes && rc == MNV_OK; ++i, off += half) {
    const int b = i & 1;
    const size_t n = bytes - off < half ? bytes - off : half;
    if (i >= 2) rc = mnv_event_sync(drained[b]);  // this half has left for the device
    if (rc != MNV_OK) break;
    std::memcpy(area->base + b * half, src + off, n);
    rc = mnv_memcpy_h2d(dst + off, area->base + b * half, n, stream);
    if (rc == MNV_OK) rc = mnv_event_record(drained[b], stream);
  }
  const int rs = mnv_stream_sync(stream);
  if (drained[0]) mnv_event_destroy(drained[0]);
  if (drained[1]) mnv_event_destroy(drained[1]);
  return rc != MNV_OK ? rc : rs;
}

}  // namespace minerva
