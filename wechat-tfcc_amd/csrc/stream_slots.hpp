// Scratch memory that belongs to one stream at a time: numbers for pieces of static device memory, or pieces that are asked
// for when a stream first needs one.  Launches on one stream run in order and share a piece; streams that may overlap get one
// each.  A graph may replay beside its stream's own work, so a stream that is being captured gets none, and neither does
// one that comes when all pieces are given out: the caller has a path without.
#pragma once

#include <map>
#include <mutex>
#include <utility>
#include <vector>

#include <hip/hip_runtime.h>

namespace tfcc_rocm {

// Whether the stream is one whose launches run in order and right away.
inline bool runs_in_order_now(hipStream_t stream) {
  if (stream == hipStreamPerThread) return false;  // one handle, a stream per thread
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &capturing) != hipSuccess) {  // the null stream beside a capture
    (void)hipGetLastError();
    return false;
  }
  return capturing == hipStreamCaptureStatusNone;
}

// Device memory, null if there is none: an allocation that breaks no capture that another thread has under way, and leaves no error.
inline void* allocate_beside_captures(size_t bytes) {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  const bool relaxed = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
  void* mem = nullptr;
  const bool made = relaxed && hipMalloc(&mem, bytes) == hipSuccess;
  if (relaxed) (void)hipThreadExchangeStreamCaptureMode(&mode);
  if (made) return mem;
  (void)hipGetLastError();
  return nullptr;
}

class StreamSlots {
 public:
  explicit StreamSlots(unsigned count) : count_(count) {}
  bool of(int dev, hipStream_t stream, unsigned* slot) {
    if (!runs_in_order_now(stream)) return false;
    std::lock_guard<std::mutex> lock(mutex_);
    const auto found = given_.find({dev, stream});
    if (found != given_.end()) {
      *slot = found->second;
      return true;
    }
    if (free_.empty() && next_ == count_) return false;
    if (free_.empty()) {
      *slot = next_++;
    } else {
      *slot = free_.back();
      free_.pop_back();
    }
    given_[{dev, stream}] = *slot;
    return true;
  }
  // the stream, which is idle, goes away
  void release(int dev, hipStream_t stream) {
    std::lock_guard<std::mutex> lock(mutex_);
    const auto found = given_.find({dev, stream});
    if (found == given_.end()) return;
    free_.push_back(found->second);
    given_.erase(found);
  }

 private:
  const unsigned count_;
  std::mutex mutex_;
  std::map<std::pair<int, hipStream_t>, unsigned> given_;
  std::vector<unsigned> free_;
  unsigned next_ = 0;
};

class StreamPieces {
 public:
  // prepare: makes a new piece ready on the stream it is for; 0 for success
  StreamPieces(size_t bytes, unsigned count, int (*prepare)(hipStream_t, void*)) : bytes_(bytes), count_(count), prepare_(prepare) {}
  void* of(int dev, hipStream_t stream) {
    if (!runs_in_order_now(stream)) return nullptr;
    std::lock_guard<std::mutex> lock(mutex_);
    const auto found = given_.find({dev, stream});
    if (found != given_.end()) return found->second;
    if (given_.size() == count_) return nullptr;
    void* const piece = allocate_beside_captures(bytes_);
    if (piece == nullptr) return nullptr;
    if (prepare_(stream, piece) != 0) {
      (void)hipFree(piece);
      return nullptr;
    }
    given_[{dev, stream}] = piece;
    return piece;
  }
  // the stream, which is idle, goes away
  void release(int dev, hipStream_t stream) {
    std::lock_guard<std::mutex> lock(mutex_);
    const auto found = given_.find({dev, stream});
    if (found == given_.end()) return;
    (void)hipFree(found->second);
    given_.erase(found);
  }

 private:
  const size_t bytes_;
  const unsigned count_;
  int (*const prepare_)(hipStream_t, void*);
  std::mutex mutex_;
  std::map<std::pair<int, hipStream_t>, void*> given_;
};

}  // namespace tfcc_rocm
