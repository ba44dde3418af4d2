// Numbers for pieces of static device memory that belong to one stream at a time.  Launches on one stream run in order and
// share a piece; streams that may overlap get one each.  A graph may replay beside its stream's own work, so a stream that
// is being captured gets none, and neither does one that comes when all pieces are given out: the caller has a path without.
#pragma once

#include <map>
#include <mutex>
#include <utility>
#include <vector>

#include <hip/hip_runtime.h>

namespace tfcc_rocm {

class StreamSlots {
 public:
  explicit StreamSlots(unsigned count) : count_(count) {}
  bool of(int dev, hipStream_t stream, unsigned* slot) {
    if (stream == hipStreamPerThread) return false;  // one handle, a stream per thread
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &capturing) != hipSuccess) {  // the null stream beside a capture
      (void)hipGetLastError();
      return false;
    }
    if (capturing != hipStreamCaptureStatusNone) return false;
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

}  // namespace tfcc_rocm
