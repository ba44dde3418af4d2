// Where an upload is cut into the pieces and launches that it travels in.  Plain arithmetic, compiled for the session and for the
// tests.
#pragma once

#include <algorithm>
#include <cstddef>

namespace tfcc {

// The first launch is short so that the GPU starts early, the later ones long because each costs a launch, but no longer than the
// GPU has work for meanwhile; small inputs share one.  An encoder layer of 8 x 128 x 768 served, us, by the first and the
// longest chunk in KB: 256 and 1024 308, 256 and 512 297, 256 and 256 309, 384 and 768 294.
class UploadCut {
 public:
  // What a piece takes of the staging block and of its launch: whole lines, so that only the end of an input is no multiple of
  // one, and every piece begins on one.  (A piece at an odd address travels byte by byte: a mask of 301 floats in front of
  // 301 x 768 hidden states, counted as it is, did that to 533 of the 925 KB.)
  static constexpr size_t kLine = 64;
  static constexpr size_t padded(size_t bytes) { return (bytes + kLine - 1) / kLine * kLine; }

  // bytes of the next piece of an input that has `left`, with room for `room`, a multiple of kLine, in the staging block
  size_t next(size_t left, size_t room) const { return std::min(std::min(left, _chunk - _gathered), room); }
  // that piece is put down; true: the pieces so far are a launch
  bool put(size_t bytes) {
    _gathered += padded(bytes);
    return _gathered >= _chunk;
  }
  void launched() {
    _gathered = 0;
    _chunk = std::min(2 * _chunk, kLongest);
  }

 private:
  static constexpr size_t kFirst = size_t(384) << 10, kLongest = size_t(768) << 10;
  static_assert(kFirst % kLine == 0 && kLongest % kLine == 0, "whole lines");
  size_t _chunk = kFirst, _gathered = 0;
};

}  // namespace tfcc
