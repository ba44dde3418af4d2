// A quantize in one launch whose workgroups tell one another their minimum and maximum: the words by which they do, and how
// many workgroups there are.  Plain functions of integers, compiled for the kernel, its launch and the tests.
#pragma once

#include <mutex>

namespace tfcc_rocm {
namespace quantize_exchange {

// A word is half of a value, 16 bits, and the number of the call in the other 48, so that a reader knows from a word alone
// whether it is this call's.  A call has a number that no other one of the process has for 2^48 calls, 44 years at 5 us each (32
// bits, with a whole value to a word, are used up in six hours).  Numbers begin with 1: memory that nobody has written holds 0.
constexpr unsigned kWords = 4;  // of a workgroup: its minimum, its maximum, the low half first
constexpr unsigned long long kNumbers = 1ull << 48;

constexpr unsigned long long number_of(unsigned long long calls) { return calls % (kNumbers - 1) + 1; }
constexpr unsigned long long word_of(unsigned long long number, unsigned value, bool high) {
  return number << 16 | (high ? value >> 16 : value & 0xffffu);
}
constexpr bool belongs_to(unsigned long long word, unsigned long long number) { return word >> 16 == number; }
constexpr unsigned value_of(unsigned long long low, unsigned long long high) {
  return (unsigned)(low & 0xffffu) | (unsigned)(high & 0xffffu) << 16;
}

constexpr unsigned kWorkgroups = 256;  // at most
constexpr unsigned kPiece = 4096;      // elements that 1024 threads read with a 16-byte load each

constexpr unsigned long long workgroups(unsigned long long total, unsigned quads) {
  return (total + (unsigned long long)kPiece * quads - 1) / ((unsigned long long)kPiece * quads);
}
// Loads of a thread: one, two, four or eight, as few as leave a CU of this GPU for every workgroup (as many workgroups as there
// may be: the loads of a thread are all on their way at once, and the words are read side by side); 0: not even with eight.  A
// workgroup that finds no CU keeps the others waiting, which on a part of a partitioned GPU would be every call.
constexpr unsigned quads_of(unsigned long long total, int cus) {
  const unsigned long long room = cus <= 0 ? 0 : (unsigned)cus < kWorkgroups ? (unsigned)cus : kWorkgroups;
  for (unsigned quads = 1; quads <= 8; quads *= 2)
    if (workgroups(total, quads) <= room) return quads;
  return 0;
}

// From how many streams in turn calls may come with so many loads to a thread.  The launches of more streams than that find no
// CU for all of their workgroups, and those of each wait for one another until they give up.  us a call, streams side by
// side, in one launch / in two: 2 M elements on 4 streams 6.3 / 9.1, on 8 10.2 / 9.0; 4 M on 2 8.5 / 10.1, on 3 17.0 / 9.8, on 8
// 19.5 / 9.3; 8 M on 2 14.7 / 15.4, on 3 24.7 / 14.5, on 8 28.2 / 14.8.  One load to a thread is better on any number of streams.
constexpr unsigned streams_of(unsigned quads) { return quads <= 1 ? ~0u : quads == 2 ? 4 : 2; }

// The streams of a device's last calls.
class LastStreams {
 public:
  // another call on this stream; of how many streams the last kCalls calls are, this one among them
  unsigned with(const void* stream) {
    std::lock_guard<std::mutex> lock(mutex_);
    last_[next_++ % kCalls] = stream;
    const unsigned known = next_ < kCalls ? next_ : kCalls;
    if (next_ == 2 * kCalls) next_ = kCalls;
    unsigned streams = 0;
    for (unsigned i = 0; i < known; ++i) {
      bool again = false;
      for (unsigned j = 0; j < i; ++j) again = again || last_[j] == last_[i];
      streams += again ? 0 : 1;
    }
    return streams;
  }

 private:
  static constexpr unsigned kCalls = 8;
  std::mutex mutex_;
  const void* last_[kCalls] = {};
  unsigned next_ = 0;
};

}  // namespace quantize_exchange
}  // namespace tfcc_rocm
