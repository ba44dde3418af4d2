// The words by which the workgroups of a one-launch quantize tell one another their minimum and maximum.  Plain functions of
// integers, compiled for the kernel and for the tests.
#pragma once

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

}  // namespace quantize_exchange
}  // namespace tfcc_rocm
