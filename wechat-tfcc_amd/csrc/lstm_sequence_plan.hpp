// Which LSTM sequences run in one launch, and what memory they need.  Plain functions of integers, compiled for the
// launcher and for a host-side test.
#pragma once

#include <cstddef>

namespace tfcc_rocm {
namespace lstm_plan {

constexpr unsigned kUnitsPerWorkgroup = 8;  // one wavefront each

inline unsigned padded_units(unsigned units) { return units <= 256 ? 256 : units <= 512 ? 512 : 1024; }

inline unsigned workgroups(unsigned units, unsigned directions) {
  return (units + kUnitsPerWorkgroup - 1) / kUnitsPerWorkgroup * directions;
}

// Bytes of the workspace; 0: not a sequence for one launch.  Its workgroups wait for one another, so each needs a CU: 1024
// units in both directions fill the 256 of a whole GPU, a part of a partitioned one has room for fewer.
inline size_t workspace_bytes(unsigned batch, unsigned units, unsigned directions, int cus) {
  if (batch < 1 || batch > 16 || units < 1 || units > 1024 || directions < 1 || directions > 2) return 0;
  if (cus < 0 || workgroups(units, directions) > (unsigned)cus) return 0;
  return (size_t)2 * directions * batch * padded_units(units) * 8 + 64;
}

constexpr unsigned kXcds = 8, kCusOfXcd = 32;  // of a whole GPU; workgroups are dispatched to the XCDs in turn

// Rows of the batch that the workgroups of one XCD take, where a direction's state kernel fits the registers of one; 0: it does
// not, or the GPU is a part of one.  Beyond 768 units it would take all of them.
inline unsigned rows_of_xcd(unsigned batch, unsigned units, unsigned directions, int cus) {
  if (units > 768 || cus < (int)(kXcds * kCusOfXcd)) return 0;
  const unsigned groups = kXcds / directions;
  return (batch + groups - 1) / groups;
}

}  // namespace lstm_plan
}  // namespace tfcc_rocm
