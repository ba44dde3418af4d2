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

}  // namespace lstm_plan
}  // namespace tfcc_rocm
