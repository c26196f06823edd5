// How long rows are reduced, shared by the eager reductions and the fused row
// kernels, whose results must agree bit for bit.  Host code, no HIP includes.
#pragma once

#include <algorithm>
#include <cstdint>

namespace lmp_hip {

// Rows of at least this many values take a workgroup of kRowLanes lanes (or
// several) each, shorter ones a wave or less.
constexpr uint64_t kLongRow = 2048;
constexpr int kRowLanes = 256;

// Workgroups per long row of `units` (16 bytes, or one value): enough to fill
// the chip twice over, more than one only when the rows alone cannot.
inline uint64_t row_parts(uint64_t cus, uint64_t rows, uint64_t units) {
  const uint64_t target = cus * 8;
  uint64_t parts = 1;
  if (rows < target)
    parts = std::min((target + rows - 1) / rows, std::max<uint64_t>(1, units / 1024));
  const uint64_t seg = (units + parts - 1) / parts;
  return (units + seg - 1) / seg;
}

}  // namespace lmp_hip
