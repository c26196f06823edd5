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

// Units of 16 bytes of fp32 values, or anything else: units of one value, of two
// float64, ...  They differ in how a row is cut and its sums meet.
enum class RowUnits { Float4, Other };

// Workgroups per long row of `units`: enough to fill the chip twice over, more
// than one only when the rows alone cannot, and a part long enough to pay for the
// second launch.  A workgroup's lanes take four units at a time: four rounds a
// part of float4s, 16 (64 units a lane, all that a fused row holds) of others, whose
// second launch costs more than it saves below that ([256, 3001] fp32 5.8 us in
// two parts, 4.1 whole; [64, 6000] float64 6.1 and 4.6).
inline uint64_t row_parts(uint64_t cus, uint64_t rows, uint64_t units, RowUnits kind) {
  const uint64_t target = cus * 8, least = kind == RowUnits::Float4 ? 1024 : 64 * kRowLanes;
  uint64_t parts = 1;
  if (rows < target)
    parts = std::min((target + rows - 1) / rows, std::max<uint64_t>(1, units / least));
  const uint64_t seg = (units + parts - 1) / parts;
  return (units + seg - 1) / seg;
}

}  // namespace lmp_hip
