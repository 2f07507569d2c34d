// Entry of the queue of box edge lines (pc_direct.hip): a point of the cloud and
// which of its lines (0: first, 1: last column).  64 bits, for a cloud may have
// 2^30 points and more.
#pragma once

#include <cstdint>

namespace ohx {

constexpr int64_t line_entry(int64_t point, int side) { return point * 2 + side; }
constexpr int64_t line_point(int64_t e) { return e >> 1; }
constexpr int line_side(int64_t e) { return (int)(e & 1); }

}  // namespace ohx
