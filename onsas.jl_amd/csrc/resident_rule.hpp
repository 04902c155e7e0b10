// resident_rule.hpp -- which launches of workgroups that wait for one another may be
// made (host code): all of them have to be resident at once, so the grid is held to what
// the device says that its CUs take of the kernel (registers, LDS, waves).
#pragma once

#include <algorithm>
#include <cstdint>

namespace onsas {

constexpr int kXcdCus = 32;  // CUs of an XCD
// Most workgroups of a launch on a CU of one XCD; more have not been measured there.
constexpr int kXcdBlocks = 3;

// a grid of a kernel of which a CU takes `blocks`, on the whole device of `cus` CUs
inline bool fits_device(int64_t grid, int blocks, int cus) { return grid <= (int64_t)blocks * cus; }
// ... and on one XCD of it
inline bool fits_one_xcd(int64_t grid, int blocks, int cus) {
  return grid <= (int64_t)std::min(blocks, kXcdBlocks) * std::min(cus, kXcdCus);
}

}  // namespace onsas
