// The residency rule of the one-launch solvers (onsas.jl_amd/csrc/resident_rule.hpp):
// no grid is allowed that the CUs do not take at once.
#include <cstdio>
#include <cstdlib>

#include "resident_rule.hpp"

using namespace onsas;

int main() {
  for (int cus : {8, 32, 64, 128, 256, 304})
    for (int blocks = 0; blocks <= 8; ++blocks)
      for (int64_t grid = 1; grid <= 128; ++grid) {
        const int64_t xcd = (int64_t)blocks * (cus < 32 ? cus : 32);
        if (fits_device(grid, blocks, cus) != (grid <= (int64_t)blocks * cus)) std::abort();
        if (fits_one_xcd(grid, blocks, cus) && grid > xcd) std::abort();
        if (fits_one_xcd(grid, blocks, cus) && !fits_device(grid, blocks, cus)) std::abort();
        // up to three workgroups a CU the XCD is used for all that it takes
        if (blocks <= 3 && grid <= xcd && !fits_one_xcd(grid, blocks, cus)) std::abort();
      }
  std::puts("ok");
}
