// Answers questions about the library's dispatch rules, asked of its own
// objects, for tests/test_dispatch.py. Input lines and the line each prints:
//
//   fused <m> <n> <k> <planes>  "<form> <slices> <k_slice> <workspace bytes>"
//     (choose_fused_shape), form none, tile, residue or digits
//   grid <units> <slots>        workgroups of a persistent launch
#include <cstdint>
#include <iostream>
#include <string>

#include "kernels.hpp"

int main() {
  std::string what;
  while (std::cin >> what) {
    if (what == "fused") {
      int64_t m, n, k;
      uint32_t planes;
      std::cin >> m >> n >> k >> planes;
      rns8x::FusedShape s{};
      const char* form = "none";
      if (rns8x::choose_fused_shape(m, n, k, planes, rns8x::padded_ld(n), s))
        form = s.skinny == 2 ? "digits" : s.skinny ? "residue" : "tile";
      std::cout << form << " " << s.slices << " " << s.k_slice << " " << s.ws_bytes << "\n";
    } else if (what == "grid") {
      uint64_t units, slots;
      std::cin >> units >> slots;
      std::cout << rns8x::persistent_grid(units, slots) << "\n";
    } else {
      return 2;
    }
  }
  return 0;
}
