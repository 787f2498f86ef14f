// Prints which form of the fused native GEMM each product runs
// (choose_fused_shape of the library's own objects), for
// tests/test_fused_forms.py. Input: lines "m n k planes"; output per line:
// "<form> <slices> <k_slice> <workspace bytes>", form none, tile, residue or
// digits.
#include <cstdint>
#include <iostream>

#include "kernels.hpp"

int main() {
  int64_t m, n, k;
  uint32_t planes;
  while (std::cin >> m >> n >> k >> planes) {
    rns8x::FusedShape s{};
    const char* form = "none";
    if (rns8x::choose_fused_shape(m, n, k, planes, rns8x::padded_ld(n), s))
      form = s.skinny == 2 ? "digits" : s.skinny ? "residue" : "tile";
    std::cout << form << " " << s.slices << " " << s.k_slice << " " << s.ws_bytes << "\n";
  }
  return 0;
}
