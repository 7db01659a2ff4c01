// Prints the share GEMM's kernel choice: one line per line "x w w_bits M K N" of stdin (x, w: addresses).
#include <cstdio>

#include "gemm_rule.hpp"

int main() {
  static const char* names[] = {"few", "dma2", "dma3", "reg", "fused", "zero"};
  unsigned long long x, w;
  int bits, m, k, n;
  while (std::scanf("%llu %llu %d %d %d %d", &x, &w, &bits, &m, &k, &n) == 6) {
    const auto c = praghip::gemm_choice(reinterpret_cast<const void*>(x), reinterpret_cast<const void*>(w), bits, m, k, n);
    std::printf("%s %d %d %d %d\n", names[c.kernel], c.k_split, c.splits, c.planes, c.adds ? 1 : 0);
  }
}
