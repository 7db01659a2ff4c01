// CPU check of the products modulo primes just below a power of two (mul_pm,
// fold_pm, canon_pm) and of the bounds ArPM's butterflies keep, against
// 128-bit host arithmetic: every stage's outputs must be congruent to the
// butterfly's and stay below that stage's bound, from inputs at the bound of
// the stage before, and no sum may wrap.  Plants a wrong folding constant and
// a missing fold.
#include <cstdio>
#include <random>
#include <vector>

#include "ntt_core.hpp"
using namespace praghip;
using u128 = unsigned __int128;

static NttPrime prime_of(uint64_t q) {
  NttPrime p{};
  p.q = q;
  p.pm_bits = pm_bits(q);
  return p;
}
static ulonglong2 pair_of(uint64_t w, uint64_t q) {
  return make_ulonglong2(pm_split(w), pm_split(uint64_t(((u128)w << 32) % q)));
}

// mode 0: as it is; 1: a wrong folding constant; 2: forward stage 4 without its fold
static int check(uint64_t q, int mode, std::mt19937_64& rng) {
  int bad = 0;
  NttPrime pr = prime_of(q);
  if (!pr.pm_bits) return -1;
  ArPM ar(pr);
  if (mode == 1) ar.c2 += 2;
  const uint64_t unit = 1ull << 60, eps = 1ull << 35, m = q << (60 - pr.pm_bits), top = ~0ull;
  const auto res = [&](u128 x) { return uint64_t(x % q); };
  const auto some = [&](uint64_t limit) {  // edges and random words below `limit`
    std::vector<uint64_t> v = {0, 1, limit - 1, limit - 2, limit / 2, 0xffffffffull < limit ? 0xffffffffull : 3};
    for (int i = 0; i < 40; ++i) v.push_back(rng() % limit);
    return v;
  };
  const std::vector<uint64_t> ws = some(q);
  for (uint64_t w : ws) {
    const ulonglong2 p = pair_of(w, q);
    for (uint64_t a : some(top)) {
      const uint64_t t = mul_pm(a, p.x, p.y, ar.c2);
      if (t >= ar.m3 || res(t) != res((u128)a * w)) ++bad;
    }
  }
  for (uint64_t a : some(top)) {
    if (fold_pm(a, ar.c1) > unit + eps || res(fold_pm(a, ar.c1)) != res(a)) ++bad;
    if (ar.to_u64_fwd(a) != res(a)) ++bad;
  }
  // forward: bound after stage s from the bound before it
  uint64_t before = q;
  for (int s = 0; s < 14; ++s) {
    const int run = s % 4 + 1;  // stages since the last fold
    const uint64_t after = unit + eps + uint64_t(run) * 3 * unit;
    for (uint64_t w : {uint64_t(0), uint64_t(1), q - 1, uint64_t(rng() % q)}) {
      const ulonglong2 p = pair_of(w, q);
      for (uint64_t x : some(before))
        for (uint64_t y : some(before)) {
          uint64_t a = x, b = y;
          ar.fwd_at(mode == 2 && s == 4 ? 1 : s, a, b, p);
          const uint64_t t = res((u128)y * w);
          if (a >= after || b >= after || res(a) != res((u128)x + t) || res(b) != res((u128)x + q - t)) ++bad;
        }
    }
    before = after;
  }
  // inverse: below 4M before even stages, below 8M before odd ones
  pr.ninv = pair_of(q - 2, q).x, pr.ninv_q = pair_of(q - 2, q).y;
  pr.last = pair_of(q / 3, q).x, pr.last_q = pair_of(q / 3, q).y;
  for (int l = 0; l < 2; ++l) {
    const uint64_t in = (l % 2 ? 8 : 4) * m, out = (l % 2 ? 4 : 8) * m;
    for (uint64_t w : {uint64_t(0), uint64_t(1), q - 1, uint64_t(rng() % q)}) {
      const ulonglong2 p = pair_of(w, q);
      for (uint64_t x : some(in))
        for (uint64_t y : some(in)) {
          uint64_t a = x, b = y;
          ar.inv_at(l, a, b, p);
          const uint64_t d = res((u128)x + 16 * (u128)m - y);
          if (a >= out || b >= out || res(a) != res((u128)x + y) || res(b) != res((u128)d * w)) ++bad;
          a = x, b = y;
          ar.inv_last(a, b, pr);
          if (a >= 4 * m || b >= 4 * m || res(a) != res((u128)res((u128)x + y) * (q - 2)) ||
              res(b) != res((u128)d * (q / 3)))
            ++bad;
        }
    }
  }
  return bad;
}

int main() {
  std::mt19937_64 rng(2025);
  // the arithmetic needs no primality: the locked primes' extremes, the
  // smallest and largest distance below 2^60, 2^54 and 2^50 that pm_bits takes
  std::vector<uint64_t> qs = {0xfffffffff898001ull, 0xffffffffffe8001ull, (1ull << 60) - 1, (1ull << 60) - (1ull << 27) + 2,
                              (1ull << 54) - 3, (1ull << 54) - (1ull << 25) + 1, (1ull << 57) - (1ull << 27) + 2,
                              (1ull << 50) - 1, (1ull << 50) - (1ull << 21) + 1};
  int bad = 0, planted = 0;
  for (uint64_t q : qs) {
    const int b = check(q, 0, rng);
    if (b) printf("q=%llx bad=%d\n", (unsigned long long)q, b);
    bad += b != 0;
    planted += check(q, 1, rng) > 0;
    planted += check(q, 2, rng) > 0;
  }
  // refused: too far below the power of two, 61 bits, 49 bits
  for (uint64_t q : {(1ull << 60) - (1ull << 27) - 1, (1ull << 61) - 1, (1ull << 49) - 1, (1ull << 50) - (1ull << 21) - 1,
                     3ull << 57})
    bad += pm_bits(q) != 0;
  printf("bad=%d planted=%d\n", bad, planted);
  const bool ok = bad == 0 && planted == int(2 * qs.size());
  printf(ok ? "ALL OK\n" : "FAIL\n");
  return !ok;
}
