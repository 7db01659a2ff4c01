// Three-phase keyswitch at N = 16384, and the choice of the shapes that take it.
#include "keyswitch_rows.hpp"

namespace praghip {

template <int LOG>
hipError_t run_keyswitch_rows_small(const KsArgs& a, const KsConst* kc_dev, const KsConst& kc, const NttDevice& d,
                                    hipStream_t s);

// N = 4096, 8192 and 16384 with digits of up to three primes.  Key primes of
// 2^60 and more (Harvey bounds) only at N = 16384.
bool keyswitch_rows_supported(const KsConst& kc) {
  if (kc.dnum < 1 || kc.dig_lo[1] > 3) return false;  // the first digits are the largest
  return kc.log_n == 14 || ((kc.log_n == 12 || kc.log_n == 13) && kc.lazy);
}

// 64 at N = 16384.  Below it a chunk of 64 ciphertexts of few digits and primes is
// soon over (22 us at N = 4096 with one digit of one prime), so large batches paid
// their launches over and over: chunks of as many ciphertexts as expand to 64 MiB,
// and 64 at least.  us, chunks of 64 / these / the whole-limb kernel: N = 4096, one
// data prime, 512 ciphertexts 177 / 93 / 126; two digits of one 50-bit prime, 512,
// 256 / 180 / 222; N = 8192, one data prime, 512, 258 / 168 / 237; six digits of one
// prime stay at 64.
size_t keyswitch_rows_chunk(const KsConst& kc) {
  if (kc.log_n == 14) return 64;
  const size_t expanded = size_t(kc.dnum) * size_t(kc.K) * 8 << kc.log_n;
  return std::max<size_t>(64, (size_t(64) << 20) / expanded);
}

hipError_t launch_keyswitch_rows(const KsArgs& a, const KsConst* kc_dev, const KsConst& kc, const NttDevice& d,
                                 hipStream_t s) {
  if (!keyswitch_rows_supported(kc) || !a.inter || a.inter_cts == 0) return hipErrorNotSupported;
  switch (kc.log_n) {
    case 12: return run_keyswitch_rows_small<12>(a, kc_dev, kc, d, s);
    case 13: return run_keyswitch_rows_small<13>(a, kc_dev, kc, d, s);
    default: return run_keyswitch_rows<14>(a, kc_dev, kc, d, s);
  }
}

}  // namespace praghip
