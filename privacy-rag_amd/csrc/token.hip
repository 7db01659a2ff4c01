// Element-wise kernels of the token-resident path and of the acyclic packing
// tree:
//   pack_prepare: right * x^shift, then the sum and the Galois image of the
//     difference of a packing pair (switch.cu:49-58 packing_prepare);
//   pack_finish: the two switched halves added (switch.cu:59-61).
// All residues stay canonical (< q < 2^62, so a + b never wraps).  Each kernel
// is a single HBM pass; one thread per output coefficient, contiguous in the
// coefficient index so reads and writes coalesce except the Galois-permuted
// reads, which stay inside one 2^log_n-word limb.
#include <type_traits>

#include "kernels.hpp"

namespace praghip {

static unsigned elem_grid(size_t items) {
  return unsigned(std::min<size_t>(std::max<size_t>((items + 255) / 256, 1), 1u << 20));
}

// Sum of products of a batch of weight columns against the resident inputs:
//   out[c][l][z] = sum_b in[b][l][z] * w[c][b][l % P][z]  mod q_{l % P}
// (resident.cu:38-45 accumulate), for every column c of the batch.
//
// For primes below 2^60 no product is reduced: with both words split
// at 30 bits a product is four 32 x 32 multiply-adds into three sums (weights
// 1, 2^30, 2^60), and the sums are brought below q once per sixteen blocks
// (the middle sum takes two products a block and is carried into the upper one
// after eight) - about 7
// instructions per product at 19 blocks instead of 20 with a Shoup product
// each.  A thread holds KL limbs (of one prime) x kMacCoords columns of one
// coefficient; every input word then meets four columns and every weight word
// KL limbs.
//
// It then stands between its bounds (below), so workgroups are numbered for the L2:
// the ones on one XCD (blockIdx % 8) that share a prime's 256 coefficients come
// one after the other - every column group and limb tile of them - and the
// input words (19 blocks x 8 limbs: 311 KB) are read from HBM once.
// 64 columns, 19 blocks, 48 limbs at N = 16384: 796 us with Shoup products and the
// columns walked over all of N, 441 here: 1,076 MB read (weights 956, inputs 120)
// and 403 written at 3.4 TB/s, VALU busy 59%.
//
// MODE: kMacPm   - primes just below 2^60 (2^60 == c): the sums are brought
//                  together by three multiply-adds;
//       kMacNarrow - any primes below 2^60: by a Shoup product by 2^60;
//       kMacWide - primes of 2^60 and more.
//
// Primes of 2^60 and more: a Shoup quotient per weight word (from the Barrett
// ratio), Shoup products and canonical sums; one or two columns in a loop of their
// own (one column of two 62-bit primes, 19 blocks and 2 slots, N = 4096, the whole
// evaluation, us: 61 with four columns formed and one stored, 42 so).
constexpr int kMacCoords = 4;
enum MacMode { kMacPm, kMacNarrow, kMacWide };

struct MacConst {
  uint64_t q, one_q, c60, c60_q;  // q, Shoup quotient of 1, c60 = 2^60 mod q with its quotient
  uint32_t c;                     // kMacPm: M = q 2^(60-b) = 2^60 - c (pm_bits b, c < 2^28)
  int bits;
};

// s0 + s1 2^30 + s2 2^60 mod q as some word below 2^62.
template <MacMode MODE>
__device__ __forceinline__ uint64_t mac_fold(uint64_t s0, uint64_t s1, uint64_t s2, const MacConst& m) {
  if constexpr (MODE == kMacPm) return sum_pm(s0, s1, s2, m.c);
  s1 += s0 >> 30;
  s2 += s1 >> 30;
  return mul_shoup_lazy(s2, m.c60, m.c60_q, m.q) + (((s1 & kLow30) << 30) | (s0 & kLow30));
}

template <MacMode MODE, int KL>
__global__ void __launch_bounds__(256)
    token_mac_kernel(const uint64_t* __restrict__ in, const uint64_t* __restrict__ w, uint64_t* __restrict__ out,
                     unsigned coords, unsigned blocks, unsigned limbs, int log_n, BarrettList bl, unsigned tiles,
                     unsigned groups, unsigned places) {
  // blockIdx = ((place / 8) * groups * tiles + group * tiles + tile) * 8 + place % 8,
  // place = (prime, 256 coefficients)
  const unsigned x8 = blockIdx.x & 7u, y = blockIdx.x >> 3, inner = groups * tiles;
  const unsigned place = (y / inner) * 8u + x8, gt = y % inner;
  if (place >= places) return;
  const unsigned P = unsigned(bl.count), n = 1u << log_n, zs = (n + 255u) / 256u;
  const unsigned p = place / zs, z = (place % zs) * 256u + threadIdx.x;
  if (z >= n) return;
  const unsigned c0 = (gt / tiles) * unsigned(kMacCoords);
  const unsigned l0 = p + (gt % tiles) * unsigned(KL) * P;  // limbs l0, l0 + P, ...
  if (l0 >= limbs) return;
  const Barrett m = bl.m[p];
  const size_t words = size_t(limbs) << log_n, wcol = (size_t(blocks) * P) << log_n;
  const unsigned cn = coords - c0 < unsigned(kMacCoords) ? coords - c0 : unsigned(kMacCoords);
  // past the last limb or column a thread works on the first one again and
  // does not store it: no branch in the loop
  size_t xo[KL], wo[kMacCoords];
#pragma unroll
  for (int k = 0; k < KL; ++k) {
    const unsigned l = l0 + unsigned(k) * P;
    xo[k] = size_t(l < limbs ? l : l0) << log_n;
  }
#pragma unroll
  for (int c = 0; c < kMacCoords; ++c)
    wo[c] = (c0 + (unsigned(c) < cn ? unsigned(c) : 0u)) * wcol + (size_t(p) << log_n);
  const auto store = [&](int c, int k, uint64_t v) {
    const unsigned l = l0 + unsigned(k) * P;
    if (unsigned(c) < cn && l < limbs) (out + (size_t(c0) + unsigned(c)) * words + (size_t(l) << log_n))[z] = v;
  };
  if constexpr (MODE != kMacWide) {
    MacConst mc;
    mc.q = m.q;
    mc.one_q = m.r1;                                // floor(2^64 / q)
    mc.c60 = (1ull << 60) - (m.r1 >> 4) * m.q;      // 2^60 mod q
    mc.c60_q = shoup_quotient(mc.c60, m);
    mc.bits = 64 - __clzll((long long)m.q);
    mc.c = uint32_t((1ull << 60) - (m.q << (60 - mc.bits)));
    uint64_t s0[kMacCoords][KL], s1[kMacCoords][KL], s2[kMacCoords][KL];
#pragma unroll
    for (int c = 0; c < kMacCoords; ++c)
#pragma unroll
      for (int k = 0; k < KL; ++k) s0[c][k] = s1[c][k] = s2[c][k] = 0;
    // the next block's words are in flight while this block's are multiplied
    uint64_t xn[KL], wn[kMacCoords];
    const auto load = [&](unsigned b) {
      const uint64_t* xb = in + size_t(b) * words;
      const uint64_t* wb = w + ((size_t(b) * P) << log_n);
#pragma unroll
      for (int k = 0; k < KL; ++k) xn[k] = (xb + xo[k])[z];
#pragma unroll
      for (int c = 0; c < kMacCoords; ++c) wn[c] = (wb + wo[c])[z];
    };
    load(0);
    for (unsigned b = 0; b < blocks; ++b) {
      uint32_t x0[KL], x1[KL], w0[kMacCoords], w1[kMacCoords];
#pragma unroll
      for (int k = 0; k < KL; ++k) x0[k] = uint32_t(xn[k]) & uint32_t(kLow30), x1[k] = uint32_t(xn[k] >> 30);
#pragma unroll
      for (int c = 0; c < kMacCoords; ++c) w0[c] = uint32_t(wn[c]) & uint32_t(kLow30), w1[c] = uint32_t(wn[c] >> 30);
      if (b + 1 < blocks) load(b + 1);
      if (b && b % 8 == 0) {
#pragma unroll
        for (int c = 0; c < kMacCoords; ++c)
#pragma unroll
          for (int k = 0; k < KL; ++k) {
            if (b % 16) {
              // sixteen products of s2 and both carries of s1 stay below 2^64: s1
              // restarts below 2^32 after a fold, so this carry is at most 2^34 - 28
              // and the fold's (with s0's) at most 2^34 - 16, and
              // 16 (2^30 - 1)^2 + 2^35 - 44 = 2^64 - 28
              s2[c][k] += s1[c][k] >> 30;
              s1[c][k] &= kLow30;
            } else {  // below 2^62: s1 restarts below 2^32
              const uint64_t r = mac_fold<MODE>(s0[c][k], s1[c][k], s2[c][k], mc);
              s0[c][k] = r & kLow30;
              s1[c][k] = r >> 30;
              s2[c][k] = 0;
            }
          }
      }
#pragma unroll
      for (int k = 0; k < KL; ++k) {
#pragma unroll
        for (int c = 0; c < kMacCoords; ++c) {
          s0[c][k] += uint64_t(x0[k]) * w0[c];
          s1[c][k] += uint64_t(x0[k]) * w1[c];
          s1[c][k] += uint64_t(x1[k]) * w0[c];
          s2[c][k] += uint64_t(x1[k]) * w1[c];
        }
      }
    }
#pragma unroll
    for (int c = 0; c < kMacCoords; ++c)
#pragma unroll
      for (int k = 0; k < KL; ++k) {
        const uint64_t r = mac_fold<MODE>(s0[c][k], s1[c][k], s2[c][k], mc);
        if constexpr (MODE == kMacPm)
          store(c, k, canon_pm(r, m.q, mc.c >> (60 - mc.bits), unsigned(mc.bits) - 32));
        else
          store(c, k, mul_shoup(r, 1, mc.one_q, m.q));
      }
  } else {
    // the products bound this loop, so one or two columns get a loop of their own
    const auto wide = [&](auto columns) {
      constexpr int C = decltype(columns)::value;
      uint64_t acc[C][KL];
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int k = 0; k < KL; ++k) acc[c][k] = 0;
      for (unsigned b = 0; b < blocks; ++b) {
        uint64_t xv[KL];
#pragma unroll
        for (int k = 0; k < KL; ++k) xv[k] = (in + size_t(b) * words + xo[k])[z];
#pragma unroll
        for (int c = 0; c < C; ++c) {
          const uint64_t wv = (w + wo[c] + ((size_t(b) * P) << log_n))[z];
          const uint64_t wq = shoup_quotient(wv, m);
#pragma unroll
          for (int k = 0; k < KL; ++k) acc[c][k] = add_mod(acc[c][k], mul_shoup(xv[k], wv, wq, m.q), m.q);
        }
      }
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int k = 0; k < KL; ++k) store(c, k, acc[c][k]);
    };
    if (cn > 2)
      wide(std::integral_constant<int, kMacCoords>{});
    else if (cn == 2)
      wide(std::integral_constant<int, 2>{});
    else
      wide(std::integral_constant<int, 1>{});
  }
}

hipError_t launch_token_mac(const uint64_t* in, const uint64_t* w, uint64_t* out, size_t coords, size_t blocks,
                            size_t limbs, int log_n, const Barrett* m, int primes, hipStream_t s) {
  BarrettList bl{};
  for (int i = 0; i < primes; ++i) bl.m[i] = m[i];
  bl.count = primes;
  MacMode mode = kMacPm;
  for (int i = 0; i < primes; ++i) {
    const int b = pm_bits(m[i].q);
    if (m[i].q >> 60)
      mode = kMacWide;
    else if (mode == kMacPm && (!b || ((1ull << 60) - (m[i].q << (60 - b))) >> 28))
      mode = kMacNarrow;
  }
  // limbs of one prime: 2 per thread for a single ciphertext's, else 4 (their 48
  // 64-bit sums are 96 registers; 8 limbs would leave two waves per SIMD)
  const unsigned per = unsigned((limbs + size_t(primes) - 1) / size_t(primes)), kl = per <= 2 ? 2 : 4;
  const unsigned tiles = (per + kl - 1) / kl, groups = unsigned((coords + kMacCoords - 1) / kMacCoords);
  const unsigned places = unsigned(primes) * unsigned(((size_t(1) << log_n) + 255) / 256);
  const dim3 grid((places + 7) / 8 * 8 * groups * tiles);
  const auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, in, w, out, unsigned(coords), unsigned(blocks), unsigned(limbs),
                       log_n, bl, tiles, groups, places);
  };
  if (mode == kMacPm)
    kl == 2 ? go(token_mac_kernel<kMacPm, 2>) : go(token_mac_kernel<kMacPm, 4>);
  else if (mode == kMacNarrow)
    kl == 2 ? go(token_mac_kernel<kMacNarrow, 2>) : go(token_mac_kernel<kMacNarrow, 4>);
  else
    kl == 2 ? go(token_mac_kernel<kMacWide, 2>) : go(token_mac_kernel<kMacWide, 4>);
  return hipGetLastError();
}

// Local pair i is pair e = first + i of the list; it reads
// left(e) = left + ((e / group) * stride + e % group) * ct and right(e) the
// same way from right (ct = 2 L N words), and writes
//   sum[i]  = left(e) + x^shift right(e)
//   diff[i] = sigma_g(left(e) - x^shift right(e)),  sigma_g: x -> x^g
// with x^shift right at j = right[j - shift], negated for j < shift.  Both
// outputs are written in coefficient order: diff at d takes the source
// coefficient u = d g^-1 mod 2N (negated when u >= N), gathered from inside
// the same limb, so no write is scattered.
// MERGE: the switched halves of a pair are added, and so are their components 0,
// which the switches only pass on: component 0 of sum takes both and that of
// diff is not written (a quarter of the writes less, and of the switches' reads).
__device__ __forceinline__ uint64_t shifted_diff(const uint64_t* __restrict__ l, const uint64_t* __restrict__ r,
                                                 size_t j, size_t n, size_t shift, uint64_t q, uint64_t& sum) {
  uint64_t v = r[(j + n - shift) & (n - 1)];
  v = (j < shift && v) ? q - v : v;
  const uint64_t a = l[j];
  sum = add_mod(a, v, q);
  return sub_mod(a, v, q);
}

template <bool MERGE>
__global__ void __launch_bounds__(256)
    pack_prepare_kernel(const uint64_t* __restrict__ left, const uint64_t* __restrict__ right,
                        uint64_t* __restrict__ sum, uint64_t* __restrict__ diff, size_t count, size_t first,
                        size_t group, size_t stride, PrimeList pl, int log_n, size_t shift, uint32_t ginv) {
  const size_t n = size_t(1) << log_n, L = size_t(pl.count), ct = 2 * L * n, total = count * ct;
  for (size_t idx = size_t(blockIdx.x) * blockDim.x + threadIdx.x; idx < total;
       idx += size_t(gridDim.x) * blockDim.x) {
    const size_t i = idx / ct, w = idx - i * ct, d = w & (n - 1), base = w - d, e = first + i;
    const size_t src = ((e / group) * stride + e % group) * ct + base;
    const uint64_t q = pl.q[(w >> log_n) % L];
    const uint64_t* l = left + src;
    const uint64_t* r = right + src;
    uint64_t s0;
    (void)shifted_diff(l, r, d, n, shift, q, s0);
    if constexpr (!MERGE) sum[i * ct + w] = s0;
    const size_t u = (d * size_t(ginv)) & (2 * n - 1);
    uint64_t unused;
    const uint64_t delta = shifted_diff(l, r, u & (n - 1), n, shift, q, unused);
    const uint64_t mapped = (u >= n && delta) ? q - delta : delta;
    if constexpr (MERGE) {
      const bool first_half = w < ct / 2;  // component 0
      sum[i * ct + w] = first_half ? add_mod(s0, mapped, q) : s0;
      if (!first_half) diff[i * ct + w] = mapped;
    } else {
      diff[i * ct + w] = mapped;
    }
  }
}

hipError_t launch_pack_prepare(const uint64_t* left, const uint64_t* right, uint64_t* sum, uint64_t* diff,
                               size_t count, size_t first, size_t group, size_t stride, const PrimeList& pl,
                               int log_n, size_t shift, uint32_t ginv, bool merge, hipStream_t s) {
  const size_t total = count * 2 * size_t(pl.count) << log_n;
  const auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(elem_grid(total)), dim3(256), 0, s, left, right, sum, diff, count, first, group,
                       stride, pl, log_n, shift, ginv);
  };
  merge ? go(pack_prepare_kernel<true>) : go(pack_prepare_kernel<false>);
  return hipGetLastError();
}

// out[w] = a[w] + b[w] mod q over count ciphertexts [count][2][L][N].
__global__ void __launch_bounds__(256)
    pack_finish_kernel(const uint64_t* __restrict__ a, const uint64_t* __restrict__ b, uint64_t* __restrict__ out,
                       size_t count, PrimeList pl, int log_n) {
  const size_t L = size_t(pl.count), total = count * 2 * L << log_n;
  for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total; i += size_t(gridDim.x) * blockDim.x)
    out[i] = add_mod(a[i], b[i], pl.q[(i >> log_n) % L]);
}

hipError_t launch_pack_finish(const uint64_t* a, const uint64_t* b, uint64_t* out, size_t count, const PrimeList& pl,
                              int log_n, hipStream_t s) {
  const size_t total = count * 2 * size_t(pl.count) << log_n;
  hipLaunchKernelGGL(pack_finish_kernel, dim3(elem_grid(total)), dim3(256), 0, s, a, b, out, count, pl, log_n);
  return hipGetLastError();
}

// Selective evaluation of a batch (evaluate_selective, matrix.cu:65-81, with
// the c0 gather of matrix.cu:41-44): c0 of every output group keeps only the
// `count` target coefficients idx[] (strictly increasing, < N) and is zero
// elsewhere; selected[g][k][j] = c0[g][k][idx[j]] when selected is given.  One
// thread per c0 coefficient finds its coefficient among the targets by binary
// search over idx staged in LDS; c1 is left as it is.
__global__ void __launch_bounds__(256)
    select_c0_kernel(uint64_t* __restrict__ out, size_t groups, int primes, int log_n,
                     const uint64_t* __restrict__ idx, unsigned count, uint64_t* __restrict__ selected) {
  __shared__ uint64_t targets[kMaxTargets];
  for (unsigned j = threadIdx.x; j < count; j += blockDim.x) targets[j] = idx[j];
  __syncthreads();
  const size_t n = size_t(1) << log_n, per_group = size_t(primes) << log_n, total = groups * per_group;
  for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total; i += size_t(gridDim.x) * blockDim.x) {
    const size_t g = i / per_group, r = i % per_group, z = r & (n - 1);
    unsigned lo = 0, hi = count;  // first target >= z
    while (lo < hi) {
      const unsigned mid = (lo + hi) >> 1;
      if (targets[mid] < z)
        lo = mid + 1;
      else
        hi = mid;
    }
    uint64_t* c0 = out + g * 2 * per_group + r;  // c0 limb k, coefficient z
    if (lo < count && targets[lo] == z) {
      if (selected) selected[(g * size_t(primes) + (r >> log_n)) * count + lo] = *c0;
    } else {
      *c0 = 0;
    }
  }
}

hipError_t launch_select_c0(uint64_t* out, size_t groups, int primes, int log_n, const uint64_t* idx,
                            unsigned count, uint64_t* selected, hipStream_t s) {
  if (count == 0 || count > kMaxTargets) return hipErrorInvalidValue;
  const size_t total = groups * size_t(primes) << log_n;
  hipLaunchKernelGGL(select_c0_kernel, dim3(elem_grid(total)), dim3(256), 0, s, out, groups, primes, log_n, idx,
                     count, selected);
  return hipGetLastError();
}

}  // namespace praghip
