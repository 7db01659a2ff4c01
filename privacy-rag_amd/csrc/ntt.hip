// Batched negacyclic NTT / INTT kernels (NttBatch::transform, ntt.cu:104-127,
// and the stage loops inside Switch / TokenWeights / Matrix / PublicZero).
//
// Layout: [limbs][N] u64, limb l uses prime index l % P (the reference's
// [batch][prime][coefficient], ntt.hpp:20).  One workgroup per limb; the
// whole limb is transformed in registers + LDS, so each launch reads and
// writes every coefficient once (the reference launches 14 stages, each a
// full HBM round trip).
#include "kernels.hpp"

namespace praghip {

// Kernel over the limbs whose prime uses arithmetic A: virtual index v maps to
// limb (v / C) * P + sel[v % C], where sel lists the C prime indices of that
// arithmetic.  Workgroup g transforms v = g, g + G, ... (G resident
// workgroups).  Each limb is loaded in the first pass's layout (coalesced),
// transformed in registers + LDS and stored in the last pass's layout.  The
// float-path forward kernel issues the next limb's loads as soon as the
// current limb no longer needs the LDS (before its last pass), so they overlap
// the last pass and the stores instead of starting after them.  The
// float-path inverse kernel loads the next limb's first-pass twiddles before
// the current limb's stores and its words after them; the other kernels have
// no registers to spare and load each limb at the top of its turn.
//
// LIFT (forward only): limb l = b P + k is not read from data but formed on
// load from ring block b, lift_word mod q_k (ring[b][z] when width = 0;
// ring[b][width-1-z] for z < width and 0 above otherwise), so the lifted limbs
// never pass through memory.
struct NttLift {
  const uint64_t* ring = nullptr;
  size_t width = 0;
};

// FINISH (inverse only): limb l = (slot * 2 + c) P + p is not stored in place but
// finished on the way out (resident.cu:54-59 add_shift): in component 0
// scaled[slot][p] is added to coefficient `lift`, and the limb times x^-lift
// goes to out, so the products are not read and written once more (64 columns
// of 4 slots, us: 271 for the transform and 176 for the finish as a pass of its
// own -> 293 together).
struct NttFinish {
  uint64_t* out = nullptr;
  const uint64_t* scaled = nullptr;
  unsigned lift = 0;
};

// The signed value of ring word v (bit 58 the sign) as a forward transform's
// input: canonical, or for ArPM below M by one masked addition of M - 2^59 (M is
// a multiple of q above 2^59 whatever q's size).
template <class A>
__device__ __forceinline__ uint64_t lift_word(const A& ar, uint64_t v, const NttPrime& pr) {
  if constexpr (std::is_same<A, ArPM>::value)
    return v + (((ar.m8 >> 3) - (1ull << 59)) & (0ull - (v >> 58)));
  else
    return lift59_residue(v, pr);
}

template <int LOGN, bool INV, class A, bool LIFT = false, bool FINISH = false>
__global__ void __launch_bounds__(ntt_threads<LOGN>())
    ntt_kernel(uint64_t* __restrict__ data, size_t count, const NttPrime* __restrict__ primes,
               const typename A::TW* __restrict__ tw, int P, const int* __restrict__ sel, int C, NttLift lift,
               NttFinish fin) {
  __shared__ __attribute__((aligned(16))) uint64_t lds[(1 << LOGN) + (1 << LOGN) / 16];
  using T = typename A::T;
  // with FINISH recomputed per limb (v < 2^40): the output indices would
  // otherwise be kept in registers across the loop and spill
  unsigned t = threadIdx.x;
  const auto limb_of = [&](size_t v) { return (v / unsigned(C)) * unsigned(P) + unsigned(sel[v % unsigned(C)]); };
  const auto in_index = [&](int j) { return INV ? inv_in_index<LOGN>(t, j) : fwd_in_index<LOGN>(t, j); };
  // the input words of limb `limb` in the first pass's register layout (with
  // LIFT the ring words, lifted by `lifted` once the limb's turn comes)
  const auto load = [&](uint64_t (&raw)[kE], size_t limb) {
    if constexpr (LIFT) {
      // coefficient z reads base[sign * z]: base = ring[b] (sign +1), or the
      // last word of the token block ring[b][width - 1] (sign -1, z < width)
      const size_t b = limb / unsigned(P);
      const bool rev = lift.width != 0;
      const uint64_t* base = lift.ring + (rev ? b * lift.width + lift.width - 1 : b << LOGN);
      const long long sign = rev ? -1 : 1;
      const unsigned limit = rev ? unsigned(lift.width) : (1u << LOGN);
#pragma unroll
      for (int j = 0; j < kE; ++j) {
        const unsigned z = in_index(j);
        raw[j] = z < limit ? base[sign * (long long)z] : 0;
      }
    } else {
      const uint64_t* x = data + (limb << LOGN);
#pragma unroll
      for (int j = 0; j < kE; ++j) raw[j] = x[in_index(j)];
    }
  };
  const auto lifted = [&](uint64_t v, const A& ar, const NttPrime& pr) {
    if constexpr (LIFT)
      return lift_word(ar, v, pr);
    else
      return v;
  };
  const auto store = [&](const A& ar, T (&x)[kE], size_t limb, const NttPrime& pr) {
    uint64_t* out = (FINISH ? fin.out : data) + (limb << LOGN);
    if constexpr (FINISH) {
      const size_t row = limb / unsigned(P), slot = row >> 1;  // row = slot * 2 + component
      const uint64_t add = row & 1 ? 0 : fin.scaled[slot * unsigned(P) + limb % unsigned(P)];
#pragma unroll
      for (int j = 0; j < kE; ++j) {
        const unsigned z = inv_out_index<LOGN>(t, j);
        uint64_t v = ar.to_u64_inv(x[j]);
        if (z == fin.lift) v = add_mod(v, add, pr.q);
        out[(z - fin.lift) & ((1u << LOGN) - 1)] = z < fin.lift && v ? pr.q - v : v;
        if ((j & 3) == 3) __builtin_amdgcn_sched_barrier(0);
      }
    } else if (!INV) {
#pragma unroll
      for (int j = 0; j < kE; j += 2)
        *reinterpret_cast<ulonglong2*>(out + fwd_out_index<LOGN>(t, j)) =
            make_ulonglong2(ar.to_u64_fwd(x[j]), ar.to_u64_fwd(x[j + 1]));
    } else {
#pragma unroll
      for (int j = 0; j < kE; ++j) out[inv_out_index<LOGN>(t, j)] = ar.to_u64_inv(x[j]);
    }
  };
  if constexpr (std::is_same<T, double>::value && !INV) {
    size_t v = blockIdx.x;
    if (v >= count) return;
    uint64_t raw[kE];
    load(raw, limb_of(v));
    for (; v < count; v += gridDim.x) {
      const size_t limb = limb_of(v);
      const int p = int(limb % unsigned(P));
      const NttPrime pr = primes[p];
      const A ar(pr);
      T x[kE];
#pragma unroll
      for (int j = 0; j < kE; ++j) x[j] = ar.from_u64(lifted(raw[j], ar, pr));
      const size_t vn = v + gridDim.x;
      ntt_regs<LOGN, INV>(x, reinterpret_cast<T*>(lds), t, tw + (size_t(p) << LOGN), ar, pr, [&] {
        if (vn < count) load(raw, limb_of(vn));
      });
      store(ar, x, limb, pr);
    }
  } else if constexpr (std::is_same<T, double>::value && INV) {
    // the next limb's first-pass twiddles are loaded before this limb's
    // stores (vector memory operations complete in order: issued behind the
    // stores they would wait for them, and the first pass waits for its
    // twiddles); its words after them (before the stores as well, they cost
    // registers and measured no faster)
    size_t v = blockIdx.x;
    if (v >= count) return;
    uint64_t raw[kE];
    typename A::TW w0[pass_twiddles<Passes<LOGN>::r(INV, 0)>()];
    {
      const size_t limb = limb_of(v);
      load(raw, limb);
      load_pass_twiddles<LOGN, INV, 0>(w0, t, tw + ((limb % unsigned(P)) << LOGN));
    }
    for (; v < count; v += gridDim.x) {
      const size_t limb = limb_of(v);
      const int p = int(limb % unsigned(P));
      const NttPrime pr = primes[p];
      const A ar(pr);
      T x[kE];
#pragma unroll
      for (int j = 0; j < kE; ++j) x[j] = ar.from_u64(raw[j]);
      run_passes<LOGN, INV, 0>(x, reinterpret_cast<T*>(lds), t, tw + (size_t(p) << LOGN), ar, pr, w0, [] {});
      const size_t vn = v + gridDim.x;
      if (vn < count) load_pass_twiddles<LOGN, INV, 0>(w0, t, tw + ((limb_of(vn) % unsigned(P)) << LOGN));
      store(ar, x, limb, pr);
      if (vn < count) load(raw, limb_of(vn));
    }
  } else {
    for (size_t v = blockIdx.x; v < count; v += gridDim.x) {
      if constexpr (FINISH) t = threadIdx.x + unsigned(v >> 40);
      const size_t limb = limb_of(v);
      const int p = int(limb % unsigned(P));
      const NttPrime pr = primes[p];
      const A ar(pr);
      uint64_t raw[kE];
      load(raw, limb);
      T x[kE];
#pragma unroll
      for (int j = 0; j < kE; ++j) x[j] = ar.from_u64(lifted(raw[j], ar, pr));
      ntt_regs<LOGN, INV>(x, reinterpret_cast<T*>(lds), t, tw + (size_t(p) << LOGN), ar, pr);
      store(ar, x, limb, pr);
    }
  }
}

// Few limbs (no more than CUs): one workgroup per limb on twice the threads of
// ntt_kernel, eight coefficients each.  A limb alone on its CU is bound by
// latency: with sixteen coefficients per thread a SIMD holds one wave at
// N = 4096, which issues a multiply-add every 8.8 cycles; two waves issue one
// every 4.4, and the next pass's twiddles are on their way during a pass.
// 32 limbs at N = 4096, forward and inverse: 15.9 -> 12.6 us.  Not at N = 8192, whose
// sixteen waves would name coefficient bits that the second pass needs.
constexpr int kFewLE = 3;
template <int LOGN, bool INV, class A>
__global__ void __launch_bounds__((ntt_threads<LOGN, kFewLE>()))
    ntt_few_kernel(uint64_t* __restrict__ data, size_t count, const NttPrime* __restrict__ primes,
                   const typename A::TW* __restrict__ tw, int P, const int* __restrict__ sel, int C) {
  constexpr int E = 1 << kFewLE;
  // the second pass's gap bits end where the wave bits begin
  static_assert(LOGN - kFewLE <= LOGN - Passes<LOGN, kFewLE>::WAVE_BITS);
  __shared__ __attribute__((aligned(16))) uint64_t lds[(1 << LOGN) + (1 << LOGN) / 16];
  using T = typename A::T;
  const unsigned t = threadIdx.x, v = blockIdx.x;
  if (v >= count) return;
  const size_t limb = size_t(v / unsigned(C)) * unsigned(P) + unsigned(sel[v % unsigned(C)]);
  const int p = int(limb % unsigned(P));
  const typename A::TW* tab = tw + (size_t(p) << LOGN);
  uint64_t* d = data + (limb << LOGN);
  uint64_t raw[E];
#pragma unroll
  for (int j = 0; j < E; ++j)
    raw[j] = d[INV ? inv_in_index<LOGN, kFewLE>(t, j) : fwd_in_index<LOGN, kFewLE>(t, j)];
  typename A::TW w0[(pass_tw_count<LOGN, INV, 0, kFewLE>())];
  load_pass_twiddles_e<LOGN, INV, 0, kFewLE>(w0, t, tab);
  const NttPrime pr = primes[p];
  const A ar(pr);
  T x[E];
#pragma unroll
  for (int j = 0; j < E; ++j) x[j] = ar.from_u64(raw[j]);
  run_passes_wide<LOGN, INV, 0>(x, reinterpret_cast<T*>(lds), t, tab, ar, pr, w0);
  if constexpr (!INV) {
#pragma unroll
    for (int j = 0; j < E; j += 2)
      *reinterpret_cast<ulonglong2*>(d + fwd_out_index<LOGN, kFewLE>(t, j)) =
          make_ulonglong2(ar.to_u64_fwd(x[j]), ar.to_u64_fwd(x[j + 1]));
  } else {
#pragma unroll
    for (int j = 0; j < E; ++j) d[inv_out_index<LOGN, kFewLE>(t, j)] = ar.to_u64_inv(x[j]);
  }
}

static unsigned device_cus() {
  static unsigned cached = 0;
  if (!cached) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
      cus = 256;
    cached = unsigned(cus);
  }
  return cached;
}

// Resident workgroups per CU times the CU count, cached per kernel.
template <int LOGN, bool INV, class A, bool LIFT, bool FINISH>
static unsigned persistent_grid() {
  static unsigned grid = 0;
  if (!grid) {
    int dev = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      cus = 256;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (ntt_kernel<LOGN, INV, A, LIFT, FINISH>), ntt_threads<LOGN>(),
                                                     0) !=
            hipSuccess ||
        per_cu < 1)
      per_cu = 1;
    grid = unsigned(cus * per_cu);
  }
  return grid;
}

// Number of limbs among the first `limbs` whose prime index is in sel[0..C).
static size_t subset_count(size_t limbs, int P, const int* host_sel, int C) {
  size_t count = (limbs / unsigned(P)) * unsigned(C);
  const size_t tail = limbs % unsigned(P);
  for (int c = 0; c < C; ++c) count += size_t(host_sel[c]) < tail ? 1 : 0;
  return count;
}

template <int LOGN, bool INV, class A, bool LIFT = false, bool FINISH = false>
static hipError_t launch_subset(uint64_t* data, size_t limbs, const NttDevice& d, const typename A::TW* tw,
                                const int* sel_dev, const int* sel_host, int C, hipStream_t s, NttLift lift = {},
                                NttFinish fin = {}) {
  if (!C) return hipSuccess;
  const size_t count = subset_count(limbs, d.P, sel_host, C);
  if (!count) return hipSuccess;
  if constexpr (!LIFT && !FINISH && LOGN >= 10 && LOGN <= 12) {
    if (count <= device_cus()) {
      hipLaunchKernelGGL((ntt_few_kernel<LOGN, INV, A>), dim3(unsigned(count)), dim3(ntt_threads<LOGN, kFewLE>()), 0, s,
                         data, count, d.primes, tw, d.P, sel_dev, C);
      return hipGetLastError();
    }
  }
  const dim3 block{unsigned(ntt_threads<LOGN>())};
  const dim3 grid{unsigned(std::min<size_t>(count, persistent_grid<LOGN, INV, A, LIFT, FINISH>()))};
  hipLaunchKernelGGL((ntt_kernel<LOGN, INV, A, LIFT, FINISH>), grid, block, 0, s, data, count, d.primes, tw, d.P,
                     sel_dev, C, lift, fin);
  return hipGetLastError();
}

template <class A>
struct TypeTag {
  using type = A;
};

template <int LOGN>
static hipError_t launch_ntt_n(bool inverse, uint64_t* data, size_t limbs, const NttDevice& d,
                               hipStream_t s) {
  // integer-path primes all just below a power of two: ArPM; all below 2^60:
  // the lazy transforms (ArU64L)
  const auto u64 = [&](auto tag, bool inv) {
    using A = typename decltype(tag)::type;
    return inv ? launch_subset<LOGN, true, A>(data, limbs, d, d.tw_inv_u, d.sel_u64, d.host_sel_u64, d.n_u64, s)
               : launch_subset<LOGN, false, A>(data, limbs, d, d.tw_fwd_u, d.sel_u64, d.host_sel_u64, d.n_u64, s);
  };
  hipError_t e;
  if (inverse)
    e = launch_subset<LOGN, true, ArF64T>(data, limbs, d, d.tw_inv_f, d.sel_f64, d.host_sel_f64, d.n_f64, s);
  else
    e = launch_subset<LOGN, false, ArF64T>(data, limbs, d, d.tw_fwd_f, d.sel_f64, d.host_sel_f64, d.n_f64, s);
  if (e == hipSuccess && d.n_u64) e = d.pm_u64 ? u64(TypeTag<ArPM>{}, inverse) : d.lazy_u64 ? u64(TypeTag<ArU64L>{}, inverse) : u64(TypeTag<ArU64>{}, inverse);
  return e;
}

// The lifted transform at N = 16384 by half limbs.  A whole limb's exchange
// buffer (136 KiB) leaves one workgroup on a CU, whose loads, stages and stores
// follow one another; two half-limb workgroups (68 KiB, 512 threads) fill the
// same registers and run each other's gaps.  Stage 0 pairs the halves, so each
// workgroup forms it from the ring words of both and keeps its own side - the
// ring is not written, so there is no order between the two.  When the ring
// block reaches half the limb at most (kReversedLow) the upper half is
// zero, the stage changes nothing and costs nothing.  Every limb half of a ring
// block runs on one XCD (workgroup % 8), whose L2 then holds the block.
// 7,296 limbs (19 blocks x 64 columns x 6 primes), width 8192: 660 us by whole
// limbs, 560 to 601 here: VALU busy 75% of the launch, 251 M instructions.
constexpr int kHalfLog = 13;
enum HalfInput { kPlain, kReversed, kReversedLow };  // width 0, above N / 2, up to N / 2
template <class A, HalfInput IN>
__global__ void __launch_bounds__(1 << (kHalfLog - kLogE)) __attribute__((amdgpu_waves_per_eu(4)))
    ntt_lift_half_kernel(uint64_t* __restrict__ out, size_t blocks, const NttPrime* __restrict__ primes,
                         const typename A::TW* __restrict__ tw, int P, const int* __restrict__ sel, int C,
                         NttLift lift) {
  constexpr unsigned kHalf = 1u << kHalfLog;
  __shared__ __attribute__((aligned(16))) uint64_t lds[kHalf + kHalf / 16];
  const unsigned items = 2 * unsigned(C);
  const size_t total = (blocks + 7) / 8 * 8 * items;
  for (size_t v = blockIdx.x; v < total; v += gridDim.x) {  // gridDim is a multiple of 8
    const size_t seq = v >> 3, b = seq / items * 8 + (v & 7);
    if (b >= blocks) continue;
    const unsigned t = threadIdx.x + unsigned(v >> 40);  // recomputed per item: no index kept across the loop
    const unsigned sub = unsigned(seq % items), h = sub & 1u, p = unsigned(sel[sub >> 1]);
    const NttPrime pr = primes[p];
    const A ar(pr);
    // coefficient z is ring[b][z], or ring[b][width - 1 - z] and zero from width on
    const typename A::TW* tab = tw + (size_t(p) << (kHalfLog + 1));
    const unsigned z0 = fwd_in_index<kHalfLog>(t, 0), width = unsigned(lift.width);
    const uint64_t* first = IN == kPlain ? lift.ring + (b << (kHalfLog + 1)) + z0
                                         : lift.ring + b * lift.width + lift.width - 1 - (long long)z0;
    const auto word = [&](unsigned d) {  // of coefficient z0 + d
      if constexpr (IN == kPlain)
        return first[d];
      else
        return z0 + d < width ? *(first - d) : 0;
    };
    uint64_t x[kE];
#pragma unroll
    for (int j = 0; j < kE; ++j) x[j] = word(PassMap<kHalfLog, false, 0>::reg_field(j));
#pragma unroll
    for (int j = 0; j < kE; ++j) x[j] = ar.from_u64(lift_word(ar, x[j], pr));
    if constexpr (IN != kReversedLow) {
      const typename A::TW w = load_invariant(tab + 1);
#pragma unroll
      for (int j = 0; j < kE; ++j) {
        uint64_t y = ar.from_u64(lift_word(ar, word(PassMap<kHalfLog, false, 0>::reg_field(j) + kHalf), pr));
        ar.template fwd_at<true>(0, x[j], y, w);
        x[j] = h ? y : x[j];
        if ((j & 3) == 3) __builtin_amdgcn_sched_barrier(0);  // four words of the other half in registers at a time
      }
    }
    run_part_passes<kHalfLog + 1, kHalfLog, 0>(x, lds, t, h, tab, ar);
    uint64_t* o = out + ((b * unsigned(P) + p) << (kHalfLog + 1)) + size_t(h) * kHalf;
#pragma unroll
    for (int j = 0; j < kE; j += 2)
      *reinterpret_cast<ulonglong2*>(o + fwd_out_index<kHalfLog>(t, j)) =
          make_ulonglong2(ar.to_u64_fwd(x[j]), ar.to_u64_fwd(x[j + 1]));
    __syncthreads();  // the next half's first exchange reuses the LDS
  }
}

template <class A, HalfInput IN>
static hipError_t launch_lift_half(uint64_t* out, size_t blocks, const NttDevice& d, NttLift lift, hipStream_t s) {
  const unsigned resident = (device_cus() + 7) / 8 * 8 * 2;
  const size_t total = (blocks + 7) / 8 * 8 * 2 * size_t(d.n_u64);
  hipLaunchKernelGGL((ntt_lift_half_kernel<A, IN>), dim3(unsigned(std::min<size_t>(total, resident))),
                     dim3(1 << (kHalfLog - kLogE)), 0, s, out, blocks, d.primes, d.tw_fwd_u, d.P, d.sel_u64, d.n_u64,
                     lift);
  return hipGetLastError();
}

template <int LOGN>
static hipError_t launch_ntt_lift_n(const uint64_t* ring, size_t width, uint64_t* out, size_t limbs,
                                    const NttDevice& d, hipStream_t s) {
  const NttLift lift{ring, width};
  const auto go = [&](auto tag) {
    if constexpr (LOGN == kHalfLog + 1) {
      using A = typename decltype(tag)::type;
      const size_t blocks = limbs / unsigned(d.P);
      return !width ? launch_lift_half<A, kPlain>(out, blocks, d, lift, s)
             : width > (size_t(1) << kHalfLog) ? launch_lift_half<A, kReversed>(out, blocks, d, lift, s)
                                               : launch_lift_half<A, kReversedLow>(out, blocks, d, lift, s);
    } else {
      return launch_subset<LOGN, false, typename decltype(tag)::type, true>(out, limbs, d, d.tw_fwd_u, d.sel_u64,
                                                                            d.host_sel_u64, d.n_u64, s, lift);
    }
  };
  return d.pm_u64 ? go(TypeTag<ArPM>{}) : d.lazy_u64 ? go(TypeTag<ArU64L>{}) : go(TypeTag<ArU64>{});
}

// Every prime on the integer path: the lift is done by the transform's loads.
// With float-path primes (whose kernel has no registers left for the lift's
// arithmetic) the lift kernel writes the limbs first and the transform runs
// in place.
hipError_t launch_ntt_lift(const uint64_t* ring, size_t width, uint64_t* out, size_t blocks, const PrimeList& pl,
                           const NttDevice& d, hipStream_t s) {
  const size_t limbs = blocks * size_t(d.P);
  if (limbs == 0) return hipSuccess;
  if (d.n_f64) {
    const hipError_t e = launch_lift59(ring, out, blocks, d.log_n, width, pl, s);
    return e == hipSuccess ? launch_ntt(false, out, limbs, d, s) : e;
  }
  switch (d.log_n) {
    case 4: return launch_ntt_lift_n<4>(ring, width, out, limbs, d, s);
    case 5: return launch_ntt_lift_n<5>(ring, width, out, limbs, d, s);
    case 6: return launch_ntt_lift_n<6>(ring, width, out, limbs, d, s);
    case 7: return launch_ntt_lift_n<7>(ring, width, out, limbs, d, s);
    case 8: return launch_ntt_lift_n<8>(ring, width, out, limbs, d, s);
    case 9: return launch_ntt_lift_n<9>(ring, width, out, limbs, d, s);
    case 10: return launch_ntt_lift_n<10>(ring, width, out, limbs, d, s);
    case 11: return launch_ntt_lift_n<11>(ring, width, out, limbs, d, s);
    case 12: return launch_ntt_lift_n<12>(ring, width, out, limbs, d, s);
    case 13: return launch_ntt_lift_n<13>(ring, width, out, limbs, d, s);
    case 14: return launch_ntt_lift_n<14>(ring, width, out, limbs, d, s);
    default: return hipErrorInvalidValue;
  }
}

template <int LOGN>
static hipError_t launch_ntt_finish_n(uint64_t* data, size_t limbs, const NttDevice& d, NttFinish fin, hipStream_t s) {
  hipError_t e = launch_subset<LOGN, true, ArF64T, false, true>(data, limbs, d, d.tw_inv_f, d.sel_f64, d.host_sel_f64,
                                                                d.n_f64, s, {}, fin);
  const auto go = [&](auto tag) {
    return launch_subset<LOGN, true, typename decltype(tag)::type, false, true>(data, limbs, d, d.tw_inv_u, d.sel_u64,
                                                                                d.host_sel_u64, d.n_u64, s, {}, fin);
  };
  if (e == hipSuccess && d.n_u64)
    e = d.pm_u64 ? go(TypeTag<ArPM>{}) : d.lazy_u64 ? go(TypeTag<ArU64L>{}) : go(TypeTag<ArU64>{});
  return e;
}

hipError_t launch_ntt_finish(uint64_t* data, const uint64_t* scaled, uint64_t* out, size_t slots, size_t width,
                             const NttDevice& d, hipStream_t s) {
  const size_t limbs = slots * 2 * size_t(d.P);
  if (limbs == 0) return hipSuccess;
  const NttFinish fin{out, scaled, unsigned(width - 1)};
  switch (d.log_n) {
    case 4: return launch_ntt_finish_n<4>(data, limbs, d, fin, s);
    case 5: return launch_ntt_finish_n<5>(data, limbs, d, fin, s);
    case 6: return launch_ntt_finish_n<6>(data, limbs, d, fin, s);
    case 7: return launch_ntt_finish_n<7>(data, limbs, d, fin, s);
    case 8: return launch_ntt_finish_n<8>(data, limbs, d, fin, s);
    case 9: return launch_ntt_finish_n<9>(data, limbs, d, fin, s);
    case 10: return launch_ntt_finish_n<10>(data, limbs, d, fin, s);
    case 11: return launch_ntt_finish_n<11>(data, limbs, d, fin, s);
    case 12: return launch_ntt_finish_n<12>(data, limbs, d, fin, s);
    case 13: return launch_ntt_finish_n<13>(data, limbs, d, fin, s);
    case 14: return launch_ntt_finish_n<14>(data, limbs, d, fin, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_ntt(bool inverse, uint64_t* data, size_t limbs, const NttDevice& d, hipStream_t s) {
  if (limbs == 0) return hipSuccess;
  switch (d.log_n) {
    case 4: return launch_ntt_n<4>(inverse, data, limbs, d, s);
    case 5: return launch_ntt_n<5>(inverse, data, limbs, d, s);
    case 6: return launch_ntt_n<6>(inverse, data, limbs, d, s);
    case 7: return launch_ntt_n<7>(inverse, data, limbs, d, s);
    case 8: return launch_ntt_n<8>(inverse, data, limbs, d, s);
    case 9: return launch_ntt_n<9>(inverse, data, limbs, d, s);
    case 10: return launch_ntt_n<10>(inverse, data, limbs, d, s);
    case 11: return launch_ntt_n<11>(inverse, data, limbs, d, s);
    case 12: return launch_ntt_n<12>(inverse, data, limbs, d, s);
    case 13: return launch_ntt_n<13>(inverse, data, limbs, d, s);
    case 14: return launch_ntt_n<14>(inverse, data, limbs, d, s);
    default: return hipErrorInvalidValue;
  }
}

// Products of a batch of small polynomials u with both components of a
// resident public key, in coefficient form (enc0.cu:99-114 before its ModDown):
//   prod[e][c][t] = INTT(NTT(u[e][t]) (.) pk[c][t]),  u[e][t] at samples + e stride + t N.
// One workgroup per (encryption, prime): the forward transform's registers are
// the inverse transform's, position by position, so the product happens in
// registers and the transform of u goes to memory only to be read again for the
// second component (`work`, each thread its own words).  The key is held as
// ArPM's pairs, and the forward values need no reduction before the product.
// 64 encryptions at N = 16384, seven 60-bit primes, us: a copy of u, its
// transform, the products and the inverse as launches of their own 211, 162 here.
// SPLIT: a workgroup per component as well, each transforming u for itself - two
// transforms in series instead of three, while even that leaves CUs idle (two
// encryptions, us: launches of their own 61, three in series 64, SPLIT 43).
template <int LOGN, bool SPLIT>
__global__ void __launch_bounds__(ntt_threads<LOGN>())
    enc0_products_kernel(const uint64_t* __restrict__ samples, size_t stride, const ulonglong2* __restrict__ pk,
                         uint64_t* __restrict__ work, uint64_t* __restrict__ prod, size_t count,
                         const NttPrime* __restrict__ primes, const ulonglong2* __restrict__ tw_fwd,
                         const ulonglong2* __restrict__ tw_inv, unsigned K) {
  __shared__ __attribute__((aligned(16))) uint64_t lds[(1 << LOGN) + (1 << LOGN) / 16];
  constexpr unsigned TH = ntt_threads<LOGN>();
  for (size_t i = blockIdx.x; i < (SPLIT ? 2 : 1) * count * K; i += gridDim.x) {
    const unsigned t = threadIdx.x + unsigned(i >> 40);  // recomputed per item: no index kept across the loop
    const size_t v = SPLIT ? i / 2 : i, e = v / K;
    const unsigned p = unsigned(v % K);
    const NttPrime pr = primes[p];
    const ArPM ar(pr);
    uint64_t x[kE];
    const uint64_t* u = samples + e * stride + (size_t(p) << LOGN);
#pragma unroll
    for (int j = 0; j < kE; ++j) x[j] = u[fwd_in_index<LOGN>(t, j)];
    ntt_regs<LOGN, false>(x, lds, t, tw_fwd + (size_t(p) << LOGN), ar, pr);
    uint64_t* own = work + (v << LOGN) + t;
    if constexpr (!SPLIT) {
#pragma unroll
      for (int j = 0; j < kE; ++j) own[unsigned(j) * TH] = x[j];
    }
    const unsigned c_first = SPLIT ? unsigned(i & 1) : 0u, c_end = SPLIT ? c_first + 1 : 2u;
#pragma unroll 1
    for (unsigned c = c_first; c < c_end; ++c) {
      const unsigned t2 = t + unsigned((v + c) >> 40);
      if (!SPLIT && c) {
#pragma unroll
        for (int j = 0; j < kE; ++j) x[j] = own[unsigned(j) * TH];
      }
      const ulonglong2* k = pk + (size_t(c * K + p) << LOGN);
#pragma unroll
      for (int j = 0; j < kE; ++j) {
        const ulonglong2 w = k[fwd_out_index<LOGN>(t2, j)];
        x[j] = mul_pm(x[j], w.x, w.y, ar.c2);  // below 3M, the inverse's input bound is 4M
        if ((j & 3) == 3) __builtin_amdgcn_sched_barrier(0);  // four pairs in registers at a time
      }
      // no barrier between the transforms: the forward one's last exchanges and
      // the inverse one's first stay in the same wave's part of the LDS, and an
      // exchange across waves begins and ends with one
      ntt_regs<LOGN, true>(x, lds, t2, tw_inv + (size_t(p) << LOGN), ar, pr);
      uint64_t* out = prod + (((e * 2 + c) * K + p) << LOGN);
#pragma unroll
      for (int j = 0; j < kE; ++j) out[inv_out_index<LOGN>(t2, j)] = ar.to_u64_inv(x[j]);
    }
  }
}

template <int LOGN>
static hipError_t launch_enc0_products_n(const uint64_t* samples, size_t stride, const ulonglong2* pk, uint64_t* work,
                                         uint64_t* prod, size_t count, const NttDevice& d, hipStream_t s) {
  const size_t items = count * size_t(d.P);
  const bool split = 2 * items <= device_cus();
  const unsigned grid =
      unsigned(std::min<size_t>((split ? 2 : 1) * items, persistent_grid<LOGN, true, ArPM, false, false>()));
  const auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(ntt_threads<LOGN>()), 0, s, samples, stride, pk, work, prod, count,
                       d.primes, d.tw_fwd_u, d.tw_inv_u, unsigned(d.P));
  };
  split ? go(enc0_products_kernel<LOGN, true>) : go(enc0_products_kernel<LOGN, false>);
  return hipGetLastError();
}

hipError_t launch_enc0_products(const uint64_t* samples, size_t stride, const ulonglong2* pk, uint64_t* work,
                                uint64_t* prod, size_t count, const NttDevice& d, hipStream_t s) {
  if (count == 0) return hipSuccess;
  switch (d.log_n) {
    case 4: return launch_enc0_products_n<4>(samples, stride, pk, work, prod, count, d, s);
    case 5: return launch_enc0_products_n<5>(samples, stride, pk, work, prod, count, d, s);
    case 6: return launch_enc0_products_n<6>(samples, stride, pk, work, prod, count, d, s);
    case 7: return launch_enc0_products_n<7>(samples, stride, pk, work, prod, count, d, s);
    case 8: return launch_enc0_products_n<8>(samples, stride, pk, work, prod, count, d, s);
    case 9: return launch_enc0_products_n<9>(samples, stride, pk, work, prod, count, d, s);
    case 10: return launch_enc0_products_n<10>(samples, stride, pk, work, prod, count, d, s);
    case 11: return launch_enc0_products_n<11>(samples, stride, pk, work, prod, count, d, s);
    case 12: return launch_enc0_products_n<12>(samples, stride, pk, work, prod, count, d, s);
    case 13: return launch_enc0_products_n<13>(samples, stride, pk, work, prod, count, d, s);
    case 14: return launch_enc0_products_n<14>(samples, stride, pk, work, prod, count, d, s);
    default: return hipErrorInvalidValue;
  }
}

// ArPM's pairs of `words` residues [..][P][N] (a plan's resident key).
__global__ void pm_pairs_kernel(const uint64_t* __restrict__ in, ulonglong2* __restrict__ out, BarrettList bl,
                                int log_n, size_t words) {
  for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < words; i += size_t(gridDim.x) * blockDim.x) {
    const uint64_t w = in[i];
    out[i] = make_ulonglong2(pm_split(w), pm_split(mul_barrett(w, 1ull << 32, bl.m[(i >> log_n) % unsigned(bl.count)])));
  }
}

hipError_t launch_pm_pairs(const uint64_t* in, ulonglong2* out, size_t words, int log_n, const Barrett* m, int primes,
                           hipStream_t s) {
  BarrettList bl{};
  for (int i = 0; i < primes; ++i) bl.m[i] = m[i];
  bl.count = primes;
  const unsigned blocks = unsigned(std::min<size_t>((words + 255) / 256, 4096));
  hipLaunchKernelGGL(pm_pairs_kernel, dim3(blocks), dim3(256), 0, s, in, out, bl, log_n, words);
  return hipGetLastError();
}

// Pointwise product with a per-prime operand in Shoup form (client_dyadic,
// ntt.cu:55-57): data[l][k] = data[l][k] * key[l % P][k] mod q.
__global__ void dyadic_shoup_kernel(uint64_t* __restrict__ data, const ulonglong2* __restrict__ key,
                                    const NttPrime* __restrict__ primes, int P, int log_n, size_t words) {
  for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < words; i += size_t(gridDim.x) * blockDim.x) {
    const size_t limb = i >> log_n;
    const int p = int(limb % unsigned(P));
    const ulonglong2 w = key[(size_t(p) << log_n) + (i & ((size_t(1) << log_n) - 1))];
    data[i] = mul_shoup(data[i], w.x, w.y, primes[p].q);
  }
}

hipError_t launch_dyadic_shoup(uint64_t* data, const ulonglong2* key, const NttDevice& d, size_t words,
                               hipStream_t s) {
  if (!words) return hipSuccess;
  const unsigned blocks = unsigned(std::min<size_t>((words + 255) / 256, 65536));
  hipLaunchKernelGGL(dyadic_shoup_kernel, dim3(blocks), dim3(256), 0, s, data, key, d.primes, d.P, d.log_n, words);
  return hipGetLastError();
}

}  // namespace praghip
