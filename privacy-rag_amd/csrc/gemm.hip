// Party-local share GEMM over Z_2^64 on the i8 matrix cores of gfx950.
//
//   y[m][n] = ((sum_k x[m][k] * w[n][k]) << s_n)  mod 2^mask_bits
//
// (bfv_matrix.inc:101-105 / 156-160 / 177-182: the reference runs this as a
// scalar triple loop on the protocol thread.)
//
// Exactness.  Each u64 share is split into its 8 bytes b_d and re-centred as
// signed digits a_d = b_d - 128 (one XOR with 0x80 per byte), so that
//   x = sum_d (a_d + 128) 256^d
//   sum_k x w = sum_d 256^d (sum_k a_d w)  +  0x8080808080808080 * sum_k w   (mod 2^64).
// Every digit product a_d * w fits i8 x i8, and each column of partial sums
// fits the i32 accumulator (|a_d w| <= 2^14, K < 2^17).  int32 weights in
// [-0x808080, 0x7F7F7F] (the reference f12 domain is |w| <= 2^20) are split
// into three balanced signed bytes w = sum_e w_e 256^e and run as one pass per
// weight byte, each pass shifting its contribution by 8e and accumulating
// mod 2^64.
//
// Tiling.  One MFMA v_mfma_i32_32x32x32_i8 covers 32 "digit rows" = 4 share
// rows x 8 digits (32x32 accumulator layout: lane l, register r -> column l%32,
// row 8(r/4) + 4(l/32) + r%4), so that a lane holds, for its column, four
// digits of each share row and the digit sum is formed in registers with one
// exchange across the wave's halves.  Large products run as 32-row x 128- or
// 192-column tiles (LDS DMA, or staged through registers), products of few
// rows on a kernel that splits K over the waves of a workgroup.
#include "gemm_rule.hpp"
#include "kernels.hpp"
#include "praghip.h"

#include <vector>

namespace praghip {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kPitch = 80, kThreads = 256;

// o_d byte e = a_e byte d, for four dwords a0..a3.
__device__ __forceinline__ void transpose4(uint32_t a0, uint32_t a1, uint32_t a2, uint32_t a3, uint32_t& o0,
                                           uint32_t& o1, uint32_t& o2, uint32_t& o3) {
  const uint32_t p0 = __builtin_amdgcn_perm(a1, a0, 0x05010400u);
  const uint32_t p1 = __builtin_amdgcn_perm(a1, a0, 0x07030602u);
  const uint32_t p2 = __builtin_amdgcn_perm(a3, a2, 0x05010400u);
  const uint32_t p3 = __builtin_amdgcn_perm(a3, a2, 0x07030602u);
  o0 = __builtin_amdgcn_perm(p2, p0, 0x05040100u);
  o1 = __builtin_amdgcn_perm(p2, p0, 0x07060302u);
  o2 = __builtin_amdgcn_perm(p3, p1, 0x05040100u);
  o3 = __builtin_amdgcn_perm(p3, p1, 0x07060302u);
}

// Balanced signed byte e (e < 3) of a weight in [-0x808080, 0x7F7F7F].
__device__ __forceinline__ int weight_digit(int w, int e) {
  for (int i = 0; i < e; ++i) {
    const int lo = (int)(int8_t)(w & 0xff);
    w = (w - lo) >> 8;
  }
  return (int)(int8_t)(w & 0xff);
}

// Global tile of one K step held in registers: the share loader's 8 u64 and
// the weight loader's 32 weight bytes (as 8 words).
struct TileRegs {
  uint64_t xs[8];
  uint32_t wb[8];
};

__device__ __forceinline__ void load_tile(TileRegs& tr, const uint64_t* __restrict__ xrow, bool x_row_ok,
                                          const int8_t* __restrict__ wrow, bool w_row_ok, int k0, int K, int ak, int wk,
                                          int w_vec) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int kk = k0 + ak + e;
    tr.xs[e] = (x_row_ok && kk < K) ? xrow[kk] : 0;
  }
  const int kk = k0 + wk;
  if (w_row_ok && kk + 32 <= K && w_vec) {
    const uint4 a = *reinterpret_cast<const uint4*>(wrow + kk);
    const uint4 b = *reinterpret_cast<const uint4*>(wrow + kk + 16);
    tr.wb[0] = a.x; tr.wb[1] = a.y; tr.wb[2] = a.z; tr.wb[3] = a.w;
    tr.wb[4] = b.x; tr.wb[5] = b.y; tr.wb[6] = b.z; tr.wb[7] = b.w;
  } else {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      uint32_t word = 0;
#pragma unroll
      for (int bb = 0; bb < 4; ++bb) {
        const int kq = kk + 4 * q + bb;
        const uint32_t byte = (w_row_ok && kq < K) ? uint8_t(wrow[kq]) : 0u;
        word |= byte << (8 * bb);
      }
      tr.wb[q] = word;
    }
  }
}

// ------------------------------------------------------------- VALU form
// The same product with VALU dot products instead of the matrix cores: the
// tiles are staged as digit planes of the offset-binary share bytes (byte
// transpose with v_perm) and int8 weight rows, and each thread forms a 4 x 4
// block of outputs with v_dot4_i32_i8, one per (row, column, digit) and four
// k.  It exists as the measured alternative to the MFMA kernels (int8
// weights).
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
    share_gemm_valu_kernel(const uint64_t* __restrict__ x, const int8_t* __restrict__ w,
                           const int8_t* __restrict__ shifts, uint64_t* __restrict__ y, int M, int K, int N,
                           uint64_t mask, int w_vec) {
  __shared__ __attribute__((aligned(16))) uint8_t a_lds[8][kBM][kPitch];
  __shared__ __attribute__((aligned(16))) uint8_t w_lds[kBN][kPitch];
  __shared__ int csum[kThreads];
  const int t = threadIdx.x;
  const int m0 = blockIdx.y * kBM, n0 = blockIdx.x * kBN;
  const int ar = t >> 3, ak = (t & 7) * 8, wr = t >> 1, wk = (t & 1) * 32;
  const int rg = t >> 5, cg = t & 31;  // rows rg + 8i, columns cg + 32j
  int colsum = 0;
  int acc[4][4][8];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int d = 0; d < 8; ++d) acc[i][j][d] = 0;
  const bool x_row_ok = (m0 + ar) < M, w_row_ok = (n0 + wr) < N;
  const uint64_t* xrow = x + size_t(m0 + ar) * K;
  const int8_t* wrow = w + size_t(n0 + wr) * K;
  TileRegs tr;
  load_tile(tr, xrow, x_row_ok, wrow, w_row_ok, 0, K, ak, wk, w_vec);
  for (int k0 = 0; k0 < K; k0 += kBK) {
    uint32_t d[16];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      d[2 * e] = uint32_t(tr.xs[e]) ^ 0x80808080u;
      d[2 * e + 1] = uint32_t(tr.xs[e] >> 32) ^ 0x80808080u;
    }
    uint32_t o[4][4];
    transpose4(d[0], d[2], d[4], d[6], o[0][0], o[0][1], o[0][2], o[0][3]);
    transpose4(d[8], d[10], d[12], d[14], o[1][0], o[1][1], o[1][2], o[1][3]);
    transpose4(d[1], d[3], d[5], d[7], o[2][0], o[2][1], o[2][2], o[2][3]);
    transpose4(d[9], d[11], d[13], d[15], o[3][0], o[3][1], o[3][2], o[3][3]);
#pragma unroll
    for (int dg = 0; dg < 4; ++dg) {
      *reinterpret_cast<uint2*>(&a_lds[dg][ar][ak]) = make_uint2(o[0][dg], o[1][dg]);
      *reinterpret_cast<uint2*>(&a_lds[dg + 4][ar][ak]) = make_uint2(o[2][dg], o[3][dg]);
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) colsum = __builtin_amdgcn_sdot4(int(tr.wb[q]), 0x01010101, colsum, false);
    *reinterpret_cast<uint4*>(&w_lds[wr][wk]) = make_uint4(tr.wb[0], tr.wb[1], tr.wb[2], tr.wb[3]);
    *reinterpret_cast<uint4*>(&w_lds[wr][wk + 16]) = make_uint4(tr.wb[4], tr.wb[5], tr.wb[6], tr.wb[7]);
    __syncthreads();
#pragma unroll 1
    for (int kk = 0; kk < kBK; kk += 4) {
      int wv[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) wv[j] = *reinterpret_cast<const int*>(&w_lds[cg + 32 * j][kk]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int dg = 0; dg < 8; ++dg) {
          const int xv = *reinterpret_cast<const int*>(&a_lds[dg][rg + 8 * i][kk]);
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[i][j][dg] = __builtin_amdgcn_sdot4(xv, wv[j], acc[i][j][dg], false);
        }
      }
    }
    __syncthreads();
    // the next step's tile is loaded after the dot products (the 128
    // accumulators leave no registers to hold it during them)
    if (k0 + kBK < K) load_tile(tr, xrow, x_row_ok, wrow, w_row_ok, k0 + kBK, K, ak, wk, w_vec);
  }
  csum[t] = colsum;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int cl = cg + 32 * j, col = n0 + cl;
    if (col >= N) continue;
    const int64_t s_n = int64_t(csum[2 * cl]) + int64_t(csum[2 * cl + 1]);
    const uint64_t corr = 0x8080808080808080ull * uint64_t(s_n);
    const int sh = shifts ? int(shifts[col]) : 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = m0 + rg + 8 * i;
      if (row >= M) continue;
      uint64_t v = corr;
#pragma unroll
      for (int dg = 0; dg < 8; ++dg) v += uint64_t(int64_t(acc[i][j][dg])) << (8 * dg);
      v = sh < 64 ? (v << sh) : 0;
      y[size_t(row) * N + col] = v & mask;
    }
  }
}

hipError_t launch_share_gemm_valu(const uint64_t* x, const int8_t* w, const int8_t* shifts, uint64_t* y, int M,
                                  int K, int N, int mask_bits, hipStream_t s) {
  const uint64_t mask = mask_bits >= 64 ? ~0ull : ((1ull << mask_bits) - 1);
  const int w_vec = (K % 16 == 0) && (reinterpret_cast<uintptr_t>(w) % 16 == 0);
  const dim3 grid((N + kBN - 1) / kBN, (M + kBM - 1) / kBM);
  hipLaunchKernelGGL(share_gemm_valu_kernel, grid, dim3(kThreads), 0, s, x, w, shifts, y, M, K, N, mask, w_vec);
  return hipGetLastError();
}

// ---------------------------------------------------------------- DMA path
// For K % 64 == 0 and int8 weights (16-byte aligned x, w): the raw tiles go
// from global memory straight into a three-stage LDS ring with
// global_load_lds_dwordx4 (no registers, no wait until the stage is used), so
// the next two K steps' loads are in flight during the current step's MFMAs;
// two workgroups per CU overlap each other's waits as well.  The MFMA share
// operands are read from the raw u64 tile with ds_read_b64_tr_b8, which hands
// every lane one byte position of eight words: with the eight words of a row
// k..k+7 as the source, lane i of each 8-lane half of a 16-lane group receives
// digit i of those eight shares (the byte transpose is done by the LDS read,
// with no VALU shuffle, no digit-plane copy and no second barrier per step).
//
// MFMA rows of one 32x32x32 product: lane l of the A operand is digit l % 8 of
// share row (l % 32) / 8, so a lane's 16 accumulator registers hold, for its
// column, digits 4(l/32)..4(l/32)+3 of four share rows; the two halves of the
// wave add their digit sums with one cross-half exchange.
//
// LDS: raw shares [3][32 rows][512 B] with the 16-byte chunk c of row r at
// chunk c ^ 4(r & 7) (each 8-word read of a row stays one 64-byte block, and
// the four rows of one read land on distinct banks), weights [3][128 rows][64 B]
// with chunk c of row r at c ^ wt_swizzle(r).  DMA writes 64 lanes x 16 bytes in
// order, so each lane loads the global chunk that belongs at its LDS slot.
constexpr int kRawRow = kBK * 8;  // bytes of one raw share row per step

// 16 bytes per lane from global memory straight into LDS at M0 + lane * 16
// (global_load_lds_dwordx4).  Issued from inline asm, so the compiler adds no
// wait of its own for it: the caller waits with s_waitcnt vmcnt(0) before any
// wave reads what was loaded.  The LDS DMA reads M0 one wait state after the
// scalar write that sets it (the compiler's own global_load_lds always leaves
// one instruction there); the compiler cannot see that dependency into the
// asm, so the asm starts with s_nop 0.
__device__ __forceinline__ void dma16(const void* src, void* lds_wave_base) {
  const unsigned lds = unsigned(reinterpret_cast<uintptr_t>((void __attribute__((address_space(3)))*)(lds_wave_base)));
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "{m0}"(__builtin_amdgcn_readfirstlane(lds))
               : "memory");
}

// Byte offset of share word k of raw row r in a stage buffer.
__device__ __forceinline__ int raw_offset(int r, int k) {
  return r * kRawRow + ((((k >> 1) ^ (4 * (r & 7)))) << 4) + ((k & 1) << 3);
}

// Chunk swizzle of weight row r (64-byte rows, four 16-byte chunks): 16-byte
// reads of 8 consecutive rows land on 8 distinct 16-byte bank slots of a
// 128-byte bank line, and those of rows r, r + 4, r + 8, r + 12 on 4 distinct
// slots of a 256-byte one (bits: 2 (r/4 % 2) + (r/2 % 2 ^ r/8 % 2)).
__device__ __forceinline__ int wt_swizzle(int r) { return 2 * ((r >> 2) & 1) + (((r >> 1) ^ (r >> 3)) & 1); }

typedef int v2i __attribute__((ext_vector_type(2)));

// Eight bytes of the LDS transpose read at byte offset `off` of `base`.
__device__ __forceinline__ v2i tr8(const uint8_t* base, int off) {
  return __builtin_amdgcn_ds_read_tr8_b64_v2i32((v2i __attribute__((address_space(3)))*)(base + off));
}

// One K step of the DMA path on stage buffers (raw, wt); the next step's DMAs
// go to (raw_n, wt_n).  Distinct __shared__ objects per stage let the
// compiler see that this step's LDS reads do not depend on the DMAs just
// issued into the other stage (it would otherwise wait for them).
struct DmaCtx {
  const uint8_t* xsrc[4];
  const int8_t* wsrc[3];
  int wave, i, khalf, wm, wn, tr_row, tr_k;
  // operand read offsets within a stage: share word run h (k + 8h) of row
  // block 0 at K step 0 is a_off[h]; row block rb, K step ks adds
  // 2048 rb + 256 (ks ^ (rb & 1)).  Weight chunk of K step ks for block 0 is
  // w_off[ks]; block cb adds 2048 cb.  (raw_offset and wt_swizzle, with the
  // lane-independent parts moved into immediates.)
  int a_off[2], w_off[2];
};

// CB 32-column blocks per wave: a workgroup tile is 32 share rows x 64 CB
// columns (waves 2 x 2, each 16 rows x 32 CB columns).
template <int CB, class RAW, class WT>
__device__ __forceinline__ void dma_issue(const DmaCtx& c, int k0, RAW& raw, WT& wt) {
#pragma unroll
  for (int j = 0; j < 4; ++j) dma16(c.xsrc[j] + size_t(k0) * 8, &raw[(2 * (4 * c.wave + j)) * kRawRow]);
#pragma unroll
  for (int j = 0; j < CB; ++j) dma16(c.wsrc[j] + k0, &wt[(16 * (CB * c.wave + j)) * kBK]);
}

// One K step of MFMAs on stage buffers (raw, wt).
template <int CB, class RAW, class WT>
__device__ __forceinline__ void mfma_step(const DmaCtx& c, const RAW& raw, const WT& wt, int (&colsum)[CB],
                                          v16i (&acc)[4][CB]) {
  // ---- every operand of the step first (16 transpose reads, 2 CB weight
  // reads), so that the MFMAs then issue back to back behind one LDS wait
  v4i aop[kBK / 32][4], bop[kBK / 32][CB];
#pragma unroll
  for (int ks = 0; ks < kBK / 32; ++ks) {
    const int chunk = ks * 2 + c.khalf;  // logical 16-byte chunk of the weight rows
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      const int row = c.wn * 32 * CB + cb * 32 + c.i;
      bop[ks][cb] = *reinterpret_cast<const v4i*>(&wt[row * kBK + ((chunk ^ wt_swizzle(row)) * 16)]);
    }
    const int k = ks * 32 + c.tr_k;
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
      const int r = c.wm * 16 + rb * 4 + c.tr_row;
      const v2i lo = tr8(raw, raw_offset(r, k)), hi = tr8(raw, raw_offset(r, k + 8));
      aop[ks][rb] = v4i{lo.x, lo.y, hi.x, hi.y};
    }
  }
  // ---- MFMA over the two 32-wide K steps
#pragma unroll
  for (int ks = 0; ks < kBK / 32; ++ks) {
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
      // offset-binary digits: a_d = b_d - 128
      const v4i a = aop[ks][rb] ^ int(0x80808080u);
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
        acc[rb][cb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, bop[ks][cb], acc[rb][cb], 0, 0, 0);
    }
  }
  // ---- column sums from the weight operands already in registers (lanes l
  // and l ^ 32 hold the two halves of each row's K chunk; VALU work beside
  // the MFMAs)
#pragma unroll
  for (int ks = 0; ks < kBK / 32; ++ks)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int e = 0; e < 4; ++e) colsum[cb] = __builtin_amdgcn_sdot4(bop[ks][cb][e], 0x01010101, colsum[cb], false);
}

// Three stages: step s computes on stage s % 3 while the DMAs of steps s + 1
// (issued one step earlier) and s + 2 (issued here, into the stage step s - 1
// read) are in flight.
template <int CB, class RAW, class WT, class RAWN, class WTN>
__device__ __forceinline__ void dma_step(const DmaCtx& c, bool ahead, bool next, int k_next, const RAW& raw,
                                         const WT& wt, RAWN& raw_n, WTN& wt_n, int (&colsum)[CB],
                                         v16i (&acc)[4][CB]) {
  // this wave's DMAs for this step are done: loads complete in order, and
  // `ahead` says whether the next step's 4 + CB are still allowed in flight;
  // after the barrier every wave's are, and every wave has finished reading
  // the stage the new DMAs overwrite
  if (ahead) {
    if (CB == 2)
      asm volatile("s_waitcnt vmcnt(6)\n\ts_barrier" ::: "memory");
    else
      asm volatile("s_waitcnt vmcnt(7)\n\ts_barrier" ::: "memory");
  } else {
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  }
  if (next) dma_issue<CB>(c, k_next, raw_n, wt_n);
  mfma_step<CB>(c, raw, wt, colsum, acc);
}

// Software-pipelined form (CB = 3, one wave per SIMD): each step runs as two
// halves of one 32-wide K step each, and the operands of the next half are
// read from LDS while the MFMAs of the current half run, so LDS reads and the
// matrix cores overlap within the wave with two operand sets in registers.
template <int CB>
struct HalfOps {
  v4i a[4], b[CB];
};

template <int CB, int KS, class RAW, class WT>
__device__ __forceinline__ void read_half(const DmaCtx& c, const RAW& raw, const WT& wt, HalfOps<CB>& o) {
  constexpr int ks = KS;
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) o.b[cb] = *reinterpret_cast<const v4i*>(&wt[c.w_off[ks] + 2048 * cb]);
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) {
    const int blk = 2048 * rb + 256 * (ks ^ (rb & 1));
    const v2i lo = tr8(raw, c.a_off[0] + blk), hi = tr8(raw, c.a_off[1] + blk);
    o.a[rb] = v4i{lo.x, lo.y, hi.x, hi.y};
  }
}

template <int CB>
__device__ __forceinline__ void mfma_half(HalfOps<CB>& o, int (&colsum)[CB], v16i (&acc)[4][CB]) {
  // offset-binary digits, in place, all four before the first MFMA (a VALU
  // write just before the MFMA that reads it stalls the issue)
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) o.a[rb] ^= int(0x80808080u);
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) {
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
      acc[rb][cb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(o.a[rb], o.b[cb], acc[rb][cb], 0, 0, 0);
  }
  // column sums from the weight operands (lanes l and l ^ 32 hold the two
  // halves of each row's K chunk)
#pragma unroll
  for (int cb = 0; cb < CB; ++cb)
#pragma unroll
    for (int e = 0; e < 4; ++e) colsum[cb] = __builtin_amdgcn_sdot4(o.b[cb][e], 0x01010101, colsum[cb], false);
}

// 3 + 8 LDS reads among the 4 CB MFMAs of a half.
template <int CB>
__device__ __forceinline__ void interleave_half() {
  __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);  // the four digit XORs
#pragma unroll
  for (int j = 0; j < CB + 8; ++j) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one LDS read
  }
}

// Step s: half A reads K step 1 of stage s (raw_s, wt_s) into h1 while the
// MFMAs of K step 0 run from h0; then the wait for step s + 1's stage and the
// refill of stage s with step s + 3 (past the last step: the last step's tile
// again, never read); half B reads K step 0 of stage s + 1 (raw_n, wt_n; past
// the last step: stale data, never used) into h0 while the MFMAs of K step 1
// run from h1.
template <int CB, class RAWS, class WTS, class RAWN, class WTN>
__device__ __forceinline__ void piped_step(const DmaCtx& c, int s, int steps, int k_begin, RAWS raw_s, WTS wt_s,
                                           RAWN raw_n, WTN wt_n, HalfOps<CB>& h0, HalfOps<CB>& h1,
                                           int (&colsum)[CB], v16i (&acc)[4][CB]) {
  read_half<CB, 1>(c, raw_s, wt_s, h1);
  mfma_half<CB>(h0, colsum, acc);
  interleave_half<CB>();
  // step s + 1's DMAs are done when only step s + 2's (4 + CB = 7) remain in
  // flight, and this wave's reads of stage s are done; after the barrier both
  // hold for every wave, so stage s may be refilled
  asm volatile("s_waitcnt vmcnt(7) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  dma_issue<CB>(c, k_begin + min(s + 3, steps - 1) * kBK, raw_s, wt_s);
  read_half<CB, 0>(c, raw_n, wt_n, h0);
  mfma_half<CB>(h1, colsum, acc);
  interleave_half<CB>();
}

// a m + c for signed 32-bit a, m and a 64-bit c, as one v_mad_i64_i32 (the
// compiler expands a product by a power of two into a sign extension and
// 64-bit shifts and adds, several instructions per term).  Its carry-out
// lane mask is not read.
__device__ __forceinline__ int64_t mad_i64(int a, int m, int64_t c) {
  int64_t r;
  uint64_t unused;
  asm("v_mad_i64_i32 %0, %1, %2, %3, %4" : "=v"(r), "=s"(unused) : "v"(a), "s"(m), "v"(c));
  return r;
}

// Tile (tm, tn) of workgroup t in a TM x TN tile grid.
// Workgroups go to the 8 XCDs round robin (linear id mod 8), so when the grid
// holds a multiple of 8 tiles XCD x is given the contiguous range
// [x nt/8, (x+1) nt/8) of a grouped order (8 tile rows at a time, column by
// column within the group): a compact block of tiles whose share rows and
// weight columns stay in that XCD's L2 (512 x 3072 in 32 x 192 tiles: each
// XCD 8 x 4 tiles, 2 MiB of shares and 768 KiB of weights).  Any bijection
// is correct; this one only places the reuse.
__device__ __forceinline__ void tile_of(int& tm, int& tn, int TN, int TM, int t) {
  const int nt = TN * TM;
  if (nt % 8 == 0) t = (t % 8) * (nt / 8) + t / 8;
  constexpr int G = 8;
  const int group = t / (G * TN), first = group * G, rows = min(G, TM - first);
  const int in = t - group * G * TN;
  tm = first + in % rows;
  tn = in / rows;
}

// Digit sums of one accumulator tile of a wave: rows r0 .. r0 + 3, of which this
// lane takes r0 + 2 khalf (sum[0]) and r0 + 2 khalf + 1 (sum[1]) of its column.
// The lane holds, for its column, digits 4 khalf .. 4 khalf + 3 of the four rows
// in register groups g (rows r0 + g); the halves of the wave add their digit
// sums with v_permlane32_swap: swapping lanes 32-63 of part[g] with lanes 0-31
// of part[g + 2] leaves every lane with its own half's value and the other
// half's for the row it takes, one in each register.
__device__ __forceinline__ void tile_sums(const v16i& a, int khalf, uint64_t (&sum)[2]) {
  uint64_t part[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    // sum_ii acc_ii 256^ii fits 56 signed bits: three 32x32+64 MADs
    const int64_t v = mad_i64(a[4 * g + 3], 16777216, mad_i64(a[4 * g + 2], 65536, mad_i64(a[4 * g + 1], 256, int64_t(a[4 * g]))));
    part[g] = uint64_t(v) << (32 * khalf);
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const auto lo = __builtin_amdgcn_permlane32_swap(uint32_t(part[h]), uint32_t(part[h + 2]), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(uint32_t(part[h] >> 32), uint32_t(part[h + 2] >> 32), false, false);
    sum[h] = ((uint64_t(hi[0]) << 32) | lo[0]) + ((uint64_t(hi[1]) << 32) | lo[1]);
  }
}

// Epilogue of one accumulator tile of a wave: rows row0 .. row0 + 3, column col;
// corr is the offset-binary correction of the column, sh its shift.
__device__ __forceinline__ void store_tile(const v16i& a, int row0, int col, int khalf, uint64_t corr, int sh,
                                           bool split, uint64_t mask, uint64_t* __restrict__ y, int M, int N) {
  uint64_t sum[2];
  tile_sums(a, khalf, sum);
  if (col >= N) return;  // the same for lanes l and l ^ 32
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int row = row0 + 2 * khalf + h;
    if (row >= M) continue;
    uint64_t v = corr + sum[h];
    v = sh < 64 ? (v << sh) : 0;
    if (split)
      atomicAdd(reinterpret_cast<unsigned long long*>(y + size_t(row) * N + col), (unsigned long long)v);
    else
      y[size_t(row) * N + col] = v & mask;
  }
}

// The offset-binary correction 0x8080808080808080 sum_k w[col][k] of a column
// from this lane's column sum (lanes l and l ^ 32 hold the two halves of the
// column's K chunks; after the swap one register holds lanes 0-31's values in
// both halves, the other lanes 32-63's).
__device__ __forceinline__ uint64_t column_correction(int colsum) {
  const auto cs = __builtin_amdgcn_permlane32_swap(colsum, colsum, false, false);
  return 0x8080808080808080ull * uint64_t(int64_t(int(cs[0])) + int64_t(int(cs[1])));
}

// Operand coordinates of this lane (everything of DmaCtx but the DMA sources).
template <int CB>
__device__ __forceinline__ void lane_context(DmaCtx& c) {
  const int t = threadIdx.x, lane = t & 63;
  c.wave = t >> 6;
  c.wm = c.wave >> 1;
  c.wn = c.wave & 1;
  c.i = lane & 31;
  c.khalf = lane >> 5;
  // transpose-read source of this lane: share row 2((l/16) % 2) + l % 2 of
  // the 4-row block, word (l/2) % 8 of the 8-word run at k = 16(l/32)
  c.tr_row = 2 * ((lane >> 4) & 1) + (lane & 1);
  c.tr_k = 16 * (lane >> 5) + ((lane >> 1) & 7);
  {
    const int j = (lane >> 1) & 7;
#pragma unroll
    for (int h = 0; h < 2; ++h)
      c.a_off[h] = (c.wm * 16 + c.tr_row) * kRawRow + 16 * (((8 * c.khalf + 4 * h) ^ (4 * c.tr_row)) + (j >> 1)) +
                   8 * (j & 1);
    const int f = wt_swizzle(c.i);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
      c.w_off[ks] = (c.wn * 32 * CB + c.i) * kBK + 16 * (2 * (ks ^ (f >> 1)) + (c.khalf ^ (f & 1)));
  }
}

// The tile at (m0, n0) over the K steps [k_begin, k_begin + 64 steps) of one
// weight plane (w: its [N][K] bytes; its products enter y shifted by 8 plane).
// split: the result is added into y by 64-bit atomics, unmasked.
template <int CB>
__device__ __forceinline__ void dma_tile(const uint64_t* __restrict__ x, const int8_t* __restrict__ w,
                                         const int8_t* __restrict__ shifts, uint64_t* __restrict__ y, int M, int K,
                                         int N, uint64_t mask, int m0, int n0, int k_begin, int steps, int plane,
                                         bool split) {
  constexpr int BN = 64 * CB;
  __shared__ __attribute__((aligned(16))) uint8_t raw0[kBM * kRawRow];
  __shared__ __attribute__((aligned(16))) uint8_t raw1[kBM * kRawRow];
  __shared__ __attribute__((aligned(16))) uint8_t raw2[kBM * kRawRow];
  __shared__ __attribute__((aligned(16))) uint8_t wt0[BN * kBK];
  __shared__ __attribute__((aligned(16))) uint8_t wt1[BN * kBK];
  __shared__ __attribute__((aligned(16))) uint8_t wt2[BN * kBK];

  DmaCtx c;
  lane_context<CB>(c);
  const int lane = threadIdx.x & 63;
  // DMA sources of this lane: 4 raw-share instructions (2 rows of 512 B each)
  // and CB weight instructions (16 rows of 64 B each) per wave and step.
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int row = 2 * (4 * c.wave + j) + (lane >> 5);
    const int grow = min(m0 + row, M - 1);  // rows past M: any valid row, results dropped
    const int ck = (lane & 31) ^ (4 * (row & 7));  // logical chunk stored at physical chunk lane & 31
    c.xsrc[j] = reinterpret_cast<const uint8_t*>(x + size_t(grow) * K) + ck * 16;
  }
#pragma unroll
  for (int j = 0; j < CB; ++j) {
    const int row = 16 * (CB * c.wave + j) + (lane >> 2);
    const int grow = min(n0 + row, N - 1);
    const int ck = (lane & 3) ^ wt_swizzle(row);  // logical chunk stored at physical chunk lane & 3
    c.wsrc[j] = w + size_t(grow) * K + ck * 16;
  }
  int colsum[CB];
  v16i acc[4][CB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    colsum[cb] = 0;
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) acc[rb][cb] = v16i{0};
  }

  if constexpr (CB == 3) {
    auto raw_of = [&](int q) { return q == 0 ? raw0 : (q == 1 ? raw1 : raw2); };
    auto wt_of = [&](int q) { return q == 0 ? wt0 : (q == 1 ? wt1 : wt2); };
    // steps 0..2 in flight (past the last step: the last step's tile again)
    dma_issue<CB>(c, k_begin, raw0, wt0);
    dma_issue<CB>(c, k_begin + min(1, steps - 1) * kBK, raw1, wt1);
    dma_issue<CB>(c, k_begin + min(2, steps - 1) * kBK, raw2, wt2);
    asm volatile("s_waitcnt vmcnt(14)\n\ts_barrier" ::: "memory");
    HalfOps<CB> h0, h1;
    read_half<CB, 0>(c, raw0, wt0, h0);
    int q = 0;  // stage of step s
    for (int s = 0; s < steps; ++s) {
      const int qn = q == 2 ? 0 : q + 1;
      piped_step<CB>(c, s, steps, k_begin, raw_of(q), wt_of(q), raw_of(qn), wt_of(qn), h0, h1, colsum, acc);
      q = qn;
    }
    // the refills past the last step land before the workgroup ends
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  } else {
  dma_issue<CB>(c, k_begin, raw0, wt0);
  if (steps > 1) dma_issue<CB>(c, k_begin + kBK, raw1, wt1);
  for (int s = 0; s < steps; s += 3) {
    const int kn = k_begin + (s + 2) * kBK;
    dma_step<CB>(c, s + 1 < steps, s + 2 < steps, kn, raw0, wt0, raw2, wt2, colsum, acc);
    if (s + 1 < steps) dma_step<CB>(c, s + 2 < steps, s + 3 < steps, kn + kBK, raw1, wt1, raw0, wt0, colsum, acc);
    if (s + 2 < steps) dma_step<CB>(c, s + 3 < steps, s + 4 < steps, kn + 2 * kBK, raw2, wt2, raw1, wt1, colsum, acc);
  }
  }
  // ---- epilogue: column sums, digit recombination, shift, mask
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    const int col = n0 + c.wn * 32 * CB + cb * 32 + c.i;
    const uint64_t corr = column_correction(colsum[cb]);
    const int sh = 8 * plane + (shifts && col < N ? int(shifts[col]) : 0);
#pragma unroll
    for (int rb = 0; rb < 4; ++rb)
      store_tile(acc[rb][cb], m0 + c.wm * 16 + rb * 4, col, c.khalf, corr, sh, split, mask, y, M, N);
  }
}

// Weight planes: w holds `planes` int8 matrices [planes][N][K], plane e the
// signed byte of weight digit e (planes = 1: int8 weights; 3: the pre-split
// f12 weights).  Workgroup z takes plane z / splits and K split z % splits;
// plane e's products enter y shifted by 8e.  CB = 2: 128-column tiles, two
// workgroups (two waves per SIMD) per CU, whose waits overlap; CB = 3:
// 192-column tiles, one workgroup per CU, 12 accumulator tiles per wave, so
// that every MFMA takes fewer operand bytes from L2 and LDS.
// split-K: workgroup z takes K steps [z k_split, (z+1) k_split); with more
// than one split the partial products are added into y (zeroed first) by
// 64-bit atomics, exact mod 2^64 in any order.
template <int CB>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(CB == 2 ? 2 : 1, CB == 2 ? 2 : 1)))
    share_gemm_dma_kernel(const uint64_t* __restrict__ x, const int8_t* __restrict__ w,
                          const int8_t* __restrict__ shifts, uint64_t* __restrict__ y, int M, int K, int N,
                          uint64_t mask, int k_split, int splits) {
  const int plane = int(blockIdx.z) / splits, k_begin = (int(blockIdx.z) % splits) * k_split;
  int tm, tn;
  tile_of(tm, tn, int(gridDim.x), int(gridDim.y), int(blockIdx.y * gridDim.x + blockIdx.x));
  dma_tile<CB>(x, w + size_t(plane) * size_t(N) * size_t(K), shifts, y, M, K, N, mask, tm * kBM, tn * 64 * CB, k_begin,
               min(k_split, K - k_begin) / kBK, plane, gridDim.z > 1);
}

// ------------------------------------------------------- products of a batch
// The tiles of up to kGroupMax independent products in one launch: workgroup
// g takes tile g - first of the product whose range [first, first + tiles)
// holds g.  Apart, each product pays its own launch, ring fill, epilogue and
// last round of tiles (about 10 us of the 26 us of a 512-row Qwen3 product);
// in one grid a CU's next tile, of whatever product, starts as soon as one of
// its two workgroups ends, so fills and epilogues run beside other tiles'
// MFMAs, and no product needs its K split (and the clear and the atomics of
// one) to fill the chip.
constexpr int kGroupMax = 32;
struct GemmGroup {
  struct Item {
    const uint64_t* x;
    const int8_t* w;
    const int8_t* shifts;
    uint64_t* y;
    int M, K, N;
    int mask_bits;
    int tiles_n, tiles_m;
    unsigned first;  // index of its first tile in the grid
    int pad;
  } item[kGroupMax];
  int count;
};
__device__ __forceinline__ const GemmGroup::Item& group_item(const GemmGroup& g, unsigned tile) {
  int lo = 0, hi = g.count;  // the last item whose first tile is at or below `tile`
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (g.item[mid].first <= tile)
      lo = mid;
    else
      hi = mid;
  }
  return g.item[lo];
}
__device__ __forceinline__ uint64_t group_mask(int bits) { return bits >= 64 ? ~0ull : (1ull << bits) - 1; }

__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
    share_gemm_group_kernel(GemmGroup g) {
  const GemmGroup::Item& it = group_item(g, blockIdx.x);
  int tm, tn;
  tile_of(tm, tn, it.tiles_n, it.tiles_m, int(blockIdx.x - it.first));
  dma_tile<2>(it.x, it.w, it.shifts, it.y, it.M, it.K, it.N, group_mask(it.mask_bits), tm * kBM, tn * kBN, 0,
              it.K / kBK, 0, false);
}

// ------------------------------------------------- any K, any weight form
// Weight forms of the kernels below: int8 rows, three int8 planes [3][N][K],
// or int32 words in [-0x808080, 0x7F7F7F].  For those
//   w + 0x808080 = sum_e b_e 256^e (bytes b_e),  w = sum_e (b_e - 128) 256^e,
// so balanced digit e is byte e of w + 0x808080 with its top bit flipped.
enum { kW8 = 0, kWPlanes = 1, kW32 = 2 };

// 16 bytes from any address (one global_load_dwordx4: gfx950 loads need no
// alignment).
__device__ __forceinline__ uint4 load16(const void* p) {
  uint4 v;
  __builtin_memcpy(&v, (const __attribute__((address_space(1))) char*)(p), 16);
  return v;
}

// Share words k, k + 1 of a row of K; zero past K.  Nothing past K is read.
__device__ __forceinline__ uint4 load_x2(const uint64_t* row, int k, int K) {
  if (k + 2 <= K) return load16(row + k);
  if (k < K) {
    const uint64_t v = row[k];
    return make_uint4(uint32_t(v), uint32_t(v >> 32), 0, 0);
  }
  return make_uint4(0, 0, 0, 0);
}

// Weight bytes k .. k + 15 of a row of K; zero past K.  Nothing past K is
// read: a piece that K cuts is taken from the 16 bytes that end at K.
__device__ __forceinline__ uint4 load_w16(const int8_t* row, int k, int K) {
  if (k + 16 <= K) return load16(row + k);
  unsigned __int128 v = 0;
  if (k < K) {
    if (K >= 16) {
      const uint4 t = load16(row + K - 16);
      v = ((unsigned __int128)((uint64_t(t.w) << 32) | t.z) << 64) | ((uint64_t(t.y) << 32) | t.x);
      v >>= 8 * (k + 16 - K);
    } else {
      for (int b = k; b < K; ++b) v |= (unsigned __int128)(uint8_t(row[b])) << (8 * (b - k));
    }
  }
  const uint64_t lo = uint64_t(v), hi = uint64_t(v >> 64);
  return make_uint4(uint32_t(lo), uint32_t(lo >> 32), uint32_t(hi), uint32_t(hi >> 32));
}

// int32 weights k .. k + 3 of a row of K; zero past K.
__device__ __forceinline__ uint4 load_w4(const int32_t* row, int k, int K) {
  if (k + 4 <= K) return load16(row + k);
  return make_uint4(k < K ? row[k] : 0, k + 1 < K ? row[k + 1] : 0, k + 2 < K ? row[k + 2] : 0, 0);
}

// ------------------------------------------------------ register-staged tile
// The 32 x 128 tile of the DMA kernel for operands its LDS DMA cannot take: K
// not a multiple of 64, weight rows off 16 bytes, int32 weights.  The next K
// step's words are loaded into registers during the current step's MFMAs and
// written to the other of two LDS stages, in the DMA path's swizzled layout;
// the MFMA part is the same.  One barrier per step: a stage is rewritten two
// steps after it was read.  Workgroup z as in the DMA kernel.
//
// FUSED: the workgroup takes the three planes one after the other and keeps the
// outputs' sums in registers, so that y is written once: no clear, no atomics and
// no mask pass, which move y nine times.  They are the cost where K is short:
// three planes 1000x16x3072 71 -> 24 us, int32 78 -> 34.  Each step's words are
// loaded as it starts (the sums take the registers that the next step's would).
template <int WT>
struct RegTile {
  uint4 x[4], w[WT == kW32 ? 8 : 2];
};

template <int WT>
__device__ __forceinline__ void reg_load(RegTile<WT>& r, const uint64_t* const (&xrow)[4], const void* const (&wrow)[2],
                                         int kx, int kw, int K) {
#pragma unroll
  for (int j = 0; j < 4; ++j) r.x[j] = load_x2(xrow[j], kx, K);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    if constexpr (WT == kW32) {
#pragma unroll
      for (int q = 0; q < 4; ++q) r.w[4 * j + q] = load_w4(static_cast<const int32_t*>(wrow[j]), kw + 4 * q, K);
    } else {
      r.w[j] = load_w16(static_cast<const int8_t*>(wrow[j]), kw, K);
    }
  }
}

// Balanced digit e of four int32 weights as four bytes (sel: byte e of both
// v_perm operands).
__device__ __forceinline__ uint32_t digit4(uint4 w, uint32_t sel) {
  const uint32_t o = 0x808080u;
  const uint32_t lo = __builtin_amdgcn_perm(w.y + o, w.x + o, sel), hi = __builtin_amdgcn_perm(w.w + o, w.z + o, sel);
  return __builtin_amdgcn_perm(hi, lo, 0x05040100u) ^ 0x80808080u;
}

template <int WT, bool FUSED = false>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
    share_gemm_reg_kernel(const uint64_t* __restrict__ x, const void* __restrict__ wv,
                          const int8_t* __restrict__ shifts, uint64_t* __restrict__ y, int M, int K, int N,
                          uint64_t mask, int k_split, int splits) {
  constexpr int CB = 2;
  __shared__ __attribute__((aligned(16))) uint8_t raw[2][kBM * kRawRow];
  __shared__ __attribute__((aligned(16))) uint8_t wt[2][kBN * kBK];
  const int first = FUSED ? 0 : int(blockIdx.z) / splits, k_begin = (int(blockIdx.z) % splits) * k_split;
  const int k_end = min(k_begin + k_split, K);
  int tm, tn;
  tile_of(tm, tn, int(gridDim.x), int(gridDim.y), int(blockIdx.y * gridDim.x + blockIdx.x));
  const int m0 = tm * kBM, n0 = tn * kBN;
  DmaCtx c;
  lane_context<CB>(c);
  const int lane = threadIdx.x & 63, xc = lane & 31, wc = lane & 3;
  const uint64_t* xrow[4];
  const void* wrow[2];
  int x_at[4], w_at[2];  // this lane's LDS slots
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int row = 2 * (4 * c.wave + j) + (lane >> 5);
    xrow[j] = x + size_t(min(m0 + row, M - 1)) * K;  // rows past M: any valid row, results dropped
    x_at[j] = row * kRawRow + ((xc ^ (4 * (row & 7))) << 4);
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int row = 16 * (2 * c.wave + j) + (lane >> 2);
    const size_t off = size_t(min(n0 + row, N - 1)) * K;
    wrow[j] = WT == kW32 ? static_cast<const void*>(static_cast<const int32_t*>(wv) + off)
                         : static_cast<const void*>(static_cast<const int8_t*>(wv) + off + size_t(first) * N * K);
    w_at[j] = row * kBK + ((wc ^ wt_swizzle(row)) << 4);
  }
  // the K loop of weight plane `plane`
  const auto products = [&](int plane, int (&colsum)[CB], v16i (&acc)[4][CB]) {
    const uint32_t sel = 0x0c0c0400u + 0x0101u * unsigned(plane);
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      colsum[cb] = 0;
#pragma unroll
      for (int rb = 0; rb < 4; ++rb) acc[rb][cb] = v16i{0};
    }
    RegTile<WT> r;
    if constexpr (!FUSED) reg_load<WT>(r, xrow, wrow, k_begin + 2 * xc, k_begin + 16 * wc, k_end);
    const auto step = [&](uint8_t* rs, uint8_t* ws, int k) {
      if constexpr (FUSED) reg_load<WT>(r, xrow, wrow, k + 2 * xc, k + 16 * wc, k_end);
#pragma unroll
      for (int j = 0; j < 4; ++j) *reinterpret_cast<uint4*>(rs + x_at[j]) = r.x[j];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if constexpr (WT == kW32)
          *reinterpret_cast<uint4*>(ws + w_at[j]) = make_uint4(digit4(r.w[4 * j], sel), digit4(r.w[4 * j + 1], sel),
                                                               digit4(r.w[4 * j + 2], sel), digit4(r.w[4 * j + 3], sel));
        else
          *reinterpret_cast<uint4*>(ws + w_at[j]) = r.w[j];
      }
      __syncthreads();
      const int kn = k + kBK;
      if (!FUSED && kn < k_end) reg_load<WT>(r, xrow, wrow, kn + 2 * xc, kn + 16 * wc, k_end);
      mfma_step<CB>(c, static_cast<const uint8_t*>(rs), static_cast<const uint8_t*>(ws), colsum, acc);
    };
    for (int k = k_begin; k < k_end; k += 2 * kBK) {
      step(raw[0], wt[0], k);
      if (k + kBK < k_end) step(raw[1], wt[1], k + kBK);
    }
  };
  int colsum[CB];
  v16i acc[4][CB];
  if constexpr (!FUSED) {
    products(first, colsum, acc);
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      const int col = n0 + c.wn * 32 * CB + cb * 32 + c.i;
      const uint64_t corr = column_correction(colsum[cb]);
      const int sh = 8 * first + (shifts && col < N ? int(shifts[col]) : 0);
#pragma unroll
      for (int rb = 0; rb < 4; ++rb)
        store_tile(acc[rb][cb], m0 + c.wm * 16 + rb * 4, col, c.khalf, corr, sh, gridDim.z > 1, mask, y, M, N);
    }
  } else {
    uint64_t total[4][CB][2];
#pragma unroll
    for (int rb = 0; rb < 4; ++rb)
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) total[rb][cb][0] = total[rb][cb][1] = 0;
#pragma unroll 1
    for (int plane = 0; plane < 3; ++plane) {
      products(plane, colsum, acc);
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) {
        const uint64_t corr = column_correction(colsum[cb]);
#pragma unroll
        for (int rb = 0; rb < 4; ++rb) {
          uint64_t sum[2];
          tile_sums(acc[rb][cb], c.khalf, sum);
#pragma unroll
          for (int h = 0; h < 2; ++h) total[rb][cb][h] += (corr + sum[h]) << (8 * plane);
        }
      }
      if constexpr (WT == kWPlanes) {
#pragma unroll
        for (int j = 0; j < 2; ++j) wrow[j] = static_cast<const int8_t*>(wrow[j]) + size_t(N) * K;
      }
      __syncthreads();  // both stages are read: the next plane writes them
    }
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      const int col = n0 + c.wn * 32 * CB + cb * 32 + c.i;
      if (col >= N) continue;
      const int sh = shifts ? int(shifts[col]) : 0;
#pragma unroll
      for (int rb = 0; rb < 4; ++rb)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int row = m0 + c.wm * 16 + rb * 4 + 2 * c.khalf + h;
          if (row < M) y[size_t(row) * N + col] = (sh < 64 ? total[rb][cb][h] << sh : 0) & mask;
        }
    }
  }
}

// ---------------------------------------------------------------- few rows
// Products of few share rows (decoding, short prompts) read every weight once
// and have little to compute: what counts is how many bytes are in flight and
// how many launches there are.  A workgroup of eight waves takes 4 RB share
// rows x 32 columns over the whole K: wave v takes the 128-wide K chunks v, v +
// 8, ..., so that the workgroup reads K/128 chunks at once, and the waves' sums
// meet in LDS at the end: one launch, no clear, no atomics, no mask pass, and
// eight times the waves of a 128-column tile grid.  Any K and weight form.
//
// Weights go from memory straight into the MFMA's B registers: lane l holds 64
// bytes of column l % 32, the chunk's half l / 32, and MFMA j of a chunk takes
// bytes 16 j .. 16 j + 15 of both halves (any assignment of k to MFMAs is
// exact, as long as A follows the same).  Shares go through a wave-private LDS
// buffer of 4 rows x 128 words and are read as digits by the transpose read, as
// in the DMA kernel.  LDS operations of one wave complete in order, so the
// buffer needs no barrier.  Pre-split and int32 weights keep one accumulator
// set per plane, so the shares are staged once for all three.
constexpr int kFewRow = kFewChunk * 8;  // bytes of one staged share row

template <int WT>
constexpr int few_planes() { return WT == kW8 ? 1 : 3; }

template <int RB, int WT>
__global__ void __launch_bounds__(64 * kFewWaves) __attribute__((amdgpu_waves_per_eu(2)))
    share_gemm_few_kernel(GemmGroup g) {
  constexpr int P = few_planes<WT>();
  constexpr int kStage = kFewWaves * 4 * kFewRow, kSums = kFewWaves * RB * 4 * 64 * 8;
  __shared__ __attribute__((aligned(16))) uint8_t lds[kStage > kSums ? kStage : kSums];
  const GemmGroup::Item& it = group_item(g, blockIdx.x);
  const int M = it.M, K = it.K, N = it.N;
  const int tile = int(blockIdx.x - it.first), m0 = (tile / it.tiles_n) * 4 * RB, n0 = (tile % it.tiles_n) * kFewCols;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, half = lane >> 5;
  const size_t col = size_t(min(n0 + (lane & 31), N - 1)) * K;  // columns past N: any valid one, results dropped
  const int8_t* w8 = it.w + col;
  const int32_t* w32 = reinterpret_cast<const int32_t*>(it.w) + col;
  const size_t plane_step = size_t(N) * K;
  uint8_t* buf = lds + wave * 4 * kFewRow;
  // transpose-read source: row tr_row, words 64 half + 16 j + tr_k (+ 8)
  const int tr_row = 2 * ((lane >> 4) & 1) + (lane & 1), tr_k = (lane >> 1) & 7;
  v16i acc[P][RB];
  int colsum[P];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    colsum[p] = 0;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) acc[p][rb] = v16i{0};
  }
  for (int k0 = wave * kFewChunk; k0 < K; k0 += kFewWaves * kFewChunk) {
    const int kw = k0 + 64 * half;
    v4i b[P][4];
    if constexpr (WT == kW32) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint4 v = load_w4(w32, kw + 16 * j + 4 * q, K);
#pragma unroll
          for (int p = 0; p < P; ++p) b[p][j][q] = int(digit4(v, 0x0c0c0400u + 0x0101u * unsigned(p)));
        }
      }
    } else {
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint4 v = load_w16(w8 + p * plane_step, kw + 16 * j, K);
          b[p][j] = v4i{int(v.x), int(v.y), int(v.z), int(v.w)};
        }
    }
    uint4 xv[RB][4];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        xv[rb][r] = load_x2(it.x + size_t(min(m0 + 4 * rb + r, M - 1)) * K, k0 + 2 * lane, K);
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
#pragma unroll
      for (int r = 0; r < 4; ++r) *reinterpret_cast<uint4*>(buf + r * kFewRow + ((lane ^ (4 * r)) << 4)) = xv[rb][r];
      __builtin_amdgcn_wave_barrier();
      v4i a[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = 64 * half + 16 * j + tr_k;
        const v2i lo = tr8(buf, tr_row * kFewRow + (((k >> 1) ^ (4 * tr_row)) << 4) + ((k & 1) << 3));
        const v2i hi = tr8(buf, tr_row * kFewRow + ((((k + 8) >> 1) ^ (4 * tr_row)) << 4) + ((k & 1) << 3));
        a[j] = v4i{lo.x, lo.y, hi.x, hi.y} ^ int(0x80808080u);
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int p = 0; p < P; ++p)
          acc[p][rb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[j], b[p][j], acc[p][rb], 0, 0, 0);
    }
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) colsum[p] = __builtin_amdgcn_sdot4(b[p][j][e], 0x01010101, colsum[p], false);
  }
  // this lane's part of rows 4 rb + gq: digits 4 half .. 4 half + 3 and its
  // half of the column's offset correction
  __syncthreads();
  uint64_t* sums = reinterpret_cast<uint64_t*>(lds);  // [wave][row][lane]
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) {
      uint64_t v = 0;
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const v16i& a = acc[p][rb];
        const int64_t d = mad_i64(a[4 * gq + 3], 16777216,
                                  mad_i64(a[4 * gq + 2], 65536, mad_i64(a[4 * gq + 1], 256, int64_t(a[4 * gq]))));
        v += ((uint64_t(d) << (32 * half)) + 0x8080808080808080ull * uint64_t(int64_t(colsum[p]))) << (8 * p);
      }
      sums[(wave * 4 * RB + 4 * rb + gq) * 64 + lane] = v;
    }
  __syncthreads();
  const int row = t >> 5, cl = t & 31;
  if (row < 4 * RB && m0 + row < M && n0 + cl < N) {
    uint64_t v = 0;
#pragma unroll
    for (int w = 0; w < kFewWaves; ++w) {
      const uint64_t* s = sums + (w * 4 * RB + row) * 64 + cl;
      v += s[0] + s[32];
    }
    const int sh = it.shifts ? int(it.shifts[n0 + cl]) : 0;
    v = sh < 64 ? (v << sh) : 0;
    it.y[size_t(m0 + row) * N + n0 + cl] = v & group_mask(it.mask_bits);
  }
}

// y = 0 before a split-K product (keep = 0); y &= mask after one (mask_bits < 64).
__global__ void __launch_bounds__(256) gemm_clear_kernel(uint64_t* __restrict__ y, size_t n, uint64_t keep) {
  for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x)
    y[i] = keep ? (y[i] & keep) : 0;
}

// Pre-split weights: planes[e][i] = balanced signed byte e of w[i] (w in
// [-0x808080, 0x7F7F7F]), so that w = sum_e planes[e] 256^e.
__global__ void __launch_bounds__(256) weight_split_kernel(const int32_t* __restrict__ w, int8_t* __restrict__ planes,
                                                           size_t count) {
  for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < count; i += size_t(gridDim.x) * blockDim.x) {
    const int v = w[i];
#pragma unroll
    for (int e = 0; e < 3; ++e) planes[size_t(e) * count + i] = int8_t(weight_digit(v, e));
  }
}

hipError_t launch_weight_split(const int32_t* w, int8_t* planes, size_t count, hipStream_t s) {
  if (!count) return hipSuccess;
  const unsigned grid = unsigned(std::min<size_t>((count + 255) / 256, 8192));
  hipLaunchKernelGGL(weight_split_kernel, dim3(grid), dim3(256), 0, s, w, planes, count);
  return hipGetLastError();
}

// Zero several outputs in one launch (a batch's split-K products): blockIdx.y
// names the buffer.
constexpr int kGemmClearMax = 64;
struct GemmClearList {
  uint64_t* ptr[kGemmClearMax];
  size_t words[kGemmClearMax];
  int count;
};
__global__ void __launch_bounds__(256) gemm_clear_list_kernel(GemmClearList l) {
  uint64_t* y = l.ptr[blockIdx.y];
  const size_t n = l.words[blockIdx.y];
  for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x) y[i] = 0;
}

static GemmGroup::Item group_entry(const uint64_t* x, const void* w, const int8_t* shifts, uint64_t* y, int M, int K,
                                   int N, int mask_bits, int tile_m, int tile_n, unsigned first) {
  return GemmGroup::Item{x, static_cast<const int8_t*>(w), shifts, y, M, K, N, mask_bits,
                         (N + tile_n - 1) / tile_n, (M + tile_m - 1) / tile_m, first, 0};
}

static hipError_t launch_few(const GemmGroup& g, int rb, int w_bits, unsigned tiles, hipStream_t s) {
  const auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(tiles), dim3(64 * kFewWaves), 0, s, g); };
  if (w_bits == 8)
    rb == 1 ? go(share_gemm_few_kernel<1, kW8>) : rb == 2 ? go(share_gemm_few_kernel<2, kW8>) : go(share_gemm_few_kernel<4, kW8>);
  else if (w_bits == 24)
    rb == 1 ? go(share_gemm_few_kernel<1, kWPlanes>) : go(share_gemm_few_kernel<2, kWPlanes>);
  else
    rb == 1 ? go(share_gemm_few_kernel<1, kW32>) : go(share_gemm_few_kernel<2, kW32>);
  return hipGetLastError();
}

static hipError_t run_share_gemm(const uint64_t* x, const void* w, int w_bits, const int8_t* shifts, uint64_t* y,
                                 int M, int K, int N, int mask_bits, hipStream_t s, bool y_zero) {
  const uint64_t mask = mask_bits >= 64 ? ~0ull : ((1ull << mask_bits) - 1);
  const GemmChoice c = gemm_choice(x, w, w_bits, M, K, N);
  if (c.kernel == kGemmFew) {
    GemmGroup g;
    g.count = 1;
    g.item[0] = group_entry(x, w, shifts, y, M, K, N, mask_bits, 4 * c.rb, kFewCols, 0);
    return launch_few(g, c.rb, w_bits, unsigned(g.item[0].tiles_m) * unsigned(g.item[0].tiles_n), s);
  }
  const size_t words = size_t(M) * N;
  const unsigned fgrid = unsigned(std::min<size_t>((words + 255) / 256, 4096));
  // several planes or K splits add their partial products into y; the empty sum is y = 0
  if (c.kernel == kGemmZero || (c.adds && !y_zero)) {
    hipLaunchKernelGGL(gemm_clear_kernel, dim3(fgrid), dim3(256), 0, s, y, words, 0ull);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || c.kernel == kGemmZero) return e;
  }
  const dim3 block(kThreads);
  const unsigned gy = unsigned((M + kBM - 1) / kBM), gz = c.kernel == kGemmRegFused ? 1u : unsigned(c.splits * c.planes);
  const dim3 grid2(unsigned((N + kBN - 1) / kBN), gy, gz);
  const auto reg = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid2, block, 0, s, x, w, shifts, y, M, K, N, mask, c.k_split, c.splits);
  };
  if (c.kernel == kGemmRegFused)
    w_bits == 32 ? reg(share_gemm_reg_kernel<kW32, true>) : reg(share_gemm_reg_kernel<kWPlanes, true>);
  else if (c.kernel == kGemmReg)
    w_bits == 32 ? reg(share_gemm_reg_kernel<kW32>) : reg(share_gemm_reg_kernel<kW8>);
  else if (c.kernel == kGemmDma2)
    hipLaunchKernelGGL(share_gemm_dma_kernel<2>, grid2, block, 0, s, x, static_cast<const int8_t*>(w), shifts, y, M, K,
                       N, mask, c.k_split, c.splits);
  else
    hipLaunchKernelGGL(share_gemm_dma_kernel<3>, dim3(unsigned((N + 191) / 192), gy, gz), block, 0, s, x,
                       static_cast<const int8_t*>(w), shifts, y, M, K, N, mask, c.k_split, c.splits);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess && c.adds && mask != ~0ull) {
    hipLaunchKernelGGL(gemm_clear_kernel, dim3(fgrid), dim3(256), 0, s, y, words, mask);
    e = hipGetLastError();
  }
  return e;
}

hipError_t launch_share_gemm(const uint64_t* x, const void* w, int w_bits, const int8_t* shifts, uint64_t* y,
                             int M, int K, int N, int mask_bits, hipStream_t s) {
  return run_share_gemm(x, w, w_bits, shifts, y, M, K, N, mask_bits, s, false);
}

// Products whose order does not matter: those of few rows in launches of up to
// kGroupMax by their weight form and row blocks, the DMA path's int8 ones as
// 128-column tiles, longest K first (the last round of tiles is then one of
// short ones); the rest one by one, the outputs they add into zeroed together.
// A grid of many products fills the chip with either kernel, and then the bytes
// per product decide: for every 32 columns and k a tile moves 96, the few-row
// kernel 64 (up to 4 rows), 96 or 160.  56 products of 16 rows: tiles 85 us,
// few-row 142 us; of one row: 77 and 60 us.
// A grid of tiles has no need of K splits, but one product alone may: where the
// split saves 16 K steps and more it takes its own path.  us, unsplit / split with
// its clear and mask: 200x3072x1024 (48 steps to 12) 31.0 / 18.4, 512x3072x1024 (48 to
// 24) 31.8 / 28.4, 200x1024x3072 (16 to 8) 13.9 / 20.4.  Four three-plane products
// 16x3072x1024 64 us one after the other (64 workgroups each), 17 together.
hipError_t launch_share_gemm_group(const praghip_gemm_desc* list, size_t count, hipStream_t s) {
  std::vector<const praghip_gemm_desc*> few[3][3], dma, rest;
  hipError_t e = hipSuccess;
  size_t moved = 0;
  for (size_t i = 0; i < count; ++i)
    if (list[i].m && list[i].n && list[i].w_bits == 8)
      moved += few_bytes(8, int(list[i].m), int(list[i].k), int(list[i].n));
  for (size_t i = 0; i < count; ++i) {
    const praghip_gemm_desc& d = list[i];
    if (d.m == 0 || d.n == 0) continue;
    GemmChoice c = gemm_choice(d.x, d.w, d.w_bits, int(d.m), int(d.k), int(d.n));
    if (d.w_bits == 8 && c.kernel == kGemmFew && d.m > 4 && moved > kFewBytes) {
      const GemmChoice t = gemm_choice(d.x, d.w, 8, int(d.m), int(d.k), int(d.n), false);
      if (t.kernel == kGemmDma2 || t.kernel == kGemmDma3) c = t;
    }
    const size_t tiles = ((d.m + 3) / 4) * ((d.n + kFewCols - 1) / kFewCols);
    if (c.kernel == kGemmFew && tiles < (1u << 24))
      few[d.w_bits == 8 ? 0 : d.w_bits == 24 ? 1 : 2][c.rb >> 1].push_back(&d);
    else if (d.w_bits == 8 && (c.kernel == kGemmDma2 || c.kernel == kGemmDma3) && tiles < (1u << 24))
      dma.push_back(&d);
    else
      rest.push_back(&d);
  }
  if (dma.size() == 1) {
    const praghip_gemm_desc& d = *dma[0];
    if (int(d.k) - gemm_choice(d.x, d.w, 8, int(d.m), int(d.k), int(d.n), false).k_split >= 16 * kBK) {
      rest.push_back(dma[0]);
      dma.clear();
    }
  }
  std::vector<const praghip_gemm_desc*> adds;
  for (const praghip_gemm_desc* d : rest)
    if (gemm_choice(d->x, d->w, d->w_bits, int(d->m), int(d->k), int(d->n)).adds) adds.push_back(d);
  const bool together = adds.size() > 1;
  for (size_t a0 = 0; together && a0 < adds.size() && e == hipSuccess; a0 += kGemmClearMax) {
    GemmClearList l{};
    for (size_t a = a0; a < adds.size() && l.count < kGemmClearMax; ++a) {
      l.ptr[l.count] = adds[a]->y;
      l.words[l.count++] = adds[a]->m * adds[a]->n;
    }
    hipLaunchKernelGGL(gemm_clear_list_kernel, dim3(512, unsigned(l.count)), dim3(256), 0, s, l);
    e = hipGetLastError();
  }
  for (size_t i = 0; i < rest.size() && e == hipSuccess; ++i) {
    const praghip_gemm_desc& d = *rest[i];
    e = run_share_gemm(d.x, d.w, d.w_bits, d.shifts, d.y, int(d.m), int(d.k), int(d.n), d.mask_bits, s, together);
  }
  std::stable_sort(dma.begin(), dma.end(), [](auto* a, auto* b) { return a->k > b->k; });
  const auto run = [&](const std::vector<const praghip_gemm_desc*>& v, int tile_m, int tile_n, auto&& launch) {
    for (size_t i0 = 0; i0 < v.size() && e == hipSuccess; i0 += kGroupMax) {
      GemmGroup g;
      g.count = int(std::min<size_t>(kGroupMax, v.size() - i0));
      unsigned tiles = 0;
      for (int i = 0; i < g.count; ++i) {
        const praghip_gemm_desc& d = *v[i0 + size_t(i)];
        g.item[i] = group_entry(d.x, d.w, d.shifts, d.y, int(d.m), int(d.k), int(d.n), d.mask_bits, tile_m, tile_n, tiles);
        tiles += unsigned(g.item[i].tiles_m) * unsigned(g.item[i].tiles_n);
      }
      e = launch(g, tiles);
    }
  };
  for (int f = 0; f < 3; ++f)
    for (int i = 0; i < 3; ++i) {
      const int bits = f == 0 ? 8 : f == 1 ? 24 : 32, rb = 1 << i;
      run(few[f][i], 4 * rb, kFewCols, [&](const GemmGroup& g, unsigned tiles) { return launch_few(g, rb, bits, tiles, s); });
    }
  run(dma, kBM, kBN, [&](const GemmGroup& g, unsigned tiles) {
    hipLaunchKernelGGL(share_gemm_group_kernel, dim3(tiles), dim3(kThreads), 0, s, g);
    return hipGetLastError();
  });
  return e;
}

}  // namespace praghip
