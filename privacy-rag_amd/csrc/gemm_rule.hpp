// Which kernel a share product takes, and how its K is split: host code without
// HIP, so that it can be checked apart from the kernels (gemm.hip).
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace praghip {

constexpr int kBM = 32, kBN = 128, kBK = 64;  // rows and columns of a tile, words of a K step
constexpr int kFewWaves = 8, kFewChunk = 128, kFewCols = 32;  // few-row kernel: waves, K words of a wave's turn, columns

// The few-row kernel's workgroups each read 4 rb share rows and 32 weight
// columns whole, so what it moves through L2 grows with M N K, while a tile
// kernel pays a clear, a mask pass and a ring fill.  Measured (us, few-row /
// tile kernel, int8): 1x1024x4096 11.9 / 17.5 and 64x1024x4096 12.0 / 17.7
// (both at the host's issue rate), 100x1024x3001 15.5 / 17.7 (108 MB),
// 32x4096x8192 26.4 / 22.4 (335 MB), 100x3072x4096 35.1 / 25.9 (440 MB); three
// planes: 64x3072x1024 15.3 / 18.2 (126 MB), 77x3072x1024 28.2 / 21.2 (157 MB);
// int32: 13x1024x3001 12.7 / 18.7 (37 MB), 13x3072x4096 32.9 / 29.5 (151 MB).
constexpr size_t kFewBytes = size_t(128) << 20;
// K counts as at least the eight waves' 1024 words: below it some of them have no
// chunk.  us, few-row / tiles: int8 486x90x1131 27.8 / 9.3, 200x130x4000 34.2 / 9.4,
// 700x500x700 24.2 / 12.6; int32 486x90x1131 61.2 / 24.8, 40x700x5000 46.0 / 24.4.
inline int few_rb(int w_bits, int M) { return M <= 4 ? 1 : (M <= 8 || w_bits != 8) ? 2 : 4; }
inline size_t few_bytes(int w_bits, int M, int K, int N) {
  const size_t rb = size_t(few_rb(w_bits, M)), wgs = (size_t(M) + 4 * rb - 1) / (4 * rb) * ((size_t(N) + 31) / 32);
  return wgs * size_t(std::max(K, kFewWaves * kFewChunk)) * 32 * (rb + (w_bits == 8 ? 1 : w_bits == 24 ? 3 : 4));
}

// kGemmRegFused: the register-staged tile with the three planes in one workgroup;
// kGemmZero: K = 0, the empty sum; y is zeroed.
enum GemmKernel { kGemmFew, kGemmDma2, kGemmDma3, kGemmReg, kGemmRegFused, kGemmZero };
struct GemmChoice {
  GemmKernel kernel;
  int rb;               // kGemmFew: 4-row blocks per workgroup
  int k_split, splits;  // K words per workgroup, K splits (tile kernels)
  int planes;
  bool adds;  // the workgroups of one tile add into y (atomics): y is zeroed first, masked after
};

inline GemmChoice gemm_choice(const void* x, const void* w, int w_bits, int M, int K, int N,
                              size_t few_limit = kFewBytes) {
  GemmChoice c{};
  c.planes = w_bits == 8 ? 1 : 3;
  c.rb = few_rb(w_bits, M);
  if (K == 0) {
    c.kernel = kGemmZero;
    return c;
  }
  if (few_bytes(w_bits, M, K, N) <= few_limit) {
    c.kernel = kGemmFew;
    return c;
  }
  // LDS DMA: whole 64-wide K steps, 16-byte aligned rows
  const bool dma = w_bits != 32 && K % kBK == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(x) % 16 == 0;
  // 128-column tiles (CB = 2, up to two workgroups per CU), K split while
  // the tiles fill fewer than 256 workgroups and each split keeps >= 8
  // steps.  192-column tiles (CB = 3, one workgroup per CU) only where
  // they fill the 256 CUs in one round while the 128-column grid would
  // leave the CUs unevenly loaded (between one and two workgroups each):
  // 512 x 1024 x 3072 int8 runs 21.4 us against 22.8 us; every other
  // Qwen3 shape and the f12 planes run faster with CB = 2 (measured).
  const int ksteps = (K + kBK - 1) / kBK;
  const long tiles2 = long((N + kBN - 1) / kBN) * long((M + kBM - 1) / kBM);
  const long tiles3 = long((N + 191) / 192) * long((M + kBM - 1) / kBM);
  int splits = 1;
  while (splits < 4 && tiles2 * splits < 256 && ksteps / (splits * 2) >= 8) splits *= 2;
  const long wg2 = tiles2 * splits * c.planes;
  c.kernel = !dma ? kGemmReg : (splits == 1 && c.planes == 1 && wg2 > 256 && wg2 < 512 && tiles3 <= 256) ? kGemmDma3 : kGemmDma2;
  c.k_split = (ksteps + splits - 1) / splits * kBK;
  c.splits = (K + c.k_split - 1) / c.k_split;
  // Three planes in one workgroup: a third of the workgroups, but no clear, atomics
  // and mask over y, which cost most while K is short.  us, planes apart /
  // together - three planes: 1000x16x1024 (256 tiles, 1 step) 29.4 / 11.9,
  // 1000x700x1024 (256, 11) 51.3 / 41.4, 1000x200x512 (128, 4) 20.6 / 20.0,
  // 1000x300x512 (128, 5) 21.4 / 23.1, 200x47x1024 (56, 1) 11.9 / 12.1; int32:
  // 1000x200x1024 (256, 4) 41.7 / 31.6, 1000x512x1024 (256, 8) 45.8 / 45.8,
  // 1000x100x512 (128, 2) 21.9 / 21.3, 1000x200x512 (128, 4) 24.0 / 29.8.
  const int most = w_bits == 24 ? (tiles2 >= 256 ? 15 : tiles2 >= 128 ? 4 : tiles2 >= 64 ? 1 : 0)
                                : (tiles2 >= 256 ? 4 : tiles2 >= 128 ? 2 : 0);
  if (c.kernel == kGemmReg && c.planes == 3 && ksteps <= most) {
    c.kernel = kGemmRegFused;
    return c;
  }
  c.adds = c.splits * c.planes > 1;
  return c;
}

}  // namespace praghip
