// Which kernel a share product takes, and how its K is split: host code without
// HIP, so that it can be checked apart from the kernels (gemm.hip).
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace praghip {

constexpr int kBM = 32, kBN = 128, kBK = 64;  // rows and columns of a tile, words of a K step
constexpr int kFewWaves = 8, kFewChunk = 128, kFewCols = 32;  // few-row kernel: waves, K words of a wave's turn, columns

// The few-row kernel: 4 rb share rows x 32 columns to a workgroup, which reads
// these rows and columns whole.
inline int few_rb(int w_bits, int M) { return M <= 4 ? 1 : (M <= 8 || w_bits != 8) ? 2 : 4; }
inline size_t few_groups(int w_bits, int M, int N) {
  const size_t rows = 4 * size_t(few_rb(w_bits, M));
  return (size_t(M) + rows - 1) / rows * ((size_t(N) + kFewCols - 1) / kFewCols);
}
// What it moves through L2, which grows with M N K; K counts as at least the eight
// waves' 1024 words.  us, few-row / tiles, above the limit: int8 32x4096x8192 26.4
// / 22.4 (335 MB), 100x3072x4096 35.1 / 25.9 (440 MB); three planes 77x3072x1024
// 28.2 / 21.2 (157 MB); int32 13x3072x4096 32.9 / 29.5 (151 MB).
constexpr size_t kFewBytes = size_t(128) << 20;
inline size_t few_bytes(int w_bits, int M, int K, int N) {
  return few_groups(w_bits, M, N) * size_t(std::max(K, kFewWaves * kFewChunk)) * 32 *
         (size_t(few_rb(w_bits, M)) + (w_bits == 8 ? 1 : w_bits == 24 ? 3 : 4));
}
// Below the limit it is a matter of rounds: one workgroup fills a CU, so each 256
// of them are a round of about 5 us, and a second round already meets tiles that
// are done in one.  GPU time, us, few-row / tiles (workgroups):
//   int8, one round: 64x1024x1024 6.3 / 12.8, 8x64x8000 4.9 / 4.9; but a single K
//   step of the LDS DMA is over sooner: 64x64x1024 6.7 / 5.4.  Two rounds, while a
//   tile's K loop is long or split and each wave has a chunk or so: 400x512x512
//   9.3 / 9.7 (400), 200x1024x1024 11.2 / 14.2 (416), but 400x300x512 12.0 / 10.8 (400),
//   64x64x3072 11.8 / 5.6 (384).  Three and more: 1000x100x300 16.8 / 8.4 (630),
//   1000x64x300 17.1 / 5.7 (630), 400x64x1024 21.7 / 5.8 (800);
//   three planes: 64x64x1024 6.8 / 9.0 (256), 16x3072x1024 15.2 / 15.8, but 8x4096x1024
//   19.4 / 17.1 where the DMA tiles' splits still fit one round (1x3804x308, on no
//   DMA, 13.5 / 18.8); 200x128x512 8.3 / 10.2 (400), 200x1024x512 13.7 / 15.0 (400),
//   406x28x178 11.0 / 13.0 (306), but 32x2048x3072 23.5 / 19.1 (384), 64x64x3072 17.2 /
//   10.4 (768);
//   int32, whose tiles split the digits at every use: 13x3072x1024 20.8 / 23.3,
//   200x512x512 13.4 / 19.5 (400), 1024x800x100 22.8 / 25.7 (512), but 400x64x300 15.7 /
//   11.6 (500), 400x1024x300 27.3 / 21.2 (500: from 1024 on the tiles split K).
// Shares beyond the L2s are read once per 32 columns here and once per 128 by the
// tiles: int8 1000x3072x128 19.2 / 16.4, but 1000x3072x64 12.3 / 15.8; three planes
// 4000x1024x32 14.3 / 30.7, int32 27.5 / 40.4 (500), where the tiles pad N to 128.
inline bool few_pays(int w_bits, bool dma, long tile_groups, int M, int K, int N) {
  const size_t rounds = (few_groups(w_bits, M, N) + 255) / 256;
  const bool near = N <= 64 || size_t(M) * size_t(K) <= (size_t(1) << 21);
  if (w_bits == 8)
    return near && (rounds == 1 ? !(dma && K <= kBK && M > 8) : rounds == 2 && K >= 448 && K <= 1024);
  if (w_bits == 24)
    return rounds == 1 ? K <= 3072 || !dma || M <= 4 || tile_groups > 256 : rounds == 2 && near && (K > kBK || !dma) && K <= 1024;
  return rounds == 1 || (K >= 100 && ((rounds == 2 && (K < 1024 || N <= 64)) || (rounds <= 4 && K <= 600)));
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

// few: false leaves the few-row kernel out.
inline GemmChoice gemm_choice(const void* x, const void* w, int w_bits, int M, int K, int N, bool few = true) {
  GemmChoice c{};
  c.planes = w_bits == 8 ? 1 : 3;
  c.rb = few_rb(w_bits, M);
  if (K == 0) {
    c.kernel = kGemmZero;
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
  if (few && few_bytes(w_bits, M, K, N) <= kFewBytes &&
      few_pays(w_bits, dma, tiles2 * splits * c.planes, M, K, N)) {
    c.kernel = kGemmFew;
    return c;
  }
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
