// Rules that choose a kernel from sizes and types. Plain functions of their
// arguments (the number of CUs among them), so that the CPU tests can run them.
#pragma once

#include <stdint.h>

namespace qo {

// fp16 / bf16 shapes and token counts at which fq_mfma_kernel's zero-padded
// fragments are faster than fq_tile_kernel: where one round of tile workgroups
// fills every CU (four of 56 x 64, two of the others), their set-ups share the
// CU's LDS and the LDS-DMA copies of fq_mfma_kernel do not; and 64 x 80 fp16
// beyond two tokens per CU, whose 99 registers let two workgroups of five waves
// share a CU and not three (bf16: 93, three). Measured on 256 CUs, kernel alone,
// packed codes, fp16, tile -> mfma: 80 x 112, 300 tokens 10.6 -> 9.4 us, 512
// tokens 11.1 -> 9.9 us (256 tokens 8.0 against 8.3, 600 tokens 16.3 against
// 21.1); 72 x 96, 512 tokens 10.1 -> 9.8 us; 64 x 112, 512 tokens 9.1 -> 8.7 us
// (bf16 the same on both); 56 x 64, 1021 tokens 8.5 -> 8.1 us; 64 x 80, 1024
// tokens 13.6 -> 9.8 us, 4096 tokens 27.7 -> 21.3 us (bf16 21.2 against 24.4).
inline bool fq_padded_mfma(int M, int N, int64_t tokens, bool f16, int64_t cus) {
  const int64_t per_cu = (tokens + cus - 1) / cus;
  if (M == 56 && N == 64) return per_cu == 4;
  if (M == 64 && N == 80) return f16 && per_cu > 2;
  if ((M == 64 && N == 112) || (M == 72 && N == 96) || (M == 80 && N == 112)) return per_cu == 2;
  return false;
}

// Quantize calls of a few features and fewer tokens than CUs that the generic
// kernel finishes sooner than fq_tile_kernel / fq_f32_kernel, whose set-up
// (operand fragments of 16 rows and columns) is then most of the time. Its
// fast form needs M and N to be multiples of 4, and packing costs it an
// exchange. Measured, 1 token, int8 codes, fragment kernel -> generic: float32
// 4 x 4 4.7 -> 3.8 us, 8 x 8 4.5 -> 4.0 us, 8 x 12 4.4 -> 4.1 us (12 x 12 4.4
// against 4.3); 4 x 6 4.8 -> 4.5 us; fp16 4 x 8 4.5 -> 4.2 us, 8 x 8 4.4 -> 4.3
// us (8 x 12 the same, 5 x 8 4.3 against 6.3); packed float32 4 x 4 4.7 -> 4.3 us
// (4 x 8 the same). At 256 tokens the fragment kernels win from 24 features.
inline bool fq_generic_few(int M, int N, int64_t tokens, bool f32, bool pack, int64_t cus) {
  const int64_t F = (int64_t)M * N;
  if (tokens >= cus) return false;
  if (pack) return f32 && F <= 16;
  if (M % 4 == 0 && N % 4 == 0) return F <= (f32 ? 96 : 64);
  return f32 && F <= 32;
}

// Ragged products (N % 4 != 0 or K % 128 != 0) that the generic GEMM kernel
// finishes sooner than the small-M kernel (`over_skinny`) or the FP6 route. A
// workgroup of the generic kernel makes 16 x 16 outputs; two per CU run beside
// each other, further rounds of them cost more (in ns, per k: 20 for the first
// round on W.t(), 25 on [K/8, N], 26 for each further one). The small-M kernel
// takes 3.7 to 5 us whatever K is here, the FP6 route's two launches 6 to 9 us
// of the device and 9.3 us of the host (one launch: 5.8 us), so the line lies
// where the generic kernel's estimate passes the device's time but not yet the
// host's (8 us; single shapes there differ by 2 us either way). Measured on W.t(),
// FP6 route -> generic: 300 x 64 x 8 6.6 -> 2.4 us, 256 x 37 x 64 7.0 -> 3.5 us,
// 128 x 1001 x 200 7.9 -> 7.1 us, 128 x 513 x 264 8.8 -> 8.1 us, 256 x 1001 x 64
// (two rounds) 7.7 -> 6.4 us, but 512 x 1001 x 64 (four) 8.1 against 10.5 and
// 65 x 1001 x 320 7.5 against 9.1; [K/8, N] 65 x 1001 x 264 7.6 against 9.0.
// Small-M kernel -> generic: 64 x 37 x 64 4.3 -> 3.5 us, 64 x 2051 x 32 4.7 -> 3.4
// us, 16 x 513 x 96 4.0 either way.
inline bool gemm_generic_small(int64_t M, int64_t N, int64_t K, bool b_nk, bool over_skinny, int64_t cus) {
  const int64_t blocks = ((M + 15) / 16) * ((N + 15) / 16);
  const int64_t rounds = (blocks + 2 * cus - 1) / (2 * cus);
  if (over_skinny) return K * rounds <= 64;
  return 2000 + K * ((b_nk ? 20 : 25) + 26 * (rounds - 1)) <= 8000;
}

// The output tile of an M x N x K product, by an estimate of its time in ns: k-blocks
// times the time of a round's stages, plus what a round takes besides them. A
// stage is bound by the CU's LDS traffic (its operand reads at about 128 bytes
// per clock, the copies from L2 at 64), so a larger tile costs less per product
// but leaves more CUs idle. Per stage, measured at 4096 columns x 14336: 256-row
// tiles 740 (850 with every CU busy, 256 columns wide), 128 x 128 430 for one
// workgroup on a CU and 700 for two, 128 x 64 345 and 480; per round 8 us and 4 us.
// Split tiles (one per CU, two groups of waves) take 670 and 510 for a pair of
// stages, and 1 us more a round for the sums' exchange: they win where a round
// leaves CUs with one tile and K is 1536 or more. Kernel alone, unsplit -> split:
// 512 x 4096 x 14336 38.6 -> 33.8 us, 640 x 3584 x 18944 61.1 -> 49.2 us,
// 400 x 8192 x 28672 94.6 -> 80.2 us, 1024 x 4096 x 14336 49.7 -> 42.1 us,
// 300 x 2048 x 2048 7.7 -> 7.4 us.
// With 256-row tiles alone M = 512 took 83.7 us there (38 tiles on 256 CUs); 512 x 14336 x 4096 33 -> 25 us on 128 x 128; 2048 x
// 4096 x 4096 34 -> 25 us; 2048 x 14336 x 4096 keeps 256 x 224 (87 us against 94).
enum F6Tile { kF6Tile224, kF6Tile256, kF6Tile128, kF6Tile64, kF6Split128, kF6Split64 };
inline F6Tile f6_tile(int64_t M, int64_t N, int64_t K, bool f32, int64_t cus) {
  const int64_t nk = (K + 127) / 128;
  auto tiles = [&](int64_t bm, int64_t bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  auto wide = [&](int64_t t, int64_t stage) { return (t + cus - 1) / cus * (nk * stage + 8000); };
  auto pair = [&](int64_t t, int64_t one, int64_t two) {   // rounds of two workgroups per CU
    const int64_t full = t / (2 * cus), rest = t % (2 * cus);
    return full * (nk * two + 4000) + (rest == 0 ? 0 : nk * (rest <= cus ? one : two) + 4000);
  };
  auto split = [&](int64_t t, int64_t stage) { return (t + cus - 1) / cus * ((nk + 1) / 2 * stage + 5000); };
  const int64_t est[6] = {wide(tiles(256, 224), 745), wide(tiles(256, 256), 850), pair(tiles(128, 128), 430, 700),
                          pair(tiles(128, 64), 345, 480), split(tiles(128, 128), 670), split(tiles(128, 64), 510)};
  int best = f32 ? 2 : 0;   // the 256-row kernel stages 16-bit values
  for (int i = best + 1; i < 6; ++i)
    if (est[i] < est[best]) best = i;
  return (F6Tile)best;
}

}  // namespace qo
