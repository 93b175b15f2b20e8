// bi_gemm_gen.h — launches of the dense tiles (gemm_big, gemm_tall) for a
// batch of matrices in one grid, a right-hand side stored row-major (b[k][n])
// and K that is not a multiple of 64. 2-byte types; the same steps per output
// element as every other dense launch, so the same bits.
#pragma once

#include "bi_matmul_impl.h"

namespace bi {

enum GenForm { kGen32x64 = 0, kGen64x64, kGen128x64, kGen128x128, kGen256x128, kGenForms };
constexpr int kGenRows[kGenForms] = {32, 64, 128, 128, 256};
constexpr int kGenCols[kGenForms] = {64, 64, 64, 128, 128};

struct GenPlan {
  int form = kGen64x64;
  int chunks = 1, cg = 0;   // K chunks of cg groups (tall forms, row-major B)
};

// fold_groups over a batch: slice blockIdx.y of part[slice][g][M N].
template <typename T>
__global__ __launch_bounds__(256) void fold_groups_batch(const float* __restrict__ part, T* __restrict__ out,
                                                         int64_t MN, int G, int64_t out_stride) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= MN) return;
  part += blockIdx.y * MN * G;
  float total = 0.0f;
#pragma unroll 8
  for (int g = 0; g < G; ++g) total = total + part[(int64_t)g * MN + idx];
  out[blockIdx.y * out_stride + idx] = to_store<T>(total);
}

static inline int64_t gen_tiles(int64_t batch, int64_t M, int64_t N, int form) {
  return batch * ceil_div(M, kGenRows[form]) * ceil_div(N, kGenCols[form]);
}

// The form (a function of the shape only; bits never depend on it). Measured
// on one MI355X, bf16, us by form 64x64 / 128x64 / 128x128 / 256x128 (either B
// layout within 5%):
//   128 x [512, 128, K 512]  37 / 32 / 43 / 60   (256 tiles of 256 x 128)
//   128 x [512, 512, K 128]  71 / 47 / 51 / 44   (1024)
//   8 x [512, 128, K 1024]   13 / 8.8 / 12 / 16  (8)
//   32 x [200, 64, K 776]    13 / 12.4 / 14.5 / 19
//   [515, 4096, K 4096]      81 / 38 / 34 / 46   (96)
//   [2000, 4096, K 4096]     194 / 82 / 84 / 64  (256)
//   [3000, 14336, K 4096]    920 / 470 / 442 / 376
//   [333, 896, K 4864]       51 / 26 / 38 / 53   (42 tiles of 128 x 64; 64 x 64 in 7 K chunks 23, row-major B only)
// 256 x 128 runs one workgroup per CU, so it wants several rounds of tiles or a
// long K; 128 x 64 runs two and hides each other's prologue and stores. Rows up
// to 64 take the tall tiles (64 x [64, 128, K 512]: 64x64 8.7, 128x64 19), more
// rows only with K split. A row-major B with few tiles splits K: [64, 4096, K
// 4096] 42 -> 17 us in 8 chunks, [1, 1024, K 4096] 31 -> 6.2 in 16, [16, 14336,
// K 4096] 31 -> 28 in 2; and so does a small batch, whose chain of K stages is
// otherwise longer than one launch per matrix with K split was: 2 x [1, 64, K
// 65536] 75 by matrix, 462 unsplit, 18 split; 2 x [64, 64, K 4096] 26 / 44 / 9.7;
// 4 x [512, 128, K 16384] 145 / 167 / 57; 2 x [33, 64, K 1000] 38 / 14 / 9.5.
static inline GenPlan gen_plan(int64_t batch, int64_t M, int64_t N, int64_t K, BMode mode, bool split = true) {
  GenPlan p;
  const int G = ceil_div(K, kGroupK);
  p.cg = G;
  const int64_t t256 = gen_tiles(batch, M, N, kGen256x128), t128 = gen_tiles(batch, M, N, kGen128x128),
                t64 = gen_tiles(batch, M, N, kGen128x64);
  if (M <= 32) p.form = kGen32x64;
  else if (M <= 64) p.form = kGen64x64;
  else if (t256 >= 512 || (t256 >= 192 && K >= 1024)) p.form = kGen256x128;
  else if (t64 > 256 && t128 <= 256 && K >= 1024) p.form = kGen128x128;
  else if (t64 >= 48) p.form = kGen128x64;
  else p.form = kGen64x64;
  if (split && p.form <= kGen64x64 && mode == kBColumns) {
    const int64_t t = gen_tiles(batch, M, N, p.form);
    if (batch == 1 ? t < 256 && G >= 2 : t <= (M <= 16 ? 31 : 64) && G >= 4) {
      p.cg = ceil_div(G, std::min<int64_t>(G, ceil_div(512, t)));
      p.chunks = ceil_div(G, p.cg);
    }
  }
  if (M > 64 && p.form == kGen64x64 && p.chunks == 1) p.form = kGen128x64;
  return p;
}

// A batch of bt[n][k] matrices in one grid, against one launch per matrix: one
// grid when its tiles come near to filling the chip, or when the chain of K
// stages one workgroup walks (about 0.5 us each) is shorter than the launches
// it replaces (5 - 8 us each). Up to 16 rows the launches are the streaming
// GEMV, which reads a large matrix faster than the tiles, so there only the
// chain counts. Measured, one launch per matrix -> one grid, bf16 us: 128 x
// [512, 128, K 512] 580 -> 32; 3 x [512, 4096, K 4096] 90 -> 65; 8 x [200,
// 4096, K 512] 54 -> 24; 64 x [4, 128, K 2048] 241 -> 24; 4 x [1, 4096, K
// 4096] 31.5 against 33.5 (stays).
static inline bool gen_batch(int64_t batch, int64_t M, int64_t N, int64_t K) {
  if (batch < 2) return false;
  if (M <= 16) return N * K < ((int64_t)1 << 25) && K <= 640 * (batch - 1);
  const GenPlan p = gen_plan(batch, M, N, K, kBRows);
  return gen_tiles(batch, M, N, p.form) >= 192 || K <= 512 * (batch - 1);
}

// Operands a launch of `mode` can address: 32-bit byte offsets within a tile
// row range (kBRows) or within the whole of b (kBColumns).
static inline bool gen_fits(BMode mode, int64_t lda, int64_t ldb, int64_t K) {
  if (lda >= kBigMaxLd || lda % 8 || ldb % 8) return false;
  return mode == kBColumns ? (K + 512) * ldb < ((int64_t)1 << 30) : ldb < kBigMaxLd;
}

template <typename T, BMode MODE, int WM, int BN>
static void launch_gen_big(const T* a, int64_t lda, const T* b, int64_t ldb, T* out, int batch, BatchStride bs, int M,
                           int N, int K, hipStream_t st) {
  const int tm = ceil_div(M, 64 * WM), tn = ceil_div(N, BN);
  const dim3 grid((tm * tn + 7) / 8 * 8, batch);
  gemm_big<T, WM, BN, MODE><<<grid, big_threads<WM, BN>(), 0, st>>>(a, lda, b, ldb, out, M, N, K, tm, tn, bs);
}

template <typename T, BMode MODE, int TI, int RMAX>
static void launch_gen_tall(const T* a, int64_t lda, const T* b, int64_t ldb, T* out, float* ws, int batch,
                            BatchStride bs, int M, int N, int K, const GenPlan& p, hipStream_t st) {
  const int G = ceil_div(K, kGroupK);
  if constexpr (MODE == kBColumns) {
    if (p.chunks > 1) {                       // few tiles: batch * chunks stays below 65,536
      const dim3 grid(ceil_div(N, 64), ceil_div(M, 16 * TI), batch * p.chunks);
      bs.chunks = p.chunks;
      gemm_tall<T, TI, 1, 4, 64, true, RMAX, MODE><<<grid, 256, 0, st>>>(a, lda, b, ldb, out, ws, M, N, K, G, p.cg, bs);
      const int64_t MN = (int64_t)M * N;
      const dim3 fold((unsigned)((MN + 255) / 256), batch);
      if (batch == 1) fold_groups<T><<<fold, 256, 0, st>>>(ws, out, MN, G);
      else fold_groups_batch<T><<<fold, 256, 0, st>>>(ws, out, MN, G, bs.out);
      return;
    }
  }
  const dim3 grid(ceil_div(N, 64), ceil_div(M, 16 * TI), batch);
  gemm_tall<T, TI, 1, 4, 64, false, RMAX, MODE><<<grid, 256, 0, st>>>(a, lda, b, ldb, out, ws, M, N, K, G, G, bs);
}

template <typename T, BMode MODE>
static void launch_gen(const GenPlan& p, const T* a, int64_t lda, const T* b, int64_t ldb, T* out, float* ws,
                       int64_t batch, BatchStride bs, int M, int N, int K, hipStream_t st) {
  constexpr int64_t kMost = 65535;  // matrices per launch (grid.y / grid.z)
  for (int64_t i = 0; i < batch; i += kMost) {
    const int n = (int)std::min<int64_t>(kMost, batch - i);
    const T* ai = a + i * bs.a;
    const T* bi_ = b + i * bs.b;
    T* oi = out + i * bs.out;
    switch (p.form) {
      case kGen256x128: launch_gen_big<T, MODE, 4, 128>(ai, lda, bi_, ldb, oi, n, bs, M, N, K, st); break;
      case kGen128x128: launch_gen_big<T, MODE, 2, 128>(ai, lda, bi_, ldb, oi, n, bs, M, N, K, st); break;
      case kGen128x64: launch_gen_big<T, MODE, 2, 64>(ai, lda, bi_, ldb, oi, n, bs, M, N, K, st); break;
      case kGen64x64: launch_gen_tall<T, MODE, 4, 4>(ai, lda, bi_, ldb, oi, ws, n, bs, M, N, K, p, st); break;
      default: launch_gen_tall<T, MODE, 2, 5>(ai, lda, bi_, ldb, oi, ws, n, bs, M, N, K, p, st); break;
    }
  }
}

// bi_matmul_gen.hip: one launch (or grid.y / grid.z rounds of one) per call.
int gen_matmul_bf16(BMode mode, const void* a, int64_t lda, const void* b, int64_t ldb, void* out, void* ws,
                    int64_t batch, BatchStride bs, int M, int N, int K, hipStream_t st, const char* what);
int gen_matmul_f16(BMode mode, const void* a, int64_t lda, const void* b, int64_t ldb, void* out, void* ws,
                   int64_t batch, BatchStride bs, int M, int N, int K, hipStream_t st, const char* what);

}  // namespace bi
