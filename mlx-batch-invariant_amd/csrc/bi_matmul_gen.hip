// bi_matmul_gen.hip — the dense tiles of bi_gemm_gen.h (a batch of matrices in
// one grid, a row-major right-hand side, K not a multiple of 64), in a
// translation unit of their own so the build compiles them in parallel.
#include "bi_gemm_gen.h"

namespace bi {

template <typename T>
static int gen_matmul(BMode mode, const void* a, int64_t lda, const void* b, int64_t ldb, void* out, void* ws,
                      int64_t batch, BatchStride bs, int M, int N, int K, hipStream_t st, const char* what) {
  const GenPlan p = gen_plan(batch, M, N, K, mode, ws != nullptr);
  const T* ap = static_cast<const T*>(a);
  const T* bp = static_cast<const T*>(b);
  T* op = static_cast<T*>(out);
  if (mode == kBColumns)
    launch_gen<T, kBColumns>(p, ap, lda, bp, ldb, op, static_cast<float*>(ws), batch, bs, M, N, K, st);
  else launch_gen<T, kBRows>(p, ap, lda, bp, ldb, op, static_cast<float*>(ws), batch, bs, M, N, K, st);
  return bi_host::launch_status(what);
}

int gen_matmul_bf16(BMode mode, const void* a, int64_t lda, const void* b, int64_t ldb, void* out, void* ws,
                    int64_t batch, BatchStride bs, int M, int N, int K, hipStream_t st, const char* what) {
  return gen_matmul<bf16>(mode, a, lda, b, ldb, out, ws, batch, bs, M, N, K, st, what);
}
int gen_matmul_f16(BMode mode, const void* a, int64_t lda, const void* b, int64_t ldb, void* out, void* ws,
                   int64_t batch, BatchStride bs, int M, int N, int K, hipStream_t st, const char* what) {
  return gen_matmul<f16>(mode, a, lda, b, ldb, out, ws, batch, bs, M, N, K, st, what);
}

}  // namespace bi
