// bi_pad.hip — rows of any length and alignment copied into 16-byte aligned rows
// zero-padded to a given length: what the matmul kernels read in place of an
// operand whose inner size is not a multiple of 8 or whose rows are not
// 16-byte aligned.
//
// Bound by memory: each element is read once and each output byte written once
// (as a zero fill and a strided elementwise copy the output was written twice,
// an element at a time). One thread per 16 output bytes, the source read as
// 16 bytes at its own alignment (global loads need none); the last chunk of a
// row by element. bf16 [14299, 4067]: zero fill and copy 60 us, this 38.
#include <algorithm>

#include "bi_common.h"

namespace bi {

template <typename E>
__global__ __launch_bounds__(256) void pad_rows_kernel(const E* __restrict__ in, int64_t bs, int64_t rs,
                                                       E* __restrict__ out, int64_t rows, int64_t out_bs, int cols,
                                                       int chunks) {
  constexpr int kE = 16 / (int)sizeof(E);
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (id >= rows * chunks) return;
  const int64_t row = id / chunks;
  const int c = (int)(id % chunks) * kE;
  const E* src = in + blockIdx.y * bs + row * rs + c;
  u32x4 v = {0u, 0u, 0u, 0u};
  if (c + kE <= cols) {
    __builtin_memcpy(&v, src, 16);
  } else {
    E e[kE];
#pragma unroll
    for (int i = 0; i < kE; ++i) e[i] = c + i < cols ? src[i] : (E)0;
    __builtin_memcpy(&v, e, 16);
  }
  *reinterpret_cast<u32x4*>(out + blockIdx.y * out_bs + row * chunks * kE + c) = v;
}

}  // namespace bi

extern "C" int bi_pad_rows(const void* in, int64_t batch_stride, int64_t row_stride, void* out, int64_t batch,
                           int64_t rows, int64_t cols, int64_t cols_out, int elem_bytes, void* stream) {
  using namespace bi_host;
  const char* what = "bi_pad_rows";
  if (elem_bytes != 2 && elem_bytes != 4) return fail(BI_E_UNSUPPORTED, "%s: %d-byte elements", what, elem_bytes);
  const int64_t unit = 16 / elem_bytes;
  if (batch < 0 || rows < 0 || cols < 0 || cols_out < cols || cols_out % unit || batch_stride < 0 || row_stride < 0)
    return fail(BI_E_INVALID_ARG, "%s: batch=%lld rows=%lld cols=%lld cols_out=%lld (a multiple of 16 bytes, >= cols)",
                what, (long long)batch, (long long)rows, (long long)cols, (long long)cols_out);
  if (batch == 0 || rows == 0 || cols_out == 0) return BI_OK;
  if (!in || !out || !aligned16(out) || reinterpret_cast<uintptr_t>(in) % (unsigned)elem_bytes)
    return fail(BI_E_INVALID_ARG, "%s: null or misaligned operand", what);
  const int64_t chunks = cols_out / unit;
  if (cols_out > 0x7fffffffLL || rows > 0x7fffffffLL) return fail(BI_E_UNSUPPORTED, "%s: shape too large", what);
  // A launch holds fewer than 2^32 threads (64 GiB of output): larger operands
  // take several.
  const int64_t most = std::max<int64_t>(1, ((int64_t)1 << 31) / chunks);
  hipStream_t st = static_cast<hipStream_t>(stream);
  for (int64_t b = 0; b < batch; b += 65535) {
    for (int64_t r = 0; r < rows; r += most) {
      const int64_t n = std::min(most, rows - r);
      const dim3 grid((unsigned)((n * chunks + 255) / 256), (unsigned)std::min<int64_t>(batch - b, 65535));
      const char* src = static_cast<const char*>(in) + (b * batch_stride + r * row_stride) * elem_bytes;
      char* dst = static_cast<char*>(out) + (b * rows + r) * cols_out * elem_bytes;
      if (elem_bytes == 2)
        bi::pad_rows_kernel<uint16_t><<<grid, 256, 0, st>>>(reinterpret_cast<const uint16_t*>(src), batch_stride,
                                                            row_stride, reinterpret_cast<uint16_t*>(dst), n,
                                                            rows * cols_out, (int)cols, (int)chunks);
      else
        bi::pad_rows_kernel<uint32_t><<<grid, 256, 0, st>>>(reinterpret_cast<const uint32_t*>(src), batch_stride,
                                                            row_stride, reinterpret_cast<uint32_t*>(dst), n,
                                                            rows * cols_out, (int)cols, (int)chunks);
    }
  }
  return launch_status(what);
}
