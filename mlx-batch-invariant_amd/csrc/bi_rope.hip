// bi_rope.hip — rotary embedding of a decoder block's queries and keys, and the
// write of its keys and values into the K/V cache, in one launch.
//
// Per element the same roundings as the elementwise ops it stands for (each
// product and the sum rounded to T): with the halves x1, x2 of a head,
//   y1 = T(T(x1 cos) - T(x2 sin)),  y2 = T(T(x2 cos) + T(x1 sin));
// values are copied. Every output element depends on its own inputs only.
//
// Bound by launches, not bytes: a decode step moves a few tens of KB here,
// and as 14 elementwise ops and two strided copies it took 16 launches of 2-3
// us each in a replayed graph; one thread per 8 + 8 elements of a head, one
// launch: Llama-3-8B block and head, 4-bit, B = 4 152 -> 107 us a step.
#include "bi_common.h"

namespace bi {

struct RopeArgs {
  const void *q, *k, *v, *cos, *sin;
  void *qo, *kc, *vc;
  int64_t q_row, k_row, v_row;                  // elements between tokens of q, k, v
  int64_t kc_sb, kc_sh, kc_sl, vc_sb, vc_sh, vc_sl;
  int B, T, Hq, Hkv, D, pos;
};

template <typename T>
__global__ __launch_bounds__(256) void rope_cache_kernel(RopeArgs a) {
  const int cph = a.D / 16;                     // 8 + 8 element chunks per head
  const int heads = a.Hq + 2 * a.Hkv;
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (id >= (int64_t)a.B * a.T * heads * cph) return;
  const int c = (int)(id % cph);
  const int h = (int)(id / cph % heads);
  const int64_t bt = id / cph / heads;
  const int b = (int)(bt / a.T), t = (int)(bt % a.T);
  const int half = a.D / 2, d = 8 * c;
  const bool is_q = h < a.Hq, is_k = !is_q && h < a.Hq + a.Hkv;
  const int hh = is_q ? h : is_k ? h - a.Hq : h - a.Hq - a.Hkv;
  const T* src = is_q ? static_cast<const T*>(a.q) + bt * a.q_row
                      : is_k ? static_cast<const T*>(a.k) + bt * a.k_row : static_cast<const T*>(a.v) + bt * a.v_row;
  src += (int64_t)hh * a.D + d;
  T* dst = is_q ? static_cast<T*>(a.qo) + (((int64_t)b * a.Hq + hh) * a.T + t) * a.D
                : is_k ? static_cast<T*>(a.kc) + b * a.kc_sb + hh * a.kc_sh + (int64_t)(a.pos + t) * a.kc_sl
                       : static_cast<T*>(a.vc) + b * a.vc_sb + hh * a.vc_sh + (int64_t)(a.pos + t) * a.vc_sl;
  dst += d;
  float x1[8], x2[8];
  load8<T>(src, x1);
  load8<T>(src + half, x2);
  if (is_q || is_k) {
    float co[8], si[8];
    load8<T>(static_cast<const T*>(a.cos) + (int64_t)t * half + d, co);
    load8<T>(static_cast<const T*>(a.sin) + (int64_t)t * half + d, si);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float a1 = to_f32(to_store<T>(x1[e] * co[e])), b1 = to_f32(to_store<T>(x2[e] * si[e]));
      const float a2 = to_f32(to_store<T>(x2[e] * co[e])), b2 = to_f32(to_store<T>(x1[e] * si[e]));
      x1[e] = a1 - b1;
      x2[e] = a2 + b2;
    }
  }
  store8<T>(dst, x1);
  store8<T>(dst + half, x2);
}

}  // namespace bi

extern "C" int bi_rope_cache(const void* q, int64_t q_row, const void* k, int64_t k_row, const void* v, int64_t v_row,
                             const void* cos, const void* sin, void* q_out, void* k_cache, void* v_cache, int64_t B,
                             int64_t T, int64_t Hq, int64_t Hkv, int64_t D, int64_t pos, int64_t max_len,
                             const int64_t* strides, int dtype, void* stream) {
  using namespace bi_host;
  const char* what = "bi_rope_cache";
  if (B < 0 || T < 0 || Hq <= 0 || Hkv <= 0 || D <= 0 || D % 16 || pos < 0 || pos + T > max_len || !strides)
    return fail(BI_E_INVALID_ARG, "%s: bad shape B=%lld T=%lld Hq=%lld Hkv=%lld D=%lld pos=%lld max_len=%lld", what,
                (long long)B, (long long)T, (long long)Hq, (long long)Hkv, (long long)D, (long long)pos,
                (long long)max_len);
  if (dtype != BI_BF16 && dtype != BI_F16 && dtype != BI_F32)
    return fail(BI_E_UNSUPPORTED, "%s: unknown dtype %d", what, dtype);
  if (B > 0x7fffffffLL || T > 0x7fffffffLL || max_len > 0x7fffffffLL || Hq > 65536 || Hkv > 65536 || D > 65536 ||
      B * T > ((int64_t)1 << 31) || B * T * (Hq + 2 * Hkv) * (D / 16) > ((int64_t)1 << 32) - 256)  // threads
    return fail(BI_E_UNSUPPORTED, "%s: shape too large", what);
  if (B == 0 || T == 0) return BI_OK;
  const int64_t unit = 16 / (int64_t)dtype_size(dtype);
  bool ok = q && k && v && cos && sin && q_out && k_cache && v_cache && q_row >= Hq * D && k_row >= Hkv * D &&
            v_row >= Hkv * D && q_row % unit == 0 && k_row % unit == 0 && v_row % unit == 0;
  for (const void* p : {q, k, v, cos, sin, (const void*)q_out, (const void*)k_cache, (const void*)v_cache})
    ok = ok && aligned16(p);
  for (int i = 0; i < 6; ++i) ok = ok && strides[i] >= 0 && strides[i] % unit == 0;
  if (!ok)
    return fail(BI_E_INVALID_ARG, "%s: null or misaligned operand (16-byte aligned rows, rows of at least H * D)", what);
  bi::RopeArgs a{q, k, v, cos, sin, q_out, k_cache, v_cache, q_row, k_row, v_row, strides[0], strides[1], strides[2],
                 strides[3], strides[4], strides[5], (int)B, (int)T, (int)Hq, (int)Hkv, (int)D, (int)pos};
  const int64_t n = B * T * (Hq + 2 * Hkv) * (D / 16);
  const unsigned grid = (unsigned)((n + 255) / 256);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == BI_BF16) bi::rope_cache_kernel<bi::bf16><<<grid, 256, 0, st>>>(a);
  else if (dtype == BI_F16) bi::rope_cache_kernel<bi::f16><<<grid, 256, 0, st>>>(a);
  else bi::rope_cache_kernel<float><<<grid, 256, 0, st>>>(a);
  return launch_status(what);
}
