// int8_row codec on gfx950: decode (bit-exact with the reference decode) and encode.
//
// Format (selas/codecs.py:86-96): a weight [rows, ...] is stored as q, int8 of
// the same shape, and one fp32 scale per row: scale = absmax(row) / 127 (1 for
// an all-zero row), q = clamp(round_half_even(w / scale), -127, 127).
// Decode (selas/codecs.py:273-277) computes q.to(dt) * scale.to(dt) in the
// output type dt: q converts exactly, the scale is rounded to dt, and their
// product (exact in fp32 for bf16 and fp16) is rounded once to dt.
#include "common.h"

namespace selas {
namespace {

constexpr int kThreads = 256;

// The row scale as the reference's decode sees it: rounded to the output type.
template <int DT>
__device__ __forceinline__ float scale_as(float s) {
  if constexpr (DT == SELAS_F32) return s;
  else if constexpr (DT == SELAS_F16) return f16_bits_to_f32(f16_bits_rne(s));
  else return bf16_bits_to_f32(bf16_bits_rne(s));
}

// --------------------------------------------------------------------------- decode

// Vector path (cols % 8 == 0): lane i of a wave decodes 8-byte chunk i of 64 consecutive ones, so that its 16-byte
// stores (fp32: two) and the loads cover consecutive addresses; each thread takes kDequantPer chunks, kThreads apart,
// all loaded before the first is decoded. HBM-bound: 19.6 us for a 12288 x 3072 weight to bf16, 5.8 TB/s (fp32 39.5
// us); with 16 values per lane, stores 32 bytes apart and a 64-bit division for the row, 20.5 us (54.1).
constexpr int kDequantPer = 2;

template <int DT>
__global__ __launch_bounds__(kThreads) void int8_row_dequant_vec8(const uint2 *__restrict__ q,
                                                                  const float *__restrict__ scale, uint32_t n8,
                                                                  FastDiv chunks_per_row, void *__restrict__ out) {
  const uint32_t i0 = blockIdx.x * (kThreads * kDequantPer) + threadIdx.x;
  uint2 w[kDequantPer];
  float s[kDequantPer];
#pragma unroll
  for (int j = 0; j < kDequantPer; ++j) {
    const uint32_t i = i0 + j * kThreads;
    w[j] = i < n8 ? q[i] : make_uint2(0u, 0u);
    s[j] = i < n8 ? scale_as<DT>(scale[div31(i, chunks_per_row)]) : 0.0f;
  }
#pragma unroll
  for (int j = 0; j < kDequantPer; ++j) {
    const uint32_t i = i0 + j * kThreads;
    if (i >= n8) return;
    const uint32_t words[2] = {w[j].x, w[j].y};
    float v[8];
#pragma unroll
    for (int t = 0; t < 8; ++t)
      v[t] = static_cast<float>(static_cast<int8_t>((words[t >> 2] >> (8 * (t & 3))) & 0xffu)) * s[j];
    if constexpr (DT == SELAS_F32) {
      float4 *o = reinterpret_cast<float4 *>(out) + static_cast<int64_t>(i) * 2;
      o[0] = make_float4(v[0], v[1], v[2], v[3]);
      o[1] = make_float4(v[4], v[5], v[6], v[7]);
    } else {
      uint32_t pr[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if constexpr (DT == SELAS_BF16)
          pr[t] = bf16_bits_rne(v[2 * t]) | (static_cast<uint32_t>(bf16_bits_rne(v[2 * t + 1])) << 16);
        else
          pr[t] = f16_bits_rne(v[2 * t]) | (static_cast<uint32_t>(f16_bits_rne(v[2 * t + 1])) << 16);
      }
      reinterpret_cast<uint4 *>(out)[i] = make_uint4(pr[0], pr[1], pr[2], pr[3]);
    }
  }
}

// Generic path: one value per thread.
template <int DT>
__global__ __launch_bounds__(kThreads) void int8_row_dequant_elems(const int8_t *__restrict__ q,
                                                                   const float *__restrict__ scale, int64_t n,
                                                                   int64_t cols, void *__restrict__ out) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (i >= n) return;
  store_f<DT>(out, i, static_cast<float>(q[i]) * scale_as<DT>(scale[i / cols]));
}

template <int DT>
int dequant_typed(const int8_t *q, const float *scale, int64_t rows, int64_t cols, void *out, hipStream_t stream) {
  const int64_t n = rows * cols;
  if (cols % 8 == 0 && aligned(q, 8) && aligned(out, 16) && n / 8 < (1ll << 31) - 4096) {
    const int64_t n8 = n / 8;
    int8_row_dequant_vec8<DT><<<dim3(static_cast<uint32_t>(cdiv(n8, kThreads * kDequantPer))), dim3(kThreads), 0,
                                stream>>>(reinterpret_cast<const uint2 *>(q), scale, static_cast<uint32_t>(n8),
                                          fast_div(static_cast<uint32_t>(cols / 8)), out);
  } else {
    int8_row_dequant_elems<DT><<<dim3(static_cast<uint32_t>(cdiv(n, kThreads))), dim3(kThreads), 0, stream>>>(
        q, scale, n, cols, out);
  }
  return check_launch("int8_row_dequant");
}

// --------------------------------------------------------------------------- encode

// NaN-propagating max, as torch.amax.
__device__ __forceinline__ float max_nan(float a, float b) {
  if (a != a) return a;
  if (b != b) return b;
  return a > b ? a : b;
}

// q of one element by IEEE division and round half to even (torch.round). NaN gives -127, as the clamp does.
__device__ __forceinline__ int quantize(float w, float sc) {
  return static_cast<int>(fminf(fmaxf(rintf(w / sc), -127.0f), 127.0f));
}

// Rows of 8 * R * kThreads elements at most, 16-byte aligned: one workgroup per row, which stays in registers between
// the maximum and the rounding (16-byte loads, 8-byte stores). An element is multiplied by the reciprocal of the scale,
// at most 3e-5 from w / scale; a thread with an element that close to a half, and rows without a safe reciprocal
// (scale subnormal, huge, Inf, NaN), divide theirs, so every element has the value of the division.
// HBM-bound: 26 us for a 12288 x 3072 bf16 weight, 4.3 TB/s (fp32 35 us); a 4-byte load per element, twice, and a
// division each took 86 us for the fp32 weight and 12 more for a bf16 weight's conversion.
template <int DT, int R>
__global__ __launch_bounds__(kThreads) void int8_row_encode_vec(const void *__restrict__ w, int64_t rows, int cols8,
                                                                uint2 *__restrict__ q, float *__restrict__ scale) {
  __shared__ uint32_t part[2][kThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int buf = 0;
  for (int64_t r = blockIdx.x; r < rows; r += gridDim.x, buf ^= 1) {
    float v[R][8];
    uint32_t m = 0;  // magnitude bits order like the values, NaN above Inf: the maximum propagates NaN
#pragma unroll
    for (int c = 0; c < R; ++c) {
      const int i = tid + c * kThreads;
      if (i < cols8) m = max(m, load8<DT>(w, r * cols8 + i, v[c]));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = max(m, static_cast<uint32_t>(__shfl_xor(static_cast<int>(m), o, 64)));
    if (lane == 0) part[buf][wave] = m;
    __syncthreads();  // one barrier a row: the next row writes the other buffer
    m = max(max(part[buf][0], part[buf][1]), max(part[buf][2], part[buf][3]));
    const float a = __uint_as_float(m), sc = a > 0.0f ? a / 127.0f : 1.0f;
    const bool plain = sc > 0x1p-100f && sc < 0x1p100f && a == a;
    const float inv = 1.0f / sc;
#pragma unroll
    for (int c = 0; c < R; ++c) {
      const int i = tid + c * kThreads;
      if (i >= cols8) break;
      int qi[8];
      float off = 0.0f;
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const float x = v[c][t] * inv, n = rintf(x);
        off = fmaxf(off, fabsf(x - n));
        qi[t] = static_cast<int>(__builtin_amdgcn_fmed3f(n, -127.0f, 127.0f));
      }
      if (!plain || off > 0.4999f) {
#pragma unroll
        for (int t = 0; t < 8; ++t) qi[t] = quantize(v[c][t], sc);
      }
      uint32_t o[2];
#pragma unroll
      for (int h = 0; h < 2; ++h)
        o[h] = (qi[4 * h] & 0xff) | ((qi[4 * h + 1] & 0xff) << 8) | ((qi[4 * h + 2] & 0xff) << 16) |
               (static_cast<uint32_t>(qi[4 * h + 3]) << 24);
      q[r * cols8 + i] = make_uint2(o[0], o[1]);
    }
    if (tid == 0) scale[r] = sc;
  }
}

// Any shape and alignment, fp32 input. One workgroup per row (grid-stride): |w| max over the row, scale = max / 127
// (1 when the max is not positive, as torch.where(absmax > 0, ...) picks), then
// q = clamp(rint(w / scale), -127, 127) with IEEE division and round half to even
// (torch.round).
__global__ __launch_bounds__(kThreads) void int8_row_encode_rows(const float *__restrict__ w, int64_t rows,
                                                                 int64_t cols, int8_t *__restrict__ q,
                                                                 float *__restrict__ scale) {
  __shared__ float part[kThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
    const float *src = w + r * cols;
    float m = 0.0f;
    for (int64_t j = tid; j < cols; j += kThreads) m = max_nan(m, fabsf(src[j]));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = max_nan(m, __shfl_xor(m, o, 64));
    if (lane == 0) part[wave] = m;
    __syncthreads();
    m = max_nan(max_nan(part[0], part[1]), max_nan(part[2], part[3]));
    __syncthreads();  // part is rewritten by the next row
    const float sc = m > 0.0f ? m / 127.0f : 1.0f;
    for (int64_t j = tid; j < cols; j += kThreads) {
      q[r * cols + j] = static_cast<int8_t>(quantize(src[j], sc));
    }
    if (tid == 0) scale[r] = sc;
  }
}

}  // namespace
}  // namespace selas

using namespace selas;

extern "C" int selas_int8_row_dequant(const int8_t *q, const float *scale, int64_t rows, int64_t cols, void *out,
                                      int out_dtype, void *stream) {
  if (rows < 0 || cols < 0)
    return set_error(SELAS_EINVAL, "int8_row_dequant: bad shape %lld x %lld", (long long)rows, (long long)cols);
  if (!valid_dtype(out_dtype)) return set_error(SELAS_EINVAL, "int8_row_dequant: bad output dtype %d", out_dtype);
  if (rows == 0 || cols == 0) return ok();
  if (!q || !scale || !out) return set_error(SELAS_EINVAL, "int8_row_dequant: null pointer");
  if (rows * cols / kThreads >= (1ll << 31))
    return set_error(SELAS_EUNSUPPORTED, "int8_row_dequant: %lld elements exceed one launch", (long long)(rows * cols));
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (out_dtype) {
    case SELAS_F32: return dequant_typed<SELAS_F32>(q, scale, rows, cols, out, s);
    case SELAS_F16: return dequant_typed<SELAS_F16>(q, scale, rows, cols, out, s);
    default: return dequant_typed<SELAS_BF16>(q, scale, rows, cols, out, s);
  }
}

namespace {
template <int DT>
void launch_encode_vec(const void *w, int64_t rows, int64_t cols, int8_t *q, float *scale, hipStream_t st) {
  const dim3 grid(static_cast<uint32_t>(rows < 65536 ? rows : 65536)), blk(kThreads);
  const int c8 = static_cast<int>(cols / 8);
  uint2 *q8 = reinterpret_cast<uint2 *>(q);
  if (c8 <= 2 * kThreads) int8_row_encode_vec<DT, 2><<<grid, blk, 0, st>>>(w, rows, c8, q8, scale);
  else if (c8 <= 4 * kThreads) int8_row_encode_vec<DT, 4><<<grid, blk, 0, st>>>(w, rows, c8, q8, scale);
  else int8_row_encode_vec<DT, 8><<<grid, blk, 0, st>>>(w, rows, c8, q8, scale);
}

int encode_any(const char *what, const void *w, int w_dtype, int64_t rows, int64_t cols, int8_t *q, float *scale,
               hipStream_t st) {
  if (rows < 0 || cols < 0)
    return set_error(SELAS_EINVAL, "%s: bad shape %lld x %lld", what, (long long)rows, (long long)cols);
  if (!valid_dtype(w_dtype)) return set_error(SELAS_EINVAL, "%s: bad input dtype %d", what, w_dtype);
  if (rows == 0) return ok();
  if (!w || !q || !scale) return set_error(SELAS_EINVAL, "%s: null pointer", what);
  if (cols % 8 == 0 && cols > 0 && cols <= 8 * 8 * kThreads && aligned(w, 16) && aligned(q, 8)) {
    switch (w_dtype) {
      case SELAS_F32: launch_encode_vec<SELAS_F32>(w, rows, cols, q, scale, st); break;
      case SELAS_F16: launch_encode_vec<SELAS_F16>(w, rows, cols, q, scale, st); break;
      default: launch_encode_vec<SELAS_BF16>(w, rows, cols, q, scale, st);
    }
    return check_launch(what);
  }
  if (w_dtype != SELAS_F32)
    return set_error(SELAS_EUNSUPPORTED, "%s: 16-bit input needs rows of 8 to %d elements, a multiple of 8, 16-byte "
                                         "aligned", what, 8 * 8 * kThreads);
  const int64_t grid = rows < 65536 ? rows : 65536;
  int8_row_encode_rows<<<dim3(static_cast<uint32_t>(grid)), dim3(kThreads), 0, st>>>(static_cast<const float *>(w), rows,
                                                                                     cols, q, scale);
  return check_launch(what);
}
}  // namespace

extern "C" int selas_int8_row_encode(const float *w, int64_t rows, int64_t cols, int8_t *q, float *scale,
                                     void *stream) {
  return encode_any("int8_row_encode", w, SELAS_F32, rows, cols, q, scale, static_cast<hipStream_t>(stream));
}

extern "C" int selas_int8_row_encode_typed(const void *w, int w_dtype, int64_t rows, int64_t cols, int8_t *q,
                                           float *scale, void *stream) {
  return encode_any("int8_row_encode_typed", w, w_dtype, rows, cols, q, scale, static_cast<hipStream_t>(stream));
}
