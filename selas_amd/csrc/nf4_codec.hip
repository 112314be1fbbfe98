// NF4 codec on gfx950: decode (bit-exact with the reference decode) and encode.
//
// Decode restates selas/codecs.py:178-199 (nf4_dequant_torch) and :207-228
// (the Triton kernel): value = code[nibble] * absmax[block] in fp32, rounded
// once to the output type. Encode restates selas/codecs.py:99-119.
#include <algorithm>
#include <cstring>

#include "common.h"

namespace selas {
namespace {

constexpr int kThreads = 256;

// --------------------------------------------------------------------------- decode

// Vector path (blocksize % 8 == 0): lane i of a wave decodes dword i of 64 consecutive ones, 8 values, so that
// its 16-byte stores (fp32: two) and the loads cover consecutive addresses; each thread takes kDequantPer dwords,
// kThreads apart, all loaded before the first is decoded. HBM-bound: 16.5 us for a 12288 x 3072 weight to bf16, 5.9
// TB/s (fp32 37.7 us); with 16 bytes read per lane and its four stores 64 bytes apart, 26.2 us (60.6).
constexpr int kDequantPer = 4;

template <int DT>
__global__ __launch_bounds__(kThreads) void nf4_dequant_vec4(const uint32_t *__restrict__ packed,
                                                             const float *__restrict__ absmax, uint32_t n4,
                                                             FastDiv dwords_per_block, Code16 code,
                                                             void *__restrict__ out) {
  __shared__ float s_code[16];
  if (threadIdx.x < 16) s_code[threadIdx.x] = code.v[threadIdx.x];
  __syncthreads();
  const uint32_t i0 = blockIdx.x * (kThreads * kDequantPer) + threadIdx.x;
  uint32_t w[kDequantPer];
  float a[kDequantPer];
#pragma unroll
  for (int j = 0; j < kDequantPer; ++j) {
    const uint32_t i = i0 + j * kThreads;
    w[j] = i < n4 ? packed[i] : 0u;
    a[j] = i < n4 ? absmax[div31(i, dwords_per_block)] : 0.0f;
  }
#pragma unroll
  for (int j = 0; j < kDequantPer; ++j) {
    const uint32_t i = i0 + j * kThreads;
    if (i >= n4) return;
    float v[8];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const uint32_t byte = (w[j] >> (8 * t)) & 0xffu;
      v[2 * t] = s_code[byte >> 4] * a[j];
      v[2 * t + 1] = s_code[byte & 15u] * a[j];
    }
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

// Generic path: one byte per thread, any even blocksize and any alignment.
template <int DT>
__global__ __launch_bounds__(kThreads) void nf4_dequant_bytes(const uint8_t *__restrict__ packed,
                                                              const float *__restrict__ absmax, int64_t begin,
                                                              int64_t n_bytes, int64_t bytes_per_block, Code16 code,
                                                              void *__restrict__ out) {
  __shared__ float s_code[16];
  if (threadIdx.x < 16) s_code[threadIdx.x] = code.v[threadIdx.x];
  __syncthreads();
  const int64_t i = begin + static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (i >= n_bytes) return;
  const uint32_t byte = packed[i];
  const float a = absmax[i / bytes_per_block];
  store_f<DT>(out, 2 * i, s_code[byte >> 4] * a);
  store_f<DT>(out, 2 * i + 1, s_code[byte & 15u] * a);
}

template <int DT>
int dequant_typed(const uint8_t *packed, const float *absmax, int64_t n_bytes, int64_t bpb, const Code16 &code,
                  void *out, hipStream_t stream) {
  int64_t done = 0;
  if (bpb % 4 == 0 && aligned(packed, 4) && aligned(out, 16) && n_bytes >= 4 && n_bytes / 4 < (1ll << 31) - 4096) {
    const int64_t n4 = n_bytes / 4;
    const int64_t grid = cdiv(n4, kThreads * kDequantPer);
    // The dwords past a first block of more than n4 do not exist: n4 gives the same quotients, 0, in 32 bits.
    const FastDiv per_block = fast_div(static_cast<uint32_t>(std::min(bpb / 4, n4)));
    nf4_dequant_vec4<DT><<<dim3(static_cast<uint32_t>(grid)), dim3(kThreads), 0, stream>>>(
        reinterpret_cast<const uint32_t *>(packed), absmax, static_cast<uint32_t>(n4), per_block, code, out);
    done = n4 * 4;
  }
  if (done < n_bytes) {
    const int64_t grid = cdiv(n_bytes - done, kThreads);
    nf4_dequant_bytes<DT><<<dim3(static_cast<uint32_t>(grid)), dim3(kThreads), 0, stream>>>(
        packed, absmax, done, n_bytes, bpb, code, out);
  }
  return check_launch("nf4_dequant");
}

// --------------------------------------------------------------------------- encode

struct Mids15 {
  float v[15];
};

// NaN-propagating max, as torch.amax.
__device__ __forceinline__ float max_nan(float a, float b) {
  if (a != a) return a;
  if (b != b) return b;
  return a > b ? a : b;
}

// Code index of x: the number of midpoints m with !(m >= x) (torch.bucketize with right=False counts exactly these).
__device__ __forceinline__ uint32_t code_index(float x, const Mids15 &mids) {
  uint32_t idx = 0;
#pragma unroll
  for (int t = 0; t < 15; ++t) idx += !(mids.v[t] >= x) ? 1u : 0u;
  return idx;
}

// Search table over 64 equal buckets of [-1, 1], each with at most one midpoint: the midpoint's bits with the low four
// replaced by the number of midpoints in lower buckets (4.0, above every x, where there is no midpoint). 64 words in LDS
// (1.4 conflict cycles counted per LDS instruction of the kernel, the maximum's shuffles included; HBM-bound with them).
struct SearchTable {
  uint32_t e[64];
};
__host__ __device__ __forceinline__ float bucket_of(float x) { return __builtin_fmaf(x, 31.999f, 32.0f); }
// x = w * (1 / absmax) is within 2e-7 of w / absmax, and an entry within 16 ulp (1e-6) of its midpoint: closer than
// this the elements are divided and searched exactly. x meets only the entry of its own bucket, so search_table takes
// no midpoint from which x could be off into the next bucket.
constexpr float kNearMid = 2e-6f;

// Blocks of 64, 16-byte aligned input. Eight lanes per block, eight consecutive elements per lane: 16-byte loads (fp32:
// two), one dword of codes stored per lane; each thread takes kEncodePer dwords, kThreads apart, all loaded first.
// An element costs a multiplication by the block's reciprocal, its bucket, one table read, one comparison with the
// entry and the check that the comparison cannot be off (11 VALU); a thread with an element near a midpoint, and
// blocks whose absmax has no safe reciprocal (0, subnormal, huge, Inf, NaN), redo theirs by IEEE division and 15
// comparisons, which gives every element the code that alone would. A wave per block with that for every element was
// VALU-bound: 240 us for a 21504 x 3072 weight, and 57 us more for a bf16 weight's conversion to fp32; this takes
// 37 us for the bf16 weight, 4.6 TB/s.
constexpr int kEncodePer = 2;

template <int DT>
__global__ __launch_bounds__(kThreads) void nf4_encode_64(const void *__restrict__ w, int64_t n8, Mids15 mids,
                                                          SearchTable table, uint32_t *__restrict__ packed,
                                                          float *__restrict__ absmax) {
  __shared__ uint32_t entry[64];
  if (threadIdx.x < 64) entry[threadIdx.x] = table.e[threadIdx.x];
  __syncthreads();
  const int64_t i0 = static_cast<int64_t>(blockIdx.x) * (kThreads * kEncodePer) + threadIdx.x;
  float v[kEncodePer][8];
  uint32_t m[kEncodePer];
#pragma unroll
  for (int j = 0; j < kEncodePer; ++j) {
    m[j] = 0;
    const int64_t i = i0 + j * kThreads;  // n8 is a multiple of 8: a block's eight lanes are all in or all out
    if (i < n8) m[j] = load8<DT>(w, i, v[j]);
  }
#pragma unroll
  for (int j = 0; j < kEncodePer; ++j) {
    const int64_t i = i0 + j * kThreads;
    if (i >= n8) return;
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) m[j] = max(m[j], static_cast<uint32_t>(__shfl_xor(static_cast<int>(m[j]), o, 64)));
    const float a = __uint_as_float(m[j]);
    const bool plain = a > 0x1p-100f && a < 0x1p100f;
    const float r = 1.0f / a;
    uint32_t codes = 0;
    float near = 1.0f;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const float x = v[j][t ^ 1] * r;  // element 2i goes to the high nibble of byte i
      const uint32_t e = entry[static_cast<uint32_t>(__builtin_amdgcn_fmed3f(bucket_of(x), 0.0f, 63.0f))];
      const float mid = __uint_as_float(e);
      near = fminf(near, fabsf(x - mid));
      const uint32_t c = e + (x > mid ? 1u : 0u);
      codes = __builtin_amdgcn_alignbit(c, codes, 4);  // low four bits of c into the top nibble
    }
    if (!plain || near < kNearMid) {
      const float safe = a > 0.0f ? a : 1.0f;
      codes = 0;
      for (int t = 0; t < 8; ++t) {
        float x = v[j][0];
#pragma unroll
        for (int k = 1; k < 8; ++k) x = (t ^ 1) == k ? v[j][k] : x;
        codes |= code_index(x / safe, mids) << (4 * t);
      }
    }
    packed[i] = codes;
    if ((threadIdx.x & 7) == 0) absmax[i >> 3] = a;
  }
}

// Fills `table` when nf4_encode_64 can use these midpoints: ascending, at most one per bucket, and none within kNearMid
// of its bucket's edges. (0 lies on an edge and may: x has the sign of w / absmax, and below 1e-6 bucket_of rounds to
// the edge, whose bucket holds the entry.)
bool search_table(const Mids15 &mids, SearchTable &table) {
  int bucket[15];
  for (int i = 0; i < 15; ++i) {
    if (!(mids.v[i] > -1.0f && mids.v[i] < 1.0f) || (i > 0 && !(mids.v[i] > mids.v[i - 1]))) return false;
    bucket[i] = static_cast<int>(bucket_of(mids.v[i]));
    if (i > 0 && bucket[i] == bucket[i - 1]) return false;
    if (mids.v[i] != 0.0f && (static_cast<int>(bucket_of(mids.v[i] - kNearMid)) != bucket[i] ||
                              static_cast<int>(bucket_of(mids.v[i] + kNearMid)) != bucket[i]))
      return false;
  }
  int below = 0;
  for (int b = 0; b < 64; ++b) {
    const bool here = below < 15 && bucket[below] == b;
    uint32_t bits = 0x40800000u;
    if (here) std::memcpy(&bits, &mids.v[below], 4);
    table.e[b] = (bits & ~15u) | static_cast<uint32_t>(below);
    below += here;
  }
  return true;
}

// Any blocksize and alignment, fp32 input. One wavefront per block: |w| max across the block, then each element's code
// index, packed two per byte, first element high.
__global__ __launch_bounds__(kThreads) void nf4_encode_waves(const float *__restrict__ w, int64_t nblocks,
                                                             int blocksize, Mids15 mids, uint8_t *__restrict__ packed,
                                                             float *__restrict__ absmax) {
  const int lane = threadIdx.x & 63;
  const int64_t wave = (static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x) >> 6;
  const int64_t nwaves = (static_cast<int64_t>(gridDim.x) * kThreads) >> 6;
  for (int64_t b = wave; b < nblocks; b += nwaves) {
    const float *src = w + b * blocksize;
    float m = 0.0f;
    for (int j = lane; j < blocksize; j += 64) m = max_nan(m, fabsf(src[j]));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = max_nan(m, __shfl_xor(m, o, 64));
    const float safe = m > 0.0f ? m : 1.0f;
    for (int j0 = 0; j0 < blocksize; j0 += 64) {
      const int j = j0 + lane;
      uint32_t idx = 0;
      if (j < blocksize) idx = code_index(src[j] / safe, mids);
      const uint32_t next = __shfl_down(idx, 1, 64);
      if (j < blocksize && (lane & 1) == 0) packed[(b * blocksize + j) >> 1] = static_cast<uint8_t>((idx << 4) | next);
    }
    if (lane == 0) absmax[b] = m;
  }
}

}  // namespace
}  // namespace selas

using namespace selas;

extern "C" int selas_nf4_dequant(const uint8_t *packed, const float *absmax, int64_t n_bytes, int64_t blocksize,
                                 const float code[16], void *out, int out_dtype, void *stream) {
  if (n_bytes < 0) return set_error(SELAS_EINVAL, "nf4_dequant: negative byte count %lld", (long long)n_bytes);
  if (blocksize <= 0 || blocksize % 2)
    return set_error(SELAS_EINVAL, "nf4_dequant: blocksize must be positive and even, got %lld", (long long)blocksize);
  if (!valid_dtype(out_dtype)) return set_error(SELAS_EINVAL, "nf4_dequant: bad output dtype %d", out_dtype);
  if (n_bytes == 0) return ok();
  if (!packed || !absmax || !out || !code) return set_error(SELAS_EINVAL, "nf4_dequant: null pointer");
  Code16 c;
  for (int i = 0; i < 16; ++i) c.v[i] = code[i];
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t bpb = blocksize / 2;
  switch (out_dtype) {
    case SELAS_F32: return dequant_typed<SELAS_F32>(packed, absmax, n_bytes, bpb, c, out, s);
    case SELAS_F16: return dequant_typed<SELAS_F16>(packed, absmax, n_bytes, bpb, c, out, s);
    default: return dequant_typed<SELAS_BF16>(packed, absmax, n_bytes, bpb, c, out, s);
  }
}

namespace {
int encode_any(const char *what, const void *w, int w_dtype, int64_t n, int64_t blocksize, const float *code,
               uint8_t *packed, float *absmax, hipStream_t stream) {
  if (blocksize <= 0 || blocksize % 2 || blocksize > (1 << 20))
    return set_error(SELAS_EINVAL, "%s: blocksize must be positive and even, got %lld", what, (long long)blocksize);
  if (n < 0 || n % blocksize)
    return set_error(SELAS_EINVAL, "nf4 needs numel divisible by blocksize (%lld %% %lld)", (long long)n,
                     (long long)blocksize);
  if (!valid_dtype(w_dtype)) return set_error(SELAS_EINVAL, "%s: bad input dtype %d", what, w_dtype);
  if (n == 0) return ok();
  if (!w || !packed || !absmax || !code) return set_error(SELAS_EINVAL, "%s: null pointer", what);
  Mids15 mids;
  // Midpoints in fp32 exactly as (code[1:] + code[:-1]) / 2 evaluates them.
  for (int i = 0; i < 15; ++i) mids.v[i] = (code[i + 1] + code[i]) / 2.0f;
  SearchTable table;
  if (blocksize == 64 && aligned(w, 16) && aligned(packed, 4) && search_table(mids, table)) {
    const int64_t n8 = n / 8, grid = cdiv(n8, kThreads * kEncodePer);
    if (grid >= (1ll << 31)) return set_error(SELAS_EUNSUPPORTED, "%s: too many elements", what);
    const dim3 g(static_cast<uint32_t>(grid)), b(kThreads);
    uint32_t *p4 = reinterpret_cast<uint32_t *>(packed);
    switch (w_dtype) {
      case SELAS_F32: nf4_encode_64<SELAS_F32><<<g, b, 0, stream>>>(w, n8, mids, table, p4, absmax); break;
      case SELAS_F16: nf4_encode_64<SELAS_F16><<<g, b, 0, stream>>>(w, n8, mids, table, p4, absmax); break;
      default: nf4_encode_64<SELAS_BF16><<<g, b, 0, stream>>>(w, n8, mids, table, p4, absmax);
    }
    return check_launch(what);
  }
  if (w_dtype != SELAS_F32)
    return set_error(SELAS_EUNSUPPORTED, "%s: 16-bit input needs blocksize 64, a 16-byte aligned tensor and a codebook "
                                         "with spread midpoints", what);
  const int64_t nblocks = n / blocksize;
  int64_t grid = cdiv(nblocks, kThreads / 64);
  if (grid > 65536) grid = 65536;
  nf4_encode_waves<<<dim3(static_cast<uint32_t>(grid)), dim3(kThreads), 0, stream>>>(
      static_cast<const float *>(w), nblocks, static_cast<int>(blocksize), mids, packed, absmax);
  return check_launch(what);
}
}  // namespace

extern "C" int selas_nf4_encode(const float *w, int64_t n, int64_t blocksize, const float code[16], uint8_t *packed,
                                float *absmax, void *stream) {
  return encode_any("nf4_encode", w, SELAS_F32, n, blocksize, code, packed, absmax, static_cast<hipStream_t>(stream));
}

extern "C" int selas_nf4_encode_typed(const void *w, int w_dtype, int64_t n, int64_t blocksize, const float code[16],
                                      uint8_t *packed, float *absmax, void *stream) {
  return encode_any("nf4_encode_typed", w, w_dtype, n, blocksize, code, packed, absmax,
                    static_cast<hipStream_t>(stream));
}
