// Fused attention forward of the FLUX blocks (head dim 128, no mask) for gfx950:
// softmax(q k^T / sqrt(128)) v for every (batch, head), written straight into the
// [B, L, H * 128] layout the projection linear reads.
//
// One workgroup = NWV waves (8 or 4, see the launch) = 32 * NWV queries of
// one (batch, head); wave w owns queries 32w .. 32w+31. The keys stream through
// LDS in tiles of 64 (K rows and the matching V rows, double-buffered,
// loaded by buffer->LDS DMA, shared by all the workgroup's waves). Per tile:
//   * S^T = K Q^T on 32x32x16 MFMAs (16 per wave): K from LDS is the A operand,
//     Q (held in registers for the whole loop) the B operand, so lane l holds 32
//     scores of query l % 32 (lanes l and l^32 together hold its 64 keys);
//   * online softmax in the exp2 domain: the running maximum is raised only when
//     a tile's maximum exceeds it by more than 8 (2^8 headroom in fp32 and in the
//     bf16 probabilities), so the rescale of the output is rare;
//   * O^T += V^T P^T (16 MFMAs): the probabilities, rounded to bf16, are the B
//     operand straight from the score registers. For that, the K rows of a 32-key
//     block are loaded with bits 2 and 3 of the row index swapped: lane (q, h)
//     register r then holds key 16*(r/8) + 8*h + r%8, i.e. 8 consecutive keys per
//     MFMA k-step, as the V^T operand holds, transposed by the LDS reads
//     (ds_read_b64_tr_b16). With v^T laid out by a kernel of its own (16-byte
//     operand reads) the product itself ran 1 % faster at L = 4592, 241 us, but
//     that kernel takes 10 us there and half a call's time at L < 1024. Call
//     against call: 258.6 -> 247.5 us for B1 L 4592, 53.6 -> 40.2 for B1 L 1536.
// LDS tiles are XOR-swizzled in 16-byte chunks so that the fragment reads (16
// lanes per LDS cycle) hit 16 distinct 4-bank groups.
// Any sequence length: key and query rows past L read as zeros (buffer range),
// the last key tile's missing keys get score -inf, and query rows past L are not
// stored; value rows past L read as zeros too (v^T: padded to 64 tokens).
//
// LDS bandwidth bounds this kernel: every MFMA reads a 1 KiB A fragment from LDS
// (halving those reads ran 24 % faster). Two query blocks per wave would share
// each fragment, but need about 500 registers (one wave per SIMD); that version
// ran 25 % slower, because a lone wave cannot overlap its softmax with MFMAs.
// Eight waves per workgroup (one workgroup per CU) share each tile's DMA among
// 256 queries instead of 128, which cuts the LDS traffic per query by a tenth.
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "common.h"

namespace selas {
namespace {

constexpr int kDh = 128;                   // head dim
constexpr int kKT = 64;                    // keys per tile
constexpr int kTileBytes = kKT * kDh * 2;  // one K tile or V^T tile: 16 KiB
constexpr int kStageBytes = 2 * kTileBytes;

// MFMA row rho of a 32-key block reads K row swap23(rho): bits 2 and 3 exchanged.
__device__ __forceinline__ int swap23(int r) { return (r & ~12) | ((r & 4) << 1) | ((r & 8) >> 1); }

// max / sum of v over lanes l and l ^ 32 (the two halves of one query's keys), by
// v_permlane32_swap: its first result holds lanes 0-31's v in every lane, the
// second lanes 32-63's.
__device__ __forceinline__ float pair_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pair_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Two probabilities to packed bf16 (round to nearest even), one v_cvt_pk_bf16_f32.
// The caller materializes each probability once, where it is produced, and adds
// the same registers into the row sum; materializing again inside the pack made
// the compiler copy every value (32 moves per tile).
__device__ __forceinline__ uint32_t pack_probs(float lo, float hi) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const bf16x2 v = {static_cast<__bf16>(lo), static_cast<__bf16>(hi)};
  return __builtin_bit_cast(uint32_t, v);
}

// Of every image's `items` work items the last `tail` run as `parts` ranges of `per` key tiles each
// (selas_attention_split); a range leaves each wave's output, not yet divided, and its queries' maxima and sums in
// `partial`.
struct AttnSplit {
  int items, tail, parts, per;
  float *partial;
  // Work item of whole item w, of split item s.
  __host__ __device__ int whole_item(int w) const { return w + w / (items - tail) * tail; }
  __host__ __device__ int split_item(int s) const { return (s / tail + 1) * items - tail + s % tail; }
};
// Per wave and range: 64 x 64 outputs in the order of the registers (1 KiB per store instruction), then per lane the
// running maximum and the sum.
constexpr int kPartialFloats = 64 * 64 + 2 * 64;

// VT: the values come as v^T [B*H, 128, Lp] (selas_attention, for callers of the C ABI that have them so), else as v
// [B*H, L, 128].
template <int NWV, bool VT, bool SPLIT = false>
__global__ __launch_bounds__(64 * NWV, 2) void attn_fwd_kernel(const uint16_t *__restrict__ q,
                                                               const uint16_t *__restrict__ k,
                                                               const uint16_t *__restrict__ v,
                                                               uint16_t *__restrict__ out, int64_t ldo, int H, int L,
                                                               int qtiles, int per_xcd, int total, float c2,
                                                               AttnSplit sp) {
  constexpr int kQT = 32 * NWV;  // queries per workgroup
  constexpr int KJ = 16 / NWV;   // DMA instructions per wave and tile, for K and for V^T each
  // An array per stage: the compiler then knows that reads of one stage do not touch the DMA into the other. With one
  // array for both it waited for the next tile's loads before the first transposing read of a tile: 254 -> 250 us for
  // B1 L 4592 on inputs that come from HBM.
  __shared__ __attribute__((aligned(1024))) uint8_t smem0[kStageBytes], smem1[kStageBytes];
  // Work item t = (b % 8) * per_xcd + b / 8: each XCD takes a contiguous range,
  // so the query tiles of one head share that head's K and V^T in its L2.
  // Split: the whole items first, then the ranges, a range's parts on different XCDs.
  int t = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3), range = -1;
  if constexpr (SPLIT) {
    if (static_cast<int>(blockIdx.x) >= 8 * per_xcd) {
      range = blockIdx.x - 8 * per_xcd;
      t = sp.split_item(range / sp.parts);
    } else {
      if (t >= total) return;
      t = sp.whole_item(t);
    }
  } else {
    if (t >= total) return;
  }
  const int bh = t / qtiles, qt = t - bh * qtiles;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int h = lane >> 5, c = lane & 31;
  // q, k, v: [B*H, L, 128]; v^T: [B*H, 128, Lp] with Lp = L rounded up to the 64-key tile
  // (zero-filled). Query, key and value rows past L read as zeros through the buffer range.
  const int Lp = (L + kKT - 1) / kKT * kKT;
  const int64_t head = static_cast<int64_t>(bh) * L * kDh;  // elements
  const uint32_t head_bytes = static_cast<uint32_t>(L) * kDh * 2;
  const __amdgpu_buffer_rsrc_t qr = make_rsrc(q + head, head_bytes);
  const __amdgpu_buffer_rsrc_t kr = make_rsrc(k + head, head_bytes);
  const __amdgpu_buffer_rsrc_t vr = VT ? make_rsrc(v + static_cast<int64_t>(bh) * Lp * kDh,
                                                   static_cast<uint32_t>(Lp) * kDh * 2)
                                       : make_rsrc(v + head, head_bytes);

  // Q as the B operand of S^T = K Q^T: lane (query c of this wave, h) holds d = 16s + 8h .. +8.
  const int q_row = qt * kQT + 32 * wave + c;
  bf16x8 qf[8];
#pragma unroll
  for (int s = 0; s < 8; ++s)
    qf[s] = __builtin_bit_cast(bf16x8, load_b128(qr, static_cast<uint32_t>(q_row) * 256u + (16 * s + 8 * h) * 2, 0));

  // DMA per tile: 16 instructions of 1 KiB for K and V (4 rows of 256 B each; V^T:
  // 8 rows of 128 B) each, KJ + KJ per wave. Lane i of instruction J fills row
  // r = 4J + i/16, physical chunk i%16, with logical chunk (i%16) ^ (r%16) of K,
  // (i%16) ^ 4(r%4) of V; lane i of V^T instruction J fills row d = 8J + i/8,
  // physical chunk i%8, with logical chunk (i%8) ^ ((d/2)%8). The tile's first key
  // goes in the scalar offset.
  uint32_t k_voff[KJ], v_voff[KJ];
#pragma unroll
  for (int j = 0; j < KJ; ++j) {
    const int J = KJ * wave + j;
    const int r = 4 * J + (lane >> 4);
    k_voff[j] = static_cast<uint32_t>(r) * 256u + ((static_cast<uint32_t>(lane & 15) ^ (r & 15)) << 4);
    if constexpr (VT) {
      const int d = 8 * J + (lane >> 3);
      v_voff[j] = static_cast<uint32_t>(d) * static_cast<uint32_t>(Lp) * 2u +
                  ((static_cast<uint32_t>(lane & 7) ^ ((d >> 1) & 7)) << 4);
    } else {
      v_voff[j] = static_cast<uint32_t>(r) * 256u + ((static_cast<uint32_t>(lane & 15) ^ (4 * (lane >> 4))) << 4);
    }
  }
  auto issue = [&](int stage, int kt) {
    uint8_t *base = stage ? smem1 : smem0;
    const uint32_t key0 = static_cast<uint32_t>(kt) * kKT;
#pragma unroll
    for (int j = 0; j < KJ; ++j) load_lds16(kr, base + (KJ * wave + j) * 1024, k_voff[j], key0 * 256u);
#pragma unroll
    for (int j = 0; j < KJ; ++j) load_lds16(vr, base + kTileBytes + (KJ * wave + j) * 1024, v_voff[j], key0 * (VT ? 2u : 256u));
  };
  // A-operand fragments: K row of MFMA row c in key block kb, d-chunk 2s+h; V^T
  // row d = 32db + c, key chunk 4kb + 2t + h (keys 32kb + 16t + 8h .. +8).
  const int krow = swap23(c);
  auto kfrag = [&](int stage, int kb, int s) {
    const int r = 32 * kb + krow;
    const int cc = 2 * s + h;
    return *reinterpret_cast<const bf16x8 *>((stage ? smem1 : smem0) + r * 256 + ((cc ^ (r & 15)) << 4));
  };
  // V as the A operand of O^T += V^T P^T: lane (c, h) needs channel 32db + c of the keys 32kb + 16t + 8h .. +8.
  // ds_read_b64_tr_b16 transposes on the way: the 16 lanes of a group each address 4 channels of one of 4 keys (lane
  // i: key i/4, channels 4(i%4) .. +4), and lane i receives channel i of the 4 keys. Two reads make an operand. The
  // swizzle puts the 4 keys of a read in 4 different quarters of the 256-byte rows, so it is free of bank conflicts.
  uint32_t v_rd[4];
  {
    const int r = (lane >> 2) & 3, x = 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);
#pragma unroll
    for (int db = 0; db < 4; ++db) v_rd[db] = (8 * h + r) * 256 + ((db ^ r) << 6) + x * 16 + 8 * (lane & 1);
  }
  auto vfrag = [&](int stage, int db, int kb, int t2) {
    uint8_t *vs = (stage ? smem1 : smem0) + kTileBytes;
    if constexpr (VT) {
      const int d = 32 * db + c;
      const int cc = 4 * kb + 2 * t2 + h;
      return *reinterpret_cast<const bf16x8 *>(vs + d * 128 + ((cc ^ ((d >> 1) & 7)) << 4));
    } else {
      typedef short s16x4 __attribute__((ext_vector_type(4)));
      auto read = [&](int u) {
        return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(
            vs + v_rd[db] + kb * 8192 + t2 * 4096 + u * 1024));
      };
      const s16x4 lo = read(0), hi = read(1);
      return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
  };

  f32x16 o[4];
#pragma unroll
  for (int db = 0; db < 4; ++db) o[db] = f32x16{};
  // Split: a range may hold only scores of -inf, which then weigh nothing beside the other ranges.
  float m_run = SPLIT ? -3.402823466e38f : -__builtin_inff(), l_run = 0.0f;
  int kt = 0, ntiles = Lp / kKT;
  if constexpr (SPLIT) {
    if (range >= 0) {
      kt = range % sp.parts * sp.per;
      ntiles = min(ntiles, kt + sp.per);
    }
  }

  issue(0, kt);
  wait_vmcnt<0>();
  __syncthreads();

  // kMasked: the last tile of a sequence that is not a multiple of 64. The mask
  // is a separate instantiation so that full tiles carry no per-score selects
  // (a runtime test on every tile was turned into 93 selects and compares).
  auto tile = [&](int stage, int kt, auto masked) {
    constexpr bool kMasked = decltype(masked)::value;
    if (kt + 1 < ntiles) issue(stage ^ 1, kt + 1);
    // Scores: 16 MFMAs over (key block kb, d-chunk s) = (i / 8, i % 8). The K
    // fragments go through a ring of kKAhead registers, each read kKAhead MFMAs
    // before its use, so that no MFMA waits on a read issued just before it.
    constexpr int kKAhead = 4;
    f32x16 sc[2] = {f32x16{}, f32x16{}};
    bf16x8 kf[kKAhead];
#pragma unroll
    for (int i = 0; i < kKAhead; ++i) kf[i] = kfrag(stage, i / 8, i % 8);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      sc[i / 8] = mfma32(kf[i % kKAhead], qf[i % 8], sc[i / 8]);
      if (i + kKAhead < 16) kf[i % kKAhead] = kfrag(stage, (i + kKAhead) / 8, (i + kKAhead) % 8);
    }
    // The same order for the scheduler, which otherwise issues the first key
    // block's reads right before their MFMAs where registers are tight.
    __builtin_amdgcn_sched_group_barrier(0x100, kKAhead, 0);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      if (i + kKAhead < 16) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    if constexpr (kMasked) {
      // Keys past L do not exist. Register r of score block kb holds key
      // 32 kb + 16 (r/8) + 8 h + r % 8.
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (kt * kKT + 32 * kb + 16 * (r >> 3) + 8 * h + (r & 7) >= L) sc[kb][r] = -__builtin_inff();
    }
    float mx = sc[0][0];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sc[kb][r]);
    mx = pair_max(mx) * c2;
    const bool raise = mx > m_run + 8.0f;
    // Skipped for the whole wave unless some query's maximum moved (rare after the
    // first tiles); lanes whose maximum stays multiply by exactly 1.
    if (__builtin_amdgcn_ballot_w64(raise)) {
      const float alpha = raise ? __builtin_amdgcn_exp2f(m_run - mx) : 1.0f;
#pragma unroll
      for (int db = 0; db < 4; ++db) o[db] *= alpha;
      l_run *= alpha;
      m_run = raise ? mx : m_run;
    }
    // V^T fragments of the second product (db, kb, t2) = (i / 4, (i / 2) % 2, i % 2),
    // each read kVAhead MFMAs ahead.
    // Two reads a fragment from V: 6 ahead measured 0.3 % faster at L 4592, up to 1.5 % slower at other lengths.
    constexpr int kVAhead = VT ? 8 : 4;
    bf16x8 vf[kVAhead];
#pragma unroll
    for (int i = 0; i < kVAhead; ++i) vf[i] = vfrag(stage, i / 4, (i / 2) % 2, i % 2);
    float ls = 0.0f;
    bf16x8 pb[2][2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) {
        uint32_t w[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float p0 = materialize(__builtin_amdgcn_exp2f(__builtin_fmaf(sc[kb][8 * t2 + 2 * e], c2, -m_run)));
          const float p1 = materialize(__builtin_amdgcn_exp2f(__builtin_fmaf(sc[kb][8 * t2 + 2 * e + 1], c2, -m_run)));
          ls += p0 + p1;
          w[e] = pack_probs(p0, p1);
        }
        pb[kb][t2] = __builtin_bit_cast(bf16x8, make_uint4(w[0], w[1], w[2], w[3]));
      }
    l_run += ls;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      o[i / 4] = mfma32(vf[i % kVAhead], pb[(i / 2) % 2][i % 2], o[i / 4]);
      const int j = i + kVAhead;
      if (j < 16) vf[i % kVAhead] = vfrag(stage, j / 4, (j / 2) % 2, j % 2);
    }
    // The same order for the scheduler, which otherwise issues most of the transposing reads in fours right before
    // their MFMAs: 240.7 -> 235.4 us for B1 L 4592.
    if constexpr (!VT) {
      __builtin_amdgcn_sched_group_barrier(0x100, 2 * kVAhead, 0);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (i + kVAhead < 16) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
    }
    // The next tile has landed for this wave; the barrier then covers every wave
    // and orders this tile's LDS reads before the DMA that reuses its stage.
    wait_vmcnt<0>();
    __syncthreads();
  };
  const std::integral_constant<bool, false> full{};
  const std::integral_constant<bool, true> last{};
  const int kt0 = kt, nfull = SPLIT ? min(L / kKT, ntiles) : L / kKT;  // tiles whose 64 keys all exist
  for (; kt + 2 <= nfull; kt += 2) {
    tile(0, kt, full);
    tile(1, kt + 1, full);
  }
  if (kt < nfull) tile(0, kt++, full);
  if (kt < ntiles) {  // a partial last tile
    if ((kt - kt0) & 1) tile(1, kt, last);
    else tile(0, kt, last);
  }

  // out[(b*L + q) * ldo + hh*128 + d] = O^T[d][q] / l, d = 32db + 8g + 4h + e for register 4g + e.
  if constexpr (SPLIT) {
    if (range >= 0) {
      float *w = sp.partial + static_cast<int64_t>(range * NWV + wave) * kPartialFloats;
#pragma unroll
      for (int i = 0; i < 16; ++i)
        *reinterpret_cast<float4 *>(w + (i * 64 + lane) * 4) =
            make_float4(o[i >> 2][4 * (i & 3)], o[i >> 2][4 * (i & 3) + 1], o[i >> 2][4 * (i & 3) + 2],
                        o[i >> 2][4 * (i & 3) + 3]);
      *reinterpret_cast<float2 *>(w + 4096 + 2 * lane) = make_float2(m_run, pair_sum(l_run));
      return;
    }
  }
  const float inv = 1.0f / pair_sum(l_run);
  const int b = bh / H, hh = bh - b * H;
  if (q_row >= L) return;  // a last query tile past the sequence end
  uint16_t *orow = out + (static_cast<int64_t>(b) * L + q_row) * ldo + hh * kDh;
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d = 32 * db + 8 * g + 4 * h;
      *reinterpret_cast<uint2 *>(orow + d) = make_uint2(pack_bf16x2(o[db][4 * g] * inv, o[db][4 * g + 1] * inv),
                                                        pack_bf16x2(o[db][4 * g + 2] * inv, o[db][4 * g + 3] * inv));
    }
}

// The split items' outputs from their ranges, added in key order: a workgroup of one wave per 32 queries and 32
// channels, in the lane order of attn_fwd_kernel. Bounded by the reads of the partial outputs (L2, Infinity Cache).
__global__ __launch_bounds__(64) void attn_merge_kernel(uint16_t *__restrict__ out,
                                                        int64_t ldo, int H, int L, int qtiles, int nwv,
                                                        AttnSplit sp) {
  const int lane = threadIdx.x, db = blockIdx.x & 3, wave = (blockIdx.x >> 2) % nwv, item = (blockIdx.x >> 2) / nwv;
  const int t = sp.split_item(item), bh = t / qtiles, qt = t - bh * qtiles, parts = sp.parts;
  const int64_t step = static_cast<int64_t>(nwv) * kPartialFloats;  // from one range to the next
  const float *__restrict__ w = sp.partial + (static_cast<int64_t>(item) * parts * nwv + wave) * kPartialFloats;
  float m = -__builtin_inff();
  for (int p = 0; p < parts; ++p) m = fmaxf(m, w[p * step + 4096 + 2 * lane]);
  float l = 0.0f;
  float4 o[4] = {};
#pragma unroll 2
  for (int p = 0; p < parts; ++p) {
    const float2 ml = *reinterpret_cast<const float2 *>(w + p * step + 4096 + 2 * lane);
    const float a = __builtin_amdgcn_exp2f(ml.x - m);
    l += a * ml.y;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const float4 x = *reinterpret_cast<const float4 *>(w + p * step + ((4 * db + g) * 64 + lane) * 4);
      o[g].x += a * x.x;
      o[g].y += a * x.y;
      o[g].z += a * x.z;
      o[g].w += a * x.w;
    }
  }
  const int q_row = qt * 32 * nwv + 32 * wave + (lane & 31);
  if (q_row >= L) return;
  const float inv = 1.0f / l;
  const int b = bh / H, hh = bh - b * H;
  uint16_t *orow = out + (static_cast<int64_t>(b) * L + q_row) * ldo + hh * kDh + 32 * db + 4 * (lane >> 5);
#pragma unroll
  for (int g = 0; g < 4; ++g)
    *reinterpret_cast<uint2 *>(orow + 8 * g) =
        make_uint2(pack_bf16x2(o[g].x * inv, o[g].y * inv), pack_bf16x2(o[g].z * inv, o[g].w * inv));
}

// vt[bh][d][l] = v[bh][l][d] for 64 tokens x 128 channels per workgroup, through LDS;
// vt rows hold Lp = L rounded up to 64 tokens, the ones past L zero. The tile is
// [token][channel] with a 65-word row: the row writes (lane = token r % 4, channel
// chunk) fall in 64 distinct banks, and the transposed 2-byte reads (lane = channel d,
// token chunk) in 32 distinct words, two lanes per word.
__global__ __launch_bounds__(256) void transpose_heads_kernel(const uint16_t *__restrict__ v, uint16_t *__restrict__ vt,
                                                              int L, int Lp) {
  constexpr int kRow = kDh + 2;  // 260-byte rows
  __shared__ __attribute__((aligned(16))) uint16_t tile[kKT * kRow];
  const int l0 = blockIdx.x * kKT;
  const int64_t head = static_cast<int64_t>(blockIdx.y) * L * kDh;
  const int tid = threadIdx.x;
#pragma unroll
  for (int i = 0; i < 4; ++i) {  // token r, channels 8c .. 8c+7
    const int r = (tid >> 4) + 16 * i, ch = tid & 15;
    const uint4 x = l0 + r < L ? *reinterpret_cast<const uint4 *>(v + head + static_cast<int64_t>(l0 + r) * kDh + 8 * ch)
                               : make_uint4(0, 0, 0, 0);
    uint32_t *dst = reinterpret_cast<uint32_t *>(tile + r * kRow + 8 * ch);  // 4-byte aligned
    dst[0] = x.x;
    dst[1] = x.y;
    dst[2] = x.z;
    dst[3] = x.w;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {  // channel d, tokens 8c .. 8c+7
    const int d = (tid >> 3) + 32 * i, ch = tid & 7;
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      w[e] = static_cast<uint32_t>(tile[(8 * ch + 2 * e) * kRow + d]) |
             (static_cast<uint32_t>(tile[(8 * ch + 2 * e + 1) * kRow + d]) << 16);
    *reinterpret_cast<uint4 *>(vt + static_cast<int64_t>(blockIdx.y) * Lp * kDh + static_cast<int64_t>(d) * Lp + l0 +
                               8 * ch) = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

}  // namespace
}  // namespace selas

using namespace selas;

namespace {
int check_heads(const char *what, int64_t B, int64_t H, int64_t L, int64_t Dh, int dtype) {
  if (B < 0 || H < 0 || L < 0 || Dh <= 0)
    return set_error(SELAS_EINVAL, "%s: bad shape B=%lld H=%lld L=%lld Dh=%lld", what, (long long)B, (long long)H,
                     (long long)L, (long long)Dh);
  if (!valid_dtype(dtype)) return set_error(SELAS_EINVAL, "%s: bad dtype %d", what, dtype);
  if (dtype != SELAS_BF16 || Dh != kDh)
    return set_error(SELAS_EUNSUPPORTED, "%s: fused attention takes bf16 and head_dim 128 (got %s, %lld)", what,
                     dtype_name(dtype), (long long)Dh);
  if ((L + kKT) * Dh * 2 >= (1ll << 32) || B * H >= (1ll << 31) / 64)
    return set_error(SELAS_EUNSUPPORTED, "%s: a head above 4 GiB", what);
  return SELAS_OK;
}
}  // namespace

namespace {
// The GPU's CU count (256 on MI355X), asked of the runtime once per device.
int attn_cu_count() {
  static std::atomic<int> counts[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
    (void)hipGetLastError();
    dev = 0;
  }
  int v = counts[dev].load(std::memory_order_relaxed);
  if (v > 0) return v;
  if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) {
    (void)hipGetLastError();
    v = 256;
  }
  counts[dev].store(v, std::memory_order_relaxed);
  return v;
}

// How a call is cut up: the workgroup size, and a last round of few eight-wave items split over the keys.
struct AttnPlan {
  int nwv = 8;
  AttnSplit split{0, 0, 0, 0, nullptr};  // parts 0: not split
};

// Eight waves share each tile among more queries but run one workgroup per CU; of the four-wave workgroups two
// run on a CU, or one, faster, when there are no more than CUs left. Relative time per key tile of a round of each
// (us, fitted to B 1 and 4 at L = 768 to 4608 with 24 heads): 1.74, 1.9 and 1.3. Measured when fitted, four waves
// against eight, us: B1 L 4608 274 / 251, B1 L 1536 45.7 / 42.4, B2 L 2300 145 / 135, B4 L 1536 127 / 142, B1 L 768
// 18 / 25.
constexpr double kTile8 = 1.74, kTile4 = 1.9, kTile4Half = 1.3;

double rounds8(int64_t B, int64_t H, int64_t L) {
  return kTile8 * static_cast<double>(cdiv(B * H * cdiv(L, 256), static_cast<int64_t>(attn_cu_count())));
}
double rounds4(int64_t B, int64_t H, int64_t L) {
  const int64_t cu = attn_cu_count(), n4 = B * H * cdiv(L, 128), rest = n4 % (2 * cu);
  return kTile4 * static_cast<double>(n4 / (2 * cu)) + (rest == 0 ? 0.0 : rest <= cu ? kTile4Half : kTile4);
}

// The eight-wave items that an image has beyond full rounds of the CUs run as ranges of keys on the idle CUs. Whether
// and how is decided for one image, from H, L and the CU count: an image has the same bits in every batch. So the cut
// has to serve two to four images too, whose items fill rounds that one image leaves partly idle: at most an eighth of
// a round is cut up per full round, into at most half a round of ranges. Not where four-wave workgroups need less (L
// 2688: 92 us), and not for fewer than 40 key tiles (a range's prologue, its partial output and the merge take 8 us).
// Unsplit / split, us, batch 1 to 4, 24 heads: L 2700 125 / 104, 206 / 188, 308 / 271, 392 / 359; L 3072 138 / 119,
// 232 / 221, 343 / 334, 446 / 438 (six images 639 / 651, eight 829 / 873); L 5632 406 / 353, 764 / 682; L 6144
// 448 / 425, 834 / 802. Past the line: L 3328 (56 items over one round) in 4 ranges 152 / 137, 259 / 266, 381 / 397,
// 494 / 530, in 2 151 / 144, 257 / 254, 382 / 395; L 3584 (80) in 3 167 / 156, 299 / 301, 425 / 451; L 4096 (128)
// 196 / 194, 361 / 379; 32 heads, L 2100 (33 key tiles) 97 / 88 and, batch 4, 304 / 312.
AttnSplit plan_split(int64_t H, int64_t L) {
  AttnSplit split{0, 0, 0, 0, nullptr};
  const int64_t cu = attn_cu_count(), items = H * cdiv(L, 256), tail = items % cu, full = items / cu, tiles = cdiv(L, kKT);
  if (tail == 0 || 8 * tail > cu * full || 4 * tail > cu || tiles < 40) return split;
  const int64_t per = cdiv(tiles, std::min<int64_t>(8, cu / (2 * tail))), parts = cdiv(tiles, per);
  const double cut = kTile8 * (static_cast<double>(full) + 1.0 / static_cast<double>(parts));
  if (cut > 0.95 * std::min(rounds8(1, H, L), rounds4(1, H, L))) return split;
  return {static_cast<int>(items), static_cast<int>(tail), static_cast<int>(parts), static_cast<int>(per), nullptr};
}

AttnPlan plan_attention(int64_t B, int64_t H, int64_t L, bool may_split) {
  AttnPlan plan;
  if (may_split) plan.split = plan_split(H, L);
  if (plan.split.parts == 0 && rounds8(B, H, L) >= rounds4(B, H, L)) plan.nwv = 4;
  return plan;
}

int64_t split_bytes(const AttnPlan &plan, int64_t B) {
  return B * plan.split.tail * plan.split.parts * plan.nwv * kPartialFloats * static_cast<int64_t>(sizeof(float));
}

template <bool VT>
int attention_any(const char *what, const void *q, const void *k, const void *v, int64_t B, int64_t H, int64_t L,
                  int64_t Dh, void *out, int64_t ldo, int dtype, bool may_split, void *workspace,
                  int64_t workspace_bytes, void *stream) {
  if (int e = check_heads(what, B, H, L, Dh, dtype)) return e;
  if (B == 0 || H == 0 || L == 0) return ok();
  if (!q || !k || !v || !out) return set_error(SELAS_EINVAL, "%s: null pointer", what);
  if (ldo < H * Dh) return set_error(SELAS_EINVAL, "%s: out row stride %lld below H*Dh", what, (long long)ldo);
  if (!aligned(q, 16) || !aligned(k, 16) || !aligned(v, 16) || !aligned(out, 8) || ldo % 4)
    return set_error(SELAS_EUNSUPPORTED, "%s: q, k and the values must be 16-byte aligned, out rows 8-byte aligned", what);
  const float c2 = 1.4426950408889634f / sqrtf(static_cast<float>(Dh));  // log2(e) / sqrt(Dh)
  AttnPlan plan = plan_attention(B, H, L, may_split);
  const int qtiles = static_cast<int>(cdiv(L, 32 * plan.nwv));
  const int64_t total = B * H * qtiles;
  const hipStream_t st = static_cast<hipStream_t>(stream);
  auto launch = [&](auto kernel, int64_t whole, int64_t ranges) {
    const int per_xcd = static_cast<int>(cdiv(whole, 8));
    kernel<<<dim3(static_cast<uint32_t>(per_xcd * 8 + ranges)), dim3(64 * plan.nwv), 0, st>>>(
        static_cast<const uint16_t *>(q), static_cast<const uint16_t *>(k), static_cast<const uint16_t *>(v),
        static_cast<uint16_t *>(out), ldo, static_cast<int>(H), static_cast<int>(L), qtiles, per_xcd,
        static_cast<int>(whole), c2, plan.split);
  };
  if constexpr (!VT) {
    if (plan.split.parts) {
      const int64_t bytes = split_bytes(plan, B), tail = B * plan.split.tail;
      if (workspace_bytes < bytes || !workspace || !aligned(workspace, 16))
        return set_error(SELAS_EINVAL, "%s: needs a 16-byte aligned workspace of %lld bytes", what, (long long)bytes);
      plan.split.partial = static_cast<float *>(workspace);
      launch(attn_fwd_kernel<8, VT, true>, total - tail, tail * plan.split.parts);
      if (int e = check_launch(what)) return e;
      attn_merge_kernel<<<dim3(static_cast<uint32_t>(4 * plan.nwv * tail)), dim3(64), 0, st>>>(
          static_cast<uint16_t *>(out), ldo, static_cast<int>(H), static_cast<int>(L), qtiles, plan.nwv, plan.split);
      return check_launch(what);
    }
  }
  if (plan.nwv == 8) launch(attn_fwd_kernel<8, VT>, total, 0);
  else launch(attn_fwd_kernel<4, VT>, total, 0);
  return check_launch(what);
}
}  // namespace

extern "C" int selas_attention(const void *q, const void *k, const void *vt, int64_t B, int64_t H, int64_t L,
                               int64_t Dh, void *out, int64_t ldo, int dtype, void *stream) {
  return attention_any<true>("attention", q, k, vt, B, H, L, Dh, out, ldo, dtype, false, nullptr, 0, stream);
}

extern "C" int selas_attention_v(const void *q, const void *k, const void *v, int64_t B, int64_t H, int64_t L,
                                 int64_t Dh, void *out, int64_t ldo, int dtype, void *stream) {
  if (B >= 0 && H >= 0 && B * H > 65535)
    return set_error(SELAS_EUNSUPPORTED, "attention_v: more than 65535 heads");
  return attention_any<false>("attention_v", q, k, v, B, H, L, Dh, out, ldo, dtype, false, nullptr, 0, stream);
}

extern "C" int selas_attention_workspace_bytes(int64_t B, int64_t H, int64_t L, int64_t *bytes) {
  if (!bytes) return set_error(SELAS_EINVAL, "attention_workspace_bytes: null pointer");
  *bytes = 0;
  if (int e = check_heads("attention_workspace_bytes", B, H, L, kDh, SELAS_BF16)) return e;
  if (B && H && L) *bytes = split_bytes(plan_attention(B, H, L, true), B);
  return ok();
}

extern "C" int selas_attention_split(const void *q, const void *k, const void *v, int64_t B, int64_t H, int64_t L,
                                     int64_t Dh, void *out, int64_t ldo, int dtype, void *workspace,
                                     int64_t workspace_bytes, void *stream) {
  if (B >= 0 && H >= 0 && B * H > 65535)
    return set_error(SELAS_EUNSUPPORTED, "attention_split: more than 65535 heads");
  return attention_any<false>("attention_split", q, k, v, B, H, L, Dh, out, ldo, dtype, true, workspace, workspace_bytes,
                              stream);
}

extern "C" int selas_transpose_heads(const void *v, int64_t BH, int64_t L, int64_t Dh, void *vt, int dtype,
                                     void *stream) {
  if (int e = check_heads("transpose_heads", 1, BH, L, Dh, dtype)) return e;
  if (BH == 0 || L == 0) return ok();
  if (!v || !vt) return set_error(SELAS_EINVAL, "transpose_heads: null pointer");
  if (!aligned(v, 16) || !aligned(vt, 16))
    return set_error(SELAS_EUNSUPPORTED, "transpose_heads: v and v^T must be 16-byte aligned");
  if (BH > 65535) return set_error(SELAS_EUNSUPPORTED, "transpose_heads: more than 65535 heads");
  const int64_t Lp = cdiv(L, kKT) * kKT;
  transpose_heads_kernel<<<dim3(static_cast<uint32_t>(Lp / kKT), static_cast<uint32_t>(BH)), dim3(256), 0,
                           static_cast<hipStream_t>(stream)>>>(static_cast<const uint16_t *>(v),
                                                               static_cast<uint16_t *>(vt), static_cast<int>(L),
                                                               static_cast<int>(Lp));
  return check_launch("transpose_heads");
}
