// Indexer input producer: RoPE, Hadamard rotation and fp8-e4m3 per-row quantisation of the
// lightning indexer's query / key rows in one pass (DeepSeek-V3.2 Indexer.forward and
// DeepSeek-V4 Indexer.forward up to the index-score einsum).
//
// Per row x of D = 128 bf16 values (one query head or one key):
//   1. RoPE on the rope_dim features starting at rope_start, in fp32, rounded to bf16:
//      pairs (a, b) -> (a c - b s, a s + b c) with (c, s) = cs[pos][i] for pair i; the pairs
//      are (rope_start + 2i, rope_start + 2i + 1) when interleaved and
//      (rope_start + i, rope_start + i + rope_dim/2) otherwise (the V3.2 indexer's blocked
//      layout);
//   2. y = bf16(bf16(H x) * D^-0.5) with H the Sylvester Hadamard matrix (natural order,
//      H[i][j] = (-1)^popcount(i & j)), summed in fp32 by a radix-2 butterfly;
//   3. optionally fp8: scale = max(amax |y| / 448, 1e-12), q = e4m3fn(y / scale) rounded to
//      nearest even (the rule of dsa_quantize_fp8_rows).
// The bf16 rounding points are the reference's: RoPE output cast to the model dtype, the
// bf16 linear, then the bf16 scale multiply.
//
// A 16-lane group per row (four rows per wave and step), lane l holding features
// 8l .. 8l+7 (16-byte loads and stores coalesced along the row).  Every cross-lane step --
// the butterfly's strides 8 .. 64, the V3.2 rope partner four lanes away and the amax --
// is a DPP lane exchange inside the 16-lane row.
#include "dsa_common.h"

namespace dsa {
namespace {

constexpr int kD = 128;
constexpr int kThreads = 256;

// fp32 pair -> bf16 pair and back (one conversion instruction for both)
__device__ __forceinline__ uint32_t round2(float& a, float& b) {
  const uint32_t w = pack_bf16x2(a, b);
  a = bf16_lo(w);
  b = bf16_hi(w);
  return w;
}

// Each 16-lane group takes kRows rows a grid apart and issues all their loads (the row, its
// position, then its cos / sin entries) before the first is used.  What bounds it is the
// vector work per element as much as HBM, hence the paired conversions, the row quotient
// (dsa_common.h) instead of a divide, and 32-bit row arithmetic (idx_t) up to 2^31 rows.
// 8192 tokens x 64 heads, bf16 and fp8 out: 109.9 us (3.1 TB/s) before, 85.0 us
// (4.0 TB/s) after; one row or four per group 2 % and 4 % slower.
constexpr int kRows = 2;
enum class Rope { kNone, kInterleaved, kBlocked };

template <Rope kRope, typename idx_t>
__global__ void __launch_bounds__(kThreads)
indexer_prep_kernel(const uint16_t* __restrict__ x, uint16_t* __restrict__ y, uint8_t* __restrict__ q8,
                    float* __restrict__ scale, idx_t vecs, idx_t heads, idx_t seq_len, const float* __restrict__ cs,
                    int64_t n_pos, const int32_t* __restrict__ positions, int64_t pos_offset, int rope_dim,
                    int rope_start, int hadamard) {
  const idx_t g0 = ((idx_t)blockIdx.x * kThreads + threadIdx.x) >> 4;
  const idx_t ng = ((idx_t)gridDim.x * kThreads) >> 4;
  const int l = threadIdx.x & 15;
  const int f0 = 8 * l;
  const int lf = f0 - rope_start;  // local feature of the lane's first
  const bool lane_rope = kRope != Rope::kNone && lf >= 0 && lf < rope_dim;
  u32x4 w[kRows];
  float4 c4[kRows][kRope == Rope::kBlocked ? 4 : 2];
  bool in_rope[kRows];
#pragma unroll
  for (int i = 0; i < kRows; ++i) {
    const idx_t v = min(g0 + i * ng, vecs - 1);  // (idle groups redo the last row)
    w[i] = reinterpret_cast<const u32x4*>(x + (int64_t)v * kD)[l];
  }
  if constexpr (kRope != Rope::kNone) {
    int64_t pos[kRows];
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
      const idx_t row = min(g0 + i * ng, vecs - 1) / heads;
      pos[i] = positions ? (int64_t)positions[row] : pos_offset + (int64_t)(row % seq_len);
    }
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
      const bool pos_ok = pos[i] >= 0 && pos[i] < n_pos;  // rows outside the table keep their features
      in_rope[i] = pos_ok && lane_rope;
      const float* cp = cs + (pos_ok ? pos[i] : 0) * rope_dim;
      // interleaved: the (cos, sin) of angles lf/2 .. +3; blocked: of angles lf % 32 .. +7
      const int a0 = !lane_rope ? 0 : kRope == Rope::kInterleaved ? lf : 2 * (lf & 31);
#pragma unroll
      for (int k = 0; k < (kRope == Rope::kBlocked ? 4 : 2); ++k)
        c4[i][k] = *reinterpret_cast<const float4*>(cp + a0 + 4 * k);
    }
  }
#pragma unroll
  for (int i = 0; i < kRows; ++i) {
    const idx_t v = g0 + i * ng;
    const bool active = v < vecs;
    float e[8];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      e[2 * k] = bf16_lo(w[i][k]);
      e[2 * k + 1] = bf16_hi(w[i][k]);
    }
    // ---- 1. RoPE (fp32, rounded to bf16) ----
    if constexpr (kRope == Rope::kInterleaved) {
      // pairs (lf + 2k, lf + 2k + 1) inside the lane, angles lf/2 + k
      const float cc[4] = {c4[i][0].x, c4[i][0].z, c4[i][1].x, c4[i][1].z};
      const float ss[4] = {c4[i][0].y, c4[i][0].w, c4[i][1].y, c4[i][1].w};
      if (in_rope[i]) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float a = e[2 * k], b = e[2 * k + 1];
          e[2 * k] = a * cc[k] - b * ss[k];
          e[2 * k + 1] = a * ss[k] + b * cc[k];
          round2(e[2 * k], e[2 * k + 1]);
        }
      }
    } else if constexpr (kRope == Rope::kBlocked) {
      // pairs (k, k + 32) of a 64-feature block: the partner lane is four lanes away
      float p[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) p[k] = lane_xor<4>(e[k]);
      if (in_rope[i]) {
        const bool lower = lf < 32;
#pragma unroll
        for (int k = 0; k < 8; k += 2) {
          const float4 c = c4[i][k >> 1];
          e[k] = lower ? e[k] * c.x - p[k] * c.y : p[k] * c.y + e[k] * c.x;
          e[k + 1] = lower ? e[k + 1] * c.z - p[k + 1] * c.w : p[k + 1] * c.w + e[k + 1] * c.z;
          round2(e[k], e[k + 1]);
        }
      }
    }
    // ---- 2. Hadamard: y = bf16(bf16(H x) * D^-0.5) ----
    u32x4 yw;
    if (hadamard) {
      // feature strides 1, 2, 4 inside the lane
#pragma unroll
      for (int h = 1; h < 8; h <<= 1)
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (!(k & h)) {
            const float a = e[k], b = e[k + h];
            e[k] = a + b;
            e[k + h] = a - b;
          }
      // strides 8 .. 64 across the lanes of the row: lane bit k <-> feature stride 8 * 2^k
      static_for<4>([&](auto kc) {
        constexpr int m = 1 << decltype(kc)::value;
        const float sg = (l & m) ? -1.f : 1.f;  // upper lanes: partner - own
#pragma unroll
        for (int k = 0; k < 8; ++k) e[k] = fmaf(sg, e[k], lane_xor<m>(e[k]));
      });
      const float sc = 0.08838834764831845f;  // 128^-0.5 rounded to fp32
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        round2(e[2 * k], e[2 * k + 1]);
        e[2 * k] *= sc;
        e[2 * k + 1] *= sc;
        yw[k] = round2(e[2 * k], e[2 * k + 1]);
      }
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) yw[k] = pack_bf16x2(e[2 * k], e[2 * k + 1]);
    }
    if (y && active) reinterpret_cast<u32x4*>(y + (int64_t)v * kD)[l] = yw;

    // ---- 3. fp8-e4m3 with a per-row scale ----
    if (q8) {
      float amax = 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float a = fabsf(e[k]);
        amax = (a > amax || a != a) ? a : amax;  // a NaN makes the row's amax NaN
      }
      static_for<4>([&](auto kc) {
        constexpr int m = 1 << decltype(kc)::value;
        const float o = lane_xor<m>(amax);
        amax = (o > amax || o != o) ? o : amax;
      });
      float s = amax / 448.0f;
      s = s < 1e-12f ? 1e-12f : s;  // (keeps NaN)
      if (active) {
        typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
        uint32_t b[2];
        e4m3_row8(e, s, b);
        reinterpret_cast<u32x2*>(q8 + (int64_t)v * kD)[l] = (u32x2){b[0], b[1]};
        if (l == 0 && scale) scale[v] = s;
      }
    }
  }
}

template <typename idx_t>
void launch_prep(Rope rope, const uint16_t* x, uint16_t* y, uint8_t* q8, float* scale, int64_t vecs, int64_t heads,
                 int64_t seq_len, const float* cs, int64_t n_pos, const int32_t* positions, int64_t pos_offset,
                 int rope_dim, int rope_start, int hadamard, unsigned grid, hipStream_t st) {
  auto* kern = rope == Rope::kNone          ? indexer_prep_kernel<Rope::kNone, idx_t>
               : rope == Rope::kInterleaved ? indexer_prep_kernel<Rope::kInterleaved, idx_t>
                                            : indexer_prep_kernel<Rope::kBlocked, idx_t>;
  kern<<<grid, kThreads, 0, st>>>(x, y, q8, scale, (idx_t)vecs, (idx_t)heads, (idx_t)seq_len, cs, n_pos, positions,
                                  pos_offset, rope_dim, rope_start, hadamard);
}

}  // namespace
}  // namespace dsa

extern "C" int dsa_indexer_prep(const void* x, void* y, uint8_t* q8, float* scale, int64_t rows, int64_t heads,
                                int64_t d, int64_t seq_len, const float* rope_cs, int64_t n_pos,
                                const int32_t* positions, int64_t pos_offset, int64_t rope_dim, int64_t rope_start,
                                int interleaved, int hadamard, void* stream) {
  using namespace dsa;
  if (!x) return set_error(DSA_ERR_INVALID_ARG, "dsa_indexer_prep: null input");
  if (!y && !q8) return set_error(DSA_ERR_INVALID_ARG, "dsa_indexer_prep: no output requested");
  if (q8 && !scale) return set_error(DSA_ERR_INVALID_ARG, "dsa_indexer_prep: fp8 output needs the scale output");
  if (rows < 0 || heads <= 0 || seq_len <= 0) return set_error(DSA_ERR_INVALID_ARG, "dsa_indexer_prep: bad sizes");
  if (d != kD) return set_error(DSA_ERR_UNSUPPORTED, "dsa_indexer_prep: D=%lld (the producer takes D = 128)",
                                (long long)d);
  if (rope_dim < 0 || rope_start < 0 || rope_start + rope_dim > kD ||
      (rope_dim > 0 && (interleaved ? (rope_dim % 8 || rope_start % 8) : (rope_dim != 64 || rope_start % 64))))
    return set_error(DSA_ERR_UNSUPPORTED, "dsa_indexer_prep: rope features [%lld, %lld) (interleaved: multiples of "
                     "8; blocked: 64 features starting at 0 or 64)", (long long)rope_start,
                     (long long)(rope_start + rope_dim));
  if (rope_dim > 0 && (!rope_cs || n_pos <= 0))
    return set_error(DSA_ERR_INVALID_ARG, "dsa_indexer_prep: RoPE needs the cos/sin table");
  const int64_t vecs = rows * heads;
  if (vecs == 0) return DSA_OK;
  const int64_t grid = ((vecs + kRows - 1) / kRows * 16 + kThreads - 1) / kThreads;
  if (grid > INT32_MAX) return set_error(DSA_ERR_INVALID_ARG, "dsa_indexer_prep: too many rows");
  const TimedLaunch tl("indexer_prep_kernel", (hipStream_t)stream);
  const Rope rope = rope_dim == 0 ? Rope::kNone : interleaved ? Rope::kInterleaved : Rope::kBlocked;
  // 32-bit rows where the thread index (16 per row) and the sequence length fit 31 bits
  const bool small = grid * kThreads * (kRows + 1) <= INT32_MAX && seq_len <= INT32_MAX && heads <= INT32_MAX;
  auto* launch = small ? launch_prep<uint32_t> : launch_prep<int64_t>;
  launch(rope, (const uint16_t*)x, (uint16_t*)y, q8, scale, vecs, heads, seq_len, rope_cs, n_pos, positions, pos_offset,
         (int)rope_dim, (int)rope_start, hadamard ? 1 : 0, (unsigned)grid, (hipStream_t)stream);
  return check_launch("dsa_indexer_prep");
}
