// MLA weight absorption, the per-head products around the absorbed attention
// (DeepSeek-V3.2 PreAttention / PostAttention, models/deepseek_v32/model.py:520-535, :574-575):
//   C[t, h, 0:N] = A[t, h, 0:K] . W[h]          (W = Wt[h]^T, Wt [H, N, K] row-major)
//   C[t, h, N:N+E] = E[t, h, 0:E]               (optional append: q_pe behind the absorbed q_nope)
// for (K, N) = (128, 512) (q_nope . w_uk, and the backward of the output projection) or
// (512, 128) (attention output . w_uv, and the backward of the query projection).
//
// Workgroup = one head x (8 waves x T 32-token tiles).  The head's Wt (N x K bf16, 128 KB)
// is staged once in LDS with 16-byte chunk c of row n at c ^ (n & 15) (conflict-free b128
// reads by 16 rows).  Per 32-token tile the wave computes C^T[32 n x 32 tokens] = Wt[n-tile]
// . A^T on v_mfma_f32_32x32x16_bf16 (A operand = 8 consecutive k of an Wt row from LDS, B
// operand = 8 consecutive k of a token's A row from global memory), fp32 accumulation, bf16
// output: lane (token, half) holds n = 8j + 4 half + i; a lane exchange between the two
// half-waves turns them into 16-byte stores.  Each Wt operand read from LDS feeds the
// wave's T token tiles (LDS traffic per MFMA / T):
//   (K, N) = (128, 512), T = 2: the tiles' A rows stay in VGPRs (8 k-steps x 2 tiles), the
//          16 n-tiles run in pairs (a whole 128-byte output line per iteration);
//   (K, N) = (512, 128), T = 2: the 4 n-tiles x 2 token tiles accumulate together while the
//          32 k-steps stream the A rows from global memory three steps ahead.
// Each workgroup stages its weight once and then walks token chunks; the waves share no
// state after the staging barrier.
//
// kKRows: the weight is given as W [H, K, N], the parameter's own layout in both forward
// products, and staged as it is, 16-byte chunk c of row k at c ^ 4 (k & 3); the A operand (8
// consecutive k of column n) is then read transposed, two ds_read_b64_tr_b16 of four rows
// each, whose lanes take distinct banks.  It saves the caller a transposed copy of the weight
// (18 to 31 us each): both products, forward + backward, 4096 tokens, 128 heads 1087 -> 1027 us;
// 100 tokens, 128 heads 191 -> 147; 1000 tokens, 32 heads 198 -> 164.  The products and their
// order are the same, so are the results.
#include <algorithm>

#include "dsa_common.h"

namespace dsa {
namespace {

constexpr int kWaves = 8;
constexpr int kThreads = 64 * kWaves;
constexpr int64_t kTargetWgs = 512;
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

template <int K, int N>
__device__ __forceinline__ void stage_wt(u32x4* ws, const uint16_t* __restrict__ wt, int h, int tid) {
  constexpr int kChunks = K / 8, kPer = N * kChunks / kThreads;
  static_assert(N * kChunks % kThreads == 0, "whole chunks per thread");
  const u32x4* wsrc = reinterpret_cast<const u32x4*>(wt + (int64_t)h * N * K);
  u32x4 v[kPer];  // every load in flight before the first LDS write
#pragma unroll
  for (int j = 0; j < kPer; ++j) v[j] = wsrc[tid + j * kThreads];
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int i = tid + j * kThreads, n = i / kChunks, ch = i - n * kChunks;
    ws[n * kChunks + (ch ^ (n & 15))] = v[j];
  }
}

template <int K, int N>
__device__ __forceinline__ void stage_w_rows(u32x4* ws, const uint16_t* __restrict__ w, int h, int tid) {
  constexpr int kChunks = N / 8, kPer = K * kChunks / kThreads;
  const u32x4* wsrc = reinterpret_cast<const u32x4*>(w + (int64_t)h * N * K);
  u32x4 v[kPer];
#pragma unroll
  for (int j = 0; j < kPer; ++j) v[j] = wsrc[tid + j * kThreads];
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int i = tid + j * kThreads, k = i / kChunks, ch = i - k * kChunks;
    ws[k * kChunks + (ch ^ (4 * (k & 3)))] = v[j];
  }
}

// Lane terms of the transposed reads of columns 32 nt .. +31, k = 16 s + 8 half .. +7: lane group
// G = lane / 16 covers columns 16 (G & 1) .. +15 of k half G >> 1; source lane c16 supplies row
// 8 (G >> 1) + c16 / 4 (+ 4 second read), columns 4 (c16 % 4) .. +3
struct TrLane {
  uint32_t base;  // row and chunk bits that do not depend on nt or s, bytes
  int rx;         // row & 3, the swizzle of nt
};
template <int N>
__device__ __forceinline__ TrLane tr_lane(int lane) {
  const int c16 = lane & 15, G = lane >> 4;
  const int row = 8 * (G >> 1) + (c16 >> 2);
  return {(uint32_t)(row * N * 2 + 32 * (G & 1) + 16 * ((c16 & 3) >> 1) + 8 * (c16 & 1)), c16 >> 2};
}
// A operand of n-tile nt, k-step s: `at` = base + 64 (nt ^ rx)
template <int N>
__device__ __forceinline__ u32x4 read_tr(const lds_char* wl, uint32_t at, int s) {
  const lds_char* p = wl + at + s * (16 * N * 2);
  return lds_read_tr_pair(p, p + 4 * N * 2);
}

// store one 32x32 C^T tile: lane (token col, half) holds rows n = n0 + 8 j + 4 half + i.
// A v_permlane32_swap per j pair gives each lane 8 consecutive n: the lower half-wave
// n0 + 16 q .. + 7, the upper n0 + 16 q + 8 .. + 15, so every store is 16 bytes and a
// token's 32 bytes leave in one instruction.
__device__ __forceinline__ void store_tile(uint16_t* crow, int n0, int half, const f32x16& acc) {
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const uint32_t x0 = pack_bf16x2(acc[8 * q], acc[8 * q + 1]), x1 = pack_bf16x2(acc[8 * q + 2], acc[8 * q + 3]);
    const uint32_t y0 = pack_bf16x2(acc[8 * q + 4], acc[8 * q + 5]), y1 = pack_bf16x2(acc[8 * q + 6], acc[8 * q + 7]);
    // (vdst, src) -> lower lanes (own vdst, upper partner's vdst), upper lanes (lower partner's src, own src)
    const auto r0 = __builtin_amdgcn_permlane32_swap(x0, y0, false, false);
    const auto r1 = __builtin_amdgcn_permlane32_swap(x1, y1, false, false);
    const u32x4 v = {r0[0], r1[0], r0[1], r1[1]};
    *reinterpret_cast<u32x4*>(crow + n0 + 16 * q + 8 * half) = v;
  }
}

__device__ __forceinline__ void append_cols(uint16_t* crow, const uint16_t* erow, int N, int app_w, int half) {
  for (int e = 8 * half; e < app_w; e += 16)
    *reinterpret_cast<u32x4*>(crow + N + e) = *reinterpret_cast<const u32x4*>(erow + e);
}

// (K, N) = (128, 512): the A rows of T token tiles stay in VGPRs; the n-tiles run in pairs,
// so each 128-byte line of a token's output is written whole within one iteration
template <bool kKRows>
__global__ void __launch_bounds__(kThreads, 1)
mla_absorb_q_kernel(const uint16_t* __restrict__ a, int64_t lda, const uint16_t* __restrict__ wt,
                    uint16_t* __restrict__ c, int64_t ldc, const uint16_t* __restrict__ app, int64_t ld_app,
                    int app_w, int64_t tokens, int heads) {
  constexpr int K = 128, N = 512, T = 2, kChunks = K / 8, kSteps = K / 16;
  __shared__ u32x4 ws[N * kChunks];  // 128 KB
  const int h = blockIdx.y;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int col = lane & 31, half = lane >> 5;
  if constexpr (kKRows) stage_w_rows<K, N>(ws, wt, h, tid);
  else stage_wt<K, N>(ws, wt, h, tid);
  __syncthreads();  // the only barrier: the waves run the chunks independently afterwards
  const lds_char* wl = lds_bytes(&ws[0]);
  for (int64_t t0 = ((int64_t)blockIdx.x * kWaves + wave) * (32 * T); t0 < tokens;
       t0 += (int64_t)gridDim.x * kWaves * (32 * T)) {
    int64_t row[T];
    bool ok[T];
    u32x4 bk[T][kSteps];
#pragma unroll
    for (int u = 0; u < T; ++u) {
      const int64_t tok = t0 + 32 * u + col;
      ok[u] = tok < tokens;
      row[u] = (ok[u] ? tok : tokens - 1) * heads + h;
      const u32x4* arow = reinterpret_cast<const u32x4*>(a + row[u] * lda);
#pragma unroll
      for (int s = 0; s < kSteps; ++s) bk[u][s] = arow[2 * s + half];
    }
    // LDS address of chunk (2s + half) ^ (n & 15) of row n = 32 nt + col: lane term lo,
    // chunk (2s) ^ xm; kept opaque so that the compiler does not hoist every address
    uint32_t lo = 16u * (uint32_t)(col * kChunks);
    int xm = (col & 15) ^ half;
    TrLane tr = tr_lane<N>(lane);
    asm volatile("" : "+v"(lo), "+v"(xm), "+v"(tr.base), "+v"(tr.rx));
#pragma unroll 1
    for (int np = 0; np < N / 64; ++np) {
      f32x16 acc[2][T];
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int u = 0; u < T; ++u)
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[p][u][i] = 0.f;
#pragma unroll
      for (int s = 0; s < kSteps; ++s) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          u32x4 av;
          if constexpr (kKRows) av = read_tr<N>(wl, tr.base + 64u * (uint32_t)((2 * np + p) ^ tr.rx), s);
          else av = lds_read16(wl + lo + 16 * ((64 * np + 32 * p) * kChunks + ((2 * s) ^ xm)));
#pragma unroll
          for (int u = 0; u < T; ++u) acc[p][u] = mfma32x32x16(as_bf16x8(av), as_bf16x8(bk[u][s]), acc[p][u]);
        }
      }
#pragma unroll
      for (int u = 0; u < T; ++u) {
        uint16_t* crow = c + row[u] * ldc;
        if (ok[u]) {
          store_tile(crow, 64 * np, half, acc[0][u]);
          store_tile(crow, 64 * np + 32, half, acc[1][u]);
        }
      }
    }
    if (app)
#pragma unroll
      for (int u = 0; u < T; ++u)
        if (ok[u]) append_cols(c + row[u] * ldc, app + row[u] * ld_app, N, app_w, half);
  }
}

// (K, N) = (512, 128): all n-tiles accumulate together, the A rows stream over the k-steps
template <bool kKRows>
__global__ void __launch_bounds__(kThreads, 1)
mla_absorb_o_kernel(const uint16_t* __restrict__ a, int64_t lda, const uint16_t* __restrict__ wt,
                    uint16_t* __restrict__ c, int64_t ldc, const uint16_t* __restrict__ app, int64_t ld_app,
                    int app_w, int64_t tokens, int heads) {
  constexpr int K = 512, N = 128, T = 2, kChunks = K / 8, kSteps = K / 16, kNT = N / 32, kAhead = 3;
  __shared__ u32x4 ws[N * kChunks];  // 128 KB
  const int h = blockIdx.y;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int col = lane & 31, half = lane >> 5;
  if constexpr (kKRows) stage_w_rows<K, N>(ws, wt, h, tid);
  else stage_wt<K, N>(ws, wt, h, tid);
  __syncthreads();  // the only barrier: the waves run the chunks independently afterwards
  const lds_char* wl = lds_bytes(&ws[0]);
  for (int64_t t0 = ((int64_t)blockIdx.x * kWaves + wave) * (32 * T); t0 < tokens;
       t0 += (int64_t)gridDim.x * kWaves * (32 * T)) {
    int64_t row[T];
    bool ok[T];
    const u32x4* arow[T];
#pragma unroll
    for (int u = 0; u < T; ++u) {
      const int64_t tok = t0 + 32 * u + col;
      ok[u] = tok < tokens;
      row[u] = (ok[u] ? tok : tokens - 1) * heads + h;
      arow[u] = reinterpret_cast<const u32x4*>(a + row[u] * lda);
    }
    // B operands of k-steps s .. s + kAhead - 1 in a register ring
    u32x4 bk[kAhead][T];
#pragma unroll
    for (int s = 0; s < kAhead; ++s)
#pragma unroll
      for (int u = 0; u < T; ++u) bk[s][u] = arow[u][2 * s + half];
    // lane terms of the LDS addresses, opaque to the compiler so that it does not hoist the
    // 128 addresses of the k-loop out of the chunk loop (they would not fit in registers)
    uint32_t lo = 16u * (uint32_t)(col * kChunks);
    int xm = (col & 15) ^ half;
    TrLane tr = tr_lane<N>(lane);
    asm volatile("" : "+v"(lo), "+v"(xm), "+v"(tr.base), "+v"(tr.rx));
    f32x16 acc[kNT][T];
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt)
#pragma unroll
      for (int u = 0; u < T; ++u)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[nt][u][i] = 0.f;
    static_for<kSteps>([&](auto sc) {
      constexpr int s = decltype(sc)::value;
      constexpr int slot = s % kAhead;
      // chunk (2s + half) ^ (n & 15) of row n = 32 nt + col; (n & 15) = (col & 15)
      const int sw = (16 * (s >> 3)) + ((2 * (s & 7)) ^ xm);
#pragma unroll
      for (int nt = 0; nt < kNT; ++nt) {
        u32x4 av;
        if constexpr (kKRows) av = read_tr<N>(wl, tr.base + 64u * (uint32_t)(nt ^ tr.rx), s);
        else av = lds_read16(wl + lo + 16 * (32 * nt * kChunks + sw));
#pragma unroll
        for (int u = 0; u < T; ++u) acc[nt][u] = mfma32x32x16(as_bf16x8(av), as_bf16x8(bk[slot][u]), acc[nt][u]);
      }
      if constexpr (s + kAhead < kSteps) {
#pragma unroll
        for (int u = 0; u < T; ++u) bk[slot][u] = arow[u][2 * (s + kAhead) + half];
      }
    });
#pragma unroll
    for (int u = 0; u < T; ++u) {
      if (!ok[u]) continue;
      uint16_t* crow = c + row[u] * ldc;
#pragma unroll
      for (int nt = 0; nt < kNT; ++nt) store_tile(crow, 32 * nt, half, acc[nt][u]);
      if (app) append_cols(crow, app + row[u] * ld_app, N, app_w, half);
    }
  }
}

// Weight gradient of either product, per head h:
//   G[i, j] = sum_t A[t, h, i] . B[t, h, j]   (A rows 128 wide, B rows 512 wide, fp32 sums)
// written as [128, 512] (the query projection's w_uk) or transposed, [512, 128] (w_uv).
//
// Bound by one read of A and B (each row element is used in 512 or 128 products of its own
// token only).  Workgroup = head x 256 of B's columns, 8 waves of 64 x 64 outputs on
// v_mfma_f32_32x32x16_bf16; the tokens are the k dimension, so both operands are read
// transposed (ds_read_b64_tr_b16) out of 32-token tiles that are DMA'd into three LDS buffers
// two tiles ahead (16-byte chunk c of row r at c ^ 4 (r & 3): the four rows of a transposed read
// take distinct banks).  The two workgroups of a head run on one XCD (head = blockIdx.x), so
// A's second read comes from its L2.  Few heads: the tokens are split over workgroups too
// (about 256 in all), whose fp32 partial sums wgrad_sum_kernel adds in order.
// 4096 tokens, 128 heads: permuting copies, fp32 conversions and an fp32 library product
// 1.73 ms -> 0.128 ms (w_uk; 5.2 TB/s of operand bytes) and 0.166 ms (w_uv, transposed stores).
constexpr int kGTok = 32;             // tokens per tile
constexpr int kGThreads = 512;
constexpr int kNar = 128, kWide = 512, kGCols = 256;
constexpr int64_t kGElems = (int64_t)kNar * kWide;

template <bool kWideRows>
__global__ void __launch_bounds__(kGThreads, 2)
mla_absorb_wgrad_kernel(const uint16_t* __restrict__ a, int64_t lda, const uint16_t* __restrict__ b, int64_t ldb,
                        void* __restrict__ out, int out_bf16, float* __restrict__ part, int64_t tokens, int heads,
                        int64_t per_split) {
  __shared__ u32x4 ta[3][kGTok * kNar / 8];
  __shared__ u32x4 tb[3][kGTok * kGCols / 8];
  const int h = blockIdx.x, cpart = blockIdx.y, sp = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;  // 64 columns of A, of B
  const int64_t t_beg = sp * per_split, t_end = min(tokens, t_beg + per_split);
  const int n_tiles = t_end > t_beg ? (int)((t_end - t_beg + kGTok - 1) / kGTok) : 0;
  const uint32_t sa = (uint32_t)(heads * lda * 2), sb = (uint32_t)(heads * ldb * 2);  // bytes per token
  auto issue = [&](int tl, int buf) {  // three instructions per wave: 4 rows of A, 2 x 2 rows of B
    const int64_t t0 = t_beg + (int64_t)tl * kGTok;
    const int last = (int)min<int64_t>(kGTok - 1, t_end - 1 - t0);
    const uint16_t* ab = a + (t0 * heads + h) * lda;
    const uint16_t* bb = b + (t0 * heads + h) * ldb + cpart * kGCols;
    {
      const int r = 4 * wave + (lane >> 4), c = (lane & 15) ^ (4 * (r & 3));
      dma16_to_lds(ab, (uint32_t)min(r, last) * sa + 16u * c, (uint32_t)(uintptr_t)&ta[buf][64 * wave]);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int J = wave + 8 * i, r = 2 * J + (lane >> 5), c = (lane & 31) ^ (4 * (r & 3));
      dma16_to_lds(bb, (uint32_t)min(r, last) * sb + 16u * c, (uint32_t)(uintptr_t)&tb[buf][64 * J]);
    }
  };
  // transposed operand reads (the lane pattern of the attention forward's V reads): lane group
  // G = lane / 16 covers columns 16 (G & 1) .. +15 and token half G >> 1; source lane c
  // supplies token 8x + 4 (G >> 1) + c / 4 and columns 4 (c % 4) .. +3
  const int c16 = lane & 15, G = lane >> 4, n = lane & 31, half = lane >> 5;
  uint32_t oa[2][2], ob[2][2];  // [32-column tile][x], bytes
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      const int r = 8 * x + 4 * half + (c16 >> 2);
      const int ca = 8 * wm + 4 * y + 2 * (G & 1) + ((c16 & 3) >> 1), cb = 8 * wn + 4 * y + 2 * (G & 1) + ((c16 & 3) >> 1);
      oa[y][x] = r * (kNar * 2) + 16 * (ca ^ (4 * (r & 3))) + 8 * (c16 & 1);
      ob[y][x] = r * (kGCols * 2) + 16 * (cb ^ (4 * (r & 3))) + 8 * (c16 & 1);
    }
  f32x16 acc[2][2];  // [A tile][B tile]
#pragma unroll
  for (int y = 0; y < 2; ++y)
#pragma unroll
    for (int z = 0; z < 2; ++z) acc[y][z] = (f32x16){0.f};
  if (n_tiles > 0) issue(0, 0);
  if (n_tiles > 1) issue(1, 1);
  int buf = 0;
  for (int tl = 0; tl < n_tiles; ++tl) {
    if (tl + 1 < n_tiles) {
      asm volatile("s_waitcnt vmcnt(3)" ::: "memory");  // (the next tile's three may be in flight)
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __syncthreads();  // every wave's part landed; the buffer of the tile before is free
    if (tl + 2 < n_tiles) issue(tl + 2, buf == 0 ? 2 : buf - 1);
    const int valid = (int)min<int64_t>(kGTok, t_end - t_beg - (int64_t)tl * kGTok);
    if (valid < kGTok) {  // (workgroup-uniform, the last tile) rows past the last token add nothing
      for (int i = tid; i < (kGTok - valid) * (kNar / 8); i += kGThreads) ta[buf][valid * (kNar / 8) + i] = (u32x4){0u, 0u, 0u, 0u};
      for (int i = tid; i < (kGTok - valid) * (kGCols / 8); i += kGThreads) tb[buf][valid * (kGCols / 8) + i] = (u32x4){0u, 0u, 0u, 0u};
      __syncthreads();
    }
    const lds_char* pa = lds_bytes(&ta[buf][0]);
    const lds_char* pb = lds_bytes(&tb[buf][0]);
#pragma unroll
    for (int ks = 0; ks < kGTok / 16; ++ks) {
      u32x4 va[2], vb[2];
#pragma unroll
      for (int y = 0; y < 2; ++y) {
        va[y] = lds_read_tr_pair(pa + oa[y][0] + ks * 16 * kNar * 2, pa + oa[y][1] + ks * 16 * kNar * 2);
        vb[y] = lds_read_tr_pair(pb + ob[y][0] + ks * 16 * kGCols * 2, pb + ob[y][1] + ks * 16 * kGCols * 2);
      }
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int z = 0; z < 2; ++z)
          acc[y][z] = kWideRows ? mfma32x32x16(as_bf16x8(vb[z]), as_bf16x8(va[y]), acc[y][z])
                                : mfma32x32x16(as_bf16x8(va[y]), as_bf16x8(vb[z]), acc[y][z]);
    }
    buf = buf == 2 ? 0 : buf + 1;
  }
  // lane holds rows 8j + 4 half + i of the first operand's tile, column n of the second's
  float* po = part ? part + ((int64_t)sp * heads + h) * kGElems : nullptr;
#pragma unroll
  for (int y = 0; y < 2; ++y)
#pragma unroll
    for (int z = 0; z < 2; ++z)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int r = 8 * (v >> 2) + 4 * half + (v & 3);
        const int ia = 64 * wm + 32 * y, ib = cpart * kGCols + 64 * wn + 32 * z;
        const int64_t e = kWideRows ? (int64_t)(ib + r) * kNar + ia + n : (int64_t)(ia + r) * kWide + ib + n;
        if (po) po[e] = acc[y][z][v];
        else if (out_bf16) reinterpret_cast<uint16_t*>(out)[h * kGElems + e] = f_to_bf16(acc[y][z][v]);
        else reinterpret_cast<float*>(out)[h * kGElems + e] = acc[y][z][v];
      }
}

// out = sum of the token splits' partial sums, in order; four elements per thread
__global__ void __launch_bounds__(256)
wgrad_sum_kernel(const float* __restrict__ part, void* __restrict__ out, int out_bf16, int64_t n4, int splits) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  f32x4 s = reinterpret_cast<const f32x4*>(part)[i];
  for (int k = 1; k < splits; ++k) s += reinterpret_cast<const f32x4*>(part)[k * n4 + i];
  if (out_bf16) reinterpret_cast<uint2*>(out)[i] = make_uint2(pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3]));
  else reinterpret_cast<f32x4*>(out)[i] = s;
}

// token splits: about 256 workgroups, 256 tokens or more each (a split costs a write and a
// read of the fp32 gradient)
int wgrad_splits(int64_t tokens, int64_t heads) {
  const int64_t wgs = heads * (kWide / kGCols);
  return (int)std::max<int64_t>(1, std::min<int64_t>(256 / wgs, tokens / 256));
}

}  // namespace
}  // namespace dsa

extern "C" int64_t dsa_mla_absorb_wgrad_workspace_size(int64_t tokens, int64_t heads) {
  if (tokens <= 0 || heads <= 0) return 0;
  const int s = dsa::wgrad_splits(tokens, heads);
  return s > 1 ? s * heads * dsa::kGElems * 4 : 0;
}

extern "C" int dsa_mla_absorb_wgrad(const void* a, int64_t lda, const void* b, int64_t ldb, void* out, int out_dtype,
                                    int wide_rows, int64_t tokens, int64_t heads, void* workspace,
                                    int64_t workspace_bytes, void* stream) {
  using namespace dsa;
  const char* what = "dsa_mla_absorb_wgrad";
  if (!a || !b || !out) return set_error(DSA_ERR_INVALID_ARG, "%s: null pointer", what);
  if (tokens < 0 || heads <= 0 || heads > 65535) return set_error(DSA_ERR_INVALID_ARG, "%s: bad sizes", what);
  if (out_dtype != DSA_BF16 && out_dtype != DSA_F32)
    return set_error(DSA_ERR_UNSUPPORTED, "%s: out dtype %d", what, out_dtype);
  if (lda < kNar || ldb < kWide || lda % 8 || ldb % 8)
    return set_error(DSA_ERR_INVALID_ARG, "%s: leading dimensions (lda %lld, ldb %lld; multiples of 8 elements)", what,
                     (long long)lda, (long long)ldb);
  if (heads * std::max(lda, ldb) * 2 * kGTok > (int64_t)UINT32_MAX)
    return set_error(DSA_ERR_UNSUPPORTED, "%s: a tile of %d tokens exceeds 4 GiB", what, kGTok);
  if (((uintptr_t)a | (uintptr_t)b | (uintptr_t)out) % 16)
    return set_error(DSA_ERR_INVALID_ARG, "%s: operands must be 16-byte aligned", what);
  int splits = wgrad_splits(tokens, heads);
  if (splits > 1 && (!workspace || workspace_bytes < splits * heads * kGElems * 4 || (uintptr_t)workspace % 16)) splits = 1;
  int64_t per = (tokens + splits - 1) / splits;
  per = std::max<int64_t>(kGTok, (per + kGTok - 1) / kGTok * kGTok);
  hipStream_t st = (hipStream_t)stream;
  float* part = splits > 1 ? (float*)workspace : nullptr;
  {
    const TimedLaunch tl("mla_absorb_wgrad_kernel", st);
    auto* kern = wide_rows ? mla_absorb_wgrad_kernel<true> : mla_absorb_wgrad_kernel<false>;
    kern<<<dim3((unsigned)heads, kWide / kGCols, (unsigned)splits), kGThreads, 0, st>>>(
        (const uint16_t*)a, lda, (const uint16_t*)b, ldb, out, out_dtype == DSA_BF16, part, tokens, (int)heads, per);
  }
  if (int rc = check_launch(what)) return rc;
  if (splits > 1) {
    const int64_t n4 = heads * kGElems / 4;
    const TimedLaunch tl("wgrad_sum_kernel", st);
    wgrad_sum_kernel<<<ceil_div(n4, 256), 256, 0, st>>>(part, out, out_dtype == DSA_BF16, n4, splits);
    return check_launch(what);
  }
  return DSA_OK;
}

namespace dsa {
static int absorb_impl(const void* a, int64_t lda, const void* wt, bool k_rows, void* c, int64_t ldc,
                       const void* append, int64_t ld_append, int64_t append_width, int64_t tokens, int64_t heads,
                       int64_t k, int64_t n, void* stream) {
  if (!a || !wt || !c) return set_error(DSA_ERR_INVALID_ARG, "dsa_mla_absorb: null pointer");
  if (tokens < 0 || heads <= 0 || heads > 65535) return set_error(DSA_ERR_INVALID_ARG, "dsa_mla_absorb: bad sizes");
  const bool q_shape = k == 128 && n == 512, o_shape = k == 512 && n == 128;
  if (!q_shape && !o_shape)
    return set_error(DSA_ERR_UNSUPPORTED, "dsa_mla_absorb: (K, N) = (%lld, %lld); (128, 512) or (512, 128)",
                     (long long)k, (long long)n);
  if (lda < k || ldc < n + (append ? append_width : 0) || lda % 8 || ldc % 8 ||
      (append && (append_width <= 0 || append_width % 8 || ld_append < append_width || ld_append % 8)))
    return set_error(DSA_ERR_INVALID_ARG, "dsa_mla_absorb: leading dimensions (lda %lld, ldc %lld, append %lld/%lld; "
                     "multiples of 8 elements)", (long long)lda, (long long)ldc, (long long)append_width,
                     (long long)ld_append);
  if (((uintptr_t)a | (uintptr_t)wt | (uintptr_t)c) % 16 || (append && (uintptr_t)append % 16))
    return set_error(DSA_ERR_INVALID_ARG, "dsa_mla_absorb: operands must be 16-byte aligned");
  if (tokens == 0) return DSA_OK;
  // Each workgroup stages its head's weight once and then walks token chunks of
  // per_wg tokens gx apart: about kTargetWgs workgroups in all (every CU holds one).
  const int64_t per_wg = (int64_t)kWaves * 32 * 2;
  const int64_t chunks = (tokens + per_wg - 1) / per_wg;
  const int64_t gx = std::max<int64_t>(1, std::min<int64_t>(chunks, (kTargetWgs + heads - 1) / heads));
  dim3 grid((unsigned)gx, (unsigned)heads);
  hipStream_t st = (hipStream_t)stream;
  const uint16_t* ap = (const uint16_t*)a;
  const uint16_t* wp = (const uint16_t*)wt;
  const uint16_t* ep = (const uint16_t*)append;
  const TimedLaunch tl(q_shape ? "mla_absorb_q_kernel" : "mla_absorb_o_kernel", st);
  auto* kern = q_shape ? (k_rows ? mla_absorb_q_kernel<true> : mla_absorb_q_kernel<false>)
                       : (k_rows ? mla_absorb_o_kernel<true> : mla_absorb_o_kernel<false>);
  kern<<<grid, kThreads, 0, st>>>(ap, lda, wp, (uint16_t*)c, ldc, ep, ld_append, (int)append_width, tokens, (int)heads);
  return check_launch("dsa_mla_absorb");
}
}  // namespace dsa

extern "C" int dsa_mla_absorb(const void* a, int64_t lda, const void* wt, void* c, int64_t ldc, const void* append,
                              int64_t ld_append, int64_t append_width, int64_t tokens, int64_t heads, int64_t k,
                              int64_t n, void* stream) {
  return dsa::absorb_impl(a, lda, wt, false, c, ldc, append, ld_append, append_width, tokens, heads, k, n, stream);
}

extern "C" int dsa_mla_absorb_rows(const void* a, int64_t lda, const void* w, void* c, int64_t ldc, const void* append,
                                   int64_t ld_append, int64_t append_width, int64_t tokens, int64_t heads, int64_t k,
                                   int64_t n, void* stream) {
  return dsa::absorb_impl(a, lda, w, true, c, ldc, append, ld_append, append_width, tokens, heads, k, n, stream);
}
