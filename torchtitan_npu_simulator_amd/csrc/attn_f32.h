// fp32 gathered attention on the matrix units (attn_f32.hip).
#pragma once
#include "dsa_common.h"

namespace dsa {

// widths the tile kernels take, and operands they can read 16 bytes at a time
bool attn_f32_fits(int64_t d_qk, int64_t d_v, int64_t n_heads);
bool attn_f32_aligned(const void* a, const void* b, const void* c = nullptr, const void* d = nullptr);
int attn_f32_fwd(const float* q, const float* kv, const int32_t* indices, float* out, float* smax, float* ssum,
                 int64_t batch, int64_t s_q, int64_t s_kv, int64_t n_heads, int64_t d_qk, int64_t d_v, int64_t topk,
                 float scale, int64_t q_offset, const float* sinks, hipStream_t st);
int attn_f32_bwd(const float* q, const float* kv, const int32_t* indices, const float* out, const float* dout,
                 const float* smax, const float* ssum, float* dq, float* dkv, int64_t batch, int64_t s_q, int64_t s_kv,
                 int64_t n_heads, int64_t d_qk, int64_t d_v, int64_t topk, float scale, int64_t q_offset,
                 const float* sinks, float* dsink, hipStream_t st);

}  // namespace dsa
