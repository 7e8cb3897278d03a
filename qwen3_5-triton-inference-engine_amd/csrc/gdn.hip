// Gated DeltaNet (GDN) delta-rule recurrence on gfx950: the decode update of
// the cached state (the varlen prefill is in gdn_scan.hip).
//
// Per token t and value head h, with the state S [DK, DV] fp32:
//   S      = exp(g_t) * S
//   mem    = k_t^T S                         [DV]
//   delta  = beta_t * (v_t - mem)            [DV]
//   S      = S + k_t delta^T
//   out_t  = q_t^T S                         [DV]  (stored as bf16)
// Reference: gdn_recurrent_prefill.py:151-246 (decode kernel), op :1185-1260.
//
// The lane layout and the step itself are in gdn_common.h.  The output uses
// q^T S_new = q^T S_decayed + (q^T k) delta, the same value as the reference's
// q^T S_new, so the two reductions of a token (k^T S and q^T S, plus q^T k)
// run together, before the update.
#include "gdn_common.h"

using namespace wy;
using namespace wy::gdn;

namespace {

__device__ __forceinline__ float *state_block(const GdnArgs &a, int b, int h, int kg, int col) {
  return a.state + b * a.s_b + h * a.s_h + int64_t(kg * kRows) * a.s_k + col;
}

// Decode: one token per sequence, S read from and written back to the cache.
// Workgroup = 8 wavefronts = 128 value columns of one (sequence, head); all
// 8 state loads of a lane are issued before the first use.
template <bool kContig>
__global__ __launch_bounds__(512) void gdn_recurrent_decode_kernel(const GdnArgs a) {
  const int bh = blockIdx.x;
  const int b = bh / a.heads, h = bh - b * a.heads;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int kg = lane & 15, cg = lane >> 4;
  const int col = blockIdx.y * 128 + wave * kWaveCols + cg * kCols;
  float *sp = state_block(a, b, h, kg, col);
  float s[kRows][kCols];
#pragma unroll
  for (int i = 0; i < kRows; ++i) {
    const float4 x = *reinterpret_cast<const float4 *>(sp + i * a.s_k);
    s[i][0] = x.x;
    s[i][1] = x.y;
    s[i][2] = x.z;
    s[i][3] = x.w;
  }
  TokenIn in;
  load_token<kContig>(a, b, h, kg, col, in);
  float o[kCols];
  gdn_step(s, in, o);
#pragma unroll
  for (int i = 0; i < kRows; ++i)
    *reinterpret_cast<float4 *>(sp + i * a.s_k) = make_float4(s[i][0], s[i][1], s[i][2], s[i][3]);
  if (kg == 0) store4<kContig>(a.out + b * a.o_t + h * a.o_h + col * a.o_d, a.o_d, o);
}

}  // namespace

extern "C" int wy_gdn_recurrent_decode(const void *q, const int64_t *q_strides, const void *k,
                                       const int64_t *k_strides, const void *v,
                                       const int64_t *v_strides, const float *beta,
                                       const int64_t *beta_strides, const float *g,
                                       const int64_t *g_strides, void *out,
                                       const int64_t *out_strides, float *state,
                                       const int64_t *state_strides, int batch, int num_heads,
                                       int key_dim, int value_dim, void *stream) {
  GdnArgs a;
  bool contig = false;
  const int rc = gdn_setup(a, contig, q, q_strides, k, k_strides, v, v_strides, beta,
                           beta_strides, g, g_strides, out, out_strides, state, state_strides,
                           num_heads, key_dim, value_dim);
  if (rc != WY_OK) return rc;
  if (batch < 0) return WY_E_SHAPE;
  if (batch == 0) return WY_OK;
  const dim3 grid(unsigned(batch * num_heads), unsigned(value_dim / 128));
  const hipStream_t st = static_cast<hipStream_t>(stream);
  if (contig)
    gdn_recurrent_decode_kernel<true><<<grid, 512, 0, st>>>(a);
  else
    gdn_recurrent_decode_kernel<false><<<grid, 512, 0, st>>>(a);
  return wyh::launch_status();
}
