// Gated DeltaNet varlen prefill on gfx950: the delta rule over a packed batch,
// 32 tokens at a time on bf16 MFMAs at fp32 accuracy.
//
// Per chunk of 32 tokens and head, with G = cumsum(g) inside the chunk and S
// the state entering it:
//   L[t, i] = beta_t exp(G_t - G_i) <k_t, k_i>   (i < t),   T = (I + L)^-1 diag(beta)
//   delta   = T (v - exp(G) (k S))
//   out     = exp(G) (q S) + A delta,  A[t, i] = exp(G_t - G_i) <q_t, k_i>  (i <= t)
//   S       = exp(G_last) S + k^T (exp(G_last - G) delta)
// the same values as the token-by-token recurrence
// (gdn_recurrent_prefill.py:52-143, op :1050-1146).
//
// Precision: q and k are bf16 and enter the MFMAs exactly; an fp32 operand x
// is cut by truncation into three bf16 pieces with x = h + m + l exactly, so a
// bf16 x fp32 product is three MFMAs with exact products summed in fp32, and a
// fp32 x fp32 product the six of weight >= 2^-16 (what is left out is below
// 2^-24 of the product).  G is summed in fp64 and kept as an fp32 pair, since
// a strongly decaying token would otherwise cost the small differences
// G_t - G_i after it their low bits.
//
// Layout: one wavefront owns 32 value columns of one head with all 128 key
// rows of S in registers, in the C layout of v_mfma_f32_32x32x16_bf16 (lane =
// column l % 32; register r of a 32-row tile = row (r & 3) + 8 (r >> 2) + 4
// (l / 32)).  Its registers 8s .. 8s + 7 are, up to an order of the rows that
// the A operand can share, exactly a B operand of k-step s: S, v - k S and
// delta go from one product into the next without leaving their lanes.  The A
// operands (k, q, T, A; k transposed by the LDS) are common to the workgroup's
// four wavefronts and lie in LDS with that row order: token or key 4 hf + (i &
// 3) + 8 (i >> 2) of a 16-group in slot 8 hf + i.
//
// Segments: a sequence longer than seg_len tokens is cut into segments that run
// side by side.  A first launch walks every segment but the last from a zero
// state and, as 128 further columns with v = 0 from the identity, its
// homogeneous solution P; a second folds S_{s+1} = P_s S_s + U_s along the
// segments; the last launch walks all segments from their true states.  In a
// packed batch seg_len is kSeg, so that a sequence gives the same bits in every
// batch; a prompt given as one alone has the chip to itself and takes the
// length that suits it (prompt_segment).
//
// Values that are not finite (infinities and NaN in the inputs, sums past
// FLT_MAX): the products spread them further than the recurrence does, and a
// cut infinity is NaN.  They are kept out of earlier tokens' and other
// columns' results, and a wavefront that met an infinity walks its columns once
// more token by token, putting the recurrence's own value wherever its output or
// state is not finite.  (A NaN needs no walk; a segment behind the one of the
// infinity gets NaN.)
//
// What bounds it: a chunk is 96 MFMAs of 32 cycles and ~750 VALU operations
// (cutting fp32 values is most of them) per wavefront, and T's chain (~4000
// cycles per group) holds up the workgroup's four; two workgroups per CU fill
// one another's gaps (LDS and 256 VGPRs allow no third).  Measured (16 heads,
// recurrence alone, against the walk of whole sequences token by token): 32 x
// 128 tokens 188 -> 42 us (48 where the longest sequence is not known), 24
// prompts of 22..4096 tokens (23772) 2.09 -> 0.51 ms, a packed batch of one
// sequence of 1000 tokens 308 -> 145 us, one prompt of 5003 alone 278 (chunk
// ops of csrc/gdn_chunk.hip) -> 181 us; one of 9 to 16 tokens 6.4 to 8.6 -> 9.5
// us, the chunk's fixed cost.
#include "gdn_common.h"

using namespace wy;
using namespace wy::gdn;

namespace {

constexpr int kC = 32;        // tokens per chunk
constexpr int kG = 64;        // tokens staged together (two chunks)
// Tokens per segment of a packed batch.  Shorter ones fill the chip when few
// sequences are there, longer ones save walking twice what fills it anyway: 128
// / 256 / 512 / 1024 tokens: 24 prompts of 22..4096 tokens 755 / 579 / 512 / 422
// us, 32 of 600 489 / 400 / 396 / 191, one of 5003 269 / 213 / 206 / 293, one of
// 1000 77 / 92 / 146 / 155.  One length for every sequence is a compromise of
// these.
#ifndef WY_GDN_SEG
#define WY_GDN_SEG 512
#endif
constexpr int kSeg = WY_GDN_SEG;
static_assert(kSeg % kG == 0, "segments hold whole groups");
// Sequences of at most kWalk tokens are walked token by token: a chunk costs
// the same whatever it holds.  One prompt, us a launch, walked by
// gdn_walk_kernel / as a chunk: 1 token 3.6 / 9.5, 8 tokens 6.3 / 9.5, 16
// tokens 8.6 / 9.5.  In batches the chunk wins earlier: 16 sequences of 8
// tokens 13.4 / 12.3, of 16 tokens 19.6 / 12.6, 64 of 8 32 / 29, of 16 55 / 37;
// the line is one for all, so that a sequence gives the same bits in every
// batch.
#ifndef WY_GDN_WALK
#define WY_GDN_WALK 8
#endif
constexpr int kWalk = WY_GDN_WALK;
// A batch of such sequences alone (known from the longest one's length, or from
// the token total) is gdn_walk_kernel's up to kWalkBatch sequences.  Inside
// the scan kernel, 8 columns a lane, a short sequence waits on its chains where
// the chip is not full, and saves the re-read q and k where it is: 64 sequences
// of 4 tokens 22 us / 28 inside, 256 of 4 80 / 105, 1024 of 4 490 / 404, 4096
// of one 1.9 ms / 1.2.
constexpr int kWalkBatch = 512;
constexpr int kKP = kDK + 8;  // LDS row pitch of k and q (bf16): 16-byte reads of 16 rows fill all banks
constexpr int kTP = kC + 8;   // of T and A
constexpr int kLP = kC + 4;   // of L (fp32)
constexpr int kWCols = 32;    // value columns per wavefront
constexpr float kMaxFinite = 3.402823466e38f;   // FLT_MAX: |x| <= it is false for inf and NaN

struct ScanLds {
  bf16_t K[kG][kKP];
  bf16_t Q[kG][kKP];
  bf16_t T[2][3][kC][kTP];    // chunk, piece (h, m, l), row t, columns i in slot order
  bf16_t A[2][3][kC][kTP];
  float Lt[2][kC * kLP + 16]; // L transposed: Lt[j kLP + i] = L[i][j], zero for i <= j (the
                              // padding keeps the chunks' rows in different banks); the blocks
                              // of X = (I + L)^-1 take the place of the diagonal ones and of the
                              // zero one
  float Gh[kG], Gl[kG], beta[kG];
  float eG[kG], E[kG], eL[4];
  int wild;   // an infinity in L, A, k, q, beta or g
};
static_assert(sizeof(ScanLds) <= 80 * 1024, "two workgroups per CU");
static_assert(offsetof(ScanLds, T) % 16 == 0 && offsetof(ScanLds, A) % 16 == 0 &&
                  offsetof(ScanLds, Lt) % 16 == 0 && offsetof(ScanLds, Gh) % 16 == 0 &&
                  offsetof(ScanLds, eG) % 16 == 0 && (kKP * 2) % 16 == 0 && (kTP * 2) % 16 == 0,
              "16-byte LDS accesses");

__device__ __forceinline__ f32x16_t mfma32(u32x4_t a, u32x4_t b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                 __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// the high halves of two words: bf16 truncations of two floats
__device__ __forceinline__ uint32_t hi_pair(float lo, float hi) {
  return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}
__device__ __forceinline__ float trunc_bf16(float x) {
  return __uint_as_float(__float_as_uint(x) & 0xffff0000u);
}

// Eight floats as three bf16 operands, x = p[0] + p[1] + p[2] exactly.
struct Pieces {
  u32x4_t p[3];
};
__device__ __forceinline__ Pieces cut8(const float (&x)[8]) {
  Pieces o;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float a = x[2 * e], b = x[2 * e + 1];
    const float a1 = a - trunc_bf16(a), b1 = b - trunc_bf16(b);
    const float a2 = a1 - trunc_bf16(a1), b2 = b1 - trunc_bf16(b1);
    o.p[0][e] = hi_pair(a, b);
    o.p[1][e] = hi_pair(a1, b1);
    o.p[2][e] = hi_pair(a2, b2);
  }
  return o;
}
template <int kFrom>
__device__ __forceinline__ Pieces cut_regs(const f32x16_t &v) {
  float x[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = v[kFrom + e];
  return cut8(x);
}

__device__ __forceinline__ f32x16_t zero16() {
  f32x16_t z;
#pragma unroll
  for (int e = 0; e < 16; ++e) z[e] = 0.f;
  return z;
}

__device__ __forceinline__ u32x2_t read_tr16(const bf16_t *p) {
  typedef short i16x4_t __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                         (__attribute__((address_space(3))) i16x4_t *)(p)));
}

// A 32 x 32 fp32 matrix in LDS pieces (row lr, k-steps 0 and 1) times R; the
// operands of k-step 0 are read ahead, those of k-step 1 under its MFMAs
struct Op3 {
  u32x4_t m[3];
};
__device__ __forceinline__ Op3 load_op(const bf16_t (*M)[kC][kTP], int s, int lr, int hf) {
  Op3 o;
#pragma unroll
  for (int n = 0; n < 3; ++n) o.m[n] = ld16(&M[n][lr][16 * s + 8 * hf]);
  return o;
}
__device__ __forceinline__ f32x16_t apply3(const Op3 &o, const Pieces &r, f32x16_t acc) {
  acc = mfma32(o.m[2], r.p[0], acc);
  acc = mfma32(o.m[1], r.p[1], acc);
  acc = mfma32(o.m[0], r.p[2], acc);
  acc = mfma32(o.m[1], r.p[0], acc);
  acc = mfma32(o.m[0], r.p[1], acc);
  return mfma32(o.m[0], r.p[0], acc);
}
// both k-steps; the second half of x is cut between the first six MFMAs
__device__ __forceinline__ f32x16_t apply(const bf16_t (*M)[kC][kTP], const Op3 &o0,
                                          const f32x16_t &x, int lr, int hf, f32x16_t acc) {
  const Op3 o1 = load_op(M, 1, lr, hf);
  const Pieces r0 = cut_regs<0>(x);
  acc = apply3(o0, r0, acc);
  const Pieces r1 = cut_regs<8>(x);
  return apply3(o1, r1, acc);
}

// Scheduling: a fence, and "kVops VALU operations behind each of kN MFMAs" --
// an MFMA keeps the matrix pipe for 32 cycles, in which its wave can issue
// eight VALU operations that do not depend on it.
__device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }
template <int kN, int kVops>
__device__ __forceinline__ void weave() {
#pragma unroll
  for (int i = 0; i < kN; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x2, kVops, 0);
  }
}

__device__ __forceinline__ uint32_t lane_xor1(uint32_t x) {   // quad_perm [1, 0, 3, 2]
  return __builtin_amdgcn_update_dpp(0, int(x), 0xB1, 0xf, 0xf, true);
}

// x plus the x of the lanes before it in DPP order (0 where there is none)
template <int kCtrl, int kRows>
__device__ __forceinline__ double dpp_add(double x) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, int(u), kCtrl, kRows, 0xf, false);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, int(u >> 32), kCtrl, kRows, 0xf, false);
  return x + __builtin_bit_cast(double, (uint64_t(hi) << 32) | lo);
}
// inclusive prefix sum over each half wave (32 lanes)
__device__ __forceinline__ double half_prefix(double x) {
  x = dpp_add<0x111, 0xf>(x);   // row_shr:1, 2, 4, 8 within 16 lanes
  x = dpp_add<0x112, 0xf>(x);
  x = dpp_add<0x114, 0xf>(x);
  x = dpp_add<0x118, 0xf>(x);
  return dpp_add<0x142, 0xa>(x);   // row_bcast:15 into the odd rows
}
__device__ __forceinline__ double lane_of(double x, int l) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = __builtin_amdgcn_readlane(int(u), l);
  const uint32_t hi = __builtin_amdgcn_readlane(int(u >> 32), l);
  return __builtin_bit_cast(double, (uint64_t(hi) << 32) | lo);
}

// first token of sequence i of the packed batch (no cu_seqlens: one sequence)
__device__ __forceinline__ int seq_start(const int32_t *cu, int token_num, int i) {
  return cu ? cu[i] : i ? token_num : 0;
}
__device__ __forceinline__ int seg_count(int len, int seg_len) {
  return len > seg_len ? (len - 1) / seg_len + 1 : 1;
}

// Item `item` of the packed batch's segments (of all of them, or of all but
// each sequence's last): its sequence, segment and the number of non-last
// segments in the sequences before it (its workspace slots start there).
// Each wavefront scans 64 sequences at a time.
__device__ __forceinline__ bool find_segment(const int32_t *cu, int token_num, int batch, int seg_len,
                                             int item, bool nonlast, int &b, int &s, int &slot0) {
  const int lane = threadIdx.x & 63;
  int items = 0, slots = 0;
  for (int b0 = 0; b0 < batch; b0 += 64) {
    const int i = b0 + lane;
    const int n =
        i < batch ? seg_count(seq_start(cu, token_num, i + 1) - seq_start(cu, token_num, i), seg_len)
                  : 0;
    const int extra = n > 0 ? n - 1 : 0, cnt = nonlast ? extra : n;
    int ci = cnt, si = extra;   // inclusive prefix sums
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int yc = __shfl_up(ci, o), ys = __shfl_up(si, o);
      if (lane >= o) {
        ci += yc;
        si += ys;
      }
    }
    const uint64_t hit = __ballot(items + ci > item);
    if (hit) {
      const int l = __builtin_ctzll(hit);   // uniform, like everything read from lane l
      b = b0 + l;
      s = item - items - __builtin_amdgcn_readlane(ci - cnt, l);
      slot0 = slots + __builtin_amdgcn_readlane(si - extra, l);
      return true;
    }
    items += __builtin_amdgcn_readlane(ci, 63);
    slots += __builtin_amdgcn_readlane(si, 63);
  }
  return false;
}

// Non-last segments in the sequences before b (of a batch with cu_seqlens).
__device__ __forceinline__ int slots_before(const int32_t *cu, int seg_len, int b, int lane) {
  int n = 0;
  for (int b0 = 0; b0 < b; b0 += 64) {
    const int i = b0 + lane;
    int x = i < b ? seg_count(cu[i + 1] - cu[i], seg_len) - 1 : 0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
    n += x;
  }
  return n;
}

// Two workspace blocks per (slot, head): the state after the segment (value
// columns: dv of them) and its homogeneous solution P [128][128].
struct Seg {
  float *state, *hom;
};
__device__ __forceinline__ Seg seg_block(float *ws, int slot, int h, int heads, int dv) {
  float *p = ws + (int64_t(slot) * heads + h) * kDK * (dv + kDK);
  return {p, p + int64_t(kDK) * dv};
}

// n rows of `pitch` bytes as a buffer resource that ends `width` bytes into the
// last one: reads past it give zero, writes are dropped (pitch >= width, so no
// row past the end lies inside; the launch checks).
template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(const T *p, int pitch, int n,
                                                            int width) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(p), 0, (n - 1) * pitch + width,
                                           0x00020000);
}
// a scalar the compiler must not form products of ahead of their use
__device__ __forceinline__ int opaque(int x) {
  asm volatile("" : "+s"(x));
  return x;
}
// element-wise form of a 16-byte piece, for other strides
__device__ __forceinline__ u32x4_t gather8(const bf16_t *p, int64_t stride) {
  u32x4_t w;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    w[e] = uint32_t(p[2 * e * stride]) | (uint32_t(p[(2 * e + 1) * stride]) << 16);
  return w;
}

// The kernel's first argument, read from the argument segment where it is used,
// and the lane, counted there (held in registers through the chunks, they would
// make others spill).
__device__ __forceinline__ GdnArgs args_again() {
  auto p = __builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  GdnArgs a;
  __builtin_memcpy(&a, (const void *)p, sizeof(a));
  return a;
}
__device__ __forceinline__ int lane_again() {
  const int all = opaque(-1);
  return __builtin_amdgcn_mbcnt_hi(all, __builtin_amdgcn_mbcnt_lo(all, 0));
}

// ---- the recurrence token by token: lane = kg + 16 cg holds key rows 8 kg ..
// + 7 of NC value columns, so every reduction stays inside a 16-lane DPP row.

// One token's inputs as loaded (bf16 bits, fp32 g / beta): the unpack happens
// at the step, so later tokens' loads stay in flight while a step runs.  g and
// beta are read through VGPR addresses: vector loads complete in order, a wait
// on a scalar load is a wait on all.
template <int NC>
struct TokenRaw {
  u32x4_t k, q;
  uint32_t v[(NC + 1) / 2];
  float g, beta;
};
typedef const __attribute__((address_space(1))) float gfloat_t;

template <bool kContig, int NC>
__device__ __forceinline__ void load_token_raw(const GdnArgs &a, int64_t t, int h, int kg, int col,
                                               TokenRaw<NC> &r) {
  const bf16_t *kp = a.k + t * a.k_t + h * a.k_h + kg * kRows * a.k_d;
  const bf16_t *qp = a.q + t * a.q_t + h * a.q_h + kg * kRows * a.q_d;
  const bf16_t *vp = a.v + t * a.v_t + h * a.v_h + col * a.v_d;
  if constexpr (kContig) {
    r.k = ld16(kp);
    r.q = ld16(qp);
    if constexpr (NC == 1) {
      r.v[0] = vp[0];
    } else {
#pragma unroll
      for (int e = 0; e < NC / 4; ++e) {   // rows of v are aligned to 8 bytes
        const u32x2_t w = *reinterpret_cast<const u32x2_t *>(vp + 4 * e);
        r.v[2 * e] = w[0];
        r.v[2 * e + 1] = w[1];
      }
    }
  } else {
    r.k = gather8(kp, a.k_d);
    r.q = gather8(qp, a.q_d);
    r.v[0] = vp[0];
#pragma unroll
    for (int e = 0; e < NC / 2; ++e)
      r.v[e] = uint32_t(vp[2 * e * a.v_d]) | (uint32_t(vp[(2 * e + 1) * a.v_d]) << 16);
  }
  gfloat_t *gp = (gfloat_t *)(a.g + t * a.g_t + h * a.g_h);
  gfloat_t *bp = (gfloat_t *)(a.beta + t * a.beta_t + h * a.beta_h);
  asm volatile("" : "+v"(gp), "+v"(bp));
  r.g = *gp;
  r.beta = *bp;
}

// One step on a lazily decayed state: the true state is c * s.  The decay only
// scales c; the reductions use s and are scaled by c, the rank-1 update adds
// k (delta / c).  When c drops below 2^-32 it is folded into s first (c = 0, a
// full decay, clears s).
template <int NC>
__device__ __forceinline__ void step_scaled(float (&s)[kRows][NC], float &c, const TokenRaw<NC> &in,
                                            float (&o)[NC]) {
  float k[kRows], q[kRows];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    k[2 * e] = bf16_lo(in.k[e]);
    k[2 * e + 1] = bf16_hi(in.k[e]);
    q[2 * e] = bf16_lo(in.q[e]);
    q[2 * e + 1] = bf16_hi(in.q[e]);
  }
  c *= __expf(in.g);
  if (c < 0x1p-32f) {   // uniform: c depends on the token only
#pragma unroll
    for (int i = 0; i < kRows; ++i)
#pragma unroll
      for (int j = 0; j < NC; ++j) s[i][j] *= c;
    c = 1.f;
  }
  float mem[NC], qs[NC], qk = 0.f;
#pragma unroll
  for (int j = 0; j < NC; ++j) mem[j] = qs[j] = 0.f;
#pragma unroll
  for (int i = 0; i < kRows; ++i) {
    qk = __fmaf_rn(q[i], k[i], qk);
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      mem[j] = __fmaf_rn(k[i], s[i][j], mem[j]);
      qs[j] = __fmaf_rn(q[i], s[i][j], qs[j]);
    }
  }
  qk = sum16(qk);
  const float inv_c = __builtin_amdgcn_rcpf(c);   // 1 ulp: only scales the update
  float dsc[NC];
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    const float vj = (j & 1) ? bf16_hi(in.v[j / 2]) : bf16_lo(in.v[j / 2]);
    const float delta = in.beta * (vj - c * sum16(mem[j]));
    o[j] = __fmaf_rn(qk, delta, c * sum16(qs[j]));
    dsc[j] = delta * inv_c;
  }
#pragma unroll
  for (int i = 0; i < kRows; ++i)
#pragma unroll
    for (int j = 0; j < NC; ++j) s[i][j] = __fmaf_rn(k[i], dsc[j], s[i][j]);
}

// Tokens [0, len) of the sequence at s0 from a zero state, the wavefront's 4 NC
// columns from col0; the state goes to sp (null: nowhere).  The sums keep one
// order whatever NC is: the same bits.  kAhead tokens are in flight: every load
// and store is unconditional (a request past the end re-reads the last token, the
// 16 lanes of a row store the same output), so a wait names exactly the token a
// step needs.
// kMend: only what is there and not finite is replaced, outputs from t_lo on.
template <bool kContig, int NC, bool kMend = false>
__device__ __forceinline__ void walk(const GdnArgs &a, int s0, int len, int h, int col0, int lane,
                                     float *sp, int t_lo = 0) {
  constexpr int kAhead = NC == 1 ? 4 : 2;
  const int kg = lane & 15, col = col0 + NC * (lane >> 4);
  float s[kRows][NC], c = 1.f;
#pragma unroll
  for (int i = 0; i < kRows; ++i)
#pragma unroll
    for (int j = 0; j < NC; ++j) s[i][j] = 0.f;
  if (len > 0) {
    auto put = [&](int t, const float (&o)[NC]) {
      bf16_t *op = a.out + int64_t(s0 + t) * a.o_t + h * a.o_h + col * a.o_d;
      if constexpr (kMend) {
        if (t < t_lo) return;
#pragma unroll
        for (int j = 0; j < NC; ++j)
          if ((op[j * a.o_d] & 0x7f80) == 0x7f80) op[j * a.o_d] = bf16_t(f32_to_bf16_bits(o[j]));
      } else if constexpr (!kContig || NC == 1) {
#pragma unroll
        for (int j = 0; j < NC; ++j) op[j * a.o_d] = bf16_t(f32_to_bf16_bits(o[j]));
      } else {
#pragma unroll
        for (int j = 0; j < NC; j += 4)   // rows of out are aligned to 8 bytes
          *reinterpret_cast<u32x2_t *>(op + j) =
              u32x2_t{pack_bf16x2(o[j], o[j + 1]), pack_bf16x2(o[j + 2], o[j + 3])};
      }
    };
    TokenRaw<NC> in[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
      load_token_raw<kContig, NC>(a, s0 + min(u, len - 1), h, kg, col, in[u]);
    const int whole = len - len % kAhead;
    for (int t = 0; t < whole; t += kAhead) {
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        float o[NC];
        step_scaled<NC>(s, c, in[u], o);
        put(t + u, o);
        load_token_raw<kContig, NC>(a, s0 + min(t + u + kAhead, len - 1), h, kg, col, in[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < kAhead - 1; ++u)
      if (whole + u < len) {
        float o[NC];
        step_scaled<NC>(s, c, in[u], o);
        put(whole + u, o);
      }
  }
  if (kMend && sp == nullptr) return;
  sp += int64_t(kg * kRows) * a.s_k + col;
#pragma unroll
  for (int i = 0; i < kRows; ++i)
#pragma unroll
    for (int j = 0; j < NC; ++j)
      if (!kMend || !(fabsf(sp[i * a.s_k + j]) <= kMaxFinite)) sp[i * a.s_k + j] = c * s[i][j];
}

// A batch of sequences of at most kWalk tokens each: one wavefront to 4 NC
// columns of a (sequence, head), sequence fastest.
template <bool kContig, int NC>
__global__ __launch_bounds__(64) void gdn_walk_kernel(const GdnArgs a, int token_num, int batch) {
  const int b = blockIdx.x % batch;
  const int h = (blockIdx.x / batch) % a.heads;
  const int col0 = blockIdx.x / (batch * a.heads) * 4 * NC;
  const int s0 = seq_start(a.cu_seqlens, token_num, b);
  walk<kContig, NC>(a, s0, seq_start(a.cu_seqlens, token_num, b + 1) - s0, h, col0, threadIdx.x,
                    a.state + b * a.s_b + h * a.s_h);
}

// ---- infinities.  (fmaxf passes NaN by.)
__device__ __forceinline__ bool has_inf(const f32x16_t &v) {
  float m = 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) m = fmaxf(m, fabsf(v[r]));
  return m > kMaxFinite;
}
__device__ __forceinline__ bool has_inf(const f32x16_t (&S)[4]) {
  return has_inf(S[0]) || has_inf(S[1]) || has_inf(S[2]) || has_inf(S[3]);
}
// one in keys 64 hf .. + 63 of a row of k or q
__device__ __forceinline__ bool row_has_inf(const bf16_t *row, int hf) {
  int found = 0;
#pragma unroll 1
  for (int i = 64 * hf; i < 64 * hf + 64; ++i) found |= (row[i] & 0x7fff) == 0x7f80;
  return found != 0;
}

// kState: a non-last segment's state (and homogeneous solution) only.
template <bool kContig, bool kState>
__global__ __launch_bounds__(256, 2) void gdn_scan_kernel(const GdnArgs a, int token_num, int batch,
                                                          float *ws, int slots, int seg_len) {
  extern __shared__ __align__(16) unsigned char scan_smem[];
  ScanLds &L = *reinterpret_cast<ScanLds *>(scan_smem);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, hf = lane >> 5;
  const int vblocks = a.dv / 128;
  // grid: head fastest, then column block (kState: one more, the homogeneous
  // columns), then segment
  const int cols = kState ? vblocks + 1 : vblocks;
  const int h = blockIdx.x % a.heads;
  const int vb = (blockIdx.x / a.heads) % cols;
  const int item = blockIdx.x / (a.heads * cols);
  const bool hom = kState && vb == vblocks;
  int b, seg = 0, slot0 = 0;
  // A search costs a memory round trip for every 64 sequences.  Larger batches
  // list the non-last segments (few, and the longest walks) first and then every
  // sequence's last one, whose sequence is the item's number: 4096 sequences of
  // 8 tokens searched for took 4.0 ms, listed 2.2.
  const bool listed = !kState && batch > 64 && item >= slots;
  if (slots == 0) {
    b = item;   // no segments: one item per sequence
    if (b >= batch) return;
  } else if (listed) {
    b = item - slots;
  } else if (!find_segment(a.cu_seqlens, token_num, batch, seg_len, item, kState || batch > 64,
                           b, seg, slot0)) {
    return;
  }
  // the same in every lane: pointers and buffer resources built from them
  // stay in scalar registers
  b = __builtin_amdgcn_readfirstlane(b);
  seg = __builtin_amdgcn_readfirstlane(seg);
  slot0 = __builtin_amdgcn_readfirstlane(slot0);
  const int s0 = seq_start(a.cu_seqlens, token_num, b);
  const int len = seq_start(a.cu_seqlens, token_num, b + 1) - s0;
  if constexpr (!kState) {
    if (len <= kWalk) {
      const GdnArgs ar = args_again();
      walk<kContig, 8>(ar, s0, len, h, vb * 128 + wave * kWCols, lane_again(),
                       ar.state + b * ar.s_b + h * ar.s_h);
      return;
    }
  }
  const int nseg = slots == 0 ? 1 : seg_count(len, seg_len);
  if (listed && nseg > 1) {
    seg = nseg - 1;
    slot0 = slots_before(a.cu_seqlens, seg_len, b, lane);
  }
  if (slot0 + nseg - 1 > slots) return;   // more tokens than the workspace was sized for
  if (hom && seg == 0) return;            // the first segment starts from a known (zero) state
  const int t_lo = slots == 0 ? 0 : seg * seg_len;
  const int t_hi = slots == 0 ? len : min(len, t_lo + seg_len);
  const int col = (hom ? 0 : vb * 128) + wave * kWCols + lr;

  // Where the state goes, and the distance of its rows: formed here, not by
  // loads of the arguments in front of the stores.
  float *dst = nullptr;
  int64_t row = a.s_k;
  if constexpr (kState) {
    const Seg blk = seg_block(ws, slot0 + seg, h, a.heads, a.dv);
    dst = hom ? blk.hom : blk.state;
    row = hom ? kDK : a.dv;
  } else if (seg == nseg - 1) {
    dst = a.state + b * a.s_b + h * a.s_h;
  }
  asm volatile("" : "+s"(dst), "+s"(row));

  f32x16_t S[4];
#pragma unroll
  for (int rt = 0; rt < 4; ++rt) S[rt] = zero16();
  if (hom) {
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        S[rt][r] = 32 * rt + (r & 3) + 8 * (r >> 2) + 4 * hf == col ? 1.f : 0.f;
  } else if (!kState && seg > 0) {
    const int pitch = opaque(a.dv * 4);
    const auto rs = rows_rsrc(seg_block(ws, slot0 + seg - 1, h, a.heads, a.dv).state, pitch, kDK,
                              pitch);
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        S[rt][r] = __builtin_bit_cast(
            float, __builtin_amdgcn_raw_buffer_load_b32(
                       rs, 4 * hf * pitch + col * 4, (32 * rt + (r & 3) + 8 * (r >> 2)) * pitch, 0));
  }

  // the next group's k and q rows (thread: 8-key piece tid & 15 of rows tid / 16 + 16 i), g and beta
  u32x4_t rk[4], rq[4];
  float rg = 0.f, rb = 0.f;
  auto load_rows = [&](u32x4_t (&r)[4], const bf16_t *src, int64_t st, int64_t sd, int64_t t,
                       int n) {
    src += t * st;
    if constexpr (kContig) {
      const int pitch = opaque(int(st) * 2);
      const auto rs = rows_rsrc(src, pitch, n, kDK * 2);
      const int off = (tid >> 4) * pitch + (tid & 15) * 16;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        r[i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                               rs, off, 16 * i * pitch, 0));
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = (tid >> 4) + 16 * i;
        r[i] = u32x4_t{0u, 0u, 0u, 0u};
        if (row < n) r[i] = gather8(src + row * st + (tid & 15) * 8 * sd, sd);
      }
    }
  };
  auto load_gate = [&](const float *src, int64_t st, int64_t t, int n) {
    src += t * st;
    if constexpr (kContig) {
      const int pitch = opaque(int(st) * 4);
      return __builtin_bit_cast(
          float, __builtin_amdgcn_raw_buffer_load_b32(rows_rsrc(src, pitch, n, 4), lane * pitch,
                                                      0, 0));
    } else {
      return lane < n ? src[lane * st] : 0.f;
    }
  };
  auto load_group = [&](int t0) {
    const int n = min(kG, t_hi - t0);
    load_rows(rk, a.k + h * a.k_h, a.k_t, a.k_d, s0 + t0, n);
    if constexpr (!kState) load_rows(rq, a.q + h * a.q_h, a.q_t, a.q_d, s0 + t0, n);
    rg = load_gate(a.g + h * a.g_h, a.g_t, s0 + t0, n);   // (used by wave 3)
    rb = load_gate(a.beta + h * a.beta_h, a.beta_t, s0 + t0, n);
  };
  // a 16-byte piece (8 keys) into slot order: keys 4 .. 7 of a 16-group's half
  // go 8 slots behind keys 0 .. 3
  const int kslot = 16 * ((tid & 15) >> 1) + 4 * (tid & 1);
  auto put_row = [&](bf16_t (*dst)[kKP], int row, u32x4_t x) {
    *reinterpret_cast<u32x2_t *>(&dst[row][kslot]) = u32x2_t{x[0], x[1]};
    *reinterpret_cast<u32x2_t *>(&dst[row][kslot + 8]) = u32x2_t{x[2], x[3]};
  };

  if (tid == 192) L.wild = 0;   // (wave 3 is the first to set it)
  uint64_t wild = 0;   // not 0: this wavefront met an infinity
  // the block of T above the diagonal is zero and never written again
  for (int i = tid; i < 2 * 3 * 16 * 4; i += 256)
    *reinterpret_cast<u32x2_t *>(&L.T[i / 192][i / 64 % 3][i / 4 % 16][16 + 4 * (i % 4)]) =
        u32x2_t{0u, 0u};
  // v of the next chunk: requested when the chunk before it has used its own.
  // A lane reads two neighbouring columns of one row -- an even lane those of
  // row r, an odd lane those of row r + 1 (r even) -- and swaps at the use.
  const int odd = lane & 1;
  uint32_t v[8];
  auto load_v = [&](int tc) {
    const int n = min(kC, t_hi - tc);
    const bf16_t *vp = a.v + (s0 + tc) * a.v_t + h * a.v_h;
    if constexpr (kContig) {
      const int pitch = opaque(int(a.v_t) * 2);
      const auto rs = rows_rsrc(vp, pitch, n, a.dv * 2);
      const int off = (4 * hf + odd) * pitch + (col - odd) * 2;
#pragma unroll
      for (int r2 = 0; r2 < 8; ++r2)
        v[r2] = __builtin_amdgcn_raw_buffer_load_b32(
            rs, off, (2 * (r2 & 1) + 8 * (r2 >> 1)) * pitch, 0);
    } else {
#pragma unroll
      for (int r2 = 0; r2 < 8; ++r2) {
        const int t = 2 * (r2 & 1) + 8 * (r2 >> 1) + 4 * hf + odd;
        const bf16_t *p = vp + t * a.v_t + (col - odd) * a.v_d;
        v[r2] = t < n ? uint32_t(p[0]) | (uint32_t(p[a.v_d]) << 16) : 0u;
      }
    }
  };

  if (t_lo < t_hi) {
    load_group(t_lo);
    if (!hom) load_v(t_lo);
  }
  for (int t0 = t_lo; t0 < t_hi; t0 += kG) {
    // T's chain and the staging before it hold up all four waves: they go first
    __builtin_amdgcn_s_setprio(2);
    const int nval = min(kG, t_hi - t0);
    // ---- stage the group
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = (tid >> 4) + 16 * i;
      put_row(L.K, row, rk[i]);
      if constexpr (!kState) put_row(L.Q, row, rq[i]);
    }
    if (wave == 3) {
      // G in units of log2, summed in fp64.  The clamp keeps differences of G
      // finite where g = -inf (NaN passes) and lies so low that what it clears
      // stays cleared: later tokens' growth inside the chunk is at most 31
      // factors below 2^128 (a larger one is infinite), and 2^(-8192 + 3968)
      // is 0.  The fp32 pair holds 32 clamped tokens' sum to 2^-31.
      const double g2 = double(rg) * 1.4426950408889634074;
      const double G = half_prefix(lane < nval ? (g2 < -8192.0 ? -8192.0 : g2) : 0.0);
      const double G0 = lane_of(G, 31), G1 = lane_of(G, 63), Gl = lane < 32 ? G0 : G1;
      const float gh = float(G);
      L.Gh[lane] = gh;
      L.Gl[lane] = float(G - double(gh));
      // a beta that is not finite makes its row of v - k S (through eG) not
      // finite, and so the columns from this token on; T itself stays finite
      const bool fine = fabsf(rb) <= kMaxFinite;
      if (!kState && __ballot(lane < nval && (fabsf(rb) > kMaxFinite || rg > kMaxFinite)) != 0)
        L.wild = 1;
      L.beta[lane] = lane < nval && fine ? rb : 0.f;
      L.eG[lane] = lane >= nval || fine ? __builtin_amdgcn_exp2f(gh) : __builtin_nanf("");
      L.E[lane] = __builtin_amdgcn_exp2f(float(Gl - G));
      if ((lane & 31) == 31) L.eL[lane >> 5] = __builtin_amdgcn_exp2f(float(Gl));
    }
    __syncthreads();

    // ---- L and from it T (waves 0, 1) and A (waves 2, 3) of the two chunks,
    // from <x_i, k_j> with lane = j (L: the column; A: the row t), registers = i
    {
      // the lane, opaque: addresses and masks made from it here are not worth
      // registers across the loop
      int lane = tid & 63;
      asm volatile("" : "+v"(lane));
      const int lr = lane & 31, hf = lane >> 5;
      const int cc = wave & 1, rb0 = kC * cc;
      const bool second = wave >= 2;
      if (!second || !kState) {
        const bf16_t(*X)[kKP] = second ? L.Q : L.K;
        f32x16_t acc = zero16();
#pragma unroll
        for (int s4 = 0; s4 < 8; s4 += 4) {
          u32x4_t kf[4], xf[4];
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            kf[s] = ld16(&L.K[rb0 + lr][16 * (s4 + s) + 8 * hf]);
            xf[s] = ld16(&X[rb0 + lr][16 * (s4 + s) + 8 * hf]);
          }
          fence();
#pragma unroll
          for (int s = 0; s < 4; ++s) acc = mfma32(kf[s], xf[s], acc);
          fence();
        }
        const float gh = L.Gh[rb0 + lr], gl = L.Gl[rb0 + lr];
        if (!second) {
          float *Lt = L.Lt[cc];
          float nans = 0.f;
#pragma unroll
          for (int q4 = 0; q4 < 4; ++q4) {
            const int i0 = 8 * q4 + 4 * hf;
            const f32x4_t Gh = *reinterpret_cast<const f32x4_t *>(&L.Gh[rb0 + i0]);
            const f32x4_t Gl = *reinterpret_cast<const f32x4_t *>(&L.Gl[rb0 + i0]);
            const f32x4_t be = *reinterpret_cast<const f32x4_t *>(&L.beta[rb0 + i0]);
            f32x4_t o;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float x = be[e] * (__builtin_amdgcn_exp2f((Gh[e] - gh) + (Gl[e] - gl)) *
                                       acc[4 * q4 + e]);
              o[e] = i0 + e > lr ? x : 0.f;
              nans += o[e];
            }
            *reinterpret_cast<f32x4_t *>(&Lt[lr * kLP + i0]) = o;
          }
          if (__ballot(!(fabsf(nans) <= kMaxFinite)) != 0) {
            // as for beta: mark the rows of L that are not finite, keep T finite
            bool inf = !kState && row_has_inf(L.K[rb0 + lr], hf);
#pragma unroll 1
            for (int i = 0; i < kC; ++i) {
              const float x = Lt[lr * kLP + i];
              if (!(fabsf(x) <= kMaxFinite)) {
                inf |= fabsf(x) > kMaxFinite;
                L.eG[rb0 + i] = __builtin_nanf("");
                Lt[lr * kLP + i] = 0.f;
              }
            }
            if (!kState && __ballot(inf) != 0) L.wild = 1;
          }
          // T = (I + L)^-1 diag(beta).  The two diagonal 16 x 16 blocks by
          // back substitution of x (I + L) = e_t, a row t per lane (the upper
          // half wave repeats the lower); row j of Lt is requested while row
          // j + 1 is used.
          const int blk = (lane >> 4) & 1, t16 = lane & 15;
          const float *Lb = Lt + 16 * blk * (kLP + 1);
          float x[16];
          f32x4_t row[2][4];
          auto fetch = [&](int j) {
#pragma unroll
            for (int i4 = (j + 1) / 4; i4 < 4; ++i4)
              row[j & 1][i4] = *reinterpret_cast<const f32x4_t *>(&Lb[j * kLP + 4 * i4]);
          };
          fetch(14);
          x[15] = 15 == t16 ? 1.f : 0.f;
#pragma unroll
          for (int j = 14; j >= 0; --j) {
            if (j > 0) fetch(j - 1);
            fence();
            float a2[2] = {j == t16 ? 1.f : 0.f, 0.f};
#pragma unroll
            for (int i = j + 1; i < 16; ++i)
              a2[i & 1] = __fmaf_rn(-x[i], row[j & 1][i / 4][i % 4], a2[i & 1]);
            x[j] = a2[0] + a2[1];   // zero for j > t
            fence();
          }
          if (hf == 0) {
#pragma unroll
            for (int j4 = 0; j4 < 4; ++j4)
              *reinterpret_cast<f32x4_t *>(&Lt[(16 * blk + t16) * kLP + 16 * blk + 4 * j4]) =
                  f32x4_t{x[4 * j4], x[4 * j4 + 1], x[4 * j4 + 2], x[4 * j4 + 3]};
          }
          __builtin_amdgcn_wave_barrier();
          // The block below the diagonal, T21 = -X22 L21 X11, transposed: P =
          // L21^T X22^T, then -X11^T P, on fp32 MFMAs (lane = column l % 16 =
          // row t of T21, k index 4 (l / 16) + step, so P goes in as it came).
          const int q = lane >> 4;
          const f32x4_t l21 = *reinterpret_cast<const f32x4_t *>(&Lt[t16 * kLP + 16 + 4 * q]);
          const f32x4_t x22 = *reinterpret_cast<const f32x4_t *>(&Lt[(16 + t16) * kLP + 16 + 4 * q]);
          float x11[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) x11[e] = Lt[(4 * q + e) * kLP + t16];
          f32x4_t P = {0.f, 0.f, 0.f, 0.f}, D = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int e = 0; e < 4; ++e)
            P = __builtin_amdgcn_mfma_f32_16x16x4f32(l21[e], x22[e], P, 0, 0, 0);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            D = __builtin_amdgcn_mfma_f32_16x16x4f32(x11[e], P[e], D, 0, 0, 0);
          *reinterpret_cast<f32x4_t *>(&Lt[(16 + t16) * kLP + 4 * q]) = -D;
        } else {
          float nans = 0.f;
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            float x[8];
#pragma unroll
            for (int q2 = 0; q2 < 2; ++q2) {
              const int i0 = 16 * s + 8 * q2 + 4 * hf;
              const f32x4_t Gh = *reinterpret_cast<const f32x4_t *>(&L.Gh[rb0 + i0]);
              const f32x4_t Gl = *reinterpret_cast<const f32x4_t *>(&L.Gl[rb0 + i0]);
#pragma unroll
              for (int e = 0; e < 4; ++e)
                x[4 * q2 + e] = i0 + e <= lr
                                    ? __builtin_amdgcn_exp2f((gh - Gh[e]) + (gl - Gl[e])) *
                                          acc[8 * s + 4 * q2 + e]
                                    : 0.f;
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) nans += x[e];
            const Pieces p = cut8(x);
#pragma unroll
            for (int n = 0; n < 3; ++n) st16(&L.A[cc][n][lr][16 * s + 8 * hf], p.p[n]);
          }
          if (__ballot(!(fabsf(nans) <= kMaxFinite)) != 0) {
            bool inf = row_has_inf(L.K[rb0 + lr], hf) || row_has_inf(L.Q[rb0 + lr], hf);
#pragma unroll 1
            for (int i = 0; i < kC; ++i) inf |= (L.A[cc][0][lr][i] & 0x7fff) == 0x7f80;
            if (__ballot(inf) != 0) L.wild = 1;
          }
        }
      }
    }
    __syncthreads();
    {
      // T = (I + L)^-1 diag(beta) in pieces: eight columns of a row per thread,
      // in slot order (the block above the diagonal stays zero)
      const int g8 = tid & 3, row = (tid >> 2) & 31, cc = tid >> 7;
      const int j0 = 16 * (g8 >> 1) + 4 * (g8 & 1);
      if (16 * (g8 >> 1) <= row) {
        float y[8];
#pragma unroll
        for (int n = 0; n < 2; ++n) {
          const f32x4_t x = *reinterpret_cast<const f32x4_t *>(&L.Lt[cc][row * kLP + j0 + 8 * n]);
          const f32x4_t be = *reinterpret_cast<const f32x4_t *>(&L.beta[kC * cc + j0 + 8 * n]);
#pragma unroll
          for (int e = 0; e < 4; ++e) y[4 * n + e] = x[e] * be[e];
        }
        const Pieces p = cut8(y);
#pragma unroll
        for (int n = 0; n < 3; ++n) st16(&L.T[cc][n][row][8 * g8], p.p[n]);
      }
    }
    __syncthreads();

    __builtin_amdgcn_s_setprio(0);
    // the next group is in flight during the recurrence (defined on both
    // paths: kept from the last load, the registers would be live through T)
    if (t0 + kG < t_hi) {
      load_group(t0 + kG);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) rk[i] = rq[i] = u32x4_t{0u, 0u, 0u, 0u};
      rg = rb = 0.f;
    }
    // ---- the recurrence over the group's chunks
    for (int cc = 0; cc < 2; ++cc) {
      const int rb0 = kC * cc;
      if (rb0 >= nval) break;
      const int64_t tb = s0 + t0 + rb0;   // first token
      const int nv = min(kC, nval - rb0);
      f32x16_t ks = zero16(), qs = zero16();
      if (hom || seg > 0 || t0 + rb0 > 0) {   // a sequence's first chunk: S = 0
        // k S and q S: the next k-step's operands are read and cut between the
        // MFMAs of this one
        u32x4_t kf = ld16(&L.K[rb0 + lr][8 * hf]), qf = {};
        if constexpr (!kState) qf = ld16(&L.Q[rb0 + lr][8 * hf]);
        Pieces sp = cut_regs<0>(S[0]);
        fence();
#pragma unroll
        for (int s = 0; s < 8; ++s) {
          u32x4_t kn = kf, qn = qf;
          Pieces sn = sp;
          if (s < 7) {
            kn = ld16(&L.K[rb0 + lr][16 * (s + 1) + 8 * hf]);
            if constexpr (!kState) qn = ld16(&L.Q[rb0 + lr][16 * (s + 1) + 8 * hf]);
            sn = (s & 1) ? cut_regs<0>(S[(s + 1) >> 1]) : cut_regs<8>(S[(s + 1) >> 1]);
          }
#pragma unroll
          for (int n = 2; n >= 0; --n) {
            ks = mfma32(kf, sp.p[n], ks);
            if constexpr (!kState) qs = mfma32(qf, sp.p[n], qs);
          }
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
          if constexpr (kState)
            weave<3, 15>();
          else
            weave<6, 8>();
          fence();
          kf = kn;
          qf = qn;
          sp = sn;
        }
      }
      const Op3 To = load_op(L.T[cc], 0, lr, hf);
      f32x16_t R = zero16();
      if (!hom) {
#pragma unroll
        for (int r2 = 0; r2 < 8; ++r2) {
          // lane parity p holds columns c - p, c - p + 1 of row r + p: the own
          // column of that row, and the partner's of the other
          const uint32_t got = lane_xor1(v[r2]);
          const float own = __uint_as_float(odd ? v[r2] & 0xffff0000u : v[r2] << 16);
          const float oth = __uint_as_float(odd ? got & 0xffff0000u : got << 16);
          R[2 * r2] = odd ? oth : own;
          R[2 * r2 + 1] = odd ? own : oth;
        }
      }
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const f32x4_t eg = *reinterpret_cast<const f32x4_t *>(&L.eG[rb0 + 8 * q4 + 4 * hf]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int r = 4 * q4 + e;
          R[r] = __fmaf_rn(-eg[e], ks[r], R[r]);
          if constexpr (!kState) qs[r] *= eg[e];
        }
      }
      if (!hom && t0 + rb0 + kC < t_hi) load_v(t0 + rb0 + kC);
      fence();
      f32x16_t delta = apply(L.T[cc], To, R, lr, hf, zero16());
      Op3 Ao;
      if constexpr (!kState) Ao = load_op(L.A[cc], 0, lr, hf);
      // Row 31 of the product sees every row of R: where it is not finite, a
      // value that is not finite sits in this column of R from some token
      // t_bad on, and 0 x inf has spread it to the rows before as well.  Those
      // are formed again without it; from t_bad on the column is set to NaN
      // (which the walk at the end replaces if it came from an infinity).
      int t_bad = kC;
      const bool any = __ballot(!(fabsf(delta[15]) <= kMaxFinite) && hf == 1) != 0;
      if (any) {
        if constexpr (!kState) wild |= __ballot(has_inf(R) || has_inf(S));
#pragma unroll
        for (int r = 15; r >= 0; --r)
          if (!(fabsf(R[r]) <= kMaxFinite)) t_bad = (r & 3) + 8 * (r >> 2) + 4 * hf;
        t_bad = min(t_bad, __shfl_xor(t_bad, 32));
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if ((r & 3) + 8 * (r >> 2) + 4 * hf >= t_bad) R[r] = 0.f;
        delta = apply(L.T[cc], To, R, lr, hf, zero16());
      }
      // out = exp(G) q S + A delta
      if constexpr (!kState) {
        const f32x16_t o = apply(L.A[cc], Ao, delta, lr, hf, qs);
        // (row 31 of this product sees every row of delta)
        if (__ballot(!(fabsf(o[15]) <= kMaxFinite)) != 0)
          wild |= __ballot(has_inf(o) || has_inf(delta) || has_inf(S));
        bf16_t *op = a.out + tb * a.o_t + h * a.o_h;
        const int pitch = opaque(int(a.o_t) * 2);
        const auto rs = rows_rsrc(op, pitch, nv, a.dv * 2);
        const int off = (4 * hf + odd) * pitch + (col - odd) * 2;
#pragma unroll
        for (int r2 = 0; r2 < 8; ++r2) {
          const int t = 2 * (r2 & 1) + 8 * (r2 >> 1) + 4 * hf;
          const float x0 = any && t >= t_bad ? __builtin_nanf("") : o[2 * r2];
          const float x1 = any && t + 1 >= t_bad ? __builtin_nanf("") : o[2 * r2 + 1];
          // as for v: columns c, c + 1 of row t in the even lane, of row t + 1
          // in the odd one
          const float own = odd ? x1 : x0;
          const float got = __uint_as_float(lane_xor1(__float_as_uint(odd ? x0 : x1)));
          const uint32_t y = odd ? pack_bf16x2(got, own) : pack_bf16x2(own, got);
          if constexpr (kContig) {
            __builtin_amdgcn_raw_buffer_store_b32(y, rs, off,
                                                  (2 * (r2 & 1) + 8 * (r2 >> 1)) * pitch, 0);
          } else if (t + odd < nv) {
            bf16_t *p = op + (t + odd) * a.o_t + (col - odd) * a.o_d;
            p[0] = bf16_t(y);
            p[a.o_d] = bf16_t(y >> 16);
          }
        }
      }
      fence();   // (interleaved with what follows, this needs too many registers)
      f32x16_t dd;
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const f32x4_t ex = *reinterpret_cast<const f32x4_t *>(&L.E[rb0 + 8 * q4 + 4 * hf]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int r = 4 * q4 + e;
          float x = delta[r];
          if (any && e + 8 * q4 + 4 * hf >= t_bad) x = __builtin_nanf("");
          dd[r] = x * ex[e];
        }
      }
      const Pieces ddp[2] = {cut_regs<0>(dd), cut_regs<8>(dd)};
      const float el = L.eL[cc];
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) S[rt] *= el;
      // k transposed: the 16-lane group (keys 32 rt + 16 g + 0 .. 15, token
      // half hf) receives tokens 16 s + 4 hf + 0 .. 3 and + 8; its lane a
      // addresses token row a / 4 and the slots of keys 4 (a % 4) .. + 3
      const int ln = lane & 15, g = (lane >> 4) & 1, c4 = ln & 3;
      const bf16_t *ktp =
          &L.K[rb0 + 4 * hf + (ln >> 2)][16 * g + 8 * (c4 & 1) + 4 * (c4 >> 1)];
      auto read_kt = [&](int i) {   // i = 2 rt + s
        const bf16_t *p = ktp + 16 * (i & 1) * kKP + 32 * (i >> 1);
        const u32x2_t x0 = read_tr16(p), x1 = read_tr16(p + 8 * kKP);
        return u32x4_t{x0[0], x0[1], x1[0], x1[1]};
      };
      u32x4_t kt[2] = {read_kt(0), read_kt(1)};
      fence();
#pragma unroll
      for (int i = 0; i < 8; ++i) {
#pragma unroll
        for (int n = 2; n >= 0; --n) S[i >> 1] = mfma32(kt[i & 1], ddp[i & 1].p[n], S[i >> 1]);
        if (i < 6) kt[i & 1] = read_kt(i + 2);
        fence();
      }
    }
    __syncthreads();   // the next group rewrites the LDS
  }

  if (dst == nullptr) {
  } else if (kContig || kState) {
    const int pitch = opaque(int(row) * 4);
    const auto rs = rows_rsrc(dst, pitch, kDK, (hom ? kDK : a.dv) * 4);
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(S[rt][r]), rs,
                                              4 * hf * pitch + col * 4,
                                              (32 * rt + (r & 3) + 8 * (r >> 2)) * pitch, 0);
  } else {
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        dst[(32 * rt + (r & 3) + 8 * (r >> 2) + 4 * hf) * row + col] = S[rt][r];
  }
  if constexpr (!kState) {
    // (behind the stores, which take longer)
    float z[4] = {0.f, 0.f, 0.f, 0.f};   // NaN unless all of S is finite
#pragma unroll
    for (int r = 0; r < 16; ++r)
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) z[rt] = __fmaf_rn(S[rt][r], 0.f, z[rt]);
    if (__ballot((z[0] + z[1]) + (z[2] + z[3]) != 0.f) != 0) wild |= __ballot(has_inf(S));
    if (t_lo < t_hi) wild |= uint64_t(__builtin_amdgcn_readfirstlane(L.wild));
    if (wild != 0) {
      __threadfence_block();   // other lanes' results are read back
      walk<kContig, 8, true>(args_again(), s0, t_hi, h, vb * 128 + wave * kWCols, lane_again(), dst,
                             t_lo);
    }
  }
}

// Fold the segments' states: S_{s+1} = P_s S_s + U_s for s = 1 .. nseg - 2, in
// place of U_s.  Workgroup = one (sequence, head, 32 value columns); wave w
// forms rows 32 w .. + 31, the cut state goes through LDS in operand order.
__global__ __launch_bounds__(256) void gdn_fold_kernel(const int32_t *cu, int token_num, int heads,
                                                       int dv, float *ws, int slots, int seg_len) {
  __shared__ __align__(16) u32x4_t sp[2][8][3][64];   // k-step, piece, lane; two steps' worth
  const int h = blockIdx.x % heads;
  const int cb = (blockIdx.x / heads) % (dv / kWCols);
  const int b = blockIdx.x / (heads * (dv / kWCols));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lr = lane & 31, hf = lane >> 5;
  const int nseg =
      seg_count(seq_start(cu, token_num, b + 1) - seq_start(cu, token_num, b), seg_len);
  if (nseg < 3) return;   // S_1 = U_0 needs no fold
  const int slot0 = slots_before(cu, seg_len, b, lane);   // (b > 0: there is a cu)
  if (slot0 + nseg - 1 > slots) return;
  const int col = cb * kWCols + lr;
  const int row0 = 32 * wave + 4 * hf;
  auto publish = [&](const f32x16_t &t, int buf) {
    const Pieces lo = cut_regs<0>(t), hi = cut_regs<8>(t);
#pragma unroll
    for (int n = 0; n < 3; ++n) {
      sp[buf][2 * wave][n][lane] = lo.p[n];
      sp[buf][2 * wave + 1][n][lane] = hi.p[n];
    }
  };
  // row 32 w + lr of P, keys in the operand's order (two quads per k-step), and
  // U: requested one segment ahead
  f32x4_t x[2][8][2];
  f32x16_t u[2];
  auto fetch = [&](int seg, f32x4_t (&px)[8][2], f32x16_t &pu) {
    const Seg blk = seg_block(ws, slot0 + seg, h, heads, dv);
    const float *pr = blk.hom + (32 * wave + lr) * kDK + 4 * hf;
#pragma unroll
    for (int k = 0; k < 8; ++k)
#pragma unroll
      for (int q = 0; q < 2; ++q) px[k][q] = *reinterpret_cast<const f32x4_t *>(pr + 16 * k + 8 * q);
    const float *us = blk.state + col;
#pragma unroll
    for (int r = 0; r < 16; ++r) pu[r] = us[int64_t(row0 + (r & 3) + 8 * (r >> 2)) * dv];
  };
  {
    const float *us = seg_block(ws, slot0, h, heads, dv).state + col;
    f32x16_t t;
#pragma unroll
    for (int r = 0; r < 16; ++r) t[r] = us[int64_t(row0 + (r & 3) + 8 * (r >> 2)) * dv];
    fetch(1, x[0], u[0]);
    publish(t, 0);
  }
  for (int s0 = 1; s0 < nseg - 1; s0 += 2)
#pragma unroll
    for (int buf = 0; buf < 2; ++buf) {   // segment s uses register set and LDS buffer (s - 1) & 1
      const int s = s0 + buf;
      if (s >= nseg - 1) break;
      if (s + 1 < nseg - 1) fetch(s + 1, x[buf ^ 1], u[buf ^ 1]);
      f32x16_t t = u[buf];
      __syncthreads();   // S_s published; the other buffer's readers are done
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        float y[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] = x[buf][k][i >> 2][i & 3];
        const Pieces p = cut8(y);
        const u32x4_t bh = sp[buf][k][0][lane], bm = sp[buf][k][1][lane], bl = sp[buf][k][2][lane];
        t = mfma32(p.p[2], bh, t);
        t = mfma32(p.p[1], bm, t);
        t = mfma32(p.p[0], bl, t);
        t = mfma32(p.p[1], bh, t);
        t = mfma32(p.p[0], bm, t);
        t = mfma32(p.p[0], bh, t);
      }
      float *us = seg_block(ws, slot0 + s, h, heads, dv).state + col;
#pragma unroll
      for (int r = 0; r < 16; ++r) us[int64_t(row0 + (r & 3) + 8 * (r >> 2)) * dv] = t[r];
      publish(t, buf ^ 1);
    }
}

template <bool kContig>
int launch_walk(const GdnArgs &a, int token_num, int batch, hipStream_t st) {
  // Four columns a lane fill the chip from 2048 wavefronts on; below that one
  // a lane, whose steps are shorter chains.
  const int64_t wide = int64_t(batch) * a.heads * (a.dv / 16);
  const bool narrow = wide < 2048;
  const int64_t groups = narrow ? wide * 4 : wide;
  if (groups > 0x7fffffff) return WY_E_SHAPE;
  if (narrow)
    gdn_walk_kernel<kContig, 1><<<unsigned(groups), 64, 0, st>>>(a, token_num, batch);
  else
    gdn_walk_kernel<kContig, 4><<<unsigned(groups), 64, 0, st>>>(a, token_num, batch);
  return wyh::launch_status();
}

template <bool kContig>
int launch_scan(const GdnArgs &a, int token_num, int batch, float *ws, int slots, int seg_len,
                hipStream_t st) {
  const int vblocks = a.dv / 128;
  const int64_t main = int64_t(batch + slots) * a.heads * vblocks;
  const int64_t pre = int64_t(slots) * a.heads * (vblocks + 1);
  const int64_t fold = int64_t(batch) * a.heads * (a.dv / kWCols);
  if (main > 0x7fffffff || pre > 0x7fffffff || fold > 0x7fffffff) return WY_E_SHAPE;
  // the attribute is per function: set once (function-local statics are
  // initialised exactly once, also under concurrent first calls)
  static const hipError_t rc0 = hipFuncSetAttribute(
      reinterpret_cast<const void *>(&gdn_scan_kernel<kContig, false>),
      hipFuncAttributeMaxDynamicSharedMemorySize, int(sizeof(ScanLds)));
  static const hipError_t rc1 = hipFuncSetAttribute(
      reinterpret_cast<const void *>(&gdn_scan_kernel<kContig, true>),
      hipFuncAttributeMaxDynamicSharedMemorySize, int(sizeof(ScanLds)));
  if (rc0 != hipSuccess) return int(rc0);
  if (rc1 != hipSuccess) return int(rc1);
  if (slots > 0) {
    gdn_scan_kernel<kContig, true>
        <<<unsigned(pre), 256, sizeof(ScanLds), st>>>(a, token_num, batch, ws, slots, seg_len);
    gdn_fold_kernel<<<unsigned(fold), 256, 0, st>>>(a.cu_seqlens, token_num, a.heads, a.dv, ws,
                                                    slots, seg_len);
  }
  gdn_scan_kernel<kContig, false>
      <<<unsigned(main), 256, sizeof(ScanLds), st>>>(a, token_num, batch, ws, slots, seg_len);
  return wyh::launch_status();
}

// Segments of a batch that are not their sequence's last: at most one per
// whole kSeg tokens.
int64_t slot_bound(int64_t token_num) { return token_num > kSeg ? token_num / kSeg : 0; }

// Segment length of one prompt alone: the two walks grow with it, the fold with
// their number.  us by segment length 64 / 128 / 192 / 256 / 384 / 512 (16
// heads; before them the chunk ops of csrc/gdn_chunk.hip): 257 tokens 44: 43 /
// 50 / 59 / 75 / 49 / 49; 512 53: 56 / 56 / 68 / 79 / 107 / 80; 1000 70: 90 /
// 75 / 82 / 90 / 117 / 145; 2048 115: 170 / 115 / 112 / 110 / 133 / 156; 3000
// 168: 245 / 165 / 134 / 137 / 143 / 165; 5003 274: 403 / 269 / 213 / 208 / 182
// / 205; 8192 474: 675 / 405 / 337 / 275 / 269 / 237.
int prompt_segment(int token_num) {
  if (token_num <= 192) return 192;   // 130 tokens: 30 in one piece, 34 in three
  const int len = (token_num / 16 + 64 + kG / 2) / kG * kG;
  return len < kSeg ? len : kSeg;
}
int64_t prompt_slots(int token_num) {
  return token_num > 0 ? (token_num - 1) / prompt_segment(token_num) : 0;
}
int64_t slots_bytes(int64_t slots, int heads, int dv) {
  return slots * heads * kDK * (int64_t(dv) + kDK) * 4;
}

}  // namespace

extern "C" int64_t wy_gdn_prefill_varlen_workspace_bytes(int token_num, int num_heads,
                                                         int value_dim) {
  if (token_num <= 0 || num_heads <= 0 || value_dim <= 0) return 0;
  return slots_bytes(slot_bound(token_num), num_heads, value_dim);
}

extern "C" int64_t wy_gdn_prefill_prompt_workspace_bytes(int token_num, int num_heads,
                                                         int value_dim) {
  if (token_num <= 0 || num_heads <= 0 || value_dim <= 0) return 0;
  return slots_bytes(prompt_slots(token_num), num_heads, value_dim);
}

// slots: segments that the workspace holds (0: none are cut)
static int run_prefill(GdnArgs &a, bool contig, int token_num, int max_seqlen, int batch,
                       float *workspace, int64_t workspace_bytes, int64_t slots, int seg_len,
                       hipStream_t st) {
  const int bound = max_seqlen > 0 ? max_seqlen : token_num;   // 0: unknown
  if (bound > 0 && bound <= kWalk && batch <= kWalkBatch)
    return contig ? launch_walk<true>(a, token_num, batch, st)
                  : launch_walk<false>(a, token_num, batch, st);
  if (slots > 0x7fffffff / 2) return WY_E_SHAPE;
  if (slots > 0 && workspace_bytes < slots_bytes(slots, a.heads, a.dv)) return WY_E_CAPACITY;
  if (slots > 0 && !wyh::aligned16(workspace)) return WY_E_LAYOUT;
  // the buffer-resource form: rows at least as long as what is read of them,
  // and a group of them within 31 bits of bytes
  const auto row_ok = [](int64_t t, int64_t width) { return t >= width && t < (1 << 22); };
  contig = contig && row_ok(a.q_t, kDK) && row_ok(a.k_t, kDK) && row_ok(a.v_t, a.dv) &&
           row_ok(a.o_t, a.dv) && row_ok(a.s_k, a.dv) && row_ok(a.g_t, 1) && row_ok(a.beta_t, 1);
  return contig ? launch_scan<true>(a, token_num, batch, workspace, int(slots), seg_len, st)
                : launch_scan<false>(a, token_num, batch, workspace, int(slots), seg_len, st);
}

extern "C" int wy_gdn_prefill_varlen_max(
    const void *q, const int64_t *q_strides, const void *k, const int64_t *k_strides,
    const void *v, const int64_t *v_strides, const float *beta, const int64_t *beta_strides,
    const float *g, const int64_t *g_strides, void *out, const int64_t *out_strides,
    float *state, const int64_t *state_strides, const int32_t *cu_seqlens, int token_num,
    int max_seqlen, int batch, int num_heads, int key_dim, int value_dim, float *workspace,
    int64_t workspace_bytes, void *stream) {
  GdnArgs a;
  bool contig = false;
  const int rc = gdn_setup(a, contig, q, q_strides, k, k_strides, v, v_strides, beta,
                           beta_strides, g, g_strides, out, out_strides, state, state_strides,
                           num_heads, key_dim, value_dim);
  if (rc != WY_OK) return rc;
  if (!cu_seqlens && batch != 1) return WY_E_NULL;
  if (batch < 0 || token_num < 0 || max_seqlen < 0) return WY_E_SHAPE;
  if (batch == 0) return WY_OK;
  a.cu_seqlens = cu_seqlens;
  return run_prefill(a, contig, token_num, max_seqlen, batch, workspace, workspace_bytes,
                     workspace ? slot_bound(token_num) : 0, kSeg,
                     static_cast<hipStream_t>(stream));
}

extern "C" int wy_gdn_prefill_prompt(const void *q, const int64_t *q_strides, const void *k,
                                     const int64_t *k_strides, const void *v,
                                     const int64_t *v_strides, const float *beta,
                                     const int64_t *beta_strides, const float *g,
                                     const int64_t *g_strides, void *out,
                                     const int64_t *out_strides, float *state,
                                     const int64_t *state_strides, int token_num, int num_heads,
                                     int key_dim, int value_dim, float *workspace,
                                     int64_t workspace_bytes, void *stream) {
  GdnArgs a;
  bool contig = false;
  const int rc = gdn_setup(a, contig, q, q_strides, k, k_strides, v, v_strides, beta,
                           beta_strides, g, g_strides, out, out_strides, state, state_strides,
                           num_heads, key_dim, value_dim);
  if (rc != WY_OK) return rc;
  if (token_num <= 0) return WY_E_SHAPE;
  return run_prefill(a, contig, token_num, token_num, 1, workspace, workspace_bytes,
                     workspace ? prompt_slots(token_num) : 0, prompt_segment(token_num),
                     static_cast<hipStream_t>(stream));
}

extern "C" int wy_gdn_prefill_varlen(const void *q, const int64_t *q_strides, const void *k,
                                     const int64_t *k_strides, const void *v,
                                     const int64_t *v_strides, const float *beta,
                                     const int64_t *beta_strides, const float *g,
                                     const int64_t *g_strides, void *out,
                                     const int64_t *out_strides, float *state,
                                     const int64_t *state_strides, const int32_t *cu_seqlens,
                                     int token_num, int batch, int num_heads, int key_dim,
                                     int value_dim, float *workspace, int64_t workspace_bytes,
                                     void *stream) {
  return wy_gdn_prefill_varlen_max(q, q_strides, k, k_strides, v, v_strides, beta, beta_strides,
                                   g, g_strides, out, out_strides, state, state_strides,
                                   cu_seqlens, token_num, 0, batch, num_heads, key_dim, value_dim,
                                   workspace, workspace_bytes, stream);
}

extern "C" int wy_gdn_recurrent_prefill_sequential(
    const void *q, const int64_t *q_strides, const void *k, const int64_t *k_strides,
    const void *v, const int64_t *v_strides, const float *beta, const int64_t *beta_strides,
    const float *g, const int64_t *g_strides, void *out, const int64_t *out_strides,
    float *state, const int64_t *state_strides, const int32_t *cu_seqlens, int batch,
    int num_heads, int key_dim, int value_dim, void *stream) {
  if (!cu_seqlens) return WY_E_NULL;
  return wy_gdn_prefill_varlen(q, q_strides, k, k_strides, v, v_strides, beta, beta_strides, g,
                               g_strides, out, out_strides, state, state_strides, cu_seqlens, 0,
                               batch, num_heads, key_dim, value_dim, nullptr, 0, stream);
}
