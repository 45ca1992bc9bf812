// Per-head RMS norm + NeoX partial rotary embedding of Q and K, fused with the
// KV-cache append of the rotated K and the raw V rows.
//
// Bound: memory (36 KiB read and 18 KiB written per token) for many tokens, the
// chain of one wave for few.  A wave64 VALU instruction takes four clocks, so
// four sincosf per lane and head cost more than the bytes did: a wave takes
// one head and computes each angle once, in one lane.  K goes by 16 rows of a
// cache block (one row half of the layout), through LDS, and leaves as whole
// 1 KiB wave stores; V is gathered by column so that a store holds the eight
// rows of a V block.  Row by row, K left in 8-byte and V in 2-byte pieces of
// lines that other CUs also wrote.  Measured per call against four sincosf and
// row-wise stores: 4096 tokens 62.6 -> 36.4 us (6.2 TB/s), 1900 tokens 27.1 ->
// 18.5, 333 tokens 7.4 -> 4.9 (by row), 12 tokens 3.6 -> 2.7.  Two, four or eight heads
// to a wave (more loads in flight, fewer sincosf): 1900 tokens 18.4, 19.1 and
// 21.1 us, 12 tokens 2.9, 3.3 and 4.4.
//
// Reference semantics: q_head_norm_rope / k_head_norm_rope
// (src/math_util.rs:501-593; Metal kernels src/engine/shaders.metal:2244-2363)
// followed by kv_cache_append (math_util.rs:387-392).  K is rotated from its
// un-rotated normed values (the CPU form's `orig` copy, math_util.rs:566).
#include <algorithm>
#include <cmath>

#include "common.h"

extern "C" __device__ float __ockl_wfred_add_f32(float);

namespace {

constexpr int kMaxRotHalf = MI_ROPE_MAX_DIM / 2;

struct RopeArgs {
  const float* q_proj;    // [n][H][2*D]
  const float* k;         // [n][G][D]
  const float* v;         // [n][G][D]
  const uint16_t* q_w;    // bf16 [D]
  const uint16_t* k_w;    // bf16 [D]
  _Float16* q_out;        // [n][H][D]
  _Float16* gate_out;     // [n][H][D]
  _Float16* kc;           // cache K blocks of the layer
  _Float16* vc;           // cache V blocks of the layer
  int64_t pos;            // row of token 0
  int n, H, G, rot_half;
  int nk, nkv;            // workgroups of K, of K and V
  float eps;
  // rope_theta^(-2i/rotary_dim), computed on the host in f32 with the
  // reference's expression so that theta = pos * inv_freq rounds identically.
  float inv_freq[kMaxRotHalf];
};

// K staging: the block layout of one (block, head, row half), each column
// chunk's 16 row slots padded by 16 bytes so that a wave's 8-byte writes
// (lanes two to a chunk) spread over the banks.
constexpr int kChunkPitch = 16 * 8 + 8;  // halves
constexpr int kStageHalves = 32 * kChunkPitch;

// K rows (tokens times KV heads) from which K goes through LDS by block; fewer go
// row by row, a wave each, which has the shorter chain: by block takes 1.24 of the
// time for 195 tokens of two heads, 1.13 for 321, 0.99 for 457, 0.93 for 796; one
// head 1.22 for 434, 0.99 for 957; 4 heads 1.11 for 139, 0.96 for 232; 8 heads 1.15 for
// 73, 0.97 for 116 (rotary_dim 64; 128 to 256 cross 10 to 40 % later).
constexpr int kKRows = 900;

// RMS norm of one head, lane l holding columns 4l .. 4l+3.
__device__ __forceinline__ void head_norm(const float4& x, const ushort4& wb, float eps,
                                          float (&y)[4]) {
  const float ss = __ockl_wfred_add_f32(x.x * x.x + x.y * x.y + x.z * x.z + x.w * x.w);
  const float inv_rms = 1.0f / sqrtf(ss / (float)mi::kHeadDim + eps);
  y[0] = x.x * inv_rms * mi::bf16_to_f32(wb.x);
  y[1] = x.y * inv_rms * mi::bf16_to_f32(wb.y);
  y[2] = x.z * inv_rms * mi::bf16_to_f32(wb.z);
  y[3] = x.w * inv_rms * mi::bf16_to_f32(wb.w);
}

// NeoX rotation of a normed head; c, s: the lane's four angles (pairs
// 4l mod rot_half ..), read only where 4l < 2 rot_half.
__device__ __forceinline__ f16x4 head_rotate(float (&y)[4], const float (&c)[4],
                                             const float (&s)[4], int lane, int rh) {
  const bool lower = 4 * lane < rh;
  const int partner = lower ? lane + (rh >> 2) : lane - (rh >> 2);
  float pr[4];
#pragma unroll
  for (int e = 0; e < 4; e++) pr[e] = __shfl(y[e], partner & 63, 64);
  if (4 * lane < 2 * rh) {
#pragma unroll
    for (int e = 0; e < 4; e++)
      y[e] = lower ? y[e] * c[e] - pr[e] * s[e] : pr[e] * s[e] + y[e] * c[e];
  }
  f16x4 h;
#pragma unroll
  for (int e = 0; e < 4; e++) h[e] = (_Float16)y[e];
  return h;
}

// The lane's four angles of token tok's rotation, computed one (BIG: two) per
// lane and fetched from the lanes that hold them.
template <bool BIG>
__device__ __forceinline__ void lane_angles(const RopeArgs& a, int tok, int lane, float (&c)[4],
                                            float (&s)[4]) {
  const int rh = a.rot_half;
  const float fpos = (float)(a.pos + tok);
  float ct[BIG ? 2 : 1] = {}, st[BIG ? 2 : 1] = {};
#pragma unroll
  for (int k = 0; k < (BIG ? 2 : 1); k++)
    if (lane + 64 * k < rh) sincosf(fpos * a.inv_freq[lane + 64 * k], &st[k], &ct[k]);
  const int p0 = 4 * lane < rh ? 4 * lane : 4 * lane - rh;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    c[e] = __shfl(ct[0], (p0 + e) & 63, 64);
    s[e] = __shfl(st[0], (p0 + e) & 63, 64);
    if constexpr (BIG) {
      const float c1 = __shfl(ct[1], (p0 + e) & 63, 64), s1 = __shfl(st[1], (p0 + e) & 63, 64);
      if (p0 + e >= 64) {
        c[e] = c1;
        s[e] = s1;
      }
    }
  }
}

// One K row by one wave, stored in place (a few rows: kKRows).
template <bool BIG>
__device__ __forceinline__ void k_row(const RopeArgs& a, int item) {
  constexpr int D = mi::kHeadDim;
  const int lane = threadIdx.x & 63;
  const int tok = item / a.G, h = item - tok * a.G;
  if (tok >= a.n) return;
  const float4 x = *(const float4*)(a.k + (int64_t)item * D + 4 * lane);
  const ushort4 wb = *(const ushort4*)(a.k_w + 4 * lane);
  float y[4], c[4], s[4];
  lane_angles<BIG>(a, tok, lane, c, s);
  head_norm(x, wb, a.eps, y);
  *(f16x4*)(a.kc + mi::k_offset(a.pos + tok, h, 4 * lane, a.G, D)) =
      head_rotate(y, c, s, lane, a.rot_half);
}

// K rows of one (32-row block, KV head, row half u): 16 rows, four per wave,
// whose slots are 8 KiB of contiguous block layout.  `lds`: the stage, then
// the angles [16][rot_half] (cos, sin).  Loads are unconditional (rows outside
// [pos, pos + n) read a row inside it and are not stored), so that all are in
// flight before the first is waited for.
__device__ __forceinline__ void k_rows(const RopeArgs& a, int item, float* lds) {
  constexpr int D = mi::kHeadDim;
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int u = item & 1, bh = item >> 1;
  const int bb = bh / a.G, h = bh - bb * a.G;
  const int64_t b = a.pos / MI_KV_KBLOCK + bb;
  const int64_t row0 = b * MI_KV_KBLOCK - a.pos + 8 * w + 4 * u;  // token of the wave's first row
  const int rh = a.rot_half;
  _Float16* const stage = (_Float16*)lds;
  float2* const tab = (float2*)(lds + kStageHalves / 2) + 4 * w * rh;

  float4 x[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int64_t tok = min(max(row0 + i, (int64_t)0), (int64_t)a.n - 1);
    x[i] = *(const float4*)(a.k + (tok * a.G + h) * D + 4 * lane);
  }
  const ushort4 wb = *(const ushort4*)(a.k_w + 4 * lane);
  // the angles of the wave's new rows [i0, i1), spread over its lanes
  const int i0 = (int)min(max(-row0, (int64_t)0), (int64_t)4);
  const int i1 = (int)min(max((int64_t)a.n - row0, (int64_t)0), (int64_t)4);
  for (int idx = i0 * rh + lane; idx < i1 * rh; idx += 64) {
    const int i = (idx >= rh) + (idx >= 2 * rh) + (idx >= 3 * rh), p = idx - i * rh;
    float sn, cs;
    sincosf((float)(a.pos + row0 + i) * a.inv_freq[p], &sn, &cs);
    tab[idx] = float2{cs, sn};
  }
  // the wave's lanes read each other's entries below: LDS serves a wave in
  // order, this keeps the compiler to it
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const bool rot = 4 * lane < 2 * rh;
  const int p0 = 4 * lane < rh ? 4 * lane : 4 * lane - rh;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    float y[4], c[4], s[4];
    head_norm(x[i], wb, a.eps, y);
#pragma unroll
    for (int e = 0; e < 4; e++) {  // this wave's own table rows
      const float2 cs = rot ? tab[i * rh + p0 + e] : float2{};
      c[e] = cs.x;
      s[e] = cs.y;
    }
    *(f16x4*)(stage + (lane >> 1) * kChunkPitch + (4 * w + i) * 8 + 4 * (lane & 1)) =
        head_rotate(y, c, s, lane, rh);
  }
  __syncthreads();
  _Float16* kd = a.kc + ((b * a.G + h) * 2 + u) * (int64_t)(16 * D);
#pragma unroll
  for (int i = 0; i < 2; i++) {  // slot (chunk, j), j fastest
    const int sl = 256 * i + t, j = sl & 15;
    const int64_t tk = b * MI_KV_KBLOCK - a.pos + (((j >> 2) << 3) | (u << 2) | (j & 3));
    if (tk >= 0 && tk < a.n)
      *(f16x8*)(kd + sl * 8) = *(const f16x8*)(stage + (sl >> 4) * kChunkPitch + j * 8);
  }
}

// V rows of one (8-row block, KV head): thread t gathers column t.
__device__ __forceinline__ void v_rows(const RopeArgs& a, int item) {
  constexpr int D = mi::kHeadDim;
  const int t = threadIdx.x;
  const int bb = item / a.G, h = item - bb * a.G;
  const int64_t b = a.pos / MI_KV_VBLOCK + bb;
  const int64_t row0 = b * MI_KV_VBLOCK - a.pos;  // token of the block's first row
  float x[8];
#pragma unroll
  for (int e = 0; e < 8; e++) {
    const int64_t tok = min(max(row0 + e, (int64_t)0), (int64_t)a.n - 1);
    x[e] = a.v[(tok * a.G + h) * D + t];
  }
  _Float16* vd = a.vc + (b * a.G + h) * (int64_t)(D * MI_KV_VBLOCK) + t * 8;
  f16x8 col;
#pragma unroll
  for (int e = 0; e < 8; e++) col[e] = (_Float16)x[e];
  if (row0 >= 0 && row0 + 8 <= a.n) {
    *(f16x8*)vd = col;
  } else {  // rows outside the range keep their contents
#pragma unroll
    for (int e = 0; e < 8; e++)
      if (row0 + e >= 0 && row0 + e < a.n) vd[e] = col[e];
  }
}

// Workgroups [0, nk): K, [nk, nkv): V blocks; then one query head of one token
// per wave.  BIG: rot_half above 64, two angles a lane.
template <bool BIG>
__global__ void __launch_bounds__(256) qk_norm_rope_kernel(const RopeArgs a) {
  constexpr int D = mi::kHeadDim;
  extern __shared__ float lds[];
  const int wave = threadIdx.x >> 6;
  const int wg = blockIdx.y * gridDim.x + blockIdx.x;
  if (wg < a.nkv) {
    if (wg >= a.nk) v_rows(a, wg - a.nk);
    else if (a.n * a.G < kKRows) k_row<BIG>(a, wg * 4 + wave);
    else k_rows(a, wg, lds);
    return;
  }
  const int lane = threadIdx.x & 63;
  const int64_t head = (int64_t)(wg - a.nkv) * 4 + wave;  // tok * H + head
  const int tok = (int)(head / a.H);
  if (tok >= a.n) return;  // whole waves
  const float* src = a.q_proj + head * (2 * D) + 4 * lane;
  const float4 x = *(const float4*)src;
  const float4 g = *(const float4*)(src + D);
  const ushort4 wb = *(const ushort4*)(a.q_w + 4 * lane);
  float y[4], c[4], s[4];
  lane_angles<BIG>(a, tok, lane, c, s);
  head_norm(x, wb, a.eps, y);
  const int64_t o = head * D + 4 * lane;
  *(f16x4*)(a.q_out + o) = head_rotate(y, c, s, lane, a.rot_half);
  *(f16x4*)(a.gate_out + o) =
      f16x4{(_Float16)g.x, (_Float16)g.y, (_Float16)g.z, (_Float16)g.w};
}

}  // namespace

namespace mi {

mi_status check_rope(const mi_kv* kv, int32_t rotary_dim, float rope_theta, float eps) {
  if (rotary_dim < 0 || rotary_dim % 8 || rotary_dim > kv->D || rotary_dim > MI_ROPE_MAX_DIM)
    return fail(MI_ERR_INVALID_ARG, "rotary_dim=%d (multiple of 8, at most %d)", rotary_dim,
                std::min(kv->D, MI_ROPE_MAX_DIM));
  if (!(eps >= 0.f) || !(rope_theta > 0.f))
    return fail(MI_ERR_INVALID_ARG, "eps=%g rope_theta=%g", (double)eps, (double)rope_theta);
  return MI_OK;
}

// A model has one (rope_theta, rotary_dim): the table of the last pair is kept
// per thread, so a decode step does not pay 32 powf calls again (1.3 us).
void rope_inv_freq(float rope_theta, int32_t rotary_dim, float* inv_freq) {
  thread_local float theta = 0.f, table[kMaxRotHalf];
  thread_local int32_t dim = -1;
  const int half = rotary_dim / 2;
  if (theta != rope_theta || dim != rotary_dim) {
    for (int i = 0; i < half; i++)
      table[i] = powf(rope_theta, -2.0f * (float)i / (float)rotary_dim);
    theta = rope_theta;
    dim = rotary_dim;
  }
  std::copy(table, table + half, inv_freq);
}

}  // namespace mi

extern "C" mi_status mi_qk_norm_rope_append(mi_kv* kv, int32_t layer, const float* q_proj,
                                            const float* k, const float* v,
                                            const uint16_t* q_norm_w, const uint16_t* k_norm_w,
                                            int32_t rotary_dim, float rope_theta, float eps,
                                            int64_t pos, int32_t n, mi_f16* q_out,
                                            mi_f16* gate_out, mi_stream stream) {
  mi::clear_error();
  MI_TRY(mi::check_layer(kv, layer));
  if (!q_proj || !k || !v || !q_norm_w || !k_norm_w || !q_out || !gate_out)
    return mi::fail(MI_ERR_INVALID_ARG, "null pointer");
  if (n <= 0) return mi::fail(MI_ERR_INVALID_ARG, "n=%d", n);
  if (pos < 0) return mi::fail(MI_ERR_OUT_OF_RANGE, "pos=%lld", (long long)pos);
  MI_TRY(mi::check_rope(kv, rotary_dim, rope_theta, eps));
  MI_TRY(mi::kv_grow(kv, pos + n, (hipStream_t)stream));

  RopeArgs a{};
  a.q_proj = q_proj;
  a.k = k;
  a.v = v;
  a.q_w = q_norm_w;
  a.k_w = k_norm_w;
  a.q_out = (_Float16*)q_out;
  a.gate_out = (_Float16*)gate_out;
  a.kc = kv->k[layer];
  a.vc = kv->v[layer];
  a.pos = pos;
  a.n = n;
  a.H = kv->H;
  a.G = kv->G;
  a.rot_half = rotary_dim / 2;
  a.eps = eps;
  mi::rope_inv_freq(rope_theta, rotary_dim, a.inv_freq);

  const int64_t last = pos + n - 1;
  const bool by_row = (int64_t)n * kv->G < kKRows;
  a.nk = by_row ? (n * kv->G + 3) / 4
                : (int)(2 * (last / MI_KV_KBLOCK - pos / MI_KV_KBLOCK + 1) * kv->G);
  a.nkv = a.nk + (int)((last / MI_KV_VBLOCK - pos / MI_KV_VBLOCK + 1) * kv->G);
  const int64_t wgs = a.nkv + ((int64_t)n * kv->H + 3) / 4;
  const int64_t gx = std::min<int64_t>(wgs, 1 << 22);  // a grid row is below 2^32 threads
  const size_t lds = by_row ? 0 : kStageHalves * sizeof(_Float16) + 16 * a.rot_half * sizeof(float2);
  MI_HIP(mi::launch("qk_norm_rope",
                    a.rot_half > 64 ? qk_norm_rope_kernel<true> : qk_norm_rope_kernel<false>,
                    dim3((unsigned)gx, (unsigned)((wgs + gx - 1) / gx)), dim3(256), lds,
                    (hipStream_t)stream, a));
  kv->len[layer] = pos + n;
  return MI_OK;
}
