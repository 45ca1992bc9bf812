// Split-K flash-decoding over the f16 KV cache, for one query token (decode),
// a few query tokens with a causal tail (speculative verify), or a ragged
// batch of independent sequences.
//
// Reference semantics: attention_scores/softmax/values_batched and
// sigmoid_gate_inplace (src/math_util.rs:264-269, 323-383); the split-K
// kernels attn_sdpa_block / attn_sdpa_reduce (src/engine/shaders.metal:
// 1559-1776) dispatched by encode_pre_expert_full (src/engine/qwen35_moe/
// fused_exp2.rs:683-719); the causal bound of attn_sdpa_causal_n
// (shaders.metal:2675-2676: query i sees rows [0, past_pos + i]).
//
// Design (gfx950, wave64):
//  * One workgroup = one (sequence, KV head, chunk of keys).  The eight query
//    heads of the GQA group — times the query tokens for verify — are the
//    columns of one MFMA tile, so each K/V byte is read from HBM once per
//    group rather than once per query head.
//  * S^T = K . Q^T with v_mfma_f32_16x16x32_f16: K rows are the A operand,
//    loaded straight from HBM as 128-bit vectors (each lane streams 128
//    contiguous bytes of one key row); Q^T stays in registers.
//  * O^T += V^T . P^T with the same instruction: the V cache is stored in
//    8-row transposed blocks, so the A operand (eight keys of one value
//    column) is one 128-bit load, and the P^T operand is the S^T
//    accumulator of the same lane (the QK row order is chosen so that it
//    is) — no LDS transpose, no shuffles of P.
//  * Online softmax in base 2 per column; the column max / sum reductions
//    are two cross-lane xor steps (lanes 16 and 32 apart).
//  * The waves of a workgroup merge their (m, l, O) through LDS and write one
//    partial per chunk; attn_combine_kernel merges the chunks, normalises,
//    applies the sigmoid gate and writes f16.
#include <algorithm>
#include <cstdlib>
#include <initializer_list>
#include <type_traits>

#include "common.h"
#include "plan.h"

namespace {

constexpr int D = mi::kHeadDim;
constexpr float kNegBig = -1e30f;

// Most sequences of a ragged batch whose tile offsets the flat split
// computes itself (no plan launch); larger batches run ragged_plan_kernel.
constexpr int kFusedPlan = 256;

// Ragged batches of more tiles than workgroups, up to kChunkTiles per spare
// workgroup (grid minus sequences), are dealt out by chunks of one sequence,
// ceil(tiles / spare) tiles each, so that no workgroup crosses into a second
// sequence: a crossing runs the whole chain (Q, K, V, merge, store) twice, and
// with a tile or two per wave that chain is the launch.  Per call (us, against
// tiles dealt evenly across sequences): 8 sequences of 100..3000 rows 25.7 ->
// 15.5, 2 of 3000 32.5 -> 15.7, 32 of 500..2000 26.4 -> 24.5, 100 of 50..200 24.7
// -> 18.1.  Up to one tile per workgroup nothing crosses, and the second scan
// that the chunks need would cost 0.6 us (16 of 1..60 rows 12.0 -> 12.9).
constexpr int kChunkTiles = 16;

struct SplitArgs {
  const _Float16* k;        // K 32-row blocks (mi::k_offset)
  const _Float16* v;        // V blocks, (r,h,i) at v + ((r/8)*G + h)*D*8 + i*8 + r%8
  const int32_t* offsets;   // ragged: first row of sequence s (else null)
  const int32_t* lengths;   // ragged: rows of sequence s (else null)
  int64_t kv_len;           // non-ragged: rows the launch may read
  int64_t lim0;             // non-ragged: rows visible to query token 0
  const _Float16* q;        // [batch][nq][H][D]
  float* part_o;            // [G][nslots][ncols][D], slot = s * max_chunks + chunk
  float* part_ml;           // [G][nslots][ncols][2]  (flat ragged: slot = workgroup + s)
  int64_t nslots;
  int G, H, nq, chunk, max_chunks;
  int ntok;                 // groups: query tokens in all
  float scale_log2e;
  // Flat ragged split: tile_off[s] = 32-key tiles of sequences 0..s-1
  // (invalid descriptors count 0), tile_off[batch] = all tiles T; workgroup
  // x < nw = min(gridDim.x, T) takes tiles [x T / nw, (x+1) T / nw) of the
  // concatenation and writes one partial per sequence it touches, in slot
  // x + s.  Null otherwise.
  const int32_t* tile_off;
  // Flat split of up to kFusedPlan sequences: no plan kernel; every
  // workgroup computes the tile offsets into LDS from lengths / offsets, and
  // workgroup (0, 0) also stores them here (= tile_off) for the merge kernel.
  // Null otherwise.  With few tiles (kChunkTiles) the table counts chunks of
  // whole sequences instead, and its last entry is stored as -1 - chunks.
  int32_t* tile_off_out;
  int batch;
  // Optional fused append (decode step, verify): rows [app0, app0 + app_n)
  // of the cache are written from app_k / app_v ([app_n][G*D] token-major)
  // by the workgroup whose key chunk holds them, before it reads them.
  const _Float16* app_k;
  const _Float16* app_v;
  _Float16* kw;
  _Float16* vw;
  int64_t app0;
  int app_n;
  // In-launch merge (single sequence, one query token, one KV head per
  // workgroup): partials m / l at part_ml with a 256-byte stride per slot,
  // then merged inside the launch (merge_tail) and written to out with the
  // gate, instead of by attn_combine_kernel.  Null mcnt: off.
  int* mcnt;          // counters: XCD-local [G][8], then per KV head [G] (256 B apart)
  float* xo;          // per-XCD partials [G][8][8][D]
  float* xml;         // per-XCD (m, l) [G][8][64]
  const _Float16* gate;
  const float* gate32;
  _Float16* out;
};

// Partials are consumed once, by the combine kernel, on any XCD: written
// through to memory (sc0 sc1), so that the end of the split launch has no
// dirty partial lines to write back from the L2s.  Measured at C2 against
// streaming (nontemporal) and default stores, in one process: 19.87-19.91
// against 20.12-20.15 us per step.
__device__ __forceinline__ void store_part(float v, float* p) {
  asm volatile("global_store_dword %0, %1, off sc0 sc1" ::"v"(p), "v"(v) : "memory");
}
// A store of more than 64 bits reads its data registers after issue: the
// next instruction may not overwrite them without wait states, which the
// compiler inserts for its own stores but not for asm ones, hence the nops.
__device__ __forceinline__ void store_part(f32x4 v, f32x4* p) {
  asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1\n s_nop 1" ::"v"(p), "v"(v) : "memory");
}

// 16-byte streaming load of K/V: read once per launch, so it is not kept in
// the caches (MI_ATTN_TEMPORAL_KV=1 at build time keeps the default policy).
__device__ __forceinline__ f16x8 load16(const _Float16* p) {
#if defined(MI_ATTN_TEMPORAL_KV)
  return *(const f16x8*)p;
#else
  return __builtin_nontemporal_load((const f16x8*)p);
#endif
}

// Fused projection input of the decode step (mi_attn_step_proj): the raw
// q_proj / k / v of one token in f32, normed and rotated inside the split
// kernel.  cos / sin of the rotation angles pos * inv_freq[i] are computed on
// the host (the position is a host value), in f32 like the reference:
// cs[i] = cos, cs[rot_half + i] = sin, i < rot_half.
struct ProjInput {
  const float* q_proj;  // [H][2*D]: query then gate of each head
  const float* k;       // [G][D]
  const float* v;       // [G][D]
  const uint16_t* q_w;  // bf16 [D]
  const uint16_t* k_w;  // bf16 [D]
  float eps;
};
struct ProjArgs : ProjInput {
  int rot_half;  // host side: selects the Proj<rot_half / 32> kernel
  float cs[MI_ROPE_MAX_DIM];
};
struct NoProj {
  static constexpr int kSH = 0;
};
// The kernel argument, with the rotation width as a compile-time constant:
// rot_half = 32 * SH, SH = 0 .. 4.  It holds the 64 SH cos / sin values in
// use only: launch arguments are copied by the host at every call.
template <int SH>
struct Proj : ProjInput {
  static constexpr int kSH = SH;
  float cs[SH > 0 ? 64 * SH : 1];
};
template <class X>
struct is_proj : std::false_type {};
template <int SH>
struct is_proj<Proj<SH>> : std::true_type {};

// A lane's cos / sin of the rotation, for head columns DPT*i .. DPT*i + DPT-1
// (i = lane % TPH): read from the kernel arguments at the lane's own place.
// Against the table in scalar registers spread over the wave by selects and
// fetched by cross-lane permutes, a step from projections went from 9.2 to 8.2 us
// at 517 rows and from 23.6 to 22.5 at 32000.
template <int DPT, int SH>
struct RopeLane {
  float c[DPT], s[DPT];
  __device__ __forceinline__ void load(const Proj<SH>& x, int lane) {
    if constexpr (SH > 0) {
      constexpr int RH = 32 * SH;
      const int d0 = DPT * (lane % (D / DPT));
      const int p0 = d0 < RH ? d0 : d0 < 2 * RH ? d0 - RH : 0;
#pragma unroll
      for (int e = 0; e < DPT; e++) {
        c[e] = x.cs[p0 + e];
        s[e] = x.cs[RH + p0 + e];
      }
    }
  }
};

// Per-head RMS norm + NeoX rotation, one head per TPH = 256 / DPT adjacent
// lanes (aligned within the wave): lane index i = lane % TPH holds columns
// DPT*i .. DPT*i + DPT-1 of the head.  The rotation partner of column
// d < rot_half, d + rot_half, sits rot_half / DPT lanes up.  Split into the
// loads (issued early, ahead of the first K/V tile, so that waiting for
// them does not wait for the tile) and the arithmetic.
template <int DPT>
struct HeadPart {
  float y[DPT];
  uint32_t wb[DPT / 2];  // bf16 pairs
  __device__ __forceinline__ void load(const float* src, const uint16_t* w, int lane) {
    const int i = lane % (D / DPT);
#pragma unroll
    for (int e = 0; e < DPT; e += 4) {
      const float4 f = *(const float4*)(src + DPT * i + e);
      y[e] = f.x;
      y[e + 1] = f.y;
      y[e + 2] = f.z;
      y[e + 3] = f.w;
      const uint2 u = *(const uint2*)(w + DPT * i + e);
      wb[e / 2] = u.x;
      wb[e / 2 + 1] = u.y;
    }
  }
  template <int SH>
  __device__ __forceinline__ void norm_rope(const ProjInput& x, const RopeLane<DPT, SH>& rl,
                                            int lane) {
    constexpr int TPH = D / DPT;
    const int i = lane % TPH;
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < DPT; e++) ss += y[e] * y[e];
#pragma unroll
    for (int m = 1; m < TPH; m <<= 1) ss += __shfl_xor(ss, m, 64);
    const float inv_rms = 1.0f / sqrtf(ss / (float)D + x.eps);
#pragma unroll
    for (int e = 0; e < DPT; e++)
      y[e] = y[e] * inv_rms * mi::bf16_to_f32((uint16_t)(wb[e / 2] >> (16 * (e & 1))));
    if constexpr (SH > 0) {
      constexpr int RH = 32 * SH;
      const int d0 = DPT * i;
      const bool lower = d0 < RH;
      const int partner = lower ? lane + RH / DPT : lane - RH / DPT;
      float pr[DPT];
#pragma unroll
      for (int e = 0; e < DPT; e++) pr[e] = __shfl(y[e], partner & 63, 64);
#pragma unroll
      for (int e = 0; e < DPT; e++)
        if (d0 < 2 * RH)
          y[e] = lower ? y[e] * rl.c[e] - pr[e] * rl.s[e] : pr[e] * rl.s[e] + y[e] * rl.c[e];
    }
  }
};

// ---- in-launch merge of the chunk partials (decode of one sequence, one
// query token, one KV head per workgroup).  Workgroup b of the launch runs on
// XCD b % 8 (round-robin dispatch; checked per device when a handle is
// created, else the merge is not used).  The partials of the chunks of one
// KV head whose workgroups share an XCD are merged by the last of them to
// arrive (an XCD-local counter: stores and atomics meet in that XCD's L2,
// so no cache write-back is needed); it writes one partial per XCD through
// to memory, and the last of those (a device-scope counter) merges the
// eight, normalises, applies the gate and writes the output.  Every counter
// is reset by its last user, so the launch can be replayed in a graph.
// Off by default (decode_merge_enabled): in a probe of the protocol alone it
// added 1.9 us to a launch of 256 workgroups, but after a real C2 split the
// chain takes ~5 us, as long as the combine launch.

// Loads the compiler tracks (it places the waits itself: an asm load whose
// result the compiler copied before a separate wait would copy stale
// data).  Within the XCD a plain load: it misses this CU's L1 (which never
// held those lines in this launch; L1 is invalidated at every kernel start)
// and hits the XCD's L2, where the members' stores landed; the barrier
// before the loads keeps them after the arrival count.  Across XCDs,
// system-scope atomic loads (sc0 sc1: past this XCD's L2, from memory, where
// the data was written through).
__device__ __forceinline__ f32x4 ld_xcd4(const float* p) { return *(const f32x4*)p; }
__device__ __forceinline__ float ld_xcd1(const float* p) { return *p; }
__device__ __forceinline__ float ld_dev1(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ f32x4 ld_dev4(const float* p) {
  return f32x4{ld_dev1(p), ld_dev1(p + 1), ld_dev1(p + 2), ld_dev1(p + 3)};
}
__device__ __forceinline__ void st_dev4(float* p, f32x4 v) {  // written through to memory
  // (the nops: as for store_part, the data registers are read after issue)
  asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1\n s_nop 1" ::"v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ void st_dev1(float* p, float v) {
  asm volatile("global_store_dword %0, %1, off sc0 sc1" ::"v"(p), "v"(v) : "memory");
}
constexpr int kMergeStride = 64;  // ints between counters (256 bytes)

template <int NT>
__device__ void merge_tail(const SplitArgs& a) {
  static_assert(NT == 512, "one f32x4 of the 8 x 256 outputs per thread");
  const int t = threadIdx.x;
  const int hy = blockIdx.y;  // KV head
  const int mc = a.max_chunks;
  const int x = (blockIdx.x + mc * hy) & 7;  // this workgroup's XCD
  const int ngroups = mc < 8 ? mc : 8;
  // chunks c of this head on XCD x: c = first(x) + 8 j
  auto first_of = [&](int xx) { return ((xx - mc * hy) % 8 + 8) % 8; };
  const int first = first_of(x);
  const int nmem = first < mc ? (mc - first + 7) / 8 : 0;
  const int col = t >> 6, d4 = (t & 63) * 4;  // output column (query head) and values
  __shared__ int s_last;

  __builtin_amdgcn_s_waitcnt(0);  // this thread's partial stores have reached L2
  __syncthreads();
  if (t == 0)
    s_last = __hip_atomic_fetch_add(a.mcnt + (hy * 8 + x) * kMergeStride, 1, __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_WORKGROUP) == nmem - 1;
  __syncthreads();
  if (!s_last) return;

  // XCD level: online merge of the members' (m, l, o), 16 at a time
  float M = kNegBig, L = 0.f;
  f32x4 O = {0.f, 0.f, 0.f, 0.f};
  for (int j0 = 0; j0 < nmem; j0 += 16) {
    f32x4 o[16];
    float m[16], l[16];
#pragma unroll
    for (int u = 0; u < 16; u++) {
      const int c = first + 8 * (j0 + u < nmem ? j0 + u : j0);
      const int64_t slot = (int64_t)hy * a.nslots + c;
      o[u] = ld_xcd4(a.part_o + (slot * 8 + col) * D + d4);
      m[u] = ld_xcd1(a.part_ml + slot * 64 + 2 * col);
      l[u] = ld_xcd1(a.part_ml + slot * 64 + 2 * col + 1);
    }
    float mb = M;
#pragma unroll
    for (int u = 0; u < 16; u++)
      if (j0 + u < nmem) mb = fmaxf(mb, m[u]);
    const float r = exp2f(M - mb);
    L *= r;
    O *= r;
#pragma unroll
    for (int u = 0; u < 16; u++)
      if (j0 + u < nmem) {
        const float w = exp2f(m[u] - mb);
        L += l[u] * w;
        O += o[u] * w;
      }
    M = mb;
  }
  st_dev4(a.xo + ((hy * 8 + x) * 8 + col) * D + d4, O);
  if (d4 == 0) {
    st_dev1(a.xml + (hy * 8 + x) * 64 + 2 * col, M);
    st_dev1(a.xml + (hy * 8 + x) * 64 + 2 * col + 1, L);
  }
  __builtin_amdgcn_s_waitcnt(0);  // written through before the arrival is counted
  __syncthreads();
  if (t == 0) {
    __hip_atomic_store(a.mcnt + (hy * 8 + x) * kMergeStride, 0, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_WORKGROUP);
    int* dc = a.mcnt + (a.G * 8 + hy) * kMergeStride;
    const bool last = __hip_atomic_fetch_add(dc, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                      ngroups - 1;
    if (last) __hip_atomic_store(dc, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = last;
  }
  __syncthreads();
  if (!s_last) return;

  // head level: the XCDs that hold chunks of this head
  f32x4 o[8];
  float m[8], l[8];
#pragma unroll
  for (int xx = 0; xx < 8; xx++) {
    o[xx] = ld_dev4(a.xo + ((hy * 8 + xx) * 8 + col) * D + d4);
    m[xx] = ld_dev1(a.xml + (hy * 8 + xx) * 64 + 2 * col);
    l[xx] = ld_dev1(a.xml + (hy * 8 + xx) * 64 + 2 * col + 1);
  }
  float Mh = kNegBig;
#pragma unroll
  for (int xx = 0; xx < 8; xx++)
    if (first_of(xx) < mc) Mh = fmaxf(Mh, m[xx]);
  float Lh = 0.f;
  f32x4 Oh = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int xx = 0; xx < 8; xx++)
    if (first_of(xx) < mc) {
      const float w = exp2f(m[xx] - Mh);
      Lh += l[xx] * w;
      Oh += o[xx] * w;
    }
  // out = O / L (zero when L = 0, math_util.rs:357, 372), then the gate
  const float inv = Lh > 0.f ? 1.f / Lh : 0.f;
  const int hq = hy * 8 + col;
  f16x4 h;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    float r = Oh[e] * inv;
    if (a.gate) r = mi::gate_mul(r, (float)a.gate[hq * D + d4 + e]);
    else if (a.gate32) r = mi::gate_mul(r, a.gate32[hq * (2 * D) + D + d4 + e]);
    h[e] = (_Float16)r;
  }
  *(f16x4*)(a.out + hq * D + d4) = h;
}

// Workgroup = GH KV heads x NWH waves per head, over one chunk of keys of one
// sequence (with GH = 2 a workgroup reads one contiguous stretch of both
// heads' K and V blocks).  NCB column blocks of 16 columns (column c = token
// c / 8, query head c % 8 of the group).
// With X = Proj (decode step from projections, one token, NCB = 1) the
// kernel also norms and rotates Q per wave, and the workgroup holding row
// app0 norms, rotates and appends K and appends V.
// With GROUPS the grid's z counts groups of nq query tokens of one sequence
// (token tok0 = nq z on, the last group perhaps fewer): every group reads the
// whole range, and workgroups of a chunk that holds new rows append the same
// bytes, each before its own reads.  TILE: a tile's weights against the tile's
// own max (see attn_direct_kernel), where a wave has two tiles and the wide
// pass, which also serves these sizes, has one: up to 16384 / G rows.  Without it
// the error against 64 bits of 12 tokens after 6100 rows was 1.7 % above that
// pass's; with it 12 after 9001 rows, where the wide pass is 5 % above, would
// go from 19.5 to 20.0 us.
template <int NWH, int NCB, int GH, typename X, bool FLAT, bool GROUPS = false, bool TILE = false>
__global__ void __launch_bounds__(NWH * GH * 64)
attn_split_kernel(SplitArgs a, X x) {
  constexpr bool kProj = is_proj<X>::value;
  extern __shared__ float smem[];
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
  const int hw = wv / NWH;   // KV head of this wave within the workgroup
  const int w = wv % NWH;    // wave within the head
  const int g = lane >> 4;   // lane group: k-slot group of the MFMA operands
  const int j = lane & 15;   // column within a column block / A-operand row
  const int chunk_idx = blockIdx.x;
  const int kvh = blockIdx.y * GH + hw;
  int s = blockIdx.z;
  const int G = a.G;
  const int ncols = a.nq * 8;

  constexpr bool flat = FLAT;  // the flat ragged split (a.tile_off)
  int64_t len = 0, row0 = 0, lim0 = 0, key_begin = 0, key_end = 0;
  int64_t t_lo = 0, t_hi = 0;  // flat: this workgroup's tiles (chunks) of the concatenation
  int per_seq = 0;             // flat, by chunks of a sequence: tiles per chunk (else 0)
  // flat: the tile offsets, from the plan kernel's table or computed below
  int32_t* const ltoff = (int32_t*)(smem + GH * (NWH * ncols * (D + 4) + 2 * NWH * ncols));
  auto toff = [&](int i) -> int64_t {  // tile_off[i], i wave-uniform in [0, batch]
    return __builtin_amdgcn_readfirstlane(a.tile_off_out ? ltoff[i] : a.tile_off[i]);
  };
  if constexpr (flat) {
    if (a.tile_off_out) {  // uniform
      // Wave 0 scans the tile counts (an invalid descriptor counts 0) of up
      // to kFusedPlan sequences, 64 per step, into LDS; workgroup (0, 0)
      // also stores them for the merge kernel.
      if (wv == 0) {
        int32_t n[kFusedPlan / 64], per = 0;
#pragma unroll
        for (int c = 0; c < kFusedPlan / 64; c++) {
          const int i = 64 * c + lane;
          n[c] = 0;
          if (i < a.batch) {
            const int32_t len = a.lengths[i], off = a.offsets[i];
            const bool bad = len < 0 || len > a.kv_len || off < 0 || (off & 31);
            n[c] = bad ? 0 : (len + 31) >> 5;
          }
        }
        const bool store = blockIdx.x == 0 && blockIdx.y == 0;
        // exclusive scan of n into LDS; returns the sum
        auto scan = [&] {
          int32_t carry = 0;
#pragma unroll
          for (int c = 0; c < kFusedPlan / 64; c++) {
            int32_t inc = n[c];
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
              const int32_t y = __shfl_up(inc, d, 64);
              if (lane >= d) inc += y;
            }
            if (64 * c + lane < a.batch) ltoff[64 * c + lane] = carry + inc - n[c];
            carry += __shfl(inc, 63, 64);
          }
          return carry;
        };
        int32_t carry = scan();
        const int32_t spare = (int32_t)gridDim.x - a.batch;
        if (carry > (int32_t)gridDim.x && spare > 0 && carry <= kChunkTiles * spare) {
          per = max(1, (carry + spare - 1) / spare);
#pragma unroll
          for (int c = 0; c < kFusedPlan / 64; c++) n[c] = (n[c] + per - 1) / per;
          carry = scan();
        }
        if (store) {
#pragma unroll
          for (int c = 0; c < kFusedPlan / 64; c++)  // the wave's own LDS entries
            if (64 * c + lane < a.batch) a.tile_off_out[64 * c + lane] = ltoff[64 * c + lane];
        }
        if (lane == 0) {
          ltoff[a.batch] = carry;
          ltoff[kFusedPlan + 1] = per;
          if (store) a.tile_off_out[a.batch] = per ? -1 - carry : carry;
        }
      }
      __syncthreads();
    }
    // min(gridDim.x, T) workgroups take the tiles, each at least one
    // (uniform values: kept in scalar registers)
    if (a.tile_off_out) per_seq = __builtin_amdgcn_readfirstlane(ltoff[kFusedPlan + 1]);
    const int64_t total = toff(a.batch);
    const int64_t nw = per_seq ? total : min((int64_t)gridDim.x, total);
    if (chunk_idx >= nw) return;  // uniform
    t_lo = per_seq ? chunk_idx : (int64_t)chunk_idx * total / nw;
    t_hi = per_seq ? chunk_idx + 1 : (int64_t)(chunk_idx + 1) * total / nw;
    // the sequence holding tile t_lo: the last s with tile_off[s] <= t_lo
    int lo = 0, hi = a.batch - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (toff(mid) <= t_lo) lo = mid;
      else hi = mid - 1;
    }
    s = lo;
  } else if (a.lengths) {
    len = a.lengths[s];
    row0 = a.offsets[s];
    lim0 = len;
    // invalid descriptors are reported as NaN by the combine kernel
    if (len < 0 || len > a.kv_len || row0 < 0 || (row0 & 31)) return;
  } else {
    len = a.kv_len;
    row0 = 0;
    lim0 = a.lim0;
    if constexpr (GROUPS) lim0 += s * a.nq;
  }
  if constexpr (!flat) {
    key_begin = (int64_t)chunk_idx * a.chunk;
    // uniform over the workgroup; with the in-launch merge every workgroup
    // takes part (an empty chunk leaves an empty partial)
    if (key_begin >= len && !a.mcnt) return;
    key_end = min(key_begin + (int64_t)a.chunk, len);
  }

  // K operand rows: tile u, A-row j <-> key k0 + 8*(j/4) + 4u + j%4, so that
  // accumulator row 4g+e of tile u is key k0 + 8g + 4u + e.  In the 32-row
  // block layout this operand (chunk 4kk + g of row j, half u) is one
  // 16-byte vector, and the 16 lanes of a group read 256 contiguous bytes.
  // Whole 32-key tiles always lie inside the allocation (cache capacities
  // are multiples of 256 rows; ragged sequences own whole 32-row blocks),
  // so the loads are unconditional and straight-line.  Keys past key_end
  // are masked out of the scores below; their V values are zeroed because
  // stale rows may hold anything (NaN included) and 0 * NaN is NaN.
  // V operand: lane (g, j), value block dblk holds V^T[dblk*16 + j][keys
  // k0+8g .. k0+8g+7] = one 16-byte vector of the block layout.
  auto load_k = [&](int64_t k0, f16x8(&kf)[2][8]) {
    const _Float16* kp =
        a.k + (((row0 + k0) >> 5) * G + kvh) * (int64_t)(32 * D) + g * 128 + j * 8;
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int kk = 0; kk < 8; kk++) kf[u][kk] = load16(kp + u * (16 * D) + kk * 512);
  };
  auto load_v = [&](int64_t k0, f16x8(&vf)[16]) {
    const _Float16* vp =
        a.v + (((row0 + k0) >> 3) + g) * G * (int64_t)(D * 8) + kvh * (D * 8) + j * 8;
#pragma unroll
    for (int dblk = 0; dblk < 16; dblk++) vf[dblk] = load16(vp + dblk * 128);
  };
  // LDS: per KV head of the workgroup the merge area (below); with the
  // projection prologue then the normed, rotated f16 query rows of the
  // workgroup's GH*8 heads.
  constexpr int kLdsRow = D + 4;
  constexpr int kQRow = D + 8;
  const int per_head = NWH * ncols * kLdsRow + 2 * NWH * ncols;
  _Float16* qs = (_Float16*)(smem + GH * per_head);  // [GH*8][kQRow]
  // Projection prologue, issue side: this lane's part of the q_proj rows
  // (one query head per kTPH lanes of the workgroup).  The first K/V tile is
  // loaded in the tile loop, after the prologue: issuing it here keeps 128
  // registers live through the norm and rotation, which spills (measured
  // 2 us slower per step).
  constexpr int kTPH = NWH * 8;
  RopeLane<kProj ? D / kTPH : 4, X::kSH> tab;
  HeadPart<kProj ? D / kTPH : 4> qpart;
  f16x8 kf[2][8], vf[16];
  if constexpr (kProj) {
    qpart.load(x.q_proj + ((int64_t)blockIdx.y * GH * 8 + threadIdx.x / kTPH) * (2 * D), x.q_w,
               lane);
    tab.load(x, lane);
  }

  if constexpr (kProj) {
    const int64_t r = a.app0;
    if (key_begin <= r && r < key_end) {  // workgroup-uniform
      const int h0 = blockIdx.y * GH;
      constexpr int TPH = NWH * 8, DPT = D / TPH;
      if ((int)threadIdx.x < GH * TPH) {  // whole waves
        // K head h0 + t / TPH, columns DPT * (t % TPH) ...
        const int hk = threadIdx.x / TPH;
        HeadPart<DPT> kp;
        kp.load(x.k + (h0 + hk) * D, x.k_w, lane);
        kp.template norm_rope<X::kSH>(x, tab, lane);
        const float(&y)[DPT] = kp.y;
        if constexpr (DPT == 8) {
          f16x8 h;
#pragma unroll
          for (int e = 0; e < 8; e++) h[e] = (_Float16)y[e];
          *(f16x8*)(a.kw + mi::k_offset(r, h0 + hk, DPT * (lane % TPH), G, D)) = h;
        } else {
          f16x4 h;
#pragma unroll
          for (int e = 0; e < 4; e++) h[e] = (_Float16)y[e];
          *(f16x4*)(a.kw + mi::k_offset(r, h0 + hk, DPT * (lane % TPH), G, D)) = h;
        }
      }
      for (int it = threadIdx.x; it < GH * D; it += NWH * GH * 64) {
        const int hh = it / D, i = it % D;
        a.vw[mi::v_offset(r, h0 + hh, i, G, D)] = (_Float16)x.v[(h0 + hh) * D + i];
      }
      __syncthreads();  // the row is in L2 before any wave of this group reads it
    }
  } else if (a.app_n > 0) {
    // Fused append of the new rows that fall in this chunk, for this
    // workgroup's GH heads; nothing else reads them in this launch.
    const int64_t r_lo = max(key_begin, a.app0);
    const int64_t r_hi = min(key_end, a.app0 + a.app_n);
    if (r_lo < r_hi) {  // workgroup-uniform
      const int nrow = (int)(r_hi - r_lo);
      const int h0 = blockIdx.y * GH;
      for (int it = threadIdx.x; it < nrow * GH * (D / 8); it += NWH * GH * 64) {
        const int rr = it / (GH * (D / 8)), hh = (it / (D / 8)) % GH, c = it % (D / 8);
        const int64_t r = r_lo + rr;
        *(f16x8*)(a.kw + mi::k_offset(r, h0 + hh, 8 * c, G, D)) =
            *(const f16x8*)(a.app_k + (r - a.app0) * G * D + (h0 + hh) * D + 8 * c);
      }
      for (int it = threadIdx.x; it < nrow * GH * D; it += NWH * GH * 64) {
        const int rr = it / (GH * D), hh = (it / D) % GH, i = it % D;
        const int64_t r = r_lo + rr;
        a.vw[mi::v_offset(r, h0 + hh, i, G, D)] = a.app_v[(r - a.app0) * G * D + (h0 + hh) * D + i];
      }
      __syncthreads();  // the rows are in L2 before any wave of this group reads them
    }
  }


  // One pass per key range: once, or per sequence segment of a flat range.
  for (;;) {
  int64_t pslot = (int64_t)s * a.max_chunks + chunk_idx;  // partial slot
  if constexpr (flat) {
    const int64_t ps = toff(s);
    const int64_t pe = toff(s + 1);
    len = __builtin_amdgcn_readfirstlane(a.lengths[s]);
    row0 = __builtin_amdgcn_readfirstlane(a.offsets[s]);
    lim0 = len;
    const int64_t unit = 32 * (per_seq ? per_seq : 1);  // keys of an entry of the table
    key_begin = unit * (max(t_lo, ps) - ps);
    key_end = min(unit * (min(t_hi, pe) - ps), len);
    pslot = (int64_t)chunk_idx + s;
  }

  // Q^T operand: lane (g, j) holds q[token][head][32kk + 8g + 0..7] for its
  // column j, kk = 0..7 (the column chunk 4kk + g the K operand of the same
  // lane holds).  Padding columns are zero and fully masked.
  f16x8 qf[NCB][8];
  int64_t lim[NCB];
  if constexpr (kProj) {
    static_assert(NCB == 1, "projection input is one query token");
    // Cooperative norm + rotation of the workgroup's GH*8 query heads, one
    // head per kTPH lanes; the result goes to LDS as f16 and comes back as
    // this lane's Q^T operand (column j < 8 = query head kvh*8 + j).
    {
      constexpr int DPT = D / kTPH;
      const int hl = threadIdx.x / kTPH;
      qpart.template norm_rope<X::kSH>(x, tab, lane);
      _Float16* dst = qs + hl * kQRow + DPT * (lane % kTPH);
      if constexpr (DPT == 8) {
        f16x8 h;
#pragma unroll
        for (int e = 0; e < 8; e++) h[e] = (_Float16)qpart.y[e];
        *(f16x8*)dst = h;
      } else {
        f16x4 h;
#pragma unroll
        for (int e = 0; e < 4; e++) h[e] = (_Float16)qpart.y[e];
        *(f16x4*)dst = h;
      }
    }
    mi::sync_lds();
    const bool col = j < 8;
    const _Float16* qrow = qs + (hw * 8 + (j & 7)) * kQRow + 8 * g;
#pragma unroll
    for (int kk = 0; kk < 8; kk++) qf[0][kk] = col ? *(const f16x8*)(qrow + 32 * kk) : f16x8{};
    lim[0] = col ? a.lim0 : 0;
  } else {
#pragma unroll
  for (int cb = 0; cb < NCB; cb++) {
    const int c = cb * 16 + j;
    const int tok = c >> 3;
    if (c < ncols && (!GROUPS || s * a.nq + tok < a.ntok)) {
      const _Float16* qp =
          a.q + (((int64_t)s * a.nq + tok) * a.H + kvh * 8 + (c & 7)) * D + 8 * g;
#pragma unroll
      for (int kk = 0; kk < 8; kk++) qf[cb][kk] = *(const f16x8*)(qp + 32 * kk);
      lim[cb] = lim0 + tok;
    } else {
#pragma unroll
      for (int kk = 0; kk < 8; kk++) qf[cb][kk] = f16x8{};
      lim[cb] = 0;
    }
  }
  }

  float m[NCB], l[NCB];
  f32x4 acc[NCB][16];
#pragma unroll
  for (int cb = 0; cb < NCB; cb++) {
    m[cb] = kNegBig;
    l[cb] = 0.f;
#pragma unroll
    for (int d = 0; d < 16; d++) acc[cb][d] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // V rows of the last, partial tile past key_end are zeroed (a
  // wave-uniform branch).  The flat ragged split meets such a tile at the
  // end of every sequence segment, so there the zeroing (which waits for the
  // V loads) comes after the QK MFMAs: C3 312 against 323 us.  For single
  // sequences it stays ahead of them: a build with it after them for every
  // kernel took 15.6 against 14.6 us per C2 split launch.
  auto zero_v_tail = [&](int64_t k0) {
    const int64_t valid = key_end - (k0 + 8 * g);
#pragma unroll
    for (int dblk = 0; dblk < 16; dblk++)
#pragma unroll
      for (int e = 0; e < 8; e++)
        if (e >= valid) vf[dblk][e] = (_Float16)0.f;
  };
  // Wave w of the head takes a contiguous run of the range's 32-key tiles
  // (ceil(tiles / NWH) each).  Against tiles dealt round-robin this took the
  // C2 split from 14.6 to 14.2 us (one tile per wave either way: the loop
  // the compiler makes is what differs); verify and the ragged batch are
  // unchanged.
  const mi::WaveTiles wt = mi::split_wave_tiles(key_begin, key_end, NWH, w);
  for (int64_t k0 = wt.first; k0 < wt.last; k0 += 32) {
    load_k(k0, kf);
    load_v(k0, vf);
    if (!flat && k0 + 32 > key_end) zero_v_tail(k0);

#pragma unroll
    for (int cb = 0; cb < NCB; cb++) {
      f32x4 st[2];
#pragma unroll
      for (int u = 0; u < 2; u++) {
        f32x4 c4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < 8; kk++)
          c4 = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[u][kk], qf[cb][kk], c4, 0, 0, 0);
        st[u] = c4;
      }
      if (flat && cb == 0 && k0 + 32 > key_end) zero_v_tail(k0);
      // scale into base 2 and mask keys outside this column's window
      float mt = kNegBig;
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int64_t key = k0 + 8 * g + 4 * u + e;
          float sv = st[u][e] * a.scale_log2e;
          sv = (key < lim[cb] && key < key_end) ? sv : -INFINITY;
          st[u][e] = sv;
          mt = fmaxf(mt, sv);
        }
      mt = mi::max_rows(mt);
      const float mnew = fmaxf(m[cb], mt);
      const float alpha = exp2f(m[cb] - mnew);
      const float mref = TILE ? mt : mnew;
      const float wt = TILE ? exp2f(mt - mnew) : 1.f;
      float rs = 0.f;
      f16x8 pf;
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          // The row sum adds the f16 weights the PV MFMA uses, so that the
          // normalised weights sum to one.
          const _Float16 ph = (_Float16)exp2f(st[u][e] - mref);
          rs += (float)ph;
          pf[4 * u + e] = ph;
        }
      rs = mi::sum_rows(rs);
      l[cb] = l[cb] * alpha + (TILE ? rs * wt : rs);
      m[cb] = mnew;
#pragma unroll
      for (int dblk = 0; dblk < 16; dblk++) {
        acc[cb][dblk] *= alpha;
        if constexpr (TILE)
          acc[cb][dblk] += wt * __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                    vf[dblk], pf, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        else
          acc[cb][dblk] =
              __builtin_amdgcn_mfma_f32_16x16x32_f16(vf[dblk], pf, acc[cb][dblk], 0, 0, 0);
      }
    }
  }

  // ---- merge the NWH waves of each head through LDS.  Per head:
  // O [NWH][ncols][kLdsRow] (row padded by 4 floats so the 16 columns a
  // lane group writes fall in distinct banks), then m, l [NWH][ncols].
  float* so = smem + hw * per_head;
  float* sm = so + NWH * ncols * kLdsRow;
  float* sl = sm + NWH * ncols;
#pragma unroll
  for (int cb = 0; cb < NCB; cb++) {
    const int c = cb * 16 + j;
    if (c < ncols) {
      float* dst = so + (w * ncols + c) * kLdsRow + 4 * g;
#pragma unroll
      for (int dblk = 0; dblk < 16; dblk++) *(f32x4*)(dst + dblk * 16) = acc[cb][dblk];
      if (g == 0) {
        sm[w * ncols + c] = m[cb];
        sl[w * ncols + c] = l[cb];
      }
    }
  }
  __syncthreads();
  // merged O, four columns of d per thread; each thread derives its column's
  // merge weights 2^(m_w - M) from the NWH waves' (m, l) itself (four
  // exponentials), which saves a barrier on the kernel's critical path; the
  // threads of d4 = 0 also store the merged (M, L).
  for (int idx = threadIdx.x; idx < GH * ncols * (D / 4); idx += NWH * GH * 64) {
    const int h2 = idx / (ncols * (D / 4));
    const int c = (idx / (D / 4)) % ncols;
    const int d4 = (idx % (D / 4)) * 4;
    const float* so2 = smem + h2 * per_head;
    const float* sm2 = so2 + NWH * ncols * kLdsRow;
    const float* sl2 = sm2 + NWH * ncols;
    float M = kNegBig;
#pragma unroll
    for (int ww = 0; ww < NWH; ww++) M = fmaxf(M, sm2[ww * ncols + c]);
    float L = 0.f;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ww = 0; ww < NWH; ww++) {
      const float sc = exp2f(sm2[ww * ncols + c] - M);
      L += sl2[ww * ncols + c] * sc;
      o += *(const f32x4*)(so2 + (ww * ncols + c) * kLdsRow + d4) * sc;
    }
    const int64_t pb = ((int64_t)(blockIdx.y * GH + h2) * a.nslots + pslot) * ncols + c;
    if (!flat && a.mcnt) {
      // plain stores: the merging workgroup reads them from this XCD's L2
      if (d4 == 0) {
        float* ml = a.part_ml + ((int64_t)(blockIdx.y * GH + h2) * a.nslots + pslot) * 64 + 2 * c;
        ml[0] = M;
        ml[1] = L;
      }
      *(f32x4*)(a.part_o + pb * D + d4) = o;
    } else {
      if (d4 == 0) {
        store_part(M, a.part_ml + pb * 2 + 0);
        store_part(L, a.part_ml + pb * 2 + 1);
      }
      store_part(o, (f32x4*)(a.part_o + pb * D + d4));
    }
  }
  if constexpr (!flat) {
    if constexpr (NWH * GH == 8 && NCB == 1) {  // the forms the host merges in-launch
      if (a.mcnt) merge_tail<NWH * GH * 64>(a);
    }
    break;
  }
  if (toff(s + 1) >= t_hi) break;
  // next sequence with tiles (the range ends inside a later one)
  do s++;
  while (toff(s + 1) == toff(s));
  __syncthreads();  // the LDS merge area is reused
  }
}

// ---- one launch for few keys per query: no chunks, no partials, no merge
// launch.  A workgroup holds the 8 query heads of two tokens (16 columns) and
// NDB * 16 of the 256 value columns of one KV head, and walks every key they
// see: its four waves take 32-key tiles in turn, straight from the cache into
// registers as in attn_split_kernel, merge through LDS, and the workgroup
// normalises, gates and writes the output.  K(next) is requested when QK has
// read K, V(next) when PV has read V.
//
// Bound: the chain launch - Q - K - QK - V - PV - merge of one workgroup, then
// what one CU can load (~50 bytes a clock: 32 keys of K and V took 2.5 us for
// eight waves at once).  Hence the slices of V: with NDB = 4 a decode step
// loads K four times but on four CUs.  Four waves measured
// best (us, 2 / 4 / 8 / 16 waves at 517 rows: 10.0 with NDB = 16 / 6.0 / 6.7 /
// 11.8).  A step at 517 rows from HBM 10.9 -> 7.1 us, from projections 13.5 ->
// 9.2, four draft tokens after 300 rows 14.4 -> 5.9, 64 prompt tokens 14.9 ->
// 6.7 with their append.
struct DirectArgs {
  const _Float16* k;
  const _Float16* v;
  const _Float16* q;       // [n][H][D]
  const _Float16* gate;    // [n][H][D] or null
  const float* gate32;     // or the gate halves of q_proj [H][2*D], n = 1 (else null)
  _Float16* out;           // [n][H][D]
  const _Float16* app_k;   // rows [past, past + n) to append first ([n][G*D]), or null
  const _Float16* app_v;
  _Float16* kw;
  _Float16* vw;
  int past, n, G, H;       // token i sees keys [0, past + i]
  float scale_log2e;
};

constexpr int kDirectWaves = 4;
// TILE: a tile's weights are taken against the tile's own max, so that its
// largest is exactly 1 in f16, and its sums are weighted in f32 - the precision
// of the split forms, whose waves see one tile each at these lengths.  Against
// the wave's running max, where only one of its tiles has such a weight, the
// error against 64 bits was 3.5 % larger for a step at 517 rows, 6 % for a
// verify of 8 at 1000, 9.5 % for one of 24 at 3100.  It costs 0.1 of 7.3 us at
// 517 rows.  A prefill in slices of 16 value blocks (NDB = 16) goes without: it
// is closer than the prefill grid, which it stands for, as it is (2.44e-4 and
// 2.50e-4 for 333 tokens, 2.63e-4 and 2.87e-4 for 200 after 600 rows), and the
// weighting took the latter from 13.7 to 14.5 us.
template <int NDB, typename X, bool TILE>
__global__ void __launch_bounds__(kDirectWaves * 64, 2)
attn_direct_kernel(DirectArgs a, X x) {
  constexpr bool kProj = is_proj<X>::value;
  constexpr int NWH = kDirectWaves, TOK = 2, NCOL = 16, SL = 16 / NDB, DS = NDB * 16;
  extern __shared__ float smem[];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, j = lane & 15;
  const int G = a.G;
  const int t0 = (gridDim.x - 1 - blockIdx.x) * TOK;  // heaviest first
  const int kvh = blockIdx.y / SL, d0 = (blockIdx.y % SL) * DS;
  const int ntok = min(TOK, a.n - t0);
  const int rows = a.past + t0 + ntok;  // keys the last token sees

  // Appended rows: every workgroup writes the K rows of its head that its
  // tokens see and its own value columns of V, and reads its own writes.
  // Workgroups of one head write the same bytes to the same K rows.
  constexpr int kTPH = NWH * 8;  // lanes per query head of the projection prologue
  RopeLane<kProj ? D / kTPH : 4, X::kSH> tab;
  HeadPart<kProj ? D / kTPH : 4> qpart;
  if constexpr (kProj) {
    qpart.load(x.q_proj + (kvh * 8 + threadIdx.x / kTPH) * (2 * D), x.q_w, lane);
    tab.load(x, lane);
    if (w == 0) {  // the whole wave norms the head (twice), its first kTPH lanes store it
      constexpr int DPT = D / kTPH;
      static_assert(kTPH <= 64, "one wave holds the K head");
      HeadPart<DPT> kp;
      kp.load(x.k + kvh * D, x.k_w, lane);
      kp.template norm_rope<X::kSH>(x, tab, lane);
      typedef _Float16 fv __attribute__((ext_vector_type(DPT)));
      fv h;
#pragma unroll
      for (int e = 0; e < DPT; e++) h[e] = (_Float16)kp.y[e];
      if (lane < kTPH) *(fv*)(a.kw + mi::k_offset(a.past, kvh, DPT * lane, G, D)) = h;
    }
    for (int i = threadIdx.x; i < DS; i += NWH * 64)
      a.vw[mi::v_offset(a.past, kvh, d0 + i, G, D)] = (_Float16)x.v[kvh * D + d0 + i];
    __syncthreads();
  } else if (a.app_k) {
    const int nrow = rows - a.past;
    for (int it = threadIdx.x; it < nrow * (D / 8); it += NWH * 64) {
      const int r = it / (D / 8), c = it % (D / 8);
      *(f16x8*)(a.kw + mi::k_offset(a.past + r, kvh, 8 * c, G, D)) =
          *(const f16x8*)(a.app_k + (r * G + kvh) * D + 8 * c);
    }
    for (int it = threadIdx.x; it < nrow * DS; it += NWH * 64) {
      const int r = it / DS, i = d0 + it % DS;
      a.vw[mi::v_offset(a.past + r, kvh, i, G, D)] = a.app_v[(r * G + kvh) * D + i];
    }
    __syncthreads();
  }

  constexpr int kRow = DS + 4;  // merge rows, padded by one 16-byte slot
  _Float16* const qs = (_Float16*)(smem + NWH * NCOL * (kRow + 2));  // kProj: [8][kQRow]
  constexpr int kQRow = D + 8;
  f16x8 qf[8];
  int lim;  // keys this lane's column sees
  if constexpr (kProj) {
    constexpr int DPT = D / kTPH;
    typedef _Float16 fv __attribute__((ext_vector_type(DPT)));
    qpart.template norm_rope<X::kSH>(x, tab, lane);
    fv h;
#pragma unroll
    for (int e = 0; e < DPT; e++) h[e] = (_Float16)qpart.y[e];
    *(fv*)(qs + (threadIdx.x / kTPH) * kQRow + DPT * (lane % kTPH)) = h;
    mi::sync_lds();
#pragma unroll
    for (int kk = 0; kk < 8; kk++)
      qf[kk] = j < 8 ? *(const f16x8*)(qs + (j & 7) * kQRow + 8 * g + 32 * kk) : f16x8{};
    lim = j < 8 ? rows : 0;
  } else {
    const int tok = j >> 3;
    const bool on = tok < ntok;
    const _Float16* qp =
        a.q + ((int64_t)(t0 + (on ? tok : 0)) * a.H + kvh * 8 + (j & 7)) * D + 8 * g;
#pragma unroll
    for (int kk = 0; kk < 8; kk++) qf[kk] = *(const f16x8*)(qp + 32 * kk);
    lim = on ? a.past + t0 + tok + 1 : 0;  // a padding column sees no key
  }

  float m = kNegBig, l = 0.f;
  f32x4 acc[NDB];
#pragma unroll
  for (int d = 0; d < NDB; d++) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  f16x8 kf[2][8], vf[NDB];
  const _Float16* const kb = a.k + (int64_t)kvh * (32 * D) + g * 128 + j * 8;
  const _Float16* const vb = a.v + ((int64_t)g * G + kvh) * (D * 8) + (d0 + j) * 8;
  auto load_k = [&](int t) {
    const _Float16* kp = kb + (int64_t)t * G * (32 * D);
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int kk = 0; kk < 8; kk++) kf[u][kk] = *(const f16x8*)(kp + u * (16 * D) + kk * 512);
  };
  auto load_v = [&](int t) {
    const _Float16* vp = vb + (int64_t)t * G * (32 * D);
#pragma unroll
    for (int d = 0; d < NDB; d++) vf[d] = *(const f16x8*)(vp + d * 128);
  };
  const int ntiles = (rows + 31) / 32;
  const float c2 = a.scale_log2e;
  if (w < ntiles) {
    load_k(w);
    load_v(w);
  }
  for (int t = w; t < ntiles; t += NWH) {
    f32x4 st[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
      f32x4 c4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < 8; kk++)
        c4 = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[u][kk], qf[kk], c4, 0, 0, 0);
      st[u] = c4;
    }
    if (t + NWH < ntiles) load_k(t + NWH);
    if (32 * t + 32 > a.past + t0 + 1) {  // some column does not see the whole tile
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (32 * t + 8 * g + 4 * u + e >= lim) st[u][e] = -INFINITY;
    }
    float mt = fmaxf(st[0][0], st[1][0]);
#pragma unroll
    for (int e = 1; e < 4; e++) mt = fmaxf(mt, fmaxf(st[0][e], st[1][e]));
    mt = fmaxf(mi::max_rows(mt) * c2, kNegBig);  // (a column that sees no key: -inf)
    const float mnew = fmaxf(m, mt);
    if (__ballot(mnew != m)) {
      const float alpha = __builtin_amdgcn_exp2f(m - mnew);
      l *= alpha;
#pragma unroll
      for (int d = 0; d < NDB; d++) acc[d] *= alpha;
      m = mnew;
    }
    const float mref = TILE ? mt : m;
    const float wt = TILE ? __builtin_amdgcn_exp2f(mt - m) : 1.f;
    // The row sum adds the f16 weights the PV MFMA uses.
    float rs = 0.f;
    f16x8 pf;
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        const f16x2 ph = {(_Float16)__builtin_amdgcn_exp2f(fmaf(st[u][e], c2, -mref)),
                          (_Float16)__builtin_amdgcn_exp2f(fmaf(st[u][e + 1], c2, -mref))};
        rs = __builtin_amdgcn_fdot2(ph, f16x2{1.f16, 1.f16}, rs, false);
        pf[4 * u + e] = ph[0];
        pf[4 * u + e + 1] = ph[1];
      }
    l += mi::sum_rows(rs) * wt;
    if (32 * t + 32 > rows) {  // stale rows may hold anything, 0 * NaN is NaN
      const int valid = rows - (32 * t + 8 * g);
#pragma unroll
      for (int d = 0; d < NDB; d++)
#pragma unroll
        for (int e = 0; e < 8; e++)
          if (e >= valid) vf[d][e] = (_Float16)0.f;
    }
#pragma unroll
    for (int d = 0; d < NDB; d++) {
      if constexpr (TILE) {
        acc[d] += wt * __builtin_amdgcn_mfma_f32_16x16x32_f16(vf[d], pf, f32x4{0.f, 0.f, 0.f, 0.f},
                                                              0, 0, 0);
        // (all 16 products at once would spill)
        if (NDB == 16 && d % 2 == 1) __builtin_amdgcn_sched_barrier(0);
      } else {
        acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf[d], pf, acc[d], 0, 0, 0);
      }
    }
    if (t + NWH < ntiles) load_v(t + NWH);
  }

  // merge of the waves through LDS: O [NWH][NCOL][kRow], then (m, l)
  float* const so = smem;
  float2* const sml = (float2*)(smem + NWH * NCOL * kRow);
  float* dst = so + (w * NCOL + j) * kRow + 4 * g;
#pragma unroll
  for (int d = 0; d < NDB; d++) *(f32x4*)(dst + d * 16) = acc[d];
  if (g == 0) sml[w * NCOL + j] = float2{m, l};
  __syncthreads();
  for (int idx = threadIdx.x; idx < ntok * 8 * (DS / 4); idx += NWH * 64) {
    const int c = idx / (DS / 4), d4 = (idx % (DS / 4)) * 4;
    const int hq = kvh * 8 + (c & 7), tok = t0 + (c >> 3);
    const int64_t o0 = ((int64_t)tok * a.H + hq) * D + d0 + d4;
    f32x4 gv;
    if (a.gate) {
      const f16x4 gh = *(const f16x4*)(a.gate + o0);
#pragma unroll
      for (int e = 0; e < 4; e++) gv[e] = (float)gh[e];
    } else if (a.gate32) {
      gv = *(const f32x4*)(a.gate32 + hq * (2 * D) + D + d0 + d4);
    }
    float M = kNegBig;
#pragma unroll
    for (int ww = 0; ww < NWH; ww++) M = fmaxf(M, sml[ww * NCOL + c].x);
    float L = 0.f;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ww = 0; ww < NWH; ww++) {
      const float2 ml = sml[ww * NCOL + c];
      const float sc = __builtin_amdgcn_exp2f(ml.x - M);
      L += ml.y * sc;
      o += *(const f32x4*)(so + (ww * NCOL + c) * kRow + d4) * sc;
    }
    // out = O / L (zero when L = 0, math_util.rs:357, 372), then the gate
    const float inv = L > 0.f ? 1.f / L : 0.f;
    f16x4 h;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      float r = o[e] * inv;
      if (a.gate || a.gate32) r = mi::gate_mul(r, gv[e]);
      h[e] = (_Float16)r;
    }
    *(f16x4*)(a.out + o0) = h;
  }
}

struct CombineArgs {
  const int32_t* offsets;  // ragged (else null)
  const int32_t* lengths;  // ragged (else null)
  int64_t kv_len;          // rows (ragged: max_len)
  const float* part_o;
  const float* part_ml;
  const _Float16* gate;    // [batch][nq][H][D] or null
  const float* gate32;     // or the gate halves of q_proj [nq][H][2*D] (else null)
  _Float16* out;           // [batch][nq][H][D]
  int G, H, nq, chunk, max_chunks;
  const int32_t* tile_off;  // flat ragged split (SplitArgs::tile_off), else null
  int nwg, batch;           // flat: the split launch's gridDim.x; sequences
  int64_t nslots;           // partial slots per KV head (SplitArgs::nslots)
  int ntok;                 // token groups: query tokens in all
};

// Chunk merge.  One workgroup per (column, KV head x slice of S values of
// d, sequence), 256 threads.  Every global load is issued up front: each
// thread's (m_c, l_c) for chunks t, t+256, ... and its partial outputs o_c[d]
// (d = d0 + t%S, chunks congruent to t/S mod 256/S, up to kBatch of them).
// The max and the sum over chunks are wave reductions in DPP followed by one
// LDS exchange each.
// out = sum_c o_c 2^(m_c - M) / sum_c l_c 2^(m_c - M), zero when the
// denominator is zero (the reference's `sum > 0` guard and zero-filled
// output, math_util.rs:357, 372), then * sigmoid(gate).
constexpr int kMaxChunks = mi::kMaxSplitChunks;

extern "C" __device__ float __ockl_wfred_max_f32(float);
extern "C" __device__ float __ockl_wfred_add_f32(float);

// S = kCombineSlice values of d per workgroup: 16 for up to 16 columns
// (decode), 32 for the 32-column verify (measured: decode step 18.9 / 19.2 /
// 19.3 us with S = 16 / 32 / 8, verify 33.1 / 32.7 / 34.6 us).
// KIND: the launch's sequences (or the one) with their own lengths; the wide
// pass, where a token's partials are those of its row block; or token groups.
enum CombineKind { kSequences, kWide, kGroups };
template <int kCombineSlice, CombineKind KIND = kSequences>
__global__ void __launch_bounds__(256)
attn_combine_kernel(CombineArgs a) {
  constexpr int kCombineGroups = 256 / kCombineSlice;  // chunk groups of a workgroup
  __shared__ float red[2][4];
  __shared__ float wts[kMaxChunks];
  __shared__ float acc_s[kCombineGroups][kCombineSlice + 1];
  const int c = blockIdx.x;
  const int kvh = blockIdx.y / (D / kCombineSlice);
  const int d0 = (blockIdx.y % (D / kCombineSlice)) * kCombineSlice;
  const int s = blockIdx.z;
  const int t = threadIdx.x;
  const int wv = t >> 6;
  const int ncols = a.nq * 8;
  if (KIND == kGroups && s * a.nq + (c >> 3) >= a.ntok) return;  // whole workgroups
  int64_t len = a.kv_len;
  bool bad = false;
  if (a.lengths) {
    len = a.lengths[s];
    const int32_t off = a.offsets[s];
    bad = len < 0 || len > a.kv_len || off < 0 || (off & 31);
    if (bad) len = 0;
  }
  if constexpr (KIND == kWide) len = mi::wide_end((int)len - a.nq, a.nq, c >> 7);
  const int nch = (int)((len + a.chunk - 1) / a.chunk);
  const int64_t base = (int64_t)s * a.max_chunks;  // first partial slot of s
  const float* ml = a.part_ml + ((kvh * a.nslots + base) * ncols + c) * 2;  // chunk ch at ml[ch * mstride]
  const int64_t mstride = (int64_t)ncols * 2;
  const int dl = t % kCombineSlice, cg = t / kCombineSlice;
  const float* po = a.part_o + ((kvh * a.nslots + base) * ncols + c) * D + d0 + dl;
  const int64_t ostride = (int64_t)ncols * D;

  float mloc[kMaxChunks / 256], lloc[kMaxChunks / 256];
#pragma unroll
  for (int u = 0; u < kMaxChunks / 256; u++) {
    const int ch = t + 256 * u;
    mloc[u] = ch < nch ? ml[ch * mstride] : kNegBig;
    lloc[u] = ch < nch ? ml[ch * mstride + 1] : 0.f;
  }
  constexpr int kBatch = 16;
  float ov[kBatch];
#pragma unroll
  for (int u = 0; u < kBatch; u++) {
    const int ch = cg + kCombineGroups * u;
    ov[u] = ch < nch ? po[ch * ostride] : 0.f;
  }
  float mx = kNegBig;
#pragma unroll
  for (int u = 0; u < kMaxChunks / 256; u++) mx = fmaxf(mx, mloc[u]);
  mx = __ockl_wfred_max_f32(mx);
  if ((t & 63) == 0) red[0][wv] = mx;
  __syncthreads();
  const float M = fmaxf(fmaxf(red[0][0], red[0][1]), fmaxf(red[0][2], red[0][3]));
  float lsum = 0.f;
#pragma unroll
  for (int u = 0; u < kMaxChunks / 256; u++) {
    const int ch = t + 256 * u;
    if (ch < nch) {
      const float wgt = exp2f(mloc[u] - M);
      wts[ch] = wgt;
      lsum += lloc[u] * wgt;
    }
  }
  lsum = __ockl_wfred_add_f32(lsum);
  if ((t & 63) == 0) red[1][wv] = lsum;
  __syncthreads();  // publishes wts[] and the wave sums
  const float L = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
  float o = 0.f;
#pragma unroll
  for (int u = 0; u < kBatch; u++) {
    const int ch = cg + kCombineGroups * u;
    if (ch < nch) o += ov[u] * wts[ch];
  }
  for (int ch = cg + kCombineGroups * kBatch; ch < nch; ch += kCombineGroups)
    o += po[ch * ostride] * wts[ch];
  acc_s[cg][dl] = o;
  __syncthreads();
  if (t < kCombineSlice) {
    float r = 0.f;
#pragma unroll
    for (int i = 0; i < kCombineGroups; i++) r += acc_s[i][t];
    r = (L > 0.f) ? r / L : 0.f;
    if (bad) r = __builtin_nanf("");
    const int tok = c >> 3;
    const int hq = kvh * 8 + (c & 7);
    const int64_t oidx = (((int64_t)s * a.nq + tok) * a.H + hq) * D + d0 + t;
    if (a.gate) {
      const float gv = (float)a.gate[oidx];
      r = mi::gate_mul(r, gv);
    } else if (a.gate32) {
      const float gv =
          a.gate32[(((int64_t)s * a.nq + tok) * a.H + hq) * (2 * D) + D + d0 + t];
      r = mi::gate_mul(r, gv);
    }
    a.out[oidx] = (_Float16)r;
  }
}

// Merge for the flat ragged split: a sequence has few partials (its tiles
// span a few workgroups), so one workgroup per (column, KV head, sequence)
// with one thread per d runs a single online-softmax pass over them.
// Workgroup x < nw = min(nwg, T) of the split took tiles [x T / nw,
// (x+1) T / nw), so tile t is in workgroup ceil((t+1) nw / T) - 1 and the
// partials of sequence s are in slots first + s .. last + s.
template <int MAXB>
__global__ void __launch_bounds__(D)
attn_combine_flat_kernel(CombineArgs a) {
  const int c = blockIdx.x, kvh = blockIdx.y, s = blockIdx.z, d = threadIdx.x;
  const int ncols = a.nq * 8;
  const int32_t len = a.lengths[s], off = a.offsets[s];
  const bool bad = len < 0 || len > a.kv_len || off < 0 || (off & 31);
  const int64_t total = a.tile_off[a.batch];
  const int64_t ps = a.tile_off[s], pe = a.tile_off[s + 1];
  int64_t first = 0, nch = 0;
  if (total < 0) {  // by chunks of a sequence
    first = ps;
    nch = (s + 1 < a.batch ? pe : -1 - total) - ps;
  } else if (pe > ps) {
    const int64_t nw = min((int64_t)a.nwg, total);
    first = ((ps + 1) * nw + total - 1) / total - 1;
    nch = (pe * nw + total - 1) / total - 1 - first + 1;
  }
  const int64_t slot0 = (kvh * a.nslots + first + s) * ncols + c;
  const float* ml = a.part_ml + slot0 * 2;
  const float* po = a.part_o + slot0 * D + d;
  float M = kNegBig, L = 0.f, o = 0.f;
  // kB partials are loaded per batch, all before their use: 8, or 16 (MAXB)
  // where a sequence has more (a small batch: 8 sequences of 1550 rows 25.7 ->
  // 16.0 us per call with the chunks of one sequence; 16 for all cost 200
  // sequences of two partials 45 -> 50 us, and a kernel that holds both 256
  // sequences of 250..500 rows 53 -> 56).
  auto merge = [&](auto batch) {
    constexpr int kB = decltype(batch)::value;
    for (int64_t c0 = 0; c0 < nch; c0 += kB) {
      float mb[kB], lb[kB], ob[kB];
#pragma unroll
      for (int k = 0; k < kB; k++) {
        const bool in = c0 + k < nch;
        mb[k] = in ? ml[(c0 + k) * ncols * 2] : kNegBig;
        lb[k] = in ? ml[(c0 + k) * ncols * 2 + 1] : 0.f;
        ob[k] = in ? po[(c0 + k) * ncols * D] : 0.f;
      }
      float mx = M;
#pragma unroll
      for (int k = 0; k < kB; k++) mx = fmaxf(mx, mb[k]);
      const float sc = exp2f(M - mx);  // rescale what has been summed
      L *= sc;
      o *= sc;
      M = mx;
#pragma unroll
      for (int k = 0; k < kB; k++) {
        const float wgt = exp2f(mb[k] - M);
        L += lb[k] * wgt;
        o += ob[k] * wgt;
      }
    }
  };
  if (MAXB == 8 || nch <= 8) merge(std::integral_constant<int, 8>{});
  else merge(std::integral_constant<int, MAXB>{});
  float r = (L > 0.f) ? o / L : 0.f;
  if (bad) r = __builtin_nanf("");
  const int hq = kvh * 8 + c;
  const int64_t oidx = ((int64_t)s * a.H + hq) * D + d;
  if (a.gate) r = mi::gate_mul(r, (float)a.gate[oidx]);
  a.out[oidx] = (_Float16)r;
}

// Tile offsets of a ragged batch for the flat split: tile_off[s] = sum over
// r < s of ceil(len_r / 32) (0 for an invalid descriptor), tile_off[batch] =
// the total.  One workgroup, an exclusive scan per 256 sequences.
__global__ void __launch_bounds__(256)
ragged_plan_kernel(const int32_t* lengths, const int32_t* offsets, int batch, int64_t max_len,
                   int32_t* tile_off) {
  __shared__ int32_t scan[256];
  const int t = threadIdx.x;
  int32_t carry = 0;
  for (int b0 = 0; b0 < batch; b0 += 256) {
    const int sq = b0 + t;
    int32_t n = 0;
    if (sq < batch) {
      const int32_t len = lengths[sq], off = offsets[sq];
      const bool bad = len < 0 || len > max_len || off < 0 || (off & 31);
      n = bad ? 0 : (len + 31) >> 5;
    }
    scan[t] = n;
    __syncthreads();
    for (int d = 1; d < 256; d <<= 1) {  // inclusive scan
      const int32_t v = t >= d ? scan[t - d] : 0;
      __syncthreads();
      scan[t] += v;
      __syncthreads();
    }
    if (sq < batch) tile_off[sq] = carry + scan[t] - n;
    carry += scan[255];
    __syncthreads();
  }
  if (t == 0) tile_off[batch] = carry;
}

int env_int(const char* name, int dflt) {
  const char* e = getenv(name);
  return (e && *e) ? atoi(e) : dflt;
}

// Split-planning knobs, read once per process (measurement aids; the
// defaults are the tuned values): MI_ATTN_SPLIT_GH=2 puts both KV heads of
// a Qwen3.6 layer in one workgroup (default one head per workgroup: at C2
// the same split time with half the partials, 18.8 against 19.5 us per
// step), MI_ATTN_SPLIT_WGS sets the target workgroup count,
// MI_ATTN_SPLIT_CHUNK fixes the keys per chunk.
const mi::SplitKnobs& split_knobs() {
  static const mi::SplitKnobs k{env_int("MI_ATTN_SPLIT_GH", 1),
                                std::max(1, env_int("MI_ATTN_SPLIT_WGS", 256)),
                                std::max(0, env_int("MI_ATTN_SPLIT_CHUNK", 0))};
  return k;
}

using mi::SplitPlan;
SplitPlan plan_split(int64_t max_len, int64_t batch, int G, int nq) {
  return mi::plan_split(max_len, batch, G, nq, split_knobs());
}

template <int NWH, int NCB, int GH, typename X = NoProj, bool FLAT = false, bool GROUPS = false,
          bool TILE = false>
mi_status launch_split(const SplitArgs& a, int64_t batch, hipStream_t stream, const X& x = X()) {
  const int ncols = a.nq * 8;
  size_t lds = (size_t)GH * (NWH * ncols * (D + 4) + 2 * NWH * ncols) * sizeof(float);
  if constexpr (is_proj<X>::value) lds += (size_t)GH * 8 * (D + 8) * sizeof(_Float16);
  if constexpr (FLAT) lds += (size_t)(kFusedPlan + 2) * sizeof(int32_t);
  static std::atomic<uint64_t> lds_set{0};
  // (below 160 KiB: the kernel also holds a few bytes of static LDS)
  MI_TRY(mi::set_lds_limit((const void*)attn_split_kernel<NWH, NCB, GH, X, FLAT, GROUPS, TILE>,
                           159 * 1024, lds_set));
  dim3 grid(a.max_chunks, a.G / GH, (unsigned)batch);
  MI_HIP(mi::launch("attn_split", attn_split_kernel<NWH, NCB, GH, X, FLAT, GROUPS, TILE>, grid,
                    dim3(NWH * GH * 64), lds, stream, a, x));
  return MI_OK;
}

template <int SH>
Proj<SH> make_proj(const ProjArgs& p) {
  Proj<SH> x;
  static_cast<ProjInput&>(x) = p;
  std::copy(p.cs, p.cs + 64 * SH, x.cs);
  return x;
}

template <int SH>
mi_status launch_proj(const SplitArgs& a, const SplitPlan& plan, hipStream_t stream,
                      const ProjArgs& p) {
  const Proj<SH> x = make_proj<SH>(p);
  if (plan.gh == 2) return launch_split<4, 1, 2>(a, 1, stream, x);
  return launch_split<8, 1, 1>(a, 1, stream, x);
}

template <int NDB, bool TILE = true, typename X = NoProj>
mi_status launch_direct(const DirectArgs& a, hipStream_t stream, const X& x = X()) {
  size_t lds = (size_t)kDirectWaves * 16 * (NDB * 16 + 4 + 2) * sizeof(float);
  if constexpr (is_proj<X>::value) lds += (size_t)8 * (D + 8) * sizeof(_Float16);
  static std::atomic<uint64_t> lds_set{0};
  MI_TRY(mi::set_lds_limit((const void*)attn_direct_kernel<NDB, X, TILE>, 80 * 1024, lds_set));
  MI_HIP(mi::launch("attn_direct", attn_direct_kernel<NDB, X, TILE>,
                    dim3((a.n + 1) / 2, a.G * (16 / NDB)), dim3(kDirectWaves * 64), lds, stream, a,
                    x));
  return MI_OK;
}

template <int SH>
mi_status launch_direct_proj(const DirectArgs& a, hipStream_t stream, const ProjArgs& p) {
  return launch_direct<4>(a, stream, make_proj<SH>(p));
}

size_t split_workspace_bytes(int64_t batch, int G, int max_chunks, int nq) {
  size_t units = (size_t)batch * G * max_chunks * nq * 8;
  return units * (D + 2) * sizeof(float) + 256;
}

// The in-launch merge: partials o as usual, then (m, l) with a 256-byte
// stride per slot (workgroups of neighbouring slots run on different XCDs,
// whose L2s must not share a line); the state in mi_kv::mstate: counters,
// then per-XCD partials [G][8][8][D] and (m, l) [G][8][64].
size_t merge_workspace_bytes(int G, int max_chunks) {
  return (size_t)G * max_chunks * (8 * D + 64) * sizeof(float) + 256;
}
size_t merge_counter_bytes(int G) { return ((size_t)9 * G * kMergeStride * sizeof(int) + 4095) / 4096 * 4096; }
// The workspace a cache decode / verify launch asks for.
size_t attend_workspace_bytes(int G, int max_chunks, int nq) {
  const size_t s = split_workspace_bytes(1, G, max_chunks, nq);
  return nq == 1 ? std::max(s, merge_workspace_bytes(G, max_chunks)) : s;
}
// MI_ATTN_DECODE_MERGE=1 (read at each call) merges single-token decode
// inside the split launch; off by default: at C2 the merge chain after the
// last workgroup (store acknowledgement, XCD-local arrival, merge from L2,
// write-through, device arrival, final merge from memory) takes ~5 us, as
// long as the second launch it replaces (measured: 21.9 against 19.9 us per
// step on one box, 18.5-18.7 against ~18 us for the kernel end).
bool decode_merge_enabled() {
  const char* e = getenv("MI_ATTN_DECODE_MERGE");
  return e && *e && atoi(e) == 1;
}

// Flat ragged split: workgroups per KV-head group (one per CU), and the
// workspace: partials of nwg + batch slots, then the tile offsets.
int ragged_nwg(int G, int gh) { return std::max(1, 256 / std::max(1, G / gh)); }
size_t ragged_workspace_bytes(int64_t batch, int G, int nwg) {
  return split_workspace_bytes(1, G, nwg + (int)batch, 1) + (size_t)(batch + 1) * sizeof(int32_t);
}

// Runs split + combine for nq <= 4 query tokens per sequence, or with ntok > 0
// for ntok tokens of one sequence in `batch` groups of nq = 4.
struct AppendRows {
  const _Float16* k = nullptr;
  const _Float16* v = nullptr;
  int64_t row0 = 0;
  int n = 0;
};

mi_status run_split(const _Float16* k, const _Float16* v, const int32_t* offsets,
                    const int32_t* lengths, int64_t kv_len, int64_t lim0,
                    int64_t max_len, int64_t batch, int H, int G, int nq,
                    const _Float16* q, const _Float16* gate, _Float16* out,
                    void* ws, size_t ws_bytes, hipStream_t stream,
                    const AppendRows& app = AppendRows(), const ProjArgs* proj = nullptr,
                    const mi_kv* kv = nullptr, int ntok = 0) {
  const SplitPlan plan = ntok ? mi::plan_groups(max_len, (int)batch, G, split_knobs())
                              : plan_split(max_len, batch, G, nq);
  SplitArgs a;
  a.mcnt = nullptr;
  a.k = k;
  a.v = v;
  a.offsets = offsets;
  a.lengths = lengths;
  a.kv_len = kv_len;
  a.lim0 = lim0;
  a.q = q;
  a.G = G;
  a.H = H;
  a.nq = nq;
  a.ntok = ntok;
  a.chunk = plan.chunk;
  a.max_chunks = plan.max_chunks;
  a.scale_log2e = mi::kLog2e / sqrtf((float)D);
  a.app_k = app.k;
  a.app_v = app.v;
  a.kw = const_cast<_Float16*>(k);
  a.vw = const_cast<_Float16*>(v);
  a.app0 = app.row0;
  a.app_n = app.n;
  a.tile_off = nullptr;
  a.tile_off_out = nullptr;
  a.batch = (int)batch;
  const int nwg = ragged_nwg(G, plan.gh);
  const size_t need = lengths ? ragged_workspace_bytes(batch, G, nwg)
                              : split_workspace_bytes(batch, G, a.max_chunks, nq);
  if (ws_bytes < need)
    return mi::fail(MI_ERR_INVALID_ARG, "workspace %zu bytes < %zu needed", ws_bytes, need);
  const size_t slots = lengths ? (size_t)nwg + batch : (size_t)batch * a.max_chunks;
  a.part_o = (float*)ws;
  a.part_ml = a.part_o + slots * G * nq * 8 * D;
  a.nslots = (int64_t)slots;
  if (lengths) {
    // flat split over the concatenated sequences (one nq = 1 token each)
    if (nq != 1) return mi::fail(MI_ERR_INVALID_ARG, "ragged batches take one query token");
    if ((int64_t)batch * ((max_len + 31) / 32) >= ((int64_t)1 << 31))
      return mi::fail(MI_ERR_UNSUPPORTED, "batch * max_len / 32 beyond 2^31 tiles");
    int32_t* tile_off = (int32_t*)(a.part_ml + slots * G * nq * 8 * 2);
    if (batch <= kFusedPlan) {
      a.tile_off_out = tile_off;  // the split launch computes and stores them
    } else {
      MI_HIP(mi::launch("ragged_plan", ragged_plan_kernel, dim3(1), dim3(256), 0, stream, lengths,
                        offsets, (int)batch, kv_len, tile_off));
    }
    a.tile_off = tile_off;
    a.max_chunks = nwg;
    a.chunk = 0;
  }
  // In-launch merge: one sequence, one query token, one KV head per
  // workgroup, 8 waves (the launch_split<8, 1, 1> forms), on a device that
  // dispatches round-robin over 8 XCDs, with room for the padded (m, l).
  const bool merge = kv && kv->merge_ok && kv->mstate && !lengths && batch == 1 && nq == 1 &&
                     plan.gh == 1 && plan.ncb == 1 && plan.nwh == 8 && decode_merge_enabled() &&
                     ws_bytes >= merge_workspace_bytes(G, a.max_chunks);
  if (merge) {
    a.mcnt = (int*)kv->mstate;
    a.xo = (float*)((char*)kv->mstate + merge_counter_bytes(G));
    a.xml = a.xo + (size_t)G * 8 * 8 * D;
    a.gate = gate;
    a.gate32 = proj ? proj->q_proj : nullptr;
    a.out = out;
  }
  mi_status st;
  if (proj) {
    if (nq != 1 || batch != 1) return mi::fail(MI_ERR_INVALID_ARG, "projection input: one token");
    switch (proj->rot_half / 32) {
      case 0: st = launch_proj<0>(a, plan, stream, *proj); break;
      case 1: st = launch_proj<1>(a, plan, stream, *proj); break;
      case 2: st = launch_proj<2>(a, plan, stream, *proj); break;
      case 3: st = launch_proj<3>(a, plan, stream, *proj); break;
      case 4: st = launch_proj<4>(a, plan, stream, *proj); break;
      default: return mi::fail(MI_ERR_UNSUPPORTED, "rot_half=%d", proj->rot_half);
    }
  } else if (lengths) {
    st = plan.gh == 2 ? launch_split<4, 1, 2, NoProj, true>(a, 1, stream)
                      : launch_split<8, 1, 1, NoProj, true>(a, 1, stream);
  } else if (ntok)
    st = a.chunk > 4 * 32 && max_len * G <= 16384
             ? launch_split<4, 2, 1, NoProj, false, true, true>(a, batch, stream)
             : launch_split<4, 2, 1, NoProj, false, true>(a, batch, stream);
  else if (plan.ncb == 2)
    st = launch_split<4, 2, 1>(a, batch, stream);
  else if (plan.gh == 2)
    st = launch_split<4, 1, 2>(a, batch, stream);
  else
    st = launch_split<8, 1, 1>(a, batch, stream);
  MI_TRY(st);
  if (merge) return MI_OK;  // merged and written by the split launch
  CombineArgs c;
  c.offsets = offsets;
  c.lengths = lengths;
  c.kv_len = kv_len;
  c.part_o = a.part_o;
  c.part_ml = a.part_ml;
  c.gate = gate;
  c.gate32 = proj ? proj->q_proj : nullptr;
  c.out = out;
  c.G = G;
  c.H = H;
  c.nq = nq;
  c.chunk = a.chunk;
  c.max_chunks = a.max_chunks;
  c.tile_off = a.tile_off;
  c.nslots = a.nslots;
  c.nwg = nwg;
  c.batch = (int)batch;
  c.ntok = ntok;
  if (lengths) {
    // (128 workgroups per head leave up to 32 sequences four partials or more each)
    MI_HIP(mi::launch("attn_combine",
                      batch <= 32 ? attn_combine_flat_kernel<16> : attn_combine_flat_kernel<8>,
                      dim3(8, G, (unsigned)batch), dim3(D), 0, stream, c));
    return MI_OK;
  }
  if (ntok) {
    MI_HIP(mi::launch("attn_combine", attn_combine_kernel<32, kGroups>,
                      dim3(nq * 8, G * (D / 32), (unsigned)batch), dim3(256), 0, stream, c));
  } else if (nq > 2) {
    MI_HIP(mi::launch("attn_combine", attn_combine_kernel<32>, dim3(nq * 8, G * (D / 32), (unsigned)batch),
                      dim3(256), 0, stream, c));
  } else {
    MI_HIP(mi::launch("attn_combine", attn_combine_kernel<16>, dim3(nq * 8, G * (D / 16), (unsigned)batch),
                      dim3(256), 0, stream, c));
  }
  return MI_OK;
}

// Merge for many columns: a wave per column, four values of d per lane, so
// that a wave reads each chunk's 1 KiB row of O in one instruction.  Columns
// are (token, head) pairs; a token's partials are those of its row block of
// the wide pass: chunks [0, nch), nch from the block's last key.  Used where
// there are few chunks or many columns; attn_combine_kernel spreads the chunks
// of a column over a workgroup instead.  Bound: the partials' bytes.  512 tokens
// in 4 chunks (38 MB): 8.0 us = 4.7 TB/s, against 14.2 us for a thread per
// output value with 4-byte loads.
constexpr int kRowsBatch = 8;
__global__ void __launch_bounds__(256) attn_combine_rows_kernel(CombineArgs a) {
  const int lane = threadIdx.x & 63;
  const int c = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  const int kvh = blockIdx.y;
  const int ncols = a.nq * 8;
  const int tok = c >> 3, hq = kvh * 8 + (c & 7);
  const int nch = (mi::wide_end((int)a.kv_len - a.nq, a.nq, tok >> 4) + a.chunk - 1) / a.chunk;
  const int64_t oidx = ((int64_t)tok * a.H + hq) * D + 4 * lane;
  f16x4 gv = {};
  if (a.gate) gv = *(const f16x4*)(a.gate + oidx);
  const float* ml = a.part_ml + ((int64_t)kvh * a.nslots * ncols + c) * 2;
  const float* po = a.part_o + ((int64_t)kvh * a.nslots * ncols + c) * D + 4 * lane;
  float M = kNegBig, L = 0.f;
  f32x4 O = {0.f, 0.f, 0.f, 0.f};
  for (int c0 = 0; c0 < nch; c0 += kRowsBatch) {
    float m[kRowsBatch], l[kRowsBatch];
    f32x4 o[kRowsBatch];
#pragma unroll
    for (int k = 0; k < kRowsBatch; k++) {
      const int64_t ch = c0 + k < nch ? c0 + k : c0;  // (a repeat is not used)
      m[k] = ml[ch * ncols * 2];
      l[k] = ml[ch * ncols * 2 + 1];
      o[k] = *(const f32x4*)(po + ch * ncols * D);
    }
    float mx = M;
#pragma unroll
    for (int k = 0; k < kRowsBatch; k++) mx = fmaxf(mx, m[k]);
    const float r = exp2f(M - mx);
    L *= r;
    O *= r;
    M = mx;
#pragma unroll
    for (int k = 0; k < kRowsBatch; k++) {
      const float w = c0 + k < nch ? exp2f(m[k] - M) : 0.f;
      L += l[k] * w;
      O += o[k] * w;
    }
  }
  // out = O / L (zero when L = 0, math_util.rs:357, 372), then the gate
  const float inv = L > 0.f ? 1.f / L : 0.f;
  f16x4 h;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    float r = O[e] * inv;
    if (a.gate) r = mi::gate_mul(r, (float)gv[e]);
    h[e] = (_Float16)r;
  }
  *(f16x4*)(a.out + oidx) = h;
}

// A form's switch, read at each call: off when set to 0.
bool switched_on(const char* name) {
  const char* e = getenv(name);
  return !(e && *e && atoi(e) == 0);
}
// More than 4 query tokens in forms other than a launch pair per four tokens.
bool verify_wide_enabled() { return switched_on("MI_ATTN_VERIFY_WIDE"); }

// The wide verify's plan (mi::wide_plan) and the workspace its partials
// (O, m, l) take.
struct WideLaunch {
  int64_t chunk;
  int nchunks;
  size_t ws_bytes;
};
WideLaunch wide_launch(int G, int64_t past, int32_t n) {
  const mi::WidePlan w = mi::wide_plan(G, past, n);
  WideLaunch p;
  p.chunk = w.chunk;
  p.nchunks = w.nchunks;
  p.ws_bytes = (size_t)G * p.nchunks * 8 * n * (D + 2) * sizeof(float) + 256;
  return p;
}

mi_status wide_attend(mi_kv* kv, int32_t layer, const _Float16* q, const _Float16* gate,
                      _Float16* out, int64_t past_pos, int32_t n, hipStream_t stream,
                      const _Float16* k_new, const _Float16* v_new) {
  const int G = kv->G;
  const int64_t rows = past_pos + n;
  const WideLaunch wp = wide_launch(G, past_pos, n);
  const int64_t chunk = wp.chunk;
  const int nchunks = wp.nchunks;
  const int ncols = 8 * n;
  const size_t units = (size_t)G * nchunks * ncols;
  void* ws;
  MI_TRY(mi::kv_workspace(kv, wp.ws_bytes, stream, &ws));
  float* part_o = (float*)ws;
  float* part_ml = part_o + units * D;
  if (k_new) MI_TRY(mi::kv_append_rows(kv, layer, k_new, v_new, past_pos, n, stream));
  MI_TRY(mi::verify_wide_split(kv, layer, q, past_pos, n, chunk, nchunks, part_o, part_ml,
                               stream));
  CombineArgs c{};
  c.kv_len = rows;
  c.part_o = part_o;
  c.part_ml = part_ml;
  c.gate = gate;
  c.out = out;
  c.G = G;
  c.H = kv->H;
  c.nq = n;
  c.chunk = (int)chunk;
  c.max_chunks = nchunks;
  c.batch = 1;
  c.nslots = nchunks;
  // 16-byte lanes per column fill the CUs from 64 tokens on; for fewer with
  // many chunks (16 tokens at 65536 rows: 114), or where a wave's walk over the
  // chunks is long next to the columns (one KV head: 68 tokens in 49 chunks, 34.8
  // us a call against 31.4; 120 in 32 36.8 against 40.7), a workgroup per column
  // and 32-value slice does.  The rows form moves 8-byte pieces of gate and out.
  if ((nchunks <= 16 || (n >= 64 && 8 * nchunks <= 5 * n * G)) &&
      !(((uintptr_t)gate | (uintptr_t)out) & 7))
    MI_HIP(mi::launch("attn_combine", attn_combine_rows_kernel, dim3(n * 2, G), dim3(256), 0,
                      stream, c));
  else
    // (the kernel without the block's end where every block writes every chunk)
    MI_HIP(mi::launch("attn_combine",
                      mi::wide_full(past_pos, n, chunk, nchunks) ? attn_combine_kernel<32>
                                                                 : attn_combine_kernel<32, kWide>,
                      dim3(n * 8, G * (D / 32), 1), dim3(256), 0, stream, c));
  return MI_OK;
}

// Whether n tokens after `past` rows take the one-launch form.  MI_ATTN_DIRECT=0
// (read at each call) turns it off; MI_ATTN_SPLIT_* and, for one token,
// MI_ATTN_DECODE_MERGE (0 or 1) ask for forms of the split launch.
// `inputs`: what the launch reads beside the cache and the gate (a gate value is
// read by the thread that writes its output).  Its workgroups share them
// (slices of V read the same queries, token pairs the same new rows), so an
// output in the same memory, which the other forms take - they write it in a
// later launch, or the prefill grid from the one workgroup that read it - would
// be stored over what another workgroup has yet to read.
struct Span {
  const void* p;
  size_t bytes;
};
bool takes_direct(const mi_kv* kv, int64_t past, int32_t n, const _Float16* gate,
                  const _Float16* out, std::initializer_list<Span> inputs, bool prefill = false) {
  if (!mi::direct_rows(kv->G, past, n, prefill)) return false;
  if (((uintptr_t)gate | (uintptr_t)out) & 7) return false;  // 8-byte accesses here only
  const uintptr_t o0 = (uintptr_t)out, o1 = o0 + (size_t)n * kv->H * D * sizeof(_Float16);
  for (const Span& s : inputs)
    if (s.p && (uintptr_t)s.p < o1 && o0 < (uintptr_t)s.p + s.bytes) return false;
  if (split_knobs().chunk > 0 || split_knobs().gh != 1 || split_knobs().wgs != 256) return false;
  const char* merge = getenv("MI_ATTN_DECODE_MERGE");
  if (n == 1 && merge && *merge) return false;
  return switched_on("MI_ATTN_DIRECT");
}

// Slices of V while the launch has fewer workgroups than CUs.  Measured (us, 4 /
// 2 / 1 slices): no past, 64 tokens 3.6 / 4.3 / 5.7, 128 tokens 5.9 / 5.1 / 6.5,
// 333 tokens 15.6 / 12.5 / 11.3.
int direct_slices(int G, int32_t n) {
  const int wgs = (n + 1) / 2 * G;
  return wgs * 4 <= 256 ? 4 : wgs * 2 <= 256 ? 2 : 1;
}

// Most new rows the one-launch form appends itself (every workgroup of a head
// writes them); more go in a launch before it.
constexpr int kDirectAppend = 16;

mi_status run_direct(mi_kv* kv, int32_t layer, const _Float16* q, const _Float16* gate,
                     _Float16* out, int64_t past, int32_t n, hipStream_t stream,
                     const _Float16* k_new, const _Float16* v_new, const ProjArgs* proj,
                     bool prefill = false) {
  if (k_new && n > kDirectAppend) {
    MI_TRY(mi::kv_append_rows(kv, layer, k_new, v_new, past, n, stream));
    k_new = v_new = nullptr;
  }
  DirectArgs a;
  a.k = a.kw = kv->k[layer];
  a.v = a.vw = kv->v[layer];
  a.q = q;
  a.gate = gate;
  a.gate32 = proj ? proj->q_proj : nullptr;
  a.out = out;
  a.app_k = k_new;
  a.app_v = v_new;
  a.past = (int)past;
  a.n = n;
  a.G = kv->G;
  a.H = kv->H;
  a.scale_log2e = mi::kLog2e / sqrtf((float)D);
  if (proj) {
    switch (proj->rot_half / 32) {
      case 0: return launch_direct_proj<0>(a, stream, *proj);
      case 1: return launch_direct_proj<1>(a, stream, *proj);
      case 2: return launch_direct_proj<2>(a, stream, *proj);
      case 3: return launch_direct_proj<3>(a, stream, *proj);
      default: return launch_direct_proj<4>(a, stream, *proj);
    }
  }
  switch (direct_slices(kv->G, n)) {
    case 4: return launch_direct<4>(a, stream);
    case 2: return launch_direct<8>(a, stream);
  }
  return prefill ? launch_direct<16, false>(a, stream) : launch_direct<16>(a, stream);
}

// Verify / decode over the cache: n query tokens at positions past_pos ..
// past_pos+n-1, rows [0, past_pos+n) already in the cache.
// With k_new / v_new, the n new rows [past_pos, past_pos + n) are appended by
// the attention kernels themselves, each workgroup the rows that it reads before
// it does (in one launch for all groups, all new rows of its chunk); the wide
// form, and the one-launch form of more than kDirectAppend tokens, append them
// in a launch of their own first.  The caller has grown the cache.
mi_status cache_attend(mi_kv* kv, int32_t layer, const _Float16* q, const _Float16* gate,
                       _Float16* out, int64_t past_pos, int32_t n, hipStream_t stream,
                       const _Float16* k_new = nullptr, const _Float16* v_new = nullptr) {
  const size_t rows_bytes = (size_t)n * kv->G * D * sizeof(_Float16);
  const bool wide = n > 4 && verify_wide_enabled();
  // (in one slice of V the wide pass is the faster one from about 2400 rows: 129
  // tokens after 2900 rows 33.9 us against 39.7, after 2100 36.5 against 33.0)
  const bool direct =
      (n <= 4 || wide) && (past_pos < 2400 || direct_slices(kv->G, n) > 1) &&
      takes_direct(kv, past_pos, n, gate, out,
                   {{q, (size_t)n * kv->H * D * sizeof(_Float16)}, {k_new, rows_bytes},
                    {v_new, rows_bytes}});
  if (wide) {
    const bool groups =
        !direct && mi::verify_groups(kv->G, past_pos, n) && switched_on("MI_ATTN_VERIFY_GROUPS");
    if (!direct && !groups)
      return wide_attend(kv, layer, q, gate, out, past_pos, n, stream, k_new, v_new);
    // (the wide form's workspace too: a later captured call may count on what
    // an eager call of this size leaves)
    const int ng = (n + 3) / 4;
    size_t need = wide_launch(kv->G, past_pos, n).ws_bytes;
    if (groups)
      need = std::max(need, split_workspace_bytes(
                                ng, kv->G,
                                mi::plan_groups(past_pos + n, ng, kv->G, split_knobs()).max_chunks,
                                4));
    void* ws;
    MI_TRY(mi::kv_workspace(kv, need, stream, &ws));
    if (groups) {
      AppendRows app;
      app.k = k_new;
      app.v = v_new;
      app.row0 = past_pos;
      app.n = k_new ? n : 0;
      return run_split(kv->k[layer], kv->v[layer], nullptr, nullptr, past_pos + n, past_pos + 1,
                       past_pos + n, ng, kv->H, kv->G, 4, q, gate, out, ws, kv->ws_bytes, stream,
                       app, nullptr, kv, n);
    }
    return run_direct(kv, layer, q, gate, out, past_pos, n, stream, k_new, v_new, nullptr);
  }
  const int64_t lim0 = past_pos + 1;
  // The workspace is grown once, to the largest group's need, before any
  // launch: a growth refused under graph capture then leaves nothing of
  // this call half-recorded.
  size_t need = 0;
  for (int32_t t0 = 0; t0 < n; t0 += 4) {
    const int nq = (n - t0) < 4 ? (n - t0) : 4;
    const SplitPlan plan = plan_split(past_pos + t0 + nq, 1, kv->G, nq);
    need = std::max(need, attend_workspace_bytes(kv->G, plan.max_chunks, nq));
  }
  void* ws;
  MI_TRY(mi::kv_workspace(kv, need, stream, &ws));
  // (The one-launch form needs none, but a later captured call may count on
  // the workspace that an eager call of this size leaves.)
  if (direct)
    return run_direct(kv, layer, q, gate, out, past_pos, n, stream, k_new, v_new, nullptr);
  for (int32_t t0 = 0; t0 < n; t0 += 4) {
    const int nq = (n - t0) < 4 ? (n - t0) : 4;
    const int64_t rows = past_pos + t0 + nq;  // rows the last token of this group sees
    const int64_t qoff = (int64_t)t0 * kv->H * D;
    AppendRows app;
    if (k_new) {
      app.k = k_new + (int64_t)t0 * kv->G * D;
      app.v = v_new + (int64_t)t0 * kv->G * D;
      app.row0 = past_pos + t0;
      app.n = nq;
    }
    MI_TRY(run_split(kv->k[layer], kv->v[layer], nullptr, nullptr, rows, lim0 + t0,
                     rows, 1, kv->H, kv->G, nq, q + qoff, gate ? gate + qoff : nullptr,
                     out + qoff, ws, kv->ws_bytes, stream, app, nullptr, kv));
  }
  return MI_OK;
}

}  // namespace

namespace {
// Records the XCD each workgroup runs on (HW_REG_XCC_ID).
__global__ void xcc_probe_kernel(int* out) {
  if (threadIdx.x == 0) {
    int v;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID, 0, 4)" : "=s"(v));
    out[blockIdx.x] = v;
  }
}
}  // namespace

namespace mi {
size_t merge_state_bytes(int G) {
  return merge_counter_bytes(G) + (size_t)G * 8 * (8 * D + 64) * sizeof(float);
}

bool xcd_round_robin() {
  static std::atomic<int> known[64];  // per device: 0 unknown, 1 yes, 2 no
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return false;
  const int k = known[dev].load(std::memory_order_acquire);
  if (k) return k == 1;
  constexpr int kN = 2048;
  int* d = nullptr;
  bool ok = hipMalloc(&d, kN * sizeof(int)) == hipSuccess;
  std::vector<int> h(kN, -1);
  if (ok) {
    hipLaunchKernelGGL(xcc_probe_kernel, dim3(kN), dim3(64), 0, 0, d);
    ok = hipGetLastError() == hipSuccess &&
         hipMemcpy(h.data(), d, kN * sizeof(int), hipMemcpyDeviceToHost) == hipSuccess;
  }
  if (d) (void)hipFree(d);
  for (int b = 0; ok && b < kN; b++) ok = h[b] == b % 8;
  known[dev].store(ok ? 1 : 2, std::memory_order_release);
  return ok;
}

mi_status attend_cache(mi_kv* kv, int32_t layer, const _Float16* q, const _Float16* gate,
                       _Float16* out, int64_t past_pos, int32_t n, hipStream_t stream) {
  return cache_attend(kv, layer, q, gate, out, past_pos, n, stream);
}

bool attend_direct(mi_kv* kv, int32_t layer, const _Float16* q, const _Float16* gate,
                   _Float16* out, int64_t past, int32_t n, hipStream_t stream, mi_status* st) {
  if (!takes_direct(kv, past, n, gate, out, {{q, (size_t)n * kv->H * D * sizeof(_Float16)}}, true))
    return false;
  // Long pasts next to n: the split-K form serves them as well.  In one slice of
  // V, where the precision of its weights would have to be paid for (TILE), it is
  // the faster one: 160 tokens after 2500 rows 29.6 us against 30.8.
  const bool split = past >= 2048 && past >= 2 * (int64_t)n;
  if (split && direct_slices(kv->G, n) == 1) return false;
  // The workspace an eager split-K call of this size leaves for later captured
  // calls, although this form needs none.
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  void* ws;
  if (split && hipStreamIsCapturing(stream, &cs) == hipSuccess &&
      cs == hipStreamCaptureStatusNone &&
      (*st = mi::kv_workspace(kv, wide_launch(kv->G, past, n).ws_bytes, stream, &ws)) != MI_OK)
    return true;
  *st = run_direct(kv, layer, q, gate, out, past, n, stream, nullptr, nullptr, nullptr, true);
  return true;
}

mi_status attend_wide(mi_kv* kv, int32_t layer, const _Float16* q, const _Float16* gate,
                      _Float16* out, int64_t past, int32_t n, hipStream_t stream) {
  return wide_attend(kv, layer, q, gate, out, past, n, stream, nullptr, nullptr);
}

size_t wide_workspace_bytes(int G, int64_t past, int32_t n) {
  return wide_launch(G, past, n).ws_bytes;
}
}  // namespace mi

extern "C" mi_status mi_attn_decode(mi_kv* kv, int32_t layer, const mi_f16* q,
                                    const mi_f16* gate, mi_f16* out, int64_t seq_len,
                                    mi_stream stream) {
  mi::clear_error();
  MI_TRY(mi::check_layer(kv, layer));
  if (!q || !out) return mi::fail(MI_ERR_INVALID_ARG, "null q/out");
  if (seq_len < 0 || seq_len > kv->cap)
    return mi::fail(MI_ERR_OUT_OF_RANGE, "seq_len %lld outside [0, capacity %lld]",
                    (long long)seq_len, (long long)kv->cap);
  // seq_len == 0 runs no split work; the combine writes zeros (times the gate).
  return cache_attend(kv, layer, (const _Float16*)q, (const _Float16*)gate, (_Float16*)out,
                      seq_len - 1, 1, (hipStream_t)stream);
}

extern "C" mi_status mi_attn_step(mi_kv* kv, int32_t layer, const mi_f16* q,
                                  const mi_f16* k, const mi_f16* v, const mi_f16* gate,
                                  mi_f16* out, int64_t pos, mi_stream stream) {
  mi::clear_error();
  MI_TRY(mi::check_layer(kv, layer));
  if (!q || !k || !v || !out) return mi::fail(MI_ERR_INVALID_ARG, "null q/k/v/out");
  if (pos < 0) return mi::fail(MI_ERR_OUT_OF_RANGE, "pos=%lld", (long long)pos);
  MI_TRY(mi::kv_grow(kv, pos + 1, (hipStream_t)stream));
  MI_TRY(cache_attend(kv, layer, (const _Float16*)q, (const _Float16*)gate, (_Float16*)out, pos,
                      1, (hipStream_t)stream, (const _Float16*)k, (const _Float16*)v));
  kv->len[layer] = pos + 1;
  return MI_OK;
}

extern "C" mi_status mi_attn_verify(mi_kv* kv, int32_t layer, const mi_f16* q,
                                    const mi_f16* k, const mi_f16* v, const mi_f16* gate,
                                    mi_f16* out, int64_t past_pos, int32_t n,
                                    mi_stream stream) {
  mi::clear_error();
  MI_TRY(mi::check_layer(kv, layer));
  if (!q || !out) return mi::fail(MI_ERR_INVALID_ARG, "null q/out");
  if (!k != !v) return mi::fail(MI_ERR_INVALID_ARG, "k and v must both be given or both NULL");
  if (n <= 0) return mi::fail(MI_ERR_INVALID_ARG, "n=%d", n);
  if (past_pos < 0) return mi::fail(MI_ERR_OUT_OF_RANGE, "past_pos=%lld", (long long)past_pos);
  if (!k && past_pos + n > kv->len[layer])
    return mi::fail(MI_ERR_OUT_OF_RANGE, "k = v = NULL but rows [%lld, %lld) are not in the "
                    "cache (len %lld)", (long long)past_pos, (long long)(past_pos + n),
                    (long long)kv->len[layer]);
  MI_TRY(mi::kv_grow(kv, past_pos + n, (hipStream_t)stream));
  MI_TRY(cache_attend(kv, layer, (const _Float16*)q, (const _Float16*)gate, (_Float16*)out,
                      past_pos, n, (hipStream_t)stream, (const _Float16*)k, (const _Float16*)v));
  kv->len[layer] = past_pos + n;
  return MI_OK;
}

extern "C" size_t mi_attn_ragged_workspace_size(int32_t batch, int32_t max_len,
                                                int32_t num_q_heads, int32_t num_kv_heads,
                                                int32_t head_dim) {
  if (batch <= 0 || max_len <= 0 || num_kv_heads <= 0) return 256;
  (void)num_q_heads;
  (void)head_dim;
  const SplitPlan plan = plan_split(max_len, batch, num_kv_heads, 1);
  return ragged_workspace_bytes(batch, num_kv_heads, ragged_nwg(num_kv_heads, plan.gh));
}

extern "C" mi_status mi_attn_decode_ragged(const mi_f16* k_rows, const mi_f16* v_rows,
                                           const int32_t* offsets, const int32_t* lengths,
                                           int32_t batch, int32_t max_len,
                                           int32_t num_q_heads, int32_t num_kv_heads,
                                           int32_t head_dim, const mi_f16* q,
                                           const mi_f16* gate, mi_f16* out, void* workspace,
                                           size_t workspace_bytes, mi_stream stream) {
  mi::clear_error();
  MI_TRY(mi::check_shape(num_q_heads, num_kv_heads, head_dim));
  if (!k_rows || !v_rows || !offsets || !lengths || !q || !out || !workspace)
    return mi::fail(MI_ERR_INVALID_ARG, "null pointer argument");
  if (batch <= 0 || max_len < 0)
    return mi::fail(MI_ERR_INVALID_ARG, "batch=%d max_len=%d", batch, max_len);
  if (batch > 65535)  // the merge launch has one grid row per sequence
    return mi::fail(MI_ERR_UNSUPPORTED, "batch=%d above 65535 sequences", batch);
  const int64_t ml = max_len > 0 ? max_len : 1;
  return run_split((const _Float16*)k_rows, (const _Float16*)v_rows, offsets, lengths, ml, 0,
                   ml, batch, num_q_heads, num_kv_heads, 1, (const _Float16*)q,
                   (const _Float16*)gate, (_Float16*)out, workspace, workspace_bytes,
                   (hipStream_t)stream);
}

extern "C" mi_status mi_attn_step_proj(mi_kv* kv, int32_t layer, const float* q_proj,
                                       const float* k, const float* v,
                                       const uint16_t* q_norm_w, const uint16_t* k_norm_w,
                                       int32_t rotary_dim, float rope_theta, float eps,
                                       mi_f16* out, int64_t pos, mi_stream stream) {
  mi::clear_error();
  MI_TRY(mi::check_layer(kv, layer));
  if (!q_proj || !k || !v || !q_norm_w || !k_norm_w || !out)
    return mi::fail(MI_ERR_INVALID_ARG, "null pointer argument");
  if (pos < 0) return mi::fail(MI_ERR_OUT_OF_RANGE, "pos=%lld", (long long)pos);
  MI_TRY(mi::check_rope(kv, rotary_dim, rope_theta, eps));
  if (rotary_dim % 64)
    return mi::fail(MI_ERR_UNSUPPORTED,
                    "rotary_dim=%d: the fused step rotates whole 64-column slices; use "
                    "mi_qk_norm_rope_append + mi_attn_decode",
                    rotary_dim);
  MI_TRY(mi::kv_grow(kv, pos + 1, (hipStream_t)stream));
  ProjArgs x;
  x.q_proj = q_proj;
  x.k = k;
  x.v = v;
  x.q_w = q_norm_w;
  x.k_w = k_norm_w;
  x.rot_half = rotary_dim / 2;
  x.eps = eps;
  float inv_freq[MI_ROPE_MAX_DIM / 2];
  mi::rope_inv_freq(rope_theta, rotary_dim, inv_freq);
  const float fpos = (float)pos;
  for (int i = 0; i < x.rot_half; i++) {
    const float theta = fpos * inv_freq[i];
    sincosf(theta, &x.cs[x.rot_half + i], &x.cs[i]);
  }
  const int64_t rows = pos + 1;
  const SplitPlan plan = plan_split(rows, 1, kv->G, 1);
  void* ws;
  MI_TRY(mi::kv_workspace(kv, attend_workspace_bytes(kv->G, plan.max_chunks, 1), (hipStream_t)stream, &ws));
  const size_t q_bytes = (size_t)kv->H * 2 * D * sizeof(float);
  const size_t kv_bytes = (size_t)kv->G * D * sizeof(float), w_bytes = D * sizeof(uint16_t);
  if (takes_direct(kv, pos, 1, nullptr, (const _Float16*)out,
                   {{q_proj, q_bytes},
                    {k, kv_bytes},
                    {v, kv_bytes},
                    {q_norm_w, w_bytes},
                    {k_norm_w, w_bytes}})) {
    MI_TRY(run_direct(kv, layer, nullptr, nullptr, (_Float16*)out, pos, 1, (hipStream_t)stream,
                      nullptr, nullptr, &x));
    kv->len[layer] = pos + 1;
    return MI_OK;
  }
  AppendRows app;
  app.row0 = pos;
  app.n = 1;
  MI_TRY(run_split(kv->k[layer], kv->v[layer], nullptr, nullptr, rows, rows, rows, 1, kv->H,
                   kv->G, 1, nullptr, nullptr, (_Float16*)out, ws, kv->ws_bytes,
                   (hipStream_t)stream, app, &x, kv));
  kv->len[layer] = pos + 1;
  return MI_OK;
}

// ------------------------------------------- allocation-free ragged decode --
//
// The ragged decode's workspace (split partials + tile offsets) as a
// file-scope device array, for callers that cannot allocate.  Each device
// the library runs on holds its own copy until the process ends; host code
// reaches it only through the address hipGetSymbolAddress returns for the
// current device (the array's name in host code is not a device address).
// Nothing in it has to start at zero: the plan kernel (or, for up to
// kFusedPlan sequences, the split launch itself) writes every tile offset
// and the split kernel writes every partial slot the merge reads.
static __device__ __align__(256) unsigned char scratch[MI_NOALLOC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch_ptr[kMaxDevices];

// The current device's copy of `scratch`, looked up once per device.  The
// launch stream must belong to the current device: the copy is per device.
mi_status scratch_ptr(hipStream_t stream, void** out) {
  int dev = 0;
  MI_HIP(hipGetDevice(&dev));
  if (stream) {
    int sdev = 0;
    MI_HIP(hipStreamGetDevice(stream, &sdev));
    if (sdev != dev)
      return mi::fail(MI_ERR_INVALID_ARG, "stream on device %d, current device %d", sdev, dev);
  }
  if (dev < 0 || dev >= kMaxDevices)
    return mi::fail(MI_ERR_UNSUPPORTED, "device %d beyond the %d the library tracks", dev,
                    kMaxDevices);
  void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (!p) {
    MI_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_ptr[dev].store(p, std::memory_order_release);
  }
  *out = p;
  return MI_OK;
}
}  // namespace

extern "C" mi_status mi_attn_decode_ragged_noalloc(
    const mi_f16* k_rows, const mi_f16* v_rows, const int32_t* offsets, const int32_t* lengths,
    int32_t batch, int32_t max_len, int32_t num_q_heads, int32_t num_kv_heads,
    int32_t head_dim, const mi_f16* q, const mi_f16* gate, mi_f16* out, mi_stream stream) {
  mi::clear_error();
  MI_TRY(mi::check_shape(num_q_heads, num_kv_heads, head_dim));
  if (batch <= 0 || max_len < 0)
    return mi::fail(MI_ERR_INVALID_ARG, "batch=%d max_len=%d", batch, max_len);
  const size_t need =
      mi_attn_ragged_workspace_size(batch, max_len, num_q_heads, num_kv_heads, head_dim);
  if (need > (size_t)MI_NOALLOC_SCRATCH_BYTES)
    return mi::fail(MI_ERR_UNSUPPORTED,
                    "batch=%d needs %zu bytes of scratch; the static scratch holds %zu "
                    "(use mi_attn_decode_ragged with a workspace)",
                    batch, need, (size_t)MI_NOALLOC_SCRATCH_BYTES);
  void* ws = nullptr;
  MI_TRY(scratch_ptr((hipStream_t)stream, &ws));
  return mi_attn_decode_ragged(k_rows, v_rows, offsets, lengths, batch, max_len, num_q_heads,
                               num_kv_heads, head_dim, q, gate, out, ws,
                               (size_t)MI_NOALLOC_SCRATCH_BYTES, stream);
}
