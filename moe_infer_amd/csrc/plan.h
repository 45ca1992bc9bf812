// Launch plans shared by the kernels, their host launchers and the CPU
// model of their memory accesses (tests/copy_bounds_model.cc compiles this
// header with g++): the causal prefill's per-wave tile schedule and the
// split-K decode's chunking.  Plain C++ with no HIP dependency.
#pragma once

#include <cstdint>

#if defined(__HIPCC__)
#define MI_HD __host__ __device__
#else
#define MI_HD
#endif

namespace mi {

// ------------------------------------------------------------- prefill --

constexpr int kPrefillBQ = 128;  // queries per workgroup (4 waves of 32)
constexpr int kPrefillBK = 64;   // keys per LDS tile

// The key-tile range of one wave of the causal prefill: the wave owns
// queries q0 + 32 w .. + 31 of query tile `qtile` (positions past + i), and
// its workgroup walks key tiles 0 .. nt-1 (64 keys each) up to the last
// key any of its queries sees.  Positions are 32-bit (the host checks
// past + n + 2 * kPrefillBK < 2^31).
struct PrefillWave {
  int first;   // smallest query position of the wave
  int last;    // largest query position of the wave (may be >= kv_len: padding)
  int kv_len;  // rows in the cache after the append: past + n
  int nt;      // key tiles the workgroup walks
};

MI_HD inline PrefillWave prefill_wave(int past, int n, int qtile, int w) {
  PrefillWave p;
  const int q0 = qtile * kPrefillBQ;
  p.first = past + q0 + 32 * w;
  p.last = p.first + 31;
  p.kv_len = past + n;
  const int end = past + q0 + kPrefillBQ < p.kv_len ? past + q0 + kPrefillBQ : p.kv_len;
  p.nt = (end + kPrefillBK - 1) / kPrefillBK;
  return p;
}

// Tile t of the wave's walk: does the wave attend it (some query sees a key
// of it), is it on the wave's diagonal (needs the causal mask), and does it
// take the steady-state schedule?  The steady schedule copies K(t+1) into
// LDS unconditionally, so it is taken only when t + 1 < nt: a wave whose
// queries all lie past n (padding of the last query tile) has its diagonal
// beyond the last tile, so "not diagonal" alone would let it copy K(nt),
// 64 rows past kv_len and possibly past the allocation.  Every other tile
// copies K(t+1) only when t + 1 < nt, and V(t).
MI_HD inline bool prefill_active(const PrefillWave& p, int t) {
  return t * kPrefillBK <= p.last;
}
MI_HD inline bool prefill_diag(const PrefillWave& p, int t) {
  return t * kPrefillBK + kPrefillBK - 1 > p.first;
}
MI_HD inline bool prefill_steady(const PrefillWave& p, int t, bool pending) {
  return prefill_active(p, t) && pending && !prefill_diag(p, t) && t + 1 < p.nt;
}

// The 64-queries-per-wave form (attn_prefill64_kernel): wave (qb, kp) owns
// queries q0 + 64 qb .. + 63 and keys 32 kp .. 32 kp + 31 of every 64-key
// tile; the workgroup walks the same nt tiles as above.
struct PrefillWave64 {
  int first, last, kv_len, nt;
  int koff;  // 32 kp: the wave's key half of a tile
};

MI_HD inline PrefillWave64 prefill_wave64(int past, int n, int qtile, int qb, int kp) {
  PrefillWave64 p;
  const int q0 = qtile * kPrefillBQ;
  p.first = past + q0 + 64 * qb;
  p.last = p.first + 63;
  p.kv_len = past + n;
  const int end = past + q0 + kPrefillBQ < p.kv_len ? past + q0 + kPrefillBQ : p.kv_len;
  p.nt = (end + kPrefillBK - 1) / kPrefillBK;
  p.koff = 32 * kp;
  return p;
}
// The wide verify's form of the same: the workgroup's keys are chunk
// [kbeg, kbeg + chunk) of [0, past + n), positions relative to kbeg; its
// row block holds tokens tok0 .. tok0 + 15, rows 64 qb .. + 63 being tokens
// tok0 + 8 qb .. + 7 (each with the group's eight heads), token i seeing
// keys up to past + i.  Only chunks that hold keys of the block are launched
// (wide_place).
MI_HD inline PrefillWave64 verify_wave64(int64_t past, int n, int64_t kbeg, int64_t chunk,
                                         int tok0, int qb, int kp) {
  PrefillWave64 p;
  p.first = (int)(past - kbeg) + tok0 + 8 * qb;
  p.last = p.first + 7;
  const int tend = n < tok0 + 16 ? n : tok0 + 16;  // the block's tokens
  int64_t end = past + tend - kbeg;                 // keys they see in the chunk
  if (end > chunk) end = chunk;
  p.kv_len = (int)end;
  p.nt = (p.kv_len + kPrefillBK - 1) / kPrefillBK;
  p.koff = 32 * kp;
  return p;
}
MI_HD inline bool prefill64_active(const PrefillWave64& p, int t) {
  return t * kPrefillBK + p.koff <= p.last;
}
MI_HD inline bool prefill64_diag(const PrefillWave64& p, int t) {
  return t * kPrefillBK + p.koff + 31 > p.first;
}
// As prefill_steady: the steady schedule copies K(t+1), so t + 1 < nt.
MI_HD inline bool prefill64_steady(const PrefillWave64& p, int t, bool pending) {
  return prefill64_active(p, t) && pending && !prefill64_diag(p, t) && t + 1 < p.nt;
}

// ----------------------------------------------------------- split-K --

// The 32-key tiles wave w of nwh reads in a chunk [begin, end): a
// contiguous run of ceil(tiles / nwh) tiles from first, while k0 < last.
struct WaveTiles {
  int64_t first, last;
};
MI_HD inline WaveTiles split_wave_tiles(int64_t begin, int64_t end, int nwh, int w) {
  const int64_t per = ((end - begin + 31) / 32 + nwh - 1) / nwh;
  WaveTiles r;
  r.first = begin + 32 * per * w;
  const int64_t e = begin + 32 * per * (w + 1);
  r.last = e < end ? e : end;
  return r;
}

// Most chunks (partials) per sequence of one split launch.
constexpr int kMaxSplitChunks = 1024;

// The wide verify / split-K prefill (attn_verify_wide_kernel): one workgroup
// per KV head, row block rb of 16 tokens and chunk c that holds keys the
// block's tokens see, rows [0, end(rb)).  As items, whole chunks come first, then
// every block's last chunk, the latest block first.  No item is empty: an empty
// grid index takes a place in the round-robin over the XCDs from a workgroup,
// which then waits for another's whole chunk (with empty ones among the last
// chunks, 672 tokens after 1260 rows took 56.7 us, without 41.5).
MI_HD inline int wide_end(int past, int n, int rb) {
  return past + (n < 16 * rb + 16 ? n : 16 * rb + 16);
}
// Row blocks with a whole chunk c and keys after it: [wide_first(c), nrb).
MI_HD inline int wide_first(int past, int n, int chunk, int c) {
  const int nrb = (n + 15) / 16;
  const int x = (int)((int64_t)(c + 1) * chunk - past);  // new tokens up to the chunk's end
  if (x >= n) return nrb;
  return x <= 0 ? 0 : x / 16;
}
MI_HD inline int wide_count(int past, int n, int chunk) {  // workgroups
  const int nrb = (n + 15) / 16;
  int c = past / chunk;  // chunks whole for every block
  int items = c * nrb + nrb;
  for (; wide_first(past, n, chunk, c) < nrb; c++) items += nrb - wide_first(past, n, chunk, c);
  return items;
}
// Item idx of [0, wide_count): its row block and chunk.
MI_HD inline void wide_item(int past, int n, int chunk, int idx, int& rb, int& c) {
  const int nrb = (n + 15) / 16;
  int cc = past / chunk;
  if (idx < cc * nrb) {
    c = idx / nrb;
    rb = nrb - 1 - (idx - c * nrb);
    return;
  }
  idx -= cc * nrb;
  for (;; cc++) {
    const int first = wide_first(past, n, chunk, cc);
    if (first >= nrb) break;
    if (idx < nrb - first) {
      c = cc;
      rb = nrb - 1 - idx;
      return;
    }
    idx -= nrb - first;
  }
  rb = nrb - 1 - idx;
  c = (wide_end(past, n, rb) - 1) / chunk;
}

// How the workgroups are dealt to the XCDs (blockIdx % 8):
//   pitch > 0  (row block, chunk, KV head), the head fastest; pitch = chunks *
//              heads (a last chunk that a block lacks is left empty: only where
//              all still run at once)
//   run > 0    each XCD takes a run of `run` items in (head, chunk, row block)
//              order, so that the blocks of a chunk, which read the same K/V,
//              share its L2
//   else       (item, KV head), the head fastest: the blocks of a chunk one
//              after the other
// What decides is the K and V of all heads that the blocks share, and whether by
// block a chunk's blocks fall on one XCD (a pitch of whole rounds) as well.
// Measured (us, by block / runs / by item, from HBM; two KV heads): 17 tokens after
// 3500 rows 25.3 / 26.0 / 24.7, after 9000 25.3 / 27.8 / 26.6, after 20000 30.9 / 29.0
// / 32.5, after 65000, where the pitch is whole rounds, 52.0 / 53.0 / -; 49 after
// 12000 (whole rounds) 35.1 / 35.7 / 39.7; 51 after 49354 83.6 / 72.8 / 85.5; 128 after
// 8000 37.4 / 38.2 / 35.6, after 64000 136.3 / 136.2 / 139.2; 1 head, 28 after 12832 29.0
// / 31.3 / 28.5; 3 heads, 71 after 11540 51.4 / 45.2 / 50.7.  The lines below are where
// the means of 1800 sizes of 1 to 8 heads cross: in whole rounds by block takes
// 1.01 to 1.05 of by item below 18000 and 0.88 to 0.99 above; else by block is up to
// 5 % ahead of the others from 8000 or 13000 on, runs above 13000 to 24000.
// A single row block (a verify of up to 16 tokens) goes by block: its look-up is a
// division, the others' would cost it 0.4 of 35 us.
struct WideDeal {
  int items;  // wide_count: workgroups per KV head
  int pitch, run;
  int grid;  // workgroups launched
};
// Every block has every chunk.
inline bool wide_full(int64_t past, int n, int64_t chunk, int nchunks) {
  return wide_end((int)past, n, 0) > (int64_t)(nchunks - 1) * chunk;
}
inline WideDeal wide_deal(int G, int64_t past, int n, int64_t chunk, int nchunks) {
  WideDeal d;
  d.items = wide_count((int)past, n, (int)chunk);
  d.pitch = d.run = 0;
  d.grid = d.items * G;
  const int nrb = (n + 15) / 16;
  const int64_t kv = G * past;
  const bool shared = nchunks * G % 8 == 0;  // by block, a chunk's blocks are on one XCD
  const bool fits = nrb <= 8 && nrb * nchunks * G <= 256;
  // (2, 4 and 8 heads fall on the XCDs in turn: each reads one head's K/V, and gains
  // from runs later)
  const bool spread = G == 1 || 8 % G;
  const bool far = kv >= (nrb == 2 && !shared ? 24000 : nrb > 4 && spread ? 13000 : 18000);
  if (nrb == 1 || (fits && (shared ? far : !far && kv >= (nrb < 4 ? 13000 : 8000)))) {
    d.pitch = nchunks * G;
    d.grid = nrb * d.pitch;
  } else if (far) {
    d.run = (d.grid + 7) / 8;
    d.grid = 8 * d.run;
  }
  return d;
}
// Workgroup `block`'s row block, chunk and KV head; false for none.
MI_HD inline bool wide_place(const WideDeal& d, int G, int past, int n, int chunk, int block,
                             int& rb, int& c, int& kvh) {
  if (d.pitch) {
    rb = block / d.pitch;
    const int u = block - rb * d.pitch;
    c = u / G;
    kvh = u - c * G;
    return c * chunk < wide_end(past, n, rb);
  }
  const int idx = d.run ? (block & 7) * d.run + (block >> 3) : block;
  const int per = d.run ? d.items : G;
  const int hi = idx / per, lo = idx - hi * per;
  kvh = d.run ? hi : lo;
  if (kvh >= G) return false;
  wide_item(past, n, chunk, d.run ? lo : hi, rb, c);
  return true;
}

// Its chunking: whole 64-key tiles, at most kMaxSplitChunks chunks (the merge
// kernels' limit), and the smallest chunk whose workgroups all run at once (256
// CUs): one more than that waits for a whole chunk.  Measured after 1000 rows,
// 1000 tokens: chunks of 704 keys (more than 256 workgroups) 68 us, of 1024
// (250) 53; after 2000 rows, 500 tokens: 448 keys 60, 640 (256) 42, 832 44.
// More than 16 (256 / G) tokens cannot fit: one chunk.
struct WidePlan {
  int64_t chunk;
  int nchunks;
};
inline WidePlan wide_plan(int G, int64_t past, int n) {
  const int64_t rows = past + n, nrb = ((int64_t)n + 15) / 16;
  const int64_t most = nrb * G > 256 ? nrb : 256 / G;  // workgroups per KV head
  const int64_t keys = nrb * past + 8 * nrb * (nrb + 1);  // at least about this many to deal out
  int64_t chunk = keys / most;
  const int64_t min_chunk = (rows + kMaxSplitChunks - 1) / kMaxSplitChunks;
  if (chunk < min_chunk) chunk = min_chunk;
  chunk = (chunk + kPrefillBK - 1) / kPrefillBK * kPrefillBK;
  if (chunk < kPrefillBK) chunk = kPrefillBK;
  while (chunk < rows && wide_count((int)past, n, (int)chunk) > most) chunk += kPrefillBK;
  WidePlan p;
  p.chunk = chunk;
  p.nchunks = (int)((rows + chunk - 1) / chunk);
  return p;
}

// Whether n query tokens after `past` rows are served by the one-launch form
// (attn_direct_kernel).  Its time grows with the rows one workgroup walks and,
// once the CUs are taken, with the keys of all tokens; the split launches cost
// about 10 us whatever the length.
// Up to 16 tokens, measured from HBM (us, one launch against the split forms):
// 1 token at 517 rows 7.1 / 10.9, at 1000 9.4 / 10.8, at 1100 13.2 / 10.9; 4
// tokens at 1000 9.7 / 15.5, at 1500 16.1 / 14.4; 8 at 1500 15.5 / 15.9; 12 at
// 1500 15.1 / 16.8, at 2000 19.3 / 16.9; 16 at 1500 15.1 / 18.0, at 2000 19.5 /
// 18.2.
// More tokens, without their append (against the prefill grid / the split-K
// pass), two KV heads: 64 after 1000 rows 10.4 / 35.3 / 24.2, 128 after 3000 27.8 /
// 82.2 / 28.9, 400 after 1000 30.3 / 45.1 / 32.8, 777 from none 25.5 / 30.9 / 42.3;
// past the line: 300 after 1500 35.3 / 53.6 / 31.5, 1024 from none 36.6 / 37.0
// / 36.6, 17 after 5000 33.6 / 119.7 / 25.0.
// A prompt's line falls with the square of the KV heads: each adds its own
// workgroups here, while those it adds to the grid find idle CUs (one launch
// against the better of grid and split-K): 3 heads, 606 from none 31.1 / 33.1, 685
// 32.8 / 32.5; 4 heads, 387 from none 24.4 / 26.0, 558 33.3 / 31.6, 959 after 20 61.2
// / 42.9; 6 heads, 257 from none 21.1 / 23.4, 318 29.0 / 27.2; 8 heads, 200 from none
// 20.4 / 21.7, 277 30.6 / 27.9, 876 94.9 / 57.9.  The alternative of a verify is the
// split-K pass, which they add to as well: 4 heads, 125 after 1303 26.4 / 34.3, 129
// after 1610 41.8 / 39.3; 8 heads, 203 after 1221 61.0 / 46.5; and where a workgroup
// walks far: 8 heads, 59 after 966 22.7 / 33.1, 25 after 3017 44.2 / 38.6.
inline bool direct_rows(int G, int64_t past, int32_t n, bool prefill) {
  const int64_t rows = past + n, keys = n * (past + n / 2);
  if (n <= 4) return rows <= 1024 + 80 * (n - 1);
  if (n <= 16) return rows <= 1400 + 21 * n;
  if (rows > 3200 || keys > 480000) return false;
  return prefill ? keys * G * G <= 2200000 && n * G <= 2080 - 60 * G
                 : keys * G <= (G <= 2 ? 960000 : 860000) && rows * G <= 18000;
}

// Whether a verify of 5 to 16 tokens outside that runs as groups of four tokens
// in one split launch (and one merge, the append inside) rather than in the
// wide pass (append, pass, merge).  Every group reads the whole cache, but from
// L2 and the last-level cache after the first, and a workgroup of the wide pass
// has 8 us of Q and first tile and 6 us of epilogue.  Measured from HBM (us,
// groups / wide): 8 tokens after 2300 rows 16.1 / 20.7, after 9001 18.8 / 26.0,
// after 24000 27.6 / 28.2; 12 after 9001 19.8 / 30.9; 9 after 24000 31.0 / 29.7;
// 16 after 16000 26.0 / 33.4, after 32000 40.2 / 38.1, after 65536 100 / 49.
// More heads leave fewer chunks to a group, and where a head's chunks do not fall
// on the XCDs in turn, or three groups do not, L2 serves less of the rereads: 3
// heads, 11 after 12177 rows 26.8 / 33.4, 13 after 13436 39.9 / 33.6; 4 heads, 11
// after 16723 35.1 / 37.3 (given up for 10 after 10727, 32.1 / 29.9); 6 heads, 16
// after 4907 32.5 / 37.1, 15 after 5740 42.5 / 37.1, 8 after 8846 28.3 / 34.1, 6 after
// 12924 38.4 / 35.0; 8 heads, 9 after 6126 33.6 / 39.9, 10 after 7870 39.5 / 37.8, 16
// after 7465 45.1 / 49.9 (given up for 13 after 6228, 44.3 / 41.1), after 12960 57.5 /
// 49.9.
inline bool verify_groups(int G, int64_t past, int32_t n) {
  const int64_t rows = past + n, ng = (n + 3) / 4;
  return n <= 16 && rows <= 20480 &&
         rows * G * ng <= (8 % G ? 110000 : ng == 3 ? 163840 : 196608);
}

// Whether a prefill outside that takes the split-K pass and its merge rather
// than the prefill grid (one workgroup per 128 queries and head): the grid is
// short of workgroups and each walks the whole past.  Measured, split-K
// against the grid (us): 512 tokens after 1024 rows 34.3 / 46.8, 600 after 600
// 33.3 / 38.8, 640 after 480 32.7 / 38.8, 777 after 777 40.4 / 50.4, 850 after
// 850 44.0 / 50.4, 960 after 960 47.8 / 54.0, 1024 after 1024 49.5 / 58.0, 512
// after 16384 139 / 377.  Nowhere in 300 sizes of 100 to 1024 tokens did the
// grid win; below the line the lead shrinks with the past (777 after 291 34.4 /
// 38.1, 1024 from none 33.9 / 35.6), and with more tokens no CU is idle (1200
// from none 39.2 / 39.1).  That is for up to two KV heads; with more the grid has
// more workgroups and wins up to longer pasts: 4 heads, 630 after 993 62.6 / 58.4,
// 432 after 362 39.9 / 37.3; 6 heads, 360 after 1036 56.3 / 51.0; 8 heads, 175 after
// 263 38.6 / 32.7, 179 after 628 43.8 / 40.7; split-K takes 0.95 of the grid's time at
// 477 after 980 (4 heads), 0.78 at 188 after 1356 (6), 0.97 at 190 after 1059 (8), and
// loses where only some blocks get a second chunk (8 heads, 302 after 1482 75.2 /
// 64.3).
inline bool prefill_split_rows(int G, int64_t past, int32_t n) {
  if (n > 1024) return false;
  if (G <= 2) return past >= (n <= 640 ? n / 2 : n);
  return past >= (int64_t)n * G / 2 && past >= 125 * G && (n * G <= 2048 || past >= 2048);
}

struct SplitKnobs {
  int gh;     // KV heads per workgroup (2, or 1 when set to 1)
  int wgs;    // target workgroup count
  int chunk;  // fixed keys per chunk (0: planned)
};

struct SplitPlan {
  int nwh, gh, ncb, chunk, max_chunks;
};

// Kernel variant and chunking of one split launch over sequences of at
// most max_len rows.  Keys per chunk (per head): enough workgroups to
// cover 256 CUs about once (K/V of one key and head is 1 KiB, so a 128-key
// chunk of two heads moves 256 KiB and leaves one 8 KiB partial per head and
// query token), at least one 32-key tile, at most 2048 keys (ragged batches
// balance better with more workgroups), and at most kMaxSplitChunks chunks.
// Chunks are whole 32-key tiles; each wave of a workgroup takes a contiguous run
// of its tiles.  Decode rounds chunks to 32 keys: rounding up to 32 * NWH
// would leave up to half the CUs idle just above a power of two (ctx 32769:
// 129 workgroups instead of 256, 21.0 against 18.1 us per call).  The
// 32-column verify (nq > 2) keeps whole wave rounds (measured ~1 us faster
// at 65540 rows: 206 workgroups of 20 tiles against 242 of 17).
inline SplitPlan plan_split(int64_t max_len, int64_t batch, int G, int nq, const SplitKnobs& k) {
  SplitPlan p;
  p.ncb = nq <= 2 ? 1 : 2;
  if (p.ncb == 2) {  // 32 columns: 4 waves, one head (registers and LDS)
    p.nwh = 4;
    p.gh = 1;
  } else if (G % 2 == 0 && k.gh == 2) {
    p.nwh = 4;
    p.gh = 2;
  } else {
    p.nwh = 8;
    p.gh = 1;
  }
  const int64_t step = 32 * p.nwh;
  const int64_t target_wgs = k.wgs > 0 ? k.wgs : 1;
  int64_t chunk = k.chunk;
  if (chunk <= 0) {
    chunk = (batch * G * max_len + p.gh * target_wgs - 1) / (p.gh * target_wgs);
    if (chunk > 2048) chunk = 2048;
  }
  const int64_t min_chunk = (max_len + kMaxSplitChunks - 1) / kMaxSplitChunks;
  if (chunk < min_chunk) chunk = min_chunk;
  const int64_t gran = p.ncb == 2 ? step : 32;
  chunk = (chunk + gran - 1) / gran * gran;
  if (chunk < gran) chunk = gran;  // also for max_len == 0
  p.chunk = (int)chunk;
  p.max_chunks = (int)((max_len + chunk - 1) / chunk);
  if (p.max_chunks < 1) p.max_chunks = 1;
  return p;
}

// Chunking of a verify by `ng` groups of four tokens (the split launch's z
// planes): chunks whose workgroups all run at once, not one more (9 tokens after
// 16300 rows in 43 chunks of two heads, 258 workgroups, took 38.2 us, in 32
// chunks 25.8), and a chunk count, padded with empty chunks where those still
// fit, that puts the groups of a chunk on one XCD (blockIdx % 8), whose L2 then
// reads its K/V once: 13 tokens after 19314 rows in 31 chunks 37.0 us, padded to
// 32 29.0; after 17000 rows in 27 chunks 33.9, padded to 28 28.4.
inline SplitPlan plan_groups(int64_t rows, int ng, int G, const SplitKnobs& k) {
  SplitPlan p = plan_split(rows, ng, G, 4, k);
  const int step = 32 * p.nwh, wgs = 256;
  if (k.chunk <= 0)
    while (p.max_chunks * ng * G > wgs && p.chunk < rows) {
      p.chunk += step;
      p.max_chunks = (int)((rows + p.chunk - 1) / p.chunk);
    }
  int lanes = 8;  // chunks to a round of the XCDs
  while (lanes > 1 && lanes / 2 * G % 8 == 0) lanes /= 2;
  const int padded = (p.max_chunks + lanes - 1) / lanes * lanes;
  if (padded * ng * G <= wgs) p.max_chunks = padded;
  return p;
}

}  // namespace mi
