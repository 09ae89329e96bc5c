// The wide pass of top-p and temperature-only rows: device code of the
// chunked path's finish kernel (sampler_chunked.hip), and the general
// per-row path.
#pragma once
#include "sampler_select.h"

namespace hi_rocm {

// ==========================================================================
// Wide pass: rows that need their whole distribution (gpu.rs:820-899 with
// top_k unset; kernels.cu:7803-7867), chunk-parallel
// ==========================================================================
//
// The select pass leaves the scaled logits s in ws_s and, for top-p rows, a
// mass histogram per chunk (WideStat); then one workgroup per (chunk, row):
//   1. merges the row's chunk maxima (M) and histograms (wide_row_stats,
//      every workgroup of the row alike): a conservative weight bound w_lo
//      such that the weights >= w_lo hold at least cutoff + kWideMargin of
//      the mass, and the predicted sum before the chunk;
//   2. computes its weights w = expf(s - M) exactly (min-p zeros them), in
//      tiles of 1024 logits, and each tile's map in the vocabulary-order fold
//      for the binade its predicted start lies in (sampler_draw.h);
//   3. lists its weights >= w_lo with their indexes (bf16 logits: their
//      distinct values with counts, an LDS hash: thousands of logits share
//      one weight); f32 weights that turn out to share values in a sample
//      are counted by value as well (f32 logits that hold bf16 values, or
//      few levels);
//   4. bumps the row's counter; the last workgroup finishes the row: wave 0
//      chains the tile maps into the exact normaliser while the others
//      gather the lists, then the ranks are sorted and folded (draw_ranks;
//      bf16, and long f32 lists of few values: runs of equal weights in
//      closed form, wide_finish_runs).
// A temperature-only row's workgroups sum its 256 reference chunks instead, a
// quad of lanes a chunk, and the last one draws.
// Rows whose chunks took the select pass's exact path, whose nucleus is not
// inside the listed weights, or of more than 256 units take finish_row.
//
// A workgroup takes a unit of one or several select chunks (WideUnits): every
// workgroup of a row repeats the row statistics (about 5 us), so fewer and
// larger units win.
//
// Measured against the form before it (a workgroup's weights and maps held
// in LDS with crossing records, distinct weights in LDS hash tables, runs
// folded in closed form for every type): 32 bf16 nucleus rows of 151,936
// beside 32 greedy ones 147 -> 118 us, 32 masked f32 nucleus rows 158-883 ->
// 86 us (the tables overflowed on some), 64 nucleus rows 247 -> 122 us, with
// spiked logits 8,253 -> 249 us; 64 temperature-only rows 483 -> 60 us.
// Bound now: the chain of exact tile folds (about 14 us) and the sort and
// folds (about 10 us) of a row's last workgroup, one workgroup each, and the
// select pass before them (16-20 us).
constexpr float kWideMargin = 0.005f;  // extra probability mass of the superset
constexpr int kWideGBins = 64;         // threshold bins (binades of w below M)
constexpr int kWideTile = 64 * kDrawPer;
constexpr int kWideHash = 2048;        // distinct superset weights of a chunk, and of a row
constexpr int kWideLog2 = 11;
static_assert((1 << kWideLog2) == kWideHash, "hash size");
constexpr int kWideProbes = 64;
// A row of distinct weights whose list exceeds V / kWideListShare takes
// finish_row: 64 f32 nucleus rows of 151,936, about everything listed 8,830 us
// by the list and 2,831 by the row, about a seventh 418 and 537.
constexpr int kWideListShare = 4;
constexpr int kWidePre = kSelChunkLarge / kWideTile / (NT / 64);  // tiles of a wave, at most
static_assert(kSelChunkLarge / kWideTile == kChunkTiles, "a chunk's tile records");

// A row's units of the wide pass.
struct WideUnits {
  int n;       // of a row (at most its chunks)
  int len;     // logits of one
  int chunks;  // select chunks of one
};
__host__ __device__ inline WideUnits wide_units(int chunk, int n_chunks) {
  // units of kSelChunkLarge logits.  Units of one small chunk (one and four,
  // nucleus): 14 f32 rows of 151,936 353 and 332 us, 26 rows 412 and 358; 20
  // bf16 rows 116 and 99; 40 rows of 50,257 88 and 89, 56 rows 105 and 95,
  // 80 rows 142 and 107 (smaller batches take one launch)
  const int g = chunk < kSelChunkLarge ? kSelChunkLarge / chunk : 1;
  return WideUnits{(n_chunks + g - 1) / g, chunk * g, g};
}

// LDS of a (unit, row) workgroup.
struct WideChunkLds {
  float tr[NT / 64][64 * kTrLd];         // a wave's tile, turned
  uint64_t exptab[32];                   // exact_expf's table (wide_row_stats copies it)
  unsigned long long gmass[kWideGBins];  // wide_row_stats
  unsigned long long predfx;
  float w_lo;
  float tsum[kChunkTiles];
  uint32_t wcnt[NT / 64];
  uint32_t n, nr, last;
  // the superset's distinct weights
  uint32_t hkey[kWideHash], hcnt[kWideHash], hmin[kWideHash];
};

// LDS of the row finish over runs of equal weights.
struct WideRunLds {
  fold::WgLds<NT> fl;
  union {
    struct {
      uint32_t hkey[kWideHash];
      uint32_t hcnt[kWideHash];
      uint32_t hmin[kWideHash];
      uint64_t sortk[kWideHash];
    } mg;
    struct {
      float rx[kWideHash];     // weight of run r (rank order)
      uint32_t rm[kWideHash];  // its multiplicity
      uint32_t ri[kWideHash];  // its smallest index
      float st[kWideHash];     // cum_p before run r
      float st2[kWideHash];    // candidate weight sum before run r
    } fo;
  } u;
  uint8_t pe[kWideHash + 4];
  uint32_t noff[kDrawChunks + 1];
  uint32_t cntc[kDrawChunks];  // the drawn weight's multiplicity per chunk
  uint8_t listed[kDrawChunks];  // the unit's entries are its list (else runs)
  uint32_t cnt, rsel, csel, tok;
};

__device__ __forceinline__ uint32_t wide_hash(uint32_t key, int log2n) {
  return (key * 0x9E3779B1u) >> (32 - log2n);
}

// Inserts `count` copies of weight bits `key` with smallest index `idx`
// into an LDS table of 2^log2n slots (key 0 = empty; weights here are > 0).
// Returns false when kWideProbes slots in a row hold other weights (a table
// that fills up would otherwise be searched end to end for every weight); a
// thread soon inserts nothing more then.
__device__ __forceinline__ bool wide_insert(uint32_t* hkey, uint32_t* hcnt, uint32_t* hmin, int log2n,
                                            uint32_t key, uint32_t count, uint32_t idx) {
  const uint32_t mask = (1u << log2n) - 1u;
  uint32_t h = wide_hash(key, log2n);
  #pragma unroll 1
  for (int probe = 0; probe < kWideProbes; ++probe, h = (h + 1u) & mask) {
    const uint32_t old = atomicCAS(&hkey[h], 0u, key);
    if (old == 0u || old == key) {
      atomicAdd(&hcnt[h], count);
      atomicMin(&hmin[h], idx);
      return true;
    }
  }
  return false;
}

// A wave's tiles of the chunk [c0, c1) (tile wid, wid + 4, ...): 16 scaled
// logits a lane and tile, loaded by wide_row_stats behind its own loads, so
// that their latency hides behind the statistics.
__device__ __forceinline__ void wide_preload(const DrawRow& r, int c0, int c1, i32x4_t (&pre)[kWidePre][4]) {
  const int lane = (int)(threadIdx.x & 63u), wid = (int)(threadIdx.x >> 6);
  #pragma unroll
  for (int i = 0; i < kWidePre; ++i) {
    const int t0 = c0 + (i * (NT / 64) + wid) * kWideTile;
    if (t0 < c1) {
      #pragma unroll
      for (int j = 0; j < 4; ++j) pre[i][j] = __builtin_amdgcn_raw_buffer_load_b128(r.s, (t0 + j * 256 + lane * 4) * 4, 0, 0);
    }
  }
}

// Step 1, by every workgroup of a top-p row's chunk work: the row max of s
// (M), the superset bound w_lo and the predicted fold value before this
// workgroup's chunk, from the chunks' statistics the select pass wrote
// (WideStat).  The masses use approximate exp; they only size the superset
// and predict binades.  valid = 0: a chunk's statistics were not written by
// this call's pass, or no logit is finite (the row takes finish_row).  The
// row's finishing workgroup clears the chunks' valid flags afterwards.
struct WideRowStats {
  float M, w_lo;
  uint32_t valid;
  double pred;  // the predicted fold value before the unit
};
__device__ __forceinline__ WideRowStats wide_row_stats(WideChunkLds& L, const SampleArgs& a, int row,
                                                      const WideUnits& wu, int unit, const RowCfg& cfg,
                                                      const DrawRow& r, i32x4_t (&pre)[kWidePre][4]) {
  const int tid = threadIdx.x;
  const int nch = a.n_chunks;
  const ChunkStat* stats = a.stats + (int64_t)row * nch;
  const WideStat* wst = a.wstat + (int64_t)row * nch;
  // the loads of the first kU * NT (chunk, bin) items go out with those of
  // the chunk maxima
  constexpr int kU = 8;
  float hv0[kU], ms0[kU];
  {
    const int items0 = nch * kWideBins;
    #pragma unroll
    for (int k = 0; k < kU; ++k) {
      const int it = k * NT + tid;
      hv0[k] = 0.f;
      ms0[k] = 0.f;
      if (it < items0) {
        const WideStat& ws = wst[it / kWideBins];
        hv0[k] = ws.hist[it % kWideBins];
        ms0[k] = ws.ms;
      }
    }
  }
  // the chunk maxima and valid flags (chunks tid, tid + NT, ...): the first
  // round goes out with the loads above; then the chunk's scaled logits,
  // behind all of them, so that waiting for the statistics' loads does not
  // wait for these
  float ml0 = 0.f;
  uint32_t v0 = 1u;
  if (tid < nch) {
    ml0 = stats[tid].max_l;
    v0 = wst[tid].valid;
  }
  wide_preload(r, unit * wu.len, min((unit + 1) * wu.len, a.V), pre);
  uint32_t mk = tid < nch ? okey(ml0) : 0u, bad = tid < nch ? v0 ^ 1u : 0u;
  for (int c = tid + NT; c < nch; c += NT) {
    mk = max(mk, okey(stats[c].max_l));
    bad |= wst[c].valid ^ 1u;
  }
  if (tid < kWideGBins) L.gmass[tid] = 0ull;
  if (tid == 0) L.predfx = 0ull;
  if (tid < 32) L.exptab[tid] = exp2_tab32((uint32_t)tid);
  mk = block_max_u32<NT>(mk, L.wcnt);
  bad = block_max_u32<NT>(bad, L.wcnt);
  const float ml = okey_inv(mk);
  const float M = finitef_(ml) ? ml / cfg.t_eff : -__builtin_inff();
  if (!finitef_(M) || bad) return WideRowStats{M, 0.f, 0u, 0.0};
  // chunk masses relative to M, in fixed point (2^-32): per binade of their
  // lower end (for w_lo) and, for the chunks before this one and for this
  // one, their sums (the prediction): each thread adds its bins' shares,
  // then one wave reduction and an atomic per wave (integer sums, exact in
  // any order)
  static_assert(kWideBins == 32, "a chunk's bins are one half of a wave");
  static_assert(kWideGBins == 64, "one bin per lane");
  const int items = nch * kWideBins;
  unsigned long long bef = 0ull;
  for (int base = 0; base < items; base += kU * NT) {
    float hv[kU], msv[kU];
    #pragma unroll
    for (int k = 0; k < kU; ++k) {
      const int it = base + k * NT + tid;
      hv[k] = hv0[k];
      msv[k] = ms0[k];
      if (base != 0) {
        hv[k] = 0.f;
        if (it < items) {
          const WideStat& ws = wst[it / kWideBins];
          hv[k] = ws.hist[it % kWideBins];
          msv[k] = ws.ms;
        }
      }
    }
    #pragma unroll
    for (int k = 0; k < kU; ++k) {
      const int it = base + k * NT + tid;
      const int j = it % kWideBins;
      const float lb = (M - msv[k]) * 1.4426950408889634f;  // log2 of M's weight over the chunk max's
      const float m = hv[k] * __builtin_amdgcn_exp2f(-lb);
      const bool pos = it < items && m > 0.f;
      const unsigned long long fx = pos ? (unsigned long long)((double)m * 4294967296.0) : 0ull;
      if (pos) {
        int g = j == kWideBins - 1 ? kWideGBins - 1 : (int)floorf((float)(j + 1) + lb);
        g = g < kWideGBins ? g : kWideGBins - 1;
        atomicAdd(&L.gmass[g], fx);
      }
      const int c = it / kWideBins;
      bef += c < unit * wu.chunks ? fx : 0ull;
    }
  }
  bef = wave_reduce64(bef, 0ull, [](uint64_t x, uint64_t y) { return x + y; });
  if ((tid & 63) == 0 && bef != 0ull) atomicAdd(&L.predfx, bef);
  __syncthreads();
  // w_lo: the first binade bin where the masses from the top reach the
  // cutoff plus the margin (one wave over the 64 bins)
  if (tid < 64) {
    const int lane = tid;
    // inclusive prefix sum over the lanes (DPP row shifts and broadcasts;
    // lanes with no source add zero)
    unsigned long long inc = L.gmass[lane];
    auto up = [&](auto ctl) {
      constexpr int C = decltype(ctl)::c, RM = decltype(ctl)::rm;
      constexpr bool BC = decltype(ctl)::bc;
      inc += ((unsigned long long)dpp32<C, RM, BC>(0u, (uint32_t)(inc >> 32)) << 32) | dpp32<C, RM, BC>(0u, (uint32_t)inc);
    };
    up(fold::DppStep<kDppShr1, 0xf, true>{});
    up(fold::DppStep<kDppShr1 + 1, 0xf, true>{});
    up(fold::DppStep<kDppShr1 + 3, 0xf, true>{});
    up(fold::DppStep<kDppShr1 + 7, 0xf, true>{});
    up(fold::DppStep<kDppBcast15, 0xa, false>{});
    up(fold::DppStep<kDppBcast31, 0xc, false>{});
    const unsigned long long tot = ((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(inc >> 32), 63) << 32) |
                                   (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)inc, 63);
    const double frac = (double)cfg.cutoff + (double)kWideMargin;
    float w_lo = 0.f;
    if (cfg.cutoff < 1.f && frac < 1.0) {
      const unsigned long long target = (unsigned long long)(frac * (double)tot);
      const uint64_t hit = __ballot(lane < kWideGBins - 1 && inc >= target);
      if (hit != 0ull) w_lo = __builtin_ldexpf(1.f, -(__ffsll((unsigned long long)hit)));
    }
    if (lane == 0) L.w_lo = fmaxf(w_lo, cfg.min_p);
  }
  __syncthreads();
  const WideRowStats st = WideRowStats{M, L.w_lo, 1u, (double)L.predfx * (1.0 / 4294967296.0)};
  __syncthreads();  // L is reused by the chunk work
  return st;
}

// The row max of s over its chunks (temperature-only rows).
__device__ __forceinline__ float wide_row_max(const SampleArgs& a, int row, const RowCfg& cfg, uint32_t* red) {
  uint32_t mk = 0u;
  for (int c = threadIdx.x; c < a.n_chunks; c += NT) mk = max(mk, okey(a.stats[(int64_t)row * a.n_chunks + c].max_l));
  mk = block_max_u32<NT>(mk, red);
  const float ml = okey_inv(mk);
  return finitef_(ml) ? ml / cfg.t_eff : -__builtin_inff();
}

// Counts the n listed weights of a unit by value into its wruns, when a
// sample of them shares values; returns the number of values, or kFoldNone.
// For lists that a row could not sort at once (kDrawPiece, by the unit's
// share): there the ranks take a sort and two folds a piece, and none of
// that when a value repeats more often than a piece is long.  64 f32 rows of
// 151,936, nucleus: bf16 values 416 -> 156 us, seven levels 3,960 -> 203, all
// equal 25 ms -> 335 us; values that all differ 413 -> 416 (the sample).
__device__ __forceinline__ uint32_t wide_count_runs(WideChunkLds& L, const SampleArgs& a, int row, const WideUnits& wu,
                                                    int unit, const uint64_t* list, uint32_t n) {
  const int tid = threadIdx.x;
  const uint32_t c0 = (uint32_t)(unit * wu.len);
  for (int h = tid; h < kWideHash; h += NT) { L.hkey[h] = 0u; L.hcnt[h] = 0u; L.hmin[h] = 0xffffffffu; }
  if (tid == 0) L.nr = 0u;
  __syncthreads();
  // the sample: up to NT weights spread over the list (keys without counts)
  const uint32_t ns = min(n, (uint32_t)NT);
  if ((uint32_t)tid < ns) {
    const uint64_t e = list[(uint32_t)tid * (n / ns)];
    (void)wide_insert(L.hkey, L.hcnt, L.hmin, kWideLog2, (uint32_t)(e >> 32), 0u, (uint32_t)e - c0);
  }
  __syncthreads();
  uint32_t mine = 0u;
  for (int h = tid; h < kWideHash; h += NT) mine += L.hkey[h] != 0u ? 1u : 0u;
  mine = wave_sum_u32(mine);
  if ((tid & 63) == 0) atomicAdd(&L.nr, mine);
  __syncthreads();
  const bool few = L.nr <= ns * 3u / 4u;
  __syncthreads();
  if (!few) return kFoldNone;
  if (tid == 0) L.nr = 0u;
  bool full = false;
  constexpr int kU = 8;
  for (uint32_t base = 0; base < n; base += kU * NT) {
    uint64_t e[kU];
    #pragma unroll
    for (int k = 0; k < kU; ++k) {
      const uint32_t p = base + (uint32_t)(k * NT + tid);
      e[k] = p < n ? list[p] : 0ull;
    }
    #pragma unroll
    for (int k = 0; k < kU; ++k)
      if (e[k] != 0ull && !full)
        full = !wide_insert(L.hkey, L.hcnt, L.hmin, kWideLog2, (uint32_t)(e[k] >> 32), 1u, (uint32_t)e[k] - c0);
  }
  if (__syncthreads_or(full)) return kFoldNone;
  // (the row's last unit may have fewer chunks)
  const uint32_t cap = (uint32_t)(kChunkRuns * min(wu.chunks, a.n_chunks - unit * wu.chunks));
  uint64_t* out = a.wruns + ((int64_t)row * a.n_chunks + (int64_t)unit * wu.chunks) * kChunkRuns;
  for (int h = tid; h < kWideHash; h += NT) {
    const uint32_t k = L.hkey[h];
    if (k == 0u) continue;
    const uint32_t p = atomicAdd(&L.nr, 1u);
    if (p < cap) out[p] = ((uint64_t)k << 32) | ((uint64_t)L.hcnt[h] << 16) | (uint64_t)L.hmin[h];
  }
  __syncthreads();
  return L.nr <= cap ? L.nr : kFoldNone;
}

// Steps 2-3 for one (unit, row), with the row's M and w_lo and the unit's
// predicted start S.
__device__ __forceinline__ void wide_chunk_work(WideChunkLds& L, const SampleArgs& a, int row, const WideUnits& wu,
                                                int unit, const RowCfg& cfg, const DrawRow& r, float M, float w_lo, double S,
                                                const i32x4_t (&pre)[kWidePre][4]) {
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int c0 = unit * wu.len, c1 = min(c0 + wu.len, a.V);
  const Exp2TabLds et{L.exptab};
  float* tr = L.tr[wid];
  uint64_t* list = a.ws_list + (int64_t)row * a.list_stride + c0;
  ChunkFold* cf = a.wfold + (int64_t)row * a.n_chunks + unit;
  const bool runs = a.dtype == HI_ROCM_DTYPE_BF16;
  if (tid == 0) L.n = 0u;
  if (runs)
    for (int h = tid; h < kWideHash; h += NT) { L.hkey[h] = 0u; L.hcnt[h] = 0u; L.hmin[h] = 0xffffffffu; }
  __syncthreads();
  bool full = false;
  float x[kWidePre][kDrawPer];
  #pragma unroll
  for (int i = 0; i < kWidePre; ++i) {
    const int tl = i * (NT / 64) + wid, t0 = c0 + tl * kWideTile;
    if (t0 >= c1) break;
    float v[4][4], sum = 0.f;
    #pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int e = t0 + j * 256 + lane * 4;
      i32x4_t o;
      #pragma unroll
      for (int q = 0; q < 4; ++q) {
        float w = exact_expf_neg(__int_as_float(pre[i][j][q]) - M, et);
        w = w < cfg.min_p || e + q >= c1 ? 0.f : w;  // min-p: excluded like a zero weight
        v[j][q] = w;
        o[q] = __float_as_int(w);
        sum += w;
      }
      // the weights, for the finish's exact folds and the drawn index
      if (e + 4 <= a.V) {
        __builtin_amdgcn_raw_buffer_store_b128(o, r.w, e * 4, 0, 0);
      } else {
        #pragma unroll
        for (int q = 0; q < 4; ++q) if (e + q < a.V) __builtin_amdgcn_raw_buffer_store_b32((uint32_t)o[q], r.w, (e + q) * 4, 0, 0);
      }
    }
    sum = wave_sum_f32(sum);
    if (lane == 0) L.tsum[tl] = sum;
    draw_turn(tr, v, x[i]);
    uint32_t mk = 0u;
    #pragma unroll
    for (int q = 0; q < kDrawPer; ++q) mk |= x[i][q] > 0.f && x[i][q] >= w_lo ? 1u << q : 0u;
    if (__ballot(mk != 0u) == 0ull) continue;
    if (runs) {
      for (mk = full ? 0u : mk; mk != 0u; mk &= mk - 1u) {
        const int q = __ffs((int)mk) - 1;
        full |= !wide_insert(L.hkey, L.hcnt, L.hmin, kWideLog2, __float_as_uint(tr[lane * kTrLd + q]), 1u,
                             (uint32_t)(t0 - c0 + lane * kDrawPer + q));
      }
      continue;
    }
    const uint32_t c = (uint32_t)__popc(mk);
    const uint32_t inc = wave_incl_scan_u32(c);
    uint32_t at = 0u;
    if (lane == 63) at = atomicAdd(&L.n, inc);
    at = (uint32_t)__builtin_amdgcn_readlane((int)at, 63) + inc - c;
    for (; mk != 0u; mk &= mk - 1u, ++at) {
      const int q = __ffs((int)mk) - 1;
      list[at] = ((uint64_t)__float_as_uint(tr[lane * kTrLd + q]) << 32) | (uint32_t)(t0 + lane * kDrawPer + q);
    }
  }
  const bool ovf = __syncthreads_or(full);
  if (runs) {
    for (int h = tid; h < kWideHash; h += NT) {
      const uint32_t k = L.hkey[h];
      if (k != 0u) list[atomicAdd(&L.n, 1u)] = ((uint64_t)k << 32) | ((uint64_t)L.hcnt[h] << 16) | (uint64_t)L.hmin[h];
    }
    __syncthreads();
  }
  const uint32_t n = L.n;
  uint32_t nr = kFoldNone;
  if (__builtin_expect(!runs && n >= 64u && n * (uint32_t)wu.n > (uint32_t)kDrawPiece, 0))
    nr = wide_count_runs(L, a, row, wu, unit, list, n);
  if (tid == 0) {
    cf->n = ovf ? kFoldNone : n;
    cf->nr = nr;
  }
  #pragma unroll
  for (int i = 0; i < kWidePre; ++i) {
    const int tl = i * (NT / 64) + wid;
    if (c0 + tl * kWideTile >= c1) break;
    double B = S;
    for (int t = 0; t < tl; ++t) B += (double)L.tsum[t];
    const uint32_t bin = (uint32_t)__builtin_amdgcn_readfirstlane((int)draw_tile_bin(B, L.tsum[tl]));
    fold::Map m = fold::map_identity(), low = m;
    if ((bin & 511u) != 0u) draw_tile_map(x[i], bin, m, low);
    if (lane == 0) {
      cf->map[tl] = m;
      cf->low[tl] = low;
      cf->bin[tl] = bin;
    }
  }
}

// The ranks' weights from the chunks' lists (n_all entries, chunk c's from
// D.noff[c] on).
struct WideListSrc {
  const WideUnits& wu;
  const DrawRow& r;
  const uint64_t* list;
  int n_all;
  bool whole;  // the lists hold every positive weight of the row

  // f(chunk, entry) for entries p0, p0 + stride, ..., eight loads in flight
  template <typename F>
  __device__ __forceinline__ void each(DrawLds<NT>& D, int p0, int stride, F f) const {
    constexpr int kU = 8;
    for (int base = p0; base < n_all; base += kU * stride) {
      uint64_t v[kU];
      int c[kU];
      // the last chunk whose offset is <= p, by a search of fixed steps (the
      // kU searches interleave)
      #pragma unroll
      for (int k = 0; k < kU; ++k) c[k] = 0;
      #pragma unroll
      for (int st = kDrawChunks / 2; st >= 1; st >>= 1) {
        #pragma unroll
        for (int k = 0; k < kU; ++k) c[k] = (int)D.noff[c[k] + st] <= base + k * stride ? c[k] + st : c[k];
      }
      #pragma unroll
      for (int k = 0; k < kU; ++k) {
        const int p = base + k * stride;
        v[k] = 0ull;
        if (p < n_all) v[k] = list[(int64_t)c[k] * wu.len + (p - (int)D.noff[c[k]])];
      }
      #pragma unroll
      for (int k = 0; k < kU; ++k)
        if (base + k * stride < n_all) f(c[k], v[k]);
    }
  }
  static __device__ __forceinline__ uint64_t key_of(uint64_t e) {
    return draw_key(__uint_as_float((uint32_t)(e >> 32)), (int)(uint32_t)e);
  }
  __device__ __forceinline__ void gather(DrawLds<NT>& D, uint64_t lo, uint64_t hi) const {
    __syncthreads();
    if (threadIdx.x == 0) D.n = 0u;
    __syncthreads();
    const uint32_t top = (uint32_t)((hi - 1u) >> 23);
    each(D, (int)threadIdx.x, NT, [&](int, uint64_t e) {
      const uint64_t k = key_of(e);
      if (k >= lo && k < hi) {
        const uint32_t at = atomicAdd(&D.n, 1u);
        if (at < (uint32_t)kDrawPiece) D.u.p.key0[at] = top - (uint32_t)(e >> 32);
      }
    });
    __syncthreads();
  }
  __device__ __forceinline__ bool descend(DrawLds<NT>&, uint64_t) const { return false; }
  __device__ __forceinline__ uint32_t index(DrawLds<NT>& D, float w, uint32_t ord, uint64_t lo, uint64_t hi) const {
    // the chunk by its matches, then its weights in index order
    const int tid = threadIdx.x;
    const uint32_t wb = __float_as_uint(w);
    uint32_t* cnt = D.u.p.v.tcnt;
    if (tid < kDrawChunks) cnt[tid] = 0u;
    __syncthreads();
    each(D, tid, NT, [&](int c, uint64_t e) {
      const uint64_t k = key_of(e);
      if ((uint32_t)(e >> 32) == wb && k >= lo && k < hi) atomicAdd(&cnt[c], 1u);
    });
    __syncthreads();
    uint32_t tot;
    const uint32_t mine = tid < wu.n ? cnt[tid] : 0u;
    const uint32_t before = block_excl_scan_u32<NT>(mine, D.red, &tot);
    if (before <= ord && ord < before + mine) {
      D.bnext = (uint32_t)tid;
      D.n = ord - before;
    }
    __syncthreads();
    const int c0 = (int)D.bnext * wu.len, c1 = min(c0 + wu.len, r.V);
    uint32_t want = D.n;
    for (int b = c0; b < c1; b += NT * kDrawPer) {
      const int i0 = b + tid * kDrawPer;
      uint32_t mk = 0u;
      #pragma unroll
      for (int j = 0; j < kDrawPer; j += 4) {
        const i32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(r.w, (i0 + j) * 4, 0, 0);
        #pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int i = i0 + j + q;
          const uint64_t k = draw_key(w, i);
          mk |= (uint32_t)v[q] == wb && i < c1 && k >= lo && k < hi ? 1u << (j + q) : 0u;
        }
      }
      const uint32_t n = (uint32_t)__popc(mk);
      const uint32_t at = block_excl_scan_u32<NT>(n, D.red, &tot);
      if (at <= want && want < at + n) {
        for (uint32_t q = at; q < want; ++q) mk &= mk - 1u;
        D.token = (uint32_t)(i0 + __ffs((int)mk) - 1);
      }
      if (want < tot) break;
      want -= tot;
    }
    __syncthreads();
    return D.token;
  }
};

// Calls f(unit, weight bits, count, index) for every entry of the row's
// units, in parallel (the units' offsets in F.noff, n_all entries): a value
// with its count and smallest index, or a listed weight (F.listed) with its
// own.
template <bool BF16, typename Fn>
__device__ __forceinline__ void wide_for_each_run(WideRunLds& F, const SampleArgs& a, int row, const WideUnits& wu,
                                                  int n_all, Fn f) {
  constexpr int kU = 8;
  const int tid = threadIdx.x;
  const uint64_t* list = a.ws_list + (int64_t)row * a.list_stride;
  const uint64_t* runs = BF16 ? list : a.wruns + (int64_t)row * a.n_chunks * kChunkRuns;
  const int stride = BF16 ? wu.len : wu.chunks * kChunkRuns;
  for (int base = 0; base < n_all; base += kU * NT) {
    uint64_t v[kU];
    int c[kU];
    #pragma unroll
    for (int k = 0; k < kU; ++k) c[k] = 0;
    #pragma unroll
    for (int st = kDrawChunks / 2; st >= 1; st >>= 1) {
      #pragma unroll
      for (int k = 0; k < kU; ++k) c[k] = (int)F.noff[c[k] + st] <= base + k * NT + tid ? c[k] + st : c[k];
    }
    uint32_t one = 0u;  // bit k: a listed weight
    if (!BF16) {
      #pragma unroll
      for (int k = 0; k < kU; ++k) one |= F.listed[c[k]] != 0 ? 1u << k : 0u;
    }
    #pragma unroll
    for (int k = 0; k < kU; ++k) {
      const int p = base + k * NT + tid, at = p - (int)F.noff[c[k]];
      const uint64_t* from = (one >> k) & 1u ? list + (int64_t)c[k] * wu.len : runs + (int64_t)c[k] * stride;
      v[k] = p < n_all ? from[at] : 0ull;
    }
    #pragma unroll
    for (int k = 0; k < kU; ++k) {
      if (base + k * NT + tid >= n_all) continue;
      const uint32_t e = (uint32_t)v[k];
      const bool w = (one >> k) & 1u;
      f(c[k], (uint32_t)(v[k] >> 32), w ? 1u : e >> 16, w ? e : (uint32_t)(c[k] * wu.len) + (e & 0xffffu));
    }
  }
  __syncthreads();
}

// The ranks of a row whose superset has few distinct weights: the units'
// runs merged by weight and sorted, the rank-order folds over runs of equal
// weights in closed form.  `mine`: the entries of unit threadIdx.x, `listed`:
// they are its list; returns the token, or 0xffffffff (path kWideMergeFull:
// the table of distinct weights overflowed).  All threads call it.
template <bool BF16>
__device__ __forceinline__ uint32_t wide_finish_runs(WideRunLds& F, const SampleArgs& a, int row, const RowCfg& cfg,
                                                     const WideUnits& wu, float w_lo, float total, uint32_t mine, bool listed,
                                                     uint32_t& path) {
  const int tid = threadIdx.x;
  const int nch = wu.n;
  uint32_t n_all;
  F.noff[tid] = block_excl_scan_u32<NT>(mine, F.fl.wcnt, &n_all);
  F.listed[tid] = listed ? 1u : 0u;
  if (tid == 0) F.noff[NT] = n_all;

  // c. merge the chunks' runs by weight
  for (int h = tid; h < kWideHash; h += NT) {
    F.u.mg.hkey[h] = 0u;
    F.u.mg.hcnt[h] = 0u;
    F.u.mg.hmin[h] = 0xffffffffu;
  }
  if (tid == 0) F.cnt = 0u;
  __syncthreads();
  bool full = false;
  wide_for_each_run<BF16>(F, a, row, wu, (int)n_all, [&](int, uint32_t key, uint32_t count, uint32_t idx) {
    if (!full) full = !wide_insert(F.u.mg.hkey, F.u.mg.hcnt, F.u.mg.hmin, kWideLog2, key, count, idx);
  });
  path = kWideMergeFull;
  if (__syncthreads_or(full)) return 0xffffffffu;
  path = kWideDrawFail;
  // d. distinct weights, descending: the table's used slots compacted in
  //    order of (thread, slot) (thread t holds slots q * NT + t: their
  //    count, then a block scan of the counts), then ranked
  {
    constexpr int kSl = kWideHash / NT;
    uint32_t hk[kSl];
    uint32_t nu = 0u;
    #pragma unroll
    for (int q = 0; q < kSl; ++q) {
      hk[q] = F.u.mg.hkey[q * NT + tid];
      nu += hk[q] != 0u ? 1u : 0u;
    }
    uint32_t tot;
    uint32_t o = block_excl_scan_u32<NT>(nu, F.fl.wcnt, &tot);
    #pragma unroll
    for (int q = 0; q < kSl; ++q)
      if (hk[q] != 0u) F.u.mg.sortk[o++] = ((uint64_t)hk[q] << 32) | (uint64_t)(q * NT + tid);
    if (tid == 0) F.cnt = tot;
  }
  __syncthreads();
  const int R = (int)F.cnt;
  if (R == 0) return 0xffffffffu;
  if (R <= NT) {
    block_sort_desc<1>(F.u.mg.sortk, R);
  } else if (R <= 2 * NT) {
    block_sort_desc<2>(F.u.mg.sortk, R);
  } else if (R <= 4 * NT) {
    block_sort_desc<4>(F.u.mg.sortk, R);
  } else {
    const int n2 = next_pow2(R);
    for (int i = R + tid; i < n2; i += NT) F.u.mg.sortk[i] = 0ull;
    __syncthreads();
    for (int k = 2; k <= n2; k <<= 1) {
      for (int j = k >> 1; j > 0; j >>= 1) {
        for (int i = tid; i < n2; i += NT) {
          const int ixj = i ^ j;
          if (ixj > i) {
            const uint64_t x = F.u.mg.sortk[i], y = F.u.mg.sortk[ixj];
            const bool desc = (i & k) == 0;
            if (desc ? (x < y) : (x > y)) { F.u.mg.sortk[i] = y; F.u.mg.sortk[ixj] = x; }
          }
        }
        __syncthreads();
      }
    }
  }
  {
    // runs in rank order: read everything first, the arrays overlap
    constexpr int kPer = kWideHash / NT;
    float rx[kPer];
    uint32_t rm[kPer], ri[kPer];
    #pragma unroll
    for (int q = 0; q < kPer; ++q) {
      const int r = q * NT + tid;
      if (r < R) {
        const uint64_t k = F.u.mg.sortk[r];
        const uint32_t h = (uint32_t)k;
        rx[q] = __uint_as_float((uint32_t)(k >> 32));
        rm[q] = F.u.mg.hcnt[h];
        ri[q] = F.u.mg.hmin[h];
      }
    }
    __syncthreads();
    #pragma unroll
    for (int q = 0; q < kPer; ++q) {
      const int r = q * NT + tid;
      if (r < R) { F.u.fo.rx[r] = rx[q]; F.u.fo.rm[r] = rm[q]; F.u.fo.ri[r] = ri[q]; }
    }
    __syncthreads();
  }

  // e. cum_p += w / total in rank order (from 0.0), up to the cutoff
  auto q_of = [&](int r) { return F.u.fo.rx[r] / total; };
  auto m_of = [&](int r) { return F.u.fo.rm[r]; };
  const float cum_end = fold::fold_runs<NT>(F.fl, F.pe, R, 0.0f, q_of, m_of,
                                            [&](int r, float v) { F.u.fo.st[r] = v; });
  __syncthreads();
  int rstar = R - 1;
  uint32_t cstar = F.u.fo.rm[R - 1];
  if (cfg.cutoff < 1.f) {
    uint32_t first = 0xffffffffu;
    for (int r = tid; r < R; r += NT) {
      const float end = r + 1 < R ? F.u.fo.st[r + 1] : cum_end;
      if (end >= cfg.cutoff) first = min(first, (uint32_t)r);
    }
    first = ~block_max_u32<NT>(~first, F.fl.wcnt);
    if (first == 0xffffffffu) {
      // the cutoff is not reached inside the superset: that is the whole
      // nucleus only when the superset holds every positive weight
      if (w_lo > cfg.min_p) {
        path = kWideNoCutoff;
        return 0xffffffffu;
      }
    } else {
      rstar = (int)first;
      cstar = fold::run_find<false>(F.u.fo.st[rstar], q_of(rstar), F.u.fo.rm[rstar], cfg.cutoff, nullptr);
      if (cstar == fold::kNone) return 0xffffffffu;
    }
  }
  // f. the candidate total: the weights of the ranks before m_end (from -0.0)
  auto m2_of = [&](int r) { return r == rstar ? cstar : F.u.fo.rm[r]; };
  const float ct = fold::fold_runs<NT>(F.fl, F.pe, rstar + 1, -0.0f, [&](int r) { return F.u.fo.rx[r]; }, m2_of,
                                       [&](int r, float v) { F.u.fo.st2[r] = v; });
  __syncthreads();
  if (tid == 0) a.wtot[2 * row + 1] = ct;
  if (!(ct > 0.f) || !finitef_(ct)) return 0xffffffffu;
  // g. the inverse CDF: the first rank whose running weight passes target
  const float target = clamp_uniform(cfg.u) * ct;
  uint32_t pr = 0xffffffffu;
  for (int r = tid; r <= rstar; r += NT) {
    const float end = r < rstar ? F.u.fo.st2[r + 1] : ct;
    if (target < end) pr = min(pr, (uint32_t)r);
  }
  pr = ~block_max_u32<NT>(~pr, F.fl.wcnt);
  int rp = rstar;
  uint32_t cp = cstar;  // gpu.rs:899: the last candidate
  if (pr != 0xffffffffu) {
    const uint32_t c = fold::run_find<true>(F.u.fo.st2[pr], F.u.fo.rx[pr], m2_of((int)pr), target, nullptr);
    if (c != fold::kNone) { rp = (int)pr; cp = c; }
  }
  // h. the drawn index: the cp-th smallest index among the weights equal
  //    to the run's (equal weights rank by index)
  const uint32_t first_idx = F.u.fo.ri[rp];
  path = kWideDone;
  if (cp == 1u) return first_idx;
  const uint32_t key = __float_as_uint(F.u.fo.rx[rp]);
  __syncthreads();
  F.cntc[tid] = 0u;
  __syncthreads();
  wide_for_each_run<BF16>(F, a, row, wu, (int)n_all, [&](int c, uint32_t k, uint32_t count, uint32_t) {
    if (k == key) atomicAdd(&F.cntc[c], count);
  });
  if (tid < 64) {
    // the chunk holding the cp-th match: an inclusive scan of the chunks'
    // match counts over the lanes, 64 chunks at a time
    uint32_t seen = 0u, csel = 0xffffffffu, rsel = 0u;
    for (int cb = 0; cb < nch; cb += 64) {
      const int c = cb + tid;
      const uint32_t k = c < nch ? F.cntc[c] : 0u;
      const uint32_t inc = wave_incl_scan_u32(k);
      const uint64_t hit = __ballot(k != 0u && seen + inc >= cp);
      if (hit != 0ull) {
        const int l = __ffsll((unsigned long long)hit) - 1;
        const uint32_t before = seen + (uint32_t)__builtin_amdgcn_readlane((int)(inc - k), l);
        csel = (uint32_t)(cb + l);
        rsel = cp - before;
        break;
      }
      seen += (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
    }
    if (tid == 0) {
      F.csel = csel;
      F.rsel = rsel;
      F.tok = 0xffffffffu;
      F.cnt = 0u;
    }
  }
  __syncthreads();
  const uint32_t csel = F.csel, want = F.rsel;
  if (csel == 0xffffffffu) {
    path = kWideDrawFail;
    return 0xffffffffu;
  }
  // the want-th weight equal to key in chunk csel, in index order: the
  // chunk's weights (ws_w, written by its chunk work) in blocks of kE
  // consecutive ones per thread, all loads in flight at once; a thread's
  // count of matches before it by a scan over the threads
  const int c0 = (int)csel * wu.len;
  const int len = min(wu.len, a.V - c0);
  const float* wrow = a.ws_w + (int64_t)row * a.V + c0;
  constexpr int kE = 16;
  for (int base = 0; base < len; base += kE * NT) {
    const int i0 = base + tid * kE;
    uint32_t eqm = 0u;
    #pragma unroll
    for (int q = 0; q < kE; ++q) {
      const int i = i0 + q;
      const float x = i < len ? wrow[i] : 0.f;
      eqm |= (i < len && __float_as_uint(x) == key ? 1u : 0u) << q;
    }
    const uint32_t nm = (uint32_t)__popc(eqm);
    uint32_t tot;
    const uint32_t before = F.cnt + block_excl_scan_u32<NT>(nm, F.fl.wcnt, &tot);
    if (before < want && before + nm >= want) {
      uint32_t m = eqm;
      for (uint32_t r = want - before; r > 1u; --r) m &= m - 1u;  // drop the matches before the wanted one
      F.tok = (uint32_t)(c0 + i0 + __ffs(m) - 1);
    }
    __syncthreads();
    if (tid == 0) F.cnt += tot;
    __syncthreads();
    if (F.tok != 0xffffffffu) break;
  }
  if (F.tok == 0xffffffffu) path = kWideDrawFail;
  return F.tok;
}

// Whether the wide pass takes the rows: their units fit the tables (up to
// 4,194,304 logits in units of 16,384).  The row of its tiles, whose maps are
// chained kDrawTiles at a time.
__device__ __forceinline__ bool wide_fits(const WideUnits& wu) { return wu.n <= kDrawChunks; }
__device__ __forceinline__ DrawRow wide_row(const SampleArgs& a, int row) {
  DrawRow r = draw_row<NT>(a, row);
  r.mult = 1;
  return r;
}

// Step 4: the finish of a top-p row by its last workgroup.  Returns the
// token, or 0xffffffff when the row must take finish_row (nothing written);
// `path` gets the WidePath code.
__device__ __forceinline__ uint32_t wide_finish(DrawLds<NT>& D, const SampleArgs& a, int row, const RowCfg& cfg,
                                                const WideUnits& wu, const DrawRow& r, float w_lo, uint32_t& path) {
  const int tid = threadIdx.x, wid = tid >> 6;
  const int nch = wu.n;
  const ChunkFold* folds = a.wfold + (int64_t)row * a.n_chunks;
  const int nt = (a.V + kWideTile - 1) / kWideTile, per = wu.len / kWideTile;
  const bool runs = a.dtype == HI_ROCM_DTYPE_BF16;
  const uint32_t cn = tid < nch ? folds[tid].n : 0u;
  const bool ovf = __syncthreads_or(cn == kFoldNone);
  const uint32_t mine = ovf ? 0u : cn;
  auto load_tiles = [&](int t0) {
    if (t0 + tid < nt) {
      const ChunkFold& f = folds[(t0 + tid) / per];
      D.tmap[tid] = f.map[(t0 + tid) % per];
      D.tlow[tid] = f.low[(t0 + tid) % per];
      D.tbin[tid] = f.bin[(t0 + tid) % per];
    }
  };
  load_tiles(0);
  uint32_t n_all;
  auto lists = [&]() {
    for (int b = tid; b < kDrawBins + kDrawBins / 32; b += NT) D.hist[b] = 0u;
    D.noff[tid] = block_excl_scan_u32<NT>(mine, D.red, &n_all);
    if (tid == 0) {
      D.noff[NT] = n_all;
      D.n = n_all;
    }
  };
  lists();
  static_assert(NT == kDrawChunks && NT == kDrawTiles, "a thread per chunk and per tile");
  __syncthreads();
  const WideListSrc src{wu, r, a.ws_list + (int64_t)row * a.list_stride, (int)n_all, !(w_lo > cfg.min_p)};
  const bool one = n_all <= (uint32_t)kDrawPiece;  // every listed weight fits a piece
  // f32: the units' values, where counted, when they halve the entries
  bool counted = false;
  uint32_t entries = mine;
  bool listed = true;
  if (__builtin_expect(!runs && !one, 0)) {
    const uint32_t nr = tid < nch ? folds[tid].nr : kFoldNone;
    listed = nr == kFoldNone;
    entries = listed ? mine : nr;
    uint32_t n_runs;
    block_excl_scan_u32<NT>(entries, D.red, &n_runs);
    counted = n_runs <= n_all / 2u;
  }
  // A piece of a long list costs more than one from the row's weights, which
  // stream without a search for each entry's unit.
  const bool too_long = n_all > (uint32_t)(a.V / kWideListShare);
  path = kWideLongList;
  if (__builtin_expect(!runs && !counted && too_long, 0)) return 0xffffffffu;
  constexpr uint32_t kTop = (uint32_t)((kDrawAll - 1u) >> 23);
  auto histogram = [&](int p0, int stride) {
    src.each(D, p0, stride, [&](int, uint64_t e) {
      atomicAdd(&D.hist[draw_slot(draw_bin(__uint_as_float((uint32_t)(e >> 32))))], 1u);
    });
  };
  if (wid == 0) {
    draw_chain<NT>(D, r, 0, min(nt, kDrawTiles), -0.0f);
  } else if (runs || counted) {
  } else if (one) {
    int p = tid - 64;  // entries in order: p, p + 192, ...
    src.each(D, tid - 64, NT - 64, [&](int, uint64_t e) {
      D.u.p.key0[p] = kTop - (uint32_t)(e >> 32);
      p += NT - 64;
    });
  } else {
    histogram(tid - 64, NT - 64);
  }
  __syncthreads();
  for (int t0 = kDrawTiles; t0 < nt; t0 += kDrawTiles) {
    load_tiles(t0);
    __syncthreads();
    if (wid == 0) draw_chain<NT>(D, r, t0, min(nt - t0, kDrawTiles), D.total);
    __syncthreads();
  }
  const float total = D.total;
  if (tid == 0) a.wtot[2 * row] = total;
  path = kWideTotal;
  if (!(total > 0.f) || !finitef_(total)) return 0xffffffffu;  // argmax_host fallback (finish_row)
  path = kWideChunkFull;
  if (ovf) return 0xffffffffu;
  path = kWideNoCutoff;
  if (runs) {
    __syncthreads();
    return wide_finish_runs<true>(reinterpret_cast<WideRunLds&>(D), a, row, cfg, wu, w_lo, total, mine, false, path);
  }
  if (__builtin_expect(counted, 0)) {
    __syncthreads();
    const uint32_t tok = wide_finish_runs<false>(reinterpret_cast<WideRunLds&>(D), a, row, cfg, wu, w_lo, total, entries,
                                                 listed, path);
    if (tok != 0xffffffffu || path != kWideMergeFull) return tok;
    // too many values after all: the ranks from the lists
    if (too_long) return tok;
    __syncthreads();
    lists();
    __syncthreads();
    histogram(tid, NT);
    __syncthreads();
    path = kWideNoCutoff;
  }
  uint64_t lo = (uint64_t)max(__float_as_uint(w_lo), 1u) << 23;
  uint32_t bin = (uint32_t)kDrawBins;
  if (!one) {
    if (wid == 0) draw_bins<NT>(D, 0u, cfg.cutoff < 1.f ? (cfg.cutoff * 1.008f + 0.002f) * total : __builtin_inff());
    __syncthreads();
    bin = D.bnext;
    lo = D.lo;
    if (bin == 0xffffffffu) return 0xffffffffu;
    src.gather(D, lo, kDrawAll);
  }
  const uint32_t tok = draw_ranks<NT>(D, src, cfg, 0, total, true, lo, bin, a.wtot + 2 * row + 1);
  if (tok == kDrawRetry) return 0xffffffffu;
  path = tok == kDrawFallback ? kWideDrawFail : kWideDone;
  return tok;
}

// A temperature-only row's part of workgroup `chunk` < kTempSplit: the sums
// of 64 of the 256 reference chunks, a quad each, to the row's ws_list.
// Batches of up to kTempRows rows: beyond, one workgroup a row fills the chip
// (bf16 rows of 151,936, one workgroup and split: 64 rows 64 and 59 us, 96
// rows 68 and 69, 128 rows 81 and 95, 256 rows 124 and 176; of 50,257: 64 rows
// 39 and 39, 128 rows 50 and 59).  (A
// wave a chunk, folding 64 weights at a time, took 140 us for 64 rows of
// 151,936 against 64 us for one workgroup a row: the folds are serial, so
// they fill the chip only when every lane holds one.)
constexpr int kTempSplit = 4;
constexpr int kTempRows = 64;
__device__ __forceinline__ void wide_temperature_work(WideChunkLds& L, const SampleArgs& a, int row, int chunk,
                                                      const DrawRow& r, float M) {
  const int tid = threadIdx.x;
  if (tid < 32) L.exptab[tid] = exp2_tab32((uint32_t)tid);
  __syncthreads();
  const Exp2TabLds et{L.exptab};
  float* csum = reinterpret_cast<float*>(a.ws_list + (int64_t)row * a.list_stride);
  const int len = (a.V + 255) / 256;
  const int t = chunk * 64 + (tid >> 2);
  const int start = t * len, end = min(start + len, a.V);
  const float s = draw_chunk_sum<4>(r.s, start, end, M, et);
  if ((tid & 3) == 0) csum[t] = s;
}

// A whole row by one workgroup of NT threads, any row class: the select
// pass over kRowGeneralChunk-logit chunks in turn, then the chunked path's
// finish (finish_lean, else finish_row).  The workspace must hold the
// records of ceil(V / kRowGeneralChunk) chunks per row (general_layout);
// lds_raw must hold SelLds (plus the history table when a.hoff is given)
// and FinLds.
template <bool MASK>
__device__ __forceinline__ void general_row_path(SampleArgs& a, int row, unsigned char* lds_raw) {
  a.chunk = kRowGeneralChunk;
  a.n_chunks = (a.V + kRowGeneralChunk - 1) / kRowGeneralChunk;
  const RowCfg cfg = load_cfg(a.pv, row, a.V, a.n_lp, a.need_lse);
  for (int c = 0; c < a.n_chunks; ++c) {
    select_chunk<HI_ROCM_DTYPE_F32, kRowGeneralChunk / NT / 4, MASK>(a, row, c, lds_raw);
    __syncthreads();
  }
  if (threadIdx.x == 0) a.diag[row] = kRowPathGeneral;
  FinLds& fs = *reinterpret_cast<FinLds*>(lds_raw);
  if (finish_lean(fs, a, row, cfg)) return;
  __syncthreads();
  finish_row(fs, a, row, cfg);
}

}  // namespace hi_rocm
