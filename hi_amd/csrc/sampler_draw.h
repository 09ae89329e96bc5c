// Draws of rows that keep their whole distribution (top-p without top-k,
// min-p alone, top-k above kBuf, temperature only) by one workgroup, from
// the row's scaled logits in ws_s.
//
// The reference walks such a row three times in order: the normaliser over
// the vocabulary (gpu.rs:837), cum_p over the ranks (:843-856) and the
// candidate total with the inverse CDF (:874-899), each a left-to-right f32
// fold.  Here every fold is split across lanes with parity maps
// (exact_fold.h), and a lane's map takes two float additions a term: folding
// the terms onto 2^e and onto 2^e + ulp rounds like any sum of that binade
// with an even, or an odd, last bit.
//  1. Weights: exact expf of every scaled logit, stored in ws_w, a histogram
//     of their leading bits (64 bins a binade) and the sum of each tile.
//  2. Normaliser: the tile sums predict each tile's binade; every tile
//     becomes one map in that binade (and the one below, near its lower
//     end); wave 0 chains them from -0.0 in tile order.  A tile that leaves
//     its binade, or starts in another, is folded exactly by the wave, lane
//     by lane.
//  3. Ranks: pieces of up to kPiece weights in descending order (the
//     histogram gives the first piece's lower end so that it holds the
//     nucleus), gathered to LDS, sorted by a radix sort and folded by wave 0
//     (cum_p) and wave 1 (candidate total) until the cutoff; the drawn rank
//     is then found from the folds' start values.  Equal weights rank by
//     index, which no fold sees: only weights are sorted, and the drawn
//     weight's index is looked up at the end.
// What bounds it: the exact expf (about 31 cycles a wave and SIMD for 64
// logits) and, with four waves, the latency of the streams over ws_s and
// ws_w.  One row of 151,936 f32 logits, all launches included: nucleus 1,667
// -> 178 us (spiked logits: 2,214 -> 193), temperature only 390 -> 47 us; the
// form before it summed the normaliser and both rank folds on one thread and
// sorted in global memory.
#pragma once

#include "fold_wg.h"
#include "exact_expf.h"

namespace hi_rocm {

constexpr int kDrawBins = 2048;   // weight histogram: 64 bins a binade, 32 binades
constexpr int kDrawLast = kDrawBins + kDrawBins / 32;  // the lanes' words past the bins
constexpr int kDrawTiles = 256;   // tiles of a row
constexpr int kDrawPer = 16;      // logits of a lane's part of a tile, per step
constexpr int kDrawPiece = 4096;  // weights sorted at a time
constexpr int kDrawBlocks = 256;  // blocks of a piece in its folds
constexpr int kDrawDigitBits = 9;
constexpr int kDrawDigits = 1 << kDrawDigitBits;  // of a radix pass
constexpr int kDrawChunks = 256;  // chunks of a row whose lists a draw reads
constexpr int kDrawRecs = 64;     // pieces whose start the draw can go back to
constexpr uint32_t kOneBits = 0x3f800000u;

// A histogram bin's word: one pad word per 32, so that the lanes of the
// range search, 32 bins each, read distinct banks.
__device__ __forceinline__ uint32_t draw_slot(uint32_t bin) { return bin + (bin >> 5); }

template <int NTH>
struct DrawLds {
  static constexpr int kKeys = kDrawPiece + kDrawBlocks;  // block t's J terms at t * (J | 1)
  union {
    struct {
      uint32_t key0[kKeys];                        // the piece's sort keys, then its weights in rank order
      union {
        float tr[NTH / 64][64 * (kDrawPer + 4)];   // a wave's tile, lane-major
        struct {
          uint32_t key1[kKeys];                    // the sort's second buffer
          uint32_t cnt[NTH / 64][kDrawDigits];     // a radix pass's digit counts, then bases
        } so;
        float start[2][kDrawBlocks];               // cum_p and candidate total before each block
        uint32_t tcnt[kDrawTiles];                 // matches of the drawn weight in each tile
      } v;
    } p;
    struct {
      float csum[256], prefix[256];                // temperature-only chunks
    } to;
  } u;
  uint32_t hist[kDrawBins + kDrawBins / 32 + 64];  // (past the bins: a word per lane that nothing reads)
  fold::Map tmap[kDrawTiles], tlow[kDrawTiles];  // a tile's map in binade tbin, and in tbin - 1
  float tsum[kDrawTiles];
  uint32_t tbin[kDrawTiles];  // draw_tile_bin
  uint64_t exptab[32];
  uint64_t rec_hi[kDrawRecs];
  float rec_ct[kDrawRecs];
  uint32_t noff[kDrawChunks + 1];  // a list's entries before each chunk
  uint32_t red[NTH / 64];
  uint64_t lo;
  uint32_t n, bnext, token;
  float total, end[2], ct;
  __device__ float* wf() { return reinterpret_cast<float*>(u.p.key0); }
};

// The row's arrays as buffers, V rounded up to whole 16-byte accesses (what
// follows a row's values belongs to the workspace; the streams drop it):
// loads past them return zero and cost nothing, so the streams need no
// branches, and the 4-byte alignment of a row that starts anywhere is enough.
struct DrawRow {
  __amdgpu_buffer_rsrc_t s, w;
  int V, mult;  // a tile is 64 lanes of 16 * mult logits
  int steps;    // 16-logit steps of a wave over its tiles
};
template <int NTH>
__device__ __forceinline__ DrawRow draw_row(const SampleArgs& a, int row) {
  DrawRow r;
  const int64_t off = (int64_t)row * a.V;
  r.s = __builtin_amdgcn_make_buffer_rsrc((void*)(a.ws_s + off), 0, ((a.V + 3) & ~3) * 4, kBufferConfig);
  r.w = __builtin_amdgcn_make_buffer_rsrc((void*)(a.ws_w + off), 0, ((a.V + 3) & ~3) * 4, kBufferConfig);
  r.V = a.V;
  r.mult = (a.V + kDrawTiles * 64 * kDrawPer - 1) / (kDrawTiles * 64 * kDrawPer);
  const int nt = (a.V + 64 * kDrawPer * r.mult - 1) / (64 * kDrawPer * r.mult);
  r.steps = (nt + NTH / 64 - 1) / (NTH / 64) * r.mult;
  return r;
}

// f(tile, part, c0, x) for every step of this wave over its tiles (tile wid,
// wid + waves, ...; part < mult of it, logits from c0 on): x[j][q] is logit
// c0 + 256 j + 4 lane + q of `buf`, zero past the row.  kAhead steps are in
// flight: a step's loads take about 2,000 cycles from another XCD's stores,
// its work 600 to 2,000.
template <int NTH, typename F>
__device__ __forceinline__ void draw_stream(const DrawRow& r, __amdgpu_buffer_rsrc_t buf, F f) {
  constexpr int kAhead = NTH >= 1024 ? 1 : 2;
  const int lane = (int)(threadIdx.x & 63u);
  const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  i32x4_t x[kAhead][4];
  auto base = [&](int it) { return ((wid + it / r.mult * (NTH / 64)) * r.mult + it % r.mult) * 64 * kDrawPer; };
  auto issue = [&](int it, i32x4_t (&d)[4]) {
    // (a step past the last reads nothing: its offsets are past the row)
    const int c0 = it < r.steps ? base(it) : r.V + 4;
    #pragma unroll
    for (int j = 0; j < 4; ++j) d[j] = __builtin_amdgcn_raw_buffer_load_b128(buf, (c0 + j * 256 + lane * 4) * 4, 0, 0);
  };
  #pragma unroll
  for (int d = 0; d < kAhead; ++d) issue(d, x[d]);
  for (int it0 = 0; it0 < r.steps; it0 += kAhead) {
    #pragma unroll
    for (int d = 0; d < kAhead; ++d) {
      const int it = it0 + d;
      float v[4][4];
      #pragma unroll
      for (int j = 0; j < 4; ++j)
        #pragma unroll
        for (int q = 0; q < 4; ++q) v[j][q] = __int_as_float(x[d][j][q]);
      issue(it + kAhead, x[d]);
      if (base(it) + 64 * kDrawPer > r.V) {
        #pragma unroll
        for (int j = 0; j < 4; ++j)
          #pragma unroll
          for (int q = 0; q < 4; ++q) v[j][q] = base(it) + j * 256 + lane * 4 + q < r.V ? v[j][q] : 0.f;
      }
      if (it < r.steps) f(wid + it / r.mult * (NTH / 64), it % r.mult, base(it), v);
    }
  }
}

// The map of the terms x[0 .. N) in binade e: the terms folded onto 2^e and
// onto 2^e + ulp.  A sum that reaches the next binade saturates (every start
// of the binade then leaves it too).
template <int N>
__device__ __forceinline__ fold::Map lane_map(const float (&x)[N], int e) {
  const uint32_t b = (uint32_t)e << 23;
  float p = __uint_as_float(b), q = __uint_as_float(b + 1u);
  #pragma unroll
  for (int k = 0; k < N; ++k) {
    p = fold::fadd(p, x[k]);
    q = fold::fadd(q, x[k]);
  }
  const uint32_t top = b + 0x800000u;
  const uint32_t pb = __float_as_uint(p), qb = __float_as_uint(q);
  return fold::Map{pb >= top ? fold::kSat : pb - b, qb >= top ? fold::kSat : qb - b - 1u};
}

// The exact fold of the wave's lane blocks (lane l's terms x[0 .. N), lanes
// in order) onto acc; start(v) gets each lane's value before its block.
// While the sum stays in one binade a scan of the lane maps steps over
// lanes; the lane whose block leaves it adds its terms one by one.
template <int N, typename StartF>
__device__ __forceinline__ float wave_fold_blocks(const float (&x)[N], float acc, StartF start) {
  const int lane = (int)(threadIdx.x & 63u);
  int pos = 0;
  float mine = acc;
  while (pos < 64) {
    const int e = fold::binade(acc);
    const uint32_t A = fold::to_A(acc), p = A & 1u;
    fold::Map m = lane_map(x, e);
    if (lane < pos) m = fold::map_identity();
    const fold::Map inc = fold::wave_map_scan(m);
    const fold::Map ex = fold::wave_map_prev(inc);
    const uint32_t Ai = A + fold::apply(inc, p);  // (maps saturate below 2^27)
    const uint64_t bad = __ballot(Ai >= fold::kTop);
    const int f = bad ? __ffsll((unsigned long long)bad) - 1 : 64;
    if (lane >= pos && lane <= f) {
      const uint32_t Ab = A + fold::apply(ex, p);  // below kTop: the lanes before stayed
      mine = lane == pos ? acc : fold::from_A(Ab, e);
    }
    if (f == 64) {
      acc = fold::from_A((uint32_t)__builtin_amdgcn_readlane((int)Ai, 63), e);
      break;
    }
    float v = mine;
    #pragma unroll
    for (int k = 0; k < N; ++k) v = fold::fadd(v, x[k]);
    acc = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), f));
    pos = f + 1;
  }
  start(mine);
  return acc;
}

// rank order of a row's weights as one integer: weight bits, then the lower
// index first (V <= 2^23, weights at most 1)
__device__ __forceinline__ uint64_t draw_key(float w, int i) {
  return ((uint64_t)__float_as_uint(w) << 23) | (uint64_t)(0x7fffffu - (uint32_t)i);
}
__device__ __forceinline__ uint32_t draw_bin(float w) {
  return min((kOneBits - __float_as_uint(w)) >> 17, (uint32_t)kDrawBins - 1u);
}

// Step 1 (see the top).
template <int NTH>
__device__ __forceinline__ void draw_weights(DrawLds<NTH>& D, const DrawRow& r, float M, float min_p) {
  const int tid = threadIdx.x, lane = tid & 63;
  for (int b = tid; b < kDrawLast + 64; b += NTH) D.hist[b] = 0u;
  if (tid < 32) D.exptab[tid] = exp2_tab32((uint32_t)tid);
  __syncthreads();
  const Exp2TabLds et{D.exptab};
  float sum = 0.f;
  uint32_t small = 0u;
  draw_stream<NTH>(r, r.s, [&](int t, int g, int c0, const float (&x)[4][4]) {
    if (g == 0) sum = 0.f;
    // no branches (the waits for the loads in flight count on it): the last
    // bin's weights count in a register (its word of the lane's own takes
    // their atomics), and a lane's access that crosses the row's end stores
    // nothing
    #pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i = c0 + j * 256 + lane * 4;
      i32x4_t o;
      #pragma unroll
      for (int q = 0; q < 4; ++q) {
        float w = exact_expf_neg(x[j][q] - M, et);
        w = w < min_p || i + q >= r.V ? 0.f : w;  // min-p: excluded like a zero weight
        o[q] = __float_as_int(w);
        sum += w;
        const uint32_t bin = draw_bin(w);
        small += bin == (uint32_t)kDrawBins - 1u && w > 0.f ? 1u : 0u;
        atomicAdd(&D.hist[bin < (uint32_t)kDrawBins - 1u ? draw_slot(bin) : (uint32_t)kDrawLast + (uint32_t)lane], 1u);
      }
      __builtin_amdgcn_raw_buffer_store_b128(o, r.w, i + 4 <= r.V ? i * 4 : 0x7ffffff0, 0, 0);
    }
    if (g == r.mult - 1) {
      const float ts = wave_sum_f32(sum);
      if (lane == 0 && t < kDrawTiles) D.tsum[t] = ts;
    }
  });
  // the row's last V % 4 weights
  if (tid < (r.V & 3)) {
    const int i = (r.V & ~3) + tid;
    const float w = exact_expf_neg(__int_as_float((int)__builtin_amdgcn_raw_buffer_load_b32(r.s, i * 4, 0, 0)) - M, et);
    __builtin_amdgcn_raw_buffer_store_b32((uint32_t)__float_as_int(w < min_p ? 0.f : w), r.w, i * 4, 0, 0);
  }
  small = wave_sum_u32(small);
  if (lane == 0 && small != 0u) atomicAdd(&D.hist[draw_slot(kDrawBins - 1)], small);
  __syncthreads();
}

// The binade a tile predicted to go from S to E is mapped in (bits 0-8; 0:
// it is folded exactly), and whether the binade below is mapped too (bit 9).
// A tile without a positive weight (min-p and masks leave many) adds nothing
// in any binade.
constexpr uint32_t kTileLow = 512u, kTileZero = 1024u;
__device__ __forceinline__ uint32_t draw_tile_bin(double S, float sum) {
  if (sum == 0.f) return kTileZero;
  const double E = S + (double)sum;
  const int e = fold::binade((float)S);
  // well inside one binade (0.1%)
  const bool one = e > 1 && fold::binade((float)(S * 0.999)) == e && fold::binade((float)(E * 1.001)) == e;
  // terms below half an ulp add nothing to an f32 sum: the sum may lag the
  // prediction, so near a binade's lower end the one below is kept too
  const bool low = e > 2 && fold::binade((float)(S * 0.875)) != e;
  return one || low ? (uint32_t)e | (low ? kTileLow : 0u) : 0u;
}

// Predicted binades of the tiles (one wave), from a scan of their sums.
template <int NTH>
__device__ __forceinline__ void draw_predict(DrawLds<NTH>& D, int nt) {
  const int lane = (int)(threadIdx.x & 63u);
  static_assert(kDrawTiles % 64 == 0, "the prediction scans 64 tiles at a time");
  double before = 0.0;
  for (int tb = 0; tb < nt; tb += 64) {
    const int t = tb + lane;
    const float s = t < nt ? D.tsum[t] : 0.f;
    const double inc = fold::wave_scan_f64((double)s);
    if (t < nt) D.tbin[t] = draw_tile_bin(before + inc - (double)s, s);
    const uint64_t ib = readlane64((uint64_t)__double_as_longlong(inc), 63);
    before += __longlong_as_double((long long)ib);
  }
}

// The maps of a tile's step (lane l's terms x) in its binade and, when kept,
// in the one below: the composition over the lanes, in every lane.
__device__ __forceinline__ void draw_tile_map(const float (&x)[kDrawPer], uint32_t bin, fold::Map& m, fold::Map& low) {
  const int e = (int)(bin & 511u);
  auto total_of = [&](fold::Map lm) {
    const fold::Map inc = fold::wave_map_scan(lm);
    return fold::Map{(uint32_t)__builtin_amdgcn_readlane((int)inc.t0, 63),
                     (uint32_t)__builtin_amdgcn_readlane((int)inc.t1, 63)};
  };
  m = total_of(lane_map(x, e));
  low = fold::map_identity();
  if (bin & kTileLow) low = total_of(lane_map(x, e - 1));
}

// A tile's lane blocks of 16 terms (lane l: terms c0 + 16 l ..), straight
// from memory (the few tiles the chain folds itself).
__device__ __forceinline__ void draw_lane_terms(const DrawRow& r, int c0, float (&x)[kDrawPer]) {
  const int i = c0 + (int)(threadIdx.x & 63u) * kDrawPer;
  #pragma unroll
  for (int j = 0; j < kDrawPer; j += 4) {
    const i32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(r.w, (i + j) * 4, 0, 0);
    #pragma unroll
    for (int q = 0; q < 4; ++q) x[j + q] = i + j + q < r.V ? __int_as_float(v[q]) : 0.f;
  }
}

// A wave's step of a tile in LDS, lane l's 16 consecutive logits at l * kTrLd
// (16-byte reads of 8 lanes hit distinct banks), and in x.
constexpr int kTrLd = kDrawPer + 4;
__device__ __forceinline__ void draw_turn(float* tr, const float (&v)[4][4], float (&x)[kDrawPer]) {
  const int lane = (int)(threadIdx.x & 63u);
  wave_lds_sync();  // the step before is read
  #pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int l = j * 256 + lane * 4;
    *reinterpret_cast<float4*>(tr + (l / kDrawPer) * kTrLd + l % kDrawPer) =
        make_float4(v[j][0], v[j][1], v[j][2], v[j][3]);
  }
  wave_lds_sync();
  #pragma unroll
  for (int j = 0; j < kDrawPer; j += 4) {
    const float4 u = *reinterpret_cast<const float4*>(tr + lane * kTrLd + j);
    x[j] = u.x; x[j + 1] = u.y; x[j + 2] = u.z; x[j + 3] = u.w;
  }
}

// This wave's part of a piece [lo, hi): the sort keys of its turned weights
// x (logits c0 + 16 lane .., also in tr) that lie in it (top minus the
// weight's bits, so that descending weights ascend) go to D.u.p.key0,
// counted in D.n (past kDrawPiece: counted only).
template <int NTH>
__device__ __forceinline__ void draw_collect(DrawLds<NTH>& D, const float* tr, const float (&x)[kDrawPer], int c0,
                                             uint64_t lo, uint64_t hi, uint32_t top) {
  const int lane = (int)(threadIdx.x & 63u);
  const float wlo = __uint_as_float((uint32_t)(lo >> 23)), whi = __uint_as_float(top);
  uint32_t mk = 0u;
  #pragma unroll
  for (int q = 0; q < kDrawPer; ++q) mk |= x[q] >= wlo && x[q] <= whi ? 1u << q : 0u;
  if (__ballot(mk != 0u) == 0ull) return;
  if (((lo | hi) & 0x7fffffull) != 0ull) {
    // the piece ends inside a run of equal weights: by whole keys
    #pragma unroll
    for (int q = 0; q < kDrawPer; ++q) {
      const uint64_t k = draw_key(x[q], c0 + lane * kDrawPer + q);
      if (k < lo || k >= hi) mk &= ~(1u << q);
    }
  }
  const uint32_t c = (uint32_t)__popc(mk);
  const uint32_t inc = wave_incl_scan_u32(c);
  const uint32_t tot = wave_last_u32(inc);
  uint32_t at = 0u;
  if (lane == 0) at = atomicAdd(&D.n, tot);
  at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at) + inc - c;
  for (; mk != 0u; mk &= mk - 1u, ++at)
    if (at < (uint32_t)kDrawPiece) D.u.p.key0[at] = top - __float_as_uint(tr[lane * kTrLd + __ffs((int)mk) - 1]);
}

// The chain from `acc` over the row's tiles t0, ..., t0 + nt - 1, whose maps D
// holds (wave 0, lane l holding tile t0 + tb + l), to D.total: scans over the
// tiles of one binade, exact folds of the others.
template <int NTH>
__device__ __forceinline__ void draw_chain(DrawLds<NTH>& D, const DrawRow& r, int t0, int nt, float acc) {
  const int lane = (int)(threadIdx.x & 63u);
  const int span = 64 * kDrawPer * r.mult;
  for (int tb = 0; tb < nt; tb += 64) {
    const int n = min(64, nt - tb);
    const uint32_t bin = lane < n ? D.tbin[tb + lane] : 0u;
    const fold::Map mh = D.tmap[min(tb + lane, nt - 1)], ml = D.tlow[min(tb + lane, nt - 1)];
    int i0 = 0;
    while (i0 < n) {
      const int e = fold::binade(acc);
      const uint32_t A = fold::to_A(acc), p = A & 1u;
      const int d = (int)(bin & 511u) - e;
      fold::Map s = d == 0 ? mh : ml;
      if (!(d == 0 || (d == 1 && (bin & kTileLow)))) s = fold::Map{fold::kSat, fold::kSat};
      if (lane < i0 || bin == kTileZero) s = fold::map_identity();
      const fold::Map inc = fold::wave_map_scan(s);
      const uint32_t Ai = A + fold::apply(inc, p);
      const uint64_t bad = __ballot(lane >= i0 && lane < n && Ai >= fold::kTop);
      const int f = bad ? __ffsll((unsigned long long)bad) - 1 : n;
      if (f > i0) acc = fold::from_A((uint32_t)__builtin_amdgcn_readlane((int)Ai, f - 1), e);
      if (f < n) {
        for (int g = 0; g < r.mult; ++g) {
          float x[kDrawPer];
          draw_lane_terms(r, (t0 + tb + f) * span + g * 64 * kDrawPer, x);
          acc = wave_fold_blocks(x, acc, [](float) {});
        }
      }
      i0 = f + 1;
    }
  }
  if (lane == 0) D.total = acc;
}

// Step 2: the vocabulary-order fold of the row's weights from -0.0, in
// D.total, and the first piece [lo, hi)'s sort keys, gathered by the same
// pass.  All threads call it (D.tbin and the range are known, D.n is 0).
template <int NTH>
__device__ __forceinline__ void draw_total(DrawLds<NTH>& D, const DrawRow& r, uint64_t lo, uint64_t hi) {
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int span = 64 * kDrawPer * r.mult;
  const int nt = (r.V + span - 1) / span;
  const uint32_t top = (uint32_t)((hi - 1u) >> 23);
  // each tile's map: loads of 256 terms, turned to 16 a lane through LDS
  float* tr = D.u.p.v.tr[wid];
  fold::Map m = fold::map_identity(), low = m;
  draw_stream<NTH>(r, r.w, [&](int t, int g, int c0, const float (&v)[4][4]) {
    float x[kDrawPer];
    draw_turn(tr, v, x);
    draw_collect<NTH>(D, tr, x, c0, lo, hi, top);
    const uint32_t tb = t < nt ? D.tbin[t] : 0u;
    if ((tb & 511u) == 0u) return;
    if (g == 0) m = low = fold::map_identity();
    fold::Map sm, sl;
    draw_tile_map(x, tb, sm, sl);
    m = fold::compose(m, sm);
    low = fold::compose(low, sl);
    if (g == r.mult - 1 && lane == 0) {
      D.tmap[t] = m;
      D.tlow[t] = low;
    }
  });
  __syncthreads();
  if (wid == 0) draw_chain<NTH>(D, r, 0, nt, -0.0f);
  __syncthreads();
}

// Wave 0: the end of the next piece by the histogram: bins from bin0 on
// while they hold at most kDrawPiece weights and, before the last one, less
// than `want` mass.  D.bnext: the bin after it (~0u: bin0 alone
// holds too many); D.lo: its smallest key.
template <int NTH>
__device__ __forceinline__ void draw_bins(DrawLds<NTH>& D, uint32_t bin0, float want) {
  const int lane = (int)(threadIdx.x & 63u);
  // lane l: 32 consecutive bins from bin0 + 32 l
  const uint32_t b0 = bin0 + 32u * (uint32_t)lane;
  uint32_t h[32];
  #pragma unroll
  for (uint32_t k = 0; k < 32u; ++k) {
    const uint32_t b = b0 + k;
    h[k] = b < (uint32_t)kDrawBins ? D.hist[draw_slot(b)] : 0u;
  }
  auto mid = [](uint32_t b) { return __uint_as_float(kOneBits - (min(b, (uint32_t)kDrawBins) << 17) - 0x10000u); };
  uint32_t c = 0u;
  float ms = 0.f;
  #pragma unroll
  for (uint32_t k = 0; k < 32u; ++k) {
    c += h[k];
    ms += (float)h[k] * mid(b0 + k);
  }
  uint32_t cum = wave_incl_scan_u32(c) - c;
  float mass = (float)(fold::wave_scan_f64((double)ms) - (double)ms);
  uint32_t end = b0;  // this lane's bins [b0, end) are taken
  bool stop = false;
  #pragma unroll
  for (uint32_t k = 0; k < 32u; ++k) {
    const uint32_t b = b0 + k;
    stop = stop || b >= (uint32_t)kDrawBins || cum + h[k] > (uint32_t)kDrawPiece || mass >= want;
    cum += h[k];
    mass += (float)h[k] * mid(b);
    end = stop ? end : b + 1u;
  }
  const uint64_t st = __ballot(stop);
  const int l = st ? __ffsll((unsigned long long)st) - 1 : 63;
  const uint32_t bend = (uint32_t)__builtin_amdgcn_readlane((int)end, l);
  if (lane == 0) {
    D.bnext = bend == bin0 ? 0xffffffffu : bend;
    D.lo = bend >= (uint32_t)kDrawBins ? (1ull << 23) : (uint64_t)(kOneBits - (bend << 17) + 1u) << 23;
  }
}

// The end of the next piece below `hi` (exclusive, a draw_key) when the
// histogram gives none: a descent over the keys, 11 bits a pass over the
// row, which overwrites the histogram.  All threads call it.
template <int NTH>
__device__ __forceinline__ void draw_descend(DrawLds<NTH>& D, const DrawRow& r, uint64_t hi) {
  constexpr uint32_t kP = (uint32_t)kDrawPiece;
  const int tid = threadIdx.x, lane = tid & 63;
  // from the top, the key bins that fit; when the first nonempty one does
  // not, its own bits
  uint64_t prefix = 0ull;
  int prev = 63, shift = 42;
  while (true) {
    __syncthreads();
    for (int b = tid; b < kDrawBins + kDrawBins / 32; b += NTH) D.hist[b] = 0u;
    __syncthreads();
    const uint32_t mask = shift == 0 ? 511u : 2047u;
    draw_stream<NTH>(r, r.w, [&](int, int, int c0, const float (&x)[4][4]) {
      #pragma unroll
      for (int j = 0; j < 4; ++j) {
        #pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint64_t k = draw_key(x[j][q], c0 + j * 256 + lane * 4 + q);
          if (x[j][q] > 0.f && k < hi && (prev == 63 || (k >> prev) == prefix))
            atomicAdd(&D.hist[draw_slot((uint32_t)(k >> shift) & mask)], 1u);
        }
      }
    });
    __syncthreads();
    if (tid < 64) {
      // from bin 2047 down, 32 bins a lane (rolled for four waves: the loads
      // of all 32 in flight made this rare path those kernels' register peak,
      // 256 + 12 instead of 214; sixteen waves have 128 either way, and the
      // mixed rows of the row kernel take 0.7% longer rolled)
      constexpr int kRolled = NTH >= 1024 ? 32 : 4, kRolled1 = NTH >= 1024 ? 32 : 1;
      uint32_t c = 0u;
      #pragma unroll kRolled
      for (int k = 0; k < 32; ++k) c += D.hist[draw_slot((uint32_t)(2047 - 32 * lane - k))];
      uint32_t cum = wave_incl_scan_u32(c) - c;
      int low = -1, first = -1;  // the last bin that still fits; the first nonempty one
      bool stop = false;
      #pragma unroll kRolled1
      for (int k = 0; k < 32 && !stop; ++k) {
        const int b = 2047 - 32 * lane - k;
        const uint32_t h = D.hist[draw_slot((uint32_t)b)];
        if (h != 0u && cum == 0u && first < 0) first = b;
        if (cum + h > kP) { stop = true; break; }
        cum += h;
        low = b;
      }
      const uint64_t st = __ballot(stop);
      const int l = st ? __ffsll((unsigned long long)st) - 1 : 63;
      int lw = __builtin_amdgcn_readlane(low, l);
      const uint32_t taken = (uint32_t)__builtin_amdgcn_readlane((int)cum, l);
      if (lw < 0) lw = 2048 - 32 * l;  // none of lane l's bins: down to the lane before
      const uint64_t fb = __ballot(first >= 0);
      const int fl = fb ? __ffsll((unsigned long long)fb) - 1 : 0;
      const int fbin = __builtin_amdgcn_readlane(first, fl);
      if (lane == 0) {
        D.n = taken;
        D.token = (uint32_t)fbin;
        D.lo = (uint64_t)lw;
      }
    }
    __syncthreads();
    const uint64_t base = prev == 63 ? 0ull : prefix << prev;
    const uint64_t lw = D.lo;
    const uint32_t taken = D.n, fbin = D.token;
    __syncthreads();
    if (taken != 0u || fbin == 0xffffffffu) {
      if (tid == 0) {
        const uint64_t lo = base + (lw << shift);
        D.lo = lo < (1ull << 23) ? (1ull << 23) : lo;
      }
      break;
    }
    prefix = (base >> shift) + fbin;
    prev = shift;
    shift = shift > 11 ? shift - 11 : 0;
  }
  __syncthreads();
}

// One stable radix pass over the keys src[0 .. n) by the kDigit bits at
// `shift`, out(p, key) placing each key at its position p.  A wave takes a
// run of 64-key groups: the lanes of a digit find each other by ballots, the
// digit's count so far gives their positions within the wave, and a scan of
// the digits over the waves their bases.  Nine bits sort the 27 of a nucleus
// over 16 binades in three passes.  All threads call it.
template <int NTH, typename OutF>
__device__ __forceinline__ void draw_radix_pass(DrawLds<NTH>& D, const uint32_t* src, int n, int shift, OutF out) {
  constexpr int kW = NTH / 64;
  constexpr int kPer = kDrawPiece / NTH;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int groups = (n + 63) / 64, per = (groups + kW - 1) / kW;  // per <= kPer
  uint32_t* cnt = D.u.p.v.so.cnt[wid];
  #pragma unroll
  for (int d = 0; d < kDrawDigits; d += 64) cnt[d + lane] = 0u;
  const uint64_t below = ((uint64_t)1 << lane) - 1u;
  uint32_t key[kPer], pos[kPer];
  #pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int i = (wid * per + k) * 64 + lane;
    key[k] = k < per && i < n ? src[i] : 0u;
  }
  wave_lds_sync();
  #pragma unroll
  for (int k = 0; k < kPer; ++k) {
    if (k >= per) break;
    const int i = (wid * per + k) * 64 + lane;
    const bool on = i < n;
    const uint32_t dg = (key[k] >> shift) & (uint32_t)(kDrawDigits - 1);
    uint64_t peers = __ballot(on);
    #pragma unroll
    for (int b = 0; b < kDrawDigitBits; ++b) {
      const bool bit = (dg >> b) & 1u;
      const uint64_t m = __ballot(bit);
      peers &= bit ? m : ~m;
    }
    const uint32_t r = (uint32_t)__popcll(peers & below);
    const uint32_t old = cnt[dg];
    pos[k] = old + r;
    if (on && r == 0u) cnt[dg] = old + (uint32_t)__popcll(peers);
    wave_lds_sync();
  }
  __syncthreads();
  {
    // digit bases: thread t takes the digits 2 t and 2 t + 1
    constexpr int kD = 2;
    static_assert(kDrawDigits == kD * 256, "two digits a thread");
    uint32_t c[kD][kW], tot = 0u;
    if (tid < 256) {
      #pragma unroll
      for (int d = 0; d < kD; ++d) {
        #pragma unroll
        for (int w = 0; w < kW; ++w) {
          c[d][w] = D.u.p.v.so.cnt[w][kD * tid + d];
          tot += c[d][w];
        }
      }
    }
    uint32_t all;
    uint32_t base = block_excl_scan_u32<NTH>(tot, D.red, &all);
    if (tid < 256) {
      #pragma unroll
      for (int d = 0; d < kD; ++d) {
        #pragma unroll
        for (int w = 0; w < kW; ++w) {
          D.u.p.v.so.cnt[w][kD * tid + d] = base;
          base += c[d][w];
        }
      }
    }
  }
  __syncthreads();
  #pragma unroll
  for (int k = 0; k < kPer; ++k) {
    if (k >= per) break;
    const int i = (wid * per + k) * 64 + lane;
    if (i < n) out(cnt[(key[k] >> shift) & (uint32_t)(kDrawDigits - 1)] + pos[k], key[k]);
  }
  __syncthreads();
}

// Sorts the gathered keys of the piece [lo, hi) and puts its weights in rank
// order in D.wf(); returns their number.  All threads call it.
template <int NTH>
__device__ __forceinline__ int draw_sort(DrawLds<NTH>& D, uint64_t lo, uint64_t hi) {
  const int tid = threadIdx.x;
  const uint32_t top = (uint32_t)((hi - 1u) >> 23);
  const int n = min((int)D.n, kDrawPiece);
  const int bits = 32 - __clz((int)((top - (uint32_t)(lo >> 23)) | 1u));
  const int J = max(1, (n + kDrawBlocks - 1) / kDrawBlocks), ld = J | 1;
  uint32_t *src = D.u.p.key0, *dst = D.u.p.v.so.key1;
  for (int shift = 0; shift < bits; shift += kDrawDigitBits) {
    draw_radix_pass<NTH>(D, src, n, shift, [&](uint32_t p, uint32_t k) { dst[p] = k; });
    uint32_t* x = src;
    src = dst;
    dst = x;
  }
  constexpr int kPer = kDrawPiece / NTH;
  float x[kPer];
  #pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int i = k * NTH + tid;
    x[k] = i < n ? __uint_as_float(top - src[i]) : 0.f;
  }
  __syncthreads();  // the weights take the keys' place
  float* wf = D.wf();
  #pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int i = k * NTH + tid;
    if (i < n) wf[(i / J) * ld + i % J] = x[k];
  }
  __syncthreads();
  return n;
}

// Gathers the piece [lo, hi).  All threads call it.
template <int NTH>
__device__ __forceinline__ void draw_gather(DrawLds<NTH>& D, const DrawRow& r, uint64_t lo, uint64_t hi) {
  __syncthreads();
  if (threadIdx.x == 0) D.n = 0u;
  __syncthreads();
  const uint32_t top = (uint32_t)((hi - 1u) >> 23);
  float* tr = D.u.p.v.tr[threadIdx.x >> 6];
  draw_stream<NTH>(r, r.w, [&](int, int, int c0, const float (&v)[4][4]) {
    float x[kDrawPer];
    draw_turn(tr, v, x);
    draw_collect<NTH>(D, tr, x, c0, lo, hi, top);
  });
  __syncthreads();
}

// The ord-th (from 0) smallest index among the row's weights equal to w with
// keys in [lo, hi).  All threads call it.
template <int NTH>
__device__ __forceinline__ uint32_t draw_index(DrawLds<NTH>& D, const DrawRow& r, float w, uint32_t ord, uint64_t lo,
                                               uint64_t hi) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int span = 64 * kDrawPer * r.mult;
  const int nt = (r.V + span - 1) / span;
  const uint32_t wb = __float_as_uint(w);
  // of the equal weights, the indexes in the piece
  const int i0 = (uint32_t)((hi - 1u) >> 23) == wb ? 0x7fffff - (int)((hi - 1u) & 0x7fffffu) : 0;
  const int i1 = (uint32_t)(lo >> 23) == wb ? 0x7fffff - (int)(lo & 0x7fffffu) : 0x7fffff;
  auto is = [&](float x, int i) { return __float_as_uint(x) == wb && i >= i0 && i <= i1; };
  // matches per tile, then the tile by a scan, then its logits in order
  uint32_t c = 0u;
  draw_stream<NTH>(r, r.w, [&](int t, int g, int c0, const float (&x)[4][4]) {
    if (g == 0) c = 0u;
    #pragma unroll
    for (int j = 0; j < 4; ++j)
      #pragma unroll
      for (int q = 0; q < 4; ++q) c += is(x[j][q], c0 + j * 256 + lane * 4 + q) ? 1u : 0u;
    if (g == r.mult - 1) {
      const uint32_t s = wave_sum_u32(c);
      if (lane == 0 && t < nt) D.u.p.v.tcnt[t] = s;
    }
  });
  __syncthreads();
  if (wid == 0) {
    uint32_t seen = 0u, tok = 0u;
    for (int tb = 0; tb < nt; tb += 64) {
      const uint32_t k = tb + lane < nt ? D.u.p.v.tcnt[tb + lane] : 0u;
      const uint32_t inc = wave_incl_scan_u32(k);
      const uint64_t hit = __ballot(seen + inc > ord);
      if (hit == 0ull) {
        seen += wave_last_u32(inc);
        continue;
      }
      const int l = __ffsll((unsigned long long)hit) - 1;
      seen += (uint32_t)__builtin_amdgcn_readlane((int)(inc - k), l);
      for (int g = 0; g < r.mult; ++g) {
        const int c0 = (tb + l) * span + g * 64 * kDrawPer;
        float x[kDrawPer];
        draw_lane_terms(r, c0, x);
        uint32_t mk = 0u;
        #pragma unroll
        for (int q = 0; q < kDrawPer; ++q) mk |= is(x[q], c0 + lane * kDrawPer + q) ? 1u << q : 0u;
        const uint32_t n = (uint32_t)__popc(mk), in = wave_incl_scan_u32(n);
        const uint64_t h = __ballot(seen + in > ord);
        if (h != 0ull) {
          const int f = __ffsll((unsigned long long)h) - 1;
          for (uint32_t q = seen + in - n; q < ord; ++q) mk &= mk - 1u;  // (lane f's: the matches before)
          tok = (uint32_t)__builtin_amdgcn_readlane(c0 + lane * kDrawPer + __ffs((int)mk) - 1, f);
          break;
        }
        seen += wave_last_u32(in);
      }
      break;
    }
    if (lane == 0) D.token = tok;
  }
  __syncthreads();
  return D.token;
}

// The folds of the first `lim` of the piece's n weights: wave 0 folds w /
// total from c0, wave 1 w from t0; D.u.p.v.start gets their values before
// each block and D.end the last ones.
template <int NTH>
__device__ __forceinline__ void draw_folds(DrawLds<NTH>& D, int n, int lim, float total, float c0, float t0) {
  const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
  constexpr int kMost = kDrawPiece / kDrawBlocks;
  const int J = max(1, (n + kDrawBlocks - 1) / kDrawBlocks), ld = J | 1;
  const float* wf = D.wf();
  if (wid < 2) {
    float acc = wid == 0 ? c0 : t0;
    for (int b = 0; b * J < n; b += 64) {
      const int blk = b + lane;
      float x[kMost];
      #pragma unroll
      for (int k = 0; k < kMost; ++k) x[k] = k < J && blk * J + k < lim ? wf[blk * ld + k] : 0.f;
      if (wid == 0) {
        #pragma unroll
        for (int k = 0; k < kMost; ++k) if (k < J) x[k] = x[k] / total;
      }
      acc = wave_fold_blocks(x, acc, [&](float v) { D.u.p.v.start[wid][blk] = v; });
    }
    if (lane == 0) D.end[wid] = acc;
  }
  __syncthreads();
}

template <int NTH>
__device__ __forceinline__ uint32_t draw_block_min(DrawLds<NTH>& D, uint32_t v) {
  return ~block_max_u32<NTH>(~v, D.red);
}

// Where the ranks' weights come from: the row's weights in ws_w.
template <int NTH>
struct DrawRowSrc {
  const DrawRow& r;
  bool whole;  // holds every positive weight of the row
  __device__ __forceinline__ void gather(DrawLds<NTH>& D, uint64_t lo, uint64_t hi) const { draw_gather<NTH>(D, r, lo, hi); }
  __device__ __forceinline__ bool descend(DrawLds<NTH>& D, uint64_t hi) const {
    draw_descend<NTH>(D, r, hi);
    return true;
  }
  __device__ __forceinline__ uint32_t index(DrawLds<NTH>& D, float w, uint32_t ord, uint64_t lo, uint64_t hi) const {
    return draw_index<NTH>(D, r, w, ord, lo, hi);
  }
};

// The next piece below hi, in rank order in D.wf(): its smallest key in lo,
// its length returned, `bin` advanced to the histogram bin after it (~0u
// once pieces come from the descent).  -1: the source cannot give it.  All
// threads call it.
template <int NTH, typename Src>
__device__ __forceinline__ int draw_piece(DrawLds<NTH>& D, const Src& src, uint64_t hi, uint64_t& lo, uint32_t& bin) {
  if (bin != 0xffffffffu) {
    __syncthreads();
    if (threadIdx.x < 64) draw_bins<NTH>(D, bin, __builtin_inff());
    __syncthreads();
    bin = D.bnext;
    lo = D.lo;
  }
  if (bin == 0xffffffffu) {
    if (!src.descend(D, hi)) return -1;
    lo = D.lo;
  }
  src.gather(D, lo, hi);
  return draw_sort<NTH>(D, lo, hi);
}

constexpr uint64_t kDrawAll = ((uint64_t)kOneBits + 1u) << 23;  // above every key
constexpr uint64_t kDrawEnd = 1ull << 23;                       // no positive weight has a smaller key
constexpr uint32_t kDrawFallback = 0xffffffffu;                 // the argmax fallback
constexpr uint32_t kDrawRetry = 0xfffffffeu;                    // the source does not hold the nucleus

// Step 3, from the normaliser `total`: ranks until the cutoff (or k ranks,
// k > 0), the candidate total (also in *ct_out), the drawn index.  ready:
// the first piece [lo, kDrawAll) is gathered and `bin` is the bin after it.
// All threads call it.
template <int NTH, typename Src>
__device__ __forceinline__ uint32_t draw_ranks(DrawLds<NTH>& D, const Src& src, const RowCfg& cfg, int k, float total,
                                               bool ready, uint64_t lo, uint32_t bin, float* ct_out) {
  const int tid = threadIdx.x;
  const bool cut = cfg.cutoff < 1.f;
  const float* wf = D.wf();
  uint64_t hi = kDrawAll;
  float cum = 0.f, ct = -0.0f;
  int seen = 0, nrec = 0;  // ranks of the pieces before this one
  int n, cnt;              // the piece's ranks, and the candidates among the last one's
  float ct0;               // the candidate total before it
  while (true) {
    n = ready ? draw_sort<NTH>(D, lo, hi) : draw_piece<NTH>(D, src, hi, lo, bin);
    ready = false;
    if (n < 0) return kDrawRetry;
    if (tid == 0 && nrec < kDrawRecs) {
      D.rec_hi[nrec] = hi;
      D.rec_ct[nrec] = ct;
    }
    nrec = min(nrec + 1, kDrawRecs);
    const int lim = k ? min(n, k - seen) : n;
    draw_folds<NTH>(D, n, lim, total, cum, ct);
    ct0 = ct;
    // the first rank whose cum_p reaches the cutoff
    const int J = max(1, (n + kDrawBlocks - 1) / kDrawBlocks), ld = J | 1;
    uint32_t first = 0xffffffffu;
    if (cut && tid < kDrawBlocks && tid * J < lim) {
      float c = D.u.p.v.start[0][tid];
      for (int q = 0; q < J && tid * J + q < lim; ++q) {
        c += wf[tid * ld + q] / total;
        if (c >= cfg.cutoff) { first = (uint32_t)(tid * J + q); break; }
      }
    }
    first = draw_block_min<NTH>(D, first);
    const bool last = (k && seen + lim >= k) || lo <= kDrawEnd || bin == (uint32_t)kDrawBins;
    if (first == 0xffffffffu && last && !src.whole) return kDrawRetry;
    if (first != 0xffffffffu || last) {
      cnt = first != 0xffffffffu ? (int)first + 1 : lim;
      if (cnt == lim) {
        ct = D.end[1];
      } else {
        // the candidate total after cnt ranks, by the thread of their block
        const int b = (cnt - 1) / J;
        if (tid == b) {
          float c = D.u.p.v.start[1][b];
          for (int i = b * J; i < cnt; ++i) c += wf[b * ld + (i - b * J)];
          D.ct = c;
        }
        __syncthreads();
        ct = D.ct;
      }
      break;
    }
    cum = D.end[0];
    ct = D.end[1];
    seen += n;
    hi = lo;
    __syncthreads();
  }
  if (ct_out && tid == 0) *ct_out = ct;
  if (seen + cnt <= 0 || !(ct > 0.f) || !finitef_(ct)) return kDrawFallback;
  const float target = clamp_uniform(cfg.u) * ct;
  // the inverse CDF: in the piece in LDS, or an earlier one gathered again
  if (target < ct0) {
    __syncthreads();
    int q = 0;
    for (int p = 1; p < nrec; ++p) q = D.rec_ct[p] <= target ? p : q;
    hi = D.rec_hi[q];
    float c0 = D.rec_ct[q];
    while (true) {
      // the pieces of the first pass again: each ends where the next record
      // starts, or (past the records) where the descent says
      __syncthreads();
      if (q + 1 < nrec) {
        lo = D.rec_hi[q + 1];
      } else {
        if (!src.descend(D, hi)) return kDrawRetry;
        lo = D.lo;
      }
      src.gather(D, lo, hi);
      n = draw_sort<NTH>(D, lo, hi);
      draw_folds<NTH>(D, n, n, 1.f, 0.f, c0);
      if (target < D.end[1] || lo <= kDrawEnd) break;
      c0 = D.end[1];
      hi = lo;
      ++q;
    }
    cnt = n;
  }
  const int J = max(1, (n + kDrawBlocks - 1) / kDrawBlocks), ld = J | 1;
  uint32_t pick = 0xffffffffu;
  if (tid < kDrawBlocks && tid * J < cnt) {
    float c = D.u.p.v.start[1][tid];
    for (int q = 0; q < J && tid * J + q < cnt; ++q) {
      c += wf[tid * ld + q];
      if (target < c) { pick = (uint32_t)(tid * J + q); break; }
    }
  }
  pick = draw_block_min<NTH>(D, pick);
  if (pick == 0xffffffffu) pick = (uint32_t)max(cnt, 1) - 1u;  // gpu.rs:899: the last candidate
  // its index: equal weights rank by index, so the pick is the ord-th match
  // of its weight in the piece, ord the equal weights of lower rank
  const float w = wf[((int)pick / J) * ld + (int)pick % J];
  uint32_t same = pick;
  for (int i = tid; i < (int)pick; i += NTH)
    if (wf[(i / J) * ld + i % J] == w) same = min(same, (uint32_t)i);
  same = draw_block_min<NTH>(D, same);
  __syncthreads();
  const uint32_t tok = src.index(D, w, pick - same, lo, hi);
  __syncthreads();
  return tok;
}

// The whole draw (gpu.rs:820-899) for a top-p row, or a top-k row of more
// than kBuf ranks.  Returns the token, or kDrawFallback for the argmax
// fallback.  All threads call it.
template <int NTH>
__device__ __forceinline__ uint32_t draw_ranked(DrawLds<NTH>& D, const SampleArgs& a, int row, const RowCfg& cfg,
                                                float M) {
  const int tid = threadIdx.x;
  const DrawRow r = draw_row<NTH>(a, row);
  const DrawRowSrc<NTH> src{r, true};
  const int span = 64 * kDrawPer * r.mult;
  const int nt = (r.V + span - 1) / span;
  draw_weights<NTH>(D, r, M, cfg.min_p);
  const int k = cfg.cls == kTopK ? cfg.k_eff : 0;
  const bool cut = cfg.cutoff < 1.f;
  uint64_t lo = 0ull;
  uint32_t bin;
  bool ready = false;  // the first piece is gathered
  float total;
  if (k == 0) {
    // the first piece: the bins of the nucleus by their mass (within 0.8%)
    if (tid >= 64 && tid < 128) draw_predict<NTH>(D, nt);
    if (tid < 64) {
      float s = 0.f;
      for (int t = tid; t < nt; t += 64) s += D.tsum[t];
      draw_bins<NTH>(D, 0u, cut ? (cfg.cutoff * 1.008f + 0.002f) * wave_sum_f32(s) : __builtin_inff());
    }
    if (tid == 0) D.n = 0u;
    __syncthreads();
    bin = D.bnext;
    lo = D.lo;
    ready = bin != 0xffffffffu;
    // (no first piece by the histogram: gather nothing)
    draw_total<NTH>(D, r, ready ? lo : kDrawAll, kDrawAll);
    total = D.total;
  } else {
    // the normaliser of the top k, in rank order
    float t = -0.0f;
    int seen = 0;
    uint64_t hi = kDrawAll;
    bin = 0u;
    while (true) {
      const int n = draw_piece<NTH>(D, src, hi, lo, bin);
      draw_folds<NTH>(D, n, min(n, k - seen), 1.f, 0.f, t);
      t = D.end[1];
      seen += n;
      if (seen >= k || lo <= kDrawEnd || bin == (uint32_t)kDrawBins) break;
      hi = lo;
    }
    if (bin != 0xffffffffu) bin = 0u;  // from the top again
    total = t;
  }
  __syncthreads();
  if (!(total > 0.f) || !finitef_(total)) return kDrawFallback;
  return draw_ranks<NTH>(D, src, cfg, k, total, ready, lo, bin, nullptr);
}

// The sum of the row's reference chunk [start, end): left to right from
// +0.0, by the Q lanes of a quad (or one lane), 16 logits a step, the next
// step's loads in flight.
template <int Q>
__device__ __forceinline__ float draw_chunk_sum(__amdgpu_buffer_rsrc_t s, int start, int end, float M,
                                                const Exp2TabLds& et) {
  constexpr int kN = 16 / Q;
  const int q0 = (int)(threadIdx.x & (Q - 1)) * kN;
  i32x4_t v[kN / 4];
  auto issue = [&](int b) {
    #pragma unroll
    for (int j = 0; j < kN / 4; ++j) v[j] = __builtin_amdgcn_raw_buffer_load_b128(s, (b + q0 + 4 * j) * 4, 0, 0);
  };
  issue(start);
  float sum = 0.f;
  for (int b = start; b < end; b += 16) {
    float w[kN];
    #pragma unroll
    for (int j = 0; j < kN; ++j) w[j] = b + q0 + j < end ? __int_as_float(v[j / 4][j % 4]) : -__builtin_inff();
    issue(b + 16);
    #pragma unroll
    for (int j = 0; j < kN; ++j) w[j] = exact_expf_neg(w[j] - M, et);
    if (Q == 1) {
      #pragma unroll
      for (int j = 0; j < kN; ++j) sum += w[j];
    } else {
      auto from = [&](auto ctl) {
        constexpr int C = decltype(ctl)::c;
        #pragma unroll
        for (int j = 0; j < kN; ++j) sum += __uint_as_float(dpp32<C>(0u, __float_as_uint(w[j])));
      };
      from(fold::DppStep<0x00, 0xf, false>{});  // quad_perm [0,0,0,0], ..., [3,3,3,3]
      from(fold::DppStep<0x55, 0xf, false>{});
      from(fold::DppStep<0xaa, 0xf, false>{});
      from(fold::DppStep<0xff, 0xf, false>{});
    }
  }
  return sum;
}

// The reference's rescan of chunk [s0, s1) by one wave: the first index
// whose running sum from `c` passes target, else the last positive weight's
// (~0u: none), 512 logits loaded at a time.
__device__ __forceinline__ uint32_t draw_chunk_find(__amdgpu_buffer_rsrc_t s, int s0, int s1, float c, float target,
                                                    float M, const Exp2TabLds& et) {
  const int lane = (int)(threadIdx.x & 63u);
  constexpr int kG = 8;
  uint32_t chosen = 0xffffffffu;
  for (int b = s0; b < s1; b += 64 * kG) {
    float w[kG];
    #pragma unroll
    for (int g = 0; g < kG; ++g)
      w[g] = __int_as_float((int)__builtin_amdgcn_raw_buffer_load_b32(s, (b + 64 * g + lane) * 4, 0, 0));
    #pragma unroll
    for (int g = 0; g < kG; ++g) w[g] = b + 64 * g + lane < s1 ? exact_expf_neg(w[g] - M, et) : 0.f;
    #pragma unroll
    for (int g = 0; g < kG; ++g) {
      if (b + 64 * g >= s1) break;
      const float r = wave_fold_f32(w[g], c, 64);
      const uint64_t pos = __ballot(w[g] > 0.f);
      const uint64_t hit = __ballot(w[g] > 0.f && target < r);
      if (hit != 0ull) return (uint32_t)(b + 64 * g + __ffsll((unsigned long long)hit) - 1);
      if (pos != 0ull) chosen = (uint32_t)(b + 64 * g + 63 - __clzll((long long)pos));
      c = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(r), 63));
    }
  }
  return chosen;
}

// The draw of a temperature-only row from its reference chunks' sums
// (D.u.to.csum; the exponential's table in D.exptab): their serial prefix,
// then the owning chunk again (kernels.cu:7834-7867).  Returns the token or
// argmax_fin.  All threads call it.
template <int NTH>
__device__ __forceinline__ uint32_t draw_chunk_pick(DrawLds<NTH>& D, const DrawRow& r, float M, float u,
                                                    uint32_t argmax_fin) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int V = r.V;
  const int chunk = (V + 255) / 256;
  float* csum = D.u.to.csum;
  float* prefix = D.u.to.prefix;
  const Exp2TabLds et{D.exptab};
  if (tid < 64) {
    float acc = 0.f;
    #pragma unroll 1
    for (int b = 0; b < 256; b += 64) {
      const float inc = wave_fold_f32(csum[b + lane], acc, 64);
      const float ex = wave_fold_u(inc);  // the lane below
      prefix[b + lane] = lane == 0 ? acc : ex;
      acc = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(inc), 63));
    }
    const float total = acc;
    uint32_t tok = 0xffffffffu;
    if (total > 0.f && finitef_(total)) {
      const float uu = finitef_(u) ? fminf(fmaxf(u, 0.f), 0.99999994f) : 0.f;
      const float target = uu * total;
      wave_lds_sync();
      #pragma unroll 1
      for (int b = 0; b < 256; b += 64) {
        const int t = b + lane;
        const int start = t * chunk, end = min(start + chunk, V);
        const float lo = prefix[t], hi = lo + csum[t];
        uint64_t own = __ballot(start < end && target >= lo && (target < hi || t == 255));
        while (own != 0ull) {
          const int l = __ffsll((unsigned long long)own) - 1;
          own &= own - 1ull;
          const int s0 = (b + l) * chunk, s1 = min(s0 + chunk, V);
          const float c = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(lo), l));
          const uint32_t chosen = draw_chunk_find(r.s, s0, s1, c, target, M, et);
          tok = chosen < tok ? chosen : tok;
        }
      }
    }
    if (lane == 0) D.token = tok;
  }
  __syncthreads();
  const uint32_t tok = D.token;
  __syncthreads();
  return tok != 0xffffffffu ? tok : argmax_fin;
}

// Temperature-only rows: kernels.cu:7803-7867 with the exact weight
// function: 256 contiguous chunks, a lane (or a quad) each, then
// draw_chunk_pick.  All threads call it.
template <int NTH>
__device__ __forceinline__ uint32_t draw_temperature(DrawLds<NTH>& D, const SampleArgs& a, int row, float M, float u,
                                                     uint32_t argmax_fin) {
  constexpr int Q = NTH / 256;
  static_assert(Q == 1 || Q == 4, "a lane or a quad per reference chunk");
  const int tid = threadIdx.x, lane = tid & 63;
  const DrawRow r = draw_row<NTH>(a, row);
  const int V = r.V;
  const int chunk = (V + 255) / 256;
  float* csum = D.u.to.csum;
  if (tid < 32) D.exptab[tid] = exp2_tab32((uint32_t)tid);
  __syncthreads();
  const Exp2TabLds et{D.exptab};
  {
    const int t = tid / Q;
    const int start = t * chunk, end = min(start + chunk, V);
    const float s = draw_chunk_sum<Q>(r.s, start, end, M, et);
    if ((tid & (Q - 1)) == 0) csum[t] = s;
  }
  __syncthreads();
  return draw_chunk_pick<NTH>(D, r, M, u, argmax_fin);
}

}  // namespace hi_rocm
