// batch.hip -- many uneven scans / reduces in one persistent launch.
//
// No reference counterpart: the reference launches one scan or reduce per
// binary (scan/main.cu, Reduce/test_reduce.cu).  The segments of a batch lie one
// after another, so the batch is treated as ONE array with a head bit at every
// segment start, cut into fixed tiles whatever the segments are: a tile may
// hold many short segments or a part of a long one, and the cost of a batch
// depends on its elements, not on its segments.
//
// Scan: workgroups take tiles in increasing order from one counter (work
// stealing).  Sums are mod 2^32, a group, so a tile is scanned flat and every
// element subtracts the flat prefix at its segment's head; a wave finds that
// head with one ballot and one shuffle per 256 elements, and skips both where no
// head falls.  The carry of a tile's first segment comes from a decoupled
// look-back (Merrill & Garland, "Single-pass Parallel Prefix Scan with
// Decoupled Look-back", 2016) over its predecessors: a tile publishes a 64-bit
// status word {flag:2, value:32} with one device-scope store (the value travels
// inside the word: no cache writeback or invalidate).  A tile with a head
// publishes the sum since its last head as final at once, so a look-back never
// reaches past the segment.  The status words are cleared by a fill kernel
// before every launch.  Look-back waits are bounded: a wait that exceeds the spin
// limit records an error word and the workgroup exits.
//
// Reduce: every wave sums spans of its workgroup's share; a span with heads
// writes its flat prefixes to LDS, and lane after lane takes a segment of the
// span as a difference of two of them (a part of a segment is added to its sum
// with a device-scope atomic: uint32 wrap, order-independent, bit-exact).
//
// Every element is read once and (scan) written once: 8 / 4 bytes per element.
#include <hip/hip_runtime.h>

#include "hs_internal.hpp"
#include "hs_wave.hpp"

using namespace hs;

namespace {

constexpr int kWg = 256;  // prep and reduce
constexpr int kWaves = kWg / 64;
// Shapes of the scan's tiles: workgroup size and wave span in 256-element segments
// (4 registers per lane each).  With 128 registers a workgroup is half of a CU: two run
// on each, and one finds room beside the serving loop's workgroup (1024 threads, one
// workgroup per CU, waited there until the loop's end; 512 ragged segments in 392 us
// against 399, one of 2^24 elements in 53 against 58).
// Early: the next tile is claimed when this one's carry is known, so that the atomic's
// round trip runs beside the stores (one segment of 2^22 elements 38.1 -> 35.2 us).
// With large tiles it starts them out of order, and the look-backs wait (2^27: 229 ->
// 239 us).
struct Large { static constexpr int kWg = 512, kSegs = 16; static constexpr bool kEarly = false; };  // 32768 elements
struct Small { static constexpr int kWg = 512, kSegs = 8; static constexpr bool kEarly = true; };    // 16384 elements
constexpr int kSegsReduce = 8;
// Elements from which a scan takes the large tiles (one segment, us per call with
// small and large tiles: 2^22 35.2 / 43.9, 2^23 44.8 / 45.8, 2^24 57.7 / 59.2, 2^24.6
// 72.4 / 73.3, 2^25 87.3 / 82.9, 2^27 260 / 229): more elements per tile mean fewer
// look-backs and claims, fewer mean that more compute units have one.
constexpr uint64_t kLargeFrom = 7ull << 22;
constexpr uint64_t kFlagAgg = 1, kFlagInc = 2;
constexpr uint32_t kSpinLimit = 1u << 26;

__host__ __device__ constexpr int span_of(int segs) { return 256 * segs; }
template <class T>
constexpr int tile_of() { return T::kWg / 64 * span_of(T::kSegs); }

__device__ __forceinline__ uint64_t pack(uint64_t flag, uint32_t v) { return (flag << 32) | v; }

struct BatchArgs {
  const uint32_t *in;
  uint32_t *out;               // scan output (same layout as in) or per-segment sums (reduce)
  const uint64_t *offsets;     // [nseg+1] element offsets of the segments
  const uint32_t *span_seg;    // [nspans+1] first segment that starts at or after the span
  uint32_t nseg;
  uint64_t lo, hi;             // the batch's elements: offsets[0], offsets[nseg]
  uint64_t base;               // lo aligned down to 16 bytes: where span 0 starts
  uint64_t ntiles, nspans;
  uint64_t *status;            // [ntiles] look-back words
  uint32_t *counter;           // tile counter (zeroed by the prep kernel)
  uint32_t *error;             // set when a look-back wait gives up
};

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Next value of a counter.  atomic_inc, as the compiler rewrites a uniform add
// into one that is waited for on the spot.
__device__ __forceinline__ uint32_t claim_next(uint32_t *c) { return inc_wrap(c, 0xFFFFFFFFu); }

// One wave's span of elements starting at `base` (16-byte aligned): x[q] of lane l
// holds elements base + q*256 + 4l + 0..3, so every instruction of the wave
// touches 1 KiB of contiguous memory.  Every element is read once and written
// once, so spans inside the batch use non-temporal (streaming) 16-byte loads and
// stores: on a 2^28-element scan 0.412 ms against 0.433 ms with plain ones.
template <int SEGS>
__device__ __forceinline__ void wave_load(const uint32_t *in, uint64_t base, uint32_t lane, u32x4 (&x)[SEGS]) {
  const u32x4 *p = reinterpret_cast<const u32x4 *>(in + base) + lane;
#pragma unroll
  for (int q = 0; q < SEGS; ++q) x[q] = __builtin_nontemporal_load(p + q * 64);
}

template <int SEGS>
__device__ __forceinline__ void wave_store(uint32_t *out, uint64_t base, uint32_t lane, const u32x4 (&y)[SEGS]) {
  u32x4 *o = reinterpret_cast<u32x4 *>(out + base) + lane;
#pragma unroll
  for (int q = 0; q < SEGS; ++q) __builtin_nontemporal_store(y[q], o + q * 64);
}

// Four elements of a span that the batch's ends cut: positions [a, b) of the
// span are inside, the others read as 0 and are not written.
__device__ __forceinline__ u32x4 part_load(const uint32_t *in, uint64_t base, uint32_t i, uint32_t a, uint32_t b) {
  u32x4 v = {0u, 0u, 0u, 0u};
  if (i + 0 >= a && i + 0 < b) v.x = in[base + i + 0];
  if (i + 1 >= a && i + 1 < b) v.y = in[base + i + 1];
  if (i + 2 >= a && i + 2 < b) v.z = in[base + i + 2];
  if (i + 3 >= a && i + 3 < b) v.w = in[base + i + 3];
  return v;
}

__device__ __forceinline__ void part_store(uint32_t *out, uint64_t base, uint32_t i, uint32_t a, uint32_t b, u32x4 v) {
  if (i + 0 >= a && i + 0 < b) out[base + i + 0] = v.x;
  if (i + 1 >= a && i + 1 < b) out[base + i + 1] = v.y;
  if (i + 2 >= a && i + 2 < b) out[base + i + 2] = v.z;
  if (i + 3 >= a && i + 3 < b) out[base + i + 3] = v.w;
}

__device__ __forceinline__ uint32_t clip(uint64_t at, uint64_t base, uint32_t span) {
  return at <= base ? 0u : at - base < span ? (uint32_t)(at - base) : span;
}

__device__ __forceinline__ uint32_t ld_status_value(const uint64_t *p, uint64_t &flag) {
  const uint64_t w = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  flag = (w >> 32) & 3u;
  return (uint32_t)w;
}

// Carry into tile t: the sum since the last head before it, from the status
// words of its predecessors, 64 at a time: lane i looks at tile t-1-i (before
// tile 0: final zeros).  Waits until every lane up to the nearest final word is
// published.  Called by one whole wave.
__device__ __forceinline__ int lookback(const BatchArgs &p, uint64_t t, uint32_t lane, uint32_t &prefix) {
  prefix = 0;
  int64_t i = (int64_t)t - 1;
  uint32_t polls = 0;
  for (;;) {
    const int64_t idx = i - (int64_t)lane;
    uint64_t flag = kFlagInc;
    uint32_t v = 0;
    if (idx >= 0) v = ld_status_value(p.status + idx, flag);
    const uint64_t incm = __builtin_amdgcn_ballot_w64(flag == kFlagInc);
    const uint64_t readym = __builtin_amdgcn_ballot_w64(flag != 0);
    const uint32_t k = incm ? (uint32_t)__builtin_ctzll(incm) : 63u;
    const uint64_t need = k == 63 ? ~0ull : ((2ull << k) - 1ull);
    if ((readym & need) != need) {
      // give up uniformly across the wave (the error word is read once)
      if (++polls >= kSpinLimit || __builtin_amdgcn_readfirstlane(ld_relaxed(p.error))) return 1;
      __builtin_amdgcn_s_sleep(1);
      continue;
    }
    prefix += wave_sum(lane <= k ? v : 0u);
    if (incm) return 0;
    i -= 64;
  }
}

// Scan of 256 elements (4 per lane) behind the flat prefix `run`: `nib` holds the
// lane's four head bits, hbase the flat prefix at the last head so far.  Elements
// at or after a head subtract the flat prefix at the last head at or before them.
template <bool INCLUSIVE>
__device__ __forceinline__ void seg_scan_heads(u32x4 &x, uint32_t nib, uint32_t lane, uint32_t &run, uint32_t &hbase) {
  const uint32_t v4 = x[0] + x[1] + x[2] + x[3];
  const uint32_t inc = wave_incl_scan(v4);
  uint32_t pre = run + inc - v4;
  run += __builtin_amdgcn_readlane(inc, 63);
  const uint64_t hm = ballot(nib != 0);
  uint32_t b = hbase;
  if (hm) {
    uint32_t lh = pre;  // flat prefix at this lane's last head
    lh += nib >= 2 ? x[0] : 0u;
    lh += nib >= 4 ? x[1] : 0u;
    lh += nib >= 8 ? x[2] : 0u;
    const uint64_t m = hm & ((1ull << lane) - 1ull);
    const uint32_t got = __shfl(lh, m ? 63 - __builtin_clzll(m) : 0);
    if (m) b = got;
    hbase = __builtin_amdgcn_readlane(lh, 63 - __builtin_clzll(hm));
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t v = x[k];
      if (nib >> k & 1u) b = pre;
      x[k] = INCLUSIVE ? pre + v - b : pre - b;
      pre += v;
    }
  } else {
    pre -= b;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t v = x[k];
      if (INCLUSIVE) { pre += v; x[k] = pre; }
      else { x[k] = pre; pre += v; }
    }
  }
}

// head bits of the lane's four elements of segment q (bit i & 31 of word i >> 5)
__device__ __forceinline__ uint32_t head_bits(const uint32_t *bits, int q, uint32_t lane) {
  return (bits[q * 8 + (lane >> 3)] >> (4 * (lane & 7))) & 15u;
}

template <class T, bool INCLUSIVE>
__global__ void __launch_bounds__(T::kWg) __attribute__((amdgpu_waves_per_eu(4))) k_scan_batch(BatchArgs p) {
  constexpr int SEGS = T::kSegs;
  constexpr uint32_t kSpan = span_of(SEGS), kWaves = T::kWg / 64;
  constexpr bool kEarly = T::kEarly;
  __shared__ uint32_t s_tile, s_prefix;
  __shared__ uint32_t s_wave[kWaves], s_seen[kWaves], s_fh0;
  __shared__ uint32_t s_bits[kWaves][kSpan / 32];
  __shared__ int s_bad;
  const uint32_t lane = lane_id(), wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint32_t *bits = s_bits[wv];
  uint32_t claim = 0;
  if (kEarly && threadIdx.x == 0) claim = claim_next(p.counter);
  for (;;) {
    if (threadIdx.x == 0) s_tile = kEarly ? claim : claim_next(p.counter);
    __syncthreads();
    const uint64_t t = __builtin_amdgcn_readfirstlane(s_tile);
    if (t >= p.ntiles) return;
    const uint64_t sp = t * kWaves + wv;
    const uint64_t base = p.base + sp * kSpan;
    const uint32_t h0 = p.span_seg[sp], h1 = p.span_seg[sp + 1];  // heads of the span: [h0, h1)
    // the batch's ends cut only the first and the last tile's spans: those are
    // read twice, 256 elements at a time, and take no registers from the others
    const bool whole = base >= p.lo && base + kSpan <= p.hi;
    const uint32_t pa = clip(p.lo, base, kSpan), pb = clip(p.hi, base, kSpan);
    uint32_t fh = kSpan, run = 0, hbase = 0;
    auto mark_heads = [&]() {
      for (uint32_t i = lane; i < kSpan / 32; i += 64) bits[i] = 0;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      for (uint32_t s = h0 + lane; s < h1; s += 64) {
        const uint32_t pos = (uint32_t)(p.offsets[s] - base);
        __hip_atomic_fetch_or(bits + (pos >> 5), 1u << (pos & 31u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (h0 != h1) fh = (uint32_t)(p.offsets[h0] - base);
    };
    u32x4 x[SEGS];
    if (whole) {
      wave_load<SEGS>(p.in, base, lane, x);
      if (h0 != h1) mark_heads();
      // one path with and without heads, here and in the add below: with two, x
      // lives in two sets of registers where they meet
#pragma unroll
      for (int q = 0; q < SEGS; ++q) {
        seg_scan_heads<INCLUSIVE>(x[q], h0 != h1 ? head_bits(bits, q, lane) : 0u, lane, run, hbase);
      }
    } else {
      mark_heads();
#pragma unroll 1
      for (int q = 0; q < SEGS; ++q) {
        u32x4 v = part_load(p.in, base, q * 256 + 4 * lane, pa, pb);
        seg_scan_heads<INCLUSIVE>(v, head_bits(bits, q, lane), lane, run, hbase);
      }
    }
    run -= hbase;  // the sum since the span's last head
    if (lane == 0) {
      s_wave[wv] = run;
      s_seen[wv] = h0 != h1;
      if (wv == 0) s_fh0 = fh;
    }
    __syncthreads();
    // sum since the last head over the waves before this one, and over the tile
    uint32_t before = 0, seen_before = 0, agg = 0, seen = 0;
#pragma unroll
    for (uint32_t k = 0; k < kWaves; ++k) {
      const uint32_t w = s_wave[k], sn = s_seen[k];
      if (k < wv) { before = sn ? w : before + w; seen_before |= sn; }
      agg = sn ? w : agg + w;
      seen |= sn;
    }
    if (wv == 0) {
      // a head in the tile makes its word final at once; a head at its first
      // element makes the look-back unnecessary
      uint32_t prefix = 0;
      int bad = 0;
      const bool fin = seen || t == 0;
      if (lane == 0)
        __hip_atomic_store(p.status + t, pack(fin ? kFlagInc : kFlagAgg, agg), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      if (t != 0 && s_fh0 != 0) {
        bad = lookback(p, t, lane, prefix);
        if (lane == 0) {
          if (bad) st_relaxed(p.error, 1u);
          else if (!fin)
            __hip_atomic_store(p.status + t, pack(kFlagInc, prefix + agg), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
      }
      if (lane == 0) { s_prefix = prefix; s_bad = bad; }
    }
    __syncthreads();
    if (s_bad) return;
    if (kEarly && threadIdx.x == 0) claim = claim_next(p.counter);
    // the elements before the span's first head (at fh) belong to a segment that
    // began earlier and take its carry
    const uint32_t add = seen_before ? before : s_prefix + before;
    if (whole) {
      const uint32_t lim = fh > 4 * lane ? fh - 4 * lane : 0u;
#pragma unroll
      for (int q = 0; q < SEGS; ++q) {
#pragma unroll
        for (int k = 0; k < 4; ++k) x[q][k] += (uint32_t)(q * 256 + k) < lim ? add : 0u;
      }
      wave_store<SEGS>(p.out, base, lane, x);
    } else {
      run = hbase = 0;
#pragma unroll 1
      for (int q = 0; q < SEGS; ++q) {
        const uint32_t i = q * 256 + 4 * lane;
        u32x4 v = part_load(p.in, base, i, pa, pb);
        seg_scan_heads<INCLUSIVE>(v, head_bits(bits, q, lane), lane, run, hbase);
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] += i + k < fh ? add : 0u;
        part_store(p.out, base, i, pa, pb, v);
      }
    }
    __syncthreads();  // s_tile, s_wave and s_prefix are rewritten by the next tile
  }
}

// Each workgroup sums a contiguous share of the spans, its waves taking them in
// turn.  No workgroup waits for another, so the shares are dealt, not claimed.
// Spans of 2048 elements: 32 data registers per lane and 8 KiB of LDS per wave
// leave 5 workgroups on a CU, of which the default grid has 4 (128 KiB of loads in
// flight).
__global__ void __launch_bounds__(kWg) __attribute__((amdgpu_waves_per_eu(5))) k_reduce_batch(BatchArgs p) {
  constexpr uint32_t kSpan = span_of(kSegsReduce);
  __shared__ __align__(16) uint32_t s_pre[kWaves][kSpan];  // flat exclusive prefixes of a wave's span
  const uint32_t lane = lane_id(), wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint32_t *pre_w = s_pre[wv];
  const uint64_t a = p.nspans * blockIdx.x / gridDim.x, b = p.nspans * (blockIdx.x + 1) / gridDim.x;
  uint32_t cur = 0xFFFFFFFFu, acc = 0;  // segment that runs through the last spans, this lane's share of it
  auto flush = [&](uint32_t next) {
    if (cur != 0xFFFFFFFFu) {
      const uint32_t tot = wave_sum(acc);
      if (lane == 0 && tot) add_relaxed(p.out + cur, tot);
    }
    cur = next;
    acc = 0;
  };
  for (uint64_t sp = a + wv; sp < b; sp += kWaves) {
    const uint64_t base = p.base + sp * kSpan;
    const uint32_t h0 = p.span_seg[sp], h1 = p.span_seg[sp + 1];
    u32x4 x[kSegsReduce];
    if (base >= p.lo && base + kSpan <= p.hi) {
      wave_load<kSegsReduce>(p.in, base, lane, x);
    } else {
      const uint32_t pa = clip(p.lo, base, kSpan), pb = clip(p.hi, base, kSpan);
#pragma unroll
      for (int q = 0; q < kSegsReduce; ++q) x[q] = part_load(p.in, base, q * 256 + 4 * lane, pa, pb);
    }
    if (h0 == h1) {  // the whole span lies in segment h0 - 1
      if (cur != h0 - 1) flush(h0 - 1);
#pragma unroll
      for (int q = 0; q < kSegsReduce; ++q) acc += x[q][0] + x[q][1] + x[q][2] + x[q][3];
      continue;
    }
    uint32_t run = 0;
#pragma unroll
    for (int q = 0; q < kSegsReduce; ++q) {
      const uint32_t v4 = x[q][0] + x[q][1] + x[q][2] + x[q][3];
      const uint32_t inc = wave_incl_scan(v4);
      u32x4 e;
      e.x = run + inc - v4;
      e.y = e.x + x[q][0];
      e.z = e.y + x[q][1];
      e.w = e.z + x[q][2];
      *reinterpret_cast<u32x4 *>(pre_w + q * 256 + 4 * lane) = e;
      run += __builtin_amdgcn_readlane(inc, 63);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    // segments that meet the span: h0 - 1 (its end) and the heads h0..h1-1
    for (uint64_t s0 = h0 ? h0 - 1 : 0; s0 < h1; s0 += 64) {
      const uint64_t s = s0 + lane;
      if (s < h1) {
        const uint64_t sb = p.offsets[s], se = p.offsets[s + 1];
        const uint32_t i = sb > base ? (uint32_t)(sb - base) : 0u;
        const uint32_t j = se < base + kSpan ? (uint32_t)(se - base) : kSpan;
        const uint32_t sum = i < j ? (j < kSpan ? pre_w[j] : run) - pre_w[i] : 0u;
        if (sb >= base && se <= base + kSpan) p.out[s] = sum;  // nobody else adds to it
        else if (sum) add_relaxed(p.out + s, sum);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // read before the next span's prefixes
  }
  flush(0xFFFFFFFFu);
}

// first segment of each span, and reset of the status words, the counter, the
// error word and (reduce) the sums.  One thread per span and a binary search:
// one thread that walked all segments instead took 74 us for 512 and 4.9 ms for
// 30011 of them, this takes 4-8 us.
__global__ void __launch_bounds__(kWg) k_batch_prep(const uint64_t *offsets, uint32_t nseg, uint64_t base,
                                                   uint32_t span, uint64_t nspans, uint32_t *span_seg,
                                                   uint64_t *status, uint64_t ntiles, uint32_t *counter,
                                                   uint32_t *error, uint32_t *sums) {
  const uint64_t t0 = blockIdx.x * (uint64_t)kWg + threadIdx.x, nt = (uint64_t)gridDim.x * kWg;
  if (t0 == 0) {
    *counter = 0;
    *error = 0;
  }
  for (uint64_t i = t0; i < ntiles; i += nt) status[i] = 0;
  if (sums)
    for (uint64_t s = t0; s < nseg; s += nt) sums[s] = 0;
  for (uint64_t i = t0; i <= nspans; i += nt) {
    const uint64_t at = base + i * span;
    uint32_t lo = 0, hi = nseg;  // segments below lo start before `at`, those from hi on do not
    while (lo < hi) {
      const uint32_t mid = lo + (hi - lo) / 2;
      if (offsets[mid] < at) lo = mid + 1;
      else hi = mid;
    }
    span_seg[i] = lo;
  }
}

// The grid of spans and tiles of a batch, the same for the work size and the
// launch.
struct Shape {
  bool ok, large;
  uint64_t lo, hi, base;
  uint64_t scan_tiles, scan_spans, reduce_spans;
};

Shape batch_shape(const uint64_t *h_offsets, uint32_t nseg) {
  Shape sh{};
  uint64_t bad = 0;
  for (uint32_t i = 0; i < nseg; ++i) bad |= (uint64_t)(h_offsets[i + 1] < h_offsets[i]);
  sh.ok = !bad;
  if (bad) return sh;
  sh.lo = h_offsets[0];
  sh.hi = h_offsets[nseg];
  sh.base = sh.lo & ~3ull;
  const uint64_t len = sh.hi > sh.lo ? sh.hi - sh.base : 0;
  sh.large = len >= kLargeFrom;
  const uint64_t tile = sh.large ? tile_of<Large>() : tile_of<Small>();
  sh.scan_tiles = (len + tile - 1) / tile;
  sh.scan_spans = sh.scan_tiles * (sh.large ? Large::kWg : Small::kWg) / 64;
  sh.reduce_spans = (len + span_of(kSegsReduce) - 1) / span_of(kSegsReduce);
  return sh;
}

size_t align256(size_t b) { return (b + 255) / 256 * 256; }

// Work layout: counter (0), error (128), span_seg (256), status words.
uint64_t span_seg_bytes(const Shape &sh) {
  const uint64_t s = sh.scan_spans > sh.reduce_spans ? sh.scan_spans : sh.reduce_spans;
  return align256(sizeof(uint32_t) * (s + 1));
}

// The size covers the most tiles that this many segments and elements could be
// cut into if every segment had 32768-element tiles of its own, twice over (16
// spans of 4 bytes and an 8-byte word for each small tile), so it only grows
// with the segments and the elements.
uint64_t batch_bytes(const Shape &sh, uint32_t nseg) {
  const uint64_t cells = 2ull * nseg + 4 + (sh.hi - sh.lo + 3ull * nseg) / 32768;
  return 512 + 2 * (16 * sizeof(uint32_t) + sizeof(uint64_t)) * cells;
}
static_assert(tile_of<Small>() == 16384 && Small::kWg <= 1024, "batch_bytes counts these tiles, with 16 spans at most");

template <class T>
const void *scan_kernel(int inclusive) {
  return inclusive ? (const void *)k_scan_batch<T, true> : (const void *)k_scan_batch<T, false>;
}

int launch_batch(bool scan, const uint32_t *d_in, uint32_t *d_out, const uint64_t *d_offsets,
                 const uint64_t *h_offsets, uint32_t nseg, int inclusive, void *d_work, int num_wgs,
                 hipStream_t s) {
  if (!d_in || !d_out || !d_offsets || !h_offsets || !d_work || nseg == 0 || nseg > 65536) return HS_ERR_INVALID;
  const Shape sh = batch_shape(h_offsets, nseg);
  if (!sh.ok || sh.scan_tiles >= 0xFFFFFFFFull) return HS_ERR_INVALID;
  const void *k = !scan ? (const void *)k_reduce_batch
                        : sh.large ? scan_kernel<Large>(inclusive) : scan_kernel<Small>(inclusive);
  const int wg = !scan ? kWg : sh.large ? Large::kWg : Small::kWg;
  // a larger grid than the CUs' registers hold is refused (counted for 256
  // threads; no workgroup waits for one that has not started, so this only
  // bounds the claims)
  if (num_wgs <= 0) num_wgs = hs_host::default_grid(k, wg, 4);
  else if (num_wgs > (scan ? 2 : 3) * hs_host::device_cus()) return HS_ERR_RESIDENCY;
  BatchArgs p{};
  p.in = d_in; p.out = d_out; p.offsets = d_offsets; p.nseg = nseg;
  p.lo = sh.lo; p.hi = sh.hi; p.base = sh.base;
  p.ntiles = scan ? sh.scan_tiles : 0;
  p.nspans = scan ? sh.scan_spans : sh.reduce_spans;
  char *w = (char *)d_work;
  p.counter = (uint32_t *)w;
  p.error = (uint32_t *)(w + 128);
  uint32_t *span_seg = (uint32_t *)(w + 256);
  p.span_seg = span_seg;
  p.status = (uint64_t *)(w + 256 + span_seg_bytes(sh));
  const uint32_t span = (uint32_t)span_of(!scan ? kSegsReduce : sh.large ? Large::kSegs : Small::kSegs);
  uint64_t items = p.nspans + 1;
  if (!scan && nseg > items) items = nseg;
  const uint64_t blocks = (items + kWg - 1) / kWg;
  hipLaunchKernelGGL(k_batch_prep, dim3((uint32_t)(blocks < 1024 ? blocks : 1024)), dim3(kWg), 0, s, d_offsets, nseg,
                     sh.base, span, p.nspans, span_seg, p.status, p.ntiles, p.counter, p.error,
                     scan ? nullptr : d_out);
  HS_TRY_HIP(hipGetLastError());
  if (p.nspans == 0) return HS_OK;
  // no more workgroups than tiles (each would claim one for nothing) or than
  // the spans give every wave one
  const uint64_t most = scan ? p.ntiles : (p.nspans + kWaves - 1) / kWaves;
  if ((uint64_t)num_wgs > most) num_wgs = (int)most;
  void *args[] = {(void *)&p};
  HS_TRY_HIP(hipLaunchKernel(k, dim3(num_wgs), dim3(wg), args, 0, s));
  return HS_OK;
}

}  // namespace

extern "C" {

int hs_batch_work_size(const uint64_t *h_offsets, uint32_t nseg, uint64_t *bytes_out) {
  if (!h_offsets || !bytes_out || nseg == 0 || nseg > 65536) return HS_ERR_INVALID;
  const Shape sh = batch_shape(h_offsets, nseg);
  if (!sh.ok) return HS_ERR_INVALID;
  *bytes_out = batch_bytes(sh, nseg);
  return HS_OK;
}

// status of the last batched launch that used d_work: HS_OK or HS_ERR_TIMEOUT
int hs_batch_status(const void *d_work, void *stream) {
  if (!d_work) return HS_ERR_INVALID;
  uint32_t err = 0;
  HS_TRY_HIP(hipMemcpyAsync(&err, (const char *)d_work + 128, sizeof(err), hipMemcpyDeviceToHost,
                            (hipStream_t)stream));
  HS_TRY_HIP(hipStreamSynchronize((hipStream_t)stream));
  return err ? HS_ERR_TIMEOUT : HS_OK;
}

int hs_scan_batch_u32(const uint32_t *d_in, uint32_t *d_out, const uint64_t *d_offsets, const uint64_t *h_offsets,
                      uint32_t nseg, int inclusive, void *d_work, int num_wgs, void *stream) {
  if (((uintptr_t)d_in & 15u) || ((uintptr_t)d_out & 15u)) return HS_ERR_INVALID;
  return launch_batch(true, d_in, d_out, d_offsets, h_offsets, nseg, inclusive, d_work, num_wgs,
                      (hipStream_t)stream);
}

int hs_reduce_batch_i32(const int32_t *d_in, int32_t *d_sums, const uint64_t *d_offsets, const uint64_t *h_offsets,
                        uint32_t nseg, void *d_work, int num_wgs, void *stream) {
  if ((uintptr_t)d_in & 15u) return HS_ERR_INVALID;
  return launch_batch(false, (const uint32_t *)d_in, (uint32_t *)d_sums, d_offsets, h_offsets, nseg, 0, d_work,
                      num_wgs, (hipStream_t)stream);
}

}  // extern "C"
