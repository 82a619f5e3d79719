// graph.hip -- persistent graph kernels on CSR uint32: single-source BFS,
// 64-source bit-parallel BFS with a push/pull schedule, near/far SSSP and
// deterministic pull PageRank.  One co-resident grid, grid barriers between
// phases (any hs_barrier_kind).
//
// Reference: LONESTAR/apps/{bfs,sssp,pr}/kernel_gsrb.cu (one persistent kernel
// per app, a barrier per round), LONESTAR/rt/include/worklist.h (frontier
// queues with warp-aggregated pushes) and LONESTAR/rt/include/internal.h (NP
// expansion: TB / warp / fine-grained).  Here the expansion is wave64-native:
// each wave takes up to 64 frontier vertices, scans their degrees with DPP and
// hands the concatenated edge list out 64 edges at a time (fine grained, the
// owner found by a 6-step shuffle search); vertices of degree >= 256 are
// split into fixed chunks that every wave of the grid shares.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "hs_graph.h"
#include "hs_internal.hpp"
#include "hs_wave.hpp"
#include "hs_worklist.hpp"
#include "team_rounds.hpp"

using namespace hs;

namespace hs_host {
int prepare_barrier(hs_arena *ar, int kind, hipStream_t s);
int launch_persistent(const void *k, void **args, int kind, int num_wgs, int wg_size, size_t lds,
                      hipStream_t s);
}  // namespace hs_host

namespace {

constexpr int kWg = 256;
constexpr int32_t kInf = 0x7FFFFFFF;
constexpr uint32_t kHeavy = 256;     // degree at which a vertex leaves the fine-grained path
constexpr int kCtr = 64;             // words between counters
__device__ __forceinline__ uint32_t gtid() { return blockIdx.x * kWg + threadIdx.x; }
__device__ __forceinline__ uint32_t gthreads() { return gridDim.x * kWg; }
__device__ __forceinline__ uint32_t gwave() { return blockIdx.x * (kWg / 64) + (threadIdx.x >> 6); }
__device__ __forceinline__ uint32_t gwaves() { return gridDim.x * (kWg / 64); }

__device__ __forceinline__ int32_t ld_i32(const int32_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t ld_u64(const uint64_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// a word that every lane reads alike, in a scalar register
__device__ __forceinline__ uint32_t ld_uniform(const uint32_t *p) { return __builtin_amdgcn_readfirstlane(ld_relaxed(p)); }
__device__ __forceinline__ uint64_t shfl64(uint64_t v, uint32_t lane) {
  const uint32_t lo = __shfl((uint32_t)v, (int)lane), hi = __shfl((uint32_t)(v >> 32), (int)lane);
  return ((uint64_t)hi << 32) | lo;
}

// ===========================================================================
// single-source BFS with load balancing (LONESTAR/apps/bfs/kernel_gsrb.cu:400-626)
// Level-synchronous push.  A vertex reached at level L goes to one of the
// inputs of level L: the light queue (out-degree < kHeavy), expanded 256
// vertices per workgroup grab with the wave64 fine-grained scheme, or, when
// heavy, as chunks of kBfsChunk out-edges to the chunk list that every wave of
// the grid shares (so one hub does not serialize a level on one workgroup).
constexpr uint32_t kBfsChunk = 1024;
constexpr int kBfsCounters = 15;

struct BfsArgs {
  uint32_t n;
  const uint32_t *row, *col;
  int32_t src;
  int32_t *level;
  uint32_t *q;    // [2][n] light frontier queues
  uint64_t *hq;   // [2][hcap] heavy chunk entries v | chunk << 32
  uint64_t *lq;   // [2][hcap] load-balanced mode: balanced entries v | first edge of v
                  // in the level's balanced edge space << 32
  uint64_t hcap;
  uint32_t *ctr;  // light counts [3], steal counters [3], chunk counts [3], balanced
                  // counts [3] (u64: entries << 32 | edges), kCtr words apart
  uint32_t *stats;
  uint32_t lb_limit;  // load-balanced mode: out-degree from which a vertex is heavy
  uint32_t ng, nx;
};

__device__ __forceinline__ uint32_t *cnt_at(uint32_t *c, uint32_t i) { return c + i * kCtr; }
__device__ __forceinline__ uint32_t *steal_at(uint32_t *c, uint32_t i) { return c + (3 + i) * kCtr; }
__device__ __forceinline__ uint32_t *hcnt_at(uint32_t *c, uint32_t i) { return c + (6 + i) * kCtr; }
__device__ __forceinline__ uint64_t *lbcnt_at(uint32_t *c, uint32_t i) {
  return reinterpret_cast<uint64_t *>(c + (9 + i) * kCtr);
}

__device__ __forceinline__ uint32_t bfs_chunks(uint32_t d) {
  return d >= kHeavy ? (d + kBfsChunk - 1) / kBfsChunk : 0u;
}

constexpr int kBfsBatch = 8;

// Load-balanced mode (the -l path of the reference: the inspector that moves
// vertices of out-degree >= DEGREE_LIMIT to a work list with their degrees, the
// prefix sum over those degrees and the kernel that gives every thread an equal
// share of their edges, LONESTAR/apps/bfs/kernel_gsrb.cu:343-398,569-579,
// LONESTAR/rt/include/thread_work.h:9-79).  Here the prefix sum is taken as the
// balanced vertices are discovered: one 64-bit fetch-and-add per wave on the
// counter (entries << 32 | their out-edges) returns both the wave's first list
// slot and its first edge, so the list is ordered by first edge; the next level
// splits the edges [0, total) evenly over every wave of the grid.  Vertices
// below the limit take the paths of the plain mode (chunk list from kHeavy,
// fine-grained below), as the reference's take its NP expansion.
__device__ __forceinline__ void bfs_visit_batch_lb(const BfsArgs &p, const uint32_t (&v)[kBfsBatch], int32_t L,
                                                   uint32_t *qout, uint32_t *cout, uint64_t *hout,
                                                   uint32_t *hcout, uint64_t *lout, uint64_t *lcout) {
  bool won[kBfsBatch];
#pragma unroll
  for (int x = 0; x < kBfsBatch; ++x) {
    won[x] = false;
    if (v[x] != 0xFFFFFFFFu && ld_i32(p.level + v[x]) == kInf) {
      int32_t expected = kInf;
      won[x] = __hip_atomic_compare_exchange_strong(p.level + v[x], &expected, L, __ATOMIC_RELAXED,
                                                    __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  uint32_t d[kBfsBatch], nc[kBfsBatch];
  bool light[kBfsBatch];
  uint32_t hc = 0, hd = 0;
#pragma unroll
  for (int x = 0; x < kBfsBatch; ++x) {
    d[x] = won[x] ? p.row[v[x] + 1] - p.row[v[x]] : 0u;
    const bool bal = won[x] && d[x] >= p.lb_limit;
    nc[x] = won[x] && !bal ? bfs_chunks(d[x]) : 0u;
    light[x] = won[x] && !bal && nc[x] == 0;
    if (!bal) d[x] = 0;
    hc += bal ? 1u : 0u;
    hd += d[x];
  }
  wave_push_batch<kBfsBatch>(qout, cout, light, v);
  wave_push_chunks_batch<kBfsBatch>(hout, hcout, nc, v);
  const uint32_t ic = wave_incl_scan(hc), id = wave_incl_scan(hd);
  const uint32_t tc = __builtin_amdgcn_readlane(ic, 63), td = __builtin_amdgcn_readlane(id, 63);
  if (tc == 0) return;
  uint64_t base = 0;
  if (lane_id() == 63)
    base = __hip_atomic_fetch_add(lcout, ((uint64_t)tc << 32) | td, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const uint32_t b_lo = __builtin_amdgcn_readlane((uint32_t)base, 63);
  const uint32_t b_hi = __builtin_amdgcn_readlane((uint32_t)(base >> 32), 63);
  uint32_t slot = b_hi + ic - hc, eb = b_lo + id - hd;
#pragma unroll
  for (int x = 0; x < kBfsBatch; ++x) {
    if (d[x]) {
      lout[slot++] = v[x] | ((uint64_t)eb << 32);
      eb += d[x];
    }
  }
}

// the entry of the balanced list whose edge range holds edge q: the last entry
// whose first edge is <= q (entries ordered by first edge, the first at 0)
__device__ __forceinline__ uint32_t bfs_lb_owner(const uint64_t *lin, uint32_t nl, uint32_t q) {
  uint32_t lo = 0, hi = nl;  // first(lo) <= q < first(hi)
  while (hi - lo > 1) {
    const uint32_t mid = lo + (hi - lo) / 2;
    if ((uint32_t)(lin[mid] >> 32) <= q) lo = mid; else hi = mid;
  }
  return lo;
}

template <int KIND>
__global__ void __launch_bounds__(kWg) __attribute__((amdgpu_waves_per_eu(8))) k_bfs_lb(ArenaView a, BfsArgs p) {
  GridBarrier gb;
  gb.init(a, KIND, p.ng, p.nx);
  for (uint32_t v = gtid(); v < p.n; v += gthreads()) p.level[v] = (v == (uint32_t)p.src) ? 0 : kInf;
  if (gtid() == 0) {
    for (int i = 0; i < 3; ++i) {
      *cnt_at(p.ctr, i) = 0;
      *steal_at(p.ctr, i) = 0;
      *hcnt_at(p.ctr, i) = 0;
      *lbcnt_at(p.ctr, i) = 0;
    }
    const uint32_t d = p.row[p.src + 1] - p.row[p.src];
    const uint32_t nc = bfs_chunks(d);
    if (d >= p.lb_limit) {
      p.lq[0] = (uint32_t)p.src;
      *lbcnt_at(p.ctr, 0) = (1ull << 32) | d;
    } else if (nc) {
      for (uint32_t c = 0; c < nc; ++c) p.hq[c] = (uint32_t)p.src | ((uint64_t)c << 32);
      *hcnt_at(p.ctr, 0) = nc;
    } else {
      p.q[0] = (uint32_t)p.src;
      *cnt_at(p.ctr, 0) = 1;
    }
  }
  if (gb.sync<KIND>()) return;
  uint32_t k = 0;
  for (;; ++k) {
    const Frontier fr{p.q, p.ctr, p.ctr + 3 * kCtr, p.n, (uint32_t)kCtr};
    const uint32_t nin = fr.in_count(k);
    const uint32_t nh = ld_relaxed(hcnt_at(p.ctr, k % 3));
    const uint64_t lc = __hip_atomic_load(lbcnt_at(p.ctr, k % 3), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t nl = (uint32_t)(lc >> 32), el = (uint32_t)lc;  // balanced entries and their edges
    if (nin == 0 && nh == 0 && nl == 0) break;
    const uint32_t *qin = fr.in(k);
    uint32_t *qout = fr.out(k);
    const uint64_t *hin = p.hq + (size_t)(k & 1) * p.hcap;
    uint64_t *hout = p.hq + (size_t)((k + 1) & 1) * p.hcap;
    const uint64_t *lin = p.lq + (size_t)(k & 1) * p.hcap;
    uint64_t *lout = p.lq + (size_t)((k + 1) & 1) * p.hcap;
    uint32_t *cout = fr.out_count(k);
    uint32_t *hcout = hcnt_at(p.ctr, (k + 1) % 3);
    uint64_t *lcout = lbcnt_at(p.ctr, (k + 1) % 3);
    if (gtid() == 0) {  // counters last used two levels ago
      fr.clear_for_next(k);
      st_relaxed(hcnt_at(p.ctr, (k + 2) % 3), 0u);
      __hip_atomic_store(lbcnt_at(p.ctr, (k + 2) % 3), 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const int32_t L = (int32_t)k + 1;
    {
      // the balanced vertices' edges [0, el), an equal share per wave of the
      // grid; a lane's owner entry only moves forward as its edge does (an
      // entry holds >= kHeavy edges, a step of a lane 64 apart)
      const uint32_t W = gwaves(), w = gwave();
      const uint32_t q_lo = (uint32_t)((uint64_t)el * w / W), q_hi = (uint32_t)((uint64_t)el * (w + 1) / W);
      if (q_lo < q_hi) {
        uint32_t j = bfs_lb_owner(lin, nl, q_lo);
        uint64_t ent = lin[j];
        uint32_t rb = p.row[(uint32_t)ent];
        uint32_t next = j + 1 < nl ? (uint32_t)(lin[j + 1] >> 32) : 0xFFFFFFFFu;  // first edge of j + 1
        for (uint32_t q0 = q_lo; q0 < q_hi; q0 += kBfsBatch * 64) {
          uint32_t vb[kBfsBatch];
#pragma unroll
          for (int x = 0; x < kBfsBatch; ++x) {
            const uint32_t q = q0 + 64 * x + lane_id();
            vb[x] = 0xFFFFFFFFu;
            if (q < q_hi) {
              while (next <= q) {
                ++j;
                ent = lin[j];
                rb = p.row[(uint32_t)ent];
                next = j + 1 < nl ? (uint32_t)(lin[j + 1] >> 32) : 0xFFFFFFFFu;
              }
              vb[x] = p.col[rb + (q - (uint32_t)(ent >> 32))];
            }
          }
          bfs_visit_batch_lb(p, vb, L, qout, cout, hout, hcout, lout, lcout);
        }
      }
    }
    // heavy chunks, spread over every wave of the grid
    for (uint32_t i = gwave(); i < nh; i += gwaves()) {
      const uint64_t ent = hin[i];
      const uint32_t u = (uint32_t)ent, c = (uint32_t)(ent >> 32);
      const uint32_t eb = p.row[u] + c * kBfsChunk, ee = min(p.row[u + 1], eb + kBfsChunk);
      for (uint32_t e0 = eb; e0 < ee; e0 += kBfsBatch * 64) {
        uint32_t vb[kBfsBatch];
#pragma unroll
        for (int x = 0; x < kBfsBatch; ++x) {
          const uint32_t e = e0 + 64 * x + lane_id();
          vb[x] = e < ee ? p.col[e] : 0xFFFFFFFFu;
        }
        bfs_visit_batch_lb(p, vb, L, qout, cout, hout, hcout, lout, lcout);
      }
    }
    // light queue: 256 vertices per workgroup grab, wave64 fine-grained expansion
    __shared__ uint32_t s_base;
    for (;;) {
      if (threadIdx.x == 0) s_base = fr.grab(k, (uint32_t)kWg);
      __syncthreads();
      const uint32_t base = s_base;
      __syncthreads();
      if (base >= nin) break;
      const uint32_t i = base + threadIdx.x;
      const bool valid = i < nin;
      const uint32_t u = valid ? qin[i] : 0u;
      uint32_t b = 0, deg = 0;
      if (valid) { b = p.row[u]; deg = p.row[u + 1] - b; }
      wave_expand<kBfsBatch>(b, deg, [&](const uint32_t (&e)[kBfsBatch], const bool (&ev)[kBfsBatch],
                                         const uint32_t (&)[kBfsBatch]) {
        uint32_t vb[kBfsBatch];
#pragma unroll
        for (int x = 0; x < kBfsBatch; ++x) vb[x] = ev[x] ? p.col[e[x]] : 0xFFFFFFFFu;
        bfs_visit_batch_lb(p, vb, L, qout, cout, hout, hcout, lout, lcout);
      });
    }
    if (gb.sync<KIND>()) return;
  }
  if (gtid() == 0 && p.stats) p.stats[0] = k;
}

// ===========================================================================
// multi-source BFS: bit s of fr[v] / vis[v] / nx[v] belongs to source s
struct MsArgs {
  uint32_t n;
  uint64_t m;
  const uint32_t *row, *col, *rrow, *rcol;
  const int32_t *srcs;
  int nsrc;
  int32_t *levels;          // [nsrc][n]
  uint64_t *fb[2];          // [n] each: level L's frontier is fb[L & 1], its next frontier fb[(L + 1) & 1]
  uint64_t *vis;            // [n]
  uint64_t *fbm[2];         // [ceil(n / 64)] each: bit v & 63 of word v >> 6 of fbm[L & 1] is
                            // "v is in level L's frontier"
  uint64_t *hlist;          // [2 lists][2 parities][hcap] entries v | chunk << 32
  uint32_t *hcnt;           // [2 lists][2 parities] counters, kCtr apart
  uint64_t hcap;
  uint64_t *part;           // [2][W][4] per-WG stats
  uint64_t *planes;         // [kMsPlanes][n]: bit s of plane k = bit k of (level + 1) of (s, v)
  int schedule;
  const float *mlp;
  const uint8_t *forced;    // [HS_MSBFS_MAX_LEVELS] (device)
  uint32_t *trace;
  uint32_t ng, nxcd;
};

// Discovery levels are kept as bit-planes while the BFS runs: a vertex reached
// by source s at level L < 255 sets bit s of planes[k][v] for every bit k of
// L + 1 (a read-modify-write of 8-byte words by the vertex's owner thread,
// coalesced), and one final pass decodes them and writes levels[s][v] once per
// pair, a full row of 64 vertices per store instruction.  Writing levels[s][v]
// at discovery instead hits every cache line of the 64 x n array at several
// levels with partial writes.  Levels >= 255 (deep graphs) are written directly.
// Plane k > 0 is written whole by the update pass of the first level with bit k
// (L + 1 = 2^k) and the decode reads only the planes written: a BFS of 8 levels
// clears and reads 4 of the 8.
constexpr int kMsPlanes = 8;
// edges per chunk of a heavy vertex in the MS-BFS lists: at R-MAT scale 22 the
// push from the level-2 hubs takes 127 us with 2048, 153 us with 4096
constexpr uint32_t kMsChunk = 2048;

struct MsStats {
  uint64_t nf, mf, mu, disc;
};

constexpr int kPush = 0, kPull = 1;
constexpr int kMlpIn = 8, kMlpH = 64, kMlpOut = 8;
constexpr int kMlpParams = kMlpH * kMlpIn + kMlpH + 2 * (kMlpH * kMlpH + kMlpH) + kMlpOut * kMlpH + kMlpOut;
// A level's action: bit 0 direction (push / pull), bit 1 expansion on half of
// the workgroups (the others go straight to the barrier), bit 2 long poll
// backoff in the barrier that ends the expansion.
constexpr uint32_t kActHalf = 2, kActLongBackoff = 4;
constexpr uint32_t kLongBackoff = 32;  // s_sleep units of a long-backoff level's polls

__device__ __forceinline__ uint64_t *hl_at(const MsArgs &p, int list, uint32_t parity) {
  return p.hlist + (size_t)(list * 2 + parity) * p.hcap;
}
// The frontier and the next frontier swap buffers every level: the update pass
// after level L leaves the new frontier where the expansion wrote it and clears
// only the words of the old frontier (found from its bitmap), instead of
// copying every word and clearing the other buffer.
__device__ __forceinline__ uint64_t *fr_at(const MsArgs &p, uint32_t L) { return p.fb[L & 1u]; }
__device__ __forceinline__ uint64_t *nx_at(const MsArgs &p, uint32_t L) { return p.fb[(L + 1u) & 1u]; }
__device__ __forceinline__ uint64_t *fbm_at(const MsArgs &p, uint32_t L) { return p.fbm[L & 1u]; }

__device__ __forceinline__ uint32_t *hc_at(const MsArgs &p, int list, uint32_t parity) {
  return p.hcnt + (list * 2 + parity) * kCtr;
}
// the pull's work is claimed from kMsGroups counters per level parity (after the
// four list counters)
constexpr uint32_t kMsGroups = 64;
constexpr uint32_t kMsCounters = 4 + 2 * kMsGroups;
__device__ __forceinline__ uint32_t *claim_at(const MsArgs &p, uint32_t parity, uint32_t g) {
  return p.hcnt + (4 + parity * kMsGroups + g) * kCtr;
}

// features of a level (all schedule-invariant; hsync.sched.features computes the
// same): frontier vertices, frontier out-edges, unvisited vertices' in-edges and
// the previous level's discoveries relative to the graph, its mean degree, the
// level, the out/in edge balance, and the graph size (costs change when the
// graph stops fitting the caches)
__device__ __forceinline__ float lg1(float x) { return log2f(1.f + x); }
__device__ __forceinline__ void ms_features(const MsStats &s, uint32_t n, uint64_t m, uint32_t L,
                                            float *f) {
  const float ln = lg1((float)n), lm = lg1((float)m);
  f[0] = (lg1((float)s.nf) - ln) / 32.f;
  f[1] = (lg1((float)s.mf) - lm) / 32.f;
  f[2] = (lg1((float)s.mu) - lm) / 32.f;
  f[3] = (lg1((float)s.disc) - ln) / 32.f;
  f[4] = (lm - ln) / 8.f;
  f[5] = (float)L / 32.f;
  f[6] = (lg1((float)s.mf) - lg1((float)s.mu)) / 8.f;
  f[7] = ln / 32.f;
}

// 8 -> 64 -> 64 -> 64 -> 8 MLP, ReLU; wave 0 of the workgroup evaluates it with
// one hidden unit per lane.  Layout: W1[64][8] b1[64] W2[64][64] b2[64]
// W3[64][64] b3[64] W4[8][64] b4[8], then one more float: the judge margin.
// The plain schedule judges: the network's best action replaces the plain
// action `plain` only when its logit leads the plain action's by at least the
// margin of the graph's size band (a margin of +inf keeps the plain schedule).
// Returns the action.
__device__ int mlp_decide(const float *w, const float *x, int plain) {
  const uint32_t j = lane_id();
  const float *W1 = w, *b1 = W1 + kMlpH * kMlpIn, *W2 = b1 + kMlpH, *b2 = W2 + kMlpH * kMlpH,
              *W3 = b2 + kMlpH, *b3 = W3 + kMlpH * kMlpH, *W4 = b3 + kMlpH, *b4 = W4 + kMlpOut * kMlpH;
  // the judge's margin for this graph's size band: w[P] up to log2(n + 1) =
  // w[P + 2] (feature 7 is log2(n + 1) / 32), w[P + 1] above it
  const float margin = x[7] * 32.f <= w[kMlpParams + 2] ? w[kMlpParams] : w[kMlpParams + 1];
  // no lead reaches +inf: the plain schedule, without evaluating the network
  // (every workgroup evaluates it per level, 37 KiB of weights each)
  if (__builtin_isinf(margin) && margin > 0.f) return plain;
  float h = b1[j];
#pragma unroll
  for (int i = 0; i < kMlpIn; ++i) h = fmaf(W1[j * kMlpIn + i], x[i], h);
  h = fmaxf(h, 0.f);
  float h2 = b2[j];
  for (int k = 0; k < kMlpH; ++k) h2 = fmaf(W2[j * kMlpH + k], __shfl(h, k), h2);
  h2 = fmaxf(h2, 0.f);
  float h3 = b3[j];
  for (int k = 0; k < kMlpH; ++k) h3 = fmaf(W3[j * kMlpH + k], __shfl(h2, k), h3);
  h3 = fmaxf(h3, 0.f);
  int best = 0;
  float ob = 0.f, op = 0.f;
  for (int q = 0; q < kMlpOut; ++q) {
    float o = W4[q * kMlpH + j] * h3;
    for (int k = 32; k >= 1; k >>= 1) o += __shfl_xor(o, k);  // fixed butterfly order: identical in every wave
    o += b4[q];
    if (q == 0 || o > ob) { ob = o; best = q; }
    if (q == plain) op = o;
  }
  return (ob - op >= margin) ? best : plain;
}

// the plain schedule: pull when the frontier's out-edges exceed half of the
// unvisited vertices' in-edges (the pull scans in-edges, the push out-edges)
__device__ __forceinline__ int heuristic_dir(const MsStats &s) { return s.mf * 2 > s.mu ? kPull : kPush; }

// Blocks of 64 vertices are visited in a scattered order: block j of a wave's
// share is scatter_block(j) (a bijection of [0, 2^k): xor-shifts and odd
// multiplies, so that neighbouring j land far apart; values >= nblk are
// skipped).  A plain stride of gwaves() blocks would hand every wave blocks with
// the same low index bits, and R-MAT degrees follow the bits of the vertex id.
__device__ __forceinline__ uint32_t scatter_block(uint32_t j, uint32_t k) {
  const uint32_t mask = k >= 32 ? 0xFFFFFFFFu : ((1u << k) - 1u);
  const uint32_t sh = (k + 1) / 2;
  uint32_t h = j;
  h ^= h >> sh;
  h = (h * 0x9E3779B1u) & mask;
  h ^= h >> sh;
  h = (h * 0x85EBCA6Bu) & mask;
  h ^= h >> sh;
  return h;
}

__device__ __forceinline__ uint32_t log2_ceil(uint32_t x) {
  uint32_t k = 0;
  while ((1ull << k) < x) ++k;
  return k;
}

// The chunk entries of an update pass's heavy vertices are staged in LDS and
// published with one counter atomic per list at the end of the pass; a wave
// takes the slots of all its lanes' entries with one atomic.  A counter atomic
// per heavy vertex serialises the workgroups that hold many of them: R-MAT
// hubs have ids with few set bits, so the workgroup of ids 0..255 mod the
// grid's stride holds ~10% of all heavy vertices (R-MAT scale 22, edge factor
// 16: 2380 of ~25k vertices of in-degree >= 256) and took twice the pass's
// median time.  Entries that do not fit into the stage go straight to the
// global list, again one atomic per wave.
constexpr uint32_t kMsStage = 512;  // staged entries per list and workgroup

struct MsStage {
  uint64_t ent[2][kMsStage];
  uint32_t cnt[2];   // slots handed out (may pass kMsStage)
  uint32_t fill[2];  // end of the filled prefix of ent
  uint32_t base[2];
};

// adds chunks 0..nc-1 of this lane's vertex v to list l (nc = 0: nothing);
// every lane of the wave calls it
__device__ __forceinline__ void ms_stage_add(MsStage &s, int l, uint32_t v, uint32_t nc, uint64_t *gl,
                                             uint32_t *gc, uint64_t cap) {
  if (!__ballot(nc != 0)) return;
  const uint32_t lane = lane_id();
  uint32_t inc = nc;  // inclusive prefix sum of nc over the wave
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = __shfl_up(inc, d);
    if (lane >= (uint32_t)d) inc += y;
  }
  const uint32_t total = __shfl(inc, 63), ex = inc - nc;
  uint32_t at = lane == 63 ? atomicAdd(&s.cnt[l], total) : 0u;
  at = __shfl(at, 63);
  if (at + total <= kMsStage) {
    // slots are handed out in order, so the ranges that fit form a prefix
    for (uint32_t c = 0; c < nc; ++c) s.ent[l][at + ex + c] = v | ((uint64_t)c << 32);
    if (lane == 63) atomicMax(&s.fill[l], at + total);
  } else {
    uint32_t g = lane == 63 ? add_relaxed(gc, total) : 0u;
    g = __shfl(g, 63);
    for (uint32_t c = 0; c < nc && (uint64_t)g + ex + c < cap; ++c) gl[g + ex + c] = v | ((uint64_t)c << 32);
  }
}

// publishes the staged entries (every thread of the workgroup calls it)
__device__ void ms_stage_flush(MsStage &s, uint64_t *gl0, uint64_t *gl1, uint32_t *gc0, uint32_t *gc1,
                               uint64_t cap) {
  __syncthreads();
  if (threadIdx.x < 2) {
    const uint32_t f = s.fill[threadIdx.x];
    s.base[threadIdx.x] = f ? add_relaxed(threadIdx.x ? gc1 : gc0, f) : 0u;
  }
  __syncthreads();
  for (int l = 0; l < 2; ++l) {
    uint64_t *gl = l ? gl1 : gl0;
    const uint32_t f = s.fill[l], b = s.base[l];
    for (uint32_t i = threadIdx.x; i < f; i += kWg)
      if ((uint64_t)b + i < cap) gl[b + i] = s.ent[l][i];
  }
  __syncthreads();
  if (threadIdx.x < 2) { s.cnt[threadIdx.x] = 0; s.fill[threadIdx.x] = 0; }
  __syncthreads();
}

// one pass over all vertices: fold next into frontier/visited (unless init),
// write discovery levels, accumulate the next level's statistics and its
// heavy-vertex chunk lists
__device__ void ms_update(const MsArgs &p, uint32_t L, bool init, uint64_t allmask) {
  MsStats st{0, 0, 0, 0};
  const uint32_t lp = (L + 1) & 1u;  // lists for level L + 1 are stored at parity (L + 1) & 1
  uint64_t *hpush = hl_at(p, 0, lp), *hpull = hl_at(p, 1, lp);
  uint32_t *cpush = hc_at(p, 0, lp), *cpull = hc_at(p, 1, lp);
  __shared__ MsStage stg;
  if (threadIdx.x < 2) { stg.cnt[threadIdx.x] = 0; stg.fill[threadIdx.x] = 0; }
  __syncthreads();
  // blocks of kWg vertices in the scattered order (the workgroup of a plain
  // stride would hold every block whose middle id bits are zero: the hubs)
  const uint32_t nblk = (p.n + kWg - 1) / kWg, kb = log2_ceil(nblk), nj = 1u << kb;
  // one vertex: vis, the old frontier's clearing, the new bitmap, the levels,
  // the statistics and the heavy lists (every thread of the workgroup calls it)
  auto vertex = [&](uint32_t v, uint64_t nxv, uint64_t visv, uint64_t old) {
    const bool valid = v < p.n;
    const uint32_t w0 = v & ~63u;  // this wave's first vertex
    if (!init && nxv) {
      visv |= nxv;
      p.vis[v] = visv;
    }
    if (!init && ((old >> lane_id()) & 1u)) fr_at(p, L)[v] = 0;  // level L's frontier becomes L + 1's next
    {  // frontier bitmap of level L + 1, one word per wave (64 consecutive vertices)
      const uint64_t fm = __ballot(nxv != 0);
      if (lane_id() == 0 && w0 < p.n) fbm_at(p, L + 1)[w0 >> 6] = fm;
    }
    if (!init && L + 1 < (1u << kMsPlanes)) {
      const uint32_t l1 = L + 1;
      if ((l1 & (l1 - 1u)) == 0) {
        // L + 1 = 2^k: the first level with bit k, and this pass visits every
        // vertex, so plane k is written here instead of cleared up front
        if (valid) p.planes[(size_t)__builtin_ctz(l1) * p.n + v] = nxv;
      } else if (nxv) {  // bit-planes of L + 1
        for (int k = 0; k < kMsPlanes; ++k)
          if (l1 >> k & 1) p.planes[(size_t)k * p.n + v] |= nxv;
      }
    } else if (!init) {
      // deep levels: one source at a time for the whole wave, so each store
      // instruction covers up to 64 consecutive vertices of one row
      uint64_t any = nxv;
      for (int k = 32; k >= 1; k >>= 1) any |= shfl64(any, lane_id() ^ k);
      while (any) {
        const int src = __builtin_ctzll(any);
        any &= any - 1;
        if (nxv >> src & 1) p.levels[(size_t)src * p.n + v] = (int32_t)L;
      }
    }
    const bool active = nxv != 0;
    const bool open = valid && visv != allmask;
    // degrees only where the statistics use them: out-degrees of the frontier,
    // in-degrees of the vertices still missing a source
    const uint32_t od = active ? p.row[v + 1] - p.row[v] : 0u;
    const uint32_t id = open ? p.rrow[v + 1] - p.rrow[v] : 0u;
    st.nf += active;
    st.mf += active ? od : 0u;
    st.mu += open ? id : 0u;
    st.disc += (uint64_t)__builtin_popcountll(nxv);
    ms_stage_add(stg, 0, v, active && od >= kHeavy ? (od + kMsChunk - 1) / kMsChunk : 0u, hpush, cpush, p.hcap);
    ms_stage_add(stg, 1, v, open && id >= kHeavy ? (id + kMsChunk - 1) / kMsChunk : 0u, hpull, cpull, p.hcap);
  };
  // two blocks per round, both blocks' loads before either's stores: the pass
  // is bound by the latency of these loads, not by their bytes
  for (uint32_t j = blockIdx.x; j < nj; j += 2 * gridDim.x) {
    uint32_t vv[2];
    uint64_t nx2[2], vis2[2], old2[2];
    bool use[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const uint32_t jj = j + u * gridDim.x;
      const uint32_t blk = jj < nj ? scatter_block(jj, kb) : nblk;
      use[u] = blk < nblk;  // the same for the whole workgroup
      vv[u] = blk * kWg + threadIdx.x;
      nx2[u] = vis2[u] = old2[u] = 0;
      if (use[u] && vv[u] < p.n) {
        nx2[u] = fr_at(p, L + 1)[vv[u]];  // level L + 1's frontier, in place (the expansions add only bits not in vis)
        vis2[u] = p.vis[vv[u]];
      }
      if (use[u] && !init && (vv[u] & ~63u) < p.n) old2[u] = fbm_at(p, L)[vv[u] >> 6];
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
      if (use[u]) vertex(vv[u], nx2[u], vis2[u], old2[u]);
  }
  ms_stage_flush(stg, hpush, hpull, cpush, cpull, p.hcap);
  // workgroup totals (fixed order) -> part[(L+1)&1][wg]
  __shared__ uint64_t red[4][kWg / 64];
  uint64_t vals[4] = {st.nf, st.mf, st.mu, st.disc};
  for (int q = 0; q < 4; ++q) {
    uint64_t x = vals[q];
    for (int k = 32; k >= 1; k >>= 1) x += shfl64(x, lane_id() ^ k);
    if (lane_id() == 0) red[q][threadIdx.x >> 6] = x;
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    uint64_t t = 0;
    for (int w = 0; w < kWg / 64; ++w) t += red[threadIdx.x][w];
    p.part[((size_t)lp * gridDim.x + blockIdx.x) * 4 + threadIdx.x] = t;
  }
  __syncthreads();
}

__device__ MsStats ms_totals(const MsArgs &p, uint32_t parity) {
  __shared__ uint64_t red[4][kWg / 64];
  uint64_t acc[4] = {0, 0, 0, 0};
  for (uint32_t w = threadIdx.x; w < gridDim.x; w += kWg)
    for (int q = 0; q < 4; ++q) acc[q] += p.part[((size_t)parity * gridDim.x + w) * 4 + q];
  for (int q = 0; q < 4; ++q) {
    uint64_t x = acc[q];
    for (int k = 32; k >= 1; k >>= 1) x += shfl64(x, lane_id() ^ k);
    if (lane_id() == 0) red[q][threadIdx.x >> 6] = x;
  }
  __syncthreads();
  MsStats s;
  uint64_t t[4];
  for (int q = 0; q < 4; ++q) {
    t[q] = 0;
    for (int w = 0; w < kWg / 64; ++w) t[q] += red[q][w];
  }
  __syncthreads();
  s.nf = t[0]; s.mf = t[1]; s.mu = t[2]; s.disc = t[3];
  return s;
}

constexpr int kMsBatch = 4;  // 64-edge steps in flight per wave

// push: out-edges of frontier vertices, atomicOr of the new bits into nx
__device__ void ms_push(const MsArgs &p, uint32_t L, uint32_t nact) {
  if (gwave() >= nact) return;  // this level expands on the first nact waves only
  const uint64_t *fr = fr_at(p, L);
  uint64_t *nx = nx_at(p, L);
  const uint32_t lane = lane_id();
  const uint32_t nblk = (p.n + 63) / 64, kb = log2_ceil(nblk);
  for (uint32_t j = gwave(); j < (1u << kb); j += nact) {
    const uint32_t blk = scatter_block(j, kb);
    if (blk >= nblk) continue;
    const uint32_t v = blk * 64 + lane;
    const uint64_t f = v < p.n ? fr[v] : 0ull;
    uint32_t b = 0, deg = 0;
    if (f) { b = p.row[v]; deg = p.row[v + 1] - b; }
    wave_expand<kMsBatch>(b, deg < kHeavy ? deg : 0u, [&](const uint32_t (&e)[kMsBatch],
                                                         const bool (&ev)[kMsBatch],
                                                         const uint32_t (&own)[kMsBatch]) {
      uint32_t dst[kMsBatch];
      uint64_t of[kMsBatch], vis[kMsBatch], nxv[kMsBatch];
#pragma unroll
      for (int x = 0; x < kMsBatch; ++x) {
        of[x] = shfl64(f, own[x]);
        dst[x] = ev[x] ? __builtin_nontemporal_load(p.col + e[x]) : 0u;
      }
#pragma unroll
      for (int x = 0; x < kMsBatch; ++x) vis[x] = ev[x] ? ld_u64(p.vis + dst[x]) : ~0ull;
#pragma unroll
      for (int x = 0; x < kMsBatch; ++x) nxv[x] = (of[x] & ~vis[x]) ? ld_u64(nx + dst[x]) : ~0ull;
#pragma unroll
      for (int x = 0; x < kMsBatch; ++x) {
        const uint64_t bits = of[x] & ~vis[x];
        if (bits && (nxv[x] & bits) != bits)
          __hip_atomic_fetch_or(nx + dst[x], bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    });
  }
  (void)lane;
  // heavy vertices: chunks of kChunk out-edges, shared round-robin by all waves
  const uint32_t cnt = ld_relaxed(hc_at(p, 0, L & 1u));
  const uint64_t *hl = hl_at(p, 0, L & 1u);
  for (uint32_t i = gwave(); i < cnt && i < p.hcap; i += nact) {
    const uint64_t ent = hl[i];
    const uint32_t v = (uint32_t)ent, c = (uint32_t)(ent >> 32);
    const uint64_t f = fr[v];
    const uint32_t eb = p.row[v] + c * kMsChunk;
    const uint32_t ee = min(p.row[v + 1], eb + kMsChunk);
    for (uint32_t e0 = eb + lane_id(); e0 < ee; e0 += kMsBatch * 64) {
      uint32_t dst[kMsBatch];
      uint64_t vis[kMsBatch];
#pragma unroll
      for (int x = 0; x < kMsBatch; ++x)
        dst[x] = e0 + 64 * x < ee ? __builtin_nontemporal_load(p.col + e0 + 64 * x) : 0xFFFFFFFFu;
#pragma unroll
      for (int x = 0; x < kMsBatch; ++x) vis[x] = dst[x] != 0xFFFFFFFFu ? ld_u64(p.vis + dst[x]) : ~0ull;
#pragma unroll
      for (int x = 0; x < kMsBatch; ++x) {
        const uint64_t bits = f & ~vis[x];
        if (bits && (ld_u64(nx + dst[x]) & bits) != bits)
          __hip_atomic_fetch_or(nx + dst[x], bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
}

__device__ __forceinline__ uint64_t lds_ld64(const uint64_t *a) {
  return __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}
__device__ __forceinline__ uint64_t wave_or64(uint64_t x) {
  for (int k = 32; k >= 1; k >>= 1) x |= shfl64(x, lane_id() ^ k);
  return x;
}
// frontier bits of in-neighbour u: the bitmap word (a few hundred KiB, kept
// in L2) first, fr[u] only for frontier vertices
__device__ __forceinline__ bool ms_in_frontier(uint64_t word, uint32_t u) {
  return (word >> (u & 63u)) & 1u;
}

// pull: in-edges of not-yet-complete vertices; light vertices accumulate in LDS
// and are stored by their owner (no atomics), heavy ones use atomicOr per chunk.
// In-neighbours are tested against the frontier bitmap before fr is read.
//
// Work is claimed, not dealt: the blocks of 64 vertices (scattered order) and
// then the heavy chunks form one sequence per group of workgroups, and each
// wave claims its next item from its group's counter while it works on the
// current one.  A fixed deal of the same blocks left the slowest wave at about
// twice the mean (R-MAT scale 22: in-edge counts per block are heavy-tailed).
// A light vertex's in-edges are read in two rounds.  The first step of the
// wave (kMsBatch x 64 positions) takes the first kMsFirst in-edges of every
// lane's vertex, then as many further edges as fit; the rest of the edges of
// the vertices still missing a source follow, packed again.  A vertex whose
// first edges found every source it was missing reads no more: at the level
// that reaches most of an R-MAT graph, ~80% of the light in-edges.  The number
// of steps stays that of one packed sequence when nothing is found early.
constexpr uint32_t kMsFirst = 4;
static_assert(kMsFirst <= (uint32_t)kMsBatch, "segment 1 must fit into the first step");

// Edge arrays are read with streaming loads (col in the push, rcol in the
// pull): each is read once per level, and cached they evict the vis, frontier
// and plane words that the update pass after the expansion reads again (R-MAT
// 22: the update passes after the big pulls 60 -> 51 us and 82 -> 62 us).
__device__ __forceinline__ void ms_pull_gather(const MsArgs &p, uint32_t L, const uint32_t (&e)[kMsBatch],
                                               const bool (&ev)[kMsBatch], const uint32_t (&own)[kMsBatch],
                                               uint64_t unv, uint64_t *acc) {
  const uint64_t *fr = fr_at(p, L), *fbm = fbm_at(p, L);
  uint32_t src[kMsBatch];
  uint64_t fm[kMsBatch], fb[kMsBatch];
#pragma unroll
  for (int x = 0; x < kMsBatch; ++x) src[x] = ev[x] ? __builtin_nontemporal_load(p.rcol + e[x]) : 0u;
#pragma unroll
  for (int x = 0; x < kMsBatch; ++x) fm[x] = ev[x] ? fbm[src[x] >> 6] : 0ull;
#pragma unroll
  for (int x = 0; x < kMsBatch; ++x) fb[x] = ms_in_frontier(fm[x], src[x]) ? ld_u64(fr + src[x]) : 0ull;
#pragma unroll
  for (int x = 0; x < kMsBatch; ++x) {
    const uint64_t bits = fb[x] & shfl64(unv, own[x]);
    if (bits) __hip_atomic_fetch_or(acc + own[x], bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
  }
}

__device__ __forceinline__ void ms_pull_light(const MsArgs &p, uint32_t L, uint64_t allmask, uint32_t blk,
                                              uint64_t *acc) {
  const uint32_t lane = lane_id();
  const uint32_t v = blk * 64 + lane;
  const uint64_t unv = v < p.n ? (~p.vis[v] & allmask) : 0ull;
  uint32_t b = 0, deg = 0;
  if (unv) { b = p.rrow[v]; deg = p.rrow[v + 1] - b; }
  const uint32_t ldeg = deg < kHeavy ? deg : 0u;
  // first round: segment 1 = the first kMsFirst edges of each lane, segment 2 =
  // the others, one sequence, its first kMsBatch x 64 positions
  const uint32_t d1 = ldeg < kMsFirst ? ldeg : kMsFirst, d2 = ldeg - d1;
  const uint32_t i1 = wave_incl_scan(d1), i2 = wave_incl_scan(d2);
  const uint32_t s1 = __builtin_amdgcn_readlane(i1, 63), s2 = __builtin_amdgcn_readlane(i2, 63);
  const uint32_t x1 = i1 - d1, x2 = i2 - d2;
  if (s1 + s2 == 0) return;
  {
    uint32_t e[kMsBatch], own[kMsBatch];
    bool ev[kMsBatch];
#pragma unroll
    for (int x = 0; x < kMsBatch; ++x) {
      if (64u * x >= s1 + s2) {  // past the last edge for the whole wave
        own[x] = 0; ev[x] = false; e[x] = 0;
        continue;
      }
      const uint32_t q = 64 * x + lane;
      const bool seg1 = q < s1;
      const uint32_t q2 = seg1 ? 0u : q - s1;
      const uint32_t o1 = wave_owner(i1, seg1 ? q : s1 - 1);  // s1 > 0 whenever any edge exists
      const uint32_t o2 = wave_owner(i2, q2 < s2 ? q2 : (s2 ? s2 - 1 : 0u));
      const uint32_t bo1 = __shfl(b, (int)o1), xo1 = __shfl(x1, (int)o1);
      const uint32_t bo2 = __shfl(b, (int)o2), xo2 = __shfl(x2, (int)o2);
      own[x] = seg1 ? o1 : o2;
      ev[x] = q < s1 + s2;
      e[x] = seg1 ? bo1 + (q - xo1) : bo2 + kMsFirst + (q2 - xo2);
    }
    ms_pull_gather(p, L, e, ev, own, unv, acc);
  }
  // second round: the segment-2 edges past the first round's positions, of the
  // vertices still missing a source
  const uint32_t used2 = kMsBatch * 64 - s1;  // segment-2 positions taken by the first round
  const uint32_t rest = i2 > used2 ? i2 - (x2 > used2 ? x2 : used2) : 0u;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the lanes' LDS ORs before the reads
  const bool done = (lds_ld64(acc + lane) & unv) == unv;
  const uint32_t r = done ? 0u : rest;
  wave_expand<kMsBatch>(b + kMsFirst + (d2 - rest), r, [&](const uint32_t (&e)[kMsBatch],
                                                           const bool (&ev)[kMsBatch],
                                                           const uint32_t (&own)[kMsBatch]) {
    ms_pull_gather(p, L, e, ev, own, unv, acc);
  });
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  if (ldeg) {
    const uint64_t got = lds_ld64(acc + lane);
    if (got) nx_at(p, L)[v] = got;
  }
  acc[lane] = 0;
}

__device__ __forceinline__ void ms_pull_heavy(const MsArgs &p, uint32_t L, uint64_t allmask, uint64_t ent) {
  const uint64_t *fr = fr_at(p, L), *fbm = fbm_at(p, L);
  const uint32_t lane = lane_id();
  const uint32_t v = (uint32_t)ent, c = (uint32_t)(ent >> 32);
  const uint64_t unv = ~p.vis[v] & allmask;
  const uint32_t eb = p.rrow[v] + c * kMsChunk;
  const uint32_t ee = min(p.rrow[v + 1], eb + kMsChunk);
  uint64_t a = 0;
  for (uint32_t e00 = eb; e00 < ee; e00 += 8 * 64) {
    uint32_t src[8];
    uint64_t fm[8];
#pragma unroll
    for (int x = 0; x < 8; ++x)
      src[x] = e00 + 64 * x + lane < ee ? __builtin_nontemporal_load(p.rcol + e00 + 64 * x + lane) : 0xFFFFFFFFu;
#pragma unroll
    for (int x = 0; x < 8; ++x) fm[x] = src[x] != 0xFFFFFFFFu ? fbm[src[x] >> 6] : 0ull;
#pragma unroll
    for (int x = 0; x < 8; ++x) a |= ms_in_frontier(fm[x], src[x]) ? ld_u64(fr + src[x]) : 0ull;
    if ((wave_or64(a) & unv) == unv) break;  // this chunk found every missing source
  }
  a = wave_or64(a) & unv;
  if (lane == 0 && a) __hip_atomic_fetch_or(nx_at(p, L) + v, a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ void ms_pull(const MsArgs &p, uint32_t L, uint64_t allmask, uint32_t nact) {
  if (gwave() >= nact) return;
  __shared__ uint64_t acc_s[kWg];
  const uint32_t lane = lane_id();
  uint64_t *acc = acc_s + (threadIdx.x & ~63u);
  acc[lane] = 0;
  const uint32_t nblk = (p.n + 63) / 64, kb = log2_ceil(nblk);
  // groups: workgroup w of the active ones claims from counter w mod G, and
  // every counter has at least one active workgroup
  const uint32_t nwg = (nact + kWg / 64 - 1) / (kWg / 64);
  const uint32_t G = nwg < kMsGroups ? nwg : kMsGroups, g = blockIdx.x % G;
  const uint32_t nj = 1u << kb;
  const uint32_t nlight = g < nj ? (nj - g + G - 1) / G : 0u;  // j = g + t G < 2^kb
  uint32_t cnt = ld_relaxed(hc_at(p, 1, L & 1u));
  cnt = cnt < p.hcap ? cnt : (uint32_t)p.hcap;
  const uint32_t nheavy = g < cnt ? (cnt - g + G - 1) / G : 0u;
  const uint64_t *hl = hl_at(p, 1, L & 1u);
  uint32_t *ctr = claim_at(p, L & 1u, g);
  uint32_t t = __shfl(lane == 0 ? add_relaxed(ctr, 1u) : 0u, 0);
  while (t < nlight + nheavy) {
    const uint32_t next = __shfl(lane == 0 ? add_relaxed(ctr, 1u) : 0u, 0);
    if (t < nlight) {
      const uint32_t blk = scatter_block(g + t * G, kb);
      if (blk < nblk) ms_pull_light(p, L, allmask, blk, acc);
    } else {
      ms_pull_heavy(p, L, allmask, hl[g + (t - nlight) * G]);
    }
    t = next;
  }
}

template <int KIND>
__global__ void __launch_bounds__(kWg) k_msbfs(ArenaView a, MsArgs p) {
  GridBarrier gb;
  gb.init(a, KIND, p.ng, p.nxcd);
  const uint64_t allmask = p.nsrc >= 64 ? ~0ull : ((1ull << p.nsrc) - 1ull);
  for (uint32_t v = gtid(); v < p.n; v += gthreads()) { p.fb[0][v] = 0; p.fb[1][v] = 0; p.vis[v] = 0; }
  for (uint32_t v = gtid(); v < p.n; v += gthreads()) p.planes[v] = 0;  // plane 0 (the others: ms_update)
  if (gtid() < kMsCounters) p.hcnt[gtid() * kCtr] = 0;
  if (gb.sync<KIND>()) return;
  if (blockIdx.x == 0 && threadIdx.x < (uint32_t)p.nsrc) {
    const uint32_t s = threadIdx.x, v = (uint32_t)p.srcs[s];
    __hip_atomic_fetch_or(fr_at(p, 1) + v, 1ull << s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_fetch_or(p.vis + v, 1ull << s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_fetch_or(p.planes + v, 1ull << s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // L + 1 = 1
  }
  if (gb.sync<KIND>()) return;
  ms_update(p, 0, true, allmask);  // statistics + heavy lists of level 1
  if (gb.sync<KIND>()) return;
  __shared__ int s_dir;
  for (uint32_t L = 1;; ++L) {
    const MsStats st = ms_totals(p, L & 1u);
    if (st.nf == 0) {
      // every update is done (a barrier followed the last one): decode the
      // planes, one row segment of 64 vertices per store; unreached -> INF,
      // reached at a deep level -> already written
      // planes in use: 0 and every k with 2^k <= L (the updates reached L + 1 <= L)
      const int kuse = (32 - __builtin_clz(L)) < kMsPlanes ? (32 - __builtin_clz(L)) : kMsPlanes;
      for (uint32_t v = gtid(); v < p.n; v += gthreads()) {
        uint64_t pl[kMsPlanes];
#pragma unroll
        for (int k = 0; k < kMsPlanes; ++k) pl[k] = k < kuse ? p.planes[(size_t)k * p.n + v] : 0ull;
        const uint64_t vis = p.vis[v];
        for (int src = 0; src < p.nsrc; ++src) {
          uint32_t code = 0;
#pragma unroll
          for (int k = 0; k < kMsPlanes; ++k) code |= (uint32_t)((pl[k] >> src) & 1u) << k;
          // streaming stores: nothing here reads the 4 B x 64 x n levels again,
          // and cached they leave dirty lines that the next launch's first
          // passes pay for (clear and first update 81 -> 64 us at R-MAT 22)
          if (code) __builtin_nontemporal_store((int32_t)code - 1, p.levels + (size_t)src * p.n + v);
          else if (!((vis >> src) & 1u)) __builtin_nontemporal_store((int32_t)kInf, p.levels + (size_t)src * p.n + v);
        }
      }
      break;
    }
    if (threadIdx.x < 64) {
      int act;
      switch (p.schedule) {
        case 1: act = kPush; break;
        case 2: act = kPull; break;
        case 3: {
          float f[kMlpIn];
          ms_features(st, p.n, p.m, L, f);
          act = mlp_decide(p.mlp, f, heuristic_dir(st));
          break;
        }
        case 4: act = L <= HS_MSBFS_MAX_LEVELS ? (int)(p.forced[L - 1] & 7u) : kPush; break;
        default: act = heuristic_dir(st);
      }
      if (threadIdx.x == 0) s_dir = act;
    }
    __syncthreads();
    const int act = s_dir;
    const int dir = act & 1;
    const uint32_t nact = (act & kActHalf) ? ((gridDim.x + 1) / 2) * (kWg / 64) : gwaves();
    uint32_t t0 = 0, t1 = 0;
    if (p.trace && blockIdx.x == 0 && threadIdx.x == 0 && L <= HS_MSBFS_MAX_LEVELS) {
      const uint64_t c = wall_clock64();
      t0 = (uint32_t)c; t1 = (uint32_t)(c >> 32);
    }
    // counters of the lists for level L+1 were read at level L-1: clear them
    if (gtid() < 2) st_relaxed(hc_at(p, (int)gtid(), (L + 1) & 1u), 0u);
    if (gtid() < kMsGroups) st_relaxed(claim_at(p, (L + 1) & 1u, gtid()), 0u);
    if (dir == kPush) ms_push(p, L, nact);
    else ms_pull(p, L, allmask, nact);
    gb.poll_sleep = (act & kActLongBackoff) ? kLongBackoff : 0u;
    const int brc = gb.sync<KIND>();
    gb.poll_sleep = 0;
    if (brc) return;
    if (p.trace && blockIdx.x == 0 && threadIdx.x == 0 && L <= HS_MSBFS_MAX_LEVELS) {
      const uint64_t c = wall_clock64();
      uint32_t *tr = p.trace + (size_t)(L - 1) * HS_MSBFS_TRACE_WORDS;
      tr[0] = (uint32_t)act; tr[1] = (uint32_t)st.nf;
      tr[2] = (uint32_t)st.mf; tr[3] = (uint32_t)(st.mf >> 32);
      tr[4] = (uint32_t)st.mu; tr[5] = (uint32_t)(st.mu >> 32);
      tr[6] = (uint32_t)st.disc;
      tr[7] = t0; tr[8] = t1; tr[9] = (uint32_t)c; tr[10] = (uint32_t)(c >> 32);
    }
    ms_update(p, L, false, allmask);
    if (gb.sync<KIND>()) return;
  }
}

// ===========================================================================
// Rounds by a team: high-diameter graphs (meshes, roads) run thousands of rounds
// of a few thousand vertices each, and such a round costs one grid barrier (5-7
// us, most of it words bouncing between the XCDs' L2s) and a chain of loads that
// miss an L2 the barrier's acquire has just emptied.  While the rounds are small
// they are run by the workgroups b with b % nxcd == 0 alone, which dispatch puts
// on one XCD: there an atomic or a coherent load of the device takes 0.12 us (a
// miss 0.5 us).  What bounds a round is that chain, so it is kept short:
//  - every workgroup appends to an output segment of its own, counted in LDS (an
//    atomic on one queue counter serializes for ~11 ns and is waited for), and a
//    segment entry carries the vertex's first edge, so its edges, key and end are
//    loaded together;
//  - the team's barrier is one word per workgroup, its episode and its segment's
//    count, which every workgroup reads with one load, so that the barrier also
//    says what the next round's input is;
//  - on meshes (degree <= 4) four lanes share a vertex: one edge per lane and a
//    single pass of short code.
// Correctness does not depend on the placement: everything the rounds write is
// written and read with agent-scope operations, and every wave's stores have
// completed before its workgroup arrives.  Nor on timing: the other workgroups wait
// in the grid barrier meanwhile (a stretch is at most 256 rounds, so that wait stays
// short), and what they read before it, to find out that this stretch is
// not theirs, is not written until it is over (team_rounds.hpp: the counters of the
// phase and the report of the stretch before; the team counts in others).
// Threads per workgroup of the kernels that run team rounds: with 128 registers and
// 33 KB of LDS at most, one workgroup is half of a CU, so that two searches on two
// streams, or one beside the serving loop (one workgroup of 248 registers per CU),
// are resident together.  1024 threads fill the CU, and each of two such launches may
// get part of the CUs and wait for the rest; they take R-MAT 22 in 334 us (BFS) and
// 2.87 ms (SSSP) against 357 us and 3.20 ms, a mesh of 1.1M vertices in 13.7 ms
// against 12.9 and 200k vertices in 164 us against 135.  64 registers, for four
// searches at once, spill: 392 us, 3.34 ms and 24.6 ms.
constexpr int kTeamWg = 512;
using hs_rounds::kTeamMax;                  // workgroups of a team
constexpr uint32_t kTeamIdleSleep = 32;     // s_sleep units between the idle workgroups' polls
constexpr uint32_t kSegCap = 2048;          // entries of a workgroup's output segment; the rest goes to the queue
constexpr uint32_t kSegBlock = 16;          // entries a wave takes at once: 4 lanes each

__device__ __forceinline__ void st_u64(uint64_t *p, uint64_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Who works on a round: wave `wave` of `waves`, the waves of a workgroup far apart
// so that a small round is spread over the compute units.
struct Crew {
  uint32_t wave, waves;
  __device__ Crew(uint32_t rank, uint32_t size) {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * size + rank;
    waves = size * (kTeamWg / 64);
  }
};

// The segments' share of a round's input: lane l holds segment l's entries and the
// blocks of segments 0..l; the same in every wave.
struct Segments {
  uint32_t cnt, upto, blocks, total;
  bool queued;  // some workgroup also appended to the queues

  __device__ void none() { cnt = upto = blocks = total = 0; queued = true; }
  // word: lane l's segment count, bit 31 = "appended to the queues"
  __device__ __forceinline__ void take(uint32_t word) {
    queued = ballot(word >> 31) != 0;
    cnt = word & 0x7FFFFFFFu;
    upto = wave_incl_scan((cnt + kSegBlock - 1) / kSegBlock);
    blocks = __builtin_amdgcn_readlane(upto, 63);
    total = wave_sum(cnt);
  }
  // entry index (of all segments, kSegCap apart) of this lane in block b, or ~0
  __device__ __forceinline__ uint32_t entry(uint32_t b) const {
    const uint32_t s = (uint32_t)__builtin_popcountll(ballot(upto <= b));
    const uint32_t n = __builtin_amdgcn_readlane(cnt, s);
    const uint32_t first = __builtin_amdgcn_readlane(upto, s) - (n + kSegBlock - 1) / kSegBlock;
    const uint32_t i = (b - first) * kSegBlock + (lane_id() >> 2);
    return i < n ? s * kSegCap + i : 0xFFFFFFFFu;
  }
};

// The counters of one round and of the next: of the grid, by phase, or of the team.
struct Round {
  uint32_t *ctr;
  hs_rounds::Side side;
  uint32_t i;
  __device__ __forceinline__ uint32_t *at(hs_rounds::Counter c, uint32_t ahead = 0) const {
    return ctr + hs_rounds::slot(side, c, i + ahead) * kCtr;
  }
  // one thread: clears what the rounds after this one use
  __device__ __forceinline__ void open() const {
    hs_rounds::open_round(side, i, [&](uint32_t s) { st_relaxed(ctr + s * kCtr, 0u); });
  }
};

// What a stretch leaves to the next phase: lane l's word l, of which the last 32 are
// the segments' counts.
struct Report {
  uint32_t w;
  __device__ __forceinline__ void write(uint32_t *ctr, uint32_t k, uint32_t seg_cnt, const uint32_t (&head)[8]) {
    const uint32_t lane = lane_id(), cnt = __shfl(seg_cnt, (int)(lane & 31));
    w = cnt;
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) w = lane == i ? head[i] : w;
    st_relaxed(ctr + hs_rounds::report(k) * kCtr + lane, w);
  }
  __device__ __forceinline__ void read(const uint32_t *ctr, uint32_t k) {
    w = ld_relaxed(ctr + hs_rounds::report(k) * kCtr + lane_id());
  }
  __device__ __forceinline__ uint32_t head(int i) const { return __builtin_amdgcn_readlane(w, i); }
  // (every lane takes part in the shuffle)
  __device__ __forceinline__ uint32_t segment() const {
    const uint32_t cnt = __shfl(w, (int)(32 | (lane_id() & 31)));
    return lane_id() < 32 ? cnt : 0u;
  }
};
static_assert(kTeamMax == 32 && kCtr == 64, "a report is 32 words and the segments' counts");

struct Team {
  uint64_t *word;       // [2][kTeamMax] episode << 32 | segment word, zero before the first grid barrier
  uint32_t size, rank;  // rank: position in the team (workgroups outside it: any value)
  bool in, usable;
  uint64_t most;    // edges of a round that the team runs
  uint32_t rounds;  // of a stretch
  uint32_t episode;

  __device__ void init(const ArenaView &a, uint64_t *w, uint32_t nxcd, bool bounded) {
    const uint32_t x = nxcd < gridDim.x ? nxcd : gridDim.x;
    word = w;
    size = (gridDim.x + x - 1) / x;
    rank = blockIdx.x / x;
    in = blockIdx.x % x == 0;
    usable = hs_rounds::team_usable(size, gridDim.x, bounded);
    most = hs_rounds::team_edges(size);
    rounds = hs_rounds::team_rounds(a.spin_limit);
    episode = 0;
  }
  // Barrier of the team; `mine` (thread 0): this workgroup's segment word, `seg`:
  // everyone's.  Words alternate by parity: a workgroup writes the same word again
  // two episodes on, when all have read it.  A status uniform across the workgroup.
  __device__ __forceinline__ int sync(const ArenaView &a, uint32_t mine, Segments &seg) {
    __shared__ int rc_sh;
    __shared__ uint32_t seg_sh[64];
    ++episode;
    wait_stores();
    __syncthreads();
    if (threadIdx.x < 64) {
      uint64_t *w = word + (episode & 1) * kTeamMax;
      const uint32_t want = episode, lane = lane_id();
      // an exchange: it reaches the readers in 0.22 us, a store in 0.32
      if (lane == 0)
        (void)__hip_atomic_exchange(w + rank, ((uint64_t)want << 32) | mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      uint64_t got = 0;
      const int rc = spin_until(a, [&] {
        got = lane < size ? ld_u64(w + lane) : (uint64_t)want << 32;
        return ballot((uint32_t)(got >> 32) != want) == 0;
      }, 1);
      seg_sh[lane] = (uint32_t)got;
      if (lane == 0) rc_sh = rc;
    }
    __syncthreads();
    seg.take(seg_sh[lane_id()]);
    return rc_sh;
  }
};

// hs_worklist.hpp's wave_push_batch and wave_push_chunks_batch for readers that no
// acquire precedes: agent-scope stores.
template <int B>
__device__ __forceinline__ void team_push(uint32_t *q, uint32_t *cnt, const bool (&want)[B], const uint32_t (&v)[B]) {
  uint64_t mask[B];
  uint32_t total = 0;
#pragma unroll
  for (int x = 0; x < B; ++x) {
    mask[x] = ballot(want[x]);
    total += (uint32_t)__builtin_popcountll(mask[x]);
  }
  if (total == 0) return;
  uint32_t base = 0;
  if (lane_id() == 0) base = add_relaxed(cnt, total);
  base = __builtin_amdgcn_readfirstlane(base);
#pragma unroll
  for (int x = 0; x < B; ++x) {
    if (mask[x] >> lane_id() & 1) st_relaxed(q + base + lanes_below(mask[x]), v[x]);
    base += (uint32_t)__builtin_popcountll(mask[x]);
  }
}

template <int B>
__device__ __forceinline__ bool team_push_chunks(uint64_t *hq, uint32_t *hcnt, const uint32_t (&nc)[B],
                                                 const uint32_t (&v)[B]) {
  uint32_t ncl = 0;
#pragma unroll
  for (int x = 0; x < B; ++x) ncl += nc[x];
  if (!ballot(ncl != 0)) return false;
  const uint32_t incl = wave_incl_scan(ncl);
  const uint32_t total = __builtin_amdgcn_readlane(incl, 63);
  uint32_t base = 0;
  if (lane_id() == 63) base = add_relaxed(hcnt, total);
  base = __builtin_amdgcn_readlane(base, 63) + incl - ncl;
#pragma unroll
  for (int x = 0; x < B; ++x)
    for (uint32_t c = 0; c < nc[x]; ++c) st_u64(hq + base++, v[x] | ((uint64_t)c << 32));
  return true;
}

// A wave's appends to one queue, staged in LDS: every atomic on a queue's counter
// serializes for ~11 ns over the whole device, and with one per batch of 256 edges
// those atomics were most of a large round (R-MAT 22, one source: 7.7 -> 2.9 ms then).
// The count is the same in every lane.
template <class T, uint32_t CAP>
struct WaveList {
  T *buf;         // [CAP] LDS of this wave
  uint32_t n;
  T *q;           // the queue and its counter
  uint32_t *cnt;

  __device__ __forceinline__ void flush() {
    if (n == 0) return;
    uint32_t base = 0;
    if (lane_id() == 0) base = add_relaxed(cnt, n);
    base = __builtin_amdgcn_readfirstlane(base);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (uint32_t i = lane_id(); i < n; i += 64) put(q + base + i, buf[i]);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    n = 0;
  }
  // room for `total` more entries, in LDS (returns true) or not at all
  __device__ __forceinline__ bool room(uint32_t total) {
    if (n + total > CAP) flush();
    return total <= CAP;
  }
  static __device__ __forceinline__ void put(uint32_t *p, uint32_t v) { st_relaxed(p, v); }
  static __device__ __forceinline__ void put(uint64_t *p, uint64_t v) { st_u64(p, v); }
};

constexpr uint32_t kWaveNear = 512, kWaveFar = 256, kWaveChunks = 128;
struct WaveBuffers {
  uint64_t chunks[kTeamWg / 64][kWaveChunks];
  uint32_t near[kTeamWg / 64][kWaveNear];
};

template <int B, uint32_t CAP>
__device__ __forceinline__ void wave_list_push(WaveList<uint32_t, CAP> &l, const bool (&want)[B], const uint32_t (&v)[B]) {
  static_assert(B * 64 <= CAP, "a batch fits");
  uint64_t mask[B];
  uint32_t total = 0;
#pragma unroll
  for (int x = 0; x < B; ++x) {
    mask[x] = ballot(want[x]);
    total += (uint32_t)__builtin_popcountll(mask[x]);
  }
  if (total == 0) return;
  l.room(total);
  uint32_t at = l.n;
#pragma unroll
  for (int x = 0; x < B; ++x) {
    if (mask[x] >> lane_id() & 1) l.buf[at + lanes_below(mask[x])] = v[x];
    at += (uint32_t)__builtin_popcountll(mask[x]);
  }
  l.n = at;
}

// chunk entries v | c << 32 (c < nc[x])
template <int B, uint32_t CAP>
__device__ __forceinline__ void wave_list_push_chunks(WaveList<uint64_t, CAP> &l, const uint32_t (&nc)[B],
                                                      const uint32_t (&v)[B]) {
  uint32_t ncl = 0;
#pragma unroll
  for (int x = 0; x < B; ++x) ncl += nc[x];
  if (!ballot(ncl != 0)) return;
  const uint32_t incl = wave_incl_scan(ncl);
  const uint32_t total = __builtin_amdgcn_readlane(incl, 63);
  if (l.room(total)) {
    uint32_t at = l.n + incl - ncl;
#pragma unroll
    for (int x = 0; x < B; ++x)
      for (uint32_t c = 0; c < nc[x]; ++c) l.buf[at++] = v[x] | ((uint64_t)c << 32);
    l.n += total;
  } else {
    team_push_chunks<B>(l.q, l.cnt, nc, v);
  }
}

// A workgroup's outputs of a team round: its segment's count and whether it appended
// to the queues.
struct Output {
  // by round parity; a round clears the other one, a stretch begins with both clear
  // (the count of the last round of the stretch before is still there)
  uint32_t cnt[2], queued[2];

  __device__ void clear(uint32_t par) { cnt[par] = queued[par] = 0; }  // one thread
  __device__ uint32_t segment_word(uint32_t par) const {
    return min(cnt[par], kSegCap) | (queued[par] ? 0x80000000u : 0u);
  }
};

// A list kept in LDS over the rounds of a stretch until it is asked for (the SSSP
// far list).
constexpr uint32_t kStage = 4096;
struct Kept {
  uint32_t slots, fill;  // slots handed out of `keep`, end of the filled ones
  uint32_t keep[kStage];
  __device__ void clear() { slots = fill = 0; }  // one thread
};

// Appends vertices (with their first edges) to the workgroup's segment, those
// that do not fit to the queue.
template <int B>
__device__ __forceinline__ void segment_push(Output &out, uint32_t par, uint64_t *seg, uint32_t *q, uint32_t *cnt,
                                             const bool (&want)[B], const uint32_t (&v)[B], const uint32_t (&eb)[B]) {
  uint64_t mask[B];
  uint32_t total = 0;
#pragma unroll
  for (int x = 0; x < B; ++x) {
    mask[x] = ballot(want[x]);
    total += (uint32_t)__builtin_popcountll(mask[x]);
  }
  if (total == 0) return;
  uint32_t base = 0;
  if (lane_id() == 0) base = atomicAdd(&out.cnt[par], total);
  base = __builtin_amdgcn_readfirstlane(base);
  const bool over = base + total > kSegCap;
  bool rest[B];
#pragma unroll
  for (int x = 0; x < B; ++x) {
    const uint32_t at = base + lanes_below(mask[x]);
    const bool mine = mask[x] >> lane_id() & 1;
    if (mine && at < kSegCap) st_u64(seg + at, v[x] | ((uint64_t)eb[x] << 32));
    rest[x] = mine && at >= kSegCap;
    base += (uint32_t)__builtin_popcountll(mask[x]);
  }
  if (over) {
    team_push<B>(q, cnt, rest, v);
    if (lane_id() == 0) out.queued[par] = 1;
  }
}

// Appends to the kept list, what does not fit to its queue.
template <int B>
__device__ __forceinline__ void kept_push(Kept &k, uint32_t *q, uint32_t *cnt, const bool (&want)[B],
                                          const uint32_t (&v)[B]) {
  uint64_t mask[B];
  uint32_t total = 0;
#pragma unroll
  for (int x = 0; x < B; ++x) {
    mask[x] = ballot(want[x]);
    total += (uint32_t)__builtin_popcountll(mask[x]);
  }
  if (total == 0) return;
  uint32_t base = 0;
  if (lane_id() == 0) {
    base = atomicAdd(&k.slots, total);
    if (base + total <= kStage) atomicMax(&k.fill, base + total);  // slots in order: those that fit form a prefix
  }
  base = __builtin_amdgcn_readfirstlane(base);
  if (base + total > kStage) {
    team_push<B>(q, cnt, want, v);
    return;
  }
#pragma unroll
  for (int x = 0; x < B; ++x) {
    if (mask[x] >> lane_id() & 1) k.keep[base + lanes_below(mask[x])] = v[x];
    base += (uint32_t)__builtin_popcountll(mask[x]);
  }
}

// Moves the kept list to its queue (every thread of the workgroup calls it).
__device__ __forceinline__ void kept_flush(Kept &k, uint32_t *q, uint32_t *cnt) {
  __shared__ uint32_t base_sh;
  __syncthreads();
  const uint32_t n = k.fill;
  if (threadIdx.x == 0) base_sh = n ? add_relaxed(cnt, n) : 0u;
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < n; i += kTeamWg) st_relaxed(q + base_sh + i, k.keep[i]);
  __syncthreads();
  if (threadIdx.x == 0) k.clear();
  __syncthreads();
}

// Vertices a wave takes at once from a queue of nin: 64, fewer (at least 8) while
// that still gives no wave a second share
__device__ __forceinline__ uint32_t queue_share(uint32_t nin, uint32_t waves) {
  uint32_t s = 64;
  while (s > 8 && (uint64_t)nin * 2 <= (uint64_t)waves * s) s >>= 1;
  return s;
}

// ===========================================================================
// single-source BFS (LONESTAR/apps/bfs/kernel_gsrb.cu:400-626)
// Level-synchronous, pushing or (with the transposed graph) pulling.  A vertex
// reached at level L joins the light queue of level L (out-degree < kHeavy) or,
// when heavy, as chunks of kBfsChunk out-edges the chunk list that every wave of
// the grid shares (so one hub does not serialize a level on one workgroup).
// Small levels are pushed by a team (above).  A level whose frontier has a large
// part of the edges not yet behind it is pulled (Beamer, Asanovic & Patterson,
// "Direction-optimizing breadth-first search", 2012): the vertices not yet reached
// look for an in-neighbour in the frontier's bitmap (512 KiB at R-MAT 22, kept in
// L2) and stop at the first; no atomics, and the new bitmap is written a word per
// wave.  R-MAT 22: 1.02 ms pushed only (1.9 ms with one queue atomic per 512
// edges), 0.36 ms; a mesh of 720k vertices 13-16 -> 4.0-5.7 ms with the team, by the
// card.
struct BfsArgs1 {
  uint32_t n, m;
  const uint32_t *row, *col, *rrow, *rcol;  // rrow, rcol null: push only
  int32_t src;
  int32_t *level;
  uint32_t *q;    // [2][n] light frontier queues
  uint64_t *hq;   // [2][hcap] heavy chunk entries v | chunk << 32
  uint64_t hcap;
  uint64_t *seg;  // [2][kTeamMax][kSegCap] segments of a team: v | first edge << 32
  uint64_t *fbm[2];  // frontier bitmaps
  uint32_t *ctr;  // hs_rounds::kSlots, kCtr words apart
  uint32_t *stats;
  uint32_t mean_degree;
  uint32_t ng, nx;
};
static_assert(2 * kTeamMax * sizeof(uint64_t) <= (hs_rounds::kSlots - hs_rounds::kTeamWords) * kCtr * sizeof(uint32_t),
              "the team's words fit their slots");

struct BfInput {
  Segments seg;
  uint32_t nin, nh;
  __device__ bool any() const { return (seg.total | nin | nh) != 0; }
};

__device__ __forceinline__ uint32_t *bf_q(const BfsArgs1 &p, uint32_t r) { return p.q + (size_t)(r & 1) * p.n; }
__device__ __forceinline__ uint64_t *bf_hq(const BfsArgs1 &p, uint32_t r) { return p.hq + (size_t)(r & 1) * p.hcap; }
// chunks that the pull of phase k leaves
__device__ __forceinline__ uint32_t *bf_pcnt(const BfsArgs1 &p, uint32_t k) {
  return p.ctr + hs_rounds::other(k) * kCtr;
}
__device__ __forceinline__ uint64_t *bf_seg(const BfsArgs1 &p, uint32_t r, uint32_t rank) {
  return p.seg + ((size_t)(r & 1) * kTeamMax + rank) * kSegCap;
}

struct BfStep {
  const BfsArgs1 &p;
  uint32_t r;
  Output *out;  // of a team, else null, and the wave's lists instead
  uint32_t rank;
  WaveList<uint32_t, kWaveNear> light;
  WaveList<uint64_t, kWaveChunks> chunks;

  __device__ __forceinline__ void flush() { light.flush(); chunks.flush(); }
};

__device__ __forceinline__ BfStep bf_step(const BfsArgs1 &p, uint32_t r, const Round &rd, Output *out, uint32_t rank,
                                          WaveBuffers *wb) {
  const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  return BfStep{p, r, out, rank,
                {wb ? wb->near[wv] : nullptr, 0, bf_q(p, r + 1), rd.at(hs_rounds::kLight, 1)},
                {wb ? wb->chunks[wv] : nullptr, 0, bf_hq(p, r + 1), rd.at(hs_rounds::kChunks, 1)}};
}

// new vertices of level r + 1 to its input
template <bool TEAM, int B>
__device__ __forceinline__ void bf_push(BfStep &s, const bool (&won)[B], const uint32_t (&v)[B], const uint32_t (&eb)[B],
                                        const uint32_t (&deg)[B]) {
  uint32_t nc[B];
  bool light[B];
#pragma unroll
  for (int x = 0; x < B; ++x) {
    nc[x] = won[x] ? bfs_chunks(deg[x]) : 0u;
    light[x] = won[x] && nc[x] == 0;
  }
  if constexpr (TEAM) {
    segment_push<B>(*s.out, s.r & 1, bf_seg(s.p, s.r + 1, s.rank), s.light.q, s.light.cnt, light, v, eb);
    if (team_push_chunks<B>(s.chunks.q, s.chunks.cnt, nc, v) && lane_id() == 0) s.out->queued[s.r & 1] = 1;
  } else {
    wave_list_push<B>(s.light, light, v);
    wave_list_push_chunks<B>(s.chunks, nc, v);
  }
}

// visit (kernel_gsrb.cu:473-479) of B candidates per lane (~0: none): the minimum
// with the level says whether this visit is the vertex's first
template <bool TEAM, int B>
__device__ __forceinline__ void bf_visit(BfStep &s, const uint32_t (&v)[B]) {
  constexpr bool kBlind = TEAM && B == 1;  // as in the SSSP's relaxation
  const BfsArgs1 &p = s.p;
  const int32_t L = (int32_t)s.r + 1;
  int32_t lv[B];
#pragma unroll
  for (int x = 0; x < B; ++x) {
    lv[x] = 0;
    if (v[x] != 0xFFFFFFFFu) lv[x] = kBlind ? kInf : ld_i32(p.level + v[x]);
  }
  bool won[B];
  uint32_t eb[B], deg[B];
#pragma unroll
  for (int x = 0; x < B; ++x) {
    eb[x] = deg[x] = 0;
    if (lv[x] == kInf) {
      lv[x] = __hip_atomic_fetch_min(p.level + v[x], L, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (TEAM) { eb[x] = p.row[v[x]]; deg[x] = p.row[v[x] + 1] - eb[x]; }
    }
  }
#pragma unroll
  for (int x = 0; x < B; ++x) {
    won[x] = v[x] != 0xFFFFFFFFu && lv[x] == kInf;
    if (!TEAM) deg[x] = won[x] ? p.row[v[x] + 1] - p.row[v[x]] : 0u;
  }
  bf_push<TEAM, B>(s, won, v, eb, deg);
}

template <bool TEAM>
__device__ __forceinline__ void bf_expand(BfStep &s, uint32_t eb, uint32_t deg) {
  constexpr int kB = TEAM ? 4 : kBfsBatch;
  wave_expand<kB>(eb, deg, [&](const uint32_t (&e)[kB], const bool (&ev)[kB], const uint32_t (&)[kB]) {
    uint32_t vb[kB];
#pragma unroll
    for (int x = 0; x < kB; ++x) vb[x] = ev[x] ? s.p.col[e[x]] : 0xFFFFFFFFu;
    bf_visit<TEAM, kB>(s, vb);
  });
}

template <bool TEAM>
__device__ __forceinline__ void bf_push_level(const BfsArgs1 &p, uint32_t r, const Round &rd, const BfInput &in, const Crew &crew,
                                              Output *out, uint32_t rank, WaveBuffers *wb) {
  const uint32_t lane = lane_id();
  BfStep s = bf_step(p, r, rd, out, rank, wb);
  for (uint32_t b = crew.wave; b < in.seg.blocks; b += crew.waves) {
    const uint32_t i = in.seg.entry(b), x = lane & 3;
    const uint64_t ent = i != 0xFFFFFFFFu ? ld_u64(bf_seg(p, r, 0) + i) : 0ull;
    const uint32_t u = (uint32_t)ent, eb = (uint32_t)(ent >> 32);
    uint32_t end = eb, c = 0;
    if (i != 0xFFFFFFFFu) {
      end = p.row[u + 1];
      if (eb + x < p.m) c = p.col[eb + x];
    }
    const uint32_t deg = end - eb;
    if (TEAM && !ballot(deg > 4)) {
      const uint32_t vb[1] = {x < deg ? c : 0xFFFFFFFFu};
      bf_visit<TEAM, 1>(s, vb);
    } else {
      bf_expand<TEAM>(s, eb, x == 0 ? deg : 0u);
    }
  }
  // heavy chunks, spread over the crew
  constexpr int kB = TEAM ? 4 : kBfsBatch;
  const uint64_t *hin = bf_hq(p, r);
  for (uint32_t i = crew.wave; i < in.nh; i += crew.waves) {
    const uint64_t ent = ld_u64(hin + i);
    const uint32_t u = (uint32_t)ent, c = (uint32_t)(ent >> 32);
    const uint32_t eb = p.row[u] + c * kBfsChunk, ee = min(p.row[u + 1], eb + kBfsChunk);
    for (uint32_t e0 = eb; e0 < ee; e0 += kB * 64) {
      uint32_t vb[kB];
#pragma unroll
      for (int x = 0; x < kB; ++x) {
        const uint32_t e = e0 + 64 * x + lane;
        vb[x] = e < ee ? p.col[e] : 0xFFFFFFFFu;
      }
      bf_visit<TEAM, kB>(s, vb);
    }
  }
  // light queue: the first share of each wave is dealt, further ones are grabbed
  const uint32_t *qin = bf_q(p, r);
  const uint32_t share = queue_share(in.nin, crew.waves);
  for (uint32_t b = crew.wave; (uint64_t)b * share < in.nin;) {
    const uint32_t i = b * share + lane;
    const bool valid = lane < share && i < in.nin;
    const uint32_t u = valid ? ld_relaxed(qin + i) : 0u;
    uint32_t eb = 0, deg = 0;
    if (valid) { eb = p.row[u]; deg = p.row[u + 1] - eb; }
    bf_expand<TEAM>(s, eb, deg);
    if ((uint64_t)crew.waves * share >= in.nin) break;
    uint32_t g = 0;
    if (lane == 0) g = add_relaxed(rd.at(hs_rounds::kGrab), 1u);
    b = crew.waves + __builtin_amdgcn_readfirstlane(g);
  }
  if (!TEAM) s.flush();
}

// bitmap of level r's frontier from the levels
__device__ __forceinline__ void bf_make_bitmap(const BfsArgs1 &p, uint32_t r, const Crew &crew) {
  const uint32_t nblk = (p.n + 63) / 64;
  for (uint32_t b = crew.wave; b < nblk; b += crew.waves) {
    const uint32_t v = b * 64 + lane_id();
    const uint64_t w = ballot(v < p.n && p.level[v] == (int32_t)r);
    if (lane_id() == 0) p.fbm[r & 1][b] = w;
  }
}

__device__ __forceinline__ bool bf_in_frontier(const uint64_t *fbm, uint32_t u) { return fbm[u >> 6] >> (u & 63u) & 1u; }

// Pull: every vertex not yet reached looks through its in-edges for the frontier,
// a wave 64 consecutive vertices at a time: the first kPullFirst in-edges by the
// vertex's own lane, then the rest of the vertices still looking packed over the
// wave, in rounds of 8, 16, ... 256 edges each, so that a vertex that finds its
// parent early costs no more.  What is left of a vertex with more than kPullRest
// in-edges becomes chunks that all waves share after the level's barrier.
constexpr uint32_t kPullFirst = 4, kPullRest = 8192, kPullChunk = 4096;

__device__ __forceinline__ void bf_pull_found(BfStep &s, bool found, uint32_t v) {
  const uint32_t row = found ? s.p.row[v] : 0u, end = found ? s.p.row[v + 1] : 0u;
  const bool won[1] = {found};
  const uint32_t vs[1] = {v}, eb[1] = {row}, deg[1] = {end - row};
  bf_push<false, 1>(s, won, vs, eb, deg);
}

__device__ __forceinline__ void bf_pull_level(const BfsArgs1 &p, uint32_t r, const Round &rd, const Crew &crew, WaveBuffers *wb) {
  __shared__ uint32_t hit_sh[kTeamWg];
  const uint32_t lane = lane_id();
  uint32_t *hit = hit_sh + (threadIdx.x & ~63u);
  BfStep s = bf_step(p, r, rd, nullptr, 0, wb);
  const uint64_t *fbm = p.fbm[r & 1];
  uint64_t *nbm = p.fbm[(r + 1) & 1];
  const uint32_t nblk = (p.n + 63) / 64, kb = log2_ceil(nblk);
  for (uint32_t j = crew.wave; j < (1u << kb); j += crew.waves) {
    const uint32_t blk = scatter_block(j, kb);
    if (blk >= nblk) continue;
    const uint32_t v = blk * 64 + lane;
    const bool open = v < p.n && p.level[v] == kInf;
    uint32_t b = 0, rem = 0;
    if (open) { b = p.rrow[v]; rem = p.rrow[v + 1] - b; }
    bool found = false;
    {
      uint32_t u[kPullFirst];
      uint64_t w[kPullFirst];
#pragma unroll
      for (uint32_t x = 0; x < kPullFirst; ++x) u[x] = x < rem ? p.rcol[b + x] : 0xFFFFFFFFu;
#pragma unroll
      for (uint32_t x = 0; x < kPullFirst; ++x) w[x] = u[x] != 0xFFFFFFFFu ? fbm[u[x] >> 6] : 0ull;
#pragma unroll
      for (uint32_t x = 0; x < kPullFirst; ++x) found |= (w[x] >> (u[x] & 63u)) & 1u;
      const uint32_t took = rem < kPullFirst ? rem : kPullFirst;
      b += took;
      rem = found ? 0u : rem - took;
    }
    for (uint32_t cap = 2 * kPullFirst; ballot(rem != 0); cap = cap < 256 ? cap * 2 : 256) {
      if (cap == 256) {
        const bool rest = rem > kPullRest;
        if (ballot(rest)) {
          // the rest of a hub: chunks by first edge, for everyone
          const uint32_t nc = rest ? (rem + kPullChunk - 1) / kPullChunk : 0u;
          const uint32_t incl = wave_incl_scan(nc);
          uint32_t base = 0;
          if (lane == 63) base = add_relaxed(bf_pcnt(p, rd.i), incl);
          base = __builtin_amdgcn_readlane(base, 63) + incl - nc;
          for (uint32_t c = 0; c < nc; ++c) st_u64(bf_hq(p, r) + base + c, v | ((uint64_t)(b + c * kPullChunk) << 32));
          if (rest) rem = 0;
        }
      }
      hit[lane] = 0;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      const uint32_t take = rem < cap ? rem : cap;
      wave_expand<4>(b, take, [&](const uint32_t (&e)[4], const bool (&ev)[4], const uint32_t (&own)[4]) {
        uint32_t u[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) u[x] = ev[x] ? p.rcol[e[x]] : 0u;
#pragma unroll
        for (int x = 0; x < 4; ++x)
          if (ev[x] && bf_in_frontier(fbm, u[x])) hit[own[x]] = 1;
      });
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      const bool got = hit[lane] != 0;
      found |= got;
      b += take;
      rem = got ? 0u : rem - take;
    }
    const uint64_t fm = ballot(found);
    if (lane == 0) nbm[blk] = fm;
    if (found) p.level[v] = (int32_t)r + 1;
    if (fm) bf_pull_found(s, found, v);
  }
  s.flush();
}

// the hubs' chunks: the first wave that finds a parent reaches the vertex
__device__ __forceinline__ void bf_pull_chunks(const BfsArgs1 &p, uint32_t r, const Round &rd, uint32_t count, const Crew &crew,
                                               WaveBuffers *wb) {
  const uint32_t lane = lane_id();
  BfStep s = bf_step(p, r, rd, nullptr, 0, wb);
  const uint64_t *fbm = p.fbm[r & 1];
  for (uint32_t i = crew.wave; i < count; i += crew.waves) {
    const uint64_t ent = ld_u64(bf_hq(p, r) + i);
    const uint32_t v = (uint32_t)ent, eb = (uint32_t)(ent >> 32);
    const uint32_t ee = min(p.rrow[v + 1], eb + kPullChunk);
    bool found = false;
    for (uint32_t e0 = eb; e0 < ee && ld_i32(p.level + v) == kInf; e0 += 4 * 64) {
      bool h = false;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const uint32_t e = e0 + 64 * x + lane;
        h |= e < ee && bf_in_frontier(fbm, p.rcol[e]);
      }
      if (ballot(h)) { found = true; break; }
    }
    bool won = false;
    if (found && lane == 0)
      won = __hip_atomic_fetch_min(p.level + v, (int32_t)r + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == kInf;
    if (won) __hip_atomic_fetch_or(p.fbm[(r + 1) & 1] + (v >> 6), 1ull << (v & 63u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (ballot(won)) bf_pull_found(s, won, v);
  }
  s.flush();
}

template <int KIND>
__global__ void __launch_bounds__(kTeamWg) __attribute__((amdgpu_waves_per_eu(4))) k_bfs(ArenaView a, BfsArgs1 p) {
  GridBarrier gb;
  gb.init(a, KIND, p.ng, p.nx);
  Team team;
  team.init(a, reinterpret_cast<uint64_t *>(p.ctr + hs_rounds::kTeamWords * kCtr), p.nx, KIND != HS_BAR_COOP);
  __shared__ Output out;
  __shared__ WaveBuffers wb;
  const uint32_t t0 = blockIdx.x * kTeamWg + threadIdx.x, nt = gridDim.x * kTeamWg;
  Round grid{p.ctr, hs_rounds::kGrid, 0};   // of this phase
  Round round{p.ctr, hs_rounds::kTeam, 0};  // of the team's next round (of use to the team)
  for (uint64_t v = t0; v < p.n; v += nt) p.level[v] = v == (uint32_t)p.src ? 0 : kInf;
  if (t0 < 2 * kTeamMax) team.word[t0] = 0;
  if (t0 == 0) {
    for (uint32_t i = 0; i < hs_rounds::kReport; ++i) p.ctr[i * kCtr] = 0;
    const uint32_t nc = bfs_chunks(p.row[p.src + 1] - p.row[p.src]);
    for (uint32_t c = 0; c < nc; ++c) p.hq[c] = (uint32_t)p.src | ((uint64_t)c << 32);
    *grid.at(hs_rounds::kChunks) = nc;
    p.q[0] = (uint32_t)p.src;
    *grid.at(hs_rounds::kLight) = nc ? 0u : 1u;
  }
  if (gb.sync<KIND>()) return;
  const Crew all(blockIdx.x, gridDim.x), few(team.rank, team.size);
  uint32_t r = 0;
  uint64_t behind = 0;        // edges of the frontiers so far, by the same estimate as `ahead` below
  bool have_bitmap = false;   // of the present frontier
  BfInput in;
  auto look = [&](const Round &rd) {
    in.nin = ld_uniform(rd.at(hs_rounds::kLight));
    in.nh = ld_uniform(rd.at(hs_rounds::kChunks));
  };
  in.seg.none();
  look(grid);
  auto edges = [&]() { return (uint64_t)(in.seg.total + in.nin) * p.mean_degree + (uint64_t)in.nh * kBfsChunk; };
  while (in.any()) {
    const uint64_t ahead = edges();
    const bool by_team = team.usable && ahead <= team.most;
    const bool pull = p.rrow && !by_team && hs_rounds::pull_pays(ahead, behind, p.m, p.n);
    if (pull && !have_bitmap) {
      bf_make_bitmap(p, r, all);
      if (gb.sync<KIND>()) return;
      have_bitmap = true;
      continue;
    }
    behind += ahead;
    if (t0 == 0) {
      grid.open();
      st_relaxed(bf_pcnt(p, grid.i + 1), 0u);
    }
    if (pull) {
      bf_pull_level(p, r, grid, all, &wb);
    } else if (!by_team) {
      bf_push_level<false>(p, r, grid, in, all, nullptr, 0, &wb);
    } else if (team.in) {
      if (threadIdx.x == 0) { out.clear(0); out.clear(1); }
      __syncthreads();
      for (uint32_t q = 0; q < team.rounds; ++q) {
        const uint32_t par = r & 1;
        if (threadIdx.x == 0) out.clear(par ^ 1);
        if (t0 == 0) round.open();
        bf_push_level<true>(p, r, round, in, few, &out, team.rank, nullptr);
        ++r;
        ++round.i;
        __syncthreads();
        if (team.sync(a, out.segment_word(par), in.seg)) return;
        in.nin = in.nh = 0;
        if (in.seg.queued) look(round);
        if (!in.any() || edges() > team.most) break;
        behind += edges();
      }
      if (t0 < 64) {
        Report rep;
        rep.write(p.ctr, grid.i, in.seg.cnt, {r, in.nin, in.nh, (uint32_t)behind, (uint32_t)(behind >> 32), 0u, 0u, 0u});
      }
    } else {
      gb.poll_sleep = kTeamIdleSleep;
    }
    if (gb.sync<KIND>()) return;
    gb.poll_sleep = 0;
    have_bitmap = pull;
    if (by_team) {
      Report rep;
      rep.read(p.ctr, grid.i);
      r = rep.head(0);
      in.nin = rep.head(1);
      in.nh = rep.head(2);
      behind = rep.head(3) | (uint64_t)rep.head(4) << 32;
      in.seg.take(rep.segment());  // the segments of the last team level are still there
      ++grid.i;
      continue;
    }
    if (pull) {
      const uint32_t hubs = ld_uniform(bf_pcnt(p, grid.i));
      if (hubs) {
        bf_pull_chunks(p, r, grid, hubs, all, &wb);
        if (gb.sync<KIND>()) return;
      }
    }
    ++r;
    ++grid.i;
    in.seg.none();
    look(grid);
  }
  if (t0 == 0 && p.stats) p.stats[0] = r;
}

// ===========================================================================
// SSSP, near/far buckets (LONESTAR/apps/sssp/kernel_gsrb.cu:459-687).
struct SsspArgs {
  uint32_t n, m;
  const uint32_t *row, *col, *w;
  int32_t src, delta;
  int32_t *dist;     // output
  uint64_t *key;     // [n] distance (sign flipped: order of unsigned) << 32 | stamp of its last change
  uint32_t *nq;      // [2][n] near queues (light vertices)
  uint64_t *hq;      // [2][hcap] near chunk lists (heavy vertices, chunks of kBfsChunk edges)
  uint64_t hcap;
  uint32_t *fq;      // [3][n] far lists
  uint64_t *seg;     // [2][kTeamMax][kSegCap] near segments of a team: v | first edge << 32
  uint32_t *ctr;     // hs_rounds::kSlots, kCtr words apart
  uint32_t *stats;
  uint32_t mean_degree;  // rounded up, for the size of a round
  uint32_t ng, nx;
};
constexpr int kSsBatch = 4;

__device__ __forceinline__ uint64_t ss_key(int32_t d, uint32_t stamp) {
  return ((uint64_t)((uint32_t)d ^ 0x80000000u) << 32) | stamp;
}
__device__ __forceinline__ int32_t ss_dist(uint64_t key) { return (int32_t)((uint32_t)(key >> 32) ^ 0x80000000u); }

// where a round stands: r counts rounds and bucket steps; stamp r + 1 marks the
// changes made in it.  far_since: stamps of the changes since the bucket was opened.
struct SsState {
  uint32_t r, epoch, relax, far_since;
};

// the input of a step
struct SsInput {
  Segments seg;
  uint32_t nin, nh, nfar;
  __device__ bool near() const { return (seg.total | nin | nh) != 0; }
};

__device__ __forceinline__ int32_t ss_bound(const SsspArgs &p, uint32_t epoch) {
  return (int32_t)min((int64_t)(epoch + 1) * p.delta, (int64_t)kInf - 1);
}
__device__ __forceinline__ uint32_t *ss_near_q(const SsspArgs &p, uint32_t r) { return p.nq + (size_t)(r & 1) * p.n; }
__device__ __forceinline__ uint32_t *ss_far_q(const SsspArgs &p, uint32_t e) { return p.fq + (size_t)(e % 3) * p.n; }
__device__ __forceinline__ uint32_t *ss_far_cnt(const SsspArgs &p, uint32_t e) {
  return p.ctr + hs_rounds::other(e) * kCtr;
}
__device__ __forceinline__ uint64_t *ss_seg(const SsspArgs &p, uint32_t r, uint32_t rank) {
  return p.seg + ((size_t)(r & 1) * kTeamMax + rank) * kSegCap;
}

// Entries of the next near input (light vertices, heavy ones as chunks that every
// wave shares) and of the far list of bucket `epoch`; out: a team's, else null.
// What a wave needs of its surroundings in a step
struct SsStep {
  const SsspArgs &p;
  SsState st;
  int32_t bound;
  uint32_t far_epoch;  // bucket whose far list is appended to
  Round rd;
  Output *out;         // of a team, else null, and the wave's lists instead
  Kept *kept;
  uint32_t rank;
  WaveList<uint32_t, kWaveNear> near;
  WaveList<uint32_t, kWaveFar> far;
  WaveList<uint64_t, kWaveChunks> chunks;
};

template <bool TEAM, int B>
__device__ __forceinline__ void sssp_push(SsStep &s, const bool (&near)[B], const bool (&far)[B], const uint32_t (&v)[B],
                                          const uint32_t (&eb)[B], const uint32_t (&deg)[B]) {
  const SsspArgs &p = s.p;
  const uint32_t r = s.st.r;
  uint32_t nc[B];
  bool light[B];
#pragma unroll
  for (int x = 0; x < B; ++x) {
    nc[x] = near[x] ? bfs_chunks(deg[x]) : 0u;
    light[x] = near[x] && nc[x] == 0;
  }
  if constexpr (TEAM) {
    segment_push<B>(*s.out, r & 1, ss_seg(p, r + 1, s.rank), ss_near_q(p, r + 1), s.rd.at(hs_rounds::kLight, 1), light,
                    v, eb);
    kept_push<B>(*s.kept, ss_far_q(p, s.far_epoch), ss_far_cnt(p, s.far_epoch), far, v);
    if (team_push_chunks<B>(p.hq + (size_t)((r + 1) & 1) * p.hcap, s.rd.at(hs_rounds::kChunks, 1), nc, v) &&
        lane_id() == 0)
      s.out->queued[r & 1] = 1;
  } else {
    wave_list_push<B>(s.near, light, v);
    wave_list_push<B>(s.far, far, v);
    wave_list_push_chunks<B>(s.chunks, nc, v);
  }
}

// Relaxation (kernel_gsrb.cu:415) of B candidates per lane (v == ~0 for none),
// their loads and atomics each in flight together.  One 64-bit atomic minimum on
// (distance, stamp of the change) does the update and says whether the vertex is
// in the list already: it joins the near list when within the bucket bound, unless
// an earlier change of this round put it there (stamp r + 1 and within the bound),
// else the far list, unless a change since the bucket was opened did (beyond the
// bound).  A later stamp never lowers a key of equal distance.  Where the atomics
// would contend the present distance is looked at first; the one-edge-per-lane
// rounds of a team do not (each step of their chain of loads is 0.4-0.9 us: 16.2
// -> 11.4 ms on a mesh of 1.1M vertices), and a team loads the degree beside the
// atomic.
template <bool TEAM, int B>
__device__ __forceinline__ void sssp_relax_batch(SsStep &s, const uint32_t (&v)[B], const int32_t (&nd)[B]) {
  constexpr bool kBlind = TEAM && B == 1;
  const SsspArgs &p = s.p;
  const uint32_t stamp = s.st.r + 1;
  uint32_t eb[B], deg[B];
  bool better[B];
  uint64_t old[B];
  int32_t cur[B];
#pragma unroll
  for (int x = 0; x < B; ++x) {
    cur[x] = kInf;
    if (!kBlind && v[x] != 0xFFFFFFFFu) cur[x] = ss_dist(ld_u64(p.key + v[x]));
  }
#pragma unroll
  for (int x = 0; x < B; ++x) {
    better[x] = v[x] != 0xFFFFFFFFu && (kBlind || nd[x] < cur[x]);
    old[x] = 0;
    eb[x] = deg[x] = 0;
    if (better[x]) {
      old[x] = __hip_atomic_fetch_min(p.key + v[x], ss_key(nd[x], stamp), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (TEAM) { eb[x] = p.row[v[x]]; deg[x] = p.row[v[x] + 1] - eb[x]; }
    }
  }
  bool near[B], far[B];
#pragma unroll
  for (int x = 0; x < B; ++x) {
    const int32_t od = ss_dist(old[x]);
    const uint32_t os = (uint32_t)old[x];
    better[x] = better[x] && nd[x] < od;
    near[x] = better[x] && nd[x] <= s.bound && !(od <= s.bound && os == stamp);
    far[x] = better[x] && nd[x] > s.bound && (od == kInf || os < s.st.far_since);
    if (!TEAM) deg[x] = near[x] ? p.row[v[x] + 1] - p.row[v[x]] : 0u;
  }
  sssp_push<TEAM, B>(s, near, far, v, eb, deg);
}

// Edge destinations and weights are read with streaming loads in the rounds of
// the whole grid: each edge is read once per relaxation of its vertex, and cached
// they evict distances (R-MAT 22: 8.5 -> 8.0 ms per source; the same change slowed
// the 64-source SSSP by 2% and left BFS and PageRank unchanged, so only here).
template <bool TEAM>
__device__ __forceinline__ uint32_t ss_edge(const uint32_t *q) {
  return TEAM ? *q : __builtin_nontemporal_load(q);
}

// the edges of up to 64 vertices, one per lane (edges [eb, eb + deg), distance du)
template <bool TEAM>
__device__ __forceinline__ void sssp_expand(SsStep &s, uint32_t eb, uint32_t deg, int32_t du) {
  wave_expand<kSsBatch>(eb, deg, [&](const uint32_t (&e)[kSsBatch], const bool (&ev)[kSsBatch],
                                     const uint32_t (&own)[kSsBatch]) {
    uint32_t vb[kSsBatch];
    int32_t nd[kSsBatch];
#pragma unroll
    for (int x = 0; x < kSsBatch; ++x) {
      const int32_t odu = __shfl(du, (int)own[x]);
      vb[x] = ev[x] ? ss_edge<TEAM>(s.p.col + e[x]) : 0xFFFFFFFFu;
      nd[x] = ev[x] ? odu + (int32_t)ss_edge<TEAM>(s.p.w + e[x]) : 0;
    }
    sssp_relax_batch<TEAM, kSsBatch>(s, vb, nd);
  });
}

// a workgroup's lists: of its waves in a round of the grid, kept in a stretch
union SsLists {
  struct {
    WaveBuffers lists;
    uint32_t far[kTeamWg / 64][kWaveFar];
  } wave;
  Kept kept;
};

// One round, or with an empty near input one bucket step, by the given crew.
// `first`: the thread that clears the counters.
template <bool TEAM>
__device__ __forceinline__ void sssp_step(const SsspArgs &p, SsState &st, const Round &rd, const SsInput &in,
                                          const Crew &crew, bool first, Output *out, uint32_t rank, SsLists *lists) {
  const uint32_t r = st.r, lane = lane_id();
  if (TEAM && threadIdx.x == 0) out->clear((r + 1) & 1);
  if (TEAM && first) rd.open();
  const uint32_t far_epoch = in.near() ? st.epoch : st.epoch + 1;
  const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  SsStep s{p, st, ss_bound(p, st.epoch), far_epoch, rd, out, &lists->kept, rank,
           {TEAM ? nullptr : lists->wave.lists.near[wv], 0, ss_near_q(p, r + 1), rd.at(hs_rounds::kLight, 1)},
           {TEAM ? nullptr : lists->wave.far[wv], 0, ss_far_q(p, far_epoch), ss_far_cnt(p, far_epoch)},
           {TEAM ? nullptr : lists->wave.lists.chunks[wv], 0, p.hq + (size_t)((r + 1) & 1) * p.hcap, rd.at(hs_rounds::kChunks, 1)}};
  if (in.near()) {
    // segments of a team's round
    for (uint32_t b = crew.wave; b < in.seg.blocks; b += crew.waves) {
      const uint32_t i = in.seg.entry(b), x = lane & 3;
      const uint64_t ent = i != 0xFFFFFFFFu ? ld_u64(ss_seg(p, r, 0) + i) : 0ull;
      const uint32_t u = (uint32_t)ent, eb = (uint32_t)(ent >> 32);
      uint32_t end = eb, c = 0, w = 0;
      int32_t du = 0;
      if (i != 0xFFFFFFFFu) {
        end = p.row[u + 1];
        du = ss_dist(ld_u64(p.key + u));
        if (eb + x < p.m) { c = p.col[eb + x]; w = p.w[eb + x]; }
      }
      const uint32_t deg = end - eb;
      if (TEAM && !ballot(deg > 4)) {
        const uint32_t vb[1] = {x < deg ? c : 0xFFFFFFFFu};
        const int32_t nd[1] = {du + (int32_t)w};
        sssp_relax_batch<TEAM, 1>(s, vb, nd);
      } else {
        sssp_expand<TEAM>(s, eb, x == 0 ? deg : 0u, du);
      }
    }
    // heavy chunks of the near input, spread over the crew
    const uint64_t *hin = p.hq + (size_t)(r & 1) * p.hcap;
    for (uint32_t i = crew.wave; i < in.nh; i += crew.waves) {
      const uint64_t ent = ld_u64(hin + i);
      const uint32_t u = (uint32_t)ent, c = (uint32_t)(ent >> 32);
      const uint32_t eb = p.row[u] + c * kBfsChunk, ee = min(p.row[u + 1], eb + kBfsChunk);
      const int32_t du = ss_dist(ld_u64(p.key + u));
      for (uint32_t e0 = eb; e0 < ee; e0 += kSsBatch * 64) {
        uint32_t vb[kSsBatch];
        int32_t nd[kSsBatch];
#pragma unroll
        for (int x = 0; x < kSsBatch; ++x) {
          const uint32_t e = e0 + 64 * x + lane;
          vb[x] = e < ee ? ss_edge<TEAM>(p.col + e) : 0xFFFFFFFFu;
          nd[x] = e < ee ? du + (int32_t)ss_edge<TEAM>(p.w + e) : 0;
        }
        sssp_relax_batch<TEAM, kSsBatch>(s, vb, nd);
      }
    }
    // light near queue: the first share of each wave is dealt, further ones are
    // taken from the round's grab counter
    const uint32_t *qin = ss_near_q(p, r);
    uint32_t *grab = rd.at(hs_rounds::kGrab);
    const uint32_t share = queue_share(in.nin, crew.waves);
    for (uint32_t b = crew.wave; (uint64_t)b * share < in.nin;) {
      const uint32_t i = b * share + lane;
      const bool valid = lane < share && i < in.nin;
      const uint32_t u = valid ? ld_relaxed(qin + i) : 0u;
      uint32_t eb = 0, deg = 0;
      int32_t du = 0;
      if (valid) { eb = p.row[u]; deg = p.row[u + 1] - eb; du = ss_dist(ld_u64(p.key + u)); }
      sssp_expand<TEAM>(s, eb, deg, du);
      if ((uint64_t)crew.waves * share >= in.nin) break;
      uint32_t g = 0;
      if (lane == 0) g = add_relaxed(grab, 1u);
      b = crew.waves + __builtin_amdgcn_readfirstlane(g);
    }
    ++st.relax;
  } else {
    // near input empty: advance the bucket and split the far list
    // (remove_dups_dev + curdelta += DELTA, kernel_gsrb.cu:310-348,669-677).
    // Entries that a shorter path brought below the old bound are done already.
    const uint32_t *fin = ss_far_q(p, st.epoch);
    if (first) st_relaxed(ss_far_cnt(p, st.epoch + 2), 0u);
    const int32_t nbound = ss_bound(p, st.epoch + 1);
    for (uint64_t b = (uint64_t)crew.wave * 64; b < in.nfar; b += (uint64_t)crew.waves * 64) {
      const uint64_t i = b + lane;
      uint32_t v[1] = {0}, eb[1] = {0}, deg[1] = {0};
      bool to_near[1] = {false}, to_far[1] = {false};
      if (i < in.nfar) {
        v[0] = ld_relaxed(fin + i);
        const int32_t d = ss_dist(ld_u64(p.key + v[0]));
        to_near[0] = d > s.bound && d <= nbound;
        to_far[0] = d > nbound;
        if (to_near[0]) { eb[0] = p.row[v[0]]; deg[0] = p.row[v[0] + 1] - eb[0]; }
        if (to_far[0]) st_u64(p.key + v[0], ss_key(d, r + 1));  // in the new bucket's far list
      }
      sssp_push<TEAM, 1>(s, to_near, to_far, v, eb, deg);
    }
    ++st.epoch;
    st.far_since = r + 1;
  }
  if (!TEAM) {
    s.near.flush();
    s.far.flush();
    s.chunks.flush();
  }
  ++st.r;
}

template <int KIND>
__global__ void __launch_bounds__(kTeamWg) __attribute__((amdgpu_waves_per_eu(KIND == HS_BAR_COOP ? 8 : 4)))  // (COOP: no team)
k_sssp(ArenaView a, SsspArgs p) {
  GridBarrier gb;
  gb.init(a, KIND, p.ng, p.nx);
  Team team;
  team.init(a, reinterpret_cast<uint64_t *>(p.ctr + hs_rounds::kTeamWords * kCtr), p.nx, KIND != HS_BAR_COOP);
  __shared__ Output out;
  __shared__ SsLists lists;
  const uint32_t t0 = blockIdx.x * kTeamWg + threadIdx.x, nt = gridDim.x * kTeamWg;
  Round grid{p.ctr, hs_rounds::kGrid, 0};   // of this phase
  Round round{p.ctr, hs_rounds::kTeam, 0};  // of the team's next round (of use to the team)
  for (uint64_t v = t0; v < p.n; v += nt) p.key[v] = ss_key(v == (uint32_t)p.src ? 0 : kInf, 0);
  if (t0 < 2 * kTeamMax) team.word[t0] = 0;
  if (t0 == 0) {
    for (uint32_t i = 0; i < hs_rounds::kReport; ++i) p.ctr[i * kCtr] = 0;
    const uint32_t nc = bfs_chunks(p.row[p.src + 1] - p.row[p.src]);
    if (nc) {
      for (uint32_t c = 0; c < nc; ++c) p.hq[c] = (uint32_t)p.src | ((uint64_t)c << 32);
      *grid.at(hs_rounds::kChunks) = nc;
    } else {
      p.nq[0] = (uint32_t)p.src;
      *grid.at(hs_rounds::kLight) = 1;
    }
  }
  if (gb.sync<KIND>()) return;
  const Crew all(blockIdx.x, gridDim.x), few(team.rank, team.size);
  SsState st{0, 0, 0, 0};
  SsInput in;
  auto look = [&](const Round &rd) {
    in.nin = ld_uniform(rd.at(hs_rounds::kLight));
    in.nh = ld_uniform(rd.at(hs_rounds::kChunks));
    // a round adds to the far list, a bucket step only reads it: its count is looked
    // at where the next step is one
    in.nfar = in.near() ? 1u : ld_uniform(ss_far_cnt(p, st.epoch));
  };
  in.seg.none();
  look(grid);
  bool told = false;  // the input is a stretch's report
  auto small = [&]() {
    if (!team.usable) return false;
    if (!in.near()) return in.nfar <= team.most / 4;
    return (uint64_t)(in.seg.total + in.nin) * p.mean_degree + (uint64_t)in.nh * kBfsChunk <= team.most;
  };
  while (in.near() || in.nfar != 0) {
    const bool by_team = small();
    // the others may read the far count of this bucket as long as the stretch runs
    // (team_rounds.hpp): it stops before the bucket step that would clear it
    const bool one_bucket = !told && !in.near();
    if (t0 == 0) grid.open();
    if (!by_team) {
      sssp_step<false>(p, st, grid, in, all, t0 == 0, nullptr, 0, &lists);
    } else if (team.in) {
      if (threadIdx.x == 0) { out.clear(0); out.clear(1); lists.kept.clear(); }
      __syncthreads();
      for (uint32_t k = 0; k < team.rounds; ++k) {
        const uint32_t par = st.r & 1;
        sssp_step<true>(p, st, round, in, few, t0 == 0, &out, team.rank, &lists);
        ++round.i;
        __syncthreads();
        if (team.sync(a, out.segment_word(par), in.seg)) return;
        in.nin = in.nh = 0;
        in.nfar = 1;  // not looked at while there are near vertices
        if (in.seg.queued) look(round);
        if (!in.near()) {
          // the kept far entries join the bucket's list
          kept_flush(lists.kept, ss_far_q(p, st.epoch), ss_far_cnt(p, st.epoch));
          if (team.sync(a, 0, in.seg)) return;
          look(round);
          if (in.nfar == 0 || one_bucket) break;
        }
        if (!small()) break;
      }
      kept_flush(lists.kept, ss_far_q(p, st.epoch), ss_far_cnt(p, st.epoch));
      if (t0 < 64) {
        Report rep;
        rep.write(p.ctr, grid.i, in.seg.cnt, {st.r, st.epoch, st.relax, st.far_since, in.nin, in.nh, in.nfar, 0u});
      }
    } else {
      gb.poll_sleep = kTeamIdleSleep;
    }
    if (gb.sync<KIND>()) return;
    gb.poll_sleep = 0;
    told = by_team;
    if (by_team) {
      Report rep;
      rep.read(p.ctr, grid.i);
      st = SsState{rep.head(0), rep.head(1), rep.head(2), rep.head(3)};
      in.nin = rep.head(4);
      in.nh = rep.head(5);
      in.nfar = rep.head(6);
      in.seg.take(rep.segment());  // the segments of the last team round are still there
      ++grid.i;
    } else {
      ++grid.i;
      in.seg.none();
      look(grid);
    }
  }
  for (uint64_t v = t0; v < p.n; v += nt) p.dist[v] = ss_dist(p.key[v]);
  if (t0 == 0 && p.stats) { p.stats[0] = st.relax; p.stats[1] = st.epoch; }
}

// ===========================================================================
// PageRank, FP32 ranks and contributions, FP64 sums, pull over the transposed CSR
// in a fixed summation order.
//   x'[v] = (1-a)/n + a*(D/n + sum_{u->v} x[u]/deg(u)),  D = dangling mass
// The in-edges and the vertices form one sequence: a vertex's in-edges, then the
// vertex itself (its "end"), vertex after vertex.  Span i is positions [i S, (i+1) S)
// of it, whatever the degrees are, so every span costs about the same and a wave
// needs no other balancing; the vertices a span starts with are found once per
// launch.  A wave loads the span's sources 16 bytes per lane, gathers their
// contributions (all in flight together: the gathers' L1 lookups are what bounds an
// iteration), writes the running sums to LDS, and then each lane takes a vertex
// that ends in the span as a difference of two of them.  A vertex cut by span
// boundaries leaves one piece per span; the wave that adds the last of its pieces
// (an arrival counter at the span it ends in) sums them in span order and
// finalizes it.  So every vertex is finalized in the same phase as its sums, and an
// iteration needs one grid barrier.  The dangling mass and the L1 change are summed
// in 2^-60 fixed point (integer sums: the same bits whatever the grid or the
// order).  Every order is fixed by the graph alone, so the ranks do not depend on
// the grid.
// R-MAT 22: 0.42 ms an iteration (0.45 with 64-vertex blocks, hub chunks and
// segmented FP32 scans), 64M gathers that each miss the L1 (128-byte lines, 16 MB of
// contributions) and are bound by how many are in flight.  Streaming gathers take
// twice as long, agent-scope ones the same.  768 positions and 3 workgroups per CU are
// 240 of a SIMD's 512 registers and 74 KB of LDS, so that another launch or the
// serving loop fits beside them; in that room 512 positions and 4 workgroups take 0.44
// ms, 1024 and 2 0.46 ms (with 4, which fill the CU, 0.39 ms).
constexpr int kPrQuads = 3;                   // S = 768, of small graphs 256
constexpr uint64_t kPrLargeFrom = 1ull << 22;  // vertices and edges from which spans are large

struct PrArgs {
  uint32_t n;
  const uint32_t *row, *rrow, *rcol;
  float alpha, tol;
  int max_iter;
  float *rank;      // output
  float *x;         // [2][n] iterates
  float *contrib;   // [2][n]
  uint32_t *first;  // [nspans + 1] first vertex whose end is not before the span
  double *tail;     // [nspans] piece of the vertex that runs on past the span
  double *last;     // [nspans] last piece of the cut vertex that ends in the span
  uint32_t *arr;    // [nspans] arrivals so far of that vertex's pieces
  uint64_t *part;   // [2][W][2] dangling mass, L1 change (2^-60 fixed point)
  uint32_t nspans;
  uint32_t *stats;
  uint32_t ng, nx;
};

__device__ __forceinline__ uint64_t q60(double v) { return (uint64_t)(v * 0x1p60); }

__device__ __forceinline__ uint64_t block_sum_u64(uint64_t v) {
  __shared__ uint64_t red[kWg / 64];
  for (int k = 32; k >= 1; k >>= 1) v += shfl64(v, lane_id() ^ k);
  if (lane_id() == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  uint64_t t = 0;
  for (int w = 0; w < kWg / 64; ++w) t += red[w];
  __syncthreads();
  return t;
}

// sum of the workgroups' fixed-point partials q of one parity, as a double
__device__ double pr_fold(const uint64_t *part, uint32_t parity, int q) {
  uint64_t acc = 0;
  for (uint32_t w = threadIdx.x; w < gridDim.x; w += kWg) acc += part[((size_t)parity * gridDim.x + w) * 2 + q];
  return (double)block_sum_u64(acc) * 0x1p-60;
}

// v of another lane by a DPP control, 0 where it has none
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_f64(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0u, (uint32_t)b, CTRL, ROWS, 0xf, false);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0u, (uint32_t)(b >> 32), CTRL, ROWS, 0xf, false);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
// inclusive wave64 scan, a fixed order of additions
__device__ __forceinline__ double wave_incl_scan_f64(double v) {
  v += dpp_f64<0x111, 0xf>(v);
  v += dpp_f64<0x112, 0xf>(v);
  v += dpp_f64<0x114, 0xf>(v);
  v += dpp_f64<0x118, 0xf>(v);
  v += dpp_f64<0x142, 0xa>(v);
  v += dpp_f64<0x143, 0xc>(v);
  return v;
}
__device__ __forceinline__ double readlane_f64(double v, int lane) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)b, lane), hi = __builtin_amdgcn_readlane((uint32_t)(b >> 32), lane);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ double ld_f64(const double *q) {
  return __builtin_bit_cast(double, ld_u64(reinterpret_cast<const uint64_t *>(q)));
}

// sources of four consecutive in-edges; rcol is only 4-byte aligned there
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(4)));

template <int KIND, int QUADS>
__global__ void __launch_bounds__(kWg) __attribute__((amdgpu_waves_per_eu(QUADS > 1 ? 6 : 8)))
k_pagerank(ArenaView a, PrArgs p) {
  constexpr uint32_t S = 256 * QUADS;
  __shared__ __align__(16) double pre_s[kWg / 64][S + 2];
  GridBarrier gb;
  gb.init(a, KIND, p.ng, p.nx);
  const float inv_n = 1.0f / (float)p.n;
  const uint32_t m = p.rrow[p.n], lane = lane_id();
  const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  double *pre = pre_s[wv];
  // iteration 0 state: x = 1/n, contributions and dangling mass of x
  uint64_t dang = 0;
  for (uint32_t v = gtid(); v < p.n; v += gthreads()) {
    p.x[v] = inv_n;
    const uint32_t d = p.row[v + 1] - p.row[v];
    p.contrib[v] = d ? inv_n / (float)d : 0.f;
    if (!d) dang += q60(inv_n);
  }
  for (uint32_t i = gtid(); i <= p.nspans; i += gthreads()) {
    // vertices whose end (position rrow[v + 1] + v) is before the span
    const uint64_t at = (uint64_t)i * S;
    uint32_t lo = 0, hi = p.n;
    while (lo < hi) {
      const uint32_t mid = lo + (hi - lo) / 2;
      if ((uint64_t)p.rrow[mid + 1] + mid < at) lo = mid + 1; else hi = mid;
    }
    p.first[i] = lo;
    if (i < p.nspans) p.arr[i] = 0;
  }
  dang = block_sum_u64(dang);
  if (threadIdx.x == 0) p.part[((size_t)0 * gridDim.x + blockIdx.x) * 2 + 0] = dang;
  if (gb.sync<KIND>()) return;
  int it = 0;
  double l1 = 0;
  uint32_t cur = 0;
  for (; it < p.max_iter; ++it) {
    const float *cin = p.contrib + (size_t)cur * p.n;
    float *cout = p.contrib + (size_t)(cur ^ 1u) * p.n;
    const float *xin = p.x + (size_t)cur * p.n;
    float *xout = p.x + (size_t)(cur ^ 1u) * p.n;
    const double D = pr_fold(p.part, (uint32_t)it & 1u, 0);
    const float base = (float)((1.0 - (double)p.alpha) / p.n + (double)p.alpha * D / p.n);
    uint64_t l1q = 0, dq = 0;  // this thread's share of the L1 change and dangling mass
    // y, L1 term, next contribution and dangling term of vertex v from its sum
    auto finalize = [&](uint32_t v, float sum, float xv, uint32_t d) {
      const float y = base + p.alpha * sum;
      l1q += q60(fabs((double)y - (double)xv));
      xout[v] = y;
      cout[v] = d ? y / (float)d : 0.f;
      if (!d) dq += q60(y);
    };
    for (uint32_t i = blockIdx.x * (kWg / 64) + wv; i < p.nspans; i += gridDim.x * (kWg / 64)) {
      const uint32_t v0 = p.first[i], v1 = p.first[i + 1];
      const uint32_t e0 = (uint32_t)((uint64_t)i * S - v0);
      const uint64_t e1w = (uint64_t)(i + 1) * S - v1;
      const uint32_t e1 = e1w < m ? (uint32_t)e1w : m, cnt = e1 - e0;
      // the first 64 vertices' state is loaded beside the gathers
      uint32_t v = v0 + lane, rb = 0, re = 0, d = 0;
      float xv = 0.f;
      if (v < v1) { rb = p.rrow[v]; re = p.rrow[v + 1]; d = p.row[v + 1] - p.row[v]; xv = xin[v]; }
      float g[QUADS][4];
      {
        u32x4_any c[QUADS];
#pragma unroll
        for (int q = 0; q < QUADS; ++q) {
          const uint32_t at = q * 256 + 4 * lane;
          c[q] = u32x4_any{~0u, ~0u, ~0u, ~0u};
          if (at + 4 <= cnt) {
            c[q] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_any *>(p.rcol + e0 + at));
          } else if (at < cnt) {
            c[q].x = p.rcol[e0 + at];
            if (at + 1 < cnt) c[q].y = p.rcol[e0 + at + 1];
            if (at + 2 < cnt) c[q].z = p.rcol[e0 + at + 2];
          }
        }
#pragma unroll
        for (int q = 0; q < QUADS; ++q)
#pragma unroll
          for (int k = 0; k < 4; ++k) g[q][k] = c[q][k] != ~0u ? cin[c[q][k]] : 0.f;
      }
      double run = 0.0;
#pragma unroll
      for (int q = 0; q < QUADS; ++q) {
        const double d1 = (double)g[q][0], d2 = d1 + (double)g[q][1], d3 = d2 + (double)g[q][2], d4 = d3 + (double)g[q][3];
        const double inc = wave_incl_scan_f64(d4);
        // the lanes before this one: the scan's value one lane down
        double ex = dpp_f64<0x138, 0xf>(inc);  // wave_shr:1, 0 into lane 0
        ex += run;
        run += readlane_f64(inc, 63);
        double *o = pre + q * 256 + 4 * lane;
        o[0] = ex;
        o[1] = ex + d1;
        o[2] = ex + d2;
        o[3] = ex + d3;
      }
      if (lane == 0) pre[S] = run;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      double cut = 0.0;  // of v0, if it began before the span
      while (v0 < v1) {
        if (v < v1) {
          const double sum = pre[re - e0] - pre[rb > e0 ? rb - e0 : 0u];
          if (rb < e0) cut = sum;
          else finalize(v, (float)sum, xv, d);
        }
        if (v - lane + 64 >= v1) break;
        v += 64;
        if (v < v1) { rb = p.rrow[v]; re = p.rrow[v + 1]; d = p.row[v + 1] - p.row[v]; xv = xin[v]; }
      }
      // pieces of cut vertices: lane 0 the last one of v0, lane 1 that of v1, which
      // runs on; published, then arrived
      const uint32_t tb = v1 < p.n ? p.rrow[v1] : m, te = v1 < p.n ? p.rrow[v1 + 1] : m;
      const uint32_t hb = v0 < p.n ? p.rrow[v0] : m;
      const bool ends = v0 < v1 && hb < e0, runs = v1 < p.n && tb < e1;
      if (ends | runs) {
        const double runs_sum = runs ? run - pre[tb > e0 ? tb - e0 : 0u] : 0.0;
        uint32_t from = 0, to = 0;
        bool mine = false;
        if (lane == 0 && ends) {
          __hip_atomic_store(reinterpret_cast<uint64_t *>(p.last + i), __builtin_bit_cast(uint64_t, cut), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
          from = (uint32_t)(((uint64_t)hb + v0) / S);
          to = i;
          mine = true;
        }
        if (lane == 1 && runs) {
          __hip_atomic_store(reinterpret_cast<uint64_t *>(p.tail + i), __builtin_bit_cast(uint64_t, runs_sum),
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          from = (uint32_t)(((uint64_t)tb + v1) / S);
          to = (uint32_t)(((uint64_t)te + v1) / S);
          mine = true;
        }
        wait_stores();
        bool done = false;
        if (mine) done = add_relaxed(p.arr + to, 1u) + 1u == (uint32_t)(it + 1) * (to - from + 1);
        for (uint64_t todo = ballot(done); todo; todo &= todo - 1) {
          const uint32_t l = (uint32_t)__builtin_ctzll(todo), f = __shfl(from, (int)l), t = __shfl(to, (int)l);
          double sum = 0.0;
          for (uint32_t k = f; k < t; k += 64) {
            const double piece = k + lane < t ? ld_f64(p.tail + k + lane) : 0.0;
            sum += readlane_f64(wave_incl_scan_f64(piece), 63);
          }
          if (lane == 0) {
            sum += ld_f64(p.last + t);
            const uint32_t cv = l == 0 ? v0 : v1;
            finalize(cv, (float)sum, xin[cv], p.row[cv + 1] - p.row[cv]);
          }
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // read before the next span's sums
    }
    l1q = block_sum_u64(l1q);
    dq = block_sum_u64(dq);
    if (threadIdx.x == 0) {
      p.part[((size_t)(((uint32_t)it + 1) & 1u) * gridDim.x + blockIdx.x) * 2 + 0] = dq;
      p.part[((size_t)((uint32_t)it & 1u) * gridDim.x + blockIdx.x) * 2 + 1] = l1q;
    }
    if (gb.sync<KIND>()) return;
    cur ^= 1u;
    l1 = pr_fold(p.part, (uint32_t)it & 1u, 1);
    if (l1 < (double)p.tol) { ++it; break; }
  }
  const float *xf = p.x + (size_t)cur * p.n;
  for (uint32_t v = gtid(); v < p.n; v += gthreads()) p.rank[v] = xf[v];
  if (gtid() == 0 && p.stats) {
    p.stats[0] = (uint32_t)it;
    const float l1f = (float)l1;
    p.stats[1] = __float_as_uint(l1f);
  }
}

template <int KIND>
constexpr auto k_pagerank_large = k_pagerank<KIND, kPrQuads>;
template <int KIND>
constexpr auto k_pagerank_small = k_pagerank<KIND, 1>;

#define HS_KIND_SWITCH(KERNEL, kind)                                            \
  [&]() -> const void * {                                                       \
    switch (kind) {                                                             \
      case HS_BAR_FLAT: return (const void *)KERNEL<HS_BAR_FLAT>;               \
      case HS_BAR_TWO_LEVEL: return (const void *)KERNEL<HS_BAR_TWO_LEVEL>;     \
      case HS_BAR_XCD: return (const void *)KERNEL<HS_BAR_XCD>;                 \
      case HS_BAR_XCD_FLAT_RELEASE: return (const void *)KERNEL<HS_BAR_XCD_FLAT_RELEASE>; \
      case HS_BAR_TREE: return (const void *)KERNEL<HS_BAR_TREE>;               \
      case HS_BAR_LF: return (const void *)KERNEL<HS_BAR_LF>;                   \
      case HS_BAR_COOP: return (const void *)KERNEL<HS_BAR_COOP>;               \
      case HS_BAR_NAIVE_ALL: return (const void *)KERNEL<HS_BAR_NAIVE_ALL>;     \
      default: return nullptr;                                                  \
    }                                                                           \
  }()

size_t align256(size_t b) { return (b + 255) / 256 * 256; }

// Grid of a kernel of kTeamWg-thread workgroups: num_wgs of them (0: one per CU), at
// most one per CU.  Requests that kWg-thread workgroups could not serve (8 per CU) are
// refused as they would be there.
int team_grid_for(const void *k, hs_arena *ar, int num_wgs) {
  const int cus = hs_host::device_cus();
  if (num_wgs > 8 * cus || num_wgs > ar->view.max_blocks) return -1;
  const int g = std::min({num_wgs > 0 ? num_wgs : cus, cus, ar->view.max_blocks});
  return hs_host::check_residency(k, g, kTeamWg, 0) == HS_OK ? g : -1;
}

int grid_for(const void *k, hs_arena *ar, int num_wgs, int per_cu = 2) {
  if (num_wgs <= 0) {  // the default grid, within the arena's barrier slots
    num_wgs = hs_host::default_grid(k, kWg, per_cu);
    if (num_wgs > ar->view.max_blocks) num_wgs = ar->view.max_blocks;
  }
  if (num_wgs > ar->view.max_blocks) return -1;
  if (hs_host::check_residency(k, num_wgs, kWg, 0) != HS_OK) return -1;
  return num_wgs;
}

uint64_t ms_hcap(uint32_t n, uint64_t m) { return m / kHeavy + m / kMsChunk + 64; }

}  // namespace

extern "C" {

// ---------------------------------------------------------------- BFS
// heavy chunk list capacity: a vertex of d >= kHeavy out-edges has at most
// d / kHeavy chunks of kBfsChunk, and each vertex is reached once
static uint64_t bfs_hcap(uint64_t m) { return m / kHeavy + 64; }

// work layouts: queues, counters, chunk lists, then (load-balanced) the balanced
// lists or (plain) the bitmaps; the team's segments last
static uint64_t bfs_bitmap_bytes(uint32_t n) { return align256(sizeof(uint64_t) * ((n + 63ull) / 64)); }

int hs_bfs_work_size(uint32_t n, uint64_t m, uint64_t *bytes) {
  if (!bytes) return HS_ERR_INVALID;
  *bytes = align256(sizeof(uint32_t) * 2ull * n) + align256(sizeof(uint32_t) * hs_rounds::kSlots * kCtr) +
           2 * align256(sizeof(uint64_t) * 2 * bfs_hcap(m)) + 2 * bfs_bitmap_bytes(n) +
           align256(sizeof(uint64_t) * 2 * kTeamMax * kSegCap);
  return HS_OK;
}

static bool bfs_args_ok(hs_arena *ar, uint32_t n, uint64_t m, const uint32_t *d_row, const uint32_t *d_col, int32_t src,
                        const int32_t *d_level, const void *d_work) {
  return ar && d_row && (!m || d_col) && d_level && d_work && n != 0 && src >= 0 && (uint32_t)src < n &&
         m <= 0xFFFFFFFFull;
}

static int bfs_launch(hs_arena *ar, uint32_t n, uint64_t m, const uint32_t *d_row, const uint32_t *d_col,
                      const uint32_t *d_rrow, const uint32_t *d_rcol, int32_t src, int32_t *d_level, void *d_work,
                      int kind, int num_wgs, uint32_t *d_stats, void *stream) {
  if (!bfs_args_ok(ar, n, m, d_row, d_col, src, d_level, d_work)) return HS_ERR_INVALID;
  const void *k = HS_KIND_SWITCH(k_bfs, kind);
  if (!k) return HS_ERR_INVALID;
  const int g = team_grid_for(k, ar, num_wgs);
  if (g < 0) return HS_ERR_RESIDENCY;
  hipStream_t s = (hipStream_t)stream;
  int rc = hs_host::prepare_barrier(ar, kind, s);
  if (rc) return rc;
  BfsArgs1 p{};
  p.n = n; p.m = (uint32_t)m; p.row = d_row; p.col = d_col; p.rrow = d_rrow; p.rcol = d_rcol;
  p.src = src; p.level = d_level;
  char *w = (char *)d_work;
  p.q = (uint32_t *)w; w += align256(sizeof(uint32_t) * 2ull * n);
  p.ctr = (uint32_t *)w; w += align256(sizeof(uint32_t) * hs_rounds::kSlots * kCtr);
  p.hq = (uint64_t *)w; w += align256(sizeof(uint64_t) * 2 * bfs_hcap(m));
  p.hcap = bfs_hcap(m);
  for (auto &f : p.fbm) { f = (uint64_t *)w; w += bfs_bitmap_bytes(n); }
  p.seg = (uint64_t *)w;
  p.stats = d_stats;
  p.mean_degree = (uint32_t)((m + n - 1) / n);
  p.ng = (uint32_t)ar->view.num_groups;
  p.nx = (uint32_t)hs_host::xcd_groups(g);
  hs::ArenaView v = ar->view;
  void *args[] = {(void *)&v, (void *)&p};
  return hs_host::launch_persistent(k, args, kind, g, kTeamWg, 0, s);
}

int hs_bfs(hs_arena *ar, uint32_t n, uint64_t m, const uint32_t *d_row, const uint32_t *d_col,
           int32_t src, int32_t *d_level, void *d_work, int kind, int num_wgs, uint32_t *d_stats,
           void *stream) {
  return bfs_launch(ar, n, m, d_row, d_col, nullptr, nullptr, src, d_level, d_work, kind, num_wgs, d_stats, stream);
}

int hs_bfs_dir(hs_arena *ar, uint32_t n, uint64_t m, const uint32_t *d_row, const uint32_t *d_col,
               const uint32_t *d_rrow, const uint32_t *d_rcol, int32_t src, int32_t *d_level, void *d_work, int kind,
               int num_wgs, uint32_t *d_stats, void *stream) {
  if (!d_rrow || (m && !d_rcol)) return HS_ERR_INVALID;
  return bfs_launch(ar, n, m, d_row, d_col, d_rrow, d_rcol, src, d_level, d_work, kind, num_wgs, d_stats, stream);
}

int hs_bfs_lb(hs_arena *ar, uint32_t n, uint64_t m, const uint32_t *d_row, const uint32_t *d_col,
              int32_t src, int32_t *d_level, void *d_work, int kind, int num_wgs, int degree_limit,
              uint32_t *d_stats, void *stream) {
  if (!bfs_args_ok(ar, n, m, d_row, d_col, src, d_level, d_work) || (degree_limit != 0 && degree_limit < (int)kHeavy))
    return HS_ERR_INVALID;
  const void *k = HS_KIND_SWITCH(k_bfs_lb, kind);
  if (!k) return HS_ERR_INVALID;
  const int g = grid_for(k, ar, num_wgs);
  if (g < 0) return HS_ERR_RESIDENCY;
  hipStream_t s = (hipStream_t)stream;
  int rc = hs_host::prepare_barrier(ar, kind, s);
  if (rc) return rc;
  BfsArgs p{};
  p.n = n; p.row = d_row; p.col = d_col; p.src = src; p.level = d_level;
  p.q = (uint32_t *)d_work;
  p.ctr = (uint32_t *)((char *)d_work + align256(sizeof(uint32_t) * 2ull * n));
  p.hq = (uint64_t *)((char *)p.ctr + align256(sizeof(uint32_t) * kBfsCounters * kCtr));
  p.hcap = bfs_hcap(m);
  p.lq = (uint64_t *)((char *)p.hq + align256(sizeof(uint64_t) * 2 * p.hcap));
  p.stats = d_stats;
  // the reference's DEGREE_LIMIT under -l is the grid's thread count
  // (LONESTAR/rt/include/ggcuda.h:19-22); at least kHeavy, so that the heavy
  // list of a level (at most m / limit entries) fits hcap
  p.lb_limit = degree_limit > 0 ? (uint32_t)degree_limit : (uint32_t)g * kWg;
  p.ng = (uint32_t)ar->view.num_groups;
  p.nx = (uint32_t)hs_host::xcd_groups(g);
  hs::ArenaView v = ar->view;
  void *args[] = {(void *)&v, (void *)&p};
  return hs_host::launch_persistent(k, args, kind, g, kWg, 0, s);
}

// ---------------------------------------------------------------- MS-BFS
int hs_msbfs_work_size(uint32_t n, uint64_t m, int nsrc, uint64_t *bytes) {
  (void)nsrc;
  if (!bytes) return HS_ERR_INVALID;
  const uint64_t hcap = ms_hcap(n, m);
  *bytes = 3 * align256(sizeof(uint64_t) * n) + align256(sizeof(uint64_t) * 4 * hcap) +
           align256(sizeof(uint32_t) * kMsCounters * kCtr) + align256(sizeof(uint64_t) * 2 * 4 * 4096) +
           align256(sizeof(uint64_t) * kMsPlanes * (uint64_t)n) + 2 * align256(sizeof(uint64_t) * ((n + 63) / 64)) +
           align256(HS_MSBFS_MAX_LEVELS);
  return HS_OK;
}

int hs_msbfs(hs_arena *ar, uint32_t n, uint64_t m, const uint32_t *d_row, const uint32_t *d_col,
             const uint32_t *d_rrow, const uint32_t *d_rcol, const int32_t *d_srcs, int nsrc,
             int32_t *d_levels, void *d_work, int kind, int num_wgs, int schedule, const float *d_mlp,
             const uint8_t *h_forced, uint32_t *d_trace, void *stream) {
  if (!ar || !d_row || !d_rrow || (m && (!d_col || !d_rcol)) || !d_srcs || nsrc <= 0 || nsrc > 64 ||
      !d_levels || !d_work || n == 0 || m > 0xFFFFFFFFull || schedule < 0 || schedule > 4 ||
      (schedule == 3 && !d_mlp) || (schedule == 4 && !h_forced))
    return HS_ERR_INVALID;
  const void *k = HS_KIND_SWITCH(k_msbfs, kind);
  if (!k) return HS_ERR_INVALID;
  // 4 WGs/CU (the kernel's occupancy): at R-MAT scale 22 with 64 sources,
  // 1.95 ms against 2.41 ms at 2 WGs/CU (the pull's gathers and the update
  // passes both gain from the waves in flight)
  const int g = grid_for(k, ar, num_wgs, 4);
  if (g < 0 || g > 4096) return HS_ERR_RESIDENCY;
  hipStream_t s = (hipStream_t)stream;
  int rc = hs_host::prepare_barrier(ar, kind, s);
  if (rc) return rc;
  MsArgs p{};
  p.n = n; p.m = m; p.row = d_row; p.col = d_col; p.rrow = d_rrow; p.rcol = d_rcol;
  p.srcs = d_srcs; p.nsrc = nsrc; p.levels = d_levels;
  char *w = (char *)d_work;
  p.fb[0] = (uint64_t *)w; w += align256(sizeof(uint64_t) * n);
  p.fb[1] = (uint64_t *)w; w += align256(sizeof(uint64_t) * n);
  p.vis = (uint64_t *)w; w += align256(sizeof(uint64_t) * n);
  p.hcap = ms_hcap(n, m);
  p.hlist = (uint64_t *)w; w += align256(sizeof(uint64_t) * 4 * p.hcap);
  p.hcnt = (uint32_t *)w; w += align256(sizeof(uint32_t) * kMsCounters * kCtr);
  p.part = (uint64_t *)w; w += align256(sizeof(uint64_t) * 2 * 4 * 4096);
  p.planes = (uint64_t *)w; w += align256(sizeof(uint64_t) * kMsPlanes * (uint64_t)n);
  p.fbm[0] = (uint64_t *)w; w += align256(sizeof(uint64_t) * ((n + 63) / 64));
  p.fbm[1] = (uint64_t *)w; w += align256(sizeof(uint64_t) * ((n + 63) / 64));
  uint8_t *forced = (uint8_t *)w;
  if (schedule == 4) HS_TRY_HIP(hipMemcpyAsync(forced, h_forced, HS_MSBFS_MAX_LEVELS, hipMemcpyHostToDevice, s));
  p.schedule = schedule; p.mlp = d_mlp; p.forced = forced; p.trace = d_trace;
  p.ng = (uint32_t)ar->view.num_groups;
  p.nxcd = (uint32_t)hs_host::xcd_groups(g);
  hs::ArenaView v = ar->view;
  void *args[] = {(void *)&v, (void *)&p};
  return hs_host::launch_persistent(k, args, kind, g, kWg, 0, s);
}

// ---------------------------------------------------------------- SSSP
int hs_sssp_work_size(uint32_t n, uint64_t m, uint64_t *bytes) {
  if (!bytes) return HS_ERR_INVALID;
  *bytes = align256(sizeof(uint32_t) * 2ull * n) + align256(sizeof(uint32_t) * 3ull * n) +
           align256(sizeof(uint64_t) * (uint64_t)n) + align256(sizeof(uint32_t) * hs_rounds::kSlots * kCtr) +
           align256(sizeof(uint64_t) * 2 * kTeamMax * kSegCap) +
           align256(sizeof(uint64_t) * 2 * bfs_hcap(m));
  return HS_OK;
}

int hs_sssp(hs_arena *ar, uint32_t n, uint64_t m, const uint32_t *d_row, const uint32_t *d_col,
            const uint32_t *d_w, int32_t src, int32_t delta, int32_t *d_dist, void *d_work, int kind,
            int num_wgs, uint32_t *d_stats, void *stream) {
  if (!ar || !d_row || (m && (!d_col || !d_w)) || !d_dist || !d_work || n == 0 || src < 0 ||
      (uint32_t)src >= n || m > 0xFFFFFFFFull)
    return HS_ERR_INVALID;
  const void *k = HS_KIND_SWITCH(k_sssp, kind);
  if (!k) return HS_ERR_INVALID;
  const int g = team_grid_for(k, ar, num_wgs);
  if (g < 0) return HS_ERR_RESIDENCY;
  hipStream_t s = (hipStream_t)stream;
  int rc = hs_host::prepare_barrier(ar, kind, s);
  if (rc) return rc;
  SsspArgs p{};
  p.n = n; p.m = (uint32_t)m; p.row = d_row; p.col = d_col; p.w = d_w; p.src = src;
  p.delta = delta > 0 ? delta : 10000;  // DELTA default, LONESTAR/apps/sssp/support.cu:10
  p.dist = d_dist;
  char *w = (char *)d_work;
  p.nq = (uint32_t *)w; w += align256(sizeof(uint32_t) * 2ull * n);
  p.fq = (uint32_t *)w; w += align256(sizeof(uint32_t) * 3ull * n);
  p.key = (uint64_t *)w; w += align256(sizeof(uint64_t) * (uint64_t)n);
  p.ctr = (uint32_t *)w; w += align256(sizeof(uint32_t) * hs_rounds::kSlots * kCtr);
  p.seg = (uint64_t *)w; w += align256(sizeof(uint64_t) * 2 * kTeamMax * kSegCap);
  p.hq = (uint64_t *)w;
  p.hcap = bfs_hcap(m);
  p.stats = d_stats;
  p.mean_degree = (uint32_t)((m + n - 1) / n);
  p.ng = (uint32_t)ar->view.num_groups;
  p.nx = (uint32_t)hs_host::xcd_groups(g);
  hs::ArenaView v = ar->view;
  void *args[] = {(void *)&v, (void *)&p};
  return hs_host::launch_persistent(k, args, kind, g, kTeamWg, 0, s);
}

// ---------------------------------------------------------------- PageRank
static bool pr_large(uint32_t n, uint64_t m) { return n + m >= kPrLargeFrom; }
static uint64_t pr_spans(uint32_t n, uint64_t m) {
  const uint64_t S = 256ull * (pr_large(n, m) ? kPrQuads : 1);
  return (n + m + S - 1) / S;
}

}  // extern "C"

// half of a CU's registers
int hs_host::pagerank_wgs_per_cu(uint32_t n, uint64_t m) { return pr_large(n, m) ? 3 : 4; }

extern "C" {

int hs_pagerank_work_size(uint32_t n, uint64_t m, uint64_t *bytes) {
  if (!bytes) return HS_ERR_INVALID;
  const uint64_t ns = std::max(pr_spans(n, m), (std::min(n + m, kPrLargeFrom) + 255) / 256) + 1;  // grows with n and m
  *bytes = align256(sizeof(float) * 2ull * n) * 2 + align256(sizeof(uint64_t) * 2 * 2 * 4096) +
           align256(sizeof(uint32_t) * ns) * 2 + align256(sizeof(double) * ns) * 2;
  return HS_OK;
}

int hs_pagerank_f32(hs_arena *ar, uint32_t n, uint64_t m, const uint32_t *d_row,
                    const uint32_t *d_rrow, const uint32_t *d_rcol, float alpha, float tol,
                    int max_iter, float *d_rank, void *d_work, int kind, int num_wgs,
                    uint32_t *d_stats, void *stream) {
  if (!ar || !d_row || !d_rrow || (m && !d_rcol) || !d_rank || !d_work || n == 0 || !(alpha > 0.f) ||
      !(alpha < 1.f) || max_iter < 1 || m > 0xFFFFFFFFull)
    return HS_ERR_INVALID;
  const void *k = pr_large(n, m) ? HS_KIND_SWITCH(k_pagerank_large, kind) : HS_KIND_SWITCH(k_pagerank_small, kind);
  if (!k) return HS_ERR_INVALID;
  // larger requests than the default are served with it, up to 8 per CU
  const int cus = hs_host::device_cus(), per = hs_host::pagerank_wgs_per_cu(n, m);
  if (num_wgs > 8 * cus || num_wgs > ar->view.max_blocks) return HS_ERR_RESIDENCY;
  const int g = grid_for(k, ar, num_wgs > per * cus ? hs_host::default_grid(k, kWg, per) : num_wgs, per);
  if (g < 0 || g > 4096) return HS_ERR_RESIDENCY;
  hipStream_t s = (hipStream_t)stream;
  int rc = hs_host::prepare_barrier(ar, kind, s);
  if (rc) return rc;
  PrArgs p{};
  p.n = n; p.row = d_row; p.rrow = d_rrow; p.rcol = d_rcol; p.alpha = alpha; p.tol = tol;
  p.max_iter = max_iter; p.rank = d_rank;
  p.nspans = (uint32_t)pr_spans(n, m);
  char *w = (char *)d_work;
  p.x = (float *)w; w += align256(sizeof(float) * 2ull * n);
  p.contrib = (float *)w; w += align256(sizeof(float) * 2ull * n);
  p.part = (uint64_t *)w; w += align256(sizeof(uint64_t) * 2 * 2 * 4096);
  p.first = (uint32_t *)w; w += align256(sizeof(uint32_t) * (p.nspans + 1ull));
  p.arr = (uint32_t *)w; w += align256(sizeof(uint32_t) * (uint64_t)p.nspans);
  p.tail = (double *)w; w += align256(sizeof(double) * (uint64_t)p.nspans);
  p.last = (double *)w;
  p.stats = d_stats;
  p.ng = (uint32_t)ar->view.num_groups;
  p.nx = (uint32_t)hs_host::xcd_groups(g);
  hs::ArenaView v = ar->view;
  void *args[] = {(void *)&v, (void *)&p};
  return hs_host::launch_persistent(k, args, kind, g, kWg, 0, s);
}

}  // extern "C"
