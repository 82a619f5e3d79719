// scan.hip -- persistent u32 prefix sum with a grid barrier.
//
// Replaces gpu_prescan / gpu_add_block_sums / sum_scan_blelloch
// (scan/scan_gsrb.cu:440-804).  The reference runs a padded-LDS Blelloch scan of
// 64 elements per 32-thread block, a barrier per level, and two more host
// launches, and is correct only up to 64^3 elements.  Here one co-resident grid
// processes the input in rounds of what its registers hold, so that every element
// is read once and written once: each workgroup loads a tile (up to 64 elements
// per thread), scans it in place, publishes its sum and takes the sums of the
// workgroups before it in the round and of the rounds before.  A workgroup
// publishes a round only when it has read the whole round before, so two words per
// workgroup suffice and nobody is more than a round ahead.  The one grid barrier
// (any hs_barrier_kind) stands after the first round's words, which are all there
// behind it, and clears the second's: an input of one round waits once (1M elements:
// 12.1 us with the barrier before the first tile and the words polled, 9.9 so).
// Bound by HBM: 2^28 elements 0.57 ms when each round was summed, crossed a barrier
// and was read a second time from the Infinity Cache, 0.43 ms so (5.0 TB/s; a copy
// of that size reaches 5.2); 100M 211 -> 162 us, 30M 63 -> 53, 13M 30 -> 26, 8M and
// less as before (16 us, 12 at 4M, 10 from 2M down).
// uint32 wrap arithmetic: bit-exact for any grid and round size.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>

#include "hs_internal.hpp"
#include "hs_wave.hpp"

using namespace hs;

// Words of hs_scan_u32_noalloc.  Each device holds its own copy until the process
// ends; host code reaches it only through the address hipGetSymbolAddress returns for
// the current device.
constexpr int kNoAllocMaxWgs = 4096;  // requests above this are refused
static __device__ __align__(256) uint64_t scratch[2 * kScanMaxWgs];

namespace {

// Threads of a workgroup, one per CU: with 128 registers half of the CU, so that a scan
// and another launch, or the serving loop, are resident together (1024 threads fill the
// CU; they scan 2^28 elements in 407 us against 428, 13M in 22.8 against 26.1, 8M in
// 17.6 against 15.7).
constexpr int kWg = 512;
static_assert(kScanMaxWgs <= kWg, "a thread per workgroup's word");
constexpr int kWaves = kWg / 64;
constexpr int kSpan = 256;  // elements of a wave's segment: 4 per lane, 1 KiB per instruction
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// scan of 256 elements (4 per lane) behind the prefix `run`, in place
template <bool INCLUSIVE>
__device__ __forceinline__ void seg_scan(u32x4 &x, uint32_t &run) {
  const uint32_t v4 = x[0] + x[1] + x[2] + x[3];
  const uint32_t inc = wave_incl_scan(v4);
  uint32_t pre = run + inc - v4;
  run += __builtin_amdgcn_readlane(inc, 63);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t v = x[k];
    if (INCLUSIVE) { pre += v; x[k] = pre; }
    else { x[k] = pre; pre += v; }
  }
}

// A wave's part as a buffer: loads at or beyond its size give 0 and stores there are
// dropped, which cuts the input's end without a second path (two paths to the data
// registers took twice the registers).  Sizes are multiples of 16 bytes; the offset
// is the lane's alone, as a scalar offset would be taken off the size.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t part_buffer(const uint32_t *p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t *>(p), 0, bytes, 0x00027000);
}
constexpr int kStream = 2;  // nt: every element is read once and written once

__device__ __forceinline__ uint64_t ld_word(const uint64_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_word(uint64_t *p, uint64_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Workgroup w's tile of round r is [(r W + w) TILE, +TILE), a wave's part of it SEGS
// segments.  words[2][W]: (round + 1) << 32 | the workgroup's sum, by round parity.
template <int KIND, int SEGS, bool INCLUSIVE>
__global__ void __launch_bounds__(kWg) __attribute__((amdgpu_waves_per_eu(SEGS > 8 ? 4 : 8)))
k_scan_u32(ArenaView a, const uint32_t *in, uint32_t *out, uint64_t n, uint64_t *words, uint32_t ngroups, uint32_t nxcd) {
  constexpr uint32_t kPart = SEGS * kSpan, kTile = kWaves * kPart;
  __shared__ uint32_t s_wave[kWaves], s_carry[kWaves], s_before[kWaves];
  __shared__ int s_bad;
  GridBarrier gb;
  gb.init(a, KIND, ngroups, nxcd);
  const uint32_t W = gridDim.x, w = blockIdx.x, lane = threadIdx.x & 63;
  const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (threadIdx.x == 0) s_bad = 0;
  const uint64_t n4 = n & ~3ull;
  uint32_t carry = 0;  // sum of all rounds before
  uint32_t r = 0;
  for (uint64_t tile = (uint64_t)w * kTile;; tile += (uint64_t)W * kTile, ++r) {
    const uint64_t base = tile + (uint64_t)wv * kPart;
    const uint64_t left = base < n4 ? (n4 - base) * sizeof(uint32_t) : 0;
    const uint32_t bytes = left < kPart * sizeof(uint32_t) ? (uint32_t)left : kPart * (uint32_t)sizeof(uint32_t);
    uint32_t run = 0;
    u32x4 x[SEGS];
    {
      const auto b = part_buffer(in + base, bytes);
#pragma unroll
      for (int q = 0; q < SEGS; ++q) x[q] = __builtin_amdgcn_raw_buffer_load_b128(b, lane * 16 + q * 1024, 0, kStream);
    }
#pragma unroll
    for (int q = 0; q < SEGS; ++q) {
      seg_scan<INCLUSIVE>(x[q], run);
      // keeps the scanned values and not their parts, whose sums would otherwise be
      // put off to the stores: 16 more registers, and spills
      asm volatile("" : "+v"(x[q]));
    }
    // the whole round before, then this round's word, then the ones before it
    uint32_t got = 0;
    if (W > 1 && r > 0 && threadIdx.x < W) {
      const uint64_t *q = words + ((r - 1) & 1u) * W + threadIdx.x;
      uint64_t v = 0;
      if (spin_until(a, [&] { v = ld_word(q); return (uint32_t)(v >> 32) == r; }, 1)) s_bad = 1;
      got = (uint32_t)v;
    }
    got = __builtin_amdgcn_readlane(wave_incl_scan(got), 63);
    if (lane == 0) { s_wave[wv] = run; s_carry[wv] = got; }
    __syncthreads();
    uint32_t wave_before = 0, agg = 0;
#pragma unroll
    for (uint32_t k = 0; k < kWaves; ++k) {
      const uint32_t s = s_wave[k];
      wave_before += k < wv ? s : 0u;
      agg += s;
      carry += s_carry[k];
    }
    if (W > 1 && threadIdx.x == 0) st_word(words + (r & 1u) * W + w, ((uint64_t)(r + 1) << 32) | agg);
    if (r == 0) {
      // the first round's words and the cleared ones of the second
      if (W > 1 && threadIdx.x == 0) st_word(words + W + w, 0);
      if (gb.sync<KIND>()) return;
    }
    if (tile >= n) return;  // only in the last round, whose later words nobody needs
    got = 0;
    if (threadIdx.x < w) {
      const uint64_t *q = words + (r & 1u) * W + threadIdx.x;
      uint64_t v = 0;
      if (spin_until(a, [&] { v = ld_word(q); return (uint32_t)(v >> 32) == r + 1; }, 1)) s_bad = 1;
      got = (uint32_t)v;
    }
    got = __builtin_amdgcn_readlane(wave_incl_scan(got), 63);
    if (lane == 0) s_before[wv] = got;
    __syncthreads();
    if (s_bad) return;
    uint32_t add = carry + wave_before;
#pragma unroll
    for (uint32_t k = 0; k < kWaves; ++k) add += s_before[k];
    if (W == 1) carry += agg;
    const auto b = part_buffer(out + base, bytes);
#pragma unroll
    for (int q = 0; q < SEGS; ++q) __builtin_amdgcn_raw_buffer_store_b128(x[q] + add, b, lane * 16 + q * 1024, 0, kStream);
    // the one to three elements after the last whole four
    if (n4 < n && n4 - tile < kTile && threadIdx.x == 0) {
      uint32_t sum = add + agg;
      for (uint64_t i = n4; i < n; ++i) {
        const uint32_t v = in[i];
        out[i] = INCLUSIVE ? sum + v : sum;
        sum += v;
      }
    }
    if (tile + (uint64_t)(W - w) * kTile >= n) return;  // this was the last round
  }
}

template <int SEGS, bool INC>
const void *scan_kernel(int kind) {
  switch (kind) {
    case HS_BAR_FLAT: return (const void *)k_scan_u32<HS_BAR_FLAT, SEGS, INC>;
    case HS_BAR_TWO_LEVEL: return (const void *)k_scan_u32<HS_BAR_TWO_LEVEL, SEGS, INC>;
    case HS_BAR_XCD: return (const void *)k_scan_u32<HS_BAR_XCD, SEGS, INC>;
    case HS_BAR_XCD_FLAT_RELEASE: return (const void *)k_scan_u32<HS_BAR_XCD_FLAT_RELEASE, SEGS, INC>;
    case HS_BAR_TREE: return (const void *)k_scan_u32<HS_BAR_TREE, SEGS, INC>;
    case HS_BAR_LF: return (const void *)k_scan_u32<HS_BAR_LF, SEGS, INC>;
    case HS_BAR_COOP: return (const void *)k_scan_u32<HS_BAR_COOP, SEGS, INC>;
    case HS_BAR_NAIVE_ALL: return (const void *)k_scan_u32<HS_BAR_NAIVE_ALL, SEGS, INC>;
    default: return nullptr;
  }
}

template <int SEGS>
const void *scan_kernel(int kind, int inclusive) {
  return inclusive ? scan_kernel<SEGS, true>(kind) : scan_kernel<SEGS, false>(kind);
}

}  // namespace

namespace hs_host {
int prepare_barrier(hs_arena *ar, int kind, hipStream_t s);
int launch_persistent(const void *k, void **args, int kind, int num_wgs, int wg_size, size_t lds,
                      hipStream_t s);
}  // namespace hs_host

// Segments per wave: 16 (128 KiB per workgroup), what its registers hold, or 4 where the
// round size in force asks for less than that of the grid.  Fewer segments give more
// compute units a tile, but bring nothing (2 / 4 / 8 / 16 of them: 1M elements 10.0 /
// 10.0 / 10.1 / 10.1 us, 2M 13.1 / 10.2 / 10.1 / 10.2, 4.1M 21.5 / 14.4 / 12.1 / 12.2, 8M
// 38.6 / 25.2 / 19.1 / 15.7).
static int scan_segs(int grid, uint64_t round_bytes) {
  return (uint64_t)grid * kWaves * kSpan * 16 * sizeof(uint32_t) > round_bytes ? 4 : 16;
}

static uint64_t g_scan_round_bytes = 64ull << 20;

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
uint64_t *g_scratch_dev[kMaxDevices];  // device address of `scratch`, per device
}  // namespace

namespace hs_host {
// Looks up this device's copy of `scratch` (the device must be current).  Called
// once per device from hs_arena_create, so the no-allocation entry point itself
// makes no runtime call beyond its launches.
int scan_scratch_init(int device) {
  if (device < 0 || device >= kMaxDevices) return HS_ERR_INVALID;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch_dev[device]) return HS_OK;
  void *p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !p) {
    fprintf(stderr, "libhs: hipGetSymbolAddress(scratch) failed on device %d: %s\n", device,
            hipGetErrorString(e));
    return HS_ERR_HIP;
  }
  g_scratch_dev[device] = (uint64_t *)p;
  return HS_OK;
}
}  // namespace hs_host

extern "C" {

int hs_scan_scratch_size(int num_wgs, uint64_t n, uint64_t *elems_out) {
  (void)n;
  if (!elems_out) return HS_ERR_INVALID;
  if (num_wgs <= 0) num_wgs = 2 * hs_host::device_cus();
  *elems_out = 2ull * (uint64_t)num_wgs;
  return HS_OK;
}

int hs_scan_set_round_bytes(uint64_t bytes) {
  if (bytes < 4096) return HS_ERR_INVALID;
  g_scan_round_bytes = bytes;
  return HS_OK;
}

int hs_scan_get_round_bytes(uint64_t *bytes_out) {
  if (!bytes_out) return HS_ERR_INVALID;
  *bytes_out = g_scan_round_bytes;
  return HS_OK;
}

// The grid: num_wgs workgroups, at most one per CU.  Requests that 256-thread
// workgroups could not serve are refused as they would be (3 per CU under the XCD
// barrier, whose kernel took 136 registers, else 4).  num_wgs / 2 workgroups, as the 2
// words of d_scratch for each would have it, take twice as long on small grids (30M
// elements, 64 workgroups: 190 us against 93).
static int scan_launch(hs_arena *ar, const uint32_t *d_in, uint32_t *d_out, uint64_t n, int inclusive,
                       uint64_t *words, int kind, int num_wgs, void *stream) {
  if (((uintptr_t)d_in & 15u) || ((uintptr_t)d_out & 15u)) return HS_ERR_INVALID;
  if (!scan_kernel<4>(kind, inclusive)) return HS_ERR_INVALID;
  const int cus = hs_host::device_cus();
  if (num_wgs <= 0) num_wgs = 2 * cus;
  if (num_wgs > ar->view.max_blocks) return HS_ERR_INVALID;
  if (num_wgs > (kind == HS_BAR_XCD ? 3 : 4) * cus) return HS_ERR_RESIDENCY;
  int g = std::min({num_wgs, cus, kScanMaxWgs});
  const int segs = scan_segs(g, g_scan_round_bytes);
  const void *k = segs == 4 ? scan_kernel<4>(kind, inclusive) : scan_kernel<16>(kind, inclusive);
  int rc = hs_host::check_residency(k, g, kWg, 0);
  if (rc) return rc;
  if (n == 0) return HS_OK;
  // no more workgroups than tiles
  const uint64_t tiles = (n + (uint64_t)segs * kWaves * kSpan - 1) / ((uint64_t)segs * kWaves * kSpan);
  if ((uint64_t)g > tiles) g = (int)tiles;
  hipStream_t s = (hipStream_t)stream;
  if ((rc = hs_host::prepare_barrier(ar, kind, s))) return rc;
  hs::ArenaView v = ar->view;
  uint32_t ng = (uint32_t)v.num_groups, nx = (uint32_t)hs_host::xcd_groups(g);
  void *args[] = {(void *)&v, (void *)&d_in, (void *)&d_out, (void *)&n, (void *)&words, (void *)&ng, (void *)&nx};
  return hs_host::launch_persistent(k, args, kind, g, kWg, 0, s);
}

int hs_scan_u32(hs_arena *ar, const uint32_t *d_in, uint32_t *d_out, uint64_t n, int inclusive,
                uint32_t *d_scratch, int kind, int num_wgs, void *stream) {
  if (!ar || !d_scratch || (n && (!d_in || !d_out))) return HS_ERR_INVALID;
  return scan_launch(ar, d_in, d_out, n, inclusive, ar->scan_words, kind, num_wgs, stream);
}

int hs_scan_u32_noalloc(hs_arena *ar, const uint32_t *d_in, uint32_t *d_out, uint64_t n, int inclusive,
                        int kind, int num_wgs, void *stream) {
  if (!ar || (n && (!d_in || !d_out))) return HS_ERR_INVALID;
  if (kind == HS_BAR_COOP) {
    fprintf(stderr, "libhs: hs_scan_u32_noalloc: the cooperative-launch barrier kind is not offered\n");
    return HS_ERR_INVALID;
  }
  if (!scan_kernel<4>(kind, inclusive)) return HS_ERR_INVALID;
  if (num_wgs <= 0) num_wgs = 2 * hs_host::device_cus();
  if (num_wgs > kNoAllocMaxWgs) {
    fprintf(stderr, "libhs: hs_scan_u32_noalloc: %d workgroups exceed the static scratch (%d at most)\n",
            num_wgs, kNoAllocMaxWgs);
    return HS_ERR_INVALID;
  }
  int dev = -1;
  HS_TRY_HIP(hipGetDevice(&dev));
  if (dev != ar->device || dev < 0 || dev >= kMaxDevices) return HS_ERR_INVALID;
  uint64_t *p;
  {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    p = g_scratch_dev[dev];
  }
  if (!p) {
    fprintf(stderr, "libhs: hs_scan_u32_noalloc: no scratch address for device %d\n", dev);
    return HS_ERR_NOT_INIT;
  }
  return scan_launch(ar, d_in, d_out, n, inclusive, p, kind, num_wgs, stream);
}

}  // extern "C"
