// oic_sort.h -- device-wide exclusive scan (tiles of 256 threads x 8 items, tile sums scanned
// recursively) and a stable LSD radix sort of (uint64 key, uint64 value) pairs for gfx950.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#define SCAN_THREADS 256
#define SCAN_ITEMS   8
#define SCAN_TILE    (SCAN_THREADS * SCAN_ITEMS)

// ---------------------------------------------------------------- exclusive scan (uint64)

__device__ __forceinline__ uint64_t wave_incl_scan_u64(uint64_t v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint64_t t = __shfl_up(v, o);
    if (lane >= o) v += t;
  }
  return v;
}

// block-wide exclusive scan of one value per thread; returns exclusive prefix, total in *tot
__device__ __forceinline__ uint64_t block_excl_scan_u64(uint64_t v, uint64_t *tot) {
  __shared__ uint64_t wsum[SCAN_THREADS / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint64_t inc = wave_incl_scan_u64(v);
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  uint64_t off = 0, all = 0;
  for (int i = 0; i < SCAN_THREADS / 64; i++) {
    if (i < w) off += wsum[i];
    all += wsum[i];
  }
  __syncthreads();
  *tot = all;
  return off + inc - v;
}

template <typename T>
__global__ void __launch_bounds__(SCAN_THREADS) k_scan_tiles(const T *__restrict__ in, uint64_t *__restrict__ out,
                                                             uint64_t *__restrict__ tile_sums, uint64_t n) {
  const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + (uint64_t)threadIdx.x * SCAN_ITEMS;
  uint64_t v[SCAN_ITEMS];
  uint64_t s = 0;
#pragma unroll
  for (int i = 0; i < SCAN_ITEMS; i++) {
    v[i] = (base + i < n) ? (uint64_t)in[base + i] : 0;
    s += v[i];
  }
  uint64_t tot;
  uint64_t off = block_excl_scan_u64(s, &tot);
#pragma unroll
  for (int i = 0; i < SCAN_ITEMS; i++) {
    if (base + i < n) out[base + i] = off;
    off += v[i];
  }
  if (threadIdx.x == 0 && tile_sums) tile_sums[blockIdx.x] = tot;
}

__global__ void __launch_bounds__(SCAN_THREADS) k_scan_add(uint64_t *__restrict__ out, const uint64_t *__restrict__ tile_off,
                                                           uint64_t n) {
  const uint64_t add = tile_off[blockIdx.x];
  const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE;
  for (int i = threadIdx.x; i < SCAN_TILE; i += SCAN_THREADS)
    if (base + i < n) out[base + i] += add;
}

// scratch needed by scan_excl for n items (uint64 words)
static inline uint64_t scan_scratch_words(uint64_t n) {
  uint64_t words = 0;
  while (n > SCAN_TILE) {
    n = (n + SCAN_TILE - 1) / SCAN_TILE;
    words += 2 * n + 2;
  }
  return words + 2;
}

// out[i] = sum(in[0..i)); returns total via *total (device->host copy); scratch from scan_scratch_words
template <typename T>
static hipError_t scan_excl(const T *in, uint64_t *out, uint64_t n, uint64_t *scratch, hipStream_t st, uint64_t *total_host) {
  if (n == 0) {
    if (total_host) *total_host = 0;
    return hipSuccess;
  }
  const uint64_t tiles = (n + SCAN_TILE - 1) / SCAN_TILE;
  uint64_t *sums = scratch;
  uint64_t *sums_off = scratch + tiles + 1;
  hipLaunchKernelGGL(k_scan_tiles<T>, dim3((unsigned)tiles), dim3(SCAN_THREADS), 0, st, in, out, sums, n);
  if (tiles > 1) {
    hipError_t e = scan_excl<uint64_t>(sums, sums_off, tiles, scratch + 2 * tiles + 2, st, nullptr);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_scan_add, dim3((unsigned)tiles), dim3(SCAN_THREADS), 0, st, out, sums_off, n);
  }
  if (total_host) {
    // total = out[n-1] + in[n-1]
    uint64_t last_out = 0;
    T last_in = 0;
    hipMemcpyAsync(&last_out, out + n - 1, sizeof(uint64_t), hipMemcpyDeviceToHost, st);
    hipMemcpyAsync(&last_in, in + n - 1, sizeof(T), hipMemcpyDeviceToHost, st);
    hipError_t e = hipStreamSynchronize(st);
    if (e != hipSuccess) return e;
    *total_host = last_out + (uint64_t)last_in;
  }
  return hipGetLastError();
}

// ---------------------------------------------------------------- stable LSD radix sort
//
// One pass per BITS-bit digit (8 to 11 bits, chosen per sort so that few passes cover the key
// bits).  A pass: k_rs_hist counts each tile's digits (8192 keys per tile, LDS histogram); the
// counts, laid out digit-major (count[digit][tile]), are exclusively scanned, which gives every
// (digit, tile) its first output slot; k_rs_scatter then ranks the tile's keys among equal digits in
// input order, puts the tile in digit order in LDS and writes it from there.  Traffic per key and
// pass: the key read twice, the value once, key and value written (40 B).
//
// Bound by the writes: a tile's pairs of one digit (16 on average at 9 bits) go to one place of the
// output.  Written as they were ranked, each store instruction touched 64 lines; from the sorted
// tile, neighbouring lanes write neighbouring words.  A run still ends within a line, which the next
// tile's run continues, so an XCD takes neighbouring tiles (its own L2 then joins the two parts).
// A wavefront ranks 16 rounds of 64 keys with counters of its own, no barrier between rounds.  An
// index of 150 M positions (5 passes of 9 bits): 44.1 -> 34.3 ms for the whole call, when tiles of
// 4096 keys were written round by round before.

#define RS_THREADS 512
#define RS_ITEMS   16
#define RS_TILE    (RS_THREADS * RS_ITEMS)
#define RS_WAVES   (RS_THREADS / 64)
#define RS_XCDS    8

// workgroups go round the XCDs; each XCD takes a run of neighbouring tiles
static inline uint32_t rs_grid(uint32_t ntiles) { return (ntiles + RS_XCDS - 1) / RS_XCDS * RS_XCDS; }
__device__ __forceinline__ uint32_t rs_tile(uint32_t ntiles) {
  return (blockIdx.x % RS_XCDS) * ((ntiles + RS_XCDS - 1) / RS_XCDS) + blockIdx.x / RS_XCDS;
}

template <int BITS>
__global__ void __launch_bounds__(RS_THREADS) k_rs_hist(const uint64_t *__restrict__ keys, uint64_t n, int shift,
                                                        uint32_t *__restrict__ counts, uint32_t ntiles) {
  constexpr int NB = 1 << BITS;
  __shared__ uint32_t h[NB];
  const uint32_t tile = rs_tile(ntiles);
  if (tile >= ntiles) return;
  for (int i = threadIdx.x; i < NB; i += RS_THREADS) h[i] = 0;
  __syncthreads();
  const uint64_t base = (uint64_t)tile * RS_TILE;
#pragma unroll 4
  for (int r = 0; r < RS_ITEMS; r++) {
    const uint64_t i = base + (uint64_t)r * RS_THREADS + threadIdx.x;
    if (i < n) atomicAdd(&h[(uint32_t)(keys[i] >> shift) & (NB - 1)], 1u);
  }
  __syncthreads();
  for (int b = threadIdx.x; b < NB; b += RS_THREADS) counts[(uint64_t)b * ntiles + tile] = h[b];
}

template <int BITS>
__global__ void __launch_bounds__(RS_THREADS) __attribute__((amdgpu_waves_per_eu(4, 4))) k_rs_scatter(const uint64_t *__restrict__ kin, const uint64_t *__restrict__ vin,
                                                           uint64_t *__restrict__ kout, uint64_t *__restrict__ vout, uint64_t n,
                                                           int shift, const uint64_t *__restrict__ offs, uint32_t ntiles) {
  constexpr int NB = 1 << BITS;
  constexpr int PER = NB > RS_THREADS ? NB / RS_THREADS : 1;    // digits a thread adds up
  __shared__ uint64_t buf[RS_TILE];                // the tile's keys, then its values, in digit order
  __shared__ uint64_t gbase[NB];                   // a digit's first output slot, less its first place in the tile
  __shared__ uint16_t cnt[RS_WAVES][NB];           // keys of each digit so far per wavefront; then their first place
  __shared__ uint32_t wsum[RS_WAVES];
  const uint32_t tile = rs_tile(ntiles);
  if (tile >= ntiles) return;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const uint64_t base = (uint64_t)tile * RS_TILE;
  const uint32_t m = n - base < RS_TILE ? (uint32_t)(n - base) : RS_TILE;
  const uint32_t first = (uint32_t)w * (64 * RS_ITEMS) + lane;
  uint64_t k[RS_ITEMS], v[RS_ITEMS];
#pragma unroll
  for (int r = 0; r < RS_ITEMS; r++) {
    const uint32_t i = first + 64 * r;
    k[r] = i < m ? kin[base + i] : 0;
  }
#pragma unroll
  for (int r = 0; r < RS_ITEMS; r++) {
    const uint32_t i = first + 64 * r;
    v[r] = i < m ? vin[base + i] : 0;
  }
  for (int b = lane; b < NB; b += 64) cnt[w][b] = 0;
  const uint64_t below = (1ull << lane) - 1ull;
  uint16_t place[RS_ITEMS];
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int r = 0; r < RS_ITEMS; r++) {
    const bool valid = first + 64 * r < m;
    const uint32_t dg = (uint32_t)(k[r] >> shift) & (NB - 1);
    // lanes of this wavefront holding the same digit
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < BITS; b++) {
      const uint64_t bl = __ballot((dg >> b) & 1u);
      peers &= ((dg >> b) & 1u) ? bl : ~bl;
    }
    const uint32_t rank = (uint32_t)__builtin_popcountll(peers & below);
    const uint32_t have = *(volatile uint16_t *)&cnt[w][dg];
    place[r] = (uint16_t)(have + rank);
    // the wavefront's LDS operations complete in order: every lane has read before the first of its digit adds
    __builtin_amdgcn_wave_barrier();
    if (valid && rank == 0) *(volatile uint16_t *)&cnt[w][dg] = (uint16_t)(have + (uint32_t)__builtin_popcountll(peers));
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  // first place of each digit in the tile, and of each wavefront's keys within the digit
  uint32_t tot[PER], sum = 0;
#pragma unroll
  for (int j = 0; j < PER; j++) {
    const int b = tid * PER + j;
    tot[j] = 0;
    if (b < NB)
      for (int x = 0; x < RS_WAVES; x++) tot[j] += cnt[x][b];
    sum += tot[j];
  }
  uint32_t inc = sum;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = __shfl_up(inc, o);
    if (lane >= o) inc += t;
  }
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  uint32_t at = inc - sum;
  for (int x = 0; x < w; x++) at += wsum[x];
#pragma unroll
  for (int j = 0; j < PER; j++) {
    const int b = tid * PER + j;
    if (b < NB) {
      gbase[b] = offs[(uint64_t)b * ntiles + tile] - at;
      uint32_t p = at;
      for (int x = 0; x < RS_WAVES; x++) {
        const uint32_t c = cnt[x][b];
        cnt[x][b] = (uint16_t)p;
        p += c;
      }
    }
    at += tot[j];
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < RS_ITEMS; r++) {
    if (first + 64 * r < m) {
      place[r] = (uint16_t)(place[r] + cnt[w][(uint32_t)(k[r] >> shift) & (NB - 1)]);
      buf[place[r]] = k[r];
    }
  }
  __syncthreads();
  uint16_t digit[RS_ITEMS];                        // of the keys that this thread writes, and then of their values
#pragma unroll
  for (int r = 0; r < RS_ITEMS; r++) {
    const uint32_t i = (uint32_t)tid + RS_THREADS * r;
    digit[r] = 0;
    if (i < m) {
      const uint64_t x = buf[i];
      digit[r] = (uint16_t)((uint32_t)(x >> shift) & (NB - 1));
      kout[gbase[digit[r]] + i] = x;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < RS_ITEMS; r++)
    if (first + 64 * r < m) buf[place[r]] = v[r];
  __syncthreads();
#pragma unroll
  for (int r = 0; r < RS_ITEMS; r++) {
    const uint32_t i = (uint32_t)tid + RS_THREADS * r;
    if (i < m) vout[gbase[digit[r]] + i] = buf[i];
  }
}
