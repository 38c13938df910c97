// oic_sched.h -- processing order of candidate pairs.
//
// PLAIN, BATCHED : longest-predicted-first by a static length-based cost proxy, so the heavy tail of
//            repeat pairs starts early and the persistent waves drain evenly.  (PLAIN, one pair per
//            wavefront: a search of 11.5 thousand pairs 35.2 ms in discovery order, 29.3 ms so.)
// LEARNED  : longest-predicted-first by the cost model's predicted DP cells (oic_mlp.h).
// The order never changes a result: every pair's outcome depends on that pair alone.
//
// The order is made on the device, by the radix sort on 16-bit keys: 1024 steps per doubling of the
// cost, far finer than the estimates are good.  (Pairs copied to the host and sorted there: 5 to 9 ms
// for the 80 to 110 thousand pairs of a search that takes 41 to 68 ms.)
#pragma once

#include "oic_mlp.h"
#include "oic_search.h"

#define ORDER_BITS 16

// static proxy: one extension per match node, each about the length of the shorter read
__device__ __forceinline__ float static_cost(const PairRec &p, const int32_t *__restrict__ len) {
  const int32_t a = len[p.s_id], b = len[p.t_id];
  return (p.consistent ? 1.0f : (float)p.nnodes) * (float)(a < b ? a : b);
}

// keys that rise as the cost falls; pred: the model's log(1 + DP cells) per pair (MLP_OUT floats a pair), or null
__global__ void __launch_bounds__(256) k_order_keys(const PairRec *__restrict__ pairs, uint64_t np, const int32_t *__restrict__ len,
                                                    const float *__restrict__ pred, uint64_t *__restrict__ key, uint64_t *__restrict__ val) {
  const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  const float doublings = pred ? pred[p * MLP_OUT] * 1.44269504f : log2f(1.0f + static_cost(pairs[p], len));
  const float top = (float)((1 << ORDER_BITS) - 1);
  const float x = fminf(fmaxf(doublings * 1024.0f, 0.0f), top);
  key[p] = (uint64_t)(top - x);
  val[p] = p;
}

// the order, from the sorted values, or pair 0 alone where there are none
__global__ void __launch_bounds__(256) k_order_write(const uint64_t *__restrict__ val, uint64_t np, uint32_t *__restrict__ order) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < np) order[i] = val ? (uint32_t)val[i] : (uint32_t)i;
}

// number of pairs whose prediction is not a finite number (a diverged or corrupt model): any makes the whole batch
// fall back to the static estimate
__global__ void __launch_bounds__(256) k_not_finite(const float *__restrict__ pred, uint64_t np, uint32_t *__restrict__ bad) {
  const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p < np && !isfinite(pred[p * MLP_OUT])) atomicAdd(bad, 1u);
}
