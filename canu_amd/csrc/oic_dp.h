// oic_dp.h -- packed reads on the device: views, 16-base windows, comparisons (gfx950).
//
// Bases are 2-bit packed, 16 to a word, and compared 16 at a time with XOR and a count of trailing zeros; N bases
// match anything (an N mask, one bit a base).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#define OIC_WAVE 64

// rightward sequence view: view base i is packed base (b0 + i)
struct SeqV {
  const uint32_t *w;     // 2-bit packed, base p at word p>>4, bits 2*(p&15)
  const uint32_t *nm;    // N mask with the same base indexing, or nullptr
  int64_t b0;
};

__device__ __forceinline__ int lane_id() { return threadIdx.x & (OIC_WAVE - 1); }

// 16 N-mask bits starting at base p, spread to the even bit of each 2-bit base slot
__device__ __forceinline__ uint32_t nwin16(const uint32_t *__restrict__ nm, int64_t p) {
  const int64_t wi = p >> 5;
  const uint32_t s = (uint32_t)(p & 31);
  uint32_t v = __builtin_amdgcn_alignbit(nm[wi + 1], nm[wi], s) & 0xffffu;
  v = (v | (v << 8)) & 0x00ff00ffu;
  v = (v | (v << 4)) & 0x0f0f0f0fu;
  v = (v | (v << 2)) & 0x33333333u;
  v = (v | (v << 1)) & 0x55555555u;
  return v;
}

// equal bases (with 'n' matching anything) among the 64 from A[ia..], T[it..]: five words of each
// loaded together (each strand carries 4 guard words past its last base, so they exist)
__device__ __forceinline__ int32_t match64(const SeqV &A, int64_t ia, const SeqV &T, int64_t it) {
  const int64_t pa = A.b0 + ia, pt = T.b0 + it;
  const uint32_t *wa = A.w + (pa >> 4), *wt = T.w + (pt >> 4);
  const uint32_t sa = (uint32_t)(pa & 15) * 2u, st = (uint32_t)(pt & 15) * 2u;
  uint32_t a[5], b[5];
#pragma unroll
  for (int k = 0; k < 5; k++) {
    a[k] = wa[k];
    b[k] = wt[k];
  }
#pragma unroll
  for (int k = 0; k < 4; k++) {
    uint32_t x = __builtin_amdgcn_alignbit(a[k + 1], a[k], sa) ^ __builtin_amdgcn_alignbit(b[k + 1], b[k], st);
    x = (x | (x >> 1)) & 0x55555555u;
    if (A.nm) x &= ~nwin16(A.nm, pa + 16 * k);
    if (T.nm) x &= ~nwin16(T.nm, pt + 16 * k);
    if (x) return 16 * k + (int32_t)(__builtin_ctz(x) >> 1);
  }
  return 64;
}
