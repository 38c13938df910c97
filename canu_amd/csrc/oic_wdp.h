// oic_wdp.h -- one banded prefix edit distance DP per wavefront (gfx950).
//
// Semantics follow prefixEditDistance::forward / ::reverse
// (src/overlapInCore/liboverlap/prefixEditDistance-forward.C:93-314, -reverse.C:113-330):
//   * row e widens the band by one on each side, reads row e-1 at d-1, d, d+1 with -2 sentinels,
//   * the first diagonal (lowest d) that reaches the end of A or T ends the call,
//     with the branch-point test in double precision (forward.C:172-212),
//   * after each row, diagonals are pruned from both ends while EAL[e][d] + max(d,0) <
//     Edit_Match_Limit[e] (prefixEditDistance.H:249-257), and the first-max Longest is tracked.
// A reverse() call is run as a rightward DP over the reverse-complement strands: comparing
// X[p-r] with Y[q-r] is comparing X_rc[|X|-1-p+r] with Y_rc[|Y|-1-q+r].
//
// A call is a chain of rows, so a row's length decides wherever calls are few.  A first form of this kernel
// (barriers between a row's steps, one chunk's slides after another's, two passes for the pruned range, a
// 12-step shuffle maximum) took about 8000 cycles for the row of a 140-cell band, and its traceback followed
// the path through HBM, three dependent loads a row on one lane.  Here
//   * a row of up to 64 diagonals stays in one register per lane: neighbours come over DPP shifts, the pruned
//     range and who slides on are 64-bit scalar masks, and the row never touches LDS.  Most rows of most calls
//     are such rows (a read pair of 9 % difference keeps about 40 diagonals).  The band moves to the middle of
//     the lanes when one of its ends reaches lane 0 or 63; from 52 diagonals on it moves to the wide form
//     instead, and comes back below 40, so that a band near 64 doesn't move at each row;
//   * in the wide form lane l of chunk c holds diagonal 64 c - 32 + l, so a chunk's place in the LDS ring is
//     uniform and ballots give diagonals at once;
//   * the loads of up to WR_GROUP chunks (four words of each tail in one load each: 48 bases or more) are
//     issued before the first is compared;
//   * a slide past 48 bases is finished by the whole wavefront, 1024 bases at a time, unless many lanes slide on;
//   * the pruned range comes from one ballot per chunk; the row's maximum from the next row's own reads of the
//     band, as in sm_row (oic_batch.h), and one DPP reduction;
//   * a stored cell carries the traceback's choice at that cell in its low two bits.  The traceback loads 32
//     rows of the 64 diagonals around its own at once and walks them in scalar registers.
// One wavefront per workgroup: its LDS operations complete in order, so fences only keep the compiler's order.
// wave_rows is not inlined: the kernels' other live values would otherwise be spilled around its loops.
// Bound by the issue of a wavefront's instructions, one wavefront's chain when calls are few.  Measured as whole
// calls, first form -> wide rows only -> both: 12 DPs of 600 bases 150 -> 95 -> 89 us, 400 of 12 kbp 1.32 -> 0.97
// -> 0.90 ms, 600 extensions of 8 kbp 4.7 -> 2.7 -> 2.5 ms, a search with one candidate pair per wavefront (951
// thousand extensions of 4 %-error reads) 101 -> 51 ms and, after other steps, 44 -> 37 ms.
#pragma once

#include "oic_dp.h"

#define WR_GROUP 4                     // chunks whose loads are in flight together
// Cells of the LDS ring that holds a row.  A band of RING - 63 diagonals touches at most RING / 64 chunks.  The
// first level's bands, up to 960 diagonals (true overlaps of 3 % difference at 4.5 % outgrow 448 at about 640
// errors, 21 kbp), take 8 KB a wavefront: 16 to a CU still fit.  The second level's, up to 8190, take 128 KB.
#define WR_FIRST 1024
#define WR_WIDE  16384
#define WR_MAX_BAND 8190
template <int RING>
constexpr int wr_band() { return RING - 64 < WR_MAX_BAND ? RING - 64 : WR_MAX_BAND; }
// Row storage: cells are stored before pruning; a row adds at most two diagonals, so over a DP at most two
// cells a row are stored beyond the kept ones that val_cap counts.  Room for them:
#define WR_VAL_SLACK(rows) (2 * (int64_t)(rows) + 64)

// the wavefront's two band buffers; ring cell i at [1 + i], copies of the last and first cell around them, so
// that the three cells a lane reads are consecutive words
template <int RING>
struct WaveBand {
  int32_t b[2][RING + 2];
};

struct DPTables {
  const int32_t *error_bound;    // [2^21]
  const int32_t *match_limit;    // [max_errors]
  double   bmv;                  // Branch_Match_Value = e/(1+e)
  double   slope_min;            // MIN_BRANCH_TAIL_SLOPE
  uint32_t min_branch_end_dist;  // MIN_BRANCH_END_DIST (uint32 in the reference)
  int32_t  partial;
};

// per-wave global scratch for row storage and deltas
struct DPScratch {
  int32_t *rowm;         // [max_rows + 2] per stored row: what to add to a diagonal for its cell in rowVal
  int32_t *rowVal;       // [val_cap + WR_VAL_SLACK] cells, the value above two bits of the traceback's choice
  int64_t  val_cap;      // kept cells
  int32_t  max_rows;
  int32_t *dbuf;         // [max_rows + 4] raw traceback stack
  int32_t *ldelta;       // [max_rows + 4] Left_Delta
  int32_t *rdelta;       // [max_rows + 4] Right_Delta
};

struct DPOut {
  int32_t e, a_end, t_end, mte, leftover, ndelta;
  int32_t overflow;
};

struct __attribute__((packed, aligned(4))) Words4 { uint32_t x, y, z, w; };

// pointers of a function that is not inlined carry their address space (a plain one compiles to flat accesses)
typedef const __attribute__((address_space(1))) uint32_t *g_words;
typedef __attribute__((address_space(1))) int32_t *g_ints;
typedef __attribute__((address_space(3))) int32_t *l_ints;

__device__ __forceinline__ int32_t uni(int32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int64_t uni64(int64_t v) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int32_t)(uint32_t)v);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int32_t)(uint32_t)((uint64_t)v >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// keeps the compiler from moving LDS operations across (the hardware keeps a wavefront's in order)
__device__ __forceinline__ void wave_order() { __atomic_signal_fence(__ATOMIC_SEQ_CST); }

// maximum over the wavefront, uniform (values >= -2)
__device__ __forceinline__ int32_t wave_max_dpp(int32_t v) {
#define OIC_WMAX(ctl, rows)                                                                \
  {                                                                                        \
    const int32_t o = __builtin_amdgcn_update_dpp(-2, v, ctl, rows, 0xF, false);           \
    v = o > v ? o : v;                                                                     \
  }
  OIC_WMAX(0x111, 0xF)   // row_shr:1, 2, 4, 8
  OIC_WMAX(0x112, 0xF)
  OIC_WMAX(0x114, 0xF)
  OIC_WMAX(0x118, 0xF)
  OIC_WMAX(0x142, 0xA)   // row_bcast:15 into rows 1 and 3
  OIC_WMAX(0x143, 0xC)   // row_bcast:31 into rows 2 and 3
#undef OIC_WMAX
  return __builtin_amdgcn_readlane(v, 63);
}

// inclusive prefix sum over the wavefront's lanes: within each row of 16 lanes by row shifts
// (lanes whose source lies before the row start add 0), then each row's total carried into the
// rows after it by the row broadcasts of lane 15 (into rows 1 and 3) and lane 31 (into rows 2, 3)
__device__ __forceinline__ int32_t wave_incl_scan(int32_t v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);   // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);   // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);   // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);   // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);   // row_bcast:15
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);   // row_bcast:31
  return v;
}

// lanes whose predicate holds
__device__ __forceinline__ uint64_t lanes(bool p) { return __builtin_amdgcn_ballot_w64(p); }

// lane-wise (value, first index) maximum over the wavefront: largest v, then smallest i; v >= -1
__device__ __forceinline__ void wave_pick(int32_t &v, int32_t &i) {
  const int32_t M = wave_max_dpp(v);
  uint64_t b = lanes(v == M);
  int32_t x = __builtin_amdgcn_readlane(i, __builtin_ctzll(b));
  for (b &= b - 1; b; b &= b - 1) {
    const int32_t y = __builtin_amdgcn_readlane(i, __builtin_ctzll(b));
    x = y < x ? y : x;
  }
  v = M;
  i = x;
}

// position of the lowest set bit, all-ones where there is none (the instruction's own answer; written out,
// the compiler adds a compare and a select)
__device__ __forceinline__ uint32_t lowest_bit(uint32_t x) {
  uint32_t r;
  asm("v_ffbl_b32 %0, %1" : "=v"(r) : "v"(x));
  return r;
}

// the four words holding position p (p >= 0) of a tail: a 32-bit byte offset from the uniform base
__device__ __forceinline__ Words4 words_at(g_words w, int32_t p) {
  typedef const __attribute__((address_space(1))) uint8_t *g_bytes;
  typedef const __attribute__((address_space(1))) Words4 *g_words4;
  const g_words4 x = (g_words4)((g_bytes)w + (uint32_t)(((uint32_t)p >> 2) & ~3u));
  Words4 r;
  r.x = x->x; r.y = x->y; r.z = x->z; r.w = x->w;
  return r;
}

// both bits of every N base among 16 from position p of the N mask
__device__ __forceinline__ uint32_t nspread16(const uint32_t *__restrict__ nm, int64_t p) {
  const uint32_t n = nwin16(nm, p);
  return n | (n << 1);
}

// The two tails of a DP, uniform: words from the one holding base 0, and base 0's place in it
struct WTails {
  g_words wa, wt;
  const uint32_t *nm;        // N mask with absolute base indexing (read only for the tails that hold N)
  int64_t a0, t0;
  int32_t ra, rt;
  bool na, nt;
};

__device__ __forceinline__ WTails make_tails(const uint32_t *words, const uint32_t *nm, int64_t a0, int64_t t0, bool na, bool nt) {
  WTails W;
  W.a0 = a0;
  W.t0 = t0;
  W.wa = (g_words)words + (a0 >> 4);
  W.wt = (g_words)words + (t0 >> 4);
  W.nm = nm;
  W.ra = (int32_t)(a0 & 15);
  W.rt = (int32_t)(t0 & 15);
  W.na = na;
  W.nt = nt;
  return W;
}

// equal bases from positions p of A and q of T on, at most rem, all arguments uniform: 1024 a step
template <bool HASN>
__device__ __forceinline__ int32_t wave_run(const WTails &W, int32_t p, int32_t q, int32_t rem) {
  const int lane = lane_id();
  for (int32_t base = 0;; base += 16 * OIC_WAVE) {
    const int32_t off = base + 16 * lane, r = rem - off;
    const int32_t o = r > 0 ? off : 0;          // lanes past the end read the first window again
    const int32_t ia = W.ra + p + o, it = W.rt + q + o;
    const g_words a = W.wa + (uint32_t)(ia >> 4), b = W.wt + (uint32_t)(it >> 4);
    uint32_t x = __builtin_amdgcn_alignbit(a[1], a[0], (uint32_t)ia * 2u) ^ __builtin_amdgcn_alignbit(b[1], b[0], (uint32_t)it * 2u);
    if (HASN && W.na) x &= ~nspread16(W.nm, W.a0 + p + o);
    if (HASN && W.nt) x &= ~nspread16(W.nm, W.t0 + q + o);
    int32_t k = x ? (int32_t)(__builtin_ctz(x) >> 1) : 16;
    k = k < r ? k : (r > 0 ? r : 0);
    const uint64_t stop = lanes(k < 16 || k == r);
    if (stop) {
      const int f = __builtin_ctzll(stop);
      return base + 16 * f + __builtin_amdgcn_readlane(k, f);
    }
  }
}

// The traceback: Set_Right_Delta (prefixEditDistance-forward.C:31-71) / Set_Left_Delta (-reverse.C:35-93)
// from cell (e, d), whose value is `last`.  Returns the delta's length; the delta goes to sc.rdelta (forward)
// or sc.ldelta (reverse).  end: cells stored.
__device__ __forceinline__ int32_t wave_traceback(const DPScratch &sc, int32_t end, int32_t e, int32_t d, int32_t last, bool is_forward,
                                                  int32_t *leftover, int32_t *t_end, int32_t t_len) {
  constexpr int STEP = 32;
  const int lane = lane_id();
  int32_t *buf = is_forward ? sc.dbuf : sc.ldelta;
  int32_t nev = 0, cnt = 0, ev = 0;             // ev, lane j: the j-th entry since the last flush
  auto flush = [&]() {
    if (lane < cnt) buf[nev + lane] = ev;
    nev += cnt;
    cnt = 0;
  };
  int32_t k = e;
  while (k > 0) {
    // rows k, k - 1, .. k - 31 (row 0 at the least) around diagonal d: a step moves by one diagonal, so the
    // row STEP - 1 steps on is still entered within 31 of d, and its neighbour, read there, within 32
    const int32_t d0 = d - 32;
    const int32_t kr = k - lane > 0 ? k - lane : 0;
    const int32_t base = sc.rowm[kr];         // row kr's diagonal x is cell base + x
    int32_t w[STEP];
#pragma unroll
    for (int j = 0; j < STEP; j++) {
      const int32_t i = __builtin_amdgcn_readlane(base, j) + d0 + lane;   // outside the row: a cell never read
      w[j] = sc.rowVal[i < 0 ? 0 : (i < end ? i : end - 1)];
    }
    const int32_t k0 = k;
#pragma unroll
    for (int j = 0; j < STEP - 1; j++) {        // the last row only gives values
      if (k0 - j > 0) {
        const uint32_t c = (uint32_t)__builtin_amdgcn_readlane(w[j], d - d0) & 3u;
        if (c) {
          d += c == 1u ? -1 : 1;
          const int32_t val = __builtin_amdgcn_readlane(w[j + 1], d - d0) >> 2;
          const int32_t x = c == 1u ? val - last - 1 : last - val;
          ev = lane == cnt ? x : ev;
          last = val;
          if (++cnt == OIC_WAVE) flush();
        }
        k = k0 - j - 1;
      }
    }
  }
  if (cnt) flush();
  __threadfence_block();
  if (is_forward) {
    for (int32_t j = lane; j < nev; j += OIC_WAVE) {
      const int32_t i = nev - j, v = i == nev ? last + 1 : buf[i], w = buf[i - 1];
      sc.rdelta[j] = (v < 0 ? -v : v) * ((w > 0) - (w < 0));
    }
    return nev;
  }
  *leftover = last;
  if (nev > 1 && uni(buf[0]) == 1 && *t_end + t_len > 0) {
    for (int32_t b = 0; b + 1 < nev; b += OIC_WAVE) {     // ascending: a round reads past what it writes
      const int32_t i = b + lane;
      int32_t v = 0;
      if (i + 1 < nev) v = buf[i + 1];
      if (i == 0) v = v > 0 ? v + 1 : v - 1;
      if (i + 1 < nev) buf[i] = v;
    }
    nev--;
    (*t_end)--;
  }
  return nev;
}

// wave_rows' flags
#define WR_NA      1u    // A's read holds N
#define WR_NT      2u    // T's
#define WR_FORWARD 4u
#define WR_STORE   8u    // rows are stored
#define WR_PARTIAL 16u

// a DP's rows: where it ended and what the traceback starts from
struct WRows {
  int32_t e, d, last;        // traceback start: row, diagonal, the cell's value (< 0: the stored one)
  int32_t end;               // cells stored
  int32_t rrow;              // row reached (mte)
  uint32_t cells, slots, rows;
  uint32_t lb;               // this lane's bases compared in slides
  bool mte, overflow;
};

// Equal bases of a chunk's lanes from their positions p of A and q = p + d of T on, at most rem each (0 for lanes
// without a cell): lane l's diagonal is d0 + l, wa and wt hold its words there.
template <bool HASN>
__device__ __forceinline__ int32_t chunk_slide(const WTails &W, const Words4 &wa, const Words4 &wt, int32_t p, int32_t q, int32_t rem,
                                               int32_t d0) {
  const int lane = lane_id();
  const uint32_t sa = (uint32_t)(W.ra + p) * 2u, st = (uint32_t)(W.rt + q) * 2u;   // alignbit takes them modulo 32
  uint32_t y0 = __builtin_amdgcn_alignbit(wa.y, wa.x, sa) ^ __builtin_amdgcn_alignbit(wt.y, wt.x, st);
  uint32_t y1 = __builtin_amdgcn_alignbit(wa.z, wa.y, sa) ^ __builtin_amdgcn_alignbit(wt.z, wt.y, st);
  uint32_t y2 = __builtin_amdgcn_alignbit(wa.w, wa.z, sa) ^ __builtin_amdgcn_alignbit(wt.w, wt.z, st);
  if (HASN && W.na) {
    y0 &= ~nspread16(W.nm, W.a0 + p);
    y1 &= ~nspread16(W.nm, W.a0 + p + 16);
    y2 &= ~nspread16(W.nm, W.a0 + p + 32);
  }
  if (HASN && W.nt) {
    y0 &= ~nspread16(W.nm, W.t0 + q);
    y1 &= ~nspread16(W.nm, W.t0 + q + 16);
    y2 &= ~nspread16(W.nm, W.t0 + q + 32);
  }
  // the first differing base: lowest set bit (two bits a base); all-ones where a word has none
  const uint32_t f0 = lowest_bit(y0), f1 = lowest_bit(y1) | 32u, f2 = lowest_bit(y2) | 64u;
  uint32_t f = f0 < f1 ? f0 : f1;
  f = f < f2 ? f : f2;
  f >>= 1;                                    // 48 and more: no difference among the 48 bases
  int32_t adv = (int32_t)(f < (uint32_t)rem ? f : (uint32_t)rem);
  uint64_t more = lanes(adv >= 48);
  if (more) {
    more = lanes(f >= 48u && rem > 48);
    adv = adv < 48 ? adv : 48;
    if (__builtin_popcountll(more) <= 4) {
      while (more) {
        const int l = __builtin_ctzll(more);
        more &= more - 1;
        const int32_t P = __builtin_amdgcn_readlane(p, l);
        const int32_t k = wave_run<HASN>(W, P + 48, P + d0 + l + 48, __builtin_amdgcn_readlane(rem, l) - 48);
        adv = lane == l ? 48 + k : adv;
      }
    } else if (f >= 48u && rem > 48) {
      SeqV a, t;
      a.w = t.w = (const uint32_t *)(W.wa - (W.a0 >> 4));   // all packed reads
      a.nm = HASN && W.na ? W.nm : nullptr; a.b0 = W.a0;
      t.nm = HASN && W.nt ? W.nm : nullptr; t.b0 = W.t0;
      while (adv < rem) {
        const int32_t k = match64(a, p + adv, t, q + adv);
        adv += k;
        if (k < 64) break;
      }
      adv = adv < rem ? adv : rem;
    }
  }
  return adv;
}

// whether this lane's bit is set
__device__ __forceinline__ bool lane_in(uint64_t mask) { return __builtin_amdgcn_inverse_ballot_w64(mask); }

// Rows 1 .. limit of a DP whose row 0 reached row0.  All values but the cells are uniform.
//
// A row runs in one of two forms.  Narrow: the band lies within 64 diagonals, lane l holding diagonal base + l in a
// register, and the row's masks (band, kept range) are single 64-bit scalars; about 75 vector and 50 scalar
// instructions a row.  When the band reaches either end it is moved to the middle by one permute, or, past 52
// diagonals, to LDS.  Wide: chunks of 64 in the LDS ring, WR_GROUP chunks' loads in flight; back to narrow below 40
// diagonals.
// Not inlined: its loops then have the registers to themselves (inlined, a kernel's own values and the N form's
// took 150 and more, or spilled into the rows).  Aligned, so that its loops keep their place in the lines of the
// instruction cache whatever stands before it: moved by words, the same instructions take 23.6 to 24.2 ms for 951 thousand
// extensions in k_process_pairs and 24.5 to 25.0 ms for 150 thousand in k_extend_nodes.  The two words at its start put
// them where neither is slow (23.6 and 24.7; without them 23.9 and 24.8, two words further 23.8 and 24.7).
template <int RING, bool ROWS, bool HASN>
__device__ __attribute__((noinline, aligned(64))) WRows wave_rows(const uint32_t *words_, const uint32_t *nmask_, int64_t a0_, int64_t t0_, uint32_t flags_,
                                                     int32_t m_, int32_t n_, int32_t limit_, int32_t row0_, const int32_t *match_limit_,
                                                     double bmv, double slope_min, uint32_t end_dist_, int32_t *rowm_, int32_t *rowVal_,
                                                     int32_t val_cap_, int32_t max_rows_, int32_t *band_) {
  constexpr int32_t MASK = RING - 1;
  asm volatile("s_nop 0\n\ts_nop 0");
  const int lane = lane_id();
  const uint32_t flags = (uint32_t)uni((int32_t)flags_), end_dist = (uint32_t)uni((int32_t)end_dist_);
  const bool is_forward = flags & WR_FORWARD, store = ROWS && (flags & WR_STORE), partial = flags & WR_PARTIAL;
  const WTails W = make_tails((const uint32_t *)uni64((int64_t)words_), (const uint32_t *)uni64((int64_t)nmask_), uni64(a0_), uni64(t0_),
                              flags & WR_NA, flags & WR_NT);
  const int32_t m = uni(m_), n = uni(n_), limit = uni(limit_), val_cap = uni(val_cap_), max_rows = uni(max_rows_);
  const g_ints match_limit = (g_ints)(int32_t *)uni64((int64_t)match_limit_);
  const g_ints rowm = (g_ints)(int32_t *)uni64((int64_t)rowm_), rowVal = (g_ints)(int32_t *)uni64((int64_t)rowVal_);
  const l_ints band0 = (l_ints)band_;
  WRows o = {};
  int32_t Left = 0, Right = 0, Longest = 0, MSL = 0, MSd = 0, MSe = 0;
  double MaxScore = 0.0;
  int32_t vend = 1;                            // cells stored
  int32_t kept = 1;                            // those of them that were kept
  int32_t mlv = 0;                             // Edit_Match_Limit of 64 rows, one a lane
  int cur = 0;                                 // wide: the buffer of the previous row
  bool narrow = true;
  int32_t base = -32, v = uni(row0_);          // narrow: the previous row, -2 outside its kept range
  uint64_t km = 1ull << 32;                    // narrow: the kept range's lanes
  if (store && lane == 0) {
    rowm[0] = 0;
    rowVal[0] = v << 2;
  }
  v = lane == 32 ? v : -2;
  // Longest / Max_Score after row er, from each lane's first maximum of that row (forward.C:284-306).  With
  // Longest unchanged the score only falls, and MaxScore already holds the earlier row's.
  auto longest = [&](int32_t pv, int32_t pd, int32_t er) {
    const int32_t M = wave_max_dpp(pv);
    if (M > Longest) {
      Longest = M;
      const double Score = (double)M * bmv - (double)er;
      if (Score > MaxScore) {
        uint64_t b = lanes(pv == M);
        int32_t bd = __builtin_amdgcn_readlane(pd, __builtin_ctzll(b));
        for (b &= b - 1; b; b &= b - 1) {
          const int32_t x = __builtin_amdgcn_readlane(pd, __builtin_ctzll(b));
          bd = x < bd ? x : bd;
        }
        MaxScore = Score; MSL = M; MSd = bd; MSe = er;
      }
    }
  };
  // The end of A or T was reached in row e on diagonal rd: branch-point test (forward.C:172-212);
  // -ffp-contract=off keeps the score two roundings.  after: the previous row's cell at rd + 1.
  auto reached = [&](int32_t e, int32_t rd, int32_t rrow, int32_t after) {
    o.cells += (uint32_t)(rd - Left + 1);
    const double Score = (double)rrow * bmv - (double)e;
    const int32_t Tail_Len = rrow - MSL;
    const double slope = (double)(MaxScore - Score) / (double)Tail_Len;
    bool abort_ = false;
    if (partial && (Score < MaxScore)) abort_ = true;
    if (((uint32_t)e > end_dist / 2u) && ((uint32_t)Tail_Len >= end_dist) && (slope >= slope_min))
      abort_ = true;
    o.mte = !abort_;
    o.e = e;
    o.d = (is_forward && rrow == m && 1 + after == rrow && rd < Right) ? rd + 1 : rd;
    o.last = rrow; o.rrow = rrow;
    if (abort_) { o.e = MSe; o.d = MSd; o.rrow = MSL; o.last = -1; }
  };
  for (int32_t e = 1; e <= limit; e++) {
    if ((e & 63) == 0 || e == 1) {
      const int32_t i = (e & ~63) + lane;
      mlv = match_limit[i < limit ? i : limit];
    }
    Left--;
    Right++;
    const int32_t width = Right - Left;
    if (width + 1 > wr_band<RING>() || (store && e >= max_rows)) {
      o.overflow = true;
      return o;
    }
    const int32_t eml = __builtin_amdgcn_readlane(mlv, e & 63);
    o.rows++;
    if (store && lane == 0) rowm[e] = vend - Left;
    o.end = vend + width + 1;
    if (narrow) {
      const uint64_t act = km | km << 1 | km >> 1;
      const int32_t d = base + lane;
      const int32_t x1 = v + 1, x2 = __builtin_amdgcn_update_dpp(-2, v, 0x138, 0xF, 0xF, false);      // wave_shr:1
      const int32_t x3 = __builtin_amdgcn_update_dpp(-2, v, 0x130, 0xF, 0xF, false) + 1;              // wave_shl:1
      const int32_t x12 = x1 > x2 ? x1 : x2;
      const bool on = lane_in(act);
      const int32_t Row = on ? (x12 > x3 ? x12 : x3) : 0, q = on ? Row + d : 0;
      const Words4 wa = words_at(W.wa, W.ra + Row), wt = words_at(W.wt, W.rt + q);
      const int32_t r1 = m - Row, r2 = n - q;
      const int32_t rem = on ? (r1 < r2 ? r1 : r2) : 0;
      const int32_t adv = chunk_slide<HASN>(W, wa, wt, Row, q, rem, base);
      o.lb += (uint32_t)adv;
      o.slots += OIC_WAVE;
      const int32_t r = Row + adv;
      if (store && on) {
        // the traceback's choice (forward.C:44-56): from d unless d - 1 is larger, then d + 1 if larger still
        const int32_t code = x3 > x12 ? 2 : (x2 > x1 ? 1 : 0);
        rowVal[(uint32_t)(vend + (d - Left))] = (r << 2) | code;
      }
      const uint64_t rb = lanes(adv == rem) & act;
      if (rb) {
        const int l = __builtin_ctzll(rb);
        reached(e, base + l, __builtin_amdgcn_readlane(r, l), l < 63 ? __builtin_amdgcn_readlane(v, l + 1) : -2);
        return o;
      }
      o.cells += (uint32_t)(width + 1);
      const uint64_t kb = lanes(r + (d > 0 ? d : 0) >= eml) & act;     // not pruned (forward.C:244-282)
      if (!kb) break;
      const int32_t lo = __builtin_ctzll(kb), hi = 63 - __builtin_clzll(kb);
      km = (~0ull << lo) & (~0ull >> (63 - hi));
      v = lane_in(km) ? r : -2;
      Left = base + lo;
      Right = base + hi;
      longest(v, d, e);
      if (store) {
        kept += hi - lo + 1;
        if (kept > val_cap) { o.overflow = true; return o; }
        vend += width + 1;
      }
      if (lo == 0 || hi == 63) {
        if (hi - lo < 52) {
          const int32_t by = ((lo + hi) >> 1) - 32, i = lane + by;
          const int32_t x = __builtin_amdgcn_ds_bpermute(i << 2, v);
          v = (uint32_t)i < 64u ? x : -2;
          base += by;
          km = by < 0 ? km << -by : km >> by;
        } else {
          const l_ints nb = band0 + cur * (RING + 2);
          const int32_t i = (d + 32) & MASK;
          nb[1 + i] = v;
          if (lane < 4) nb[1 + ((lane + (lane < 2 ? Left - 2 : Right - 1) + 32) & MASK)] = -2;
          wave_order();
          if (lane < 2) nb[lane ? RING + 1 : 0] = nb[lane ? 1 : RING];
          wave_order();
          narrow = false;
        }
      }
      continue;
    }
    const int32_t Lc = (Left + 32) >> 6, Hc = (Right + 32) >> 6;
    const l_ints pb = band0 + cur * (RING + 2);
    const l_ints nb = band0 + (cur ^ 1) * (RING + 2);
    int32_t nL = 0x7fffffff, nR = 0;
    uint64_t any = 0;
    int32_t pv = -2, pd = 0;                   // this lane's first maximum of the previous row
    for (int32_t g = Lc; g <= Hc; g += WR_GROUP) {
      Words4 wa[WR_GROUP], wt[WR_GROUP];
      int32_t rw[WR_GROUP], cd[WR_GROUP];
      // recurrence and loads
#pragma unroll
      for (int i = 0; i < WR_GROUP; i++) {
        const int32_t c = g + i;
        if (c <= Hc) {
          const int32_t d = 64 * c - 32 + lane;
          const l_ints p3 = pb + 64 * (c & (RING / 64 - 1)) + lane;
          const int32_t x2 = p3[0], pc = p3[1], x1 = pc + 1, x3 = p3[2] + 1;
          const bool on = (uint32_t)(d - Left) <= (uint32_t)width;
          const int32_t pm = on ? pc : -2;     // only the band's own cells and the sentinels around it count
          pd = pm > pv ? d : pd;
          pv = pm > pv ? pm : pv;
          const int32_t x12 = x1 > x2 ? x1 : x2;
          if (ROWS) cd[i] = x3 > x12 ? 2 : (x2 > x1 ? 1 : 0);
          const int32_t Row = on ? (x12 > x3 ? x12 : x3) : 0;
          wa[i] = words_at(W.wa, W.ra + Row);
          wt[i] = words_at(W.wt, W.rt + (on ? Row + d : 0));
          rw[i] = Row;
        }
      }
      // slides, reach, prune
#pragma unroll
      for (int i = 0; i < WR_GROUP; i++) {
        const int32_t c = g + i;
        if (c <= Hc) {
          const int32_t d0 = 64 * c - 32, d = d0 + lane, p = rw[i];
          const bool on = (uint32_t)(d - Left) <= (uint32_t)width;
          const int32_t q = on ? p + d : 0, r1 = m - p, r2 = n - q;
          const int32_t rem = on ? (r1 < r2 ? r1 : r2) : 0;
          const int32_t adv = chunk_slide<HASN>(W, wa[i], wt[i], p, q, rem, d0);
          o.lb += (uint32_t)adv;
          const int32_t r = p + adv;
          if (on) {
            nb[64 * (c & (RING / 64 - 1)) + lane + 1] = r;
            if (store) rowVal[(uint32_t)(vend + (d - Left))] = (r << 2) | cd[i];
          }
          any |= lanes(on && adv == rem);
          const uint64_t kb = lanes(on && r + (d > 0 ? d : 0) >= eml);   // not pruned (forward.C:244-282)
          if (kb) {
            const int32_t first = d0 + __builtin_ctzll(kb);
            nL = first < nL ? first : nL;
            nR = d0 + 63 - __builtin_clzll(kb);
          }
        }
      }
    }
    wave_order();
    o.slots += (uint32_t)(Hc - Lc + 1) * OIC_WAVE;
    longest(pv, pd, e - 1);
    if (any) {
      // the lowest diagonal that reached an end
      int32_t rd = 0x7fffffff, rrow = 0;
      for (int32_t c = Lc; rd == 0x7fffffff; c++) {
        const int32_t d = 64 * c - 32 + lane, r = nb[64 * (c & (RING / 64 - 1)) + lane + 1];
        const uint64_t b = lanes((uint32_t)(d - Left) <= (uint32_t)width && (r == m || r + d == n));
        if (b) {
          const int l = __builtin_ctzll(b);
          rd = 64 * c - 32 + l;
          rrow = __builtin_amdgcn_readlane(r, l);
        }
      }
      reached(e, rd, rrow, uni(pb[1 + ((rd + 1 + 32) & MASK)]));
      return o;
    }
    o.cells += (uint32_t)(width + 1);
    if (nL == 0x7fffffff) break;
    if (store) {
      kept += nR - nL + 1;
      if (kept > val_cap) { o.overflow = true; return o; }
      vend += width + 1;
    }
    Left = nL;
    Right = nR;
    cur ^= 1;
    if (nR - nL < 40 || e == limit) {
      // narrow again, or the last row: its own maximum now
      int32_t bv = -2, bd = 0;
      base = ((nL + nR) >> 1) - 32;
      if (nR - nL < 40) {
        const int32_t d = base + lane;
        bv = (uint32_t)(d - nL) <= (uint32_t)(nR - nL) ? nb[1 + ((d + 32) & MASK)] : -2;
        bd = d;
        v = bv;
        km = (~0ull << (nL - base)) & (~0ull >> (63 - (nR - base)));
        narrow = true;
      } else {
        for (int32_t d = nL + lane; d <= nR; d += OIC_WAVE) {
          const int32_t x = nb[1 + ((d + 32) & MASK)];
          bd = x > bv ? d : bd;
          bv = x > bv ? x : bv;
        }
      }
      longest(bv, bd, e);
    }
    if (!narrow) {
      // the sentinels of the next row (its band's new ends and the cells past them), and the copies around the ring
      if (lane < 4) nb[1 + ((lane + (lane < 2 ? nL - 2 : nR - 1) + 32) & MASK)] = -2;
      wave_order();
      if (lane < 2) nb[lane ? RING + 1 : 0] = nb[lane ? 1 : RING];
      wave_order();
    }
  }
  // branch point, error limit exhausted or band emptied (forward.C:306-313)
  o.e = MSe; o.d = MSd; o.rrow = MSL; o.last = -1;
  return o;
}

// Run one prefix DP.  All 64 lanes call it with identical arguments; e, A_End and T_End come in the reference's
// convention (negated for reverse).
//   is_forward  : forward() semantics (force-last-error fix-up, Right_Delta) vs reverse()
//   want_delta  : store rows and run Set_*_Delta when the call ends (ROWS; without it sc is not touched)
// A band wider than wr_band, more rows than sc holds or
// more kept cells than its store counts end with out.overflow.  ends_only: no delta for a DP that does not
// reach the end.  sc.rowVal has WR_VAL_SLACK cells beyond val_cap.
template <int RING, bool ROWS>
__device__ __forceinline__ DPOut wave_prefix_dp(const SeqV &A, const int32_t m_, const SeqV &T, const int32_t n_, const int32_t limit_,
                                                      const bool is_forward, const bool want_delta_, const bool ends_only,
                                                      const DPTables &tb, WaveBand<RING> &band, const DPScratch &sc, uint64_t &cells, uint64_t &slots,
                                                      uint64_t &lane_bases, uint32_t &rows) {
  const int lane = lane_id();
  const int32_t m = uni(m_), n = uni(n_), limit = uni(limit_);
  const bool store = ROWS && uni((int32_t)want_delta_) != 0;
  // every view's words are the packed reads
  const bool na = uni(A.nm != nullptr) != 0, nt = uni(T.nm != nullptr) != 0;
  const WTails W = make_tails(A.w, na ? A.nm : T.nm, uni64(A.b0), uni64(T.b0), na, nt);
  const bool has_n = na || nt;
  DPOut out;
  out.overflow = 0;
  out.ndelta = 0;
  out.leftover = 0;
  const int32_t row0 = has_n ? wave_run<true>(W, 0, 0, m) : wave_run<false>(W, 0, 0, m);
  cells += 1;
  slots += 1;
  if (lane == 0) lane_bases += (uint64_t)row0 + 1;
  if (row0 == m) {
    out.e = 0;
    out.a_end = is_forward ? m : -m;
    out.t_end = is_forward ? m : -m;
    out.mte = 1;
    out.leftover = m;
    return out;
  }
  const uint32_t flags = (na ? WR_NA : 0u) | (nt ? WR_NT : 0u) | (is_forward ? WR_FORWARD : 0u) | (store ? WR_STORE : 0u) |
                         (tb.partial ? WR_PARTIAL : 0u);
  const WRows r = has_n ? wave_rows<RING, ROWS, true>(A.w, W.nm, W.a0, W.t0, flags, m, n, limit, row0, tb.match_limit, tb.bmv, tb.slope_min,
                                                      tb.min_branch_end_dist, sc.rowm, sc.rowVal, (int32_t)sc.val_cap, sc.max_rows, band.b[0])
                        : wave_rows<RING, ROWS, false>(A.w, W.nm, W.a0, W.t0, flags, m, n, limit, row0, tb.match_limit, tb.bmv, tb.slope_min,
                                                       tb.min_branch_end_dist, sc.rowm, sc.rowVal, (int32_t)sc.val_cap, sc.max_rows, band.b[0]);
  cells += r.cells;
  slots += r.slots;
  rows += r.rows;
  lane_bases += r.lb;
  if (lane == 0) lane_bases += r.cells;
  out.overflow = r.overflow ? 1 : 0;
  if (r.overflow) return out;
  out.e = r.e;
  out.mte = r.mte ? 1 : 0;
  out.a_end = is_forward ? r.rrow : -r.rrow;
  out.t_end = is_forward ? r.rrow + r.d : -r.rrow - r.d;
  if (store && (r.mte || !ends_only)) {
    __threadfence_block();
    int32_t last = r.last;
    if (last < 0) last = uni(sc.rowVal[uni(sc.rowm[r.e]) + r.d]) >> 2;
    int32_t lo = 0, te = out.t_end;
    out.ndelta = wave_traceback(sc, r.end, r.e, r.d, last, is_forward, &lo, &te, n);
    out.leftover = lo;
    out.t_end = te;
    __threadfence_block();
  }
  return out;
}
