// oic_rounds.h -- Process_Matches in rounds: extensions as independent tasks, pairs resolved from their results.
//
// A pair's extensions follow one another (a dovetail removes every match node on its alignment,
// overlapInCore-Process_String_Overlaps.C:473-490), so with one wavefront per pair the pair with the most
// extensions decides: of 2323 low-error pairs (14 extensions each on average) one runs five times as many,
// and the launch lasts as long as that chain while most of the machine waits.  An extension itself depends on
// nothing but its node.  Here a round has two launches:
//   k_resolve_pairs  takes each open pair through Process_Matches with the results at hand.  A pair that picks a
//                    node without a result is suspended and asks for it, and for the nodes it would pick next, up
//                    to `ahead` in all (speculation: some will be removed before they are picked);
//   k_extend_nodes   runs the asked extensions, one to a wavefront: both tails' DPs with row storage, the
//                    delta, and which of the pair's nodes lie on the alignment, as a bit mask.
// The rounds end when no pair is open.  `ahead` is chosen per round so that the asked extensions fill the
// machine a few times: many when few pairs are open (they would idle it), few when many are.
//
// Results and node masks wait in stores of a limited size (a mask has a bit per node of its pair, so the thousands
// of extensions of one satellite pair need more than any store).  When an ask does not fit, the round's other
// extensions run, one launch of k_resolve_pairs without asking uses what results there are, and the stores start
// again empty; a pair forgets the results that it has not used by then, `ahead` of them at most.  (Rounds that went on
// until the task slots were used up, and then one wavefront for the pair from its start: 1794 extensions of one tandem
// pair 598 ms, 121 launches; so 130 ms, 37.)
#pragma once

#include "oic_batch.h"

struct ExtNode {
  uint32_t pair, node;      // pair NO_PAIR: nothing to run (its arrays were full)
  uint64_t mask;            // first word of its node mask
};
#define NO_PAIR 0xffffffffu

struct ExtRec {
  int32_t kind;             // ExtOut's, or -1: the band outgrew the short rows
  int32_t s_lo, s_hi, t_lo, t_hi, errors, ndelta;
  uint32_t pad;
  uint64_t cells;
};

// a suspended pair
struct PairState {
  OlapDev olap[OIC_MAX_DISTINCT];
  int32_t ct, first;
  PairOut po;
};

struct RoundCount {         // cleared before each round but for `asked`, which runs on until the stores are emptied
  uint32_t queue, nopen, equeue;
  uint32_t full;            // 1: an ask did not fit
  unsigned long long asked; // extensions << ROUND_WORD_BITS | their mask words
};
// One atomic reserves both, so that the first ask of empty stores gets the first places of both and fits.  Asks that do
// not fit count too: those of one launch are at most 64 extensions for each of 2^20 pairs and 64 words for each pair and
// one for each match node (at most one a seed hit, which take over 100 bytes of the device's memory each), so neither
// field overflows.
#define ROUND_WORD_BITS 36

struct RoundArgs {
  ReadsDev R;
  SearchConst C;
  const PairRec *pairs;
  int4 *nodes;
  uint64_t *outc;            // per node: pack_outcome, kind 3 (OUTC_EXT): the extension's index in the low word
  const float *pred;         // the cost model's log(1 + DP cells) per pair (two floats a pair), or nullptr
  const uint32_t *order;     // the pairs of these rounds
  const uint32_t *list;      // their open ones, n places in order[], or nullptr: all n of them; those still open
  uint32_t n;                // afterwards go to open[]
  uint32_t *open;
  int resume;                // 0: the first round
  int32_t ahead;             // extensions a pair may ask for at once; 0: none, and results not used now are forgotten
  PairState *state;          // per place in order[]
  ExtNode *tasks;
  ExtRec *recs;
  uint64_t *masks;
  uint32_t task_cap, task0, task1;   // [task0, task1): k_extend_nodes' tasks of this round
  uint64_t word_cap;         // both at least 64; word_cap at least a mask of the pair with the most nodes
  RoundCount *cnt;
  OutRec *out;
  PairOut *pout;
  unsigned long long *stats;
  DPScratch sc0;
  int64_t row_stride, val_stride, delta_stride;
};

#define OUTC_EXT 3

// One open pair per wavefront at a time, as k_process_pairs, which this follows statement for statement but for
// where an extension's result comes from.
__global__ void __launch_bounds__(OIC_WAVE) k_resolve_pairs(RoundArgs A) {
  __shared__ PairState st;
  __shared__ PairStats pst;
  const int lane = lane_id();
  const SearchConst &C = A.C;
  uint64_t cells = 0, exts = 0;
  clear_pair_stats(pst);
  // a pair each, the most expensive ones, then four at a time from the queue
  uint32_t qi = blockIdx.x, qend = qi + 1;
  for (;; qi++) {
    if (qi == qend) {
      uint32_t f = 0;
      if (lane == 0) f = atomicAdd(&A.cnt->queue, 4u);
      qi = gridDim.x + (uint32_t)uni((int32_t)f);
      qend = qi + 4;
    }
    if (qi >= A.n) break;
    const uint32_t at = A.list ? A.list[qi] : qi, p = A.order[at];
    const PairRec pr = A.pairs[p];
    int4 *nodes = A.nodes + pr.hb;
    uint64_t *outc = A.outc + pr.hb;
    const int32_t nn = uni(pr.nnodes);
    const uint32_t S_ID = pr.s_id, T_ID = pr.t_id;
    const int32_t S_Len = A.R.len[S_ID], T_Len = A.R.len[T_ID];
    PairOut po = {};
    bool first = true;
    __syncthreads();
    if (A.resume) {
      const uint32_t *src = (const uint32_t *)(A.state + at);
      for (int i = lane; i < (int)(sizeof(PairState) / 4); i += OIC_WAVE) ((uint32_t *)&st)[i] = src[i];
      __syncthreads();
      po = st.po;
      first = st.first != 0;
    } else {
      // --minkmers filter (Process_String_Overlaps.C:618-621)
      if (C.min_kmers) {
        const uint64_t mk = C.min_kmers[pr.diag_end - pr.diag_bgn];
        if (mk > (uint64_t)(int64_t)(pr.he - pr.hb)) {
          if (lane == 0) { po.status = 3; A.pout[p] = po; }
          continue;
        }
      }
      if (hopeless_pair(C, pr, nodes, nn, S_Len, T_Len)) {
        if (lane == 0) {
          po.status = 2;
          A.pout[p] = po;
          pst.n[STAT_WITHOUT]++;
        }
        continue;
      }
      if (lane == 0) st.ct = 0;
      __syncthreads();
    }
    bool suspended = false, overflow = false;
    while (true) {
      // first node with the maximal Len (Process_String_Overlaps.C:424-431)
      int32_t bl = -1, bi = 0x7fffffff;
      for (int32_t i = lane; i < nn; i += OIC_WAVE) {
        const int4 nd = nodes[i];
        if (!nd.w && nd.y > bl) { bl = nd.y; bi = i; }
      }
      wave_pick(bl, bi);
      if (bl < 0) break;
      const uint64_t bo = outc[bi];
      const int kind = uni(outcome_kind(bo));
      if (kind == 1) {
        // known not to be a dovetail: removed, with all such nodes that would be picked before any other
        uint64_t cnt = 0, cs = 0;
        if (pr.consistent) {
          if (lane == 0) { cnt = 1; cs = outcome_cells(bo); nodes[bi].w = 1; }
        } else {
          int32_t ul = -1, ui = 0x7fffffff;
          for (int32_t i = lane; i < nn; i += OIC_WAVE) {
            const int4 nd = nodes[i];
            if (!nd.w && outcome_kind(outc[i]) != 1 && nd.y > ul) { ul = nd.y; ui = i; }
          }
          wave_pick(ul, ui);
          for (int32_t i = lane; i < nn; i += OIC_WAVE) {
            const int4 nd = nodes[i];
            const uint64_t oi = outc[i];
            if (!nd.w && outcome_kind(oi) == 1 && (nd.y > ul || (nd.y == ul && i < ui))) {
              nodes[i].w = 1;
              cnt++;
              cs += outcome_cells(oi);
            }
          }
        }
        for (int o = 32; o > 0; o >>= 1) { cnt += __shfl_xor(cnt, o); cs += __shfl_xor(cs, o); }
        po.n_ext += (int32_t)cnt;
        po.cells += cs;
        if (first) { po.exit_d = outcome_exit(bo); first = false; }
        __threadfence_block();
        if (pr.consistent) break;
        continue;
      }
      if (kind != OUTC_EXT && A.ahead == 0) {
        for (int32_t i = lane; i < nn; i += OIC_WAVE)
          if (outcome_kind(outc[i]) == OUTC_EXT) outc[i] = 0;
        suspended = true;
        break;
      }
      if (kind != OUTC_EXT) {
        // ask for this node's extension and for the next ones in picking order
        int32_t want = pr.consistent ? 1 : A.ahead;
        if (A.pred && want > 1) {
          // No more than the cost model expects, its cells still to come over those of an extension so far, but half of
          // what the pair may ask for at the least, and no limit once it has used up what the model expected.  (Down to
          // one, and one for each round from there on: 900 low-error reads 43.7 ms in 42 rounds, 2500 compressed reads
          // 1605 ms in 827; so 23.1 ms in 8 and 1323 in 178, as without a model, with 4 % fewer extensions of the first.)
          const float left = expm1f(A.pred[2 * (uint64_t)p]) - (float)po.cells;
          const float each = po.n_ext > 0 ? (float)po.cells / (float)po.n_ext : (float)outcome_cells(bo);
          const float k = each > 0.f ? left / each : 1.f;
          const int32_t least = want / 2;
          if (left > 0.f && k < (float)want) want = k > (float)least ? (int32_t)k : least;
        }
        want = uni(want);
        int32_t have = 0;
        for (int32_t i0 = 0; i0 < nn; i0 += OIC_WAVE) {
          const int32_t i = i0 + lane;
          const bool c = i < nn && !nodes[i].w && (outcome_kind(outc[i]) & 1) == 0;
          have += (int32_t)__builtin_popcountll(lanes(c));
        }
        const uint32_t nw = (uint32_t)(nn + 63) / 64;
        const uint64_t room = A.word_cap / nw;
        if (room < (uint64_t)want) want = (int32_t)room;
        const int32_t cnt = have < want ? have : want;
        unsigned long long before = 0;
        if (lane == 0) before = atomicAdd(&A.cnt->asked, ((unsigned long long)cnt << ROUND_WORD_BITS) + (unsigned long long)cnt * nw);
        before = (unsigned long long)uni64((int64_t)before);
        const uint32_t slot = (uint32_t)(before >> ROUND_WORD_BITS);
        const uint64_t word = before & ((1ull << ROUND_WORD_BITS) - 1);
        const bool fits = (uint64_t)slot + cnt <= A.task_cap && word + (uint64_t)cnt * nw <= A.word_cap;
        if (!fits) {
          if (lane == 0) A.cnt->full = 1;
          for (int32_t j = lane; j < cnt; j += OIC_WAVE)
            if ((uint64_t)slot + j < A.task_cap) A.tasks[slot + j].pair = NO_PAIR;
        } else if (cnt == have) {
          int32_t k = 0;
          for (int32_t i0 = 0; i0 < nn; i0 += OIC_WAVE) {
            const int32_t i = i0 + lane;
            const bool c = i < nn && !nodes[i].w && (outcome_kind(outc[i]) & 1) == 0;
            const uint64_t b = lanes(c);
            const int32_t j = k + (int32_t)__builtin_popcountll(b & ((1ull << lane) - 1));
            if (c) {
              A.tasks[slot + j] = ExtNode{p, (uint32_t)i, word + (uint64_t)j * nw};
              outc[i] = pack_outcome(OUTC_EXT, 0, slot + (uint32_t)j);
            }
            k += (int32_t)__builtin_popcountll(b);
          }
        } else {
          for (int32_t j = 0; j < cnt; j++) {
            int32_t ml = -1, mi = 0x7fffffff;
            for (int32_t i = lane; i < nn; i += OIC_WAVE) {
              const int4 nd = nodes[i];
              if (!nd.w && nd.y > ml && (outcome_kind(outc[i]) & 1) == 0) { ml = nd.y; mi = i; }
            }
            wave_pick(ml, mi);
            if (lane == 0) {
              A.tasks[slot + j] = ExtNode{p, (uint32_t)mi, word + (uint64_t)j * nw};
              outc[mi] = pack_outcome(OUTC_EXT, 0, slot + (uint32_t)j);
            }
            __threadfence_block();
          }
        }
        suspended = true;
        break;
      }
      const uint32_t ti = outcome_cells(bo);
      const ExtRec x = A.recs[ti];
      if (uni(x.kind) < 0) { overflow = true; break; }
      po.n_ext++;
      po.cells += x.cells;
      if (first) { po.exit_d = x.t_hi - x.s_hi; first = false; }
      if (x.kind == 3 || C.partial) {
        if (1 + x.s_hi - x.s_lo >= C.min_olap && 1 + x.t_hi - x.t_lo >= C.min_olap) {
          const int32_t a = x.s_hi - x.s_lo, b = x.t_hi - x.t_lo;
          const int32_t olen = 1 + (a < b ? a : b);
          const double q = (double)x.errors / (double)olen;
          if (x.errors <= C.tb.error_bound[olen]) {
            if (lane == 0) add_overlap(C, x.s_lo, x.s_hi, x.t_lo, x.t_hi, q, x.ndelta, st.olap, &st.ct);
          }
        }
      }
      if (pr.consistent) break;
      // remove the longest match and, after a dovetail, every match on the alignment (:476-490)
      if (lane == 0) nodes[bi].w = 1;
      if (x.kind == 3 || C.partial) {
        const uint64_t *mask = A.masks + A.tasks[ti].mask;
        for (int32_t i = lane; i < nn; i += OIC_WAVE)
          if ((mask[i >> 6] >> (i & 63)) & 1) nodes[i].w = 1;
      }
      __threadfence_block();
    }
    __syncthreads();
    if (suspended) {
      if (lane == 0) {
        st.po = po;
        st.first = first ? 1 : 0;
        A.open[atomicAdd(&A.cnt->nopen, 1u)] = at;
      }
      __syncthreads();
      uint32_t *dst = (uint32_t *)(A.state + at);
      for (int i = lane; i < (int)(sizeof(PairState) / 4); i += OIC_WAVE) dst[i] = ((const uint32_t *)&st)[i];
      continue;
    }
    if (overflow) {
      // the wide-band rerun takes the pair from its start
      for (int32_t i = lane; i < nn; i += OIC_WAVE) nodes[i].w = 0;
      if (lane == 0) { po = PairOut{}; po.status = 1; A.pout[p] = po; }
      continue;
    }
    exts += (uint64_t)po.n_ext;
    cells += po.cells;
    if (lane == 0) finish_pair(C, pr, S_Len, T_Len, st.olap, st.ct, po, A.out + (uint64_t)p * OIC_MAX_DISTINCT, A.pout + p, pst);
  }
  __syncthreads();
  add_pair_stats(pst, A.stats);
  if (lane == 0 && exts) {
    atomicAdd(&A.stats[STAT_CELLS], (unsigned long long)cells);
    atomicAdd(&A.stats[STAT_EXT], (unsigned long long)exts);
  }
}

__global__ void __launch_bounds__(OIC_WAVE) __attribute__((amdgpu_waves_per_eu(4, 8))) k_extend_nodes(RoundArgs A) {
  __shared__ WaveBand<WR_FIRST> band;
  const int lane = lane_id();
  const SearchConst &C = A.C;
  DPScratch sc = A.sc0;
  sc.rowm += (int64_t)blockIdx.x * A.row_stride;
  sc.rowVal += (int64_t)blockIdx.x * A.val_stride;
  sc.dbuf += (int64_t)blockIdx.x * A.delta_stride;
  sc.ldelta += (int64_t)blockIdx.x * A.delta_stride;
  sc.rdelta += (int64_t)blockIdx.x * A.delta_stride;
  uint64_t cells_acc = 0, slots = 0, bases = 0;
  uint32_t calls = 0, ran = 0;
  while (true) {
    uint32_t f = 0;
    if (lane == 0) f = atomicAdd(&A.cnt->equeue, 1u);
    const uint32_t ti = A.task0 + (uint32_t)uni((int32_t)f);
    if (ti >= A.task1) break;
    const ExtNode tk = A.tasks[ti];
    if (tk.pair == NO_PAIR) continue;
    const PairRec pr = A.pairs[tk.pair];
    const int4 *nodes = A.nodes + pr.hb;
    const int4 nd = nodes[tk.node];
    const SeqV S = read_view(A.R, pr.s_id, pr.dir), Src = read_view(A.R, pr.s_id, 1 - pr.dir);
    const SeqV T = read_view(A.R, pr.t_id, 0), Trc = read_view(A.R, pr.t_id, 1);
    uint64_t cells = 0;
    const ExtOut x = wave_extend<WR_FIRST>(nd.z, nd.x, nd.y, S, Src, A.R.len[pr.s_id], T, Trc, A.R.len[pr.t_id], C, band, sc,
                                      cells, slots, calls, bases, true);
    if (lane == 0) {
      ExtRec r;
      r.kind = x.overflow ? -1 : x.kind;
      r.s_lo = x.s_lo; r.s_hi = x.s_hi; r.t_lo = x.t_lo; r.t_hi = x.t_hi;
      r.errors = x.errors; r.ndelta = x.ndelta; r.pad = 0; r.cells = cells;
      A.recs[ti] = r;
    }
    cells_acc += cells;
    ran++;
    if (x.overflow || pr.consistent || !(x.kind == 3 || C.partial)) continue;
    // the pair's nodes on this alignment (:476-490)
    const int32_t nn = uni(pr.nnodes);
    const int32_t gl = alignment_runs(x.s_lo, x.t_lo, sc.ldelta, x.ndelta, sc.dbuf, sc.rdelta);
    __threadfence_block();
    uint64_t *mask = A.masks + tk.mask;
    for (int32_t i0 = 0; i0 < nn; i0 += OIC_WAVE) {
      const int32_t i = i0 + lane;
      bool on = false;
      if (i < nn) {
        const int4 x2 = nodes[i];
        on = x.s_lo - OIC_SHIFT_SLACK <= x2.z && x2.z + x2.y <= (x.s_hi + 1) + OIC_SHIFT_SLACK - 1 &&
             lies_on_runs(x2.z, x2.x, sc.dbuf, sc.rdelta, x.ndelta, gl);
      }
      const uint64_t b = lanes(on);
      if (lane == 0) mask[i0 >> 6] = b;
    }
  }
  for (int o = 32; o > 0; o >>= 1) bases += __shfl_xor(bases, o);
  if (lane == 0) {
    atomicAdd(&A.stats[STAT_BASES], (unsigned long long)bases);
    atomicAdd(&A.stats[STAT_PPCELLS], (unsigned long long)cells_acc);
    atomicAdd(&A.stats[STAT_SLOTS], (unsigned long long)slots);
    atomicAdd(&A.stats[STAT_DPCALLS], (unsigned long long)calls);
    atomicAdd(&A.stats[STAT_AHEAD], (unsigned long long)ran);
  }
}
