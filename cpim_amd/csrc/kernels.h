// Propagation kernels: model build, grid-wide constraint-frontier fixpoint
// (plain and persistent), and the workgroup engine (domains in LDS) used by
// block-mode GAC, batched singleton tests, the device MAC, batches of
// instances and the serving step.
#pragma once

#include "device.h"

// ===========================================================================
// Model build: dense rows -> word-major support planes (both directions).
// One wave per (binary constraint k, word w): lanes are the 64 values
// a = 64 w + lane of scope[0]; plane 0 is a transpose of word indices, plane 1
// a bit transpose done with one ballot per value b of scope[1].
// ===========================================================================
__global__ void k_build_planes(const u64* __restrict__ rel, int nb, int max_dom, int rel_words,
                               int W, int dpad, const int* __restrict__ bin_cons,
                               const ConMeta* __restrict__ con, const int* __restrict__ cap,
                               u64* __restrict__ sup) {
  const int lane = lane_id();
  const long long wave = ((long long)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  if (wave >= (long long)nb * W) return;
  const int k = (int)(wave / W);
  const int w = (int)(wave % W);
  const int c = bin_cons[k];
  const ConMeta m = con[c];
  const int cx = cap[m.scope[0]], cy = cap[m.scope[1]];
  u64* plane0 = sup + m.off;
  u64* plane1 = plane0 + (long long)W * dpad;
  const u64* rows = rel + (long long)k * max_dom * rel_words;
  // plane 0: element (w, a) = word w of row a, masked to y's capacity
  const int ybits = cy - 64 * w;
  const u64 ymask = ybits >= 64 ? ~0ull : (ybits <= 0 ? 0ull : ((1ull << ybits) - 1ull));
  for (int a0 = 0; a0 < dpad; a0 += 64) {
    const int a = a0 + lane;
    u64 v = 0ull;
    if (a < cx && w < rel_words) v = rows[(long long)a * rel_words + w] & ymask;
    plane0[(long long)w * dpad + a] = v;
  }
  // plane 1: element (w, b) = bits a in [64w, 64w+64) with (a, b) allowed
  const int a = 64 * w + lane;
  u64 acc = 0ull;
  for (int j = 0; j < W; ++j) {
    const u64 rowword = (a < cx && j < rel_words) ? rows[(long long)a * rel_words + j] : 0ull;
    for (int bb = 0; bb < 64; ++bb) {
      const int b = 64 * j + bb;
      const bool bit = b < cy && ((rowword >> bb) & 1ull);
      const u64 word = __ballot(bit);
      if (lane == bb) acc = word;
    }
    plane1[(long long)w * dpad + 64 * j + lane] = acc;
  }
}

// Domain word seen by a lane: agent scope (other XCDs' completed updates), or
// workgroup scope (LDS, or global memory that nobody writes meanwhile or whose
// stale words only keep too much).
template <bool kCoherent>
__device__ __forceinline__ u64 ld_view(const u64* p) {
  if constexpr (kCoherent) return __hip_atomic_load(const_cast<u64*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else return ld_wg(p);
}

// Open values of some lanes, settled by the whole wave: for each lane with
// todo, the 64 lanes take the values of its word one each and read the words
// of their rows (own: index in sup of the row words of the word's first value)
// against D(src), one word after the other while some value is open: the
// first word of a row is a coalesced 512-byte read and settles most values.
// kSettle arc words at a time.  Returns, in the lanes with todo, the values of
// `need` without a support; `need` unchanged in the others.
constexpr int kSettle = 8;

template <bool kCoherent>
__device__ __forceinline__ u64 wave_settle(const DevNet& net, const u64* dom, long long own, int src, u64 need,
                                           u64 todo) {
  const int W = net.W, lane = lane_id();
  while (todo) {
    int l[kSettle];
    u64 open[kSettle];
#pragma unroll
    for (int p = 0; p < kSettle; ++p) {
      l[p] = uniform_int(todo ? (int)__builtin_ctzll(todo) : l[0]);
      open[p] = todo ? readlane64(need, l[p]) : 0ull;
      todo &= todo - 1ull;
    }
    for (int j = 0; j < W; ++j) {
      u64 r[kSettle], d[kSettle], any = 0ull;
#pragma unroll
      for (int p = 0; p < kSettle; ++p) {
        const u64* row = net.sup + (long long)readlane64((u64)own, l[p]) + (long long)j * net.dpad;
        r[p] = (open[p] >> lane) & 1ull ? row[lane] : 0ull;
        d[p] = ld_view<kCoherent>(&dom[(long long)__builtin_amdgcn_readlane(src, l[p]) * W + j]);
      }
#pragma unroll
      for (int p = 0; p < kSettle; ++p) {
        open[p] &= ~__ballot((r[p] & d[p]) != 0ull);
        any |= open[p];
      }
      if (any == 0ull) break;
    }
#pragma unroll
    for (int p = kSettle - 1; p >= 0; --p)
      if (lane == l[p]) need = open[p];
  }
  return need;
}

// The values of `need` (word w of D(tgt)) without a support in D(src), for the
// constraint whose planes start at off: one arc word per lane, each with its
// own source; lanes without an arc pass need = 0.  Called by whole waves.
// Source side: the rows of four values of src at a time are ORed, and the
// values of tgt they cover are settled; a value stays open with the product of
// four tightnesses, so a few such steps settle nearly every value of a loose
// relation.  Target side: an open value is settled by the W words of its own
// row, by the lane, four reads a step.  Lanes that tight relations leave with
// more than 12 steps per four words of a domain are settled by the wave, one
// after the other (wave_settle; kTight: the searches take that path only on
// networks of wide domains and many constraints).  One-word domains get there
// with at least 57 values against 49 open ones; by the lane n=2000 d=64 e=1500
// t=0.97 takes 131 us persistent, so 122, and n=200 e=150 t=0.985 36 and 33.
template <bool kCoherent, bool kTight>
__device__ __forceinline__ u64 arcs_unsupported(const DevNet& net, const u64* dom, long long off, int src, int pos_src,
                                                int w, u64 need) {
  const int W = net.W, dpad = net.dpad;
  const long long own = off + (long long)(1 - pos_src) * W * dpad + 64 * w;
  const u64* ds = dom + (long long)src * W;
  bool wave = false;
  if (need) {
    const u64* rows = net.sup + off + (long long)(pos_src * W + w) * dpad;
    u64 x = ld_view<kCoherent>(&ds[0]);
    int left = __popcll(x);
    for (int j = 1; j < W; ++j) left += __popcll(ld_view<kCoherent>(&ds[j]));
    int j = 0, done = 0, ts = 0;
    while (need && left > 0) {
      ts = (__popcll(need) * W + 3) >> 2;
      if (left > 4 * ts && (ts <= 1 || done >= 3)) break;
      if (kTight && done >= 2 && min(left, 4 * ts) > 48 * ((W + 3) >> 2)) {
        wave = true;
        break;
      }
      u64 r[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        while (x == 0ull && j + 1 < W) x = ld_view<kCoherent>(&ds[++j]);
        const int a = x ? (int)__builtin_ctzll(x) : 0;
        r[i] = x ? rows[64 * j + a] : 0ull;
        x &= x - 1ull;
      }
      need &= ~((r[0] | r[1]) | (r[2] | r[3]));
      left -= 4;
      ++done;
    }
    if (!wave && left > 0) {  // the target side, by the lane
      const u64* mine = net.sup + own;
      u64 open = need;
      if (W == 1) {
        const u64 d = ld_view<kCoherent>(&ds[0]);
        while (open) {
          u64 r[4], bit[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            bit[i] = open & (0ull - open);
            r[i] = open ? mine[__builtin_ctzll(open)] : 0ull;
            open &= open - 1ull;
          }
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (r[i] & d) need &= ~bit[i];
        }
      }
      while (open) {
        const int b = (int)__builtin_ctzll(open);
        bool ok = false;
        for (int j0 = 0; j0 < W && !ok; j0 += 4) {
          u64 r[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) r[i] = j0 + i < W ? mine[(long long)(j0 + i) * dpad + b] : 0ull;
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (j0 + i < W) ok = ok || (r[i] & ld_view<kCoherent>(&ds[j0 + i])) != 0ull;
        }
        if (ok) need &= ~(1ull << b);
        open &= open - 1ull;
      }
    }
  }
  if (!kTight) return need;
  const u64 todo = __ballot(wave);
  return todo ? wave_settle<kCoherent>(net, dom, own, src, need, todo) : need;
}

// ===========================================================================
// Grid engine: rounds over a bitmap of the variables that changed.
// In round r a lane takes one word of one arc u <- t of the adjacency list,
// if t changed in round r - 1.  A fixpoint seeded with one variable may start
// from a level that is not at its closure, and then reaches less than the
// whole closure: as a frontier of constraints does (`pairs`: u <- t also if u
// changed), or as one of variables does.  Three bitmaps rotate: F[r % 3] is read,
// F[(r + 1) % 3] collects the round's changes, F[(r + 2) % 3] (read in round
// r - 1) is cleared.  last_push_round only grows and wipe_round is only
// lowered to the running round, so every block takes the same decision after
// a barrier.
//
// A round is bound by its chain of dependent reads (changed bit, domains,
// rows, removal), a full one by the rows' bandwidth.  The earlier rounds kept
// a frontier of constraints, each revised in both directions by a wave that
// read 64 rows of either side, and every removal marked all constraints of its
// variable.  Kernel time, before and after (host-driven rounds): n=2000 d=64
// e=40000, one round without removals 30 -> 7.2 us; its cascade at t=0.886
// (10 rounds, 6,485 removals) 255 -> 160 us, persistent 318 -> 158 us; n=500
// d=250 e=20000 t=0.963 (5 rounds) 314 -> 197 us, persistent 372 -> 183 us.
// ===========================================================================
// Outcome of a fixpoint (or of one of its host-driven rounds).
struct GacResult {
  int rounds;           // rounds executed (persistent, one workgroup)
  int converged;
  int err;              // the launch's time budget ran out
  int last_push_round;  // as in GacCtl
  int wipe_round;       // INT_MAX: no wipe-out
  int pad;
  unsigned long long deletions, revisions;
  unsigned long long ticks;  // device clock ticks of the launch
};

// Pinned host memory a kernel answers in, so that a call costs one launch and
// no copies: the kernel stores its result there (system-scope stores, which go
// through to host memory), waits until they have completed, and stores the
// call's number in `seq`, on which the host waits.
struct HostBox {
  unsigned long long seq;  // the last call answered
  int scalar;
  int pad;
  GacResult gac;
  alignas(64) unsigned long long issued;  // the last call numbered: the host's, on a line of its own
  alignas(64) unsigned long long data[1];  // kBoxDataBytes
};

__device__ __forceinline__ void box_store(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ void box_store(int* p, int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ __forceinline__ void wait_memory_ops() {
  // vmcnt(0); expcnt and lgkmcnt left at their maxima (no wait)
  __builtin_amdgcn_s_waitcnt(0x0F70);
}

// Ends a call: every thread of the (single or last) workgroup calls it.
__device__ __forceinline__ void box_publish(unsigned long long* seq_at, unsigned long long seq) {
  wait_memory_ops();
  __syncthreads();
  if (threadIdx.x == 0 && seq_at) box_store(seq_at, seq);
}

__device__ __forceinline__ void store_result(GacResult* out, int rounds, int converged, int err, int lp, int wipe,
                                             unsigned long long dels, unsigned long long revs,
                                             unsigned long long ticks) {
  box_store(&out->rounds, rounds);
  box_store(&out->converged, converged);
  box_store(&out->err, err);
  box_store(&out->last_push_round, lp);
  box_store(&out->wipe_round, wipe);
  box_store(&out->deletions, dels);
  box_store(&out->revisions, revs);
  box_store(&out->ticks, ticks);
}

// Statistics counters are spread over kStatSlots addresses (by block), and
// the grid rounds add one workgroup total per round: device-scope atomics on
// one address serialize, and one from every wave of an 8,192-wave round on
// 32 addresses took 80 of the 100 us of a C2 round.
constexpr int kStatSlots = 256;

struct GacCtl {
  int last_push_round;  // highest round that changed a domain (host-driven rounds)
  int wipe_round;       // lowest round that emptied a domain
  unsigned long long bar_ticket;  // grid barrier arrivals so far (only grows)
  int err;              // set by a block whose barrier wait ran out of time
  unsigned done;        // blocks of the running launch that finished
  unsigned long long start;  // device clock at the start of the launch
  unsigned long long deletions[kStatSlots];
  unsigned long long revisions[kStatSlots];
};

__device__ __forceinline__ int ld_agent(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One word of one arc per lane (lanes with act false do nothing).  view: the
// domains as the lane reads them (global memory, or the round's copy in LDS);
// removals go to dom.  W = 1: the word returned by the AND tells the wipe-out,
// so the size update needs no answer.
template <bool kCoherent>
__device__ __forceinline__ void grid_arc(const DevNet& net, const u64* view, u64* dom, int* size, unsigned* nxt,
                                         GacCtl* ctl, int r, const int4& e, int w, bool act, int& dels) {
  const int W = net.W, u = e.y;
  const u64 need = act ? ld_view<kCoherent>(&view[(long long)u * W + w]) : 0ull;
  const u64 gone = arcs_unsupported<kCoherent, true>(net, view, act ? e.w * (2ll * W * net.dpad) : 0ll, adj_var(e), adj_pos(e),
                                               act ? w : 0, need);
  if (gone == 0ull) return;
  const u64 old = atomicAnd(&dom[(long long)u * W + w], ~gone);
  const int lost = __popcll(old & gone);
  if (lost == 0) return;
  dels += lost;
  atomicOr(&nxt[u >> 5], 1u << (u & 31));
  bool wiped;
  if (W == 1) {
    wiped = (old & ~gone) == 0ull;
    (void)__hip_atomic_fetch_add(&size[u], -lost, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else {
    wiped = atomicSub(&size[u], lost) == lost;
  }
  if (wiped) atomicMin(&ctl->wipe_round, r);
}

// The arcs and tables of round r that this grid's waves take.  cur: the
// variables that changed (round 0: seed < 0 takes every arc and table, else
// those on variable `seed`, in both directions); pairs: later rounds take the
// changed variables' constraints in both directions too; e0: the arc of this lane's
// first turn, kept in registers by the persistent kernel (kept true).  With
// several words a wave's arcs lie nwaves apart in the list, so that the arcs
// of one variable (a late round's few changes) fall to as many waves: what
// they settle together, wave_settle does one after the other.  One-word arcs
// stay in list order, 64 neighbours to a wave (a 10-round cascade of 80,000
// arcs 162 us against 187 us spread).
template <bool kCoherent>
__device__ __forceinline__ void grid_round(const DevNet& net, const u64* view, u64* dom, int* size,
                                           const unsigned* cur, unsigned* nxt, GacCtl* ctl, int r, int seed,
                                           bool pairs, bool kept, const int4& e0, int narcs, int& revs, int& dels) {
  const int W = net.W, lane = lane_id();
  int lw = 0;
  while ((1 << lw) < W) ++lw;
  const int w = lane & ((1 << lw) - 1);
  const int nwaves = (int)(((long long)gridDim.x * blockDim.x) >> 6);
  const int gw = uniform_int((int)(((long long)blockIdx.x * blockDim.x + threadIdx.x) >> 6));
  auto changed = [&](int v) -> bool {
    const unsigned* p = &cur[v >> 5];
    const unsigned word = kCoherent ? (unsigned)ld_agent((const int*)p) : *p;
    return (word >> (v & 31)) & 1u;
  };
  // whole waves: lanes past the end take no arc
  const int4 none = make_int4(0, -1, 0, 0);
  const long long per_pass = (long long)nwaves << (6 - lw);
  for (long long base = 0; base < narcs; base += per_pass) {
    const long long i = base + (W > 1 ? (long long)(lane >> lw) * nwaves + gw : (long long)gw * 64 + lane);
    const int4 e = kept && base == 0 ? e0 : (i < narcs ? net.adj[i] : none);
    const int t = adj_var(e), u = e.y;
    const bool act =
        u >= 0 && w < W && (r > 0 ? changed(t) || (pairs && changed(u)) : (seed < 0 || t == seed || u == seed));
    const u64 m = __ballot(act && w == 0);
    if (__ballot(act) == 0ull) continue;
    revs += __popcll(m);
    grid_arc<kCoherent>(net, view, dom, size, nxt, ctl, r, e, w, act, dels);
  }
  // tables, one per wave, over the workgroups in turn, their last waves first
  const int wib = uniform_int(threadIdx.x >> 6), wpb = (int)(blockDim.x >> 6), nb = (int)gridDim.x;
  for (int k = (wpb - 1 - wib) * nb + nb - 1 - (int)blockIdx.x; k < net.ntabs; k += nwaves) {
    const int c = uniform_int(net.tabs[k]);
    const ConMeta* mp = net.con + c;
    const int y = lane < mp->arity ? mp->scope[lane] : -1;
    const u64 some = __ballot(y >= 0 && (r > 0 ? changed(y) : (seed < 0 || y == seed)));
    if (some == 0ull) continue;
    // one changed variable of a frontier of variables: its own position stays
    int skip = -1;
    if (!pairs && seed >= 0 && r > 0 && (some & (some - 1ull)) == 0ull)
      skip = __builtin_amdgcn_readlane(y, (int)__builtin_ctzll(some));
    bool wiped = false;
    auto on_removed = [&](int v, int n) {
      if (lane == 0) {
        dels += n;
        atomicOr(&nxt[v >> 5], 1u << (v & 31));
      }
    };
    revise_table<decltype(on_removed), true>(net, dom, size, c, skip, nullptr, on_removed, &wiped);
    ++revs;
    if (wiped && lane == 0) atomicMin(&ctl->wipe_round, r);
  }
}

// Binary constraints over one-word domains (W = 1), up to kAsyncPairBatch at a
// time, by one wave.  Both arcs of a constraint c = (x, y) are revised from
// the same D(x) and D(y): value a of x keeps iff row a of plane 0 meets D(y),
// value b of y keeps iff row b of plane 1 meets D(x).  With W = 1 the rows of
// every value are loaded whatever the domains, so the domain words (lane 2p:
// x of constraint p, lane 2p + 1: its y) and the 2 x 64 row words of every
// constraint of the batch are loaded together, one memory round trip for the
// batch.  Revising an arc from a domain that the other arc shrinks in the
// same step is a chaotic-iteration step like any other: the shrunk variable
// is pushed, so c is revised again in the next round, and the closure is the
// same.  The removal masks are applied with atomic AND by lanes 2p / 2p + 1;
// for a one-word domain the returned word gives the exact removals and the
// wipe-out (a non-empty word this AND empties), so the size update needs no
// returned value.
// Eight at a time: the asynchronous fixpoint's waves are few (two per CU) and
// bound by the latency of their own loads, so more rows in flight per wave
// pay (3.6-3.75 ms against 3.85-4.1 ms at four on the C2 cascade).
constexpr int kAsyncPairBatch = 8;

// The revisions of one batch; returns the mask of lanes whose variable (in
// myv) lost values, the values removed in the batch, and whether some domain
// was emptied by it.
template <bool kCoherent, int P = kAsyncPairBatch>
__device__ __forceinline__ u64 revise_pairs_w1(const DevNet& net, u64* dom, int* size, const int (&cs)[P],
                                               int k, int& myv, int& removed_total, bool& wiped_any) {
  const int lane = lane_id();
  int xs[P], ys[P];
  long long offs[P];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const ConMeta* mp = net.con + (p < k ? cs[p] : cs[0]);
    xs[p] = mp->scope[0];
    ys[p] = mp->scope[1];
    offs[p] = mp->off;
  }
  // lane 2p: D(x_p), lane 2p + 1: D(y_p)
  myv = -1;
#pragma unroll
  for (int p = 0; p < P; ++p) {
    if (p < k && lane == 2 * p) myv = xs[p];
    if (p < k && lane == 2 * p + 1) myv = ys[p];
  }
  const u64 dl = myv >= 0 ? ld_dom<kCoherent>(&dom[myv]) : 0ull;
  u64 r0[P], r1[P];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const u64* plane0 = net.sup + offs[p];
    r0[p] = p < k ? plane0[lane] : 0ull;
    r1[p] = p < k ? plane0[net.dpad + lane] : 0ull;
  }
  u64 keep_l = ~0ull;  // lane 2p: new mask of x_p, lane 2p + 1: of y_p
#pragma unroll
  for (int p = 0; p < P; ++p) {
    if (p >= k) break;
    const u64 dx = readlane64(dl, 2 * p), dy = readlane64(dl, 2 * p + 1);
    const u64 kx = __ballot(((dx >> lane) & 1ull) && (r0[p] & dy) != 0ull);
    const u64 ky = __ballot(((dy >> lane) & 1ull) && (r1[p] & dx) != 0ull);
    if (lane == 2 * p) keep_l = kx;
    if (lane == 2 * p + 1) keep_l = ky;
  }
  int removed_l = 0;
  bool wiped_l = false;
  if (myv >= 0 && (dl & ~keep_l)) {
    const u64 old = atomicAnd(&dom[myv], keep_l);
    removed_l = __popcll(old & ~keep_l);
    wiped_l = old != 0ull && (old & keep_l) == 0ull;
    if (removed_l) atomicSub(&size[myv], removed_l);
  }
  wiped_any = __ballot(wiped_l) != 0ull;
  removed_total = (int)wave_sum64_dpp((u64)removed_l);
  return __ballot(removed_l > 0);
}

// LDS of grid_finish.
struct GridEnd {
  unsigned long long tot[2];
  int last;
};

// End of a grid kernel.  Adds the lanes' removals and the waves' revisions to
// the grid's totals, one workgroup total on the workgroup's slot; the last
// workgroup to finish sums the slots, stores the outcome and, when `final` of
// the epochs says that the fixpoint is over, puts the control block and the
// bitmaps back to their first state, so that the next fixpoint starts without
// a launch to clear them.  e->tot: zero on entry.  Every thread calls it.
template <typename Final>
__device__ __forceinline__ void grid_finish(GacCtl* ctl, unsigned* F, int nvw, GridEnd* e, int revs, int dels, int rounds,
                                            int converged, unsigned long long start, Final final, GacResult* out,
                                            unsigned long long* seq_at, unsigned long long seq) {
  const int tid = threadIdx.x, lane = lane_id();
  const u64 wave_dels = wave_sum64_dpp((u64)dels);
  if (lane == 0 && (wave_dels | (u64)revs)) {
    atomicAdd(&e->tot[0], (unsigned long long)revs);
    atomicAdd(&e->tot[1], wave_dels);
  }
  wait_memory_ops();
  __syncthreads();
  if (tid == 0) {
    if (e->tot[0] | e->tot[1]) {
      atomicAdd(&ctl->revisions[blockIdx.x % kStatSlots], e->tot[0]);
      atomicAdd(&ctl->deletions[blockIdx.x % kStatSlots], e->tot[1]);
    }
    e->tot[0] = 0ull;
    e->tot[1] = 0ull;
    wait_memory_ops();
    const unsigned ticket = atomicAdd(&ctl->done, 1u);
    e->last = ticket + 1u == gridDim.x ? 1 : 0;
  }
  __syncthreads();
  if (uniform_int(e->last) == 0) return;
  u64 r = 0ull, d = 0ull;
  for (int i = tid; i < kStatSlots; i += blockDim.x) {
    r += ld_view<true>((const u64*)&ctl->revisions[i]);
    d += ld_view<true>((const u64*)&ctl->deletions[i]);
  }
  r = wave_sum64_dpp(r);
  d = wave_sum64_dpp(d);
  if (lane == 0) {
    atomicAdd(&e->tot[0], r);
    atomicAdd(&e->tot[1], d);
  }
  const int lp = uniform_int(ld_agent(&ctl->last_push_round)), wr = uniform_int(ld_agent(&ctl->wipe_round));
  const int err = uniform_int(ld_agent(&ctl->err));
  __syncthreads();
  if (tid == 0) {
    ctl->done = 0u;  // (the next round's grid may be another)
    store_result(out, rounds, converged, err, lp, wr, e->tot[1], e->tot[0],
                 wall_clock64() - (start ? start : ld_view<true>((const u64*)&ctl->start)));
  }
  if (!err && final(lp, wr)) {
    for (int i = tid; i < kStatSlots; i += blockDim.x) {
      ctl->deletions[i] = 0ull;
      ctl->revisions[i] = 0ull;
    }
    for (int i = tid; i < 3 * nvw; i += blockDim.x) F[i] = 0u;
    if (tid == 0) {
      ctl->last_push_round = -1;
      ctl->wipe_round = INT_MAX;
      ctl->bar_ticket = 0ull;
    }
  }
  box_publish(seq_at, seq);
}

constexpr int kRoundThreads = 1024;

// One round per launch (host-driven fixpoint).  A launch queued behind the
// round that ended the fixpoint only answers.
__global__ void __launch_bounds__(kRoundThreads) k_gac_round(DevNet net, u64* dom, int* size, unsigned* F, int nvw,
                                                             GacCtl* ctl, int r, int seed, int pairs, int narcs,
                                                             GacResult* out, unsigned long long* seq_at,
                                                             unsigned long long seq) {
  __shared__ GridEnd end;
  if (r > 0 && (ctl->last_push_round < r - 1 || ctl->wipe_round < r)) {
    if (blockIdx.x == 0 && threadIdx.x == 0) box_store(seq_at, seq);
    return;
  }
  if (threadIdx.x == 0) {
    end.tot[0] = 0ull;
    end.tot[1] = 0ull;
    if (blockIdx.x == 0)
      __hip_atomic_store(&ctl->start, (unsigned long long)wall_clock64(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < nvw; i += (long long)gridDim.x * blockDim.x)
    F[(long long)((r + 2) % 3) * nvw + i] = 0u;
  int revs = 0, dels = 0;
  grid_round<false>(net, dom, dom, size, F + (long long)(r % 3) * nvw, F + (long long)((r + 1) % 3) * nvw, ctl, r, seed,
                    pairs != 0, false, make_int4(0, -1, 0, 0), narcs, revs, dels);
  // the epoch only grows: skip the atomic once another wave has raised it
  if (__ballot(dels > 0) && lane_id() == 0 && ld_agent(&ctl->last_push_round) < r) atomicMax(&ctl->last_push_round, r);
  grid_finish(ctl, F, nvw, &end, revs, dels, r + 1, 0, 0ull, [&](int lp, int wr) { return lp < r || wr <= r; }, out,
              seq_at, seq);
}

// ===========================================================================
// Persistent fixpoint: every round in one launch, rounds separated by a grid
// barrier.  The host launches at most one workgroup a CU (1024 threads, at most
// 128 KB of LDS), so that all are resident at once unless other launches hold
// CUs; the bounded waits below cover that case.
//
// The barrier is a ticket count that only grows: thread 0 of each workgroup
// takes a ticket (an atomic add that returns the count) and waits until the
// count reaches the end of its ticket's round, nblocks tickets per round.
// Every wait is bounded: a waiter whose device wall clock passes the launch's
// budget, or that sees the error flag another block raised, stops waiting and
// its block leaves, so the launch always ends (an error, never a hang), even
// if the workgroups were not all resident.  Thread 0 broadcasts the outcome
// through LDS; every wave reads it back as a wave-uniform value
// (readfirstlane), so the round loop leaves through a scalar branch.
// The round decision is taken at the start of the next round from what the
// barrier made visible: wipe_round < r (a block already in round r can only
// set it to r), and no bit in the bitmap of round r - 1's changes (nobody
// writes it before the next barrier).
// ===========================================================================
// Every write a round makes that another workgroup reads in a later round
// (domain words, sizes, changed bits, wipe_round, the cleared bitmap) is an
// agent-scope atomic, and every such read is an agent-scope atomic load, so
// the data never waits in a cache that another XCD cannot see.  Before the
// barrier each wave therefore only waits until its own memory operations have
// completed (s_waitcnt vmcnt(0): atomics with and without return, and
// stores), and the barrier's own accesses are relaxed: no fence, no L2
// write-back or invalidation.  (A release fence in every wave made a barrier
// cost 37 us at 1,024 waves; with one fence-pair per workgroup a 21-round
// cascade took 1.41 ms, fence-free 1.06 ms.)  The
// asynchronous fixpoint relies on the same coherence of agent-scope
// accesses, with no barrier at all.
// Returns false when the launch's budget ran out here or elsewhere.
__device__ __forceinline__ bool grid_barrier(GacCtl* ctl, unsigned nblocks, unsigned long long t0,
                                             unsigned long long max_ticks, int* s_ok) {
  wait_memory_ops();
  __syncthreads();
  if (threadIdx.x == 0) {
    // every workgroup takes one ticket per round, so round r's tickets are
    // r * nblocks .. (r + 1) * nblocks - 1; the round is complete once the
    // count reaches the end of this ticket's round
    const unsigned long long ticket = atomicAdd(&ctl->bar_ticket, 1ull);
    const unsigned long long target = (ticket / nblocks + 1) * nblocks;
    int ok = 1;
    while (__hip_atomic_load(&ctl->bar_ticket, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target) {
      if (ld_agent(&ctl->err)) {
        ok = 0;
        break;
      }
      if (wall_clock64() - t0 > max_ticks) {
        atomicExch(&ctl->err, 1);
        ok = 0;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    *s_ok = ok;
  }
  __syncthreads();
  return uniform_int(*s_ok) != 0;
}

constexpr int kPersistentThreads = 1024;

// LDS bytes of a round's copy of the domains and of the changed bitmap.
__host__ __device__ inline long long persistent_lds_bytes(int n, int W) {
  return 8ll * n * W + 4ll * ((n + 31) / 32);
}

// kStaged: each round starts with a copy of the domains and of the changed
// bitmap into LDS (one trip to memory for both, coalesced), and every lane
// reads them there; otherwise the lanes read them from memory.  A round is
// then that copy, the rows, the removals and the barrier: a chain of four to
// six memory round trips, which is what bounds a cascade's many small rounds.
// The first arc of each lane stays in registers over the rounds.
template <bool kStaged>
__global__ void __launch_bounds__(kPersistentThreads) k_gac_persistent(DevNet net, u64* dom, int* size, unsigned* F,
                                                                       int nvw, GacCtl* ctl, int max_rounds, int seed,
                                                                       int pairs, int narcs,
                                                                       unsigned long long max_ticks,
                                                                       GacResult* out, unsigned long long* seq_at,
                                                                       unsigned long long seq) {
  extern __shared__ __align__(16) char smem[];
  __shared__ int s_ok;
  __shared__ GridEnd end;
  if (threadIdx.x == 0) {
    end.tot[0] = 0ull;
    end.tot[1] = 0ull;
  }
  __syncthreads();
  const unsigned long long t0 = wall_clock64();
  const int tid = threadIdx.x, lane = lane_id();
  const long long words = (long long)net.n * net.W;
  u64* sdom = (u64*)smem;
  unsigned* scur = (unsigned*)(smem + 8 * words);
  int lw = 0;
  while ((1 << lw) < net.W) ++lw;
  const long long i0 = (long long)blockIdx.x * blockDim.x + tid;
  const long long arc0 = net.W > 1 ? (long long)(lane >> lw) * ((gridDim.x * blockDim.x) >> 6) + (i0 >> 6) : i0;
  const int4 e0 = arc0 < narcs ? net.adj[arc0] : make_int4(0, -1, 0, 0);
  int r = 0, revs = 0, dels = 0;  // the wave's revisions and the lane's removals, over every round
  enum { NEXT, WIPE, FIXPOINT, ERROR } decision = NEXT;
  if (kStaged) {
    for (long long i = tid; i < words; i += blockDim.x) sdom[i] = ld_view<true>(&dom[i]);
    __syncthreads();
  }
  while (true) {
    unsigned* cur = F + (long long)(r % 3) * nvw;
    unsigned* nxt = F + (long long)((r + 1) % 3) * nvw;
    for (long long i = i0; i < nvw; i += (long long)gridDim.x * blockDim.x)
      __hip_atomic_store(&F[(long long)((r + 2) % 3) * nvw + i], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (kStaged) grid_round<false>(net, sdom, dom, size, scur, nxt, ctl, r, seed, pairs != 0, true, e0, narcs, revs, dels);
    else grid_round<true>(net, dom, dom, size, cur, nxt, ctl, r, seed, pairs != 0, true, e0, narcs, revs, dels);
    if (!grid_barrier(ctl, gridDim.x, t0, max_ticks, &s_ok)) {
      decision = ERROR;
      break;
    }
    ++r;
    const int wr = ld_agent(&ctl->wipe_round);
    if (kStaged) {
      for (long long i = tid; i < words; i += blockDim.x) sdom[i] = ld_view<true>(&dom[i]);
      for (int i = tid; i < nvw; i += blockDim.x) scur[i] = (unsigned)ld_agent((const int*)&nxt[i]);
      __syncthreads();
    }
    unsigned bits = 0u;
    for (int i = lane; i < nvw; i += 64) bits |= kStaged ? scur[i] : (unsigned)ld_agent((const int*)&nxt[i]);
    const bool any = __ballot(bits != 0u) != 0ull;
    if (uniform_int(wr) < r) decision = WIPE;
    else if (!any) decision = FIXPOINT;
    if (decision != NEXT || r >= max_rounds) break;
  }
  grid_finish(ctl, F, nvw, &end, revs, dels, r, decision == FIXPOINT ? 1 : 0, t0, [](int, int) { return true; }, out,
              seq_at, seq);
}

// First state of a grid fixpoint's control block and bitmaps (kept from one
// fixpoint to the next by grid_finish, but for one that ended in an error).
__global__ void k_gac_init(GacCtl* ctl, unsigned* F, int nvw) {
  const long long i0 = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i0 == 0) {
    ctl->last_push_round = -1;
    ctl->wipe_round = INT_MAX;
    ctl->bar_ticket = 0ull;
    ctl->err = 0;
    ctl->done = 0u;
    ctl->start = 0ull;
  }
  for (long long i = i0; i < kStatSlots; i += (long long)gridDim.x * blockDim.x) {
    ctl->deletions[i] = 0ull;
    ctl->revisions[i] = 0ull;
  }
  for (long long i = i0; i < 3ll * nvw; i += (long long)gridDim.x * blockDim.x) F[i] = 0u;
}

// ===========================================================================
// Asynchronous fixpoint in one launch, without any grid barrier.
//
// The frontier is a bitmap of constraints.  A wave claims a whole frontier
// word with an atomic exchange, revises the claimed constraints and pushes
// the constraints of every variable that lost values.  `pending` counts the
// queued plus the claimed-but-unfinished constraints; it is raised before a
// push sets its bits (once per revision batch, for every constraint the batch
// pushes) and lowered only after the claimed constraints are finished and
// for the pushed bits that were already set.  The lowering is kept per wave
// (`owed`) and published when the wave finds no work in a frontier chunk:
// pending never drops below the outstanding work, and it reaches 0 once the
// fixpoint is reached and every wave has gone idle.  (One atomic on pending
// per push and per claim made that word the bottleneck: 11 ms against 4 ms on
// a 23-round cascade.)
// No wave waits for another: an idle wave keeps scanning until pending is 0,
// the wipe-out flag is set, or its time budget runs out (then it sets `err`
// and leaves), so every wave exits and co-residency is not required.
// Domain and frontier words are read with agent-scope atomic loads, so a
// revision always sees removals completed by other XCDs before the push that
// queued it.
// ===========================================================================
struct AsyncCtl {
  unsigned long long pending;
  int wipe;
  int err;
  unsigned long long deletions[kStatSlots];
  unsigned long long revisions[kStatSlots];
};

// counted: pending was already raised by the caller for all of v's constraints
__device__ __forceinline__ void push_var_async(const DevNet& net, int v, unsigned* F, AsyncCtl* ctl, int& owed,
                                               bool counted = false) {
  const int lane = lane_id();
  const int b0 = net.adj_off[v], b1 = net.adj_off[v + 1];
  for (int i0 = b0; i0 < b1; i0 += 64) {
    const int k = min(64, b1 - i0);
    if (!counted && lane == 0) atomicAdd(&ctl->pending, (unsigned long long)k);
    bool already = false;
    if (lane < k) {
      const int c = net.adj[i0 + lane].x;
      const unsigned bit = 1u << (c & 31);
      already = (atomicOr(&F[c >> 5], bit) & bit) != 0u;
    }
    owed += __popcll(__ballot(already));
  }
}

__device__ __forceinline__ void async_process_constraint(const DevNet& net, u64* dom, int* size, int c,
                                                         unsigned* F, AsyncCtl* ctl,
                                                         unsigned long long& revs,
                                                         unsigned long long& dels, int& owed) {
  const ConMeta* mp = net.con + c;
  bool wiped = false;
  if (mp->kind == 0) {
    const int x = mp->scope[0], y = mp->scope[1];
    const int rx = revise_binary<true>(net, dom, size, c, x, y, 1, &wiped);
    ++revs;
    if (wiped && lane_id() == 0) atomicExch(&ctl->wipe, 1);
    if (rx) {
      dels += rx;
      push_var_async(net, x, F, ctl, owed);
    }
    const int ry = revise_binary<true>(net, dom, size, c, y, x, 0, &wiped);
    ++revs;
    if (wiped && lane_id() == 0) atomicExch(&ctl->wipe, 1);
    if (ry) {
      dels += ry;
      push_var_async(net, y, F, ctl, owed);
    }
  } else {
    auto on_removed = [&](int v, int k) {
      dels += k;
      push_var_async(net, v, F, ctl, owed);
    };
    revise_table<decltype(on_removed), true, false>(net, dom, size, c, -1, nullptr, on_removed, &wiped);
    ++revs;
    if (wiped && lane_id() == 0) atomicExch(&ctl->wipe, 1);
  }
}

__global__ void k_gac_async(DevNet net, u64* dom, int* size, unsigned* F, int nfw, AsyncCtl* ctl,
                            unsigned long long max_ticks) {
  const int lane = lane_id();
  const long long gw = ((long long)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const unsigned long long t0 = wall_clock64();
  const int nchunks = (nfw + 63) / 64;
  int chunk = (int)(gw % nchunks);
  int seen = 0;  // chunks scanned since the last claim
  int owed = 0;  // finished claims and duplicate pushes not yet taken off pending
  unsigned long long revs = 0, dels = 0;
  while (true) {
    if (__hip_atomic_load(&ctl->wipe, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ||
        __hip_atomic_load(&ctl->err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      break;
    const int wi = chunk * 64 + lane;
    unsigned bits = 0u;
    if (wi < nfw) bits = __hip_atomic_load(&F[wi], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const u64 nz = __ballot(bits != 0u);
    if (nz) {
      const int l = (int)__builtin_ctzll(nz);
      unsigned claimed = 0u;
      if (lane == 0) claimed = atomicExch(&F[chunk * 64 + l], 0u);
      claimed = __shfl(claimed, 0, 64);
      const int nclaimed = __popc(claimed);
      const int base_c = (chunk * 64 + l) * 32;
      if (net.W == 1) {
        // one-word domains: binary constraints kAsyncPairBatch at a time
        claimed = (unsigned)uniform_int((int)claimed);
        while (claimed) {
          int cs[kAsyncPairBatch] = {};
          int k = 0;
          while (claimed && k < kAsyncPairBatch) {
            const int b = __ffs(claimed) - 1;
            claimed &= claimed - 1u;
            const int c = base_c + b;
            if (net.con[c].kind != 0) {
              async_process_constraint(net, dom, size, c, F, ctl, revs, dels, owed);
              continue;
            }
#pragma unroll
            for (int p = 0; p < kAsyncPairBatch; ++p)
              if (p == k) cs[p] = c;
            ++k;
          }
          if (k) {
            int myv = -1, removed = 0;
            bool wiped = false;
            u64 changed = revise_pairs_w1<true, kAsyncPairBatch>(net, dom, size, cs, k, myv, removed, wiped);
            revs += 2 * k;
            dels += removed;
            if (wiped && lane == 0) atomicExch(&ctl->wipe, 1);
            if (changed) {
              // raise pending once for every constraint the changed
              // variables push, before any of their bits is set
              int tot = 0;
              if ((changed >> lane) & 1ull) tot = net.adj_off[myv + 1] - net.adj_off[myv];
              for (int o = 32; o > 0; o >>= 1) tot += __shfl_xor(tot, o, 64);
              if (lane == 0) atomicAdd(&ctl->pending, (unsigned long long)tot);
            }
            while (changed) {
              const int cl = (int)__builtin_ctzll(changed);
              changed &= changed - 1ull;
              push_var_async(net, __builtin_amdgcn_readlane(myv, cl), F, ctl, owed, true);
            }
          }
        }
      } else {
        while (claimed) {
          const int b = __ffs(claimed) - 1;
          claimed &= claimed - 1u;
          async_process_constraint(net, dom, size, base_c + b, F, ctl, revs, dels, owed);
        }
      }
      owed += nclaimed;
      seen = 0;
      continue;
    }
    chunk = chunk + 1 == nchunks ? 0 : chunk + 1;
    if (owed) {
      if (lane == 0) atomicSub(&ctl->pending, (unsigned long long)owed);
      owed = 0;
    }
    if (++seen >= nchunks) {
      seen = 0;
      const unsigned long long p =
          __hip_atomic_load(&ctl->pending, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (p == 0ull) break;
      if (wall_clock64() - t0 > max_ticks) {
        if (lane == 0) atomicExch(&ctl->err, 1);
        break;
      }
      __builtin_amdgcn_s_sleep(8);
    }
  }
  if (lane == 0 && (revs | dels)) {
    atomicAdd(&ctl->revisions[blockIdx.x % kStatSlots], revs);
    atomicAdd(&ctl->deletions[blockIdx.x % kStatSlots], dels);
  }
}

// First state of the asynchronous fixpoint, before k_seed_async.
__global__ void k_async_init(unsigned* F, int nfw, AsyncCtl* ctl) {
  const int i0 = blockIdx.x * blockDim.x + threadIdx.x;
  for (int i = i0; i < nfw; i += gridDim.x * blockDim.x) F[i] = 0u;
  for (int i = i0; i < kStatSlots; i += gridDim.x * blockDim.x) {
    ctl->deletions[i] = 0ull;
    ctl->revisions[i] = 0ull;
  }
  if (i0 == 0) {
    ctl->pending = 0ull;
    ctl->wipe = 0;
    ctl->err = 0;
  }
}

// Seed the asynchronous frontier: all active constraints, or those of var, or
// those of the variables in the bitmap `changed` (n variables) if there is one.
__global__ void k_seed_async(unsigned* F, int nfw, int ncons, const int* adj_off, const int4* adj, int var,
                             const unsigned* changed, int n, AsyncCtl* ctl) {
  if (changed) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n || !((changed[v >> 5] >> (v & 31)) & 1u)) return;
    int fresh = 0;
    for (int i = adj_off[v]; i < adj_off[v + 1]; ++i) {
      const unsigned bit = 1u << (adj[i].x & 31);
      if (!(atomicOr(&F[adj[i].x >> 5], bit) & bit)) ++fresh;
    }
    if (fresh) atomicAdd(&ctl->pending, (unsigned long long)fresh);
    return;
  }
  if (var < 0) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nfw) {
      const int k = ncons - (int)(i * 32);
      F[i] = k >= 32 ? 0xffffffffu : (k <= 0 ? 0u : ((1u << k) - 1u));
    }
    if (i == 0) ctl->pending = (unsigned long long)ncons;
    return;
  }
  if (blockIdx.x != 0) return;
  for (int i = adj_off[var] + threadIdx.x; i < adj_off[var + 1]; i += blockDim.x) {
    const int c = adj[i].x;
    const unsigned bit = 1u << (c & 31);
    if (!(atomicOr(&F[c >> 5], bit) & bit)) atomicAdd(&ctl->pending, 1ull);
  }
}

// Streaming copy (16-byte lanes, grid-stride): the known-traffic kernel used
// to calibrate hardware byte counters and to measure achievable bandwidth.
__global__ void k_stream_copy(const uint4* __restrict__ src, uint4* __restrict__ dst, long long n16) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n16;
       i += (long long)gridDim.x * blockDim.x)
    dst[i] = src[i];
}

// Recompute exact sizes of one level (after host-side writes).
__global__ void k_sizes(const u64* dom, int* size, int n, int W) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n) return;
  int s = 0;
  for (int w = 0; w < W; ++w) s += __popcll(dom[(long long)v * W + w]);
  size[v] = s;
}

// ===========================================================================
// Workgroup engine.  One workgroup owns one domain copy (in LDS when it fits,
// else in a per-workgroup global scratch region) and runs an AC fixpoint over
// a variable frontier: every round revises all arcs u <- t for the variables
// t that changed in the previous round, spread over the waves of the
// workgroup.  Assigned variables (asg bitmap) are never revised, as in
// AC3::enforce (src/AC3.cpp:114); the closure is the same with or without
// that skip.
// ===========================================================================
struct WgMem {
  u64* dom;       // [n * W]
  int* list;      // [n]
  int* pre;       // [n + 1]
  int* size;      // [n]
  unsigned* bm;   // [3][nvw] frontier bitmaps, rotating by round
  unsigned* asg;  // [nvw]
  int* stamp;     // [ncons] constraint stamps (dom/wdeg), NULL otherwise
  const int* aoff;   // adjacency offsets (net.adj_off)
  const int4* adj;   // adjacency entries (net.adj)
};

struct WgCtl {
  // lowest round that emptied a domain, of the running fixpoint (slot: see wg_fixpoint)
  int wipe_round[2];
  int2 flat[3];  // wg_fixpoint_flat: a round removed values, emptied a domain
  unsigned long long revs;
  u64 red[16];  // one slot per wave for block reductions
  int ok;
};

__host__ __device__ inline long long wg_mem_bytes(int n, int W) {
  const long long nvw = (n + 31) / 32;
  long long b = 8ll * n * W;
  b += 4ll * n;          // list
  b += 4ll * (n + 1);    // pre
  b += 4ll * n;          // size
  b += 4ll * nvw * 4;    // bm, asg
  return (b + 15) & ~15ll;
}

__device__ __forceinline__ WgMem wg_carve(char* base, const DevNet& net) {
  const int n = net.n, W = net.W;
  const int nvw = (n + 31) / 32;
  WgMem m;
  m.stamp = nullptr;
  m.aoff = net.adj_off;
  m.adj = net.adj;
  m.dom = (u64*)base;
  char* p = base + 8ll * n * W;
  m.list = (int*)p;
  p += 4ll * n;
  m.pre = (int*)p;
  p += 4ll * (n + 1);
  m.size = (int*)p;
  p += 4ll * n;
  m.bm = (unsigned*)p;
  p += 12ll * nvw;
  m.asg = (unsigned*)p;
  return m;
}

__device__ __forceinline__ bool bit_of(const unsigned* bm, int v) { return (bm[v >> 5] >> (v & 31)) & 1u; }

__device__ __forceinline__ int ld_wg_int(const int* p) {
  return __hip_atomic_load(const_cast<int*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Values of `need` (word w of D(u)) without a support in D(t), one arc word
// per lane, with one source t for the whole wave; lanes without an arc pass
// need = 0.  rows: word w of the rows of t's values over D(u); own: the rows
// of the values of word w of D(u) over D(t), word j at own + j dpad.
//
// As arcs_unsupported, but the values of t are wave-uniform: scalar
// instructions pick them, four rows a step (eight cost bandwidth on networks
// read from memory: 256 uneven instances 4.3 ms against 2.7 ms), and a lane
// spends one address and one load on each.  With more than two source steps
// left, the wave turns to the target side once no lane has more than a few
// open values, or (several words) after three steps if settling the others one
// after the other takes fewer steps than the rest of D(t).
template <bool kTight>
__device__ __forceinline__ u64 wave_unsupported(const DevNet& net, const u64* dom, int t, const u64* rows,
                                                const u64* own, u64 need) {
  constexpr int kStep = 4;
  const int W = net.W, dpad = net.dpad;
  const u64* dt = dom + (long long)t * W;
  int left = 0;
  for (int j = 0; j < W; ++j) left += __popcll((u64)uniform_ll((long long)ld_wg(&dt[j])));
  const int few = W == 1 ? 4 : 2;
  bool target = false;
  int done = 0;
  for (int j = 0; j < W && !target; ++j) {
    u64 x = (u64)uniform_ll((long long)ld_wg(&dt[j]));
    const u64* rj = rows + 64 * j;
    while (x) {
      // the next kStep values (the first of them again once the word is
      // exhausted), picked by scalar instructions outside the lanes' branch
      int a[kStep];
#pragma unroll
      for (int i = 0; i < kStep; ++i) {
        a[i] = uniform_int(x ? (int)__builtin_ctzll(x) : a[0]);
        x &= x - 1ull;
      }
      if (need) {
        u64 r[kStep];
#pragma unroll
        for (int i = 0; i < kStep; ++i) r[i] = rj[a[i]];
        u64 o = 0ull;
#pragma unroll
        for (int i = 0; i < kStep; ++i) o |= r[i];
        need &= ~o;
      }
      left -= kStep;
      ++done;
      if (__ballot(need != 0ull) == 0ull) return 0ull;
      if (left > 2 * kStep) {
        const u64 many = __ballot(__popcll(need) > few);
        if (many == 0ull ||
            (kTight && W > 1 && done >= 3 && (__popcll(many) + kSettle - 1) / kSettle * 2 * kStep < left)) {
          target = true;
          break;
        }
      }
    }
  }
  if (!target) return need;
  u64 settled = 0ull;  // values that the wave settled as unsupported
  if (kTight && W > 1) {
    const u64 many = __ballot(__popcll(need) > few);
    if (many) {
      const u64 left_open = wave_settle<false>(net, dom, (long long)(own - net.sup), t, need, many);
      if (__popcll(need) > few) {
        settled = left_open;
        need = 0ull;
      }
    }
  }
  u64 gone = settled;
  if (W == 1) {
    const u64 d = (u64)uniform_ll((long long)ld_wg(&dt[0]));
    while (need) {
      u64 r[4], bit[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        bit[i] = need & (0ull - need);
        r[i] = need ? own[__builtin_ctzll(need)] : ~0ull;
        need &= need - 1ull;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) gone |= (r[i] & d) ? 0ull : bit[i];
    }
    return gone;
  }
  while (need) {
    const int b = (int)__builtin_ctzll(need);
    bool ok = false;
    for (int j0 = 0; j0 < W && !ok; j0 += 4) {
      u64 r[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] = j0 + i < W ? own[(long long)(j0 + i) * dpad + b] : 0ull;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (j0 + i < W) ok = ok || (r[i] & ld_wg(&dt[j0 + i])) != 0ull;
    }
    if (!ok) gone |= 1ull << b;
    need &= need - 1ull;
  }
  return gone;
}

// Takes `gone` out of a domain word of variable u: u joins the next frontier,
// and the lane that brings its size to 0 records the wipe-out.
__device__ __forceinline__ void lane_remove(const WgMem& mem, WgCtl* ctl, unsigned* nxt, int slot, int round, int u,
                                            u64* word, u64 gone) {
  const u64 old = and_wg(word, ~gone);
  const int r = __popcll(old & gone);
  if (r) {
    atomicOr(&nxt[u >> 5], 1u << (u & 31));
    if (atomicSub(&mem.size[u], r) == r) atomicMin(&ctl->wipe_round[slot], round);
  }
}

// Frontier of a fixpoint's first round: variable `seed`, or every variable
// (seed < 0), or the bitmap `changed` if there is one; the other two bitmaps and
// the wipe-out word of `slot` are cleared.  Called by every thread, a
// __syncthreads() before wg_fixpoint.
__device__ __forceinline__ void wg_seed(const WgMem& mem, WgCtl* ctl, int n, int slot, int seed,
                                        const unsigned* changed = nullptr) {
  const int nvw = (n + 31) / 32;
  for (int i = threadIdx.x; i < 3 * nvw; i += blockDim.x) {
    unsigned v = 0u;
    if (i < nvw) {
      const int k = n - 32 * i;
      if (changed) v = changed[i];
      else if (seed < 0) v = k >= 32 ? 0xffffffffu : ((1u << k) - 1u);
      else if (i == seed >> 5) v = 1u << (seed & 31);
    }
    mem.bm[i] = v;
  }
  if (threadIdx.x == 0) ctl->wipe_round[slot] = INT_MAX;
}

// AC fixpoint from the seed that wg_seed put in mem.bm (a __syncthreads()
// lies between).  seed_both >= 0: in the first round also revise t <- u for
// every arc of this seed variable t (constraint seeding, as
// GModel::EnforceGAC(assigned_var) does).  Returns false on wipe-out.  Must
// be called by every thread of the workgroup.
//
// A unit of work is 64 / Wp arcs of one changed variable t (Wp = W rounded up
// to a power of two): lane (k, w) revises word w of the k-th arc's target.
// Every wave numbers the round's units in registers, from the frontier bitmap
// and the variables' arc counts (lane = variable), and takes every nwaves-th:
// no list, no shared counter, and one barrier per round.  Tables follow, one
// per wave, each revised once however many of its variables changed.
//
// What bounds it is the chain of dependent reads of a round (frontier,
// adjacency, domains, rows) and the barrier, not bandwidth.  With a lane per
// arc word instead of a wave per one to four arcs, one chain serves 64 / Wp
// arcs and a row read fetches one row of each instead of 64: 1000 search
// nodes of n=23 d=23 e=253 took 7.4 ms (28.2 ms before; they now take
// wg_fixpoint_flat), 256 uneven instances (n 20..200, d 8..128) of 64 nodes
// each 2.7 ms (33 ms before).  The heaviest of those, rounds of some 14,000
// arc words with the rows in memory, are bound by the cache lines that a
// wave's row reads touch: neither rows of two values a load nor adjacency
// entries read ahead gained anything.
//
// The frontier bitmaps rotate: round r reads bitmap r % 3, fills (r + 1) % 3
// and clears (r + 2) % 3, which no wave reads until the barrier of the next
// round.  A wipe-out is recorded as the round it happened in, so that a wave
// that still decides round r is not misled by one already in round r + 1.
// slot: two wipe-out words used in turn by successive fixpoints, so that
// wg_seed never resets the word a slow wave still reads.
//
// kTight: tight relations are settled by the wave (wave_unsupported).  kTabs: of
// many tables only those with a changed variable are taken up.  Each only costs
// registers on the other networks (with the look at the tables in the kernel,
// searches on n=23 d=23 e=253 and under dom/wdeg on n=100 d=50 take 3 % longer,
// the tests of n=60 d=37 e=500 3.5 %, a fixpoint of n=40 d=16 e=195 7.9 instead
// of 7.4 us): kTabs is for networks of more than kTableTurns tables a wave, and
// searches take both (kFull) where the host's full_search says so.
constexpr int kTableTurns = 4;

template <bool kTight, bool kTabs>
__device__ __forceinline__ bool wg_fixpoint(const DevNet& net, const WgMem& mem, WgCtl* ctl, int slot,
                                            int seed_both) {
  const int n = net.n, W = net.W;
  const int nvw = (n + 31) / 32;
  const int tid = threadIdx.x;
  const int nthreads = blockDim.x;
  const int wave = uniform_int(tid >> 6), nwaves = nthreads >> 6;
  const int lane = lane_id();
  int lw = 0;
  while ((1 << lw) < W) ++lw;
  const int w = lane & ((1 << lw) - 1), la = lane >> lw, per = 64 >> lw;
  const long long pair_words = 2ll * W * net.dpad;
  int revs = 0;
  bool result = true;
  int c0 = 0, c1 = nvw, c2 = 2 * nvw;
  // this wave's first table, its lanes' part kept over the rounds
  const int itab = nwaves - 1 - wave;
  const bool many_tabs = kTabs && net.ntabs > kTableTurns * nwaves;
  SmallTable tab0{};
  if (itab < net.ntabs) tab0 = load_small_table(net, uniform_int(net.tabs[itab]));
  for (int round = 0;; ++round) {
    const unsigned* cur = mem.bm + c0;
    unsigned* nxt = mem.bm + c1;
    for (int i = tid; i < nvw; i += nthreads) mem.bm[c2 + i] = 0u;
    const bool both = seed_both >= 0 && round == 0;
    int mine = wave;  // this wave's next unit, counted from the block of variables below
    bool stop = false;
    u64 some = ~0ull;  // words of the frontier with a changed variable, 64 of them from v0 / 32 on
    for (int v0 = 0; v0 < n && !stop; v0 += 64) {
      // blocks without one are passed over: a path of 2,800 variables, one
      // changed a round, took 20 us a round with every block counted
      if (n > 128) {
        if ((v0 & 2047) == 0) some = __ballot((v0 >> 5) + lane < nvw && cur[(v0 >> 5) + lane] != 0u);
        const u64 rest = some >> ((v0 >> 5) & 63);
        v0 = rest ? v0 + ((int)__builtin_ctzll(rest) >> 1) * 64 : v0 | 1984;
        if (rest == 0ull) continue;
      }
      const int v = v0 + lane;
      int a0 = 0, deg = 0;
      if (v < n) {
        a0 = mem.aoff[v];
        deg = bit_of(cur, v) ? mem.aoff[v + 1] - a0 : 0;
      }
      const int units = (deg + per - 1) >> (6 - lw);
      int total = 0;
      const int inc = wave_scan_dpp(units, &total);
      for (;; mine += nwaves) {
        const int q = uniform_int(mine);
        if (q >= total) break;
        const int wr = ld_wg_int(&ctl->wipe_round[slot]);
        const int l = (int)__builtin_ctzll(__ballot(inc > q));
        const int t = v0 + l;
        const int k0 = (q - __builtin_amdgcn_readlane(inc - units, l)) << (6 - lw);
        const int cnt = min(per, __builtin_amdgcn_readlane(deg, l) - k0);
        const int arc = __builtin_amdgcn_readlane(a0, l) + k0 + la;
        int u = -1;
        u64 need = 0ull;
        u64* word = nullptr;
        const u64* pair = net.sup;
        int pos_t = 0;
        if (la < cnt && w < W) {
          const int4 e = mem.adj[arc];
          u = e.y;
          pos_t = adj_pos(e);
          pair += e.w * pair_words;
          if (u >= 0) {  // binary
            word = mem.dom + (long long)u * W + w;
            if (!bit_of(mem.asg, u)) need = ld_wg(word);
          }
        }
        if (uniform_int(wr) <= round) {
          stop = true;
          break;
        }
        const u64 gone = wave_unsupported<kTight>(net, mem.dom, t, pair + (long long)(pos_t * W + w) * net.dpad,
                                                  pair + (long long)(1 - pos_t) * W * net.dpad + 64 * w, need);
        if (gone) lane_remove(mem, ctl, nxt, slot, round, u, word, gone);
        revs += cnt;
      }
      mine -= total;
    }
    if (both && !bit_of(mem.asg, seed_both)) {
      // t <- u of the seed's arcs, spread over the waves and settled by them, a
      // lane per value of t (by a lane per arc word, up to 64 values of it one
      // after the other, 40 arcs of 64 values at t=0.886 cost 110 us)
      const int a0 = uniform_int(mem.aoff[seed_both]), deg = uniform_int(mem.aoff[seed_both + 1]) - a0;
      for (int i0 = 0; i0 < deg; i0 += nwaves * per) {
        const int i = i0 + la * nwaves + nwaves - 1 - wave;
        int4 e = make_int4(0, -1, 0, 0);
        if (i < deg) e = mem.adj[a0 + i];
        const bool act = e.y >= 0 && w < W;
        u64* word = mem.dom + (long long)seed_both * W + (w < W ? w : 0);
        const u64 need = act ? ld_wg(word) : 0ull;
        const u64 todo = __ballot(need != 0ull);
        if (todo == 0ull) continue;
        const long long own = act ? e.w * pair_words + (long long)adj_pos(e) * W * net.dpad + 64 * w : 0ll;
        const u64 gone = wave_settle<false>(net, mem.dom, own, act ? e.y : 0, need, todo);
        if (gone) lane_remove(mem, ctl, nxt, slot, round, seed_both, word, gone);
        revs += __popcll(__ballot(act && w == 0));
      }
    }
    // Tables in turn, one a wave; where they are more than kTableTurns a wave, its
    // lanes first look which ones have a changed variable.  Small tables: each wave
    // looks at its own (every nwaves-th, so that a variable's tables, often
    // neighbours, are not left to one wave).  Larger ones cost more than the
    // look, so that every wave looks at all of them and takes every nwaves-th
    // changed one.  In turn / own / dealt, us: 300 tables of arity 5 and 3,000
    // tuples after one assignment 201 / 190 / 142, the tests of that network 1208
    // / 1013 / 774; 900 small ones 174 / 86 / 131, tests 2410 / 1273 / 1385.
    const int look = net.big_tabs ? 1 : nwaves;  // tables between two lanes'
    int seen = 0;                                // changed tables before this turn's
    for (int base = many_tabs && look == 1 ? 0 : itab; base < net.ntabs; base += many_tabs ? 64 * look : nwaves) {
      u64 found = 1ull;  // bit k: table base + k * look is this wave's
      if (kTabs && many_tabs) {
        const int k = base + lane * look;
        bool ch = false;
        if (k < net.ntabs) {
          // (unused positions of a table hold its first variable: no arity to read)
          const ConMeta* mp = net.con + net.tabs[k];
          unsigned bits = 0u;
#pragma unroll
          for (int p = 0; p < CPIM_MAX_ARITY; ++p) bits |= cur[mp->scope[p] >> 5] >> (mp->scope[p] & 31);
          ch = bits & 1u;
        }
        found = __ballot(ch);
        if (look == 1) {
          const int rank = seen + __popcll(found & ((1ull << lane) - 1ull));
          seen += __popcll(found);
          found = __ballot(ch && rank % nwaves == itab);
        }
      }
      for (; found != 0ull; found &= found - 1ull) {
        const int i = uniform_int(base + (int)__builtin_ctzll(found) * look);
        const int c = uniform_int(net.tabs[i]);
        SmallTable tab = tab0;
        if (i != itab) tab = load_small_table(net, c);
        const bool small = uniform_int(small_table(net, net.con[c].arity, tab.tw)) != 0;
        int y = tab.y;
        if (!small) y = lane < net.con[c].arity ? net.con[c].scope[lane] : -1;
        const int yy = y >= 0 ? y : 0;
        const bool mine_changed = y >= 0 && bit_of(cur, yy);
        const bool assigned = bit_of(mem.asg, yy);
        const u64 dp = small ? ld_wg(&mem.dom[yy]) : 0ull;
        const u64 changed = __ballot(mine_changed);
        if (changed == 0ull) continue;
        ++revs;
        if (small) {
          // lane 8 p removes for position p, but not for the only changed one
          u64 rows[8];
          small_table_rows(tab, rows);
          const unsigned gone = (unsigned)dp & ~small_table_keep(tab.y, tab.tw, rows, (unsigned)dp);
          const unsigned pos = (unsigned)changed & 0x01010101u;
          const u64 stays = both || (pos & (pos - 1u)) ? 0ull : pos;
          if (gone && y >= 0 && !assigned && lane < 32 && (lane & 7) == 0 && !((stays >> lane) & 1ull))
            lane_remove(mem, ctl, nxt, slot, round, y, &mem.dom[y], (u64)gone);
          continue;
        }
        // one changed variable: its own position is not revised (AC3 does not
        // either, src/AC3.cpp:106-118; at a closure its values keep their supports)
        int skip = -1;
        if (!both && (changed & (changed - 1ull)) == 0ull) skip = __builtin_amdgcn_readlane(y, (int)__builtin_ctzll(changed));
        bool wiped = false;
        revise_table(net, mem.dom, mem.size, c, skip, mem.asg,
                     [&](int v, int) {
                       if (lane == 0) atomicOr(&nxt[v >> 5], 1u << (v & 31));
                     },
                     &wiped);
        if (wiped && lane == 0) atomicMin(&ctl->wipe_round[slot], round);
      }
    }
    __syncthreads();
    const int wr = ld_wg_int(&ctl->wipe_round[slot]);
    unsigned any = 0u;
    for (int i = lane; i < nvw; i += 64) any |= nxt[i];
    if (uniform_int(wr) <= round) {
      result = false;
      break;
    }
    if (__ballot(any != 0u) == 0ull) break;
    const int c = c0;
    c0 = c1;
    c1 = c2;
    c2 = c;
  }
  if (lane == 0 && revs) atomicAdd(&ctl->revs, (unsigned long long)revs);
  return result;
}

// The same fixpoint for a search on a small network: domains of at most 32
// values (one 32-bit word), kFlatArcs arcs a lane (one if a domain has more
// than 16 values) and small tables only, one per wave.  Every lane keeps its
// arcs' support rows in registers over the whole search (32 rows of 32 bits,
// or 4 x 16 rows of 16 bits), a table's wave the rows of its table, so a round
// reads nothing but domains.  An arc is revised when its source's domain is
// not the one it last saw, so no frontier is kept; the first round revises
// the arcs of the seed only, whose domain the caller passes, so the caller's
// store of it needs no barrier before.
//
// What bounds it is a round's chain of three LDS round trips (domains,
// removal, flags), some 60 dependent instructions and the barrier; waves
// beyond those that the arcs and tables fill only add to the instructions
// each SIMD issues, hence LdsNet::flat_threads.  1000 search nodes of n=23
// d=23 e=253 take 3.3 ms; 5.8 ms with frontier bitmaps, the rows read from LDS
// every round and 1024 threads.
constexpr int kFlatArcs = 4;     // arcs per lane, of domains of at most 16 values
constexpr int kFlatTables = 16;  // one per wave

typedef short v2s __attribute__((ext_vector_type(2)));

struct FlatNet {
  int tu[kFlatArcs];  // source | target << 16, -1: no binary arc
  // rows of the source's values over the target: one a word (wide), or values
  // i and i + 8 in the halves of word i of the arc's eight; a table's wave:
  // the words of its eight rows
  unsigned rows[8 * kFlatArcs];
  int arcs;    // arcs of the wave's lanes, wave-uniform (a table's wave has none)
  bool wide;
  bool table;  // the wave has a table
  int y, tw;   // of the table: SmallTable
};

// The domains of its arcs' sources (0: of its table position's variable) that
// a lane last revised them for: D as it is, after a fixpoint.
struct FlatSeen {
  unsigned arc[kFlatArcs];
  unsigned skip;  // bit k: arc k (0: the table position) has no target, or an assigned one
};

__device__ __forceinline__ FlatNet wg_load_flat(const DevNet& net, const WgMem& mem) {
  FlatNet f;
  const int tid = threadIdx.x;
  const int lanes = blockDim.x - 64 * net.ntabs;  // that take arcs
  const int narcs = uniform_int(mem.aoff[net.n]);
  const int first = uniform_int(tid & ~63);
  f.table = first >= lanes;
  f.arcs = !f.table && first < narcs ? (narcs - first + lanes - 1) / lanes : 0;
  f.wide = net.cap > 16;
#pragma unroll
  for (int k = 0; k < kFlatArcs; ++k) {
    const int i = k * lanes + tid;
    int4 e = make_int4(0, -1, 0, 0);
    if (!f.table && i < narcs) e = mem.adj[i];
    f.tu[k] = e.y >= 0 ? adj_var(e) | (e.y << 16) : -1;
    // lanes without an arc take the rows of plane 0; rows past the source's
    // domain, of other planes or of the padding behind the last, are masked
    // by it
    const u64* row = net.sup + (e.y >= 0 ? (2 * e.w + adj_pos(e)) * net.dpad : 0);
    if (!f.wide) {
#pragma unroll
      for (int v = 0; v < 8; ++v) f.rows[8 * k + v] = ((unsigned)row[v] & 0xffffu) | ((unsigned)row[v + 8] << 16);
    } else if (k == 0) {
#pragma unroll
      for (int v = 0; v < 8 * kFlatArcs; ++v) f.rows[v] = (unsigned)row[v];
    }
  }
  f.y = -1;
  f.tw = 0;
  if (f.table) {
    const SmallTable t = load_small_table(net, uniform_int(net.tabs[(first - lanes) >> 6]));
    f.y = t.y;
    f.tw = t.tw;
    u64 r[8];
    small_table_rows(t, r);
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      f.rows[2 * v] = (unsigned)r[v];
      f.rows[2 * v + 1] = (unsigned)(r[v] >> 32);
    }
  }
  return f;
}

// Every domain and assigned variable as they are now, before the first
// fixpoint and that of a refutation (nothing may change before the next
// barrier).
__device__ __forceinline__ void wg_flat_see(const WgMem& mem, const FlatNet& f, FlatSeen& seen) {
  seen.skip = 0u;
#pragma unroll
  for (int k = 0; k < kFlatArcs; ++k)
    if (k < f.arcs) {
      const int u = f.tu[k] >> 16, uu = u >= 0 ? u : 0;
      seen.arc[k] = (unsigned)ld_wg(&mem.dom[u >= 0 ? f.tu[k] & 0xffff : 0]);
      if (u < 0 || bit_of(mem.asg, uu)) seen.skip |= 1u << k;
    }
  if (f.table) {
    const int y = f.y >= 0 ? f.y : 0;
    seen.arc[0] = (unsigned)ld_wg(&mem.dom[y]);
    if (f.y < 0 || bit_of(mem.asg, y)) seen.skip = 1u;
  }
}

// seed < 0: every arc and table.  seed_dom: D(seed); seed_assigned: the seed
// is a decision.  turn: the flags of the round (kept over the fixpoints of a
// search).  Which targets are assigned is kept with what the lanes have seen:
// read from LDS at each fixpoint, it cost 2% of a search.
__device__ __forceinline__ bool wg_fixpoint_flat(const WgMem& mem, WgCtl* ctl, const FlatNet& f, FlatSeen& seen,
                                                 int seed, unsigned seed_dom, bool seed_assigned, int& turn,
                                                 int& revs) {
  const int lane = lane_id();
  const int y = f.y >= 0 ? f.y : 0;
  if (seed_assigned) {
#pragma unroll
    for (int k = 0; k < kFlatArcs; ++k)
      if (k < f.arcs && (f.tu[k] >> 16) == seed) seen.skip |= 1u << k;
    if (f.table && y == seed) seen.skip = 1u;
  }
  const unsigned skip = seen.skip;
  bool first = true;
  while (true) {
    const int next = turn == 2 ? 0 : turn + 1;
    if (threadIdx.x == 0) ctl->flat[next] = make_int2(0, 0);
    const bool seeded = first && seed >= 0, all = first && seed < 0;
    bool changed = false, wiped = false;
    auto remove = [&](int u, unsigned gone) {
      const unsigned old = (unsigned)and_wg(&mem.dom[u], ~(u64)gone);
      const unsigned lost = old & gone;
      if (lost) {
        atomicSub(&mem.size[u], __popc(lost));
        changed = true;
        wiped = wiped || lost == old;
      }
    };
#pragma unroll
    for (int k = 0; k < kFlatArcs; ++k)
      if (k < f.arcs) {
        const int u = f.tu[k] >> 16, t = u >= 0 ? f.tu[k] & 0xffff : 0;
        const unsigned dt = (unsigned)ld_wg(&mem.dom[t]);
        const unsigned du = (unsigned)ld_wg(&mem.dom[u >= 0 ? u : 0]);
        // (the first round leaves the other arcs what they have seen: their
        // sources may be losing values already)
        const unsigned d = !seeded ? dt : t == seed ? seed_dom : seen.arc[k];
        const bool act = (seeded ? t == seed : all || d != seen.arc[k]) && !((skip >> k) & 1u);
        seen.arc[k] = d;
        const u64 active = __ballot(act);
        if (active) {
          unsigned o = 0u;
          if (!f.wide) {
            const unsigned x = (d & 0xffu) | ((d & 0xff00u) << 8);
            const v2s xs = __builtin_bit_cast(v2s, x);
#pragma unroll
            for (int v = 0; v < 8; ++v) {
              const v2s m = (v2s)(xs << (short)(15 - v)) >> (short)15;
              o |= f.rows[8 * k + v] & __builtin_bit_cast(unsigned, m);
            }
            o = (o | (o >> 16)) & 0xffffu;
          } else if (k == 0) {
#pragma unroll
            for (int b = 0; b < kFlatArcs; ++b) {
              if (__ballot(act && ((d >> (8 * b)) & 0xffu) != 0u) == 0ull) continue;
#pragma unroll
              for (int v = 8 * b; v < 8 * b + 8; ++v)
                o |= f.rows[v] & (unsigned)__builtin_amdgcn_sbfe((int)d, v, 1);
            }
          }
          const unsigned gone = act ? du & ~o : 0u;
          if (gone) remove(u, gone);
          revs += __popcll(active);
        }
      }
    if (f.table) {
      const unsigned now = (unsigned)ld_wg(&mem.dom[y]);
      const unsigned dp = seeded && y == seed ? seed_dom : now;
      const bool act = f.y >= 0 && (seeded ? y == seed : all || dp != seen.arc[0]);
      if (__ballot(act)) {
        ++revs;
        u64 r[8];
#pragma unroll
        for (int v = 0; v < 8; ++v) r[v] = ((u64)f.rows[2 * v + 1] << 32) | f.rows[2 * v];
        const unsigned keep = small_table_keep(f.y, f.tw, r, dp);
        seen.arc[0] = skip ? dp : dp & keep;  // its own removals take no tuple
        const unsigned gone = dp & ~keep;
        if (gone && !skip && lane < 32 && (lane & 7) == 0) remove(y, gone);  // lane 8 p: position p
      }
    }
    if (changed) __hip_atomic_store(&ctl->flat[turn].x, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (wiped) __hip_atomic_store(&ctl->flat[turn].y, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __syncthreads();
    const u64 flags = (u64)uniform_ll((long long)ld_wg((const u64*)&ctl->flat[turn]));
    turn = next;
    first = false;
    if (flags >> 32) return false;
    if (flags == 0ull) return true;
  }
}

__device__ __forceinline__ void wg_clear_bitmap(unsigned* bm, int nvw) {
  for (int i = threadIdx.x; i < nvw; i += blockDim.x) bm[i] = 0u;
}

__device__ __forceinline__ void wg_copy_words(u64* dst, const u64* src, long long count) {
  for (long long i = threadIdx.x; i < count; i += blockDim.x) dst[i] = src[i];
}

// Block-wide reduction helpers (all threads call; result valid in every thread).
// Workgroup reductions, called by every thread: each wave reduces over DPP,
// lane 0 publishes the wave's result, and every wave reduces the published
// results (lane i reads wave i's) the same way.
__device__ __forceinline__ u64 wg_reduce_min_u64(WgCtl* ctl, u64 v) {
  v = wave_min64_dpp(v);
  const int wave = threadIdx.x >> 6, nwaves = blockDim.x >> 6, lane = lane_id();
  if (lane == 0) ctl->red[wave] = v;
  __syncthreads();
  const u64 r = wave_min64_dpp(lane < nwaves ? ctl->red[lane] : ~0ull);
  __syncthreads();
  return (u64)uniform_ll((long long)r);
}

__device__ __forceinline__ u64 wg_reduce_sum_u64(WgCtl* ctl, u64 v) {
  v = wave_sum64_dpp(v);
  const int wave = threadIdx.x >> 6, nwaves = blockDim.x >> 6, lane = lane_id();
  if (lane == 0) ctl->red[wave] = v;
  __syncthreads();
  const u64 r = wave_sum64_dpp(lane < nwaves ? ctl->red[lane] : 0ull);
  __syncthreads();
  return (u64)uniform_ll((long long)r);
}

// ---------------------------------------------------------------------------
// Block-mode GAC on one level (one workgroup).  changed: goes on from these
// variables, where rounds over the grid left off (NULL: starts from seed_var).
// ---------------------------------------------------------------------------
template <bool kLds, bool kTabs>
__global__ void k_block_gac(DevNet net, u64* dom, int* size, int seed_var, const unsigned* changed, char* scratch,
                            GacResult* out, unsigned long long* seq_at, unsigned long long seq) {
  const unsigned long long t0 = wall_clock64();
  extern __shared__ __align__(16) char smem[];
  __shared__ WgCtl ctl;
  const int n = net.n, W = net.W;
  char* base = kLds ? smem : scratch;
  WgMem mem = wg_carve(base, net);
  if (threadIdx.x == 0) ctl.revs = 0;
  wg_copy_words(mem.dom, dom, (long long)n * W);
  for (int v = threadIdx.x; v < n; v += blockDim.x) mem.size[v] = size[v];
  wg_clear_bitmap(mem.asg, (n + 31) / 32);
  wg_seed(mem, &ctl, n, 0, seed_var, changed);
  __syncthreads();
  long long before = 0;
  for (int v = threadIdx.x; v < n; v += blockDim.x) before += mem.size[v];
  const bool ok = wg_fixpoint<true, kTabs>(net, mem, &ctl, 0, changed ? -1 : seed_var);
  long long after = 0;
  for (int v = threadIdx.x; v < n; v += blockDim.x) after += mem.size[v];
  const u64 delta = wg_reduce_sum_u64(&ctl, (u64)(before - after));
  wg_copy_words(dom, mem.dom, (long long)n * W);
  for (int v = threadIdx.x; v < n; v += blockDim.x) size[v] = mem.size[v];
  if (threadIdx.x == 0)
    store_result(out, 1, ok ? 1 : 0, 0, 0, ok ? INT_MAX : 0, delta, ctl.revs, wall_clock64() - t0);
  box_publish(seq_at, seq);
}

// ---------------------------------------------------------------------------
// Level operations, one workgroup each, answering in the host box: one launch
// a call (a call took a copy each way through the runtime's staging memory,
// three kernels and a stream synchronization).
// ---------------------------------------------------------------------------
__global__ void k_level_put(const u64* src, u64* dom, int* size, int n, int W, unsigned long long* seq_at,
                            unsigned long long seq) {
  // the words in order (a thread per variable reads host memory 8 bytes a line:
  // 64 KB took 36 us so), then the sizes
  for (int i = threadIdx.x; i < n * W; i += blockDim.x) {
    const u64 d = __hip_atomic_load(const_cast<u64*>(&src[i]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    dom[i] = d;
    if (W == 1) size[i] = __popcll(d);
  }
  if (W > 1) {
    __syncthreads();
    for (int v = threadIdx.x; v < n; v += blockDim.x) {
      int s = 0;
      for (int w = 0; w < W; ++w) s += __popcll(dom[(long long)v * W + w]);
      size[v] = s;
    }
  }
  box_publish(seq_at, seq);
}

__global__ void k_level_get(const u64* dom, unsigned long long* dst, int words, unsigned long long* seq_at,
                            unsigned long long seq) {
  for (int i = threadIdx.x; i < words; i += blockDim.x) box_store(&dst[i], dom[i]);
  box_publish(seq_at, seq);
}

__global__ void k_level_copy(const u64* src, u64* dst, const int* src_size, int* dst_size, int n, int W,
                             unsigned long long* seq_at, unsigned long long seq) {
  for (int i = threadIdx.x; i < n * W; i += blockDim.x) dst[i] = src[i];
  for (int i = threadIdx.x; i < n; i += blockDim.x) dst_size[i] = src_size[i];
  box_publish(seq_at, seq);
}

enum LevelOp {
  kOpAssign,    // D(var) = {value}
  kOpRemove,    // D(var) -= {value}; answers the new size, -1 if the value was not there
  kOpSize,      // |D(var)|
  kOpFirst,     // smallest value >= value of D(var), -1 if none
  kOpAssigned,  // the value of an assigned variable, -1 otherwise
  kOpMinVar,    // variable with the smallest |D| > 1, the lowest id on ties; -1 if none
  kOpAll        // 1: every variable is assigned
};

template <int kThreads>
__global__ void __launch_bounds__(kThreads) k_level_op(int op, u64* dom, int* size, int n, int W, int max_dom, int var,
                                                  int value, int* answer, unsigned long long* seq_at,
                                                  unsigned long long seq) {
  __shared__ u64 red[kThreads / 64];
  const int tid = threadIdx.x;
  u64* d = dom + (long long)var * W;
  int res = 0;
  if (op == kOpMinVar || op == kOpAll) {
    u64 key = ~0ull;
    for (int v = tid; v < n; v += kThreads) {
      const int s = size[v];
      const u64 k = op == kOpAll ? (u64)(s == 1) : (s > 1 ? ((u64)(unsigned)s << 32) | (unsigned)v : ~0ull);
      key = k < key ? k : key;
    }
    key = wave_min64_dpp(key);
    if (lane_id() == 0) red[tid >> 6] = key;
    __syncthreads();
    for (int i = 0; i < kThreads / 64; ++i) key = red[i] < key ? red[i] : key;
    res = op == kOpAll ? (int)(key & 1ull) : (key == ~0ull ? -1 : (int)(unsigned)key);
  } else if (tid == 0) {
    if (op == kOpAssign) {
      for (int w = 0; w < W; ++w) d[w] = w == (value >> 6) ? 1ull << (value & 63) : 0ull;
      size[var] = 1;
    } else if (op == kOpRemove) {
      const u64 bit = 1ull << (value & 63);
      res = -1;
      if (d[value >> 6] & bit) {
        d[value >> 6] &= ~bit;
        res = 0;
        for (int w = 0; w < W; ++w) res += __popcll(d[w]);
        size[var] = res;
      }
    } else if (op == kOpSize) {
      res = size[var];
    } else {
      const int start = op == kOpAssigned ? 0 : value;
      res = -1;
      if (op == kOpFirst || size[var] == 1)
        for (int w = start >> 6; w < W && res < 0; ++w) {
          u64 x = d[w];
          if (w == start >> 6) x &= ~0ull << (start & 63);
          if (x) res = 64 * w + (int)__builtin_ctzll(x);
        }
      if (res >= max_dom) res = -1;
    }
  }
  if (tid == 0) box_store(answer, res);
  box_publish(seq_at, seq);
}

// ---------------------------------------------------------------------------
// Batched singleton tests: workgroup `first + blockIdx.x` takes test (x, a),
// copies the base level into its domain copy, reduces x to {a}, marks x
// assigned and runs the fixpoint from {x}; fail[i] records a wipe-out.  The
// copies never touch HBM when they fit in LDS.  One test per workgroup: the
// kernel has no loop around its barriers, and the hardware dispatcher keeps
// every CU busy as workgroups finish at different times.
// ---------------------------------------------------------------------------
template <bool kLds, bool kTabs>
__global__ void k_singleton_tests(DevNet net, const u64* __restrict__ base_dom,
                                  const int* __restrict__ base_size, const int2* __restrict__ tests,
                                  long long ntests, long long first, unsigned char* fail,
                                  unsigned long long* revs_out, char* scratch, long long scratch_stride) {
  extern __shared__ __align__(16) char smem[];
  __shared__ WgCtl ctl;
  const long long unit = first + blockIdx.x;
  if (unit >= ntests) return;
  const int n = net.n, W = net.W;
  const int nvw = (n + 31) / 32;
  char* base = kLds ? smem : scratch + (long long)blockIdx.x * scratch_stride;
  WgMem mem = wg_carve(base, net);
  const int2 tst = tests[unit];
  const int x = uniform_int(tst.x), a = uniform_int(tst.y);
  wg_copy_words(mem.dom, base_dom, (long long)n * W);
  for (int v = threadIdx.x; v < n; v += blockDim.x) mem.size[v] = base_size[v];
  wg_clear_bitmap(mem.asg, nvw);
  wg_seed(mem, &ctl, n, 0, x);
  if (threadIdx.x == 0) ctl.revs = 0;
  __syncthreads();
  if (threadIdx.x < W) mem.dom[(long long)x * W + threadIdx.x] = (threadIdx.x == (a >> 6)) ? (1ull << (a & 63)) : 0ull;
  if (threadIdx.x == 0) {
    mem.size[x] = 1;
    mem.asg[x >> 5] |= 1u << (x & 31);
  }
  __syncthreads();
  const bool ok = wg_fixpoint<true, kTabs>(net, mem, &ctl, 0, -1);
  __syncthreads();  // every wave's revision count
  if (threadIdx.x == 0) {
    fail[unit] = ok ? 0 : 1;
    if (ctl.revs) atomicAdd(&revs_out[blockIdx.x % kStatSlots], ctl.revs);
  }
}

// ---------------------------------------------------------------------------
// Bit-sliced singleton tests (binary networks).  A workgroup runs up to 64
// singleton tests together: sl[v][b] is the 64-bit mask of the tests in
// which value b of v is alive.  Revising u <- t for all of them at once,
// value b of u keeps test k iff some value a of t with R(b, a) has bit k in
// sl[t][a].  One support row serves 64 tests, and each value stops scanning
// its supports as soon as every test that holds it has found one.
//
// Every test's bits evolve as a chaotic AC iteration of that test alone
// (a revision is monotone and idempotent, and a revision caused by another
// test's change is merely redundant), and a round ends with no change only
// when every arc is consistent in every test.  So each test reaches the GAC
// closure of its own network (unique), and test k failed iff some variable
// holds no value with bit k.  The tests' variables are not skipped as
// assigned: with x reduced to {a} the closure is the same either way.
//
// The slices live in global memory (n * dpad words per workgroup), read with
// agent-scope loads so that no stale L1 line is ever used; the source slice
// of the current work item is staged in wave-private LDS.
// ---------------------------------------------------------------------------
constexpr int kSliceArcs = 16;  // most arcs of one variable per work item

// Staged source slices: word w of t's domain occupies kStageWord entries: a
// zero entry, the masks of values 64w..64w+31, a zero entry, the masks of
// values 64w+32..64w+63.  A half-word scan reads entry ffbl(bits) of its
// half, and v_ffbl_b32 of an exhausted (zero) half is -1: the zero entry.
constexpr int kStageWord = 66;

struct SliceCtl {
  int item_ctr;
  int nchanged[2];
  int m;
  int total;
  int k;  // arcs per work item this round
  u64 act;  // tests not wiped out
  unsigned long long revs;
};

__host__ __device__ inline long long slice_lds_bytes(int n, int dpad, int nwaves) {
  const long long nvw = (n + 31) / 32;
  long long b = 4ll * n + 4ll * (n + 1) + 12ll * nvw;
  b = (b + 15) & ~15ll;
  b += 8ll * nwaves * (kStageWord * (dpad / 64) + CPIM_MAX_WORDS);
  return b;
}

__device__ __forceinline__ void slice_mark(unsigned* nxt, SliceCtl* ctl, int v, int slot) {
  const unsigned bit = 1u << (v & 31);
  const unsigned old = atomicOr(&nxt[v >> 5], bit);
  if (!(old & bit)) atomicAdd(&ctl->nchanged[slot], 1);
}


__device__ __forceinline__ int stage_pos(int v) {
  const int b = v & 63;
  return (v >> 6) * kStageWord + 1 + b + (b >> 5);
}

// Lowest set bit of x, -1 for 0 (the hardware result of v_ffbl_b32).
__device__ __forceinline__ int ffbl_raw(unsigned x) {
  int r;
  asm("v_ffbl_b32 %0, %1" : "=v"(r) : "v"(x));
  return r;
}

// pend &= ~(st[a] for every set bit a of bits), four bits per step; st[-1]
// is the zero entry.
__device__ __forceinline__ u64 clear_supported(u64 pend, unsigned bits, const u64* st) {
  while (bits && pend) {
    const int a0 = ffbl_raw(bits);
    bits &= bits - 1u;
    const int a1 = ffbl_raw(bits);
    bits &= bits - 1u;
    const int a2 = ffbl_raw(bits);
    bits &= bits - 1u;
    const int a3 = ffbl_raw(bits);
    bits &= bits - 1u;
    pend &= ~((st[a0] | st[a1]) | (st[a2] | st[a3]));
  }
  return pend;
}

// Revise u <- t for every live test (act).  plane_u: rows of the values of u
// over t's domain (element (w, b) = word w of the row of b); slu: slices of
// u; stage: slices of t in the kStageWord layout; atw[w]: values of t alive
// in some live test.  A variable no test has changed yet (touched_u false)
// still holds `all` on its base values, so its slices are derived from the
// base domain words base_u instead of being loaded; a stale "untouched"
// only yields a superset of the live tests, which costs work, not accuracy.  Returns (wave-uniform) whether some bit of u was cleared
// by this wave.
__device__ __forceinline__ bool slice_revise(const u64* __restrict__ plane_u, u64* slu,
                                             const u64* stage, const u64* atw, int W, int dpad,
                                             u64 act, bool touched_u, const u64* __restrict__ base_u,
                                             u64 all) {
  const int lane = lane_id();
  bool changed = false;
  for (int j0 = 0; j0 < W; j0 += 4) {
    u64 need[4], row0[4];
    if (touched_u) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = j0 + q;
        need[q] = j < W ? ld_wg(&slu[j * 64 + lane]) : 0ull;
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = j0 + q;
        need[q] = (j < W && ((base_u[j < W ? j : 0] >> lane) & 1ull)) ? all : 0ull;
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int j = j0 + q;
      row0[q] = j < W ? plane_u[j * 64 + lane] : 0ull;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int b = (j0 + q) * 64 + lane;
      u64 pend = need[q] & act;  // live tests holding b that still need a support
      if (pend) {
        const u64 r = row0[q] & atw[0];
        pend = clear_supported(pend, (unsigned)r, stage + 1);
        pend = clear_supported(pend, (unsigned)(r >> 32), stage + 34);
      }
      for (int w = 1; w < W && pend; ++w) {
        const u64 r = plane_u[(long long)w * dpad + b] & atw[w];
        const u64* st = stage + w * kStageWord;
        pend = clear_supported(pend, (unsigned)r, st + 1);
        pend = clear_supported(pend, (unsigned)(r >> 32), st + 34);
      }
      if (pend) {
        const u64 old = and_wg(&slu[b], ~pend);
        if (old & pend) changed = true;
      }
    }
  }
  return __ballot(changed) != 0ull;
}

// Workgroup `blockIdx.x` runs test group g (tests [gfirst[g], gfirst[g+1])
// of the list sorted by variable) in its slice region; fail[perm[i]]
// (fail[i] when perm is null) receives the outcome of sorted test i.  Blocks are mapped to groups so
// that each XCD takes a contiguous run of groups (same variables, shared
// support rows in its L2).
__global__ void k_sliced_tests(DevNet net, const u64* __restrict__ base_dom,
                               const int2* __restrict__ tests, const int* __restrict__ gfirst,
                               long long g0, const int* __restrict__ perm, unsigned char* fail,
                               unsigned long long* revs_out, u64* slices) {
  extern __shared__ __align__(16) char smem[];
  __shared__ SliceCtl ctl;
  const int n = net.n, W = net.W, dpad = net.dpad;
  const int nvw = (n + 31) / 32;
  const int tid = threadIdx.x, nthreads = blockDim.x;
  const int lane = lane_id();
  const int wave = uniform_int(tid >> 6), nwaves = nthreads >> 6;
  const int B = gridDim.x, bid = blockIdx.x;
  const int xcd = bid & 7, q = B >> 3, rem = B & 7;
  const long long g = g0 + (long long)xcd * q + (xcd < rem ? xcd : rem) + (bid >> 3);
  const int tf = gfirst[g];
  const int tc = uniform_int(gfirst[g + 1] - tf);
  const u64 all = tc >= 64 ? ~0ull : ((1ull << tc) - 1ull);
  u64* sl = slices + (long long)bid * n * dpad;

  int* list = (int*)smem;
  int* pre = list + n;
  unsigned* cur = (unsigned*)(pre + n + 1);
  unsigned* nxt = cur + nvw;
  unsigned* touched = nxt + nvw;  // variables some test has changed
  const long long head = (4ll * n + 4ll * (n + 1) + 12ll * nvw + 15) & ~15ll;
  u64* stage = (u64*)(smem + head) + (long long)wave * (kStageWord * W + CPIM_MAX_WORDS);
  u64* atw = stage + kStageWord * W;
  if (lane < 2 * W) stage[(lane >> 1) * kStageWord + 33 * (lane & 1)] = 0ull;  // zero entries

  // Slices of the base level: every test holds every base value.
  for (int v = wave; v < n; v += nwaves) {
    for (int b = lane; b < dpad; b += 64) {
      const bool in = (base_dom[(long long)v * W + (b >> 6)] >> (b & 63)) & 1ull;
      sl[(long long)v * dpad + b] = in ? all : 0ull;
    }
  }
  for (int i = tid; i < nvw; i += nthreads) {
    cur[i] = 0u;
    nxt[i] = 0u;
    touched[i] = 0u;
  }
  if (tid == 0) {
    ctl.act = all;
    ctl.revs = 0;
  }
  __syncthreads();
  // Test k reduces its variable x_k to {a_k}.
  for (int k = wave; k < tc; k += nwaves) {
    const int2 tk = tests[tf + k];
    for (int b = lane; b < dpad; b += 64) {
      u64* p = &sl[(long long)tk.x * dpad + b];
      if (b == tk.y) or_wg(p, 1ull << k);
      else and_wg(p, ~(1ull << k));
    }
  }
  if (tid < tc) {
    const int x = tests[tf + tid].x;
    atomicOr(&cur[x >> 5], 1u << (x & 31));
    atomicOr(&touched[x >> 5], 1u << (x & 31));
  }
  __syncthreads();

  unsigned long long revs = 0;
  for (int round = 0;; ++round) {
    const int slot = round & 1;
    if (wave == 0) {
      // item size: at most kSliceArcs arcs, small enough for about four
      // items per wave when the round has few arcs
      int arcs = 0;
      for (int v0 = 0; v0 < n; v0 += 64) {
        const int v = v0 + lane;
        if (v < n && bit_of(cur, v)) arcs += net.adj_off[v + 1] - net.adj_off[v];
      }
      for (int d = 32; d > 0; d >>= 1) arcs += __shfl_xor(arcs, d, 64);
      const int K = uniform_int(max(1, min(kSliceArcs, (arcs + 4 * nwaves - 1) / (4 * nwaves))));
      int base = 0, ibase = 0;
      for (int v0 = 0; v0 < n; v0 += 64) {
        const int v = v0 + lane;
        const bool f = v < n && bit_of(cur, v);
        const u64 mask = __ballot(f);
        const int rank = mbcnt(mask);
        const int items = f ? (net.adj_off[v + 1] - net.adj_off[v] + K - 1) / K : 0;
        const int inc = wave_inclusive_scan(items);
        if (f) {
          list[base + rank] = v;
          pre[base + rank] = ibase + inc - items;
        }
        base += __popcll(mask);
        ibase += __shfl(inc, 63, 64);
      }
      if (lane == 0) {
        pre[base] = ibase;
        ctl.m = base;
        ctl.total = ibase;
        ctl.k = K;
        ctl.item_ctr = 0;
        ctl.nchanged[slot] = 0;
      }
    } else {
      for (int i = tid - 64; i < nvw; i += nthreads - 64) nxt[i] = 0u;
    }
    if (nthreads == 64)
      for (int i = lane; i < nvw; i += 64) nxt[i] = 0u;
    __syncthreads();
    const int total = uniform_int(ctl.total);
    const int m = uniform_int(ctl.m);
    const int K = uniform_int(ctl.k);
    const u64 act = (u64)uniform_ll((long long)ctl.act);
    while (true) {
      int idx = 0;
      if (lane == 0) idx = atomicAdd(&ctl.item_ctr, 1);
      idx = uniform_int(__shfl(idx, 0, 64));
      if (idx >= total) break;
      int lo = 0, hi = m - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (pre[mid] <= idx) lo = mid;
        else hi = mid - 1;
      }
      const int t = uniform_int(list[lo]);
      const int s0 = net.adj_off[t] + (idx - uniform_int(pre[lo])) * K;
      const int s1 = min(s0 + K, net.adj_off[t + 1]);
      const int cnt = uniform_int(s1 - s0);
      // stage the slices of t and the values alive in some live test
      const u64* slt = sl + (long long)t * dpad;
      for (int i = lane; i < dpad; i += 64) {
        const u64 v = ld_wg(&slt[i]);
        stage[stage_pos(i)] = v;
        const u64 alive = __ballot((v & act) != 0ull);
        if (lane == 0) atw[i >> 6] = alive;
      }
      __builtin_amdgcn_wave_barrier();
      int4 e = make_int4(0, 0, 0, 0);
      if (lane < cnt) e = net.adj[s0 + lane];
      for (int i = 0; i < cnt; ++i) {
        const int u = __builtin_amdgcn_readlane(e.y, i);
        const int pos_t = __builtin_amdgcn_readlane(adj_pos(e), i);
        const long long o = (long long)__builtin_amdgcn_readlane(e.w, i) * 2 * W * dpad;
        const u64* plane_u = net.sup + o + (long long)(1 - pos_t) * W * dpad;
        const bool tu = uniform_int((int)bit_of(touched, u));
        const bool ch = slice_revise(plane_u, sl + (long long)u * dpad, stage, atw, W, dpad, act, tu,
                                     base_dom + (long long)u * W, all);
        ++revs;
        if (ch && lane == 0) slice_mark(nxt, &ctl, u, slot);
      }
      __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // Exact wipe-out check: a test wiped out at v only if v changed.
    u64 alive_all = ~0ull;
    for (int v = wave; v < n; v += nwaves) {
      if (!uniform_int((int)bit_of(nxt, v))) continue;
      u64 o = 0ull;
      for (int i = lane; i < dpad; i += 64) o |= ld_wg(&sl[(long long)v * dpad + i]);
      for (int d = 32; d > 0; d >>= 1) o |= __shfl_xor(o, d, 64);
      alive_all &= o;
    }
    if (lane == 0 && alive_all != ~0ull) atomicAnd(&ctl.act, alive_all);
    for (int i = tid; i < nvw; i += nthreads) touched[i] |= nxt[i];
    __syncthreads();
    const u64 act_now = (u64)uniform_ll((long long)ctl.act);
    if (uniform_int(ctl.nchanged[slot]) == 0 || act_now == 0ull) break;
    unsigned* tmp = cur;
    cur = nxt;
    nxt = tmp;
  }
  if (lane == 0 && revs) atomicAdd(&ctl.revs, revs);
  __syncthreads();
  if (tid < tc) fail[perm ? perm[tf + tid] : tf + tid] = ((ctl.act >> tid) & 1ull) ? 0 : 1;
  if (tid == 0 && ctl.revs) atomicAdd(&revs_out[blockIdx.x % kStatSlots], ctl.revs);
}

// ---------------------------------------------------------------------------
// Wide bit-sliced singleton tests: 64 M tests per workgroup (M = 1, 2, 4).
// Within a round the workgroup walks the changed variables t one at a time:
// all threads stage t's masks into a shared, double-buffered LDS area (one
// barrier per t), then the waves take t's arcs u <- t from a shared counter.
// One support entry serves 64 M tests; the revision is the one of
// k_sliced_tests applied to M masks at once (same fixpoint argument, same
// exact end-of-round wipe-out check).
//
// The slices hold changes from the base level, not survivors: bit k of
// sl[(v * dpad + b) * M + m] flips the base state of value b of v in test
// 64 m + k.  For a base value a set bit means the test removed it; for a
// value outside the base domain a set bit means the test holds it, which
// only the test's own value can be (a test (x, a) reduces x to {a} whether
// or not a is in the base domain).  So value b is alive in test k iff the
// bit differs from "b in the base domain".  The region of a workgroup is all
// zero when the kernel starts (every test holds exactly the base domain), a
// variable's slice is written only when some test changes one of its values,
// and the workgroup zeroes the slices of the variables it wrote (its touched
// set) before it ends, so the buffer is all zero again for the next launch.
// The caller zeroes the buffer once, when it allocates it.
// ---------------------------------------------------------------------------
template <int M>
struct WideCtl {
  int m;
  int nchanged[2];
  int pad;
  int arc_ctr[2];  // next arc of the staged variable, per stage buffer
  u64 act[M];
  unsigned long long revs;
};

// Words of one stage buffer: kStageWord * W entries of M masks, or with
// nibble tables (nib) 16 W nibbles x 16 subsets of M masks.  With nb byte
// tables the first nb bytes of word 0 have one 256-subset table each in
// place of their 2 nb nibble tables.
__host__ __device__ inline long long wide_stage_words(int W, int M, bool nib, int nb = 0) {
  if (!nib) return (long long)kStageWord * W * M;
  return 256ll * nb * M + 16ll * (16 * W - 2 * nb) * M;
}

// Stage buffers: two (double buffered) without byte tables, one with them.
__host__ __device__ inline int wide_stage_buffers(int nb) { return nb > 0 ? 1 : 2; }

// LDS bytes: list [n], cur/nxt/touched bitmaps, up to 255 bytes that align
// the stage buffers to 256 bytes, the stage buffers and as many alive-value
// rows of W words.  Every nibble-table buffer is a multiple of 256 bytes, so
// each buffer and each half-word table in it stays aligned.
__host__ __device__ inline long long wide_lds_bytes(int n, int W, int M, bool nib = false, int nb = 0) {
  const long long nvw = (n + 31) / 32;
  long long b = 4ll * n + 12ll * nvw;
  b = ((b + 15) & ~15ll) + 256;
  const int nbuf = wide_stage_buffers(nb);
  b += nbuf * 8ll * wide_stage_words(W, M, nib, nb) + nbuf * 8ll * W;
  return b;
}

template <int M>
__device__ __forceinline__ bool any_mask(const u64 (&x)[M]) {
  u64 o = 0ull;
#pragma unroll
  for (int m = 0; m < M; ++m) o |= x[m];
  return o != 0ull;
}

// pend[m] &= ~(st[a][m] for every set bit a of bits), four bits per step;
// entry -1 of st is zero (exhausted bits).  Entries hold the M masks of one
// value together (two 16-byte reads for M = 4).
template <int M>
__device__ __forceinline__ void clear_supported_wide(u64 (&pend)[M], unsigned bits, const u64* st) {
  while (bits && any_mask<M>(pend)) {
    const int a0 = ffbl_raw(bits);
    bits &= bits - 1u;
    const int a1 = ffbl_raw(bits);
    bits &= bits - 1u;
    const int a2 = ffbl_raw(bits);
    bits &= bits - 1u;
    const int a3 = ffbl_raw(bits);
    bits &= bits - 1u;
    const u64* e0 = st + (long long)a0 * M;
    const u64* e1 = st + (long long)a1 * M;
    const u64* e2 = st + (long long)a2 * M;
    const u64* e3 = st + (long long)a3 * M;
#pragma unroll
    for (int m = 0; m < M; ++m) pend[m] &= ~((e0[m] | e1[m]) | (e2[m] | e3[m]));
  }
}

// Nibble tables ("four Russians"): entry (q, s) of a half-word table holds,
// for the 4 values 4q..4q+3 of the half, the OR of the masks of the values
// in subset s (s = 0 is zero).  One lookup covers every support of a row
// nibble.  The nibbles are taken in order, kNibStep per step, by every lane
// of the wave together: the lanes of a step read the same 16-entry blocks,
// which keeps LDS bank conflicts low, and the loads of a step are
// independent.  A lane stops once its row bits or its pending tests are
// exhausted.  Four per step measured 8.2 ms per 128,000-test pass against
// 8.8 ms for two and 8.4 ms for eight (and 10.0 ms for lanes that each jump
// to their own first non-empty nibble, the earlier form).
constexpr int kNibStep = 4;
constexpr unsigned kNibStepMask = kNibStep >= 8 ? 0xffffffffu : ((1u << (4 * kNibStep)) - 1u);

// Word of mask mm of subset `sub` in the table of nibble q.  With four masks
// an entry (32 bytes) is split in two 16-byte halves kept in separate
// 256-byte planes of the nibble's block: plane h holds masks 2h, 2h + 1 of
// the 16 subsets.  The 16 entries a wave's lanes pick from in one read then
// sit on distinct banks (one 16-byte slot each) instead of colliding every
// fourth entry.
template <int M>
__device__ __forceinline__ int nib_word(int q, int sub, int mm) {
  if constexpr (M == 4) return q * 64 + (mm >> 1) * 32 + sub * 2 + (mm & 1);
  else return (q * 16 + sub) * M + mm;
}

// p & ~(a | b | c | d): one three-input OR and one gfx950 three-input logic
// op (truth table 0x10: first operand set, the other two clear).
__device__ __forceinline__ unsigned andnot_or4(unsigned p, unsigned a, unsigned b, unsigned c, unsigned d) {
  return __builtin_amdgcn_bitop3_b32(p, a | b | c, d, 0x10);
}

// (a ^ b) & c, one three-input op per 32-bit half (truth table 0x28).
__device__ __forceinline__ u64 xor_and64(u64 a, u64 b, u64 c) {
  const unsigned lo = __builtin_amdgcn_bitop3_b32((unsigned)a, (unsigned)b, (unsigned)c, 0x28);
  const unsigned hi = __builtin_amdgcn_bitop3_b32((unsigned)(a >> 32), (unsigned)(b >> 32), (unsigned)(c >> 32), 0x28);
  return (u64)lo | ((u64)hi << 32);
}

// a & b as one op per 32-bit half with b uniform (a select of b would first
// copy b out of its scalar register).
__device__ __forceinline__ u64 and64(u64 a, u64 b) {
  const unsigned lo = __builtin_amdgcn_bitop3_b32((unsigned)a, (unsigned)b, 0u, 0xC0);
  const unsigned hi = __builtin_amdgcn_bitop3_b32((unsigned)(a >> 32), (unsigned)(b >> 32), 0u, 0xC0);
  return (u64)lo | ((u64)hi << 32);
}

// 32-bit LDS byte address of a pointer into shared memory.
__device__ __forceinline__ unsigned lds_addr(const void* p) {
  return (unsigned)(size_t)(__attribute__((address_space(3))) const char*)p;
}

typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) const v4u lds_v4u;

__device__ __forceinline__ void split_masks(const u64 (&pend)[4], unsigned (&p)[8]) {
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    p[2 * m] = (unsigned)pend[m];
    p[2 * m + 1] = (unsigned)(pend[m] >> 32);
  }
}

__device__ __forceinline__ void join_masks(const unsigned (&p)[8], u64 (&pend)[4]) {
#pragma unroll
  for (int m = 0; m < 4; ++m) pend[m] = (u64)p[2 * m] | ((u64)p[2 * m + 1] << 32);
}

// Four masks, nibbles from 0, on the eight 32-bit halves p of the pending
// masks: the lookups of clear_supported_nib with the table addresses and the
// OR-and-clear written for the gfx950 ALU.  tab must be 256-byte aligned in
// LDS, so that the subset offset (16 bytes per subset) is ORed into the base
// with one three-input op ((x & vF0) | base, truth table 0xEA, vF0 = 0xF0)
// and the nibble's block offset rides in the read's immediate.  Per step of
// four lookups: 7 address ops and 16 mask ops, where the generic form takes
// 11 and 24.  live is the lane's any-pending flag: with kCheck a lane runs a
// step only while live (a live lane with no bits left in this half only
// looks up the zero subset) and live is recomputed after each step; without
// kCheck both steps run and live is computed once at the end (for the first
// half-word of a chunk, where some test of nearly every lane still lacks a
// support after 16 values).
template <bool kCheck>
__device__ __forceinline__ void nib4_run(unsigned (&p)[8], unsigned bits, const u64* tab, bool& live,
                                         unsigned vF0) {
  const unsigned base = lds_addr(tab);
#pragma unroll
  for (int q = 0; q < 8; q += 4) {
    if (kCheck && !live) break;
    v4u lo[4], hi[4];
    unsigned a[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int sh = 4 * (q + i) - 4;
      const unsigned x = sh >= 0 ? (bits >> sh) : (bits << 4);
      a[i] = __builtin_amdgcn_bitop3_b32(x, vF0, base, 0xEA) + (q + i) * 512;
      lo[i] = ((lds_v4u*)(size_t)a[i])[0];  // masks 0, 1 of the subset
    }
    p[0] = andnot_or4(p[0], lo[0].x, lo[1].x, lo[2].x, lo[3].x);
    p[1] = andnot_or4(p[1], lo[0].y, lo[1].y, lo[2].y, lo[3].y);
    p[2] = andnot_or4(p[2], lo[0].z, lo[1].z, lo[2].z, lo[3].z);
    p[3] = andnot_or4(p[3], lo[0].w, lo[1].w, lo[2].w, lo[3].w);
    // the second plane's reads after the first plane's ORs: eight reads in
    // flight at once hold 32 registers against the 64-register budget
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 4; ++i) hi[i] = ((lds_v4u*)(size_t)a[i])[16];  // masks 2, 3, 256 bytes on
    p[4] = andnot_or4(p[4], hi[0].x, hi[1].x, hi[2].x, hi[3].x);
    p[5] = andnot_or4(p[5], hi[0].y, hi[1].y, hi[2].y, hi[3].y);
    p[6] = andnot_or4(p[6], hi[0].z, hi[1].z, hi[2].z, hi[3].z);
    p[7] = andnot_or4(p[7], hi[0].w, hi[1].w, hi[2].w, hi[3].w);
    bits &= ~(0xffffu << (4 * q));
    if (kCheck) live = ((p[0] | p[1] | p[2] | p[3]) | (p[4] | p[5] | p[6] | p[7])) != 0u;
  }
  if (!kCheck) live = ((p[0] | p[1] | p[2] | p[3]) | (p[4] | p[5] | p[6] | p[7])) != 0u;
}

// nib4_run on the 64-bit pending masks (used by the byte-table variants for
// their upper half-words).
template <bool kCheck>
__device__ __forceinline__ void clear_supported_nib4(u64 (&pend)[4], unsigned bits, const u64* tab) {
  unsigned p[8];
  split_masks(pend, p);
  bool live = any_mask<4>(pend);
  nib4_run<kCheck>(p, bits, tab, live, 0xF0u);
  join_masks(p, pend);
}

template <int M, int Q0 = 0, bool kCheck = true>
__device__ __forceinline__ void clear_supported_nib(u64 (&pend)[M], unsigned bits, const u64* tab) {
  if constexpr (M == 4 && Q0 == 0 && kNibStep == 4) {
    clear_supported_nib4<kCheck>(pend, bits, tab);
    return;
  }
  for (int q = Q0; q < 8 && bits && any_mask<M>(pend); q += kNibStep) {
    u64 acc[M];
#pragma unroll
    for (int m = 0; m < M; ++m) acc[m] = 0ull;
#pragma unroll
    for (int i = 0; i < kNibStep; ++i) {
      const unsigned s = (bits >> (4 * (q + i))) & 15u;
      const u64* e = tab + nib_word<M>(q + i, (int)s, 0);
#pragma unroll
      for (int m = 0; m < M; ++m) acc[m] |= e[nib_word<M>(0, 0, m)];
    }
    bits &= ~(kNibStepMask << (4 * q));
#pragma unroll
    for (int m = 0; m < M; ++m) pend[m] &= ~acc[m];
  }
}

// Byte tables: entry (p, s) of byte p of word 0 holds the OR of the masks of
// the values 8p + i for the set bits i of s, so that one lookup covers 8
// values where a nibble table covers 4.  A support is usually found among the
// first few dozen values of a row (at tightness 0.5 a test keeps about half
// the values of each changed neighbour), so the tables cover the start of
// word 0 only; nibble tables cover the rest.  With four masks an entry is
// split in two 16-byte halves in separate planes, as in the nibble tables.
template <int M>
__device__ __forceinline__ int byte_word(int p, int sub, int mm) {
  if constexpr (M == 4) return p * 1024 + (mm >> 1) * 512 + sub * 2 + (mm & 1);
  else return (p * 256 + sub) * M + mm;
}

// Byte lookups per step: 3 for 6 tables, else 2.
__host__ __device__ constexpr int byte_step(int nb) { return nb % 3 == 0 ? 3 : 2; }

// pend[m] &= ~(masks of the supports among values 0 .. 8 NB - 1 of word 0);
// returns the row bits above them.
template <int M, int NB>
__device__ __forceinline__ u64 clear_supported_bytes(u64 (&pend)[M], u64 r, const u64* btab) {
  constexpr int S = byte_step(NB);
#pragma unroll
  for (int p = 0; p < NB; p += S) {
    if (!(r >> (8 * p)) || !any_mask<M>(pend)) break;
    u64 acc[M];
#pragma unroll
    for (int m = 0; m < M; ++m) acc[m] = 0ull;
#pragma unroll
    for (int i = 0; i < S; ++i) {
      if (p + i < NB) {
        const int sub = (int)((r >> (8 * (p + i))) & 255ull);
        const u64* e = btab + byte_word<M>(p + i, sub, 0);
#pragma unroll
        for (int m = 0; m < M; ++m) acc[m] |= e[byte_word<M>(0, 0, m)];
      }
    }
#pragma unroll
    for (int m = 0; m < M; ++m) pend[m] &= ~acc[m];
  }
  return r & ~((1ull << (8 * NB)) - 1ull);
}

// Nibble tables of a stage buffer with NB byte tables in front: nibble q of
// word 0 (q >= 2 NB) and every nibble of the later words sit where the
// nibble-only layout would put them, shifted back by the LDS the byte tables
// do not use.
template <int M, int NB>
__device__ __forceinline__ const u64* nib_base(const u64* stage) {
  return stage + (256ll * NB - 32ll * NB) * M;
}

// The M masks of one (variable, value) with plain vector loads (32 bytes for
// M = 4), issued together.
template <int M>
__device__ __forceinline__ void load_masks(const u64* p, u64 (&out)[M]) {
  if constexpr (M % 2 == 0) {
    const ulonglong2* q = reinterpret_cast<const ulonglong2*>(p);
#pragma unroll
    for (int h = 0; h < M / 2; ++h) {
      const ulonglong2 v = q[h];
      out[2 * h] = v.x;
      out[2 * h + 1] = v.y;
    }
  } else {
#pragma unroll
    for (int m = 0; m < M; ++m) out[m] = p[m];
  }
}

template <int M, bool kNib, int NB>
__device__ __forceinline__ bool wide_revise(const u64* __restrict__ plane_u, u64* slu, const u64* stage,
                                            const u64* atw, int W, int dpad, const u64 (&act)[M],
                                            bool touched_u, const u64* __restrict__ base_u,
                                            const u64 (&all)[M]) {
  const int lane = lane_id();
  bool changed = false;
  u64 aa[M];  // live tests of the group
#pragma unroll
  for (int m = 0; m < M; ++m) aa[m] = all[m] & act[m];
  const bool aa_any = any_mask<M>(aa);
  // the subset mask of the table addresses in a vector register: a
  // three-input op reads one scalar operand, and the table base is one
  unsigned vF0;
  asm volatile("v_mov_b32 %0, 0xf0" : "=v"(vF0));
  const u64 atw0 = atw[0];
  const int lane_hi = lane & 32;
  // word 0 of the next chunk's rows is loaded one chunk ahead, so that its
  // latency overlaps this chunk's lookups
  u64 row_next = plane_u[lane];
  for (int j = 0; j < W; ++j) {
    const int b = j * 64 + lane;
    const u64 row0 = row_next;
    if (j + 1 < W) row_next = plane_u[b + 64];
    // flip: all ones when b is a base value (a set slice bit flips the base
    // state), as one sign-extending bit-field extract
    const int flip32 = __builtin_amdgcn_sbfe((int)(unsigned)(base_u[j] >> lane_hi), lane & 31, 1);
    const bool in = flip32 != 0;
    const u64 flip = (u64)(long long)flip32;
    u64 pend[M];
    bool has;  // some test still holds b
    if (touched_u) {
      // plain loads, all M masks at once: another wave may be removing
      // values of u at the same time, and a load that misses those removals
      // only makes pend a superset of the live tests (the alive sets only
      // shrink), which costs lookups but not exactness, since a removal takes
      // the change from the atomic's returned word
      u64 sv[M];
      load_masks<M>(&slu[(long long)b * M], sv);
#pragma unroll
      for (int m = 0; m < M; ++m) pend[m] = xor_and64(sv[m], flip, aa[m]);
      has = any_mask<M>(pend);
    } else {
      // pend = aa for a base value, nothing otherwise; the four-mask path
      // starts from aa itself, inside the lanes that hold b
#pragma unroll
      for (int m = 0; m < M; ++m) pend[m] = (M == 4 && kNib && NB == 0) ? aa[m] : and64(flip, aa[m]);
      has = in && aa_any;
    }
    const u64* nib = nib_base<M, NB>(stage);
    bool live = has;  // some lane still holds a test without a support
    if constexpr (M == 4 && kNib && NB == 0) {
      // the four-mask path keeps live current after every step, so that
      // each step's test is computed once
      if (has) {
        unsigned p[8];
        split_masks(pend, p);
        const u64 r = row0 & atw0;
        nib4_run<false>(p, (unsigned)r, stage, live, vF0);
        nib4_run<true>(p, (unsigned)(r >> 32), stage + 128ll * M, live, vF0);
        for (int w = 1; w < W && live; ++w) {
          const u64 rw = plane_u[(long long)w * dpad + b] & atw[w];
          const u64* tb = stage + 256ll * w * M;
          nib4_run<true>(p, (unsigned)rw, tb, live, vF0);
          nib4_run<true>(p, (unsigned)(rw >> 32), tb + 128ll * M, live, vF0);
        }
        join_masks(p, pend);
      }
    } else if (has) {
      const u64 r = row0 & atw0;
      if (NB > 0) {
        const u64 rest = clear_supported_bytes<M, NB>(pend, r, stage);
        if (NB < 4) clear_supported_nib<M, 2 * NB>(pend, (unsigned)rest, nib);
        clear_supported_nib<M, (NB > 4 ? 2 * NB - 8 : 0)>(pend, (unsigned)(rest >> 32), nib + 128ll * M);
      } else if (kNib) {
        clear_supported_nib<M, 0, false>(pend, (unsigned)r, stage);
        clear_supported_nib<M>(pend, (unsigned)(r >> 32), stage + 128ll * M);
      } else {
        clear_supported_wide<M>(pend, (unsigned)r, stage + (long long)1 * M);
        clear_supported_wide<M>(pend, (unsigned)(r >> 32), stage + (long long)34 * M);
      }
    }
    if constexpr (!(M == 4 && kNib && NB == 0)) {
      for (int w = 1; w < W && any_mask<M>(pend); ++w) {
        const u64 r = plane_u[(long long)w * dpad + b] & atw[w];
        if (kNib) {
          const u64* tb = nib + 256ll * w * M;
          clear_supported_nib<M>(pend, (unsigned)r, tb);
          clear_supported_nib<M>(pend, (unsigned)(r >> 32), tb + 128ll * M);
        } else {
          const u64* st = stage + (long long)w * kStageWord * M;
          clear_supported_wide<M>(pend, (unsigned)r, st + (long long)1 * M);
          clear_supported_wide<M>(pend, (unsigned)(r >> 32), st + (long long)34 * M);
        }
      }
      live = any_mask<M>(pend);
    }
    if (live) {
#pragma unroll
      for (int m = 0; m < M; ++m) {
        if (pend[m]) {
          // removal: set the bit of a base value, clear that of a value a
          // test made present
          if (in) {
            const u64 old = or_wg(&slu[(long long)b * M + m], pend[m]);
            if (pend[m] & ~old) changed = true;
          } else {
            const u64 old = and_wg(&slu[(long long)b * M + m], ~pend[m]);
            if (pend[m] & old) changed = true;
          }
        }
      }
    }
  }
  return __ballot(changed) != 0ull;
}

// Most threads per workgroup of k_sliced_wide, and the waves per SIMD its
// register budget is set for: 8 (64 VGPRs) keeps two 1024-thread workgroups
// on every CU.  With 4 masks this spills a few registers and is still the
// fastest choice measured (11.5 ms against 13.6 ms at 512 threads and 80
// VGPRs for the 128,000-test pass).
constexpr int kWideMaxThreads = 1024;
constexpr int kWideWavesPerSimd = 8;

template <int M, bool kNib, int NB>
__global__ void __launch_bounds__(kWideMaxThreads, kWideWavesPerSimd) k_sliced_wide(DevNet net, const u64* __restrict__ base_dom,
                              const int2* __restrict__ tests, const int* __restrict__ gfirst,
                              const int* __restrict__ gorder, long long g0, const int* __restrict__ perm,
                              unsigned char* fail, unsigned long long* revs_out, u64* slices) {
  extern __shared__ __align__(16) char smem[];
  __shared__ WideCtl<M> ctl;
  const int n = net.n, W = net.W, dpad = net.dpad;
  const int nvw = (n + 31) / 32;
  const int tid = threadIdx.x, nthreads = blockDim.x;
  const int lane = lane_id();
  const int wave = uniform_int(tid >> 6), nwaves = nthreads >> 6;
  const int B = gridDim.x, bid = blockIdx.x;
  const int xcd = bid & 7, q = B >> 3, rem = B & 7;
  // slot of this workgroup (consecutive groups on one XCD), and its group
  const long long gs = g0 + (long long)xcd * q + (xcd < rem ? xcd : rem) + (bid >> 3);
  const long long g = gorder ? gorder[gs] : gs;
  const int tf = gfirst[g];
  const int tc = uniform_int(gfirst[g + 1] - tf);
  u64 all[M];
#pragma unroll
  for (int m = 0; m < M; ++m) {
    const int k = tc - 64 * m;
    all[m] = k >= 64 ? ~0ull : (k > 0 ? ((1ull << k) - 1ull) : 0ull);
  }
  u64* sl = slices + (long long)bid * n * dpad * M;

  int* list = (int*)smem;
  unsigned* cur = (unsigned*)(list + n);
  unsigned* nxt = cur + nvw;
  unsigned* touched = nxt + nvw;
  // the stage buffers start 256-byte aligned in LDS: the four-mask nibble
  // lookups OR the subset offset into the table base
  const unsigned smem0 = lds_addr(smem);
  const unsigned head_raw = (unsigned)((4ll * n + 12ll * nvw + 15) & ~15ll);
  const long long head = (long long)(((smem0 + head_raw + 255u) & ~255u) - smem0);
  u64* stage0 = (u64*)(smem + head);
  static_assert(NB == 0 || (kNib && NB <= 6), "byte tables go with nibble tables");
  const long long stage_words = wide_stage_words(W, M, kNib, NB);
  constexpr int nbuf = NB > 0 ? 1 : 2;  // double buffer without byte tables
  u64* atw0 = stage0 + nbuf * stage_words;

  for (int i = tid; i < nvw; i += nthreads) {
    cur[i] = 0u;
    nxt[i] = 0u;
    touched[i] = 0u;
  }
  // zero entries of every stage buffer (single-value layout only)
  for (int i = tid; !kNib && i < nbuf * 2 * W * M; i += nthreads) {
    const int m = i % M, k = i / M;  // k = buffer * 2W + entry
    const int buf = k / (2 * W), e = k % (2 * W);
    stage0[buf * stage_words + ((long long)(e >> 1) * kStageWord + 33 * (e & 1)) * M + m] = 0ull;
  }
  if (tid == 0) {
#pragma unroll
    for (int m = 0; m < M; ++m) ctl.act[m] = all[m];
    ctl.revs = 0;
  }
  __syncthreads();
  // test k reduces its variable x_k to {a_k}: flip every base value but a_k,
  // and a_k if it is not a base value.  The tests of a group come in runs of
  // one variable (the list is sorted by variable), so word (x, b, m) of the
  // slices is built whole by one thread from the 64 tests of mask m and
  // stored once: no atomics (one per flipped value and test, 64 to a word,
  // took a sixth of the pass).
  for (int w = tid; w < dpad * M; w += nthreads) {
    const int m = (w >> 6) % M;  // uniform: nthreads is a multiple of 64
    const int b = ((w >> 6) / M) * 64 + (w & 63);
    const int kend = min(tc, 64 * (m + 1));
    int x = -1;
    bool in = false;
    u64 word = 0ull;
    for (int k = 64 * m; k < kend; ++k) {
      const int2 tk = tests[tf + k];
      if (tk.x != x) {
        if (word) sl[((long long)x * dpad + b) * M + m] = word;
        x = tk.x;
        word = 0ull;
        in = (base_dom[(long long)x * W + (b >> 6)] >> (b & 63)) & 1ull;
      }
      if (in != (b == tk.y)) word |= 1ull << (k & 63);
    }
    if (word) sl[((long long)x * dpad + b) * M + m] = word;
  }
  if (tid < tc) {
    const int x = tests[tf + tid].x;
    atomicOr(&cur[x >> 5], 1u << (x & 31));
    atomicOr(&touched[x >> 5], 1u << (x & 31));
  }
  __syncthreads();

  unsigned long long revs = 0;
  for (int round = 0;; ++round) {
    const int slot = round & 1;
    if (wave == 0) {
      int base = 0;
      for (int v0 = 0; v0 < n; v0 += 64) {
        const int v = v0 + lane;
        const bool f = v < n && bit_of(cur, v);
        const u64 mask = __ballot(f);
        if (f) list[base + mbcnt(mask)] = v;
        base += __popcll(mask);
      }
      if (lane == 0) {
        ctl.m = base;
        ctl.nchanged[slot] = 0;
      }
    } else {
      for (int i = tid - 64; i < nvw; i += nthreads - 64) nxt[i] = 0u;
    }
    if (nthreads == 64)
      for (int i = lane; i < nvw; i += 64) nxt[i] = 0u;
    __syncthreads();
    const int mcount = uniform_int(ctl.m);
    u64 act[M];
#pragma unroll
    for (int m = 0; m < M; ++m) act[m] = (u64)uniform_ll((long long)ctl.act[m]);
    for (int i = 0; i < mcount; ++i) {
      const int t = uniform_int(list[i]);
      // one buffer: every wave finishes the previous variable's arcs first
      if (nbuf == 1 && i > 0) __syncthreads();
      u64* stage = stage0 + (i & (nbuf - 1)) * stage_words;
      u64* atw = atw0 + (i & (nbuf - 1)) * W;
      // stage t: thread v holds value v's M masks; one wave covers one word
      const u64* slt = sl + (long long)t * dpad * M;
      const u64* base_t = base_dom + (long long)t * W;
      // masks of value v of t: the live tests that still hold it.  Plain
      // loads, issued together: a wave still revising the previous
      // variable's arcs may remove values of t meanwhile, and a stage that
      // misses such a removal only keeps a support too many; t is then
      // marked changed and staged again next round.
      auto alive_of = [&](int v, int mm) -> u64 {
        const u64 flip = ((base_t[v >> 6] >> (v & 63)) & 1ull) ? ~0ull : 0ull;
        const int kk = tc - 64 * mm;
        const u64 all_m = kk >= 64 ? ~0ull : (kk > 0 ? ((1ull << kk) - 1ull) : 0ull);
        return all_m & (slt[(long long)v * M + mm] ^ flip);
      };
      // the same from a slice word already loaded
      auto alive_bits = [&](u64 raw, int v, int mm) -> u64 {
        const u64 flip = ((base_t[v >> 6] >> (v & 63)) & 1ull) ? ~0ull : 0ull;
        const int kk = tc - 64 * mm;
        const u64 all_m = kk >= 64 ? ~0ull : (kk > 0 ? ((1ull << kk) - 1ull) : 0ull);
        return all_m & (raw ^ flip);
      };
      // every wave finished the arcs of this buffer's previous variable
      // before the last barrier
      if (tid == 0) ctl.arc_ctr[i & 1] = 0;
      if (kNib) {
        // nibble tables: item (q, m) ORs the 16 subsets of values 4q..4q+3
        // (nibbles from 2 NB on); byte tables: item (p, m, h) fills the 16
        // subsets of byte p whose high nibble is h
        u64* nib = stage + (256ll * NB - 32ll * NB) * M;
        const int nib_items = (16 * W - 2 * NB) * M;
        for (int it = tid; it < nib_items + NB * M * 16; it += nthreads) {
          if (it < nib_items) {
            const int q = 2 * NB + it / M, mm = it % M;
            u64 x[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = slt[(long long)(4 * q + i) * M + mm];
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = alive_bits(x[i], 4 * q + i, mm);
#pragma unroll
            for (int sub = 0; sub < 16; ++sub) {
              u64 o = 0ull;
#pragma unroll
              for (int i = 0; i < 4; ++i)
                if (sub & (1 << i)) o |= x[i];
              nib[nib_word<M>(q, sub, mm)] = o;
            }
          } else {
            const int k = it - nib_items;
            const int h = k & 15, mm = (k >> 4) % M, p = (k >> 4) / M;
            u64 x[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = alive_of(8 * p + i, mm);
            u64 hi = 0ull;
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (h & (1 << i)) hi |= x[4 + i];
#pragma unroll
            for (int lo = 0; lo < 16; ++lo) {
              u64 o = hi;
#pragma unroll
              for (int i = 0; i < 4; ++i)
                if (lo & (1 << i)) o |= x[i];
              stage[byte_word<M>(p, (h << 4) | lo, mm)] = o;
            }
          }
        }
      }
      // the alive-any words from the waves after the table items when there
      // are enough of them, so that the two sets of slice reads overlap
      const int items = kNib ? (16 * W - 2 * NB) * M + NB * M * 16 : 0;
      const int abase = ((items + 63) & ~63) + dpad <= nthreads ? ((items + 63) & ~63) : 0;
      for (int v = tid - abase; tid >= abase && v < dpad; v += nthreads) {
        u64 alive = 0ull;
        u64* dst = stage + (long long)stage_pos(v) * M;
        u64 sv[M];
        load_masks<M>(&slt[(long long)v * M], sv);
        const u64 flip = ((base_t[v >> 6] >> (v & 63)) & 1ull) ? ~0ull : 0ull;
#pragma unroll
        for (int m = 0; m < M; ++m) {
          const u64 x = all[m] & (sv[m] ^ flip);
          if (!kNib) dst[m] = x;
          alive |= x & act[m];
        }
        const u64 word = __ballot(alive != 0ull);
        if (lane == 0) atw[v >> 6] = word;
      }
      __syncthreads();
      const int a0 = net.adj_off[t], deg = net.adj_off[t + 1] - a0;
      // waves take t's arcs one at a time from a shared counter
      while (true) {
        int j = 0;
        if (lane == 0) j = atomicAdd(&ctl.arc_ctr[i & 1], 1);
        j = __builtin_amdgcn_readfirstlane(j);
        if (j >= deg) break;
        const int4 e = net.adj[a0 + j];
        const int u = uniform_int(e.y);
        const int pos_t = uniform_int(adj_pos(e));
        const long long o = (long long)uniform_int(e.w) * 2 * W * dpad;
        const u64* plane_u = net.sup + o + (long long)(1 - pos_t) * W * dpad;
        const bool tu = uniform_int((int)bit_of(touched, u));
        const bool ch = wide_revise<M, kNib, NB>(plane_u, sl + (long long)u * dpad * M, stage, atw, W, dpad, act,
                                             tu, base_dom + (long long)u * W, all);
        ++revs;
        if (ch && lane == 0) {
          const unsigned bit = 1u << (u & 31);
          const unsigned old = atomicOr(&nxt[u >> 5], bit);
          if (!(old & bit)) atomicAdd(&ctl.nchanged[slot], 1);
        }
      }
    }
    __syncthreads();
    // exact wipe-out check: a test wiped out at v only if v changed
    u64 alive_all[M];
#pragma unroll
    for (int m = 0; m < M; ++m) alive_all[m] = ~0ull;
    for (int v = wave; v < n; v += nwaves) {
      if (!uniform_int((int)bit_of(nxt, v))) continue;
      // a lane reads the M masks of its values together, every read of the
      // variable in flight at once
      u64 o[M];
#pragma unroll
      for (int m = 0; m < M; ++m) o[m] = 0ull;
      for (int b = lane; b < dpad; b += 64) {
        const u64 flip = ((base_dom[(long long)v * W + (b >> 6)] >> (b & 63)) & 1ull) ? ~0ull : 0ull;
        u64 sv[M];
        load_masks<M>(&sl[((long long)v * dpad + b) * M], sv);
#pragma unroll
        for (int m = 0; m < M; ++m) o[m] |= all[m] & (sv[m] ^ flip);
      }
#pragma unroll
      for (int m = 0; m < M; ++m) alive_all[m] &= wave_or64_dpp(o[m]);
    }
    if (lane == 0) {
#pragma unroll
      for (int m = 0; m < M; ++m)
        if (alive_all[m] != ~0ull) atomicAnd(&ctl.act[m], alive_all[m]);
    }
    for (int i = tid; i < nvw; i += nthreads) touched[i] |= nxt[i];
    __syncthreads();
    u64 act_any = 0ull;
#pragma unroll
    for (int m = 0; m < M; ++m) act_any |= (u64)uniform_ll((long long)ctl.act[m]);
    if (uniform_int(ctl.nchanged[slot]) == 0 || act_any == 0ull) break;
    unsigned* tmp = cur;
    cur = nxt;
    nxt = tmp;
  }
  if (lane == 0 && revs) atomicAdd(&ctl.revs, revs);
  __syncthreads();
  if (tid < tc)
    fail[perm ? perm[tf + tid] : tf + tid] = ((ctl.act[tid >> 6] >> (tid & 63)) & 1ull) ? 0 : 1;
  if (tid == 0 && ctl.revs) atomicAdd(&revs_out[blockIdx.x % kStatSlots], ctl.revs);
  // leave the region all zero: clear the slices of every variable written
  for (int v = wave; v < n; v += nwaves) {
    if (!uniform_int((int)bit_of(touched, v))) continue;
    u64* p = sl + (long long)v * dpad * M;
    for (int i = lane; i < dpad * M; i += 64) p[i] = 0ull;
  }
}

// ---------------------------------------------------------------------------
// Device MAC (binary branching, dom-min over undecided variables with the
// lowest id on ties, min value), CPU MAC::enforce semantics
// (src/MAC.cpp:100-165).  The trail holds the domain of every depth: a
// positive decision at depth L saves the current domain in trail[L]; on
// failure the domain is restored from trail[L], the value removed, and the
// negative decision propagated at depth L.  The state can be suspended after
// `step_budget` nodes and resumed by a later launch (serving).
// ---------------------------------------------------------------------------
struct MacState {
  int status;  // 0 init, 1 running, 2 solution, 3 unsat or enumeration done, 4 limit reached
  int depth;
  long long npos;
  long long nneg;
  long long revisions;
  int trace_len;
  int steps;
  long long nsol;  // solutions found so far
};

struct NodeRec {
  int positive;
  int var;
  int value;
  int consistent;
  u64 dom_hash;
};

// A copy of a network laid out as it sits in LDS behind the working memory:
// adjacency offsets, adjacency, constraint metadata, support planes, tables.
// The value stride of the planes and tables is cut from dpad (64 W) to dc,
// the largest domain rounded up to an odd number, and the constraint offsets
// follow that stride.  Odd, because the lanes of a wave read the same value's
// rows of different planes: with an even stride of 16 or 32 words they would
// all meet on the same LDS banks.  The
// planes are followed by 64 W words of zeros: a target-side revision loads
// whole 64-value chunks of a row, and the lanes past dc (values that are
// never live) must still read inside the image.  bytes = 0: no image.
struct LdsNet {
  const uint4* src;  // device copy of the image
  int bytes;         // multiple of 16
  int dc;
  int o_adj, o_con, o_sup, o_tsup, o_tabs;  // byte offsets in the image
  // wg_fixpoint_flat: the smallest workgroup that can run it (0: none can) and
  // the largest that its arcs and tables fill
  int flat_min, flat_threads;
};

// Copies the image behind the working memory (at dst) and returns the
// network whose arrays are those LDS copies.  Called by every thread.
__device__ __forceinline__ DevNet wg_load_net(const DevNet& g, const LdsNet& L, char* dst) {
  uint4* d4 = (uint4*)dst;
  for (int i = threadIdx.x; i < (L.bytes >> 4); i += blockDim.x) d4[i] = L.src[i];
  __syncthreads();
  DevNet ln = g;
  ln.dpad = L.dc;
  ln.adj_off = (const int*)dst;
  ln.adj = (const int4*)(dst + L.o_adj);
  ln.con = (const ConMeta*)(dst + L.o_con);
  ln.sup = (const u64*)(dst + L.o_sup);
  ln.tsup = (const u64*)(dst + L.o_tsup);
  ln.tabs = (const int*)(dst + L.o_tabs);
  return ln;
}

struct MacArgs {
  MacState* state;
  u64* trail;          // [n + 1][n][W]; trail[0] holds the start domains
  int2* stack;         // [n]
  int* solution;       // [sol_cap][n] or NULL: solution k at solution + k n
  long long sol_cap;   // solutions the buffer holds (0 counts as 1)
  // 0 or 1: stop at the first solution; k > 1: count every solution, treat it
  // as a failed node and go on, until the tree is exhausted or k are found
  long long max_solutions;
  NodeRec* trace;      // [trace_cap] or NULL
  int trace_cap;
  long long node_limit;   // total (0 = none)
  long long step_budget;  // per launch (0 = none)
  u64 deadline;           // wall_clock64 ticks (0 = none)
  u64* root_out;          // [n][W] root-fixpoint domains, or NULL
  const int* nbr;         // [n] neighbour counts: dom/deg ordering; NULL = dom-min
  // dom/wdeg ordering (all NULL otherwise); wipe-outs are then repeated in
  // AC3's schedule so that the weights grow as the reference's do
  float* weight;          // [ncons] constraint weights, start at 1
  int* stamp_tab;         // [ncons] constraint stamps, where they do not go in LDS
  int stamp_off;          // byte offset of the constraint stamps in dynamic LDS, 0 = stamp_tab
};

enum { MAC_INIT = 0, MAC_RUNNING = 1, MAC_SAT = 2, MAC_UNSAT = 3, MAC_LIMIT = 4 };

// Records node number *len of the search (wave 0; the domains must not change
// until the workgroup's next barrier).
__device__ __forceinline__ void wg_trace(const DevNet& net, const WgMem& mem, const MacArgs& A, int* len, int positive,
                                         int var, int val, bool ok) {
  if (!A.trace) return;
  const int tl = *len;
  *len = tl + 1;
  if (tl >= A.trace_cap || threadIdx.x >= 64) return;
  u64 h = 0ull;
  if (ok) {
    for (int i = lane_id(); i < net.n * net.W; i += 64) h += mix64(mem.dom[i] + (u64)i * 0x9E3779B97F4A7C15ull);
    h = wave_sum64_dpp(h);
  }
  if (threadIdx.x == 0) {
    NodeRec r;
    r.positive = positive;
    r.var = var;
    r.value = val;
    r.consistent = ok ? 1 : 0;
    r.dom_hash = h;
    A.trace[tl] = r;
  }
}

// ---------------------------------------------------------------------------
// AC3 in the reference's schedule (AC3::enforce, src/AC3.cpp:99-141, with the
// duplicate-free FIFO var_que, src/Solver.cpp:180-218), run by one wave over
// the workgroup's domains.  The closure equals that of any other schedule;
// what the order fixes is which constraint empties a domain first, and that
// constraint's weight is raised (AC3.cpp:122-126): the input of the dom/wdeg
// ordering.
//
// The queue (ring of n + 1), the queued flags and the variable stamps use
// pre, the second frontier bitmap and list, which this schedule does not
// otherwise need.  Variable and constraint stamps restart at 0 on each call,
// as in the reference; the constraint stamps lie in LDS where they fit.
// Lane 0 does every load and store of the control state and broadcasts what
// it read, so the same code is correct whether the arrays are in LDS or in
// global scratch; control values are wave-uniform.
//
// Networks without parallel binary constraints (net.simple) revise up to 64
// of x's constraints at once.  The other variables of those constraints are
// distinct and D(x) is fixed until a revision takes values of x, so the
// revisions are independent and are all computed from the state before the
// first; they are then committed in list order (queue positions and stamps
// from the lanes' ranks) up to the first that takes values of x, or the first
// wipe-out, whose constraint gains the weight.  One after another they cost
// about 3.5 us each, a chain of dependent reads; a batch costs about 3.2 us.
// 100 nodes of 100 variables (domains of 50, 742 constraints) took 11.1 ms
// with the constraint that takes values of x revised by itself after its
// batch, and 7.3 ms with it committed as the batch's last.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int lane0_load(const int* p) {
  int v = 0;
  if (lane_id() == 0) v = *p;
  return __builtin_amdgcn_readlane(v, 0);
}

typedef int v4i __attribute__((ext_vector_type(4)));

// Adjacency entry k of a list that ends at k1; no arc past the end.  (A plain
// vector: the runtime's int4 class goes through scratch memory when a value is
// chosen between two.)
__device__ __forceinline__ v4i load_arc(const int4* adj, int k, int k1) {
  v4i e = {0, -1, 0, 0};
  if (k < k1) e = *(const v4i*)(adj + k);
  return e;
}

__device__ __forceinline__ bool wave_ac3(const DevNet& net, WgMem mem, const MacArgs& A, int seed,
                         unsigned long long* revs) {
  const int n = net.n;
  const int lane = lane_id();
  const int nvw = (n + 31) / 32;
  const int qcap = n + 1;
  int* q = mem.pre;
  unsigned* inq = mem.bm + nvw;
  int* sv = mem.list;
  int front = 0, rear = 0, t = 0;
  if (seed >= 0) {
    for (int v = lane; v < n; v += 64) sv[v] = 0;
    for (int i = lane; i < nvw; i += 64) inq[i] = 0u;
  } else {
    for (int v = lane; v < n; v += 64) {
      q[v] = v;
      sv[v] = v + 1;
    }
    for (int i = lane; i < nvw; i += 64) {
      const int k = n - 32 * i;
      inq[i] = k >= 32 ? 0xffffffffu : ((1u << k) - 1u);
    }
    rear = n;
    t = n;
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
  __builtin_amdgcn_wave_barrier();
  auto insert = [&](int v) {
    const int word = lane0_load((const int*)&inq[v >> 5]);
    if (!((word >> (v & 31)) & 1)) {
      if (lane == 0) {
        q[rear] = v;
        inq[v >> 5] = (unsigned)word | (1u << (v & 31));
      }
      rear = rear + 1 == qcap ? 0 : rear + 1;
    }
    ++t;
    if (lane == 0) sv[v] = t;
  };
  if (seed >= 0) insert(seed);
  bool ok = true;
  unsigned long long nrev = 0;
  const int W = net.W;
  int lw = 0;
  while ((1 << lw) < W) ++lw;
  const int w = lane & ((1 << lw) - 1), la = lane >> lw, per = 64 >> lw;
  const long long pair_words = 2ll * W * net.dpad;
  // pred in some lane of an arc, as a mask with one bit per arc (bit 0 of its lanes)
  u64 arc_bits = 1ull;
  for (int d = 1 << lw; d < 64; d <<= 1) arc_bits |= arc_bits << d;
  auto arcs_with = [&](bool pred) -> u64 {
    u64 m = __ballot(pred);
    for (int d = (1 << lw) >> 1; d > 0; d >>= 1) m |= m >> d;
    return m & arc_bits;
  };
  int next_x = -1, next_k0 = 0, next_k1 = 0;
  v4i next_e = {0, -1, 0, 0};
  while (ok && front != rear) {
    const int x = lane0_load(&q[front]);
    front = front + 1 == qcap ? 0 : front + 1;
    if (lane == 0) inq[x >> 5] &= ~(1u << (x & 31));
    // x's constraints; those of the next variable in the queue, if there is
    // one, are read ahead
    const bool read_ahead = x == next_x;
    const int k0 = read_ahead ? next_k0 : uniform_int(mem.aoff[x]);
    const int k1 = read_ahead ? next_k1 : uniform_int(mem.aoff[x + 1]);
    v4i first_e = next_e;
    if (!read_ahead) first_e = load_arc(mem.adj, k0 + la, k1);
    next_x = -1;
    if (net.simple && front != rear) {
      next_x = lane0_load(&q[front]);
      next_k0 = uniform_int(mem.aoff[next_x]);
      next_k1 = uniform_int(mem.aoff[next_x + 1]);
      next_e = load_arc(mem.adj, next_k0 + la, next_k1);
    }
    const bool asgx = uniform_int((int)bit_of(mem.asg, x)) != 0;
    for (int k = k0; k < k1; ++k) {
      if (net.simple) {
        // the constraints k .. k + per - 1 at once, from the state before the
        // first of them: exact up to and with the first one that takes values
        // of x (the later ones then see another D(x)), before the first table,
        // and up to the first wipe-out
        const bool in = k + la < k1 && la < per && w < W;
        v4i e = first_e;
        if (k != k0) e = load_arc(mem.adj, k + la, k1);
        const bool table = in && e.y < 0;
        const int y = in && !table ? e.y : x;
        const int px = (e.z & 15);
        const int stc = in ? ld_wg_int(&mem.stamp[e.x]) : 0;
        const int svx = ld_wg_int(&sv[x]), svy = ld_wg_int(&sv[y]);
        u64* ydom = mem.dom + (long long)y * W + w;
        const u64 dy = in && !table ? ld_wg(ydom) : 0ull;
        const bool act = in && !table && svx > stc;
        const bool yrev = act && !bit_of(mem.asg, y);
        const long long off = in && !table ? e.w * pair_words : 0ll;
        const u64 need = yrev ? dy : 0ull;
        const u64 gone = wave_unsupported<false>(net, mem.dom, x, net.sup + off + (long long)(px * W + w) * net.dpad,
                                                 net.sup + off + (long long)(1 - px) * W * net.dpad + 64 * w, need);
        const int bit0 = la << lw;
        const u64 lose = arcs_with(gone != 0ull);
        const u64 wipe_y = lose & ~arcs_with((need & ~gone) != 0ull);
        const bool mine_lose = (lose >> bit0) & 1ull;
        // x <- y: when y changed since the constraint's stamp, or lost values
        // just now.  Neither direction sees the other's removals: a value
        // removed for want of a support supported nothing there.
        const bool xrev = act && !asgx && (svy > stc || (px == 1 && mine_lose && !((wipe_y >> bit0) & 1ull)));
        const u64 dx = xrev ? ld_wg(&mem.dom[(long long)x * W + w]) : 0ull;
        const u64 xgone = arcs_unsupported<false, false>(net, mem.dom, off, y, 1 - px, in ? w : 0, dx);
        const u64 xlose = arcs_with(xgone != 0ull), tabs = arcs_with(table), acts = arcs_with(act);
        const u64 wipe = wipe_y | (xlose & ~arcs_with((dx & ~xgone) != 0ull));
        const u64 halt = xlose | tabs | wipe;
        const int stop = halt ? (int)__builtin_ctzll(halt) : 64;  // bit of the arc that ends the batch
        const u64 at = stop < 64 ? 1ull << stop : 0ull;
        const bool wiped = (wipe & at) != 0ull, last = !wiped && (xlose & at) != 0ull;
        // the arcs before it are committed, and that arc itself but for a table
        const u64 before = stop >= 64 ? ~0ull : (at - 1ull) | (tabs & at ? 0ull : at);
        const u64 done = acts & before, ins = lose & before;
        const bool commit = act && ((before >> bit0) & 1ull);
        const bool mine_last = last && bit0 == stop;
        if (commit && gone) {
          (void)and_wg(ydom, ~gone);
          atomicSub(&mem.size[y], __popcll(gone));
        }
        if (mine_last && xgone) {
          (void)and_wg(&mem.dom[(long long)x * W + w], ~xgone);
          atomicSub(&mem.size[x], __popcll(xgone));
        }
        // (a wipe-out ends its constraint with the first of the two revisions)
        const bool counted = commit && !(wiped && bit0 == stop);
        nrev += __popcll(arcs_with(yrev && counted)) + __popcll(arcs_with(xrev && counted)) + (wiped ? 1 : 0);
        if (wiped) {
          const int cw = __builtin_amdgcn_readlane(e.x, stop);
          if (lane == 0) A.weight[cw] += 1.0f;
          ok = false;
          break;
        }
        // times: an arc's removals, then its stamp; of the last arc, the first
        // position's variable first
        const u64 below = (1ull << bit0) - 1ull;
        const int t0 = t + __popcll(done & below) + __popcll(ins & below);
        const int y_late = mine_last && px == 0 ? 1 : 0, x_late = mine_last && px == 1 && mine_lose ? 1 : 0;
        if (commit && w == 0) {
          __hip_atomic_store(&mem.stamp[e.x], t0 + 1 + (mine_lose ? 1 : 0) + (mine_last ? 1 : 0), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_WORKGROUP);
          if (mine_lose) __hip_atomic_store(&sv[y], t0 + 1 + y_late, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          if (mine_last) __hip_atomic_store(&sv[x], t0 + 1 + x_late, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        const bool queued = (ld_wg_int((const int*)&inq[y >> 5]) >> (y & 31)) & 1;
        const bool xqueued = (ld_wg_int((const int*)&inq[x >> 5]) >> (x & 31)) & 1;
        const u64 add = arcs_with(commit && mine_lose && !queued);
        const int xadd = last && !xqueued ? 1 : 0;
        auto put = [&](int rank, int v) {
          int pos = rear + rank;
          pos = pos >= qcap ? pos - qcap : pos;
          __hip_atomic_store(&q[pos], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          atomicOr(&inq[v >> 5], 1u << (v & 31));
        };
        const int rank = __popcll(add & below);
        if (commit && mine_lose && !queued && w == 0) put(rank + (y_late && xadd ? 1 : 0), y);
        if (mine_last && xadd && w == 0) put(rank + (x_late && ((add >> bit0) & 1ull) ? 1 : 0), x);
        const int adds = __popcll(add) + (int)uniform_int(xadd);
        rear += adds;
        rear = rear >= qcap ? rear - qcap : rear;
        t += __popcll(done) + __popcll(ins) + (last ? 1 : 0);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        k += stop >= 64 ? per : (stop >> lw) + (last ? 1 : 0);
        if (stop >= 64 || last || k >= k1) {
          --k;
          continue;
        }
        // constraint k is a table: by itself
      }
      const int c = uniform_int(mem.adj[k].x);
      const int stc = lane0_load(&mem.stamp[c]);
      if (!(lane0_load(&sv[x]) > stc)) continue;
      const ConMeta* mp = net.con + c;
      const int arity = mp->arity;
      for (int i = 0; i < arity; ++i) {
        const int y = mp->scope[i];
        if (bit_of(mem.asg, y)) continue;
        bool aa = false;
        for (int j = 0; j < arity; ++j) {
          const int z = mp->scope[j];
          if (z != x && lane0_load(&sv[z]) > stc) aa = true;
        }
        if (y == x && !aa) continue;
        bool wiped = false;
        int removed = 0;
        if (mp->kind == 0) {
          removed = revise_binary_at(net, mem.dom, mem.size, mp->off, y, mp->scope[1 - i], 1 - i, &wiped);
        } else {
          revise_table(net, mem.dom, mem.size, c, -1, nullptr, [&](int, int r) { removed += r; }, &wiped, y);
        }
        ++nrev;
        if (removed > 0) {
          if (wiped) {
            if (lane == 0) A.weight[c] += 1.0f;
            ok = false;
            break;
          }
          insert(y);
        }
      }
      if (!ok) break;
      ++t;
      if (lane == 0) mem.stamp[c] = t;
    }
  }
  *revs += nrev;
  return ok;
}

// AC3-scheduled fixpoint for the whole workgroup: wave 0 runs it, the other
// waves wait at the barrier.
__device__ __forceinline__ bool wg_ac3(const DevNet& net, WgMem mem, WgCtl* ctl, const MacArgs& A, int seed) {
  for (int i = threadIdx.x; i < net.ncons; i += blockDim.x) mem.stamp[i] = 0;
  __syncthreads();
  if (threadIdx.x < 64) {
    unsigned long long revs = 0;
    const bool ok = wave_ac3(net, mem, A, seed, &revs);
    if (threadIdx.x == 0) {
      ctl->ok = ok ? 1 : 0;
      ctl->revs += revs;
    }
  }
  __syncthreads();
  return uniform_int(ctl->ok) != 0;
}

// MAC::select_var VRH_DOM_WDEG_MIN (src/MAC.cpp:386-411): for each undecided
// x, x_w = the sum of the weights of the constraints on x that have another
// undecided variable; key = -1 when |D(x)| = 1 or x_w = 0, else |D(x)| / x_w
// in double (IEEE division, as on the host); the lowest id among the smallest
// keys.  Non-negative doubles order as their bit patterns, -1 maps to 0.
// A row of 16 lanes sums the weights of one variable's constraints (whole
// numbers, so the sum is exact in any order).
__device__ __forceinline__ int wg_select_wdeg(const DevNet& net, const WgMem& mem, WgCtl* ctl, const MacArgs& A) {
  const int n = net.n, row = threadIdx.x >> 4, rows = blockDim.x >> 4, l = threadIdx.x & 15;
  u64 best = ~0ull;
  int bv = n;
  for (int v = row; v < n; v += rows) {
    const bool open = !bit_of(mem.asg, v);
    u64 sum = 0ull;
    const int k1 = open ? mem.aoff[v + 1] : 0;
    for (int k = open ? mem.aoff[v] + l : 0; k < k1; k += 16) {
      const int4 e = mem.adj[k];
      const float weight = A.weight[e.x];
      int cnt = 0;
      if (e.y >= 0) {
        cnt = 1 + (bit_of(mem.asg, e.y) ? 0 : 1);
      } else {
        const ConMeta* mp = net.con + e.x;
        for (int i = 0; i < mp->arity; ++i) cnt += bit_of(mem.asg, mp->scope[i]) ? 0 : 1;
      }
      if (cnt > 1) sum += (u64)weight;
    }
    sum += dpp_ror_u64_1(sum);
    sum += dpp_ror_u64_2(sum);
    sum += dpp_ror_u64_4(sum);
    sum += dpp_ror_u64_8(sum);
    if (!open) continue;
    const double xw = (double)sum;
    const int sz = mem.size[v];
    const double key = (sz == 1 || xw == 0.0) ? -1.0 : (double)sz / xw;
    const u64 k = key < 0.0 ? 0ull : (u64)__double_as_longlong(key);
    if (k < best) {
      best = k;
      bv = v;
    }
  }
  const u64 m = wg_reduce_min_u64(ctl, best);
  return (int)wg_reduce_min_u64(ctl, best == m ? (u64)bv : ~0ull);
}

// Loads one level of the trail into the working memory, less value skip_val
// of variable skip_var (skip_var < 0: nothing), and counts the sizes.
__device__ __forceinline__ void wg_load_level(const WgMem& mem, const u64* level, int n, int W, int skip_var,
                                              int skip_val) {
  for (int v = threadIdx.x; v < n; v += blockDim.x) {
    int size = 0;
    for (int w = 0; w < W; ++w) {
      u64 d = level[(long long)v * W + w];
      if (v == skip_var && w == (skip_val >> 6)) d &= ~(1ull << (skip_val & 63));
      mem.dom[(long long)v * W + w] = d;
      size += __popcll(d);
    }
    mem.size[v] = size;
  }
}

// The search.  Its control lives in registers, identical in every thread
// (every value below is wave-uniform); LDS holds the domains, the frontier
// and the decision stack.  One loop with one fixpoint in it: `phase` says
// what the fixpoint propagates (the root, a decision x = a, a refutation
// x != a).  A decision costs two barriers (one with kFlat) and a refutation
// one, beside the fixpoint's own.  kWdeg: dom/wdeg ordering, wipe-outs
// repeated in AC3's order.  kFlat: wg_fixpoint_flat propagates, and a
// refutation that follows its decision takes the domains from registers (dom
// and dom/deg only).  kFull: wg_fixpoint's kTight and kTabs.
template <bool kWdeg, bool kFlat, bool kFull>
__device__ __forceinline__ void wg_mac_run(const DevNet& net, const WgMem& mem, WgCtl* ctl, const MacArgs& A) {
  enum { ROOT, POSITIVE, NEGATIVE };
  const int n = net.n, W = net.W;
  const int nvw = (n + 31) / 32;
  const int tid = threadIdx.x, nthreads = blockDim.x, lane = lane_id();
  const long long nw = (long long)n * W;
  int status = uniform_int(A.state->status);
  int depth = uniform_int(A.state->depth);
  long long npos = uniform_ll(A.state->npos);
  long long nneg = uniform_ll(A.state->nneg);
  long long nsol = uniform_ll(A.state->nsol);
  int trace_len = uniform_int(A.state->trace_len);
  long long nodes_here = 0;
  // the stack in use: AC3's queue and stamps take list and pre under dom/wdeg
  int2* stk = kWdeg ? A.stack : (int2*)mem.list;
  int slot = 0, phase = ROOT, x = -1, a = 0;
  bool select = false;  // the domains are consistent: take the next decision
  FlatNet flat{};
  FlatSeen seen{};
  int turn = 0, flat_revs = 0;
  unsigned saved = 0u, dx = 0u;  // before the last decision: D(tid), D(x)
  if constexpr (kFlat) flat = wg_load_flat(net, mem);
  if (tid == 0) {
    ctl->revs = 0;
    if (kFlat) ctl->flat[0] = make_int2(0, 0);
  }
  wg_clear_bitmap(mem.asg, nvw);
  if (status == MAC_INIT) {
    wg_load_level(mem, A.trail, n, W, -1, 0);
    if (!kFlat) wg_seed(mem, ctl, n, slot, -1);
    status = MAC_RUNNING;
    if constexpr (kFlat) {
      __syncthreads();
      wg_flat_see(mem, flat, seen);
    }
  } else if (status == MAC_RUNNING) {
    wg_load_level(mem, A.trail + depth * nw, n, W, -1, 0);
    if (!kWdeg)
      for (int i = tid; i < depth; i += nthreads) stk[i] = A.stack[i];
    select = true;
  }
  __syncthreads();
  if (select) {
    for (int i = tid; i < depth; i += nthreads) {
      const int v = A.stack[i].x;
      atomicOr(&mem.asg[v >> 5], 1u << (v & 31));
    }
    __syncthreads();
    if constexpr (kFlat) {
      wg_flat_see(mem, flat, seen);
      __syncthreads();
    }
  }
  while (status == MAC_RUNNING) {
    if (select) {
      const bool over_nodes = A.node_limit > 0 && npos + nneg >= A.node_limit;
      const bool over_time = A.deadline && uniform_ll((long long)wall_clock64()) > (long long)A.deadline;
      if (over_nodes || over_time || (A.step_budget > 0 && nodes_here >= A.step_budget)) {
        // suspend (step budget) or stop (limits) at a consistent state of depth `depth`
        wg_copy_words(A.trail + depth * nw, mem.dom, nw);
        if (over_nodes || over_time) status = MAC_LIMIT;
        break;
      }
      // select: min key over undecided variables, lowest id on ties.  dom-min:
      // key = |D|; dom/deg: |D| / neighbours (integer), -1 without neighbours,
      // biased by one so that the packed key stays unsigned.  Every wave
      // finds it by itself.
      if (kWdeg) {
        x = wg_select_wdeg(net, mem, ctl, A);
      } else if constexpr (kFlat) {
        unsigned key = ~0u, dv = 0u;
        for (int v = lane; v < n; v += 64) {
          const unsigned d = (unsigned)ld_wg(&mem.dom[v]);
          unsigned hi = (unsigned)__popc(d);
          if (A.nbr) {
            const int g = A.nbr[v];
            hi = g == 0 ? 0u : hi / (unsigned)g + 1u;
          }
          const unsigned k = (hi << 16) | (unsigned)v;
          if (!bit_of(mem.asg, v) && k < key) {
            key = k;
            dv = d;
          }
        }
        const unsigned least = wave_min32_dpp(key);
        x = (int)(least & 0xffffu);
        dx = (unsigned)__builtin_amdgcn_readlane((int)dv, x & 63);
      } else {
        u64 key = ~0ull;
        for (int v = lane; v < n; v += 64)
          if (!bit_of(mem.asg, v)) {
            unsigned hi = (unsigned)mem.size[v];
            if (A.nbr) {
              const int g = A.nbr[v];
              hi = g == 0 ? 0u : (unsigned)(mem.size[v] / g) + 1u;
            }
            const u64 k = ((u64)hi << 32) | (unsigned)v;
            key = k < key ? k : key;
          }
        x = uniform_int((int)(wave_min64_dpp(key) & 0xffffffffu));
      }
      // min value of x (every thread scans the same words)
      a = -1;
      if constexpr (kFlat) {
        if (dx) a = (int)__builtin_ctz(dx);
      } else {
        for (int w = 0; w < W && a < 0; ++w) {
          const u64 dw = mem.dom[(long long)x * W + w];
          if (dw) a = w * 64 + (int)__builtin_ctzll(dw);
        }
        a = uniform_int(a);
      }
      if (a < 0) {
        // x has an empty domain that no revision reached (no constraints, an
        // empty initial domain): the search ends without a solution, with no
        // node recorded, as the oracle's restatement does
        status = MAC_UNSAT;
        break;
      }
      if constexpr (kFlat) {
        if (tid < n) {
          const u64 d = ld_wg(&mem.dom[tid]);
          saved = (unsigned)d;
          A.trail[depth * nw + tid] = d;
        }
      } else {
        wg_copy_words(A.trail + depth * nw, mem.dom, nw);
      }
      __syncthreads();
      if (tid < W) mem.dom[(long long)x * W + tid] = (tid == (a >> 6)) ? (1ull << (a & 63)) : 0ull;
      if (!kFlat) wg_seed(mem, ctl, n, slot, x);
      if (tid == 0) {
        A.stack[depth] = make_int2(x, a);
        if (!kWdeg) stk[depth] = make_int2(x, a);
        mem.size[x] = 1;
        mem.asg[x >> 5] |= 1u << (x & 31);
      }
      ++depth;
      ++npos;
      ++nodes_here;
      phase = POSITIVE;
      if (!kFlat) __syncthreads();
    }
    bool ok;
    if constexpr (kFlat) {
      const unsigned bit = 1u << (a & 31);
      ok = wg_fixpoint_flat(mem, ctl, flat, seen, phase == ROOT ? -1 : x, phase == POSITIVE ? bit : dx & ~bit,
                            phase == POSITIVE, turn, flat_revs);
    } else {
      ok = wg_fixpoint<kFull, kFull>(net, mem, ctl, slot, -1);
    }
    if (kWdeg && !ok) {
      // a wipe-out raises the weight of the constraint that AC3's order
      // empties a domain with first: propagate again, in that order, from the
      // domains before.  (Without a wipe-out the closure is the same in any
      // order and no weight changes.)
      const u64* level = A.trail + (phase == POSITIVE ? depth - 1 : depth) * nw;
      wg_load_level(mem, level, n, W, phase == NEGATIVE ? x : -1, a);
      __syncthreads();
      if (phase == POSITIVE) {
        if (tid < W) mem.dom[(long long)x * W + tid] = (tid == (a >> 6)) ? (1ull << (a & 63)) : 0ull;
        if (tid == 0) mem.size[x] = 1;
      }
      ok = wg_ac3(net, mem, ctl, A, phase == ROOT ? -1 : x);
    }
    slot ^= 1;
    select = true;
    if (phase == ROOT) {
      if (ok) wg_copy_words(A.trail, mem.dom, nw);
      if (A.root_out) wg_copy_words(A.root_out, mem.dom, nw);
      if (!ok) status = MAC_UNSAT;
      continue;
    }
    wg_trace(net, mem, A, &trace_len, phase == POSITIVE ? 1 : 0, x, a, ok);
    if (phase == POSITIVE && ok && depth == n) {
      if (A.solution && nsol < (A.sol_cap > 0 ? A.sol_cap : 1))
        for (int v = tid; v < n; v += nthreads) {
          int sv = -1;
          for (int w = 0; w < W && sv < 0; ++w) {
            const u64 dw = mem.dom[(long long)v * W + w];
            if (dw) sv = w * 64 + (int)__builtin_ctzll(dw);
          }
          A.solution[nsol * n + v] = sv;
        }
      ++nsol;
      if (A.max_solutions <= 1 || nsol >= A.max_solutions) {
        status = MAC_SAT;
        break;
      }
      ok = false;  // enumeration: go on as after a failed node
      __syncthreads();
    }
    if (ok) continue;
    // undo decisions until a refutation leaves its variable a value
    select = false;
    if (!kFlat) phase = NEGATIVE;
    while (true) {
      if (depth == 0) {
        status = MAC_UNSAT;
        break;
      }
      --depth;
      const int2 d = stk[depth];
      x = uniform_int(d.x);
      a = uniform_int(d.y);
      const u64* level = A.trail + depth * nw;
      u64 rest = 0ull;
      if constexpr (kFlat) {
        if (phase != POSITIVE) {
          saved = tid < n ? (unsigned)level[tid] : 0u;
          dx = (unsigned)uniform_int((int)level[x]);
        }
        phase = NEGATIVE;
        rest = dx & ~(1u << (a & 31));
        if (tid < n) {
          const unsigned d = tid == x ? (unsigned)rest : saved;
          mem.dom[tid] = d;
          mem.size[tid] = __popc(d);
        }
      } else {
        wg_load_level(mem, level, n, W, x, a);
        for (int w = 0; w < W; ++w) {
          const u64 dw = level[(long long)x * W + w];
          rest |= w == (a >> 6) ? dw & ~(1ull << (a & 63)) : dw;
        }
      }
      if (tid == 0) mem.asg[x >> 5] &= ~(1u << (x & 31));
      ++nneg;
      ++nodes_here;
      if ((u64)uniform_ll((long long)rest) != 0ull) break;
      wg_trace(net, mem, A, &trace_len, 0, x, a, false);
    }
    if (status != MAC_RUNNING) break;
    if (!kFlat) wg_seed(mem, ctl, n, slot, x);
    __syncthreads();
    if constexpr (kFlat) {
      wg_flat_see(mem, flat, seen);
      __syncthreads();
    }
  }
  if (kFlat && lane == 0 && flat_revs) atomicAdd(&ctl->revs, (unsigned long long)flat_revs);
  __syncthreads();
  if (tid == 0) {
    A.state->status = status;
    A.state->depth = depth;
    A.state->npos = npos;
    A.state->nneg = nneg;
    A.state->nsol = nsol;
    A.state->revisions += (long long)ctl->revs;
    A.state->trace_len = trace_len;
    A.state->steps += 1;
  }
}

// lnet.bytes > 0 (kLds only): the network image is copied into LDS behind
// the working memory and the search reads the network from there.  kFull: a
// network for the whole fixpoint (full_search), which has no image.
template <bool kLds, bool kWdeg, bool kFull>
__global__ void k_mac(DevNet net, MacArgs args, char* scratch, LdsNet lnet) {
  extern __shared__ __align__(16) char smem[];
  __shared__ WgCtl ctl;
  int* stamp = nullptr;
  if (kWdeg) stamp = args.stamp_off ? (int*)(smem + args.stamp_off) : args.stamp_tab;
  if (kLds && !kFull && lnet.bytes > 0) {
    const DevNet ln = wg_load_net(net, lnet, smem + wg_mem_bytes(net.n, net.W));
    WgMem mem = wg_carve(smem, ln);
    mem.stamp = stamp;
    if (!kWdeg && lnet.flat_min && lnet.flat_min <= (int)blockDim.x) wg_mac_run<false, true, false>(ln, mem, &ctl, args);
    else wg_mac_run<kWdeg, false, false>(ln, mem, &ctl, args);
  } else {
    WgMem mem = wg_carve(kLds ? smem : scratch, net);
    mem.stamp = stamp;
    wg_mac_run<kWdeg, false, kFull>(net, mem, &ctl, args);
  }
}

// ---------------------------------------------------------------------------
// Many independent MAC runs (uneven instances, serving slots): one workgroup
// per unit, units taken from a global counter (persistent) or fixed by
// `only` (one unit per launch).
// ---------------------------------------------------------------------------
struct UnitDesc {
  DevNet net;
  MacArgs args;
  long long scratch_off;  // per-unit global scratch when the domain does not fit in LDS
  int use_lds;            // 1: working memory in LDS; 2: network image in LDS as well
  int reset;              // 1: start the search over: level 0 = init, state = MAC_INIT
  int full;               // 1: the search takes the whole fixpoint (k_mac_units<true>)
  const u64* init;        // the unit's initial domains, [n][W]
  LdsNet lnet;
};

// states_out[u] receives a copy of unit u's state when its launch ends, so
// the host reads every unit's outcome with one copy.  kFull: launches with a
// unit that takes the whole fixpoint (the others of it still don't).
template <bool kFull>
__global__ void k_mac_units(const UnitDesc* __restrict__ units, int count, unsigned* counter,
                            int only, char* scratch, MacState* states_out) {
  extern __shared__ __align__(16) char smem[];
  __shared__ WgCtl ctl;
  __shared__ int unit_sh;
  while (true) {
    if (threadIdx.x == 0) unit_sh = only >= 0 ? only : (int)atomicAdd(counter, 1u);
    __syncthreads();
    const int u = uniform_int(unit_sh);
    __syncthreads();
    if (u >= count) break;
    const UnitDesc d = units[u];
    if (uniform_int(d.reset)) {
      // a new run of the batch: the workgroup restores level 0 and the state
      // itself, which spares the host two copies per unit
      const long long nw = (long long)d.net.n * d.net.W;
      for (long long i = threadIdx.x; i < nw; i += blockDim.x) d.args.trail[i] = d.init[i];
      if (threadIdx.x == 0) {
        MacState s0{};
        s0.status = MAC_INIT;
        *d.args.state = s0;
      }
      __syncthreads();
    }
    // One inlined copy of the search per place of the unit's memory (network
    // image and working memory in LDS, working memory in LDS, global
    // scratch), so that LDS accesses compile to ds_read / ds_write: one copy
    // over a pointer that may be either compiles them to flat instructions.
    const int where = uniform_int(d.use_lds);
    if (where == 2) {
      const DevNet ln = wg_load_net(d.net, d.lnet, smem + wg_mem_bytes(d.net.n, d.net.W));
      if (uniform_int(d.lnet.flat_min && d.lnet.flat_min <= (int)blockDim.x))
        wg_mac_run<false, true, false>(ln, wg_carve(smem, ln), &ctl, d.args);
      else
        wg_mac_run<false, false, false>(ln, wg_carve(smem, ln), &ctl, d.args);
    } else if (where == 1) {
      if (kFull && uniform_int(d.full)) wg_mac_run<false, false, kFull>(d.net, wg_carve(smem, d.net), &ctl, d.args);
      else wg_mac_run<false, false, false>(d.net, wg_carve(smem, d.net), &ctl, d.args);
    } else {
      const WgMem mem = wg_carve(scratch + d.scratch_off, d.net);
      if (kFull && uniform_int(d.full)) wg_mac_run<false, false, kFull>(d.net, mem, &ctl, d.args);
      else wg_mac_run<false, false, false>(d.net, mem, &ctl, d.args);
    }
    if (threadIdx.x == 0) states_out[u] = *d.args.state;
    if (only >= 0) break;
  }
}
