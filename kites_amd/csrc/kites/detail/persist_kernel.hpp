// persist_kernel.hpp -- small push frontiers in one workgroup, many
// iterations per launch.
//
// High-diameter graphs (grids, road-like meshes, paths) run thousands of
// iterations whose queues hold a few hundred or thousand vertices.  A launch
// of step_kernel per iteration then pays its dispatch, its completion and the
// next decision -- 7 to 12 us on MI355X -- for very little work.
// persist_kernel runs such iterations in one workgroup of 1,024 threads that
// synchronizes with barriers only (there is no other workgroup, so nothing
// waits on one), until the queue is empty (the run is done), the schedule
// picks a variant that is not a push, the queue outgrows the run's out-edge
// limit (the next step_kernel launch takes over), or the iteration limit is
// reached.  The engine launches it first in every chunk it replays after a
// tiny push frontier; when the coming iteration does not fit, it returns at
// once.
//
// Few edges per iteration make the loop a chain of dependent accesses, and one
// compute unit issues about one scattered access per cycle; both decide its
// form.  The queue's out-edges, not its entries, lie in LDS (edge index and
// source vertex, two lists that take turns): a thread needs no search to find
// its edges.  An iteration is three accesses long:
//   1. the edge's destination and weight and V[source];
//   2. V[destination], waited for; then a barrier, so that every thread has read
//      the values the iteration starts from;
//   3. for a candidate below that value, one returning atomic min, and beside it
//      the destination's out-offsets.  The thread whose atomic returns the
//      starting value lowered the vertex first and appends it (no other does, so
//      no bit is claimed); the waves reserve list space with one LDS atomic each
//      and write the appended vertices' edges for the next iteration.
// The decision of the next iteration is made by every thread from the totals in
// LDS (three sets of counters take turns), so the iteration has two barriers.
// Microseconds per iteration (BFS on grids of 16 / 64 / 256 / 480 columns, the
// queue two thirds of that): 1.9 / 2.1 / 3.6 / 6.1 (without the wait in front of
// the barrier 1.9 / 2.1 / 3.4 / 6.0); a form that staged the queue
// in LDS, searched each edge's entry and claimed bits took 4.3 / 4.6 / 6.0 /
// 9.2; step_kernel takes 6.2 / 6.5 / 6.9 / 7.0.  Near-far SSSP: 2.7 / 3.0 /
// 5.9 / 8.3 against 5.9 / 6.4 / 11.1 / 11.9, step_kernel 8.9 / 9.5 / 10.0 /
// 10.0.  The slope, 2.3 ns per edge, is the unit's scattered accesses, so
// BFS queues of more than about 2,048 out-edges go to step_kernel: at 4,096
// grids of 700 to 2,000 columns take 7.5 to 9.4.
//
// The queues are written to memory as step_kernel writes them (queue slot
// j & 1, offsets, the statistics entry j), the bitmap bits of a queue only when
// the loop ends: step_kernel and persist_kernel iterations follow each other
// in any order.  A step_kernel iteration j clears the bitmap slot (j + 2) % 3
// for iteration j + 1; here the slots that iterations before the launch wrote
// are cleared by its first two iterations (word by word from the queues that
// hold their bits), and the others were never set.
//
// Near-far runs (NF, unsigned values): a relaxation to a value at or above
// the threshold T claims the destination's far bit and appends it to the
// current far pile (its counter lives in a register of this launch: no other
// workgroup appends while the loop runs), and the least such value is kept.  A
// vertex is appended to the queue by the first relaxation that takes it below
// T.  When the queue runs dry with entries on the pile, the next iteration is
// a split (V_SPLIT, as in step_kernel): T becomes the least far value + delta,
// and every pile entry is dropped (its value fell below the previous
// threshold: it went through the queue), moved to the queue (below T) or kept
// on the other pile; the loop runs splits of up to 2 x the out-edge limit
// entries.
//
// The compute unit's L1 keeps lines across the iterations of one launch and
// atomics update only the L2, so every read of a location that atomics
// write (V) is an agent-scope atomic load.  Plain stores of this workgroup
// (queues, piles) pass through the same L1.
#ifndef KITES_DETAIL_PERSIST_KERNEL_HPP_
#define KITES_DETAIL_PERSIST_KERNEL_HPP_

#include <hip/hip_runtime.h>

#include <type_traits>

#include "step_kernel.hpp"
#include "wave.hpp"

namespace kites {
namespace detail {

constexpr unsigned kPersistBlock = 1024;
constexpr unsigned kPersistRounds = 4;    // edges (or pile entries) per thread
// Largest out-edge total of a queue it takes (step_core::persist_edges
// sets the run's limit, at most this): what the two lists in LDS hold.
constexpr unsigned kPersistEdges = kPersistBlock * kPersistRounds;
// Default limits.  A step_kernel iteration is 2 to 3 us dearer in near-far runs
// (two more counters to settle before it can close), so the loop pays for
// larger queues there: near-far SSSP on grids of 256 / 480 / 700 / 1111 / 2000
// columns takes 7.8 / 8.5 / 8.5 / 8.9 / 9.0 us per iteration with 2,048 and
// 6.0 / 8.4 / 8.8 / 8.5 / 8.5 with 4,096.
constexpr unsigned kPersistDefaultEdges = 2048;
constexpr unsigned kPersistFarEdges = 4096;
// options::persist_edges left alone: one of the two (no limit a caller sets).
constexpr unsigned kPersistAutoEdges = 0xFFFFFFFEu;
// Out-lists up to this long are written to the edge list by the lane that
// appends the vertex, longer ones by its wave.
constexpr unsigned kPersistLane = 16;

template <class vT>
struct persist_smem {
  unsigned idx[2][kPersistEdges];   // the queue's out-edges: index in oC, oE
  unsigned src[2][kPersistEdges];   // and source vertex
  vT slot[kPersistBlock];           // nbrComp's output, one per thread
  // Counters of an iteration, three sets that take turns: one is read, one
  // filled, one cleared.
  unsigned long long qe[3];         // packed (count, out-edges) of the next queue
  unsigned long long vmin[3];       // near-far: least far value
  unsigned maxdeg[3];
  unsigned far_add[3];              // near-far: entries appended to a pile
  float mlp[MLP_SCRATCH];           // the network's weights for an inference
};

// Whether an iteration (variant `v`; a queue with `sdeg` out-edges, or a split
// of a pile of `far_n` entries) is one persist_kernel runs.
template <bool FAR>
__device__ __forceinline__ bool persist_fits(unsigned v, unsigned long long sdeg, unsigned far_n,
                                             unsigned max_edges) {
  if (v == V_SPLIT) return FAR && far_n <= 2u * max_edges;
  return v >= V_PUSH_T && v <= V_PUSH_LB && sdeg <= max_edges;
}

template <class vT>
__device__ __forceinline__ vT load_agent(const vT* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Writes the out-edges of the lanes' vertices u (d edges from index b; d = 0:
// none) to the list at offset o, as far as the list reaches.  All 64 lanes
// active.
template <class vT>
__device__ __forceinline__ void persist_expand(persist_smem<vT>& sm, unsigned list, unsigned u,
                                               unsigned b, unsigned d, unsigned o) {
  bool const fits = d <= kPersistEdges && o <= kPersistEdges - d;
  if (fits && d <= kPersistLane)
    for (unsigned k = 0; k < d; ++k) {
      sm.idx[list][o + k] = b + k;
      sm.src[list][o + k] = u;
    }
  unsigned long long m = ballot64(fits && d > kPersistLane);
  while (m) {
    int const l = __builtin_ctzll(m);
    m &= m - 1;
    unsigned const ul = readlane(u, l), bl = readlane(b, l), dl = readlane(d, l),
                   ol = readlane(o, l);
    for (unsigned k = lane_id(); k < dl; k += WAVE_SIZE) {
      sm.idx[list][ol + k] = bl + k;
      sm.src[list][ol + k] = ul;
    }
  }
}

// Appends the lanes' vertices v[k] with `want` set (d[k] out-edges from b[k]) to
// the next queue and its edge list: one 64-bit LDS atomic per wave reserves the
// slots and the out-edge offsets.  All 64 lanes active.
template <unsigned R, class vT>
__device__ __forceinline__ void persist_append(persist_smem<vT>& sm, unsigned list, unsigned set,
                                               const bool (&want)[R], const unsigned (&v)[R],
                                               const unsigned (&b)[R], const unsigned (&d)[R],
                                               unsigned* out_q, unsigned* out_qe,
                                               unsigned& wmax) {
  unsigned cnt = 0, deg = 0;
#pragma unroll
  for (unsigned k = 0; k < R; ++k)
    if (want[k]) {
      cnt += 1;
      deg += d[k];
      wmax = d[k] > wmax ? d[k] : wmax;
    }
  if (!ballot64(cnt != 0)) return;
  unsigned const ci = wave_incl_scan(cnt), di = wave_incl_scan(deg);
  unsigned const ct = readlane(ci, 63), dt = readlane(di, 63);
  unsigned long long old = 0;
  if (lane_id() == 0) old = atomicAdd(&sm.qe[set], qe_pack(ct, dt));
  unsigned const olo = readlane(static_cast<unsigned>(old), 0);
  unsigned const ohi = readlane(static_cast<unsigned>(old >> 32), 0);
  unsigned long long const o64 = (static_cast<unsigned long long>(ohi) << 32) | olo;
  unsigned pos = qe_count(o64) + ci - cnt;
  unsigned off = qe_edges(o64) + di - deg;
#pragma unroll
  for (unsigned k = 0; k < R; ++k) {
    if (want[k]) {
      out_q[pos] = v[k];
      out_qe[pos] = off;
    }
    if (R == 1 || ballot64(want[k]))
      persist_expand(sm, list, v[k], b[k], want[k] ? d[k] : 0u, off);
    if (want[k]) {
      pos += 1;
      off += d[k];
    }
  }
}

// Appends the lanes' vertices with `want` set to a far pile at `base` + a
// position reserved with one LDS atomic per wave.  All 64 lanes active.
__device__ __forceinline__ void persist_far_append(unsigned& far_add, bool want, unsigned v,
                                                   unsigned* pile, unsigned base) {
  unsigned long long const m = ballot64(want);
  if (!m) return;
  unsigned old = 0;
  if (lane_id() == 0) old = atomicAdd(&far_add, static_cast<unsigned>(__builtin_popcountll(m)));
  old = readlane(old, 0);
  if (want) pile[base + old + rank_in(m)] = v;
}

__device__ __forceinline__ unsigned long long wave_min_u64(unsigned long long x) {
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) {
    unsigned long long const y = __shfl_xor(x, s, 64);
    x = y < x ? y : x;
  }
  return x;
}

// One push iteration over the E edges of list `cur` (0 < E <= R * kPersistBlock):
// every load of a step is issued before any is used.  Whole workgroup.
template <unsigned R, bool FAR, class P, class vT>
__device__ __forceinline__ void persist_push(P& p, persist_smem<vT>& sm, unsigned cur,
                                             unsigned set, unsigned E, unsigned long long T,
                                             unsigned* out_q, unsigned* out_qe, unsigned* far_q,
                                             unsigned fn, unsigned& wmax,
                                             unsigned long long& lvmin) {
  using eT = typename std::remove_const<typename std::remove_reference<decltype(*p.oE)>::type>::type;
  unsigned const t = threadIdx.x;
  unsigned idx[R], dst[R];
  vT val[R], cand[R], start[R];
  bool ok[R];
  // A thread without an edge repeats the list's first one and drops it; the
  // functor is called for it only if it cannot write the edge.  Functors in
  // registers are called among the loads (behind all of them near-far
  // iterations of 16 columns take 2.82 us instead of 2.76), functors in LDS
  // slots, whose flat accesses wait for every load, after them.
  constexpr bool kRead = reads_edge<decltype(p.fn), vT, eT>;
  constexpr bool kEarly = kRead && !takes_slot<decltype(p.fn), vT, eT>;
#pragma unroll
  for (unsigned k = 0; k < R; ++k) {
    unsigned const e = t + k * kPersistBlock;
    ok[k] = e < E;
    idx[k] = sm.idx[cur][ok[k] ? e : 0u];
    dst[k] = p.oC[idx[k]];
    val[k] = load_agent(p.V + sm.src[cur][ok[k] ? e : 0u]);
    cand[k] = vT{};
    if constexpr (kEarly) cand[k] = edge_value(p.fn, sm.slot[t], val[k], p.oE + idx[k]);
  }
  if constexpr (!kEarly) {
#pragma unroll
    for (unsigned k = 0; k < R; ++k)
      if (kRead || ok[k]) cand[k] = edge_value(p.fn, sm.slot[t], val[k], p.oE + idx[k]);
  }
#pragma unroll
  for (unsigned k = 0; k < R; ++k) start[k] = load_agent(p.V + dst[k]);
#pragma unroll
  for (unsigned k = 0; k < R; ++k) ok[k] = ok[k] && cand[k] < start[k];
  // (the barrier alone waits for no load: one still in flight could read what
  // another wave's atomic has written, and two threads would then take theirs
  // for the first relaxation of a vertex and append it twice)
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  vT old[R];
  unsigned b[R], deg[R];
#pragma unroll
  for (unsigned k = 0; k < R; ++k) {
    old[k] = start[k];
    b[k] = deg[k] = 0u;
    if (ok[k]) {
      old[k] = atomic_min_any(p.V + dst[k], cand[k]);
      b[k] = p.oR[dst[k]];
      deg[k] = p.oR[dst[k] + 1];
    }
  }
  bool near[R], far[R];
#pragma unroll
  for (unsigned k = 0; k < R; ++k) {
    deg[k] -= b[k];
    near[k] = ok[k] && cand[k] < old[k] && deg[k];
    far[k] = false;
    if constexpr (FAR) {
      unsigned long long const x = static_cast<unsigned long long>(cand[k]);
      if (near[k] && x >= T) {
        unsigned long long const bit = 1ull << (dst[k] & 63);
        lvmin = x < lvmin ? x : lvmin;
        far[k] = !(atomicOr(p.fbm + (dst[k] >> 6), bit) & bit);
        near[k] = false;
      }
      near[k] = near[k] && (old[k] == start[k] || static_cast<unsigned long long>(old[k]) >= T);
    } else {
      near[k] = near[k] && old[k] == start[k];
    }
  }
  persist_append(sm, cur ^ 1u, set, near, dst, b, deg, out_q, out_qe, wmax);
  if constexpr (FAR) {
#pragma unroll
    for (unsigned k = 0; k < R; ++k)
      persist_far_append(sm.far_add[set], far[k], dst[k], far_q, fn);
  }
}

template <bool NF, class P>
__global__ __launch_bounds__(kPersistBlock) void persist_kernel(P p) {
  using vT = typename std::remove_reference<decltype(*p.V)>::type;
  constexpr bool FAR = NF && std::is_unsigned<vT>::value;
  __shared__ persist_smem<vT> sm;
  unsigned const t = threadIdx.x, lane = lane_id(), wib = t >> 6;
  if (p.ctl->done) return;
  if (p.sched.mode != SCHED_PLAIN && p.sched.mode != SCHED_LEARNED) return;
  unsigned const max_edges = p.persist_edges < kPersistEdges ? p.persist_edges : kPersistEdges;
  if (max_edges == 0) return;
  unsigned iter = p.ctl->iter;
  if (iter < 2) return;
  unsigned long long const nw = p.nwords;
  unsigned long long const n = p.n;
  unsigned const max_iter = p.ctl->max_iter;
  // The state the first iteration consumes; later iterations carry it in
  // registers: the variant, the queue iteration - 1 appended (length c1,
  // out-edges e1), the length c2 of the one iteration - 2 appended, and the
  // near-far state (threshold, the previous one, pile size, least pile
  // value, current pile).
  unsigned variant = p.ctl->next_variant;
  unsigned c1 = p.ctl->q_count;
  unsigned long long e1 = p.ctl->q_edges;
  unsigned c2 = p.stats[iter - 2].count;
  unsigned long long T = ~0ull, Told = 0, fvmin = ~0ull;
  unsigned fn = 0, fsel = 0;
  if constexpr (FAR) {
    T = p.ctl->thresh;
    Told = p.ctl->thresh_prev;
    fvmin = p.ctl->far_vmin;
    fn = p.ctl->far_n;
    fsel = p.ctl->far_sel & 1u;
  }
  if (!persist_fits<FAR>(variant, e1, fn, max_edges)) return;
  // The queue's edges into list 0 (a split has no queue).
  unsigned cur = 0;
  if (!(FAR && variant == V_SPLIT)) {
    const unsigned* const in_q = p.q + (iter & 1) * n;
    const unsigned* const in_qe = p.qe + (iter & 1) * (n + 1);
    for (unsigned i0 = wib * WAVE_SIZE; i0 < c1; i0 += kPersistBlock) {
      unsigned const i = i0 + lane;
      unsigned u = 0, o = 0, b = 0, d = 0;
      if (i < c1) {
        u = in_q[i];
        o = in_qe[i];
        b = p.oR[u];
        d = p.oR[u + 1] - b;
      }
      persist_expand(sm, cur, u, b, d, o);
    }
  }
  if (t < 3) {
    sm.qe[t] = 0ull;
    sm.vmin[t] = ~0ull;
    sm.maxdeg[t] = 0u;
    sm.far_add[t] = 0u;
  }
  __syncthreads();
  unsigned set = 0;
  unsigned outside = 2;   // queues of iterations before this launch, their bits to be cleared
  for (;;) {
    bool const split = FAR && variant == V_SPLIT;
    unsigned const in_count = split ? fn : c1;
    unsigned* out_q = p.q + ((iter + 1) & 1) * n;
    unsigned* out_qe = p.qe + ((iter + 1) & 1) * (n + 1);
    // clear the bits of the queue iteration - 2 appended (it is the queue slot
    // this iteration appends to; after a large step_kernel iteration it can
    // hold up to n entries, and then the whole slot is cleared instead:
    // coalesced stores of nw words beat c2 scattered ones)
    if (outside) {
      --outside;
      unsigned long long* const clr_bm = p.bm + ((iter + 2) % 3) * nw;
      if (c2 > nw / 4) {
        for (unsigned long long w = t; w < nw; w += kPersistBlock) clr_bm[w] = 0ull;
      } else {
        for (unsigned i = t; i < c2; i += kPersistBlock) clr_bm[out_q[i] >> 6] = 0ull;
      }
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
    }
    unsigned wmax = 0;
    unsigned long long lvmin = ~0ull;   // near-far: least far value this lane saw
    unsigned long long work = 0;
    if (!split) {
      unsigned const E = static_cast<unsigned>(e1);
      work = E;
      unsigned* const far_q = FAR ? p.fq + static_cast<unsigned long long>(fsel) * n : nullptr;
      if (E == 0) {
        // nothing to relax
      } else if (E <= kPersistBlock)
        persist_push<1, FAR>(p, sm, cur, set, E, T, out_q, out_qe, far_q, fn, wmax, lvmin);
      else if (E <= 2 * kPersistBlock)
        persist_push<2, FAR>(p, sm, cur, set, E, T, out_q, out_qe, far_q, fn, wmax, lvmin);
      else if (E <= 3 * kPersistBlock)
        persist_push<3, FAR>(p, sm, cur, set, E, T, out_q, out_qe, far_q, fn, wmax, lvmin);
      else
        persist_push<kPersistRounds, FAR>(p, sm, cur, set, E, T, out_q, out_qe, far_q, fn, wmax, lvmin);
    } else if constexpr (FAR) {
      // split: every pile entry is dropped, moved to the queue or kept on the
      // other pile (far bits of entries leaving the pile cleared).  The pile
      // holds a vertex once, and the queue is empty.
      __builtin_amdgcn_s_waitcnt(0);   // the pile's entries, if this launch wrote them
      __syncthreads();
      const unsigned* const src = p.fq + static_cast<unsigned long long>(fsel) * n;
      unsigned* const keep_q = p.fq + static_cast<unsigned long long>(fsel ^ 1u) * n;
      unsigned const rounds = (in_count + kPersistBlock - 1) / kPersistBlock;   // uniform
      constexpr unsigned R = kPersistRounds;
      work = in_count;
      for (unsigned r = 0; r < rounds; r += R) {
        unsigned u[R], b[R], deg[R];
        unsigned long long x[R];
        bool ok[R], keep[R], move[R];
#pragma unroll
        for (unsigned k = 0; k < R; ++k) {
          unsigned const i = t + (r + k) * kPersistBlock;
          ok[k] = i < in_count;
          u[k] = ok[k] ? src[i] : 0u;
        }
#pragma unroll
        for (unsigned k = 0; k < R; ++k)
          x[k] = ok[k] ? static_cast<unsigned long long>(load_agent(p.V + u[k])) : ~0ull;
#pragma unroll
        for (unsigned k = 0; k < R; ++k) {
          keep[k] = ok[k] && x[k] >= T;
          move[k] = ok[k] && !keep[k] && x[k] >= Told;
          if (keep[k]) lvmin = x[k] < lvmin ? x[k] : lvmin;
          if (ok[k] && !keep[k]) atomicAnd(p.fbm + (u[k] >> 6), ~(1ull << (u[k] & 63)));
          // pile entries have out-edges (a far bit is claimed only then)
          b[k] = move[k] ? p.oR[u[k]] : 0u;
          deg[k] = move[k] ? p.oR[u[k] + 1] - b[k] : 0u;
        }
        persist_append(sm, cur ^ 1u, set, move, u, b, deg, out_q, out_qe, wmax);
#pragma unroll
        for (unsigned k = 0; k < R; ++k)
          persist_far_append(sm.far_add[set], keep[k], u[k], keep_q, 0u);
      }
      __builtin_amdgcn_s_waitcnt(0);   // the far bits, before relaxations claim them again
    }
    if (ballot64(wmax != 0)) {
      wmax = wave_max(wmax);
      if (lane == 0) atomicMax(&sm.maxdeg[set], wmax);
    }
    if constexpr (FAR) {
      if (ballot64(lvmin != ~0ull)) {
        lvmin = wave_min_u64(lvmin);
        if (lane == 0) atomicMin(&sm.vmin[set], lvmin);
      }
    }
    __syncthreads();
    // Every thread: the next queue, and whether the next iteration runs here.
    unsigned long long const qe = sm.qe[set];
    unsigned const count = qe_count(qe);
    unsigned const sdeg = qe_edges(qe);
    // near-far: the pile after this iteration
    unsigned fn_next = fn;
    unsigned long long fvmin_next = fvmin;
    bool split_next = false;
    if constexpr (FAR) {
      if (split) {
        fn_next = sm.far_add[set];
        fvmin_next = sm.vmin[set];   // exact: the least value of the entries kept
      } else {
        fn_next = fn + sm.far_add[set];
        fvmin_next = sm.vmin[set] < fvmin ? sm.vmin[set] : fvmin;
      }
      split_next = count == 0 && fn_next != 0;
    }
    bool const stop = (count == 0 && !split_next) || iter + 1 >= max_iter;
    unsigned long long T_next = T;
    if (split_next) {
      unsigned long long const tt = fvmin_next + p.sched.delta;
      T_next = tt < fvmin_next ? ~0ull : tt;
    }
    // (a queue that fits is far below the learned schedule's small-work guard,
    // which takes the plain choice)
    unsigned const fit_variant =
        split_next ? static_cast<unsigned>(V_SPLIT) : plain_variant(p.sched, sdeg, p.m);
    bool const go = !stop && persist_fits<FAR>(fit_variant, sdeg, fn_next, max_edges);
    if (t == 0) {
      unsigned const clr = set == 0 ? 2u : set - 1u;   // iteration - 1's set: all have read it
      sm.qe[clr] = 0ull;
      sm.vmin[clr] = ~0ull;
      sm.maxdeg[clr] = 0u;
      sm.far_add[clr] = 0u;
      out_qe[count] = sdeg;
      step_stats* st = p.stats + iter;
      st->count = count;
      st->variant = split ? static_cast<unsigned>(V_SPLIT) : static_cast<unsigned>(V_PERSIST);
      st->max_outdeg = sm.maxdeg[set];
      st->in_count = in_count;
      st->sum_outdeg = sdeg;
      st->work_edges = work;
      st->gathers = 0;
      st->active = in_count;
      st->qe = qe;
    }
    if (!go) {
      // The bits of the queue step_kernel goes on with, and the control line.
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      unsigned long long* const out_bm = p.bm + ((iter + 1) % 3) * nw;
      for (unsigned i = t; i < count; i += kPersistBlock)
        atomicOr(out_bm + (out_q[i] >> 6), 1ull << (out_q[i] & 63));
      if (wib != 0) return;
      unsigned next = V_CLASSIC;
      if (!stop) {
        learned_in li;
        li.scratch = sm.mlp;
        if (p.sched.mode == SCHED_LEARNED) {
          li.cache_key = p.ctl->cache_key;
          li.cache_variant = p.ctl->cache_variant;
        }
        next = split_next ? static_cast<unsigned>(V_SPLIT)
                          : choose_variant<true>(p, count, sdeg, sm.maxdeg[set], iter + 1, li);
      }
      if (lane != 0) return;
      p.ctl->next_variant = next;
      p.ctl->iter = iter + 1;
      unsigned const level = stop         ? 0u
                             : split_next ? (fn_next <= kSmallWork ? 1u : 0u)
                                          : grid_level(next, count, sdeg);
      p.ctl->small_next = level;
      p.ctl->q_count = count;
      p.ctl->q_edges = sdeg;
      if constexpr (FAR) {
        // (splits of this launch have flipped the pile and moved the threshold)
        if (split) {
          fsel ^= 1u;
          p.ctl->far_next = 0;
        }
        p.ctl->far_sel = fsel;
        p.ctl->far_n = fn_next;
        p.ctl->far_vmin = fvmin_next;
        p.ctl->thresh_prev = split_next ? T : Told;
        p.ctl->thresh = T_next;
      }
      if (stop) {
        p.ctl->done = 1;
        if (count != 0 || split_next) p.ctl->overflow = 1;
      }
      // (the iterations of the loop are part of one launch: the count of
      // launches does not move, and the host sees the loop's end)
      if (p.progress)
        __hip_atomic_store(p.progress,
                           progress_pack(iter + 1, p.ctl->launches, level, stop,
                                         stop && (count != 0 || split_next)),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      return;
    }
    variant = fit_variant;
    c2 = c1;
    c1 = count;
    e1 = sdeg;
    cur ^= 1u;
    set = set == 2 ? 0u : set + 1u;
    if constexpr (FAR) {
      if (split) fsel ^= 1u;
      fn = fn_next;
      fvmin = fvmin_next;
      if (split_next) {
        Told = T;
        T = T_next;
      }
    }
    ++iter;
  }
}

}  // namespace detail
}  // namespace kites

#endif  // KITES_DETAIL_PERSIST_KERNEL_HPP_
