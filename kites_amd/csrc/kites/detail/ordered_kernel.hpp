// ordered_kernel.hpp -- ordered (Jacobi) iterations for functor sets whose
// reduction is not idempotent (sums, PageRank-style updates).
//
// The reference runs every functor set in place with chaotic relaxation and
// combines a vertex's in-edges in an undefined tree order
// (kites/device/kernels_single_device.cuh:92-132), so a sum's result depends
// on timing and launch shape.  This mode defines both:
//   * Jacobi: iteration i reads Vin (the values after iteration i-1) and
//     writes Vout; vertices not recomputed keep their value.
//   * Combine order: for an active vertex v,
//       acc = initF(Vin[v]);
//       for each 64-edge chunk of v's in-list, in order:
//         x[l] = nbrCompF(Vin[C[e_l]], &E[e_l]) for the chunk's edges e_0..e_k-1;
//         a pairwise tree: for s = 1, 2, 4, ..., 32, x[l] = redF(x[l], x[l+s])
//           for every l divisible by 2s with l+s < k (lhs = the left operand);
//         acc = redF(acc, x[0]);
//       if updF(acc, Vin[v]): Vout[v] = acc and v's out-neighbours become
//       active for the next iteration.
//   Activeness follows the reference: the initial frontier, then the
//   out-neighbours of the vertices that changed.
// redF therefore needs neither associativity nor commutativity here, and the
// result is the same for every grid and run.
//
// The order fixes only the tree of each 64-edge chunk and the left-to-right
// fold of a vertex's chunks, so the work is cut by edges, not by vertices
// (bound: one gather of Vin per in-edge):
//   * vertices with more than 64 in-edges (ordered_shape::light; "heavy"): one wave per chunk
//     (ordered_heavy_kernel) leaves the chunk's tree in `hsum`; one lane per
//     vertex folds them in the next launch;
//   * the others: one wave takes the consecutive vertices whose in-lists start
//     in one window of ordered_shape::task_edges edges, holds all their edges' partials in LDS
//     and runs every vertex's trees at once (a lane's partner l + s belongs to
//     the same vertex exactly if both carry the same segment start).
// One wave per vertex, its chunks in sequence and one mark per out-edge, took
// 12.25 ms an iteration on R-MAT scale 20 (16M edges): a hub's in-list was one
// wave's chain.  Cut this way it takes 0.17 ms (heavy chunks 90 us, 12.2M edges
// at 136 G edges/s, bound by the L2's random reads; light vertices 78 us, 3.8M
// edges of 500K vertices, bound by the chain of dependent reads of a task).
// The light limit is one chunk: at 256 in-edges the same iteration took 0.24 ms
// (more registers, fewer waves), and full chunks are the faster form.
//
// Activity has two forms, chosen per iteration from the out-edges of the
// vertices that moved (kDenseDiv): few -- the movers' out-neighbours are
// marked (the bitmap holds active vertices); many -- only the movers are
// marked, and the next iteration, which reads every in-edge's source anyway,
// takes a vertex as active when one of its sources moved (one bit test per
// edge, 20 us above, instead of one mark per out-edge).  That form calls
// nbrCompF for edges of vertices that turn out inactive, which only functors that
// cannot write the edge allow (reads_edge).  For the others a launch in front of
// the iteration makes the active vertices' bitmap from the movers'
// (ordered_activate_kernel), and nbrCompF is called once per iteration for each
// in-edge of the active vertices and for no other.  Float PageRank in the
// reference's form, R-MAT scale 18, 76 iterations: 8.8 ms with calls for every
// edge, 13.6 with exact ones (67 when movers always marked their out-lists; one
// wave per vertex took 303).
#ifndef KITES_DETAIL_ORDERED_KERNEL_HPP_
#define KITES_DETAIL_ORDERED_KERNEL_HPP_

#include <hip/hip_runtime.h>

#include <type_traits>

#include "functor_call.hpp"
#include "ticket.hpp"
#include "wave.hpp"

namespace kites {
namespace detail {

// Shapes by value size: the partials of a task live in LDS.  4-byte values:
// 4.5 KB a wave, so eight 256-thread workgroups fit a compute unit's LDS.
template <class vT>
struct ordered_shape {
  static constexpr bool small = sizeof(vT) <= 16;
  static constexpr int block = small ? 256 : 64;
  static constexpr int waves = block / 64;
  static constexpr unsigned light = 64;       // in-edges of a light vertex, at most
  static constexpr unsigned task_edges = small ? 448 : 64;  // in-list starts per task window
  static constexpr unsigned slots = task_edges + light;     // ends of the light in-lists of a task
  static constexpr unsigned rows = slots / 64;
  static constexpr unsigned batch = small ? 4 : 2;          // rows of 64 edges in flight per wave
  static constexpr unsigned heavy_unroll = small ? 2 : 1;   // heavy chunks in flight per wave
  // A row's segment heads (4 bytes an edge) may lie where its partials will: a
  // batch of rows reads its heads before it writes its partials.  Partials of
  // more than 4 bytes would reach into the heads of later batches, which then
  // have an area of their own.
  static constexpr bool heads_apart = sizeof(vT) > sizeof(unsigned);
  static_assert(rows % batch == 0, "whole batches of rows");
};

// The next iteration tests its in-edges' sources (instead of being handed a
// list of active vertices) when the movers' out-edges * kDenseDiv >= m.
constexpr unsigned long long kDenseDiv = 8;
// ... or when one wave's movers hold more than m / kSerialDiv out-edges: a wave
// marks about 128 out-neighbours per microsecond, a pass over every in-edge
// takes about m / 65,536 us (R-MAT scale 20: hubs among a few movers made
// iterations of 1.6-2.5 ms, against 0.17 ms for the pass).
constexpr unsigned long long kSerialDiv = 512;

struct alignas(128) ordered_slot {
  unsigned long long out_edges;   // out-edges of the vertices that moved
  unsigned moved;
  unsigned most;                  // most out-edges one wave marked at once
};

// A 64-edge chunk of a heavy vertex's in-list.
struct ordered_chunk {
  unsigned begin, count, v, h;    // first edge, edges, vertex, its place in hv
};

struct ordered_ctl {
  unsigned iter;
  unsigned done;
  unsigned max_iter;
  unsigned in_moved;     // the input bitmap holds the movers (else the active vertices)
  unsigned out_moved;    // so does the output bitmap
  unsigned nheavy;       // heavy vertices and the total of their chunks
  unsigned nchunks;
  unsigned pad;
  unsigned long long heavy_cursor;   // setup: count << 32 | chunks
  ordered_slot slots[kTicketGroups];
  ticket_board board;
};

template <class vT, class eT, class FI, class FN, class FR, class FU>
struct ordered_params {
  unsigned n;
  unsigned long long m;
  const unsigned* R;    // in-edge CSR
  const unsigned* C;
  eT* E;
  const unsigned* oR;   // out-lists (activation of out-neighbours)
  const unsigned* oC;
  const unsigned* nzi;  // vertices with in-edges and their in-list starts
  const unsigned* nzR;
  unsigned nnz;
  vT* V;                // values of the even iterations (the graph's own)
  vT* W;                // and of the odd ones
  unsigned long long* bm;      // 2 bitmaps of nwords words
  unsigned long long* abm;     // functors that may write the edge: the active vertices
  unsigned long long* hasin;   // bit v: v has in-edges
  unsigned nwords;
  unsigned ntasks;
  unsigned* tstart;     // ntasks + 1 positions in nzi
  unsigned* hv;         // heavy vertices
  unsigned* hbase;      // their first chunk
  unsigned* hact;       // set when one of the vertex's sources moved
  ordered_chunk* hchunk;
  vT* hsum;             // the chunks' trees
  ordered_ctl* ctl;
  FI fi;
  FN fn;
  FR fr;
  FU fu;
  ordered_params(FI a, FN b, FR r, FU u) : fi(a), fn(b), fr(r), fu(u) {}
};

// Keeps the load of `x` (an edge's weight): the functor reads it through its
// own pointer, this only starts the round trip early.
template <class T>
__device__ __forceinline__ void ordered_touch(T const& x) {
  unsigned const b = *reinterpret_cast<unsigned char const*>(&x);
  asm volatile("" ::"v"(b));
}

__device__ __forceinline__ bool ordered_bit(const unsigned long long* bm, unsigned v) {
  return (bm[v >> 6] >> (v & 63)) & 1ull;
}

// ---- setup (once per run) -----------------------------------------------------

static __global__ void ordered_reset_kernel(ordered_ctl* ctl, unsigned max_iter, unsigned out_moved) {
  unsigned const t = threadIdx.x;
  if (t == 0) {
    ctl->iter = 0;
    ctl->done = 0;
    ctl->max_iter = max_iter;
    ctl->in_moved = 0;
    ctl->out_moved = out_moved;
    ctl->nheavy = 0;
    ctl->nchunks = 0;
    ctl->heavy_cursor = 0;
  }
  if (t < kTicketGroups) {
    ctl->slots[t].out_edges = 0;
    ctl->slots[t].moved = 0;
    ctl->slots[t].most = 0;
  }
  clear_ticket_board(ctl->board.w, t, blockDim.x);
}

// The initial active vertices into the run's first bitmap: `words` words of
// `frontier`, or every vertex when it is null.
static __global__ void ordered_frontier_kernel(const unsigned long long* __restrict__ frontier,
                                               unsigned words, unsigned n, unsigned nwords,
                                               unsigned long long* __restrict__ bm) {
  unsigned const nt = gridDim.x * blockDim.x;
  for (unsigned w = blockIdx.x * blockDim.x + threadIdx.x; w < nwords; w += nt) {
    unsigned const lo = w * 64u;
    unsigned long long const all = lo >= n ? 0ull : n - lo >= 64u ? ~0ull : (1ull << (n - lo)) - 1ull;
    bm[w] = !frontier ? all : w < words ? frontier[w] : 0ull;
  }
}

// One wave per 64 vertices: the has-in-edges word, and the heavy vertices with
// their chunk ranges (one atomic per wave that holds any; the order of the
// list does not matter).
template <unsigned LIGHT>
__global__ void ordered_vertices_kernel(const unsigned* __restrict__ R, unsigned n, unsigned nwords,
                                        unsigned long long* __restrict__ hasin,
                                        unsigned* __restrict__ hv, unsigned* __restrict__ hbase,
                                        unsigned* __restrict__ hact, ordered_ctl* ctl) {
  unsigned const lane = lane_id();
  unsigned const nw = gridDim.x * (blockDim.x / 64);
  for (unsigned w = blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6); w < nwords; w += nw) {
    unsigned const v = w * 64u + lane;
    unsigned const deg = v < n ? R[v + 1] - R[v] : 0u;
    unsigned long long const has = ballot64(deg != 0);
    if (lane == 0) hasin[w] = has;
    bool const heavy = deg > LIGHT;
    unsigned long long const hm = ballot64(heavy);
    if (!hm) continue;
    unsigned const nc = heavy ? (deg + 63u) / 64u : 0u;
    unsigned const incl = wave_incl_scan(nc);
    unsigned const total = readlane(incl, 63);
    unsigned long long old = 0;
    if (lane == 0)
      old = atomicAdd(&ctl->heavy_cursor,
                      (static_cast<unsigned long long>(__builtin_popcountll(hm)) << 32) | total);
    unsigned const chunk0 = readlane(static_cast<unsigned>(old), 0);
    unsigned const first = readlane(static_cast<unsigned>(old >> 32), 0);
    if (heavy) {
      unsigned const h = first + rank_in(hm);
      hv[h] = v;
      hbase[h] = chunk0 + incl - nc;
      hact[h] = 0;
    }
  }
}

// Task starts (the first in-list that begins at or after edge t * TE) and the
// heavy chunks.
template <unsigned TE>
__global__ void ordered_tasks_kernel(const unsigned* __restrict__ R, const unsigned* __restrict__ nzR,
                                     unsigned nnz, unsigned ntasks, unsigned* __restrict__ tstart,
                                     const unsigned* __restrict__ hv,
                                     const unsigned* __restrict__ hbase,
                                     ordered_chunk* __restrict__ hchunk, ordered_ctl* ctl) {
  unsigned const tid = blockIdx.x * blockDim.x + threadIdx.x, nt = gridDim.x * blockDim.x;
  for (unsigned t = tid; t <= ntasks; t += nt) {
    unsigned lo = 0, hi = nnz;
    unsigned long long const at = static_cast<unsigned long long>(t) * TE;
    while (lo < hi) {
      unsigned const mid = lo + (hi - lo) / 2;
      if (nzR[mid] < at) lo = mid + 1;
      else hi = mid;
    }
    tstart[t] = t == ntasks ? nnz : lo;
  }
  unsigned const nh = static_cast<unsigned>(ctl->heavy_cursor >> 32);
  if (tid == 0) {
    ctl->nheavy = nh;
    ctl->nchunks = static_cast<unsigned>(ctl->heavy_cursor);
  }
  for (unsigned h = tid >> 6; h < nh; h += nt >> 6) {
    unsigned const v = hv[h], b = hbase[h];
    unsigned const beg = R[v], deg = R[v + 1] - beg;
    for (unsigned c = lane_id(); c * 64u < deg; c += 64) {
      unsigned const left = deg - c * 64u;
      hchunk[b + c] = ordered_chunk{beg + c * 64u, left < 64u ? left : 64u, v, h};
    }
  }
}

// ---- one iteration: two launches (three for functors that may write the edge) -----

// The vertices with a mover among their in-edges' sources, when the input bitmap
// holds the movers.  One wave per 64 vertices: a lane walks a light in-list, the
// wave a heavy one, each until it meets a mover (with many movers, after an edge
// or a chunk).
template <class P>
__global__ __launch_bounds__(256) void ordered_activate_kernel(P p) {
  if (p.ctl->done || !p.ctl->in_moved) return;
  unsigned long long const* const movers =
      p.bm + static_cast<unsigned long long>(p.ctl->iter & 1) * p.nwords;
  unsigned const lane = lane_id();
  unsigned const waves = gridDim.x * (blockDim.x / 64);
  for (unsigned w = blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6); w < p.nwords; w += waves) {
    unsigned const v = w * 64u + lane;
    unsigned const b = v < p.n ? p.R[v] : 0u, e = v < p.n ? p.R[v + 1] : 0u;
    bool const heavy = e - b > 64u;
    bool on = false;
    for (unsigned k = b; !heavy && !on && k < e; ++k) on = ordered_bit(movers, p.C[k]);
    unsigned long long hm = ballot64(heavy);
    while (hm) {
      int const l = __builtin_ctzll(hm);
      hm &= hm - 1;
      unsigned const hb = readlane(b, l), he = readlane(e, l);
      bool hit = false;
      for (unsigned long long c = hb; c < he && !hit; c += 64 * 8) {
        bool any = false;
#pragma unroll
        for (unsigned u = 0; u < 8; ++u) {
          unsigned long long const k = c + u * 64 + lane;
          any = any || (k < he && ordered_bit(movers, p.C[k]));
        }
        hit = ballot64(any) != 0;
      }
      on = on || (hit && lane == static_cast<unsigned>(l));
    }
    unsigned long long const word = ballot64(on);
    if (lane == 0) p.abm[w] = word;
  }
}

// First launch: Vout = Vin, the output bitmap cleared, and the trees of the
// active heavy vertices' chunks (every heavy chunk when activity is decided
// by the sources).
template <class P>
__global__ __launch_bounds__(ordered_shape<typename std::remove_reference<decltype(*P::V)>::type>::block)
void ordered_heavy_kernel(P p) {
  using vT = typename std::remove_reference<decltype(*p.V)>::type;
  using S = ordered_shape<vT>;
  using eT = typename std::remove_reference<decltype(*p.E)>::type;
  constexpr unsigned U = S::heavy_unroll;
  constexpr bool kRead = reads_edge<decltype(p.fn), vT, eT>;
  __shared__ vT slot[S::waves][U][64];
  if (p.ctl->done) return;
  unsigned const iter = p.ctl->iter;
  bool const in_moved = p.ctl->in_moved != 0;
  bool const by_source = kRead && in_moved;
  vT const* const Vin = (iter & 1) ? p.W : p.V;
  vT* const Vout = (iter & 1) ? p.V : p.W;
  unsigned long long const* const in =
      !kRead && in_moved ? p.abm : p.bm + static_cast<unsigned long long>(iter & 1) * p.nwords;
  unsigned long long* const out = p.bm + static_cast<unsigned long long>((iter + 1) & 1) * p.nwords;
  unsigned const tid = blockIdx.x * blockDim.x + threadIdx.x, nt = gridDim.x * blockDim.x;
  for (unsigned i = tid; i < p.n; i += nt) Vout[i] = Vin[i];
  for (unsigned i = tid; i < p.nwords; i += nt) out[i] = 0ull;
  unsigned const lane = lane_id(), wib = readfirstlane(threadIdx.x >> 6);
  unsigned const nc = p.ctl->nchunks;
  unsigned const nw = gridDim.x * S::waves;
  for (unsigned c0 = (blockIdx.x * S::waves + wib) * U; c0 < nc; c0 += nw * U) {
    ordered_chunk ch[U];
    bool on[U], seen[U];
    unsigned e[U], src[U];
    vT x[U];
    eT w[U];
#pragma unroll
    for (unsigned u = 0; u < U; ++u) ch[u] = p.hchunk[c0 + u < nc ? c0 + u : nc - 1];
#pragma unroll
    for (unsigned u = 0; u < U; ++u) {
      e[u] = ch[u].begin + (lane < ch[u].count ? lane : 0u);
      src[u] = p.C[e[u]];
      w[u] = p.E[e[u]];
      on[u] = c0 + u < nc && (by_source || ordered_bit(in, ch[u].v));
      // a chunk of the same vertex may have seen a mover already (a stale read
      // only tests again)
      seen[u] = !by_source || p.hact[ch[u].h] != 0u;
    }
#pragma unroll
    for (unsigned u = 0; u < U; ++u) x[u] = Vin[src[u]];
#pragma unroll
    for (unsigned u = 0; u < U; ++u)
      // (lanes past the chunk hold its first edge's source)
      if (!seen[u] && ballot64(ordered_bit(in, src[u])) && lane == 0) p.hact[ch[u].h] = 1u;
#pragma unroll
    for (unsigned u = 0; u < U; ++u) {
      ordered_touch(w[u]);
      if (kRead || (on[u] && lane < ch[u].count))
        edge_value_at(p.fn, slot[wib][u][lane], x[u], p.E + e[u]);
    }
    wave_lds_sync();
#pragma unroll
    for (unsigned s = 1; s < 64; s <<= 1) {
#pragma unroll
      for (unsigned u = 0; u < U; ++u)
        if (on[u] && (lane & (2 * s - 1)) == 0 && lane + s < ch[u].count)
          reduce_at(p.fr, slot[wib][u][lane], slot[wib][u][lane + s]);
      wave_lds_sync();
    }
#pragma unroll
    for (unsigned u = 0; u < U; ++u)
      if (on[u] && lane == 0) p.hsum[c0 + u] = slot[wib][u][0];
    wave_lds_sync();
  }
}

// What a wave needs to publish its movers.
struct ordered_wave {
  unsigned long long* words;   // 64 words of LDS
  unsigned* excl;              // 64 entries each
  unsigned* base;
  unsigned moved = 0;
  unsigned most = 0;
  unsigned long long out_edges = 0;
};

// Marks the movers among the wave's vertices (ascending by lane), or their
// out-neighbours, in the output bitmap; [ob, oe) is the lane's out-list.  All
// 64 lanes.
template <class P>
__device__ __forceinline__ void ordered_publish(P const& p, unsigned long long* out, bool out_moved,
                                                ordered_wave& o, bool moved, unsigned v,
                                                unsigned ob, unsigned oe) {
  unsigned long long const mm = ballot64(moved);
  if (!mm) return;
  unsigned const lane = lane_id();
  unsigned const od = moved ? oe - ob : 0u;
  unsigned const incl = wave_incl_scan(od);
  unsigned const total = readlane(incl, 63);
  o.moved += moved;
  o.out_edges += od;
  o.most = total > o.most ? total : o.most;
  if (out_moved) {
    // the movers' bits, gathered per word in LDS (consecutive vertices share
    // words), one atomic per word
    unsigned const w0 = readlane(v >> 6, static_cast<int>(__builtin_ctzll(mm)));
    o.words[lane] = 0ull;
    wave_lds_sync();
    if (moved) {
      unsigned long long const bit = 1ull << (v & 63);
      unsigned const d = (v >> 6) - w0;
      if (d < 64u) atomicOr(o.words + d, bit);
      else atomicOr(out + (v >> 6), bit);
    }
    wave_lds_sync();
    unsigned long long const word = o.words[lane];
    if (word) atomicOr(out + w0 + lane, word);
    wave_lds_sync();
  } else {
    // merged walk of the movers' out-lists; a bit already seen set (bits only
    // get set here) needs no atomic
    wave_lds_sync();
    o.excl[lane] = incl - od;
    o.base[lane] = ob;
    wave_lds_sync();
    for (unsigned e0 = 0; e0 < total; e0 += 64) {
      unsigned const e = e0 + lane;
      if (e < total) {
        unsigned const own = owner_search(o.excl, e);
        unsigned const u = p.oC[o.base[own] + (e - o.excl[own])];
        unsigned long long const bit = 1ull << (u & 63);
        if (!(out[u >> 6] & bit)) atomicOr(out + (u >> 6), bit);
      }
    }
    wave_lds_sync();
  }
}

// Second launch: the heavy vertices' folds (on the first waves), the light
// vertices' trees and folds, the active vertices without in-edges; the last
// workgroup closes the iteration.
template <class P>
__global__ __launch_bounds__(ordered_shape<typename std::remove_reference<decltype(*P::V)>::type>::block) __attribute__((amdgpu_waves_per_eu(6)))
void ordered_kernel(P p) {
  using vT = typename std::remove_reference<decltype(*p.V)>::type;
  using S = ordered_shape<vT>;
  using eT = typename std::remove_reference<decltype(*p.E)>::type;
  constexpr unsigned kW = S::waves;
  constexpr unsigned kRows = S::rows, kB = S::batch;
  constexpr bool kRead = reads_edge<decltype(p.fn), vT, eT>;
  // A wave's partials; before a row's partials are written, its words hold the
  // row's segment heads (ordered_shape::heads_apart: an array of their own).
  constexpr unsigned kSlotBytes = S::slots * (sizeof(vT) < 4 ? 4 : sizeof(vT));
  __shared__ __align__(16) unsigned char slot_s[kW][(kSlotBytes + 15) / 16 * 16];
  __shared__ unsigned head_s[kW][S::heads_apart ? S::slots : 1];
  __shared__ vT acc_s[kW][64];
  __shared__ unsigned long long words_s[kW][64];
  __shared__ unsigned excl_s[kW][64], base_s[kW][64];
  __shared__ unsigned act_s[kW][(S::task_edges + 31) / 32];
  __shared__ unsigned s_moved, s_most;
  __shared__ unsigned long long s_out;
  __shared__ unsigned s_last;
  if (p.ctl->done) return;
  unsigned const iter = p.ctl->iter;
  bool const in_moved = p.ctl->in_moved != 0;
  bool const by_source = kRead && in_moved;
  bool const out_moved = p.ctl->out_moved != 0;
  vT const* const Vin = (iter & 1) ? p.W : p.V;
  vT* const Vout = (iter & 1) ? p.V : p.W;
  unsigned long long const* const in =
      !kRead && in_moved ? p.abm : p.bm + static_cast<unsigned long long>(iter & 1) * p.nwords;
  unsigned long long* const out = p.bm + static_cast<unsigned long long>((iter + 1) & 1) * p.nwords;
  unsigned const t = threadIdx.x, lane = lane_id(), wib = readfirstlane(t >> 6);
  vT* const slot = reinterpret_cast<vT*>(slot_s[wib]);
  unsigned* const head =
      S::heads_apart ? head_s[wib] : reinterpret_cast<unsigned*>(slot_s[wib]);
  vT* const acc = acc_s[wib];
  unsigned* const act = act_s[wib];
  ordered_wave ow;
  ow.words = words_s[wib];
  ow.excl = excl_s[wib];
  ow.base = base_s[wib];
  if (t == 0) {
    s_moved = 0;
    s_most = 0;
    s_out = 0;
  }
  __syncthreads();
  unsigned const wave = blockIdx.x * kW + wib, nwaves = gridDim.x * kW;
  unsigned const nh = p.ctl->nheavy;
  unsigned const hwant = (nh + 63u) / 64u;
  // the folds of hubs are the longest chains: they start first, on waves that
  // take no tasks (all waves share both when the grid is tiny)
  unsigned const hwaves = hwant < nwaves / 2 ? hwant : nwaves / 2;
  if (wave < hwaves || (hwaves == 0 && hwant)) {
    unsigned const step = hwaves ? hwaves : nwaves;
    for (unsigned g = wave; g < hwant; g += step) {
      unsigned const h = g * 64u + lane;
      unsigned v = 0, nc = 0, b = 0;
      bool moved = false;
      if (h < nh) {
        v = p.hv[h];
        bool on;
        if (by_source) {
          on = p.hact[h] != 0;
          if (on) p.hact[h] = 0u;
        } else {
          on = ordered_bit(in, v);
        }
        if (on) {
          nc = (p.R[v + 1] - p.R[v] + 63u) / 64u;
          b = p.hbase[h];
          vT const old = Vin[v];
          init_at(p.fi, acc[lane], old);
          for (unsigned c = 0; c < nc; c += 8) {
            vT x[8];
#pragma unroll
            for (unsigned u = 0; u < 8; ++u) x[u] = p.hsum[b + (c + u < nc ? c + u : nc - 1)];
#pragma unroll
            for (unsigned u = 0; u < 8; ++u)
              if (c + u < nc) {
                slot[lane] = x[u];
                reduce_at(p.fr, acc[lane], slot[lane]);
              }
          }
          moved = update_at(p.fu, acc[lane], old);
          if (moved) Vout[v] = acc[lane];
        }
      }
      // (heavy vertices are not sorted: one word at a time would not pay, the
      // marks of far words go straight to the bitmap)
      unsigned const ob = moved ? p.oR[v] : 0u, oe = moved ? p.oR[v + 1] : 0u;
      ordered_publish(p, out, out_moved, ow, moved, v, ob, oe);
    }
  }
  unsigned const wfirst = wave >= hwaves ? wave - hwaves : p.ntasks;
  for (unsigned task = wfirst; task < p.ntasks; task += nwaves - hwaves) {
    unsigned const q0 = p.tstart[task], q1 = p.tstart[task + 1];
    if (q0 == q1) continue;
    if (!by_source) {
      // skip a task whose words hold no active vertex
      unsigned const w0 = p.nzi[q0] >> 6, w1 = p.nzi[q1 - 1] >> 6;
      bool any = false;
      for (unsigned w = w0 + lane; w <= w1; w += 64) any = any || in[w] != 0ull;
      if (!ballot64(any)) continue;
    }
    unsigned const eb = p.nzR[q0];
    // 1. segment heads: (position + 1) << 12 | in-edges << 1, or with no edges
    // and the low bit for a vertex not computed here.  What the folds need of
    // the first 64 vertices (mostly all of them) is loaded now.
#pragma unroll
    for (unsigned r = 0; r < kRows; ++r) head[r * 64 + lane] = 0u;
    for (unsigned i = lane; i < (S::task_edges + 31) / 32; i += 64) act[i] = 0u;
    wave_lds_sync();
    unsigned tend = 0, longest = 0;
    unsigned pos0 = 0, len0 = 0, v0 = 0, ob0 = 0, oe0 = 0;
    vT old0{};
    for (unsigned g = q0; g < q1; g += 64) {
      unsigned const q = g + lane;
      if (q < q1) {
        unsigned const a = p.nzR[q], b = p.nzR[q + 1], v = p.nzi[q];
        bool on = b - a <= S::light;
        if (on && !by_source) on = ordered_bit(in, v);
        head[a - eb] = ((a - eb + 1u) << 12) | (on ? (b - a) << 1 : 1u);
        if (on) {
          tend = b - eb > tend ? b - eb : tend;
          longest = b - a > longest ? b - a : longest;
        }
        if (g == q0) {
          pos0 = a - eb;
          len0 = on ? b - a : 0u;
          v0 = v;
          if (on) {
            old0 = Vin[v];
            ob0 = p.oR[v];
            oe0 = p.oR[v + 1];
          }
        }
      }
    }
    tend = wave_max(tend);
    longest = wave_max(longest);
    wave_lds_sync();
    if (tend == 0) continue;
    // 2. every edge's segment (a running maximum of the heads) and partial;
    // lanes without an edge of their own read the task's first one
    unsigned seg[kRows];
    unsigned carry = 0;
#pragma unroll
    for (unsigned r0 = 0; r0 < kRows; r0 += kB) {
#pragma unroll
      for (unsigned u = 0; u < kB; ++u) seg[r0 + u] = 0u;
      if (r0 * 64 >= tend) continue;
      unsigned src[kB], e[kB];
      bool live[kB];
      eT w[kB];
      vT x[kB];
#pragma unroll
      for (unsigned u = 0; u < kB; ++u) {
        unsigned const pos = (r0 + u) * 64 + lane;
        unsigned s = wave_incl_max(head[pos]);
        s = s > carry ? s : carry;
        carry = readlane(s, 63);
        seg[r0 + u] = s;
        live[u] = pos < tend && !(s & 1u);
        e[u] = eb + (live[u] ? pos : 0u);
        src[u] = p.C[e[u]];
        w[u] = p.E[e[u]];
      }
      wave_lds_sync();   // the heads are read; their words may take the partials
#pragma unroll
      for (unsigned u = 0; u < kB; ++u) x[u] = Vin[src[u]];
      if (by_source) {
        unsigned long long wd[kB];
#pragma unroll
        for (unsigned u = 0; u < kB; ++u) wd[u] = in[src[u] >> 6];
#pragma unroll
        for (unsigned u = 0; u < kB; ++u) {
          unsigned const at = (seg[r0 + u] >> 12) - 1u;
          if (live[u] && ((wd[u] >> (src[u] & 63)) & 1ull)) atomicOr(act + (at >> 5), 1u << (at & 31));
        }
      }
#pragma unroll
      for (unsigned u = 0; u < kB; ++u) {
        ordered_touch(w[u]);
        if (kRead || live[u])
          edge_value_at(p.fn, slot[(r0 + u) * 64 + lane], x[u], p.E + e[u]);
      }
    }
    wave_lds_sync();
    // 3. the trees: the partner pos + s belongs to the same segment, and to
    // the same chunk (the offset is a multiple of 2s)
    for (unsigned s = 1; s < 64 && s < longest; s <<= 1) {
#pragma unroll
      for (unsigned r = 0; r < kRows; ++r) {
        if (r * 64 < tend) {
          unsigned const pos = r * 64 + lane;
          // (opaque copy: the offsets are recomputed per step instead of held
          // in registers for all rows)
          unsigned a = seg[r];
          asm volatile("" : "+v"(a));
          unsigned const rel = pos + 1u - (a >> 12);
          if ((rel & (2 * s - 1)) == 0 && rel + s < ((a >> 1) & 0x7ffu))
            reduce_at(p.fr, slot[pos], slot[pos + s]);
        }
      }
      wave_lds_sync();
    }
    // 4. the vertices' folds
    for (unsigned g = q0; g < q1; g += 64) {
      unsigned const q = g + lane;
      unsigned v = v0, len = len0, pos = pos0, ob = ob0, oe = oe0;
      vT old = old0;
      bool on = false;
      if (g != q0) {
        len = 0;
        if (q < q1) {
          unsigned const a = p.nzR[q];
          len = p.nzR[q + 1] - a;
          pos = a - eb;
          v = p.nzi[q];
          if (len > S::light || (!by_source && !ordered_bit(in, v))) len = 0;
          if (len) {
            old = Vin[v];
            ob = p.oR[v];
            oe = p.oR[v + 1];
          }
        }
      }
      if (len) on = !by_source || ((act[pos >> 5] >> (pos & 31)) & 1u) != 0u;
      bool moved = false;
      if (on) {
        init_at(p.fi, acc[lane], old);
        for (unsigned c = 0; c < len; c += 64) reduce_at(p.fr, acc[lane], slot[pos + c]);
        moved = update_at(p.fu, acc[lane], old);
        if (moved) Vout[v] = acc[lane];
      }
      ordered_publish(p, out, out_moved, ow, moved, v, ob, oe);
    }
    wave_lds_sync();
  }
  if (!by_source) {
    // active vertices without in-edges (none when a mover made them active)
    for (unsigned w = wave; w < p.nwords; w += nwaves) {
      unsigned long long const bits = in[w] & ~p.hasin[w];
      if (!bits) continue;
      unsigned const v = w * 64u + lane;
      bool moved = false;
      if (((bits >> lane) & 1ull) && v < p.n) {
        vT const old = Vin[v];
        init_at(p.fi, acc[lane], old);
        moved = update_at(p.fu, acc[lane], old);
        if (moved) Vout[v] = acc[lane];
      }
      unsigned const ob = moved ? p.oR[v] : 0u, oe = moved ? p.oR[v + 1] : 0u;
      ordered_publish(p, out, out_moved, ow, moved, v, ob, oe);
    }
  }
  {
    unsigned const mv = wave_sum(ow.moved);
    unsigned long long const oe = wave_sum64(ow.out_edges);
    if (lane == 0 && mv) {
      atomicAdd(&s_moved, mv);
      atomicMax(&s_most, ow.most);   // (uniform over the wave)
      atomicAdd(&s_out, oe);
    }
  }
  __syncthreads();
  if (t == 0) {
    if (s_moved) {
      ordered_slot* const g = p.ctl->slots + blockIdx.x % kTicketGroups;
      unsigned const r0 = atomicAdd(&g->moved, s_moved);
      unsigned const r1 = atomicMax(&g->most, s_most);
      unsigned long long const r2 = atomicAdd(&g->out_edges, s_out);
      asm volatile("" ::"v"(r0), "v"(r1), "v"(r2));
    }
    __builtin_amdgcn_s_waitcnt(0);
    s_last = take_ticket(p.ctl->board.w);
  }
  __syncthreads();
  if (!s_last || t >= 64) return;
  ordered_slot* const g = p.ctl->slots + lane;
  unsigned const mv = wave_sum(
      __hip_atomic_load(&g->moved, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u);
  unsigned long long const oe = wave_sum64(
      __hip_atomic_load(&g->out_edges, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  unsigned const most =
      wave_max(__hip_atomic_load(&g->most, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  g->moved = 0u;
  g->most = 0u;
  g->out_edges = 0ull;
  if (t == 0) {
    p.ctl->iter = iter + 1;
    if (mv == 0) p.ctl->done = 1;
    else if (iter + 1 >= p.ctl->max_iter) p.ctl->done = 2;   // limit reached, still moving
    p.ctl->in_moved = out_moved ? 1u : 0u;
    p.ctl->out_moved = oe * kDenseDiv >= p.m || most * kSerialDiv > p.m ? 1u : 0u;
  }
}

}  // namespace detail
}  // namespace kites

#endif  // KITES_DETAIL_ORDERED_KERNEL_HPP_
