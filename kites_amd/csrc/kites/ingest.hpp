// ingest.hpp -- a device graph built on the GPU from an edge list in HBM.
//
// Extension of the reference, which builds its graph on the host in one
// thread (kites/graph/graph_raw.h:58-190 and graph_csr.h:45-110; the
// startup bottleneck at R-MAT scale 22).  The arrays are the ones the host
// path produces for vertex-per-group 1:
//   * in-edge CSR R, C, E: in-list of v = the edges whose destination is v,
//     sorted by source id, duplicates kept in input order (graph_raw.h:102,
//     131-133; one of the orders its std::sort may produce, the one the
//     host build here produces);
//   * weighted out-edge CSR oR, oC, oE: out-list of u sorted by destination,
//     duplicates in in-list order (the host transpose);
//   * the non-empty vertex list (nzi, nzR) and the out-edge bitmap.
// With `dedup`, self-loops and every later copy of a (source, destination)
// pair are dropped (the generators' rule: the first copy keeps its weight).
// The vertex count is padded to a multiple of 128 (graph_raw.h:173-182).
//
// Two stable LSD radix sorts do the work: edges by the key (destination,
// source) with the weight as value, then the sorted edges by source with
// (destination, weight) as value.  Offsets are lower bounds over the sorted row
// ids; the non-empty list is a flag scan.  Sorting and scans use hipCUB
// (rocPRIM).  The values travel through the sorts, which read and write them in
// order: sorting positions instead and gathering by them afterwards cost two
// random gathers, 0.36 and 0.40 ms of 2.5 at 16M edges (10^6 vertices).
#ifndef KITES_INGEST_HPP_
#define KITES_INGEST_HPP_

#include <hip/hip_runtime.h>
#include <hipcub/device/device_radix_sort.hpp>
#include <hipcub/device/device_scan.hpp>

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <stdexcept>

#include "common.hpp"
#include "device.hpp"
#include "graph_device.hpp"
#include "memory.hpp"

namespace kites {
namespace detail {

constexpr unsigned kIngestBlock = 256;

inline unsigned ingest_grid(std::size_t items) {
  std::size_t const g = (items + kIngestBlock - 1) / kIngestBlock;
  return static_cast<unsigned>(g < 65535u * 16u ? (g ? g : 1) : 65535u * 16u);
}

// An out-CSR entry on its way through the second sort.
template <class eT>
struct ingest_out {
  unsigned dst;
  eT w;
};

// key[k] = (dst << nb) | src; bad[0] |= 1 for an endpoint >= n.
static __global__ void ingest_keys_kernel(const unsigned* __restrict__ src,
                                          const unsigned* __restrict__ dst, std::uint64_t m,
                                          unsigned n, unsigned nb, std::uint64_t* __restrict__ key,
                                          unsigned* __restrict__ bad) {
  std::uint64_t const stride = static_cast<std::uint64_t>(gridDim.x) * blockDim.x;
  bool oob = false;
  for (std::uint64_t k = static_cast<std::uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; k < m;
       k += stride) {
    unsigned const s = src[k], d = dst[k];
    oob |= (s >= n) || (d >= n);
    key[k] = (static_cast<std::uint64_t>(d) << nb) | s;
  }
  if (oob) atomicOr(bad, 1u);
}

// keep[i] = 1 unless dedup drops edge i of the sorted list (a self-loop, or
// the same key as edge i - 1).
static __global__ void ingest_keep_kernel(const std::uint64_t* __restrict__ key, std::uint64_t m,
                                          unsigned nb, int dedup, unsigned* __restrict__ keep) {
  std::uint64_t const stride = static_cast<std::uint64_t>(gridDim.x) * blockDim.x;
  std::uint64_t const mask = (std::uint64_t{1} << nb) - 1;
  for (std::uint64_t i = static_cast<std::uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < m;
       i += stride) {
    std::uint64_t const k = key[i];
    bool drop = false;
    if (dedup) drop = ((k >> nb) == (k & mask)) || (i > 0 && key[i - 1] == k);
    keep[i] = drop ? 0u : 1u;
  }
}

// Kept edge i (all of them without dedup: keep and pos null) goes to position
// pos[i]: C (source), E (weight), D (destination, the row id the offsets are
// searched in) and the second sort's value.
template <class eT>
__global__ void ingest_scatter_kernel(const std::uint64_t* __restrict__ key,
                                      const eT* __restrict__ w, const unsigned* __restrict__ keep,
                                      const unsigned* __restrict__ pos, std::uint64_t m,
                                      unsigned nb, unsigned* __restrict__ C, eT* __restrict__ E,
                                      unsigned* __restrict__ D, ingest_out<eT>* __restrict__ out) {
  std::uint64_t const stride = static_cast<std::uint64_t>(gridDim.x) * blockDim.x;
  std::uint64_t const mask = (std::uint64_t{1} << nb) - 1;
  for (std::uint64_t i = static_cast<std::uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < m;
       i += stride) {
    if (keep && !keep[i]) continue;
    std::uint64_t const p = pos ? pos[i] : i;
    std::uint64_t const k = key[i];
    eT const x = w[i];
    C[p] = static_cast<unsigned>(k & mask);
    D[p] = static_cast<unsigned>(k >> nb);
    E[p] = x;
    out[p] = ingest_out<eT>{static_cast<unsigned>(k >> nb), x};
  }
}

// off[v] = number of entries of the sorted `rows` below v, v = 0..n.
static __global__ void ingest_offsets_kernel(const unsigned* __restrict__ rows, unsigned m,
                                             unsigned n, unsigned* __restrict__ off) {
  unsigned const stride = gridDim.x * blockDim.x;
  for (unsigned v = blockIdx.x * blockDim.x + threadIdx.x; v <= n; v += stride) {
    unsigned lo = 0, hi = m;
    while (lo < hi) {
      unsigned const mid = lo + (hi - lo) / 2;
      if (rows[mid] < v) lo = mid + 1;
      else hi = mid;
    }
    off[v] = lo;
  }
}

// The sorted out-CSR entries into the graph's two arrays.
template <class eT>
__global__ void ingest_out_kernel(const ingest_out<eT>* __restrict__ in, unsigned m,
                                  unsigned* __restrict__ oC, eT* __restrict__ oE) {
  unsigned const stride = gridDim.x * blockDim.x;
  for (unsigned j = blockIdx.x * blockDim.x + threadIdx.x; j < m; j += stride) {
    ingest_out<eT> const x = in[j];
    oC[j] = x.dst;
    oE[j] = x.w;
  }
}

static __global__ void ingest_nz_flags_kernel(const unsigned* __restrict__ R, unsigned n,
                                              unsigned* __restrict__ flag) {
  unsigned const stride = gridDim.x * blockDim.x;
  for (unsigned v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += stride)
    flag[v] = R[v + 1] > R[v] ? 1u : 0u;
}

// nzi[pos[v]] = v and nzR[pos[v]] = R[v] for every non-empty v; the last
// thread also writes nzR[nnz] = m.
static __global__ void ingest_nz_scatter_kernel(const unsigned* __restrict__ R, unsigned n,
                                                const unsigned* __restrict__ flag,
                                                const unsigned* __restrict__ pos,
                                                unsigned* __restrict__ nzi,
                                                unsigned* __restrict__ nzR) {
  unsigned const stride = gridDim.x * blockDim.x;
  for (unsigned v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += stride) {
    if (flag[v]) {
      nzi[pos[v]] = v;
      nzR[pos[v]] = R[v];
    }
    if (v == n - 1) nzR[pos[v] + flag[v]] = R[n];
  }
}

inline unsigned id_bits(std::size_t n) {
  unsigned b = 1;
  while (b < 32 && (std::size_t{1} << b) < n) ++b;
  return b;
}

}  // namespace detail

struct ingest_report {
  std::size_t n = 0;          // padded vertex count
  std::size_t m = 0;          // edges kept
  float build_ms = 0.f;       // device time from the edge list in HBM to the finished graph
};

// Builds the device graph from m edges (src[k] -> dst[k], weight w[k]) held in
// device memory on `dev`.  n: vertex ids are < n; the graph has n rounded up
// to a multiple of 128 vertices.  Throws std::invalid_argument for an
// endpoint >= n or more than 2^32 - 1 edges.
template <class vT, class eT, class vIdxT>
graph_csr_device<vT, eT, vIdxT> make_graph_csr_from_edges(gpu& dev, std::size_t n, std::size_t m,
                                                           const vIdxT* src, const vIdxT* dst,
                                                           const eT* w, bool dedup,
                                                           ingest_report* rep = nullptr) {
  using namespace detail;
  static_assert(sizeof(vIdxT) == 4, "32-bit vertex ids");
  if (m >= 0xffffffffull) throw std::invalid_argument("ingest: at most 2^32 - 2 edges");
  if (n == 0) throw std::invalid_argument("ingest: a graph needs at least one vertex");
  if (n > 0xffffffffull - 256) throw std::invalid_argument("ingest: too many vertices");
  dev.setAsActive();
  int const did = dev.getDevIdx();
  stream& s = dev.getSsEven();
  std::size_t const np = n % VERTEX_PADDING ? (n / VERTEX_PADDING + 1) * VERTEX_PADDING : n;
  unsigned const nb = id_bits(np);
  hipEvent_t e0, e1;
  KITES_HIP_CHECK(hipEventCreate(&e0));
  KITES_HIP_CHECK(hipEventCreate(&e1));
  KITES_HIP_CHECK(hipEventRecord(e0, s.get()));

  // One scratch allocation: the sorts' keys and values in and out, the sorts'
  // and scans' own space, the row ids, flags and positions.  The second sort's
  // values and rows lie where the first one's keys and weights are done with.
  std::uint64_t *keyA = nullptr, *keyB = nullptr;
  eT* wB = nullptr;
  ingest_out<eT> *outA = nullptr, *outB = nullptr;
  unsigned *keep = nullptr, *pos = nullptr, *D = nullptr, *rows = nullptr, *bad = nullptr;
  unsigned *flag = nullptr, *fpos = nullptr;
  unsigned char* tmp = nullptr;
  std::size_t tb = 0, t1 = 0, t2 = 0, t3 = 0, t4 = 0;
  const unsigned* const no_keys = nullptr;
  if (m) {
    KITES_HIP_CHECK(hipcub::DeviceRadixSort::SortPairs(nullptr, t1, keyA, keyB, w, wB, m, 0,
                                                       static_cast<int>(2 * nb), s.get()));
    KITES_HIP_CHECK(hipcub::DeviceRadixSort::SortPairs(nullptr, t2, no_keys, rows, outA, outB, m, 0,
                                                       static_cast<int>(nb), s.get()));
    if (dedup)
      KITES_HIP_CHECK(hipcub::DeviceScan::ExclusiveSum(nullptr, t3, keep, pos, m, s.get()));
  }
  KITES_HIP_CHECK(hipcub::DeviceScan::ExclusiveSum(nullptr, t4, flag, fpos, np, s.get()));
  tb = std::max(std::max(t1, t2), std::max(t3, t4));
  device_arena scratch;
  scratch.begin();
  std::size_t const pair = std::max(sizeof(std::uint64_t), sizeof(ingest_out<eT>));
  unsigned char *pairA = nullptr, *pairB = nullptr, *wordB = nullptr;
  scratch.add(pairA, m * pair);
  scratch.add(pairB, m * pair);
  scratch.add(wordB, m * std::max(sizeof(eT), sizeof(unsigned)));
  scratch.add(D, m);
  scratch.add(keep, dedup ? m : 0);
  scratch.add(pos, dedup ? m : 0);
  scratch.add(flag, np);
  scratch.add(fpos, np);
  scratch.add(bad, 1);
  scratch.add(tmp, tb);
  scratch.commit(did);
  keyA = reinterpret_cast<std::uint64_t*>(pairA);   // read by the first sort
  outA = reinterpret_cast<ingest_out<eT>*>(pairA);  // written after it
  keyB = reinterpret_cast<std::uint64_t*>(pairB);   // read by the scatter
  outB = reinterpret_cast<ingest_out<eT>*>(pairB);  // written after it
  wB = reinterpret_cast<eT*>(wordB);
  rows = reinterpret_cast<unsigned*>(wordB);
  if (!dedup) keep = pos = nullptr;
  std::size_t mk = m;   // edges kept
  graph_csr_device<vT, eT, vIdxT> g(np, dev);
  if (m) {
    hipLaunchKernelGGL(zero_words_kernel, dim3(1), dim3(64), 0, s.get(), bad, 1u);
    hipLaunchKernelGGL(ingest_keys_kernel, dim3(ingest_grid(m)), dim3(kIngestBlock), 0, s.get(),
                       reinterpret_cast<const unsigned*>(src),
                       reinterpret_cast<const unsigned*>(dst), static_cast<std::uint64_t>(m),
                       static_cast<unsigned>(n), nb, keyA, bad);
    KITES_HIP_CHECK(hipPeekAtLastError());
    // 1. edges by (destination, source), stable: duplicates keep input order
    KITES_HIP_CHECK(hipcub::DeviceRadixSort::SortPairs(tmp, tb, keyA, keyB, w, wB, m, 0,
                                                       static_cast<int>(2 * nb), s.get()));
    // 2. kept edges and their positions
    unsigned last[2] = {0, 0};
    if (dedup) {
      hipLaunchKernelGGL(ingest_keep_kernel, dim3(ingest_grid(m)), dim3(kIngestBlock), 0, s.get(),
                         keyB, static_cast<std::uint64_t>(m), nb, 1, keep);
      KITES_HIP_CHECK(hipPeekAtLastError());
      KITES_HIP_CHECK(hipcub::DeviceScan::ExclusiveSum(tmp, tb, keep, pos, m, s.get()));
      KITES_HIP_CHECK(hipMemcpyAsync(&last[0], pos + (m - 1), 4, hipMemcpyDeviceToHost, s.get()));
      KITES_HIP_CHECK(hipMemcpyAsync(&last[1], keep + (m - 1), 4, hipMemcpyDeviceToHost, s.get()));
    }
    unsigned hbad = 0;
    KITES_HIP_CHECK(hipMemcpyAsync(&hbad, bad, 4, hipMemcpyDeviceToHost, s.get()));
    s.sync();
    if (hbad) {
      (void)hipEventDestroy(e0);
      (void)hipEventDestroy(e1);
      throw std::invalid_argument("ingest: edge endpoint out of range");
    }
    if (dedup) mk = static_cast<std::size_t>(last[0]) + last[1];
  }
  // the graph's edge arrays; the non-empty list holds at most np vertices
  std::size_t const nz_cap = std::min(np, mk);
  g.edge_arena.begin();
  g.edge_arena.add(g.C, mk ? mk : 1, did);
  g.edge_arena.add(g.E, mk ? mk : 1, did);
  g.edge_arena.add(g.oC, mk ? mk : 1, did);
  g.edge_arena.add(g.oE, mk ? mk : 1, did);
  g.edge_arena.add(g.nzi, nz_cap ? nz_cap : 1, did);
  g.edge_arena.add(g.nzR, nz_cap + 1, did);
  g.edge_arena.commit(did);
  if (m) {
    hipLaunchKernelGGL(ingest_scatter_kernel<eT>, dim3(ingest_grid(m)), dim3(kIngestBlock), 0,
                       s.get(), keyB, wB, keep, pos, static_cast<std::uint64_t>(m), nb,
                       reinterpret_cast<unsigned*>(g.C.get_ptr()), g.E.get_ptr(), D, outA);
    KITES_HIP_CHECK(hipPeekAtLastError());
  }
  unsigned const m32 = static_cast<unsigned>(mk);
  hipLaunchKernelGGL(ingest_offsets_kernel, dim3(ingest_grid(np + 1)), dim3(kIngestBlock), 0,
                     s.get(), D, m32, static_cast<unsigned>(np),
                     reinterpret_cast<unsigned*>(g.R.get_ptr()));
  KITES_HIP_CHECK(hipPeekAtLastError());
  // 3. out-CSR: the in-CSR order sorted by source, stable
  if (mk) {
    const unsigned* const ckeys = reinterpret_cast<const unsigned*>(g.C.get_ptr());
    KITES_HIP_CHECK(hipcub::DeviceRadixSort::SortPairs(tmp, tb, ckeys, rows, outA, outB, mk, 0,
                                                       static_cast<int>(nb), s.get()));
    hipLaunchKernelGGL(ingest_out_kernel<eT>, dim3(ingest_grid(mk)), dim3(kIngestBlock), 0,
                       s.get(), outB, m32, reinterpret_cast<unsigned*>(g.oC.get_ptr()),
                       g.oE.get_ptr());
    KITES_HIP_CHECK(hipPeekAtLastError());
  }
  hipLaunchKernelGGL(ingest_offsets_kernel, dim3(ingest_grid(np + 1)), dim3(kIngestBlock), 0,
                     s.get(), rows, m32, static_cast<unsigned>(np),
                     reinterpret_cast<unsigned*>(g.oR.get_ptr()));
  KITES_HIP_CHECK(hipPeekAtLastError());
  // 4. vertices with in-edges
  {
    const unsigned* const R = reinterpret_cast<const unsigned*>(g.R.get_ptr());
    hipLaunchKernelGGL(ingest_nz_flags_kernel, dim3(ingest_grid(np)), dim3(kIngestBlock), 0,
                       s.get(), R, static_cast<unsigned>(np), flag);
    KITES_HIP_CHECK(hipPeekAtLastError());
    KITES_HIP_CHECK(hipcub::DeviceScan::ExclusiveSum(tmp, tb, flag, fpos, np, s.get()));
    unsigned last[2] = {0, 0};
    KITES_HIP_CHECK(hipMemcpyAsync(&last[0], fpos + (np - 1), 4, hipMemcpyDeviceToHost, s.get()));
    KITES_HIP_CHECK(hipMemcpyAsync(&last[1], flag + (np - 1), 4, hipMemcpyDeviceToHost, s.get()));
    hipLaunchKernelGGL(ingest_nz_scatter_kernel, dim3(ingest_grid(np)), dim3(kIngestBlock), 0,
                       s.get(), R, static_cast<unsigned>(np), flag, fpos,
                       reinterpret_cast<unsigned*>(g.nzi.get_ptr()),
                       reinterpret_cast<unsigned*>(g.nzR.get_ptr()));
    KITES_HIP_CHECK(hipPeekAtLastError());
    s.sync();
    g.nnz = last[0] + last[1];
  }
  g.set_num_edges(mk);
  g.build_outbits(np, s);
  KITES_HIP_CHECK(hipEventRecord(e1, s.get()));
  s.sync();
  float ms = 0.f;
  KITES_HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (rep) {
    rep->n = np;
    rep->m = mk;
    rep->build_ms = ms;
  }
  return g;
}

}  // namespace kites

#endif  // KITES_INGEST_HPP_
