// functor_sets.hpp -- the C ABI's fixed functor sets (KITES_ALGO_*), each
// written as the reference's four __host__ __device__ lambdas
// (README.md:16-23) with plain references in place of the volatile ones, so
// that their operands stay in registers, and the edge as a pointer to const
// (kites/detail/functor_call.hpp);
// shared by the C-ABI translation units.
#ifndef KITES_AMD_FUNCTOR_SETS_HPP_
#define KITES_AMD_FUNCTOR_SETS_HPP_

#include <stdexcept>

#include "../../include/kites_amd.h"

namespace kites_capi {

// Runs `body(initF, nbrCompF, redF, updF)` with the lambdas of the
// saturating SSSP set (KITES_ALGO_SSSP).
template <class Body>
void with_sssp(Body&& body) {
  using vT = unsigned;
  using eT = unsigned;
  auto initF = [] __host__ __device__(vT& locV, vT& globV) { locV = globV; };
  // (an unreached source needs no test of its own: 0xFFFFFFFF plus any weight
  // saturates.  With one the compiler moves the weight's load behind it, 0.2 us
  // of a 2.7 us near-far iteration of the one-workgroup loop)
  auto nbr = [] __host__ __device__(vT& partialV, vT srcV, const eT* connE) {
    vT const t = srcV + *connE;
    partialV = t < srcV ? 0xFFFFFFFFu : t;
  };
  auto redMin = [] __host__ __device__(vT& lhsV, vT& rhsV) {
    if (lhsV > rhsV) lhsV = rhsV;
  };
  auto updLess = [] __host__ __device__(vT& newV, vT oldV) { return newV < oldV; };
  body(initF, nbr, redMin, updLess);
}

// Runs `body(initF, nbrCompF, redF, updF)` with the lambdas of functor set
// `algo`.
template <class Body>
void with_functors(int algo, Body&& body) {
  using vT = unsigned;
  using eT = unsigned;
  auto initF = [] __host__ __device__(vT& locV, vT& globV) { locV = globV; };
  auto redMin = [] __host__ __device__(vT& lhsV, vT& rhsV) {
    if (lhsV > rhsV) lhsV = rhsV;
  };
  auto updLess = [] __host__ __device__(vT& newV, vT oldV) { return newV < oldV; };
  switch (algo) {
    case KITES_ALGO_SSSP:
      with_sssp(body);
      break;
    case KITES_ALGO_BFS: {
      auto nbr = [] __host__ __device__(vT& partialV, vT srcV, const eT*) {
        partialV = (srcV == 0xFFFFFFFFu) ? 0xFFFFFFFFu : srcV + 1u;
      };
      body(initF, nbr, redMin, updLess);
      break;
    }
    case KITES_ALGO_CC: {
      auto nbr = [] __host__ __device__(vT& partialV, vT srcV, const eT*) { partialV = srcV; };
      body(initF, nbr, redMin, updLess);
      break;
    }
    case KITES_ALGO_SSSP_WRAP: {
      auto nbr = [] __host__ __device__(vT& partialV, vT srcV, const eT* connE) {
        partialV = srcV + (*connE);
      };
      body(initF, nbr, redMin, updLess);
      break;
    }
    case KITES_ALGO_WIDEST: {
      auto nbr = [] __host__ __device__(vT& partialV, vT srcV, const eT* connE) {
        vT const w = *connE;
        partialV = srcV < w ? srcV : w;
      };
      auto redMax = [] __host__ __device__(vT& lhsV, vT& rhsV) {
        if (lhsV < rhsV) lhsV = rhsV;
      };
      auto updMore = [] __host__ __device__(vT& newV, vT oldV) { return newV > oldV; };
      body(initF, nbr, redMax, updMore);
      break;
    }
    default:
      throw std::invalid_argument("unknown functor set");
  }
}

}  // namespace kites_capi

#endif  // KITES_AMD_FUNCTOR_SETS_HPP_
