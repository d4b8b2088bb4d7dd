// ordered_capi.hip -- C ABI of the ordered mode (declarations in
// include/kites_amd.h): float PageRank, a functor set whose reduction is a
// floating-point sum, run with options::ordered so the result is defined bit
// for bit.
#include "capi_internal.hpp"

namespace {

using kites_capi::need;

// in-edge weight 1 / outdeg(source), as float
static __global__ void inv_outdeg_kernel(const unsigned* __restrict__ oR,
                                         const unsigned* __restrict__ C, unsigned m,
                                         float* __restrict__ W) {
  unsigned const stride = gridDim.x * blockDim.x;
  for (unsigned e = blockIdx.x * blockDim.x + threadIdx.x; e < m; e += stride) {
    unsigned const u = C[e];
    W[e] = 1.0f / static_cast<float>(oR[u + 1] - oR[u]);
  }
}

static __global__ void fill_kernel(float* __restrict__ V, unsigned n, float x) {
  unsigned const stride = gridDim.x * blockDim.x;
  for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) V[i] = x;
}

}  // namespace

extern "C" {

int kites_pagerank_f32(kites_graph* g, float damping, float tol, uint32_t max_iterations,
                       float* out, kites_run_info* info) {
  KITES_API_BEGIN
  need(g != nullptr && g->g, "null graph");
  need(damping >= 0.f && damping <= 1.f, "damping must be in [0, 1]");
  need(tol >= 0.f, "tolerance must be non-negative");
  auto& src = *g->g;
  kites::gpu& dev = *g->dev;
  int const did = dev.getDevIdx();
  std::size_t const n = g->n;
  std::size_t const m = g->m;
  // The float values and the weights 1 / outdeg(source) in the handle's
  // PageRank buffer; the graph's arrays are read where they are.
  kites::stream& s = dev.getSsEven();
  dev.setAsActive();
  if (g->pr.size() < n + m) {
    g->pr.free();
    g->pr.alloc(n + m, did);
  }
  float* const V = g->pr.get_ptr();
  float* const W = V + n;
  unsigned const cus = static_cast<unsigned>(dev.numComputeUnits());
  if (m)
    hipLaunchKernelGGL(inv_outdeg_kernel, dim3(cus * 8), dim3(256), 0, s.get(),
                       reinterpret_cast<const unsigned*>(src.oR.get_ptr()),
                       reinterpret_cast<const unsigned*>(src.C.get_ptr()),
                       static_cast<unsigned>(m), W);
  // every vertex starts at 1 and active
  hipLaunchKernelGGL(fill_kernel, dim3(cus * 8), dim3(256), 0, s.get(), V,
                     static_cast<unsigned>(n), 1.0f);
  KITES_HIP_CHECK(hipPeekAtLastError());
  kites::detail::ordered_view<float, float> f;
  f.n = n;
  f.m = m;
  f.R = src.R.get_ptr();
  f.C = src.C.get_ptr();
  f.E = W;
  f.oR = src.oR.get_ptr();
  f.oC = src.oC.get_ptr();
  f.nzi = src.nzi.get_ptr();
  f.nzR = src.nzR.get_ptr();
  f.nnz = src.nnz;
  f.V = V;
  f.frontier = nullptr;
  f.frontier_bytes = 0;

  // Plain-reference functors (operands in registers); no contraction: a
  // product and a sum each round on their own, as the combine order defines.
  float const base = 1.0f - damping;
  auto initF = [base] __host__ __device__(float& locV, float&) { locV = base; };
  auto nbrF = [damping] __host__ __device__(float& partialV, float srcV, const float* connE) {
#pragma clang fp contract(off)
    partialV = damping * srcV * (*connE);
  };
  auto redF = [] __host__ __device__(float& lhsV, float& rhsV) {
#pragma clang fp contract(off)
    lhsV = lhsV + rhsV;
  };
  auto updF = [tol] __host__ __device__(float& newV, float oldV) {
#pragma clang fp contract(off)
    float const d = newV - oldV;
    return d > tol || d < -tol;
  };
  kites::run_report rep;
  kites::options o;
  o.ordered = true;
  o.max_iterations = max_iterations ? max_iterations : 10000u;
  o.report = &rep;
  kites::detail::run_ordered(f, dev, s, g->pr_ws, initF, nbrF, redF, updF, o);
  if (out && n)
    kites_capi::copy_columns(reinterpret_cast<unsigned*>(out), reinterpret_cast<const unsigned*>(V),
                             n, 1u, 1u, did, s.get());
  if (info) {
    info->iterations = rep.iterations;
    info->ms = static_cast<float>(rep.ms);
    info->delta = 0;
    info->min_fast = 0;
    info->graph_builds = 0;
  }
  KITES_API_END
}

}  // extern "C"
