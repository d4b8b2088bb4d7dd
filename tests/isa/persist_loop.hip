// persist_loop.hip -- instantiates the one-workgroup loop (plain and near-far)
// for a look at its generated code (tests/test_isa.py).
#include "kites/kites.hpp"

using vT = unsigned;
using namespace kites::detail;

auto fi = [] __host__ __device__(vT& loc, vT& glob) { loc = glob; };
auto fn = [] __host__ __device__(vT& part, vT src, vT* e) {
  vT const t = src + *e;
  part = t < src ? 0xFFFFFFFFu : t;
};
auto fr = [] __host__ __device__(vT& l, vT& r) {
  if (l > r) l = r;
};
auto fu = [] __host__ __device__(vT& nv, vT old) { return nv < old; };

using P = step_params<vT, vT, decltype(fi), decltype(fn), decltype(fr), decltype(fu)>;
template __global__ void kites::detail::persist_kernel<false, P>(P);
template __global__ void kites::detail::persist_kernel<true, P>(P);
