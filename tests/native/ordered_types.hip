// ordered_types.hip -- options::ordered on value types of 4 to 32 bytes, bit
// for bit against the combine order's definition run on the host, and the calls
// of a functor that writes its edges.
//
// The graph has no cycles (every source id is below its destination's), so any
// functor set settles; in-lists of 1 to 64 edges lie side by side, so that a
// task's window holds more than 256 light in-edges, with lists at both sides of
// the light limit (64) and of a window (448) between them.
#include "forms.hpp"
#include "native.hpp"

using namespace native;

namespace {

csr layered(unsigned seed) {
  numbers rnd(seed);
  uvec degs;
  for (unsigned d : {1u, 2u, 3u, 31u, 32u, 33u, 63u, 64u, 65u, 127u, 128u, 129u, 447u, 448u, 449u, 1000u})
    degs.push_back(d);
  // light lists that end a window at 447, 448 and 449 edges
  for (unsigned last : {63u, 64u, 1u}) {
    for (unsigned i = 0; i < 6; ++i) degs.push_back(64);
    degs.push_back(last);
  }
  for (unsigned i = 0; i < 900; ++i) degs.push_back(i % 5 == 4 ? 0 : 1 + rnd.below(64));
  csr g;
  g.n = static_cast<unsigned>(degs.size()) + 41;
  g.R.assign(1, 0);
  for (unsigned v = 0; v < g.n; ++v) {
    unsigned const d = v < 40 || v - 40 >= degs.size() ? 0 : degs[v - 40];
    uvec list(d);
    for (unsigned& s : list) s = rnd.below(v);
    std::sort(list.begin(), list.end());
    g.C.insert(g.C.end(), list.begin(), list.end());
    g.R.push_back(g.m());
  }
  g.transpose();
  return g;
}

// Order-sensitive values of any size: every byte takes part.
template <unsigned BYTES>
struct mixed {
  static constexpr unsigned words = BYTES / 4;
  unsigned w[words];
  __host__ __device__ bool operator==(mixed const& o) const {
    for (unsigned i = 0; i < words; ++i)
      if (w[i] != o.w[i]) return false;
    return true;
  }
};

template <class T>
__host__ __device__ inline T make(unsigned x) {
  T r{};
  if constexpr (std::is_arithmetic<T>::value) {
    r = static_cast<T>(x % 1021u);
  } else {
    for (unsigned i = 0; i < T::words; ++i) r.w[i] = x * 2654435761u + i;
  }
  return r;
}

template <class T>
__host__ __device__ inline T scale(T v, unsigned e) {
#pragma clang fp contract(off)
  T r{};
  if constexpr (std::is_floating_point<T>::value) {
    r = v * (static_cast<T>(1) / static_cast<T>(3u + e));
  } else if constexpr (std::is_arithmetic<T>::value) {
    r = static_cast<T>(v * (2u * e + 1u));
  } else {
    for (unsigned i = 0; i < T::words; ++i) r.w[i] = v.w[i] * (2u * e + 1u) + i;
  }
  return r;
}

template <class T>
__host__ __device__ inline T fold(T a, T b) {
#pragma clang fp contract(off)
  T r{};
  if constexpr (std::is_floating_point<T>::value) {
    r = a + b;
  } else if constexpr (std::is_arithmetic<T>::value) {
    r = static_cast<T>(a * 3u + b);
  } else {
    for (unsigned i = 0; i < T::words; ++i) r.w[i] = a.w[i] * 31u + b.w[(i + 1) % T::words];
  }
  return r;
}

// The definition (detail/ordered_kernel.hpp): returns the iterations.
template <class vT, class eT, class FI, class FN, class FR, class FU>
unsigned reference(csr const& g, std::vector<eT>& E, std::vector<vT>& V, std::vector<char> active,
                   FI fi, FN fn, FR fr, FU fu) {
  using namespace kites::detail;
  for (unsigned iter = 1;; ++iter) {
    std::vector<vT> out = V;
    std::vector<char> next(g.n, 0);
    bool moved = false;
    for (unsigned v = 0; v < g.n; ++v) {
      if (!active[v]) continue;
      vT acc{};
      init_at(fi, acc, V[v]);
      for (unsigned c0 = g.R[v]; c0 < g.R[v + 1]; c0 += 64) {
        unsigned const k = std::min(64u, g.R[v + 1] - c0);
        vT x[64] = {};
        for (unsigned l = 0; l < k; ++l) edge_value_at(fn, x[l], V[g.C[c0 + l]], &E[c0 + l]);
        for (unsigned s = 1; s < 64; s <<= 1)
          for (unsigned l = 0; l + s < k; l += 2 * s) reduce_at(fr, x[l], x[l + s]);
        reduce_at(fr, acc, x[0]);
      }
      if (update_at(fu, acc, V[v])) {
        out[v] = acc;
        moved = true;
        for (unsigned j = g.oR[v]; j < g.oR[v + 1]; ++j) next[g.oC[j]] = 1;
      }
    }
    V.swap(out);
    active.swap(next);
    if (!moved) return iter;
  }
}

template <class vT>
void run(csr const& g, kites::gpu& dev, const char* name) {
  using eT = unsigned;
  std::vector<eT> E(g.m());
  numbers rnd(11);
  for (eT& e : E) e = 1 + rnd.below(9);
  std::vector<vT> V0(g.n);
  for (unsigned v = 0; v < g.n; ++v) V0[v] = make<vT>(v + 1);
  auto fi = [] __host__ __device__(vT & loc, vT&) { loc = make<vT>(7); };
  auto fn = [] __host__ __device__(vT & part, vT src, const eT* e) { part = scale(src, *e); };
  auto fr = [] __host__ __device__(vT & l, vT & r) { l = fold(l, r); };
  auto fu = [] __host__ __device__(vT & nv, vT old) { return !(nv == old); };
  for (unsigned some : {0u, 1u}) {
    // every vertex active, or one in nine
    std::vector<char> active(g.n, 1);
    if (some)
      for (unsigned v = 0; v < g.n; ++v) active[v] = v % 9 == 4;
    std::string const what = std::string("ordered ") + name + (some ? ", some active" : ", all active");
    announce(what);
    std::vector<vT> exp = V0;
    std::vector<eT> e2 = E;
    unsigned const it = reference(g, e2, exp, active, fi, fn, fr, fu);
    auto d = upload<vT, eT>(g, E, dev);
    start(*d, V0, active);
    kites::run_report rep;
    kites::options o;
    o.ordered = true;
    o.report = &rep;
    kites::process<kites::launch::sync>(*d, dev, fi, fn, fr, fu, o);
    report(what, rep.iterations == it && same(to_host(d->V.get_ptr(), g.n), exp));
  }
}

// A functor that writes the edge counts its calls there: once per iteration and
// in-edge of the active vertices, as the definition has it.
struct counted {
  unsigned w, calls;
};
template <bool VOL, class vT>
struct counting {
  __host__ __device__ void operator()(ref<VOL, vT> part, vT src, counted* e) const {
    e->calls += 1;
    part = scale(src, e->w);
  }
};
template <bool VOL, class vT>
struct sum {
  __host__ __device__ void operator()(ref<VOL, vT> l, ref<VOL, vT> r) const {
    vT const a = l, b = r;
    l = fold(a, b);
  }
};
template <bool VOL, class vT>
struct seven {
  __host__ __device__ void operator()(ref<VOL, vT> loc, vT&) const { loc = make<vT>(7); }
};
template <bool VOL, class vT>
struct moves {
  __host__ __device__ bool operator()(ref<VOL, vT> nv, vT old) const {
    vT const x = nv;
    return !(x == old);
  }
};

template <bool VOL, class vT>
void calls(csr const& g, kites::gpu& dev, const char* name) {
  std::vector<counted> E(g.m());
  numbers rnd(12);
  for (counted& e : E) e = counted{1 + rnd.below(9), 0};
  std::vector<vT> V0(g.n);
  for (unsigned v = 0; v < g.n; ++v) V0[v] = make<vT>(v + 1);
  for (unsigned some : {0u, 1u}) {
    std::vector<char> active(g.n, 1);
    if (some)
      for (unsigned v = 0; v < g.n; ++v) active[v] = v % 9 == 4;
    std::string const what = std::string("ordered calls, ") + name + (VOL ? ", volatile" : ", plain") +
                             (some ? ", some active" : ", all active");
    announce(what);
    std::vector<vT> exp = V0;
    std::vector<counted> e2 = E;
    unsigned const it = reference(g, e2, exp, active, seven<VOL, vT>{}, counting<VOL, vT>{},
                                  sum<VOL, vT>{}, moves<VOL, vT>{});
    auto d = upload<vT, counted>(g, E, dev);
    start(*d, V0, active);
    kites::run_report rep;
    kites::options o;
    o.ordered = true;
    o.report = &rep;
    kites::process<kites::launch::sync>(*d, dev, seven<VOL, vT>{}, counting<VOL, vT>{},
                                        sum<VOL, vT>{}, moves<VOL, vT>{}, o);
    report(what, rep.iterations == it && same(to_host(d->V.get_ptr(), g.n), exp) &&
                     same(to_host(d->E.get_ptr(), g.m()), e2));
  }
}

}  // namespace

int main() {
  kites::gpu dev(0);
  csr const g = layered(5);
  run<float>(g, dev, "float");
  run<double>(g, dev, "double");
  run<long long>(g, dev, "long long");
  run<mixed<12>>(g, dev, "12-byte struct");
  run<mixed<16>>(g, dev, "16-byte struct");
  run<mixed<32>>(g, dev, "32-byte struct");
  calls<false, float>(g, dev, "float");
  calls<true, float>(g, dev, "float");
  calls<false, long long>(g, dev, "long long");
  calls<true, long long>(g, dev, "long long");
  return finish();
}
