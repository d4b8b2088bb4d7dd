// native.hpp -- what the programs of this folder share: small random graphs in
// CSR form, their device copies, host references and the report of a check.
#ifndef KITES_TESTS_NATIVE_HPP_
#define KITES_TESTS_NATIVE_HPP_

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "kites/kites.hpp"

namespace native {

using uvec = std::vector<unsigned>;

// In-edge CSR (R, C) and its transpose; slot[j] is the in-edge that entry j of
// the out-lists is.
struct csr {
  unsigned n = 0;
  uvec R, C, oR, oC, slot;
  unsigned m() const { return static_cast<unsigned>(C.size()); }
  void transpose() {
    oR.assign(n + 1, 0);
    for (unsigned s : C) ++oR[s + 1];
    for (unsigned v = 0; v < n; ++v) oR[v + 1] += oR[v];
    oC.resize(C.size());
    slot.resize(C.size());
    uvec at(oR.begin(), oR.end() - 1);
    for (unsigned v = 0; v < n; ++v)
      for (unsigned e = R[v]; e < R[v + 1]; ++e) {
        unsigned const j = at[C[e]]++;
        oC[j] = v;
        slot[j] = e;
      }
  }
};

// Deterministic 32-bit numbers (xorshift).
struct numbers {
  unsigned long long s;
  explicit numbers(unsigned long long seed) : s(seed * 0x9E3779B97F4A7C15ull + 1) {}
  unsigned operator()() {
    s ^= s << 13;
    s ^= s >> 7;
    s ^= s << 17;
    return static_cast<unsigned>(s >> 32);
  }
  unsigned below(unsigned k) { return (*this)() % k; }
};

// A device graph with the edge values e (in in-edge order).
template <class vT, class eT>
std::unique_ptr<kites::graph_csr_device<vT, eT>> upload(csr const& g, std::vector<eT> const& e,
                                                        kites::gpu& dev) {
  std::vector<eT> oe(g.m());
  for (unsigned j = 0; j < g.m(); ++j) oe[j] = e[g.slot[j]];
  return std::unique_ptr<kites::graph_csr_device<vT, eT>>(new kites::graph_csr_device<vT, eT>(
      g.n, g.m(), g.R.data(), g.C.data(), e.data(), g.oR.data(), g.oC.data(), oe.data(),
      kites::graph_property::directed, dev));
}

template <class T>
void to_device(T* d, std::vector<T> const& h) {
  if (!h.empty())
    KITES_HIP_CHECK(hipMemcpy(d, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice));
}

template <class T>
std::vector<T> to_host(const T* d, std::size_t n) {
  std::vector<T> h(n);
  if (n) KITES_HIP_CHECK(hipMemcpy(h.data(), d, n * sizeof(T), hipMemcpyDeviceToHost));
  return h;
}

// Values and frontier (one flag per vertex) of the next run.
template <class G, class vT>
void start(G& d, std::vector<vT> const& v, std::vector<char> const& active) {
  to_device(d.V.get_ptr(), v);
  std::vector<unsigned long long> words(d.vBitmapEven.size(), 0ull);
  for (std::size_t i = 0; i < active.size(); ++i)
    if (active[i]) words[i >> 6] |= 1ull << (i & 63);
  to_device(d.vBitmapEven.get_ptr(), words);
  KITES_HIP_CHECK(hipDeviceSynchronize());
}

inline int& failures() {
  static int n = 0;
  return n;
}

// Prints a check's outcome; the case was printed (and flushed) before it ran.
inline void report(std::string const& what, bool ok) {
  if (!ok) ++failures();
  std::printf("%s: %s\n", ok ? "ok" : "FAILED", what.c_str());
  std::fflush(stdout);
}

inline void announce(std::string const& what) {
  std::printf("[case] %s\n", what.c_str());
  std::fflush(stdout);
}

// Byte-wise equality (NaN equals itself).
template <class T>
bool same(std::vector<T> const& a, std::vector<T> const& b) {
  return a.size() == b.size() && (a.empty() || !std::memcmp(a.data(), b.data(), a.size() * sizeof(T)));
}

inline int finish() {
  std::printf(failures() ? "%d checks failed\n" : "all checks passed\n", failures());
  return failures() ? 1 : 0;
}

}  // namespace native

#endif  // KITES_TESTS_NATIVE_HPP_
