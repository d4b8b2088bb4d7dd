// volatile_sets.hip -- functor sets in the reference's own form (volatile
// references, eT* edges) on the paths that the C ABI's plain-reference sets take:
// shortest paths under every variant and schedule, near-far, the one-workgroup
// loop and the K-wide batch, on 32-bit, 64-bit, signed and floating values.
#include "forms.hpp"
#include "native.hpp"

using namespace native;

namespace {

using eT = unsigned;

template <class vT>
constexpr vT inf() {
  return std::is_floating_point<vT>::value ? static_cast<vT>(1e30) : std::numeric_limits<vT>::max() / 4;
}

template <class vT>
struct add {
  __host__ __device__ void operator()(volatile vT& part, vT src, eT* e) const {
    part = src + static_cast<vT>(*e);
  }
};
template <class vT>
struct take_min {
  __host__ __device__ void operator()(volatile vT& l, volatile vT& r) const {
    if (l > r) l = r;
  }
};
template <class vT>
struct less {
  __host__ __device__ bool operator()(volatile vT& nv, vT old) const { return nv < old; }
};

csr random_graph(unsigned n, unsigned seed) {
  numbers rnd(seed);
  csr g;
  g.n = n;
  g.R.assign(1, 0);
  for (unsigned v = 0; v < n; ++v) {
    unsigned const d = v % 101 == 7 ? 900 : v % 13 == 5 ? 0 : 1 + rnd.below(11);
    uvec list(d);
    for (unsigned& s : list) s = rnd.below(3) ? rnd.below(n) : rnd.below(80);
    std::sort(list.begin(), list.end());
    g.C.insert(g.C.end(), list.begin(), list.end());
    g.R.push_back(g.m());
  }
  g.transpose();
  return g;
}

csr grid(unsigned rows, unsigned cols) {
  csr g;
  g.n = rows * cols;
  g.R.assign(1, 0);
  for (unsigned r = 0; r < rows; ++r)
    for (unsigned c = 0; c < cols; ++c) {
      unsigned const v = r * cols + c;
      if (r) g.C.push_back(v - cols);
      if (c) g.C.push_back(v - 1);
      if (c + 1 < cols) g.C.push_back(v + 1);
      if (r + 1 < rows) g.C.push_back(v + cols);
      g.R.push_back(g.m());
    }
  g.transpose();
  return g;
}

// In 64-bit integers (path sums of all types here are exact).
std::vector<long long> distances(csr const& g, std::vector<eT> const& w, unsigned src) {
  long long const far = 1ll << 60;
  std::vector<long long> V(g.n, far);
  V[src] = 0;
  for (bool moved = true; moved;) {
    moved = false;
    auto pass = [&](unsigned v) {
      for (unsigned e = g.R[v]; e < g.R[v + 1]; ++e)
        if (V[g.C[e]] != far && V[g.C[e]] + w[e] < V[v]) {
          V[v] = V[g.C[e]] + w[e];
          moved = true;
        }
    };
    for (unsigned v = 0; v < g.n; ++v) pass(v);
    for (unsigned v = g.n; v-- > 0;) pass(v);
  }
  return V;
}

struct problem {
  std::string name;
  csr g;
  std::vector<eT> w;
  unsigned src;
  std::vector<long long> want;
  template <class vT>
  std::vector<vT> wanted() const {
    std::vector<vT> r(g.n);
    for (unsigned v = 0; v < g.n; ++v) r[v] = want[v] == 1ll << 60 ? inf<vT>() : static_cast<vT>(want[v]);
    return r;
  }
};

template <class vT>
void run(problem const& p, kites::gpu& dev, const char* type, bool near_far) {
  auto d = upload<vT, eT>(p.g, p.w, dev);
  std::vector<vT> const want = p.wanted<vT>();
  std::vector<vT> V0(p.g.n, inf<vT>());
  V0[p.src] = 0;
  std::vector<char> active(p.g.n, 0);
  for (unsigned j = p.g.oR[p.src]; j < p.g.oR[p.src + 1]; ++j) active[p.g.oC[j]] = 1;
  auto one = [&](std::string const& how, kites::options o) {
    std::string const what = p.name + ", " + type + ", " + how;
    announce(what);
    start(*d, V0, active);
    kites::process<kites::launch::sync>(*d, dev, copy_init<true, vT>{}, add<vT>{}, take_min<vT>{},
                                        less<vT>{}, o);
    report(what, same(to_host(d->V.get_ptr(), p.g.n), want));
  };
  one("default", kites::options{});
  kites::options c;
  c.sched = kites::schedule::classic;
  one("classic", c);
  if (std::is_floating_point<vT>::value) return;     // (no delta schedules)
  for (unsigned v = 1; v <= 8; ++v) {
    kites::options o;
    o.sched = kites::schedule::forced;
    o.forced_variant = v;
    one("forced " + std::to_string(v), o);
  }
  kites::options s;
  s.sched = kites::schedule::plain;
  s.seed = kites::options::seeding::source;
  s.seed_source = p.src;
  for (bool loop : {true, false}) {
    s.persist = loop;
    s.delta = 0;
    one(loop ? "from its source" : "from its source, without the loop", s);
    for (unsigned delta : {20u, 300u}) {
      s.delta = delta;
      if (near_far)
        one("near-far " + std::to_string(delta) + (loop ? "" : ", without the loop"), s);
    }
  }
  s.persist = true;
  s.delta = 0;
  s.split_pull = true;
  s.alpha = 1e9f;
  one("split pulls", s);
}

// The K-wide batch, one column per source.
void batch(problem const& p, kites::gpu& dev) {
  using vT = unsigned;
  auto d = upload<vT, eT>(p.g, p.w, dev);
  uvec sources;
  for (unsigned k = 0; k < 5; ++k) sources.push_back((p.src + k * 37) % p.g.n);
  for (bool masks : {false, true}) {
    std::string const what = p.name + ", K-wide batch" + (masks ? " with masks" : "");
    announce(what);
    kites::device_buffer<vT> rows;
    kites::batch_options o;
    o.per_source_masks = masks;
    kites::process_batch<kites::launch::sync>(*d, dev, sources, vT(0), inf<vT>(), rows,
                                              copy_init<true, vT>{}, add<vT>{}, take_min<vT>{},
                                              less<vT>{}, o);
    std::vector<vT> const got = to_host(rows.get_ptr(), std::size_t(p.g.n) * 64);
    bool ok = true;
    for (unsigned k = 0; k < sources.size(); ++k) {
      std::vector<long long> const want = distances(p.g, p.w, sources[k]);
      for (unsigned v = 0; v < p.g.n; ++v)
        ok = ok && got[std::size_t(v) * 64 + k] ==
                       (want[v] == 1ll << 60 ? inf<vT>() : static_cast<vT>(want[v]));
    }
    report(what, ok);
  }
}

}  // namespace

int main() {
  kites::gpu dev(0);
  for (bool second : {false, true}) {
    problem p{second ? "grid" : "random", second ? grid(40, 120) : random_graph(4001, 9), {}, 0, {}};
    numbers rnd(2);
    p.w.resize(p.g.m());
    for (eT& x : p.w) x = 1 + rnd.below(60);
    for (unsigned v = 0; v < p.g.n && !second; ++v)
      if (p.g.oR[v + 1] - p.g.oR[v] > p.g.oR[p.src + 1] - p.g.oR[p.src]) p.src = v;
    p.want = distances(p.g, p.w, p.src);
    run<unsigned>(p, dev, "unsigned", true);
    run<int>(p, dev, "int", false);
    run<unsigned long long>(p, dev, "unsigned long long", true);
    run<long long>(p, dev, "long long", false);
    run<float>(p, dev, "float", false);
    run<double>(p, dev, "double", false);
    batch(p, dev);
  }
  return finish();
}
