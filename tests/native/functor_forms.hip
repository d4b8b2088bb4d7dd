// functor_forms.hip -- a max-min functor set (widest paths: no native min)
// through kites::process with every mix of reference forms (volatile or plain)
// of nbrCompF, redF and updF, under every schedule and variant.
#include "forms.hpp"
#include "native.hpp"

using namespace native;

namespace {

using vT = int;
using eT = unsigned;

csr random_graph(unsigned n, unsigned per, unsigned seed) {
  numbers rnd(seed);
  csr g;
  g.n = n;
  g.R.assign(1, 0);
  for (unsigned v = 0; v < n; ++v) {
    // a few hubs, some vertices without in-edges
    unsigned const d = v % 97 == 3 ? 700 : v % 11 == 5 ? 0 : 1 + rnd.below(2 * per - 1);
    uvec list(d);
    for (unsigned& s : list) s = rnd.below(3) ? rnd.below(n) : rnd.below(64);
    std::sort(list.begin(), list.end());
    g.C.insert(g.C.end(), list.begin(), list.end());
    g.R.push_back(g.m());
  }
  g.transpose();
  return g;
}

// A ring with chords: many iterations of small frontiers.
csr ring(unsigned n) {
  csr g;
  g.n = n;
  g.R.assign(1, 0);
  for (unsigned v = 0; v < n; ++v) {
    uvec list{(v + n - 1) % n, (v + n - 3) % n};
    std::sort(list.begin(), list.end());
    g.C.insert(g.C.end(), list.begin(), list.end());
    g.R.push_back(g.m());
  }
  g.transpose();
  return g;
}

std::vector<vT> widest(csr const& g, std::vector<eT> const& E, unsigned src) {
  std::vector<vT> V(g.n, 0);
  V[src] = 1 << 30;
  for (bool moved = true; moved;) {
    moved = false;
    for (unsigned v = 0; v < g.n; ++v)
      for (unsigned e = g.R[v]; e < g.R[v + 1]; ++e) {
        vT const c = std::min<vT>(V[g.C[e]], static_cast<vT>(E[e]));
        if (c > V[v]) {
          V[v] = c;
          moved = true;
        }
      }
  }
  return V;
}

template <bool N, bool R, bool U>
void run(csr const& g, std::vector<eT> const& E, std::vector<vT> const& want, unsigned src,
         kites::gpu& dev, std::string const& graph) {
  auto d = upload<vT, eT>(g, E, dev);
  std::vector<vT> V0(g.n, 0);
  V0[src] = 1 << 30;
  std::vector<char> active(g.n, 0);
  for (unsigned j = g.oR[src]; j < g.oR[src + 1]; ++j) active[g.oC[j]] = 1;
  std::string const name =
      graph + std::string(", nbr ") + (N ? "v" : "p") + " red " + (R ? "v" : "p") + " upd " + (U ? "v" : "p");
  auto one = [&](std::string const& how, kites::options o) {
    announce(name + ", " + how);
    start(*d, V0, active);
    kites::process<kites::launch::sync>(*d, dev, copy_init<(N && R), vT>{}, narrow<N, vT, eT>{},
                                        take_max<R, vT>{}, more<U, vT>{}, o);
    report(name + ", " + how, same(to_host(d->V.get_ptr(), g.n), want));
  };
  for (unsigned v = 1; v <= 8; ++v) {
    kites::options o;
    o.sched = kites::schedule::forced;
    o.forced_variant = v;
    one("forced " + std::to_string(v), o);
    o.seed = kites::options::seeding::source;
    o.seed_source = src;
    one("forced " + std::to_string(v) + " from its source", o);
  }
  for (unsigned gr = 0; gr < 4; ++gr) {
    kites::options o;
    o.sched = kites::schedule::plain;
    o.gran = static_cast<kites::granularity>(gr);
    one("plain " + std::to_string(gr), o);
  }
  kites::options o;
  o.sched = kites::schedule::classic;
  one("classic", o);
}

template <bool N, bool R, bool U>
void runs(kites::gpu& dev) {
  numbers rnd(3);
  for (bool second : {false, true}) {
    csr const g = second ? ring(3000) : random_graph(5003, 6, 8);
    std::vector<eT> E(g.m());
    for (eT& e : E) e = 1 + rnd.below(1000);
    unsigned src = 0;
    for (unsigned v = 0; v < g.n; ++v)
      if (g.oR[v + 1] - g.oR[v] > g.oR[src + 1] - g.oR[src]) src = v;
    run<N, R, U>(g, E, widest(g, E, src), src, dev, second ? "ring" : "random");
  }
}

}  // namespace

int main() {
  kites::gpu dev(0);
  runs<false, false, false>(dev);
  runs<false, false, true>(dev);
  runs<false, true, false>(dev);
  runs<false, true, true>(dev);
  runs<true, false, false>(dev);
  runs<true, false, true>(dev);
  runs<true, true, false>(dev);
  runs<true, true, true>(dev);
  return finish();
}
