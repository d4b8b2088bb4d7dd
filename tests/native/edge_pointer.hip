// edge_pointer.hip -- nbrCompF's edge pointer is the edge's place in the graph's
// array in every kernel: functors that look their weight up in a table of their
// own by that place, and ones that count their calls in the edge.
#include "forms.hpp"
#include "native.hpp"

using namespace native;

namespace {

using vT = unsigned;
constexpr vT kInf = 0xFFFFFFFFu;

// A grid of rows x cols, edges to the four neighbours: many iterations of small
// frontiers (the one-workgroup loop's case).
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

std::vector<vT> distances(csr const& g, std::vector<vT> const& w, unsigned src) {
  std::vector<vT> V(g.n, kInf);
  V[src] = 0;
  for (bool moved = true; moved;) {
    moved = false;
    auto pass = [&](unsigned v) {
      for (unsigned e = g.R[v]; e < g.R[v + 1]; ++e) {
        vT const s = V[g.C[e]];
        if (s != kInf && s + w[e] < V[v]) {
          V[v] = s + w[e];
          moved = true;
        }
      }
    };
    for (unsigned v = 0; v < g.n; ++v) pass(v);
    for (unsigned v = g.n; v-- > 0;) pass(v);
  }
  return V;
}

template <bool VOL>
struct take_min {
  __host__ __device__ void operator()(ref<VOL, vT> l, ref<VOL, vT> r) const {
    if (l > r) l = r;
  }
};
template <bool VOL>
struct less {
  __host__ __device__ bool operator()(ref<VOL, vT> nv, vT old) const { return nv < old; }
};

// The edge value is not used: the weight lies in `table` at the edge's place.
// EDGE is the edge type or its const form.
template <bool VOL, class EDGE>
struct by_place {
  const unsigned* oE;
  const vT* table;
  __host__ __device__ void operator()(ref<VOL, vT> part, vT src, EDGE* e) const {
    part = src == kInf ? kInf : src + table[e - oE];
  }
};

// Counts its calls in the edge: weight in the low half.
struct counted {
  unsigned short w, calls;
};
template <bool VOL>
struct counting {
  __host__ __device__ void operator()(ref<VOL, vT> part, vT src, counted* e) const {
    e->calls = static_cast<unsigned short>(e->calls + 1);
    part = src == kInf ? kInf : src + e->w;
  }
};

template <bool VOL, class EDGE>
void places(csr const& g, std::vector<vT> const& w, std::vector<vT> const& want, kites::gpu& dev,
            std::string const& form) {
  std::vector<unsigned> zero(g.m(), 0u);
  auto d = upload<vT, unsigned>(g, zero, dev);
  std::vector<vT> ow(g.m());
  for (unsigned j = 0; j < g.m(); ++j) ow[j] = w[g.slot[j]];
  kites::device_buffer<vT> table(g.m(), 0);
  to_device(table.get_ptr(), ow);
  for (unsigned delta : {0u, 150u}) {
    std::string const what = "edge places, " + form + (delta ? ", near-far" : "");
    announce(what);
    std::vector<vT> V0(g.n, kInf);
    V0[0] = 0;
    start(*d, V0, std::vector<char>(g.n, 0));
    kites::run_report rep;
    kites::options o;
    o.sched = kites::schedule::plain;
    o.alpha = 0.f;               // push only: out-edge places
    o.delta = delta;
    o.seed = kites::options::seeding::source;
    o.seed_source = 0;
    o.keep_stats = true;
    o.report = &rep;
    kites::process<kites::launch::sync>(
        *d, dev, copy_init<VOL, vT>{},
        by_place<VOL, EDGE>{reinterpret_cast<const unsigned*>(d->oE.get_ptr()), table.get_ptr()},
        take_min<VOL>{}, less<VOL>{}, o);
    unsigned loop = 0;
    for (auto const& s : rep.stats) loop += s.variant == kites::detail::V_PERSIST;
    report(what, loop > 100 && same(to_host(d->V.get_ptr(), g.n), want));
  }
}

// Every call of a push run leaves its mark: an edge is expanded once for each
// time its source was in a queue, so the calls add up to the edges walked.
template <bool VOL>
void calls(csr const& g, std::vector<vT> const& w, std::vector<vT> const& want, kites::gpu& dev,
           std::string const& form) {
  std::vector<counted> E(g.m());
  for (unsigned e = 0; e < g.m(); ++e) E[e] = counted{static_cast<unsigned short>(w[e]), 0};
  auto d = upload<vT, counted>(g, E, dev);
  std::string const what = "calls counted in the edges, " + form;
  announce(what);
  std::vector<vT> V0(g.n, kInf);
  V0[0] = 0;
  start(*d, V0, std::vector<char>(g.n, 0));
  kites::run_report rep;
  kites::options o;
  o.sched = kites::schedule::plain;
  o.alpha = 0.f;
  o.seed = kites::options::seeding::source;
  o.seed_source = 0;
  o.keep_stats = true;
  o.report = &rep;
  kites::process<kites::launch::sync>(*d, dev, copy_init<VOL, vT>{}, counting<VOL>{},
                                      take_min<VOL>{}, less<VOL>{}, o);
  unsigned long long walked = 0, counts = 0;
  unsigned loop = 0;
  for (auto const& s : rep.stats) {
    walked += s.work_edges;
    loop += s.variant == kites::detail::V_PERSIST;
  }
  for (counted const& c : to_host(d->oE.get_ptr(), g.m())) counts += c.calls;
  report(what, loop > 100 && counts == walked && same(to_host(d->V.get_ptr(), g.n), want));
}

}  // namespace

int main() {
  kites::gpu dev(0);
  csr const g = grid(300, 70);
  std::vector<vT> w(g.m());
  numbers rnd(6);
  for (vT& x : w) x = 1 + rnd.below(40);
  std::vector<vT> const want = distances(g, w, 0);
  places<false, unsigned>(g, w, want, dev, "plain");
  places<true, unsigned>(g, w, want, dev, "volatile");
  places<false, const unsigned>(g, w, want, dev, "plain, const edge");
  places<true, const unsigned>(g, w, want, dev, "volatile, const edge");
  calls<false>(g, w, want, dev, "plain");
  calls<true>(g, w, want, dev, "volatile");
  return finish();
}
