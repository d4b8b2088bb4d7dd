// host_forms.hip -- checks of the engine's headers that need no GPU.
#include "forms.hpp"
#include "native.hpp"

#include <sstream>

#include "host_copy.hpp"

using namespace native;

namespace {

// The LDS words of an ordered task (detail/ordered_kernel.hpp): rows go in
// batches, a batch's segment heads are read, then its partials are written.  No
// partial may lie on a head that a later batch reads.
template <unsigned BYTES>
struct value {
  unsigned char b[BYTES];
};

template <unsigned BYTES>
void ordered_layout() {
  using S = kites::detail::ordered_shape<value<BYTES>>;
  std::vector<char> written(S::slots * std::max(BYTES, 4u), 0);
  unsigned bad = 0;
  for (unsigned r0 = 0; r0 < S::rows; r0 += S::batch) {
    for (unsigned p = r0 * 64; p < (r0 + S::batch) * 64; ++p)
      for (unsigned k = 0; k < 4 && !S::heads_apart; ++k) bad += written[p * 4 + k];
    for (unsigned p = r0 * 64; p < (r0 + S::batch) * 64; ++p)
      for (unsigned k = 0; k < BYTES; ++k) written[p * BYTES + k] = 1;
  }
  report("ordered segment heads of " + std::to_string(BYTES) + "-byte values", bad == 0);
}

// The four functors of a max-min set, each in either form, through the helpers
// the kernels call them with.  The slots hold what an earlier edge left.
template <bool I, bool N, bool R, bool U>
void functor_mix() {
  using namespace kites::detail;
  using vT = int;
  copy_init<I, vT> fi;
  narrow<N, vT, unsigned> fn;
  take_max<R, vT> fr;
  more<U, vT> fu;
  bool ok = true;
  for (vT old : {0, 3, 7, 9})
    for (vT src : {0, 2, 7, 100})
      for (unsigned w : {1u, 7u, 50u})
        for (vT left : {-1, 0, 8, 1000}) {
          vT const cand = src < static_cast<vT>(w) ? src : static_cast<vT>(w);
          vT const want = old < cand ? cand : old;
          unsigned e = w;
          vT slot = left, work = left, nv = left;
          ok = ok && edge_value(fn, slot, src, &e) == cand;
          // a push: the partial as returned, the slots as edge_value left them
          slot = N ? cand : left;
          bool const moved = combine(fr, fu, old, cand, work, slot, nv);
          ok = ok && moved == (want > old) && (!moved || nv == want);
          // a pull: slots in place
          vT acc = left, part = left;
          init_at(fi, acc, old);
          edge_value_at(fn, part, src, &e);
          reduce_at(fr, acc, part);
          ok = ok && part == cand && acc == want && update_at(fu, acc, old) == (want > old);
        }
  std::string const names = std::string("functor forms ") + (I ? "v" : "p") + (N ? "v" : "p") +
                            (R ? "v" : "p") + (U ? "v" : "p");
  report(names, ok);
}

template <bool I, bool N, bool R>
void functor_mixes() {
  functor_mix<I, N, R, false>();
  functor_mix<I, N, R, true>();
}

// CPUs of a container's limit, and a copy's threads within it.
void cpu_limits() {
  using namespace kites_capi;
  std::size_t const none = std::numeric_limits<std::size_t>::max();
  auto two = [](const char* text) {
    std::istringstream in(text);
    return quota_cpus(in, in);
  };
  auto split = [](const char* quota, const char* period) {
    std::istringstream q(quota), p(period);
    return quota_cpus(q, p);
  };
  report("container limits", two("1600000 100000\n") == 16 && two("150000 100000") == 1 &&
                                 two("20000 100000") == 1 && two("max 100000") == none &&
                                 two("") == none && two("100000") == none &&
                                 split("400000\n", "100000\n") == 4 &&
                                 split("-1\n", "100000\n") == none && split("", "") == none);
  std::size_t const most = std::min<std::size_t>(container_cpus(), kCopyThreads);
  report("copy threads", copy_threads(0) == 1 && copy_threads(std::size_t(1) << 20) == 1 &&
                             copy_threads(std::size_t(1) << 30) <= most);
}

// Whether a functor may write its edge is read off its signature; a generic one's
// body is not looked at with a pointer to const (it need not compile with one).
struct overloaded {
  __host__ __device__ void operator()(int& part, int src, int* e) const { part = src + *e; }
  __host__ __device__ void operator()(int& part, int src, float* e) const { part = src + (*e > 0); }
};

void edge_writers() {
  using kites::detail::edge_value_at;
  using kites::detail::reads_edge;
  auto generic = [] __host__ __device__(auto& part, auto src, auto* e) {
    *e += 1;
    part = src + *e;
  };
  auto reader = [] __host__ __device__(int& part, int src, const int* e) { part = src + *e; };
  auto writer = [] __host__ __device__(int& part, int src, int* e) { part = src + *e; };
  auto counter = [n = 0] __host__ __device__(volatile int& part, int src, int const* e) mutable noexcept {
    part = src + *e + n;
  };
  int slot = 0, edge = 4;
  edge_value_at(generic, slot, 1, &edge);
  report("functors that may write the edge",
         slot == 6 && edge == 5 && !reads_edge<decltype(generic), int, int> &&
             reads_edge<decltype(reader), int, int> && !reads_edge<decltype(writer), int, int> &&
             reads_edge<decltype(counter), int, int> && !reads_edge<overloaded, int, int>);
}

}  // namespace

int main() {
  edge_writers();
  cpu_limits();
  functor_mixes<false, false, false>();
  functor_mixes<false, false, true>();
  functor_mixes<false, true, false>();
  functor_mixes<false, true, true>();
  functor_mixes<true, false, false>();
  functor_mixes<true, false, true>();
  functor_mixes<true, true, false>();
  functor_mixes<true, true, true>();
  ordered_layout<1>();
  ordered_layout<2>();
  ordered_layout<4>();
  ordered_layout<8>();
  ordered_layout<12>();
  ordered_layout<16>();
  ordered_layout<20>();
  ordered_layout<32>();
  return finish();
}
