// host_forms.hip -- checks of the engine's headers that need no GPU.
#include "native.hpp"

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

}  // namespace

int main() {
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
