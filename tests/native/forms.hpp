// forms.hpp -- functors in the reference's form (volatile references) or with
// plain references, one template argument each.
#ifndef KITES_TESTS_FORMS_HPP_
#define KITES_TESTS_FORMS_HPP_

#include <type_traits>

namespace native {

template <bool VOL, class vT>
using ref = std::conditional_t<VOL, volatile vT&, vT&>;

// initF: the value itself.
template <bool VOL, class vT>
struct copy_init {
  __host__ __device__ void operator()(ref<VOL, vT> loc, vT& old) const { loc = old; }
};

// Widest paths: max over in-edges of min(source, weight).
template <bool VOL, class vT, class eT>
struct narrow {
  __host__ __device__ void operator()(ref<VOL, vT> part, vT src, eT* e) const {
    vT const w = static_cast<vT>(*e);
    part = src < w ? src : w;
  }
};
template <bool VOL, class vT>
struct take_max {
  __host__ __device__ void operator()(ref<VOL, vT> l, ref<VOL, vT> r) const {
    if (l < r) l = r;
  }
};
template <bool VOL, class vT>
struct more {
  __host__ __device__ bool operator()(ref<VOL, vT> nv, vT old) const { return nv > old; }
};

}  // namespace native

#endif  // KITES_TESTS_FORMS_HPP_
