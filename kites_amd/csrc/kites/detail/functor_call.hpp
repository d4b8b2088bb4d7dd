// functor_call.hpp -- how the kernels call the four functors.
//
// The reference's signatures take volatile references (README.md:16-23).  A
// volatile access through a reference stays a flat access with system scope
// (flat_load / flat_store sc0 sc1) even when it points into LDS, and the wave
// then waits for every load it has in flight.  Functors that take plain
// references instead ("vT&" where the reference has "volatile vT&"; the
// library's own sets do) work on registers.  Which form a functor has is seen
// from its signature: a plain reference does not bind to a volatile lvalue.
//
// The *_at forms work on LDS slots in place; edge_value returns the partial.
// (The host's probe of a functor set calls them on locals.)
#ifndef KITES_DETAIL_FUNCTOR_CALL_HPP_
#define KITES_DETAIL_FUNCTOR_CALL_HPP_

#include <hip/hip_runtime.h>

#include <type_traits>

namespace kites {
namespace detail {

template <class T>
__host__ __device__ __forceinline__ volatile T& as_volatile(T& x) {
  return *reinterpret_cast<volatile T*>(&x);
}

// nbrCompF takes the edge as a pointer to const: it can only read it, so a
// kernel may call it for an edge whose partial is then dropped.  (One that takes
// the reference's eT* may write through it: each call then stands for one walk
// of that edge.)  Either way the pointer is the edge's place in the graph's array.
// Read off the type of its call operator; generic and overloaded functors count
// as ones that may write.
template <class R, class C, class A, class B, class E>
E edge_param(R (C::*)(A, B, E));
template <class R, class C, class A, class B, class E>
E edge_param(R (C::*)(A, B, E) const);
template <class R, class C, class A, class B, class E>
E edge_param(R (C::*)(A, B, E) noexcept);
template <class R, class C, class A, class B, class E>
E edge_param(R (C::*)(A, B, E) const noexcept);

template <class FN, class eT, class = void>
struct edge_reader : std::false_type {};
template <class FN, class eT>
struct edge_reader<FN, eT, std::void_t<decltype(edge_param(&FN::operator()))>>
    : std::is_same<decltype(edge_param(&FN::operator())), const eT*> {};

template <class FN, class vT, class eT>
constexpr bool reads_edge = edge_reader<FN, eT>::value;

// nbrCompF works on its lane's LDS slot (volatile references).
template <class FN, class vT, class eT>
constexpr bool takes_slot = std::is_invocable<FN&, volatile vT&, vT, eT*>::value;

// nbrCompF(partial, srcV, edge); `slot`: an LDS slot of the calling lane.
template <class FN, class vT, class eT>
__host__ __device__ __forceinline__ vT edge_value(FN& fn, vT& slot, vT src, eT* edge) {
  if constexpr (std::is_invocable<FN&, volatile vT&, vT, eT*>::value) {
    fn(as_volatile(slot), src, edge);
    return slot;
  } else {
    vT r{};
    fn(r, src, edge);
    return r;
  }
}

template <class FN, class vT, class eT>
__host__ __device__ __forceinline__ void edge_value_at(FN& fn, vT& slot, vT src, eT* edge) {
  if constexpr (std::is_invocable<FN&, volatile vT&, vT, eT*>::value) {
    fn(as_volatile(slot), src, edge);
  } else {
    vT r{};
    fn(r, src, edge);
    slot = r;
  }
}

// initF(local, global)
template <class FI, class vT>
__host__ __device__ __forceinline__ void init_at(FI& fi, vT& slot, vT global) {
  vT g = global;
  if constexpr (std::is_invocable<FI&, volatile vT&, vT&>::value) {
    fi(as_volatile(slot), g);
  } else {
    vT r{};
    fi(r, g);
    slot = r;
  }
}

// redF(lhs, rhs)
template <class FR, class vT>
__host__ __device__ __forceinline__ void reduce_at(FR& fr, vT& lhs, vT& rhs) {
  if constexpr (std::is_invocable<FR&, volatile vT&, volatile vT&>::value) {
    fr(as_volatile(lhs), as_volatile(rhs));
  } else {
    vT l = lhs, r = rhs;
    fr(l, r);
    lhs = l;
  }
}

// updF(newV, oldV)
template <class FU, class vT>
__host__ __device__ __forceinline__ bool update_at(FU& fu, vT& slot, vT old) {
  if constexpr (std::is_invocable<FU&, volatile vT&, vT>::value) {
    return fu(as_volatile(slot), old);
  } else {
    vT nv = slot;
    bool const u = fu(nv, old);
    slot = nv;
    return u;
  }
}

// nv = redF(old, cand); returns updF(nv, old).  `work` and `slot`: LDS slots of
// the lane (edge_value leaves `cand` in no slot when nbrCompF takes plain
// references, so a volatile redF gets it put there).
template <class FR, class FU, class vT>
__host__ __device__ __forceinline__ bool combine(FR& fr, FU& fu, vT old, vT cand, vT& work, vT& slot,
                                        vT& nv) {
  if constexpr (std::is_invocable<FR&, volatile vT&, volatile vT&>::value) {
    as_volatile(work) = old;
    as_volatile(slot) = cand;
    fr(as_volatile(work), as_volatile(slot));
    bool const u = update_at(fu, work, old);
    nv = as_volatile(work);
    return u;
  } else {
    vT l = old, r = cand;
    fr(l, r);
    if constexpr (std::is_invocable<FU&, volatile vT&, vT>::value) {
      as_volatile(work) = l;
      bool const u = fu(as_volatile(work), old);
      nv = as_volatile(work);
      return u;
    } else {
      bool const u = fu(l, old);
      nv = l;
      return u;
    }
  }
}

}  // namespace detail
}  // namespace kites

#endif  // KITES_DETAIL_FUNCTOR_CALL_HPP_
