// host_copy.hpp -- results from device memory into the caller's (pageable)
// arrays.
//
// hipMemcpy into fresh pageable memory reaches about 4-17 GB/s (it stages or
// pins inside the runtime, and one thread takes all page faults), and
// hipMemcpy2D of n short rows goes row by row (65,536 rows of 57 values: 0.43
// s).  Here copy_out_kernel writes the wanted columns contiguously into pinned
// memory, 16 KB blocks in order, and raises each block's flag; the caller and
// up to kCopyThreads - 1 helpers move finished chunks on while the kernel goes
// on, so PCIe (57 GB/s), the page faults and the copies overlap.  Results of up
// to kCopySmall bytes take one hipMemcpyAsync and one copy (12 us for 28 KB).
//
// The pinned buffers (2 MB, or 16 MB for results above kCopyMiddle bytes) are
// kept between calls: at most kKeepRings of each size in the process, all but
// one small one given back when the last graph handle is destroyed (a program
// that builds, solves and drops one graph after the other would pay 1.5 ms for
// a large one each time).  A buffer serves one call at a time (concurrent calls
// take or make their own).
#ifndef KITES_AMD_HOST_COPY_HPP_
#define KITES_AMD_HOST_COPY_HPP_

#include <hip/hip_runtime.h>
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <fstream>
#include <istream>
#include <limits>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include "kites/common.hpp"

namespace kites_capi {

constexpr unsigned kCopyThreads = 8;
constexpr std::size_t kCopyBlock = std::size_t(1) << 14;    // bytes per flag
constexpr std::size_t kCopyChunk = std::size_t(1) << 18;    // bytes a thread moves at a time
constexpr std::size_t kCopyHalves[2] = {std::size_t(1) << 20, std::size_t(1) << 23};  // bytes of
                                                            // one launch, small and large ring
constexpr std::size_t kCopySmall = kCopyHalves[0];          // one hipMemcpyAsync up to here
constexpr std::size_t kCopyMiddle = std::size_t(1) << 22;   // the small ring up to here
// Workgroups of a launch: 64 blocks in flight keep PCIe busy, and blocks still
// finish in order a megabyte at a time.
constexpr unsigned kCopyGrid = 32;
constexpr std::size_t kKeepRings = 2;

// One call's pinned memory: two halves of data and a flag per block (the number
// of the launch that last filled the block).
struct copy_ring {
  int device = -1;
  std::size_t bytes;           // of a half
  unsigned char* mem = nullptr;
  unsigned launches = 0;       // numbers the launches of all calls it served
  copy_ring(int d, std::size_t half_bytes) : device(d), bytes(half_bytes) {
    std::size_t const marks = 2 * (bytes / kCopyBlock) * sizeof(unsigned);
    KITES_HIP_CHECK(hipHostMalloc(reinterpret_cast<void**>(&mem), 2 * bytes + marks,
                                  hipHostMallocPortable | hipHostMallocCoherent));
    std::memset(mem + 2 * bytes, 0, marks);
  }
  copy_ring(copy_ring const&) = delete;
  copy_ring& operator=(copy_ring const&) = delete;
  ~copy_ring() {
    if (mem) (void)hipHostFree(mem);
  }
  unsigned char* half(std::size_t launch) const { return mem + (launch & 1) * bytes; }
  unsigned* flags(std::size_t launch) const {
    return reinterpret_cast<unsigned*>(mem + 2 * bytes) + (launch & 1) * (bytes / kCopyBlock);
  }
};

struct copy_pool {
  std::mutex mu;
  std::vector<std::unique_ptr<copy_ring>> idle;
  std::size_t handles = 0;
  // (never destroyed: the HIP runtime may be gone when statics are)
  static copy_pool& get() {
    static copy_pool* const p = new copy_pool();
    return *p;
  }
  std::unique_ptr<copy_ring> take(int device, std::size_t half) {
    {
      std::lock_guard<std::mutex> l(mu);
      for (std::size_t i = 0; i < idle.size(); ++i)
        if (idle[i]->device == device && idle[i]->bytes == half) {
          std::unique_ptr<copy_ring> got = std::move(idle[i]);
          idle.erase(idle.begin() + static_cast<std::ptrdiff_t>(i));
          return got;
        }
    }
    return std::unique_ptr<copy_ring>(new copy_ring(device, half));
  }
  void give(std::unique_ptr<copy_ring> r) {
    std::lock_guard<std::mutex> l(mu);
    std::size_t same = 0;
    for (auto const& x : idle) same += x->bytes == r->bytes;
    if (same < kKeepRings) idle.push_back(std::move(r));
  }
};

// Held by every graph handle: with the last one the pinned memory goes back.
struct copy_user {
  copy_user() {
    auto& p = copy_pool::get();
    std::lock_guard<std::mutex> l(p.mu);
    ++p.handles;
  }
  copy_user(copy_user const&) = delete;
  copy_user& operator=(copy_user const&) = delete;
  ~copy_user() {
    auto& p = copy_pool::get();
    std::vector<std::unique_ptr<copy_ring>> gone;
    std::lock_guard<std::mutex> l(p.mu);
    if (--p.handles) return;
    gone.swap(p.idle);
    for (auto& r : gone)
      if (p.idle.empty() && r->bytes == kCopyHalves[0]) p.idle.push_back(std::move(r));
  }
};

// Values [first, first + count) of the n x K result (row-major, the first K of
// the 32-bit columns of rows `stride` values apart) into out, four per thread
// and store, in blocks of kCopyBlock bytes: a block's flag takes `number` after
// its values have reached the host (first is a multiple of 4, out and flags are
// pinned).
static __global__ __launch_bounds__(256) void copy_out_kernel(const unsigned* __restrict__ rows,
                                                              unsigned stride, unsigned K,
                                                              unsigned long long first,
                                                              unsigned count, unsigned* out,
                                                              unsigned* flags, unsigned number) {
  constexpr unsigned kValues = static_cast<unsigned>(kCopyBlock / sizeof(unsigned));
  unsigned const blocks = (count + kValues - 1) / kValues;
  for (unsigned b = blockIdx.x; b < blocks; b += gridDim.x) {
    unsigned const end = (b + 1) * kValues < count ? (b + 1) * kValues : count;
    for (unsigned i = b * kValues + 4u * threadIdx.x; i < end; i += 4u * 256u) {
      unsigned long long const at = first + i;
      unsigned const left = end - i;
      if (K == stride && left >= 4) {
        *reinterpret_cast<uint4*>(out + i) = *reinterpret_cast<uint4 const*>(rows + at);
        continue;
      }
      unsigned long long v = at / K;
      unsigned k = static_cast<unsigned>(at - v * K);
      unsigned x[4];
#pragma unroll
      for (unsigned q = 0; q < 4; ++q) {
        x[q] = q < left ? rows[v * stride + k] : 0u;
        if (++k == K) {
          k = 0;
          ++v;
        }
      }
      if (left >= 4) {
        *reinterpret_cast<uint4*>(out + i) = make_uint4(x[0], x[1], x[2], x[3]);
      } else {
        for (unsigned q = 0; q < left; ++q) out[i + q] = x[q];
      }
    }
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0)
      __hip_atomic_store(flags + b, number, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// Whole CPUs of a control group's CPU time (quota microseconds per period): at
// least one, all when there is no limit ("max", or a negative quota).
inline std::size_t quota_cpus(std::istream& quota, std::istream& period) {
  long long q = 0, p = 0;
  if (!(quota >> q) || !(period >> p) || q <= 0 || p <= 0)
    return std::numeric_limits<std::size_t>::max();
  return static_cast<std::size_t>(std::max(1ll, q / p));
}

// The limit of the container the process runs in (read once: 40 us).
inline std::size_t container_cpus() {
  static std::size_t const cpus = [] {
    std::ifstream both("/sys/fs/cgroup/cpu.max");
    if (both) return quota_cpus(both, both);
    std::ifstream q("/sys/fs/cgroup/cpu/cpu.cfs_quota_us"), p("/sys/fs/cgroup/cpu/cpu.cfs_period_us");
    return quota_cpus(q, p);
  }();
  return cpus;
}

// Threads for a copy: one per megabyte (a helper takes about 20 us to start), as
// many as the process may run at once.
inline unsigned copy_threads(std::size_t bytes) {
  cpu_set_t set;
  std::size_t cpus = 1;
  if (sched_getaffinity(0, sizeof(set), &set) == 0)
    cpus = static_cast<std::size_t>(std::max(1, CPU_COUNT(&set)));
  return static_cast<unsigned>(std::max<std::size_t>(
      1, std::min<std::size_t>({kCopyThreads, cpus, container_cpus(), bytes >> 20})));
}

// n x K values (row-major) from device rows `stride` values apart (16-byte
// aligned); returns when all of dst is written.
inline void copy_columns(unsigned* dst, const unsigned* rows, std::size_t n, unsigned stride,
                         unsigned K, int device, hipStream_t s) {
  std::size_t const bytes = n * K * sizeof(unsigned);
  if (!bytes) return;
  auto& pool = copy_pool::get();
  KITES_HIP_CHECK(hipSetDevice(device));
  std::size_t const half = kCopyHalves[bytes > kCopyMiddle];
  std::unique_ptr<copy_ring> ring = pool.take(device, half);
  if (bytes <= kCopySmall && K == stride) {
    hipError_t const e = hipMemcpyAsync(ring->half(0), rows, bytes, hipMemcpyDeviceToHost, s);
    KITES_HIP_CHECK(hipStreamSynchronize(s));
    KITES_HIP_CHECK(e);
    std::memcpy(dst, ring->half(0), bytes);
    pool.give(std::move(ring));
    return;
  }
  std::size_t const launches = (bytes + half - 1) / half;
  std::size_t const chunks = (bytes + kCopyChunk - 1) / kCopyChunk;
  std::size_t const per_half = half / kCopyChunk;
  unsigned const base = ring->launches + 1;      // launch l is number base + l
  if (base + launches < base || base + launches > 0xfffffff0ull) {
    // (the numbers ran out: start over with cleared flags)
    ring.reset(new copy_ring(device, half));
  }
  unsigned const number = ring->launches + 1;
  ring->launches += static_cast<unsigned>(launches);
  std::atomic<std::size_t> next{0}, issued{0};
  std::atomic<int> error{0};
  std::vector<std::atomic<unsigned>> moved(launches);   // chunks of each launch moved on
  for (auto& m : moved) m.store(0);
  auto chunks_of = [&](std::size_t l) { return std::min(per_half, chunks - l * per_half); };
  std::mutex issue_mu;
  // Queues, in order, every launch whose half is free: launch l reuses the
  // half of l - 2, so all chunks of that one have to have been moved on (the
  // launches finish moving in any order).
  auto issue = [&]() {
    std::lock_guard<std::mutex> lock(issue_mu);
    for (std::size_t l = issued.load();
         l < launches && (l < 2 || moved[l - 2].load() == chunks_of(l - 2)); ++l) {
      std::size_t const at = l * half, count = std::min(half, bytes - at);
      unsigned long long first = at / sizeof(unsigned);
      unsigned values = static_cast<unsigned>(count / sizeof(unsigned));
      unsigned* to = reinterpret_cast<unsigned*>(ring->half(l));
      unsigned* flags = ring->flags(l);
      unsigned mark = number + static_cast<unsigned>(l), step = stride, columns = K;
      const unsigned* from = rows;
      void* args[] = {&from, &step, &columns, &first, &values, &to, &flags, &mark};
      // (this launch's own status: the thread's last error may be an earlier
      // call's, which was reported there)
      hipError_t const e = hipLaunchKernel(reinterpret_cast<const void*>(&copy_out_kernel),
                                           dim3(kCopyGrid), dim3(256), args, 0, s);
      if (e != hipSuccess) error.store(static_cast<int>(e));
      issued.store(l + 1);
    }
  };
  auto work = [&](bool helper) {
    if (helper && hipSetDevice(device) != hipSuccess) return;   // (the others take its share)
    for (;;) {
      std::size_t const c = next.fetch_add(1);
      if (c >= chunks) return;
      std::size_t const l = c / per_half, at = c * kCopyChunk, in = at - l * half;
      std::size_t const count = std::min(kCopyChunk, bytes - at);
      unsigned const* const flag = ring->flags(l) + in / kCopyBlock;
      for (std::size_t b = 0; b * kCopyBlock < count; ++b) {
        unsigned spins = 0;
        auto since = std::chrono::steady_clock::now();
        while (__atomic_load_n(flag + b, __ATOMIC_ACQUIRE) != number + l) {
          if (error.load()) return;
          kites::detail::wait_turn(spins);
          // A stream that has failed, or has been idle for seconds, raises no
          // more flags.  (Asked rarely: hipStreamQuery beside a launch by
          // another thread can report an idle stream.)
          if (++spins % 65536 == 0 &&
              std::chrono::steady_clock::now() - since > std::chrono::seconds(5)) {
            hipError_t const e = hipStreamQuery(s);
            if (e != hipErrorNotReady &&
                __atomic_load_n(flag + b, __ATOMIC_ACQUIRE) != number + l) {
              error.store(static_cast<int>(e == hipSuccess ? hipErrorUnknown : e));
              return;
            }
            since = std::chrono::steady_clock::now();
          }
        }
      }
      std::memcpy(reinterpret_cast<unsigned char*>(dst) + at, ring->half(l) + in, count);
      if (moved[l].fetch_add(1) + 1 == chunks_of(l)) issue();
    }
  };
  issue();
  std::vector<std::thread> helpers;
  unsigned const threads = copy_threads(bytes);
  try {
    helpers.reserve(threads);
    for (unsigned t = 1; t < threads; ++t) helpers.emplace_back(work, true);
  } catch (std::exception const&) {
    // (fewer helpers, or none)
  }
  work(false);
  for (auto& h : helpers) h.join();
  // nothing of this call may still write into the pinned memory
  hipError_t const last = hipStreamSynchronize(s);
  KITES_HIP_CHECK(static_cast<hipError_t>(error.load()));
  KITES_HIP_CHECK(last);
  pool.give(std::move(ring));
}

}  // namespace kites_capi

#endif  // KITES_AMD_HOST_COPY_HPP_
