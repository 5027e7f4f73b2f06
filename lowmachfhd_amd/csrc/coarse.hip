// coarse.hip -- the one-workgroup coarse V-cycle kernels (coarse.h), a translation unit of its
// own, so that they compile beside the rest of the library.
#include <hip/hip_runtime.h>

#include <type_traits>
#include <vector>

#include "coarse.h"

namespace lmfhd {

#ifndef LMFHD_HOST_DEBUG
// the phases of a body on the device: each thread runs f on its own state, then a barrier
template <class State>
struct DevX {
  State st;
  __device__ __forceinline__ int threads() const { return (int)blockDim.x; }
  __device__ __forceinline__ int uniform(int v) const { return __builtin_amdgcn_readfirstlane(v); }
  // no instruction moves across: with several slots a thread it keeps one's temporaries from
  // living beside the next one's
  __device__ __forceinline__ void fence() const { __builtin_amdgcn_sched_barrier(0); }
  template <class S, class F>
  __device__ __forceinline__ void each(const F& f) {
    f((int)threadIdx.x, st);
    __syncthreads();
  }
  // x[0, n) minus its mean (workgroup reduction in FP64, a fixed order)
  template <typename T>
  __device__ __forceinline__ void mean(T* x, long n) const {
    __shared__ double sh[COARSE_THREADS / 64];
    double s = 0.0;
    for (long e = threadIdx.x; e < n; e += blockDim.x) s += (double)x[e];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    double tot = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) tot += sh[w];
    const double m = tot / (double)n;
    for (long e = threadIdx.x; e < n; e += blockDim.x) x[e] = T((double)x[e] - m);
    __syncthreads();
  }
};

// n elements from src to dst by the workgroup, 16 bytes a thread (blocks of 64 elements, both
// ends 16-byte aligned)
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
template <typename T>
__device__ __forceinline__ void blk_copy(T* dst, const T* src, int n) {
  const int n16 = n * (int)sizeof(T) / 16;
  for (int e = threadIdx.x; e < n16; e += blockDim.x) ((u32x4*)dst)[e] = ((const u32x4*)src)[e];
}
template <int STAGED, typename T, class Body>
__device__ __forceinline__ void run_on_work(T* work, int phi, int span, const Body& body) {
  if constexpr (STAGED) {
    __shared__ __align__(16) unsigned char buf[COARSE_LDS];
    T* W = (T*)buf;
    blk_copy(W + phi, work + phi, 2 * span);  // phi and rhs
    __syncthreads();
    body(W);
    blk_copy(work + phi, W + phi, span);  // body ends on a barrier
  } else {
    body(work);
  }
}
// the argument block behind a device address: an integer in the functor, so that the compiler
// keeps the constant address space instead of finding the plain pointer behind the cast
template <class Args>
__device__ __forceinline__ const LMFHD_CONST Args* const_args(unsigned long long a) {
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)a);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(a >> 32));
  return (const LMFHD_CONST Args*)(((unsigned long long)hi << 32) | lo);
}
#else
// the same phases on the CPU: every thread's state kept, f run for each in turn
template <class State>
struct HostX {
  int nt;
  std::vector<State> st;
  explicit HostX(int n) : nt(n), st(n) {}
  int threads() const { return nt; }
  int uniform(int v) const { return v; }
  void fence() const {}
  template <class S, class F>
  void each(const F& f) {
    for (int t = 0; t < nt; ++t) f(t, st[t]);
  }
  template <typename T>
  void mean(T* x, long n) const {
    double acc = 0.0;
    for (long e = 0; e < n; ++e) acc += (double)x[e];
    const double m = acc / (double)n;
    for (long e = 0; e < n; ++e) x[e] = T((double)x[e] - m);
  }
};
template <int STAGED, typename T, class Body>
void run_on_work_host(T* work, int phi, int span, const Body& body) {
  if (!STAGED) {
    body(work);
    return;
  }
  std::vector<T> W(COARSE_LDS / sizeof(T), T(7));  // nothing but phi and rhs is read before it is written
  memcpy(W.data() + phi, work + phi, 2 * (size_t)span * sizeof(T));
  body(W.data());
  memcpy(work + phi, W.data() + phi, (size_t)span * sizeof(T));
}
#endif

template <typename T, int VT, int DM, int STAGED, int KM, int SMALL>
struct StagCoarseBlk {
  static constexpr int BS = COARSE_THREADS;
  unsigned long long A;  // the device address of a StagCoarseArgs<T>
  int nt;
#ifdef LMFHD_HOST_DEBUG
  void block_host(int) const {
    const StagCoarseArgs<T>& a = *(const StagCoarseArgs<T>*)A;
    HostX<StagState<T, VT, DM, KM>> x(nt);
    run_on_work_host<STAGED>(a.work, a.L[a.l0].phi, a.L[a.l0].span, [&](T* W) { stag_coarse_body<T, VT, DM, KM, SMALL>(a, W, x); });
  }
#else
  __device__ __forceinline__ void block(int) const {
    auto& a = *const_args<StagCoarseArgs<T>>(A);
    DevX<StagState<T, VT, DM, KM>> x;
    run_on_work<STAGED>(a.work, a.L[a.l0].phi, a.L[a.l0].span,
                        [&](T* W) __attribute__((always_inline)) { stag_coarse_body<T, VT, DM, KM, SMALL>(a, W, x); });
  }
#endif
};
template <typename T, int DM, int STAGED, int KM, int SMALL>
struct MacCoarseBlk {
  static constexpr int BS = COARSE_THREADS;
  unsigned long long A;
  int nt;
#ifdef LMFHD_HOST_DEBUG
  void block_host(int) const {
    const MacCoarseArgs<T>& a = *(const MacCoarseArgs<T>*)A;
    HostX<MacState<T, DM, KM>> x(nt);
    run_on_work_host<STAGED>(a.work, a.L[a.l0].phi, a.L[a.l0].span, [&](T* W) { mac_coarse_body<T, DM, KM, SMALL>(a, W, x); });
  }
#else
  __device__ __forceinline__ void block(int) const {
    auto& a = *const_args<MacCoarseArgs<T>>(A);
    DevX<MacState<T, DM, KM>> x;
    run_on_work<STAGED>(a.work, a.L[a.l0].phi, a.L[a.l0].span,
                        [&](T* W) __attribute__((always_inline)) { mac_coarse_body<T, DM, KM, SMALL>(a, W, x); });
  }
#endif
};

template <typename T>
void launch_stag_coarse(hipStream_t s, int vt, int dm, int nt, CoarseForm form, const StagCoarseArgs<T>* Ap) {
  const unsigned long long A = (unsigned long long)Ap;
  dispatch_vd(vt, dm, [&](auto V, auto D) {
    constexpr int VT = decltype(V)::value, DM = decltype(D)::value, KM = stag_slots_max<T>(VT);
    if (form == CoarseForm::lds_small) launch_blocks(s, 1, StagCoarseBlk<T, VT, DM, 1, SLOTS_SMALL, 1>{A, nt}, nt);
    else if (form == CoarseForm::lds) launch_blocks(s, 1, StagCoarseBlk<T, VT, DM, 1, KM, 0>{A, nt}, nt);
    else launch_blocks(s, 1, StagCoarseBlk<T, VT, DM, 0, KM, 0>{A, nt}, nt);
  });
}
template <typename T>
void launch_mac_coarse(hipStream_t s, int dm, int nt, CoarseForm form, const MacCoarseArgs<T>* Ap) {
  const unsigned long long A = (unsigned long long)Ap;
  auto go = [&](auto D) {
    constexpr int DM = decltype(D)::value, KM = mac_slots_max<T>(DM);
    if (form == CoarseForm::lds_small) launch_blocks(s, 1, MacCoarseBlk<T, DM, 1, SLOTS_SMALL, 1>{A, nt}, nt);
    else if (form == CoarseForm::lds) launch_blocks(s, 1, MacCoarseBlk<T, DM, 1, KM, 0>{A, nt}, nt);
    else launch_blocks(s, 1, MacCoarseBlk<T, DM, 0, KM, 0>{A, nt}, nt);
  };
  if (dm == 3) go(std::integral_constant<int, 3>{});
  else go(std::integral_constant<int, 2>{});
}
// LMFHD_COARSE_T: the one precision this object holds (the build compiles the file once for each)
#define LMFHD_COARSE(T)                                                                               \
  template void launch_stag_coarse<T>(hipStream_t, int, int, int, CoarseForm, const StagCoarseArgs<T>*); \
  template void launch_mac_coarse<T>(hipStream_t, int, int, CoarseForm, const MacCoarseArgs<T>*);
#ifdef LMFHD_COARSE_T
LMFHD_COARSE(LMFHD_COARSE_T)
#else
LMFHD_COARSE(float)
LMFHD_COARSE(double)
#endif

}  // namespace lmfhd
