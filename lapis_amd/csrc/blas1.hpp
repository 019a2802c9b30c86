// Internal interface of the dot kernel, shared with the CG driver.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace lapis {

constexpr int kDotMaxBlocks = 2048;  // upper bound of dot_grid(); sizes the partials scratch

// Number of blocks (= partial sums) a dot over n elements uses.
int dot_grid(int64_t n);

// *result = init + sum x[i]*y[i].  `partials` holds kDotMaxBlocks elements of T.
template <typename T>
int launch_dot(int64_t n, const T *x, const T *y, T init, T *result, T *partials, hipStream_t st);

// A dot product on its way to the host: its kernel leaves one partial sum per block in pinned memory, and dot_finish
// adds them up as they arrive (blas1.hip).
struct HostSum {
  double *parts = nullptr;  // kDotMaxBlocks
  int count = 0;
  double init = 0.0;
  bool f32 = false;  // the parts are floats and added up as such
  hipStream_t stream = nullptr;
};
// For a kernel that will leave `count` parts: take one, launch, hand it to dot_finish (or dot_abandon).
int take_host_sum(int count, double init, bool f32, hipStream_t st, HostSum **out);
template <typename T>
int dot_start(int64_t n, const T *x, const T *y, double init, hipStream_t st, HostSum **out);
template <typename T>
int axpby_dot_start(int64_t n, T a, const T *x, T b, const T *y, T *dst, const T *z, double init, hipStream_t st, HostSum **out);
int dot_finish(HostSum *sum, double *result);  // init + the parts; gives the sum back whatever it returns
void dot_abandon(HostSum *sum);                // after an error: waits and gives it back

#ifdef __HIPCC__
// A store that reaches pinned host memory when it is made, not when the kernel ends.
__device__ __forceinline__ void tell_host(double *where, double v) {
  __hip_atomic_store(where, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
#endif

// Per-device set-up of lapis_hip_dot_f64_noalloc (address of its fixed scratch array) and
// release of the allocated ring of partials the other dot entry points use.
int dot_noalloc_setup();
void dot_release_scratch();
// Gives back the scratch of finished CG solves (cg.hip).
void cg_release_scratch();

}  // namespace lapis
