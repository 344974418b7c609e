// rsg_state.hip -- a handle's state between its internal order and the caller's.
//
// The arrays V[3][nn], S[6][nc] in the caller's numbering form one index space; a launch moves a
// range of it between the device's state and a chunk of pinned host memory, in the handle's
// precision.  The kernels read or write the chunk in order, so what crosses the bus is whole
// lines, and the scattered side of the reordering is in HBM.  Bound by the bus: the 283 MB FP64
// state of a 3.9 M-cell plate takes 6.3 ms (45 GB/s) to the caller's arrays, where whole-array
// copies and a reordering loop on the host took 67 ms.
#include <hip/hip_runtime.h>

#include "rsg_internal.h"

namespace rsg {
namespace {

// The state's value at index g of the caller's arrays.
template <typename T>
__device__ __forceinline__ T* state_at(const StateArgs<T>& a, int64_t g) {
  const int64_t v = (int64_t)3 * a.nn;
  if (g < v) {
    const int d = (int)(g / a.nn);
    return a.V[d] + a.node_at[g - (int64_t)d * a.nn];
  }
  const int s = (int)((g - v) / a.nc);
  return a.S[s] + a.cell_at[g - v - (int64_t)s * a.nc];
}

template <typename T>
__global__ __launch_bounds__(256) void state_read_kernel(StateArgs<T> a, int64_t g0, int n, T* __restrict__ out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = *state_at(a, g0 + i);
}

template <typename T>
__global__ __launch_bounds__(256) void state_write_kernel(StateArgs<T> a, int64_t g0, int n,
                                                          const T* __restrict__ in) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) *state_at(a, g0 + i) = in[i];
}

template <typename T>
hipError_t launch(const StateArgs<T>& a, int64_t g0, int n, T* chunk, bool write, hipStream_t s) {
  if (n <= 0 || n > kStateChunk || g0 < 0 || g0 + n > (int64_t)3 * a.nn + (int64_t)6 * a.nc || !chunk)
    return hipErrorInvalidValue;
  // (hipLaunchKernel's own result: the thread's last error may be another call's)
  const void* const fn = write ? reinterpret_cast<const void*>(&state_write_kernel<T>)
                               : reinterpret_cast<const void*>(&state_read_kernel<T>);
  StateArgs<T> arg = a;
  void* args[4] = {&arg, &g0, &n, &chunk};
  return hipLaunchKernel(fn, dim3((n + 255) / 256), dim3(256), args, 0, s);
}

}  // namespace

hipError_t launch_state_f64(const StateArgs<double>& a, int64_t g0, int n, double* chunk, bool write, hipStream_t s) {
  return launch<double>(a, g0, n, chunk, write, s);
}
hipError_t launch_state_f32(const StateArgs<float>& a, int64_t g0, int n, float* chunk, bool write, hipStream_t s) {
  return launch<float>(a, g0, n, chunk, write, s);
}

}  // namespace rsg
