// The batched scenes' kernels with the device libm (a file of its own: they compile for a minute).
#include "batch_kernels.hpp"

namespace pe_amd {

void launch_batch_fast(int model, const Bodies& B, const RawContacts& R, const SolverContacts& C, const BatchArgs& A,
                      uint32_t grid, uint32_t threads, bool wide, hipStream_t s) {
  batch_dispatch<TrigFast>(model, B, R, C, A, grid, threads, wide, s);
}

__global__ void k_batch_begin(uint32_t* queue, uint32_t add_steps) {
  if (threadIdx.x == 0) {
    queue[0] = 0;
    queue[1] += add_steps;
  }
}

void launch_batch_begin(uint32_t* queue, uint32_t add_steps, hipStream_t s) {
  hipLaunchKernelGGL(k_batch_begin, dim3(1), dim3(64), 0, s, queue, add_steps);
}

void launch_batch(int model, bool exact_trig, const Bodies& B, const RawContacts& R, const SolverContacts& C,
                  const BatchArgs& A, uint32_t grid, uint32_t threads, bool wide, hipStream_t s) {
  if (exact_trig) launch_batch_exact(model, B, R, C, A, grid, threads, wide, s);
  else launch_batch_fast(model, B, R, C, A, grid, threads, wide, s);
}

}  // namespace pe_amd
