// The batched scenes' kernels with correctly rounded trig (a file of its own: they compile for a minute).
#include "batch_kernels.hpp"

namespace pe_amd {

void launch_batch_exact(int model, const Bodies& B, const RawContacts& R, const SolverContacts& C, const BatchArgs& A,
                      uint32_t grid, uint32_t threads, bool wide, hipStream_t s) {
  batch_dispatch<TrigExact>(model, B, R, C, A, grid, threads, wide, s);
}

}  // namespace pe_amd
