// The BF16 rows a request keeps beside its pages (sinks and the window ring): rows of a prompt, of a prompt chunk or of a
// decode step copied to their ring slots, the key half with the static mean removed (FP32 subtraction, one BF16 rounding).
// Slot of position p: p < S ? p : S + (p - S) % W (integrations/vllm_flagrot/vllm_flagrot/attention/backend.py:1266-1325).
//
// Bound by its launch: 132 rows of 8 + 8 heads are 1 MB.  One thread moves four channels (8 bytes: what the writers ask
// of a row's alignment), so a row of 4 KB is two workgroups' width and every access is contiguous.  The positions that
// stay are two ranges known to the host -- nothing is searched for on the device and the host does not wait (as torch
// operations over boolean masks: 28 kernels and two waits for the device, 130 us of a prompt of 8192 tokens; 5 us here).
#include "ring_rows.hpp"

namespace fr {
namespace {

__global__ void __launch_bounds__(256) k_ring_rows(const RingRowsParams p) {
  ring_quad(p, static_cast<long long>(blockIdx.x) * 256 + threadIdx.x);
}

}  // namespace

int ring_rows_launch(const RingRowsParams& p, hipStream_t st) {
  const long long threads = ring_quads(p);
  if (threads == 0) return 0;
  hipLaunchKernelGGL(k_ring_rows, dim3(static_cast<unsigned>((threads + 255) / 256)), dim3(256), 0, st, p);
  return hipPeekAtLastError() == hipSuccess ? 0 : -1;
}

}  // namespace fr
