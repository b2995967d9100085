// The BF16 rows a request keeps beside its pages (sinks and the window ring): rows of a prompt, of a prompt chunk or of a
// decode step copied to their ring slots, the key half with the static mean removed (FP32 subtraction, one BF16 rounding).
// Slot of position p: p < S ? p : S + (p - S) % W (integrations/vllm_flagrot/vllm_flagrot/attention/backend.py:1266-1325).
//
// Bound by its launch: 132 rows of 8 + 8 heads are 1 MB.  One thread moves four channels (8 bytes: what the writers ask
// of a row's alignment), so a row of 4 KB is two workgroups' width and every access is contiguous.  The positions that
// stay are two ranges known to the host -- nothing is searched for on the device and the host does not wait (as torch
// operations over boolean masks: 28 kernels and two waits for the device, 130 us of a prompt of 8192 tokens; 5 us here).
#include "fr_common.hpp"
#include "fr_launch.hpp"

namespace fr {
namespace {

DEVI uint32_t bf16_row_rn(float f) { return f != f ? 0x7FC0u : bf16_rn(f); }      // (the rounding alone may lose a NaN)

__global__ void __launch_bounds__(256) k_ring_rows(const RingRowsParams p) {
  const int quads = p.width / 4;                           // of one row: K heads, then V heads
  const long long at = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
  if (at >= static_cast<long long>(p.rows) * quads) return;
  const int r = static_cast<int>(at / quads), c = 4 * static_cast<int>(at % quads);
  int t = r;
  long long slot;
  if (p.dest != nullptr) slot = p.dest[r];
  else {                                                   // the leading sinks of the chunk, then the rows of its window
    t = r < p.sinks ? r : p.win0 + (r - p.sinks);
    const int pos = p.start + t;
    slot = p.base + (pos < p.S ? pos : p.S + (pos - p.S) % p.W);
  }
  if (slot < 0 || slot >= p.ring_rows) return;
  uint2 raw = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(p.kv) + static_cast<long long>(t) * p.kv_ts + c);
  if (p.kmu != nullptr && c < p.width / 2) {
    const float4 m = *reinterpret_cast<const float4*>(p.kmu + c);
    raw.x = bf16_row_rn(bf16_lo(raw.x) - m.x) | (bf16_row_rn(bf16_hi(raw.x) - m.y) << 16);
    raw.y = bf16_row_rn(bf16_lo(raw.y) - m.z) | (bf16_row_rn(bf16_hi(raw.y) - m.w) << 16);
  }
  *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p.ring) + slot * p.width + c) = raw;
}

}  // namespace

int ring_rows_launch(const RingRowsParams& p, hipStream_t st) {
  const long long threads = static_cast<long long>(p.rows) * (p.width / 4);
  if (threads == 0) return 0;
  hipLaunchKernelGGL(k_ring_rows, dim3(static_cast<unsigned>((threads + 255) / 256)), dim3(256), 0, st, p);
  return hipPeekAtLastError() == hipSuccess ? 0 : -1;
}

}  // namespace fr
