// Selecting writer of a decode step: a handful of tokens, one workgroup per (token, KV head) (writer_exact.hpp).
// Same bytes as k_k2_write (writer.hip).
//
// Bound by latency: launch, one trip to memory and the chains of the exact evaluation.  Call of 32 tokens x 8 heads of
// 128, 4-bit / 2-bit pages: 11.6 / 13.4 -> 5.7 us (before: four half waves per token, C_q^T staged in LDS, 2-bit value
// fields that met on one word); 16 tokens x 4 heads of 256: 47 -> 6.8 us (one half wave per token).
#include "ring_rows.hpp"
#include "writer_exact.hpp"

namespace fr {
namespace {

// RING: workgroups behind the tokens' copy their BF16 rows.  A kernel of its own: the test alone is 1 to 2 % of a call without
// rows (graph of calls, 100 tokens x 8 heads on 4-bit pages 9.62 -> 9.44 us, 100 x 4 heads of 256 12.35 -> 12.12).
template <int QM, int P, int D, bool RING>
__global__ void __launch_bounds__(2 * D) k_k2_step(const K2WriteParams p) {
  __shared__ StepSmem<D> S;
  const int h = blockIdx.x, t = blockIdx.y;
  if constexpr (RING) {
    if (t >= p.T) {
      ring_quad(p.ring, (static_cast<long long>(t - p.T) * p.Hkv + h) * (2 * D) + threadIdx.x);
      return;
    }
  }
  const long long slot = p.slots[static_cast<long long>(t) * (p.slot_ph ? p.Hkv : 1) + (p.slot_ph ? h : 0)];
  if (slot < 0) return;                            // the whole workgroup
  CqRegs<D> C;
  k2_exact_token<QM, P, D, true>(p, S, C, h, t, slot);
}

template <int QM, int P>
void step(const K2WriteParams& p, hipStream_t st) {
  const long long per_row = static_cast<long long>(p.Hkv) * 256;                            // quads of a row of workgroups
  const dim3 grid(p.Hkv, p.T + static_cast<unsigned>((ring_quads(p.ring) + per_row - 1) / per_row));
  if (p.hd == 256) hipLaunchKernelGGL((k_k2_step<QM, P, 256, false>), grid, dim3(512), 0, st, p);
  else if (p.ring.rows > 0) hipLaunchKernelGGL((k_k2_step<QM, P, 128, true>), grid, dim3(256), 0, st, p);
  else hipLaunchKernelGGL((k_k2_step<QM, P, 128, false>), grid, dim3(256), 0, st, p);
}
template <int QM>
int step_qm(const K2WriteParams& p, hipStream_t st) {
  if (p.page == 16) step<QM, 16>(p, st);
  else if (p.page == 32) step<QM, 32>(p, st);
  else return -5;
  return hipPeekAtLastError() == hipSuccess ? 0 : -1;
}

}  // namespace

int k2_step_launch(int kind, const K2WriteParams& p, hipStream_t st) {
  switch (kind) {
    case KIND_KONLY: return step_qm<QM_SYM4>(p, st);
    case KIND_KONLYA: return step_qm<QM_ASYM4>(p, st);
    case KIND_KONLYA2: return step_qm<QM_ASYM2>(p, st);
  }
  return -4;
}

}  // namespace fr
