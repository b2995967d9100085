// KIVI-style FlagRot INT2 pages for gfx950: per-token value writer and the bf16 LSE merge (the key group
// encoder is in kivi_kenc.hip, the dequantiser in kivi_read.hip).  Compiled with -ffp-contract=off: the quantiser (scale, codes,
// reconstruction) rounds every operation on its own, as the reference's (integrations/vllm_flagrot/csrc/kivi.cu:94-125).
//
// Page chunk per (16-token page, KV head), D = 128: KC @0 [16][32] key codes (32-bit words of 16 channels, channel i at
// bit 2 (i >> 1) + 16 (i & 1)) | KM @512 [16][4] (fp16 scale, fp16 min) of the token's GROUP: cell i = position % 32
// holds channels [4 i, 4 i + 4) | VC @768 [16][32] value codes (byte c / 4, bits 2 (c % 4)) | VM @1280 [16][4]
// (fp16 scale with sign = H32, fp16 min) | VF @1536 [16] u8 (value uses H_128).  Key flags: scale sign of channel
// j < 4 = sub-vector j is H32; of channel 4 = whole head H_128.
//
// FP8-meta pages (F8; kivi.cu:28-35, 84-88, 123-128): scale and min are rounded to E4M3 (nearest even, saturating at
// +-448) BEFORE the codes are computed, so the codes belong to the stored values.  Chunk of 1280 bytes: KC @0 | KM8 @512
// [16][4] byte pairs (s8 | flag << 7, m8) | VC @640 | VM8 @1152 [16][4] byte pairs (bit 7 of s8 = H32).  Key flags: bit 7
// of the scale byte of channel 4 j (slot 0 of cell j) = sub-vector j is H32, of channel 16 (slot 0 of cell 4) = whole
// head.  Bit 7 of the KEY scale byte in slot 3 of a cell is the whole-head flag of the VALUE row stored in that cell: the
// value writer sets it with a byte read-modify-write, the key encoder keeps what it finds there.
//
// One half wave (32 lanes) owns a 128-d row, 4 channels per lane (the helpers of fr_common.hpp).
#include "fr_common.hpp"
#include "kivi_launch.hpp"
#include "kivi_quant.hpp"
#include "kivi_vrow.hpp"
#include "ring_rows.hpp"

namespace frkv {
using namespace fr;
namespace {

template <bool F8> constexpr long long CHUNK = F8 ? 1280 : 1552;
template <bool F8> constexpr int VC_AT = F8 ? 640 : 768;
template <bool F8> constexpr int VM_AT = F8 ? 1152 : 1280;

// ------------------------------------------------------------------------------------------------ value writer
// Half wave per (token, KV head): the three trials, the picks, the stores (kivi_vrow.hpp has the per-row work; the
// kernel loads the row and knows where the chunk keeps what).  WMAT: the picks weigh the miss vectors by a full matrix
// per head (kivi.cu:213-287) and need an LDS strip per half wave; `ident` stores the row as it is, `vfix` takes the
// picks from a word per head (bits 0..3: H32 per sub-vector, bit 16: whole head).
template <bool F8, bool WMAT>
__global__ void __launch_bounds__(256) k_v_write(const uint16_t* __restrict__ kv, long long kv_rs, int n, int Hkv,
                                                 const long long* __restrict__ slots, const float* __restrict__ co,
                                                 const float* __restrict__ M, uint8_t* __restrict__ pool, int ident,
                                                 const int* __restrict__ vfix, const RingRowsParams ring) {
  __shared__ float strips[WMAT ? 8 : 1][WMAT ? 3 * 128 : 1];
  const int l32 = threadIdx.x & 31;
  const long long items = static_cast<long long>(n) * Hkv, groups = (items + 7) / 8;
  if (blockIdx.x >= groups) {                            // behind the values: the BF16 rows of the tokens
    ring_quad(ring, (static_cast<long long>(blockIdx.x) - groups) * 256 + threadIdx.x);
    return;
  }
  const long long item = static_cast<long long>(blockIdx.x) * 8 + (threadIdx.x >> 5);
  if (item >= items) return;
  const int t = static_cast<int>(item / Hkv), h = static_cast<int>(item % Hkv);
  const long long slot = slots[t];
  if (slot < 0) return;
  const uint2 raw = *reinterpret_cast<const uint2*>(kv + static_cast<long long>(t) * kv_rs + (Hkv + h) * 128 + 4 * l32);
  const float x[1][4] = {{bf16_lo(raw.x), bf16_hi(raw.x), bf16_lo(raw.y), bf16_hi(raw.y)}};
  vrow::Trial<1> tr[3];
  vrow::trial_in_basis<1, vrow::AS_STORED, F8>(x, l32, tr[0]);
  vrow::trial_in_basis<1, vrow::BLOCK32, F8>(x, l32, tr[1]);
  vrow::trial_in_basis<1, vrow::WHOLE, F8>(x, l32, tr[2]);
  const int j = l32 >> 3;
  vrow::Picks pk{0u, false};
  if (ident) {
  } else if (vfix != nullptr) {
    pk.whole = (vfix[h] >> 16) & 1;
    pk.block32 = (vfix[h] >> j) & 1u;
  } else if constexpr (WMAT) {
    pk = vrow::pick_matrix<1>(tr, M + static_cast<long long>(h) * 128 * 128, strips[threadIdx.x >> 5], l32);
  } else {
    const float4 c4 = *reinterpret_cast<const float4*>(co + h * 128 + 4 * l32);
    const float w[1][4] = {{c4.x, c4.y, c4.z, c4.w}};
    pk = vrow::pick_diagonal<1>(tr, w, l32);
  }
  const int basis = vrow::basis_of<1>(pk, 0);
  uint8_t* chunk = pool + ((slot / 16) * Hkv + h) * CHUNK<F8>;
  const int off = static_cast<int>(slot % 16);
  chunk[VC_AT<F8> + off * 32 + l32] = static_cast<uint8_t>(vrow::chosen_byte<1>(tr, basis, 0));
  if ((l32 & 7) == 0) {
    const uint32_t meta = vrow::chosen_meta<1, F8>(tr, basis, 0);
    if (F8) *reinterpret_cast<uint16_t*>(chunk + VM_AT<true> + off * 8 + 2 * j) = static_cast<uint16_t>(meta);
    else *reinterpret_cast<uint32_t*>(chunk + VM_AT<false> + off * 16 + 4 * j) = meta;
  }
  if (l32 == 0) {
    if (F8) {                                            // bit 7 of the key scale byte in slot 3 of this token's cell
      uint8_t* kb = chunk + 512 + off * 8 + 6;
      *kb = static_cast<uint8_t>((*kb & 0x7Fu) | (pk.whole ? 0x80u : 0u));
    } else chunk[1536 + off] = pk.whole ? 1 : 0;
  }
}

// ------------------------------------------------------------------------------------------------ LSE merge
__global__ void k_lse_merge(const uint16_t* __restrict__ oa, const float* __restrict__ la, long long la_hs,
                            const uint16_t* __restrict__ ob, const float* __restrict__ lb, long long lb_hs,
                            uint16_t* __restrict__ out, long long out_rs, int na, int H, int D) {
  const long long e = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= static_cast<long long>(na) * H * D) return;
  const int c = static_cast<int>(e % D);
  const long long rh = e / D;
  const int hh = static_cast<int>(rh % H);
  const long long r = rh / H;
  float a = la[hh * la_hs + r], b = lb[hh * lb_hs + r];
  if (a == INFINITY) a = -INFINITY;
  if (b == INFINITY) b = -INFINITY;
  const float m = (a != a || b != b) ? NAN : fmaxf(a, b);
  const float wa = expf(a - m), wb = expf(b - m);
  const float va = bf16_lo(oa[(r * H + hh) * D + c]), vb = bf16_lo(ob[(r * H + hh) * D + c]);
  const float num = va * wa + vb * wb;
  out[r * out_rs + static_cast<long long>(hh) * D + c] = static_cast<uint16_t>(bf16_rn(num / (wa + wb)));
}

}  // namespace

int v_write_launch(const void* kv, long long kv_rs, int n, int Hkv, const long long* slots, const float* co, uint8_t* pool,
                   const float* M, int ident, const int* vfix, int f8, hipStream_t st, const RingRowsParams& ring) {
  const long long items = static_cast<long long>(n) * Hkv;
  const bool wmat = M != nullptr && !ident && vfix == nullptr;
  const auto kern = wmat ? (f8 ? k_v_write<true, true> : k_v_write<false, true>) : (f8 ? k_v_write<true, false> : k_v_write<false, false>);
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>((items + 7) / 8 + (ring_quads(ring) + 255) / 256)), dim3(256), 0, st,
                     static_cast<const uint16_t*>(kv), kv_rs, n, Hkv, slots, co, M, pool, ident, vfix, ring);
  return hipPeekAtLastError() == hipSuccess ? 0 : 1;
}

int lse_merge_launch(const void* oa, const float* la, long long la_hs, const void* ob, const float* lb, long long lb_hs,
                     void* out, long long out_rs, int na, int H, int D, hipStream_t st) {
  const long long tot = static_cast<long long>(na) * H * D;
  hipLaunchKernelGGL(k_lse_merge, dim3(static_cast<unsigned>((tot + 255) / 256)), dim3(256), 0, st,
                     static_cast<const uint16_t*>(oa), la, la_hs, static_cast<const uint16_t*>(ob), lb, lb_hs,
                     static_cast<uint16_t*>(out), out_rs, na, H, D);
  return hipPeekAtLastError() == hipSuccess ? 0 : 1;
}

}  // namespace frkv
