// KIVI-style FlagRot INT2 pages at head dim 256 for gfx950: value writer, page dequantiser and the decode attention
// with its split merge (integrations/vllm_flagrot/csrc/kivi.cu:163-328 k_v_write<256>, :2067-2300 the dequantisers,
// :1997-2036 the 256-d attention launches); the key group encoder is in kivi_kenc.hip.  Compiled with
// -ffp-contract=off like the 128-d writers: the quantiser rounds every operation on its own.
//
// Page chunk per (16-token page, KV head), D = 256, NV = 8 sub-vectors (kivi.cu:15-35):
//   FP16 meta, 3088 bytes: KC @0 [16][64] key codes (32-bit words of 16 channels, channel i at bit 2 (i >> 1) +
//     16 (i & 1)) | KM @1024 [16][8] (fp16 scale, fp16 min) of the token's GROUP: cell i = position % 32 holds channels
//     [8 i, 8 i + 8) | VC @1536 [16][64] value codes | VM @2560 [16][8] (fp16 scale with sign = H32, fp16 min) |
//     VF @3072 [16] u8 (value uses H_256).  Key flags: scale sign of channel j < 8 = sub-vector j is H32, of channel 8 =
//     whole head H_256.
//   FP8 meta, 2560 bytes: KC @0 | KM8 @1024 [16][8] byte pairs | VC @1280 | VM8 @2304 [16][8] byte pairs.  Key flags:
//     bit 7 of the scale byte of channel 8 j (slot 0 of cell j), of channel 64 (slot 0 of cell 8) = whole head; bit 7 of
//     the key scale byte in slot 7 of a cell = whole-head flag of the VALUE row stored in that cell.
//
// A half wave (32 lanes) owns a 256-d row as two 128-d halves: lane l holds channels 128 s + 4 l + i (s = 0, 1), so the
// 32-blocks and the 128-d butterflies are the helpers of fr_common.hpp on each half, and H_256 adds the stage of
// distance 128 between the two registers of a lane and the exact factor 1/16.  The staged butterflies meet their
// partners in the reference's order (distance 1, 2, 4, ..), so every transformed value is the reference's bit for bit.
//
// The attention kernel here is the plain fp32 form (no matrix cores): per 32-token group, scores by (token, sub-vector)
// threads against the three rotated queries, one softmax per head in a half wave, values by channel threads into one
// accumulator per (head, basis), the two inverse transforms once at the end.  It runs only when
// FLAGROT_KIVI_WIDE_PLAIN=1 asks for it: the launches go through the matrix-pipe kernel of kivi_decode_wide.hip.
// Same partials either way, one merge kernel.
#include <cstdlib>

#include "fr_common.hpp"
#include "kivi_launch.hpp"
#include "kivi_merge.hpp"
#include "kivi_quant.hpp"
#include "kivi_vrow.hpp"

namespace frkv {
using namespace fr;
namespace {

constexpr int D2 = 256, NV2 = 8;
template <bool F8> constexpr long long CHUNK2 = F8 ? 2560 : 3088;
constexpr int KM2 = 1024;
template <bool F8> constexpr int VC2 = F8 ? 1280 : 1536;
template <bool F8> constexpr int VM2 = F8 ? 2304 : 2560;
constexpr int VF2 = 3072;
template <bool F8> constexpr int CELL = F8 ? 16 : 32;                 // bytes of meta per cell (8 entries)

template <int C> DEVI void to_basis2(float (&y)[2][4], int l32) {     // candidate 0 identity, 1 H32, 2 H256 (involutions)
  if (C == 1) { fwht<32>(y[0], l32); fwht<32>(y[1], l32); }
  if (C == 2) h256(y, l32);
}
DEVI void load_row(const uint16_t* row, int l32, float (&x)[2][4]) {  // bf16 row of 256
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const uint2 raw = *reinterpret_cast<const uint2*>(row + 128 * s + 4 * l32);
    x[s][0] = bf16_lo(raw.x); x[s][1] = bf16_hi(raw.x); x[s][2] = bf16_lo(raw.y); x[s][3] = bf16_hi(raw.y);
  }
}
template <bool F8> DEVI void meta_read(const uint8_t* at, float& s, float& mn, bool& flag) {   // one (scale, min) entry
  if (F8) { flag = at[0] >> 7; s = e4m3_value(at[0] & 0x7Fu); mn = e4m3_value(at[1]); }
  else {
    const uint32_t w = *reinterpret_cast<const uint32_t*>(at);
    flag = (w >> 15) & 1u; s = f16_value(w & 0x7FFFu); mn = f16_value(w >> 16);
  }
}
template <bool F8> DEVI bool value_whole(const uint8_t* chunk, int cell) {
  return F8 ? (chunk[KM2 + cell * 16 + 14] >> 7) != 0 : chunk[VF2 + cell] != 0;
}

// ------------------------------------------------------------------------------------------------ value writer
// Half wave per (token, KV head), the row as two halves of 128 channels: the three trials, the picks, the stores
// (kivi_vrow.hpp has the per-row work).  WMAT: picks by a full 256 x 256 matrix per head (kivi.cu:213-287) through an
// LDS strip per half wave; `vfix` bits 0..7: H32 per sub-vector, bit 16: whole head.
template <bool F8, bool WMAT>
__global__ void __launch_bounds__(256) k_v_write256(const uint16_t* __restrict__ kv, long long kv_rs, int n, int Hkv,
                                                    const long long* __restrict__ slots, const float* __restrict__ co,
                                                    const float* __restrict__ M, uint8_t* __restrict__ pool, int ident,
                                                    const int* __restrict__ vfix) {
  __shared__ float strips[WMAT ? 8 : 1][WMAT ? 3 * D2 : 1];
  const int l32 = threadIdx.x & 31;
  const long long item = static_cast<long long>(blockIdx.x) * 8 + (threadIdx.x >> 5);
  if (item >= static_cast<long long>(n) * Hkv) return;
  const int t = static_cast<int>(item / Hkv), h = static_cast<int>(item % Hkv);
  const long long slot = slots[t];
  if (slot < 0) return;
  float x[2][4];
  load_row(kv + static_cast<long long>(t) * kv_rs + static_cast<long long>(Hkv + h) * D2, l32, x);
  vrow::Trial<2> tr[3];
  vrow::trial_in_basis<2, vrow::AS_STORED, F8>(x, l32, tr[0]);
  vrow::trial_in_basis<2, vrow::BLOCK32, F8>(x, l32, tr[1]);
  vrow::trial_in_basis<2, vrow::WHOLE, F8>(x, l32, tr[2]);
  const int j = l32 >> 3;
  vrow::Picks pk{0u, false};
  if (ident) {
  } else if (vfix != nullptr) {
    pk.whole = (vfix[h] >> 16) & 1;
    pk.block32 = ((vfix[h] >> j) & 1u) | (((vfix[h] >> (4 + j)) & 1u) << 1);
  } else if constexpr (WMAT) {
    pk = vrow::pick_matrix<2>(tr, M + static_cast<long long>(h) * D2 * D2, strips[threadIdx.x >> 5], l32);
  } else {
    float w[2][4];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const float4 c4 = *reinterpret_cast<const float4*>(co + h * D2 + 128 * s + 4 * l32);
      w[s][0] = c4.x; w[s][1] = c4.y; w[s][2] = c4.z; w[s][3] = c4.w;
    }
    pk = vrow::pick_diagonal<2>(tr, w, l32);
  }
  uint8_t* chunk = pool + ((slot / 16) * Hkv + h) * CHUNK2<F8>;
  const int off = static_cast<int>(slot % 16);
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int basis = vrow::basis_of<2>(pk, s);
    chunk[VC2<F8> + off * 64 + 32 * s + l32] = static_cast<uint8_t>(vrow::chosen_byte<2>(tr, basis, s));
    if ((l32 & 7) == 0) {
      const uint32_t meta = vrow::chosen_meta<2, F8>(tr, basis, s);
      const int jj = 4 * s + j;
      if (F8) *reinterpret_cast<uint16_t*>(chunk + VM2<true> + off * 16 + 2 * jj) = static_cast<uint16_t>(meta);
      else *reinterpret_cast<uint32_t*>(chunk + VM2<false> + off * 32 + 4 * jj) = meta;
    }
  }
  if (l32 == 0) {
    if (F8) {                                              // bit 7 of the key scale byte in slot 7 of this token's cell
      uint8_t* kb = chunk + KM2 + off * 16 + 14;
      *kb = static_cast<uint8_t>((*kb & 0x7Fu) | (pk.whole ? 0x80u : 0u));
    } else chunk[VF2 + off] = pk.whole ? 1 : 0;
  }
}

DEVI void lds_row(const float* row, int l32, float (&x)[2][4]) {
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const float4 v = *reinterpret_cast<const float4*>(row + 128 * s + 4 * l32);
    x[s][0] = v.x; x[s][1] = v.y; x[s][2] = v.z; x[s][3] = v.w;
  }
}
DEVI void lds_put(float* row, int l32, const float (&x)[2][4]) {
#pragma unroll
  for (int s = 0; s < 2; ++s) *reinterpret_cast<float4*>(row + 128 * s + 4 * l32) = make_float4(x[s][0], x[s][1], x[s][2], x[s][3]);
}

// ------------------------------------------------------------------------------------------------ dequantiser
template <bool F8> DEVI uint32_t key_flags(const uint8_t* chA) {
  uint32_t f = 0;
  if (F8) {
    for (int j = 0; j < 9; ++j) f |= static_cast<uint32_t>(chA[KM2 + 16 * j] >> 7) << j;
  } else {
    const uint32_t* m0 = reinterpret_cast<const uint32_t*>(chA + KM2);           // cell 0 slots 0..7, cell 1 slot 0
    for (int j = 0; j < 9; ++j) f |= ((m0[j] >> 15) & 1u) << j;
  }
  return f;
}

// ------------------------------------------------------------------------------------------------ decode attention
constexpr int GW = 8;                                     // query heads per KV head, at most
struct WideAttn {
  float qv[3][GW][D2];                                    // query x qscale: as it is, H32 per sub-vector, H256
  float ks[D2], kmn[D2];                                  // channel (scale, min) of the current group
  float part[NV2][GW][32];                                // partial scores per sub-vector
  float pr[GW][32];                                       // probabilities of the group
  float alpha[GW];
  float vs[32][NV2], vmn[32][NV2];
  int vcls[32][NV2];                                      // basis of (token, sub-vector): 0 identity, 1 H32, 2 H256
  int kfl;
};

// One workgroup per (sequence, KV head, split).  Split sp < NS: page tokens [max(sp chunk, kv_start), min((sp + 1) chunk,
// cached)); split NS: the BF16 ring rows.  Partials: opart fp32 [G][256] unnormalised, ml fp32 [G][2] = (max, sum).
template <bool F8>
__global__ void __launch_bounds__(256) k_attn256(const uint16_t* __restrict__ q, long long q_rs,
                                                 const uint8_t* __restrict__ pool, const int* __restrict__ bt, long long bt_rs,
                                                 const int* __restrict__ cached, int kv_start, int Hkv, int G, int NS,
                                                 int chunk, float qscale, const uint16_t* __restrict__ ring,
                                                 const int* __restrict__ tail_len, const int* __restrict__ tail_idx, int T,
                                                 float* __restrict__ opart, float* __restrict__ ml) {
  extern __shared__ __align__(16) uint8_t lds[];
  WideAttn& S = *reinterpret_cast<WideAttn*>(lds);
  const int b = blockIdx.x, h = blockIdx.y, sp = blockIdx.z;
  const int tid = threadIdx.x, hw = tid >> 5, l32 = tid & 31;
  const long long pidx = (static_cast<long long>(b) * Hkv + h) * (NS + 1) + sp;
  float* op = opart + pidx * G * D2;
  float* mlp = ml + pidx * G * 2;
  const bool tail = sp == NS;
  int t0, t1;
  if (tail) { t0 = 0; t1 = tail_len != nullptr ? tail_len[b] : 0; }
  else { t0 = max(sp * chunk, kv_start); t1 = min((sp + 1) * chunk, cached[b]); }
  if (t1 <= t0) {
    if (tid < G) { mlp[2 * tid] = -INFINITY; mlp[2 * tid + 1] = 0.f; }
    return;
  }
  // rotated queries: half wave hw <-> head hw (zero rows past the group)
  {
    float x[2][4];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i) x[s][i] = 0.f;
    if (hw < G) load_row(q + static_cast<long long>(b) * q_rs + (static_cast<long long>(h) * G + hw) * D2, l32, x);
    float y[2][4], z[2][4];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i) { y[s][i] = x[s][i]; z[s][i] = x[s][i]; }
    to_basis2<1>(y, l32);
    to_basis2<2>(z, l32);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i) { x[s][i] *= qscale; y[s][i] *= qscale; z[s][i] *= qscale; }
    lds_put(S.qv[0][hw], l32, x);
    lds_put(S.qv[1][hw], l32, y);
    lds_put(S.qv[2][hw], l32, z);
  }
  const int* btb = bt + static_cast<long long>(b) * bt_rs;
  const uint16_t* rbase = tail ? ring + static_cast<long long>(tail_idx != nullptr ? tail_idx[b] : 0) * T * 2 * Hkv * D2 : nullptr;
  float m_run = -INFINITY, l_run = 0.f;                   // of head hw (the same in every lane of the half wave)
  float o[3][GW];                                         // channel tid, per basis and head
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int g = 0; g < GW; ++g) o[c][g] = 0.f;
  const int g_first = t0 / 32, g_end = (t1 + 31) / 32;
  for (int grp = g_first; grp < g_end; ++grp) {
    __syncthreads();                                      // the previous group's values are done with the staged fields
    const uint8_t *chA = nullptr, *chB = nullptr;
    if (!tail) {
      chA = pool + (static_cast<long long>(btb[2 * grp]) * Hkv + h) * CHUNK2<F8>;
      chB = pool + (static_cast<long long>(btb[2 * grp + 1]) * Hkv + h) * CHUNK2<F8>;
      {                                                   // channel tid: cell tid >> 3 (page B from cell 16 on), slot tid & 7
        const int cell = tid >> 3;
        bool fl;
        meta_read<F8>((cell < 16 ? chA : chB) + KM2 + (cell & 15) * CELL<F8> + (tid & 7) * (F8 ? 2 : 4), S.ks[tid], S.kmn[tid], fl);
      }
      if (tid == 0) S.kfl = static_cast<int>(key_flags<F8>(chA));
      {                                                   // value meta of (token l32, sub-vector hw)
        const uint8_t* cht = l32 < 16 ? chA : chB;
        bool fl;
        meta_read<F8>(cht + VM2<F8> + (l32 & 15) * CELL<F8> + hw * (F8 ? 2 : 4), S.vs[l32][hw], S.vmn[l32][hw], fl);
        S.vcls[l32][hw] = value_whole<F8>(cht, l32 & 15) ? 2 : (fl ? 1 : 0);
      }
    }
    __syncthreads();
    // scores: thread (token l32, sub-vector hw)
    {
      const int pos = 32 * grp + l32;
      float acc[GW];
#pragma unroll
      for (int g = 0; g < GW; ++g) acc[g] = 0.f;
      if (tail) {
        if (pos < t1) {
          const uint16_t* row = rbase + static_cast<long long>(pos) * 2 * Hkv * D2 + static_cast<long long>(h) * D2 + 32 * hw;
          for (int c8 = 0; c8 < 4; ++c8) {
            const uint4 raw = *reinterpret_cast<const uint4*>(row + 8 * c8);
            const float kf[8] = {bf16_lo(raw.x), bf16_hi(raw.x), bf16_lo(raw.y), bf16_hi(raw.y),
                                 bf16_lo(raw.z), bf16_hi(raw.z), bf16_lo(raw.w), bf16_hi(raw.w)};
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
              for (int g = 0; g < GW; ++g) acc[g] += kf[i] * S.qv[0][g][32 * hw + 8 * c8 + i];
          }
        }
      } else {
        const int var = (S.kfl >> 8) & 1 ? 2 : (S.kfl >> hw) & 1;
        const uint8_t* cht = l32 < 16 ? chA : chB;
        const uint2 w2 = *reinterpret_cast<const uint2*>(cht + (l32 & 15) * 64 + 8 * hw);
        const float (*qr)[D2] = S.qv[var];
#pragma unroll
        for (int wi = 0; wi < 2; ++wi) {
          const uint32_t w = wi ? w2.y : w2.x;
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int c = 32 * hw + 16 * wi + i;
            const float k = static_cast<float>((w >> (2 * (i >> 1) + 16 * (i & 1))) & 3u) * S.ks[c] + S.kmn[c];
#pragma unroll
            for (int g = 0; g < GW; ++g) acc[g] += k * qr[g][c];
          }
        }
      }
#pragma unroll
      for (int g = 0; g < GW; ++g) S.part[hw][g][l32] = acc[g];
    }
    __syncthreads();
    // softmax: half wave hw <-> head hw, lane <-> token
    {
      const int pos = 32 * grp + l32;
      float sc = 0.f;
#pragma unroll
      for (int j = 0; j < NV2; ++j) sc += S.part[j][hw][l32];
      if (pos < t0 || pos >= t1) sc = -INFINITY;
      float mx = sc;
#pragma unroll
      for (int m = 1; m < 32; m <<= 1) mx = fmaxf(mx, hx(mx, m));
      const float m_new = fmaxf(m_run, mx);
      const float p = sc == -INFINITY ? 0.f : exp2f(sc - m_new);
      const float a = m_run == -INFINITY ? 0.f : exp2f(m_run - m_new);
      float ps = p;
#pragma unroll
      for (int m = 1; m < 32; m <<= 1) ps += hx(ps, m);
      l_run = l_run * a + ps;
      m_run = m_new;
      S.pr[hw][l32] = p;
      if (l32 == 0) S.alpha[hw] = m_new == -INFINITY ? 1.f : a;
    }
    __syncthreads();
    // values: thread <-> channel tid
    {
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int g = 0; g < GW; ++g) o[c][g] *= S.alpha[g];
      const int j = tid >> 5, nrow = min(32, t1 - 32 * grp);
      for (int t = max(0, t0 - 32 * grp); t < nrow; ++t) {
        float v;
        int cls = 0;
        if (tail) v = bf16_lo(rbase[static_cast<long long>(32 * grp + t) * 2 * Hkv * D2 + static_cast<long long>(Hkv + h) * D2 + tid]);
        else {
          const uint8_t* cht = t < 16 ? chA : chB;
          const uint32_t byte = cht[VC2<F8> + (t & 15) * 64 + (tid >> 2)];
          v = static_cast<float>((byte >> (2 * (tid & 3))) & 3u) * S.vs[t][j] + S.vmn[t][j];
          cls = S.vcls[t][j];
        }
        const float v0 = cls == 0 ? v : 0.f, v1 = cls == 1 ? v : 0.f, v2 = cls == 2 ? v : 0.f;
#pragma unroll
        for (int g = 0; g < GW; ++g) {
          const float p = S.pr[g][t];
          o[0][g] += p * v0; o[1][g] += p * v1; o[2][g] += p * v2;
        }
      }
    }
  }
  // back to the original basis: the H32 and the H256 accumulators through LDS (the query rows are free now)
  __syncthreads();
#pragma unroll
  for (int c = 1; c < 3; ++c)
#pragma unroll
    for (int g = 0; g < GW; ++g) S.qv[c][g][tid] = o[c][g];
  __syncthreads();
  {
    float y[2][4], z[2][4];
    lds_row(S.qv[1][hw], l32, y);
    lds_row(S.qv[2][hw], l32, z);
    to_basis2<1>(y, l32);
    to_basis2<2>(z, l32);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i) y[s][i] += z[s][i];
    lds_put(S.qv[1][hw], l32, y);
  }
  __syncthreads();
  for (int g = 0; g < G; ++g) op[g * D2 + tid] = o[0][g] + S.qv[1][g][tid];
  if (l32 == 0 && hw < G) { mlp[2 * hw] = m_run; mlp[2 * hw + 1] = l_run; }
}

template <typename K> bool carve(K kern, size_t bytes) {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                             static_cast<int>(bytes)) == hipSuccess;
}

}  // namespace

int v_write256_launch(const void* kv, long long kv_rs, int n, int Hkv, const long long* slots, const float* co, uint8_t* pool,
                      const float* M, int ident, const int* vfix, int f8, hipStream_t st) {
  const long long items = static_cast<long long>(n) * Hkv;
  const bool wmat = M != nullptr && !ident && vfix == nullptr;
  const auto kern = wmat ? (f8 ? k_v_write256<true, true> : k_v_write256<false, true>)
                         : (f8 ? k_v_write256<true, false> : k_v_write256<false, false>);
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>((items + 7) / 8)), dim3(256), 0, st, static_cast<const uint16_t*>(kv),
                     kv_rs, n, Hkv, slots, co, M, pool, ident, vfix);
  return hipPeekAtLastError() == hipSuccess ? 0 : 1;
}

int attn256_launch(int G, const void* q, long long q_rs, const void* pool, const void* bt, long long bt_rs, const void* cached,
                   int kv_start, int B, int Hkv, int NS, int chunk, float qscale, const void* ring, const void* tail_len,
                   const void* tail_idx, int T, void* opart, void* ml, void* out, long long out_rs, int f8, hipStream_t st) {
  if (G < 1 || G > GW) return 2;
  static bool attr = false;
  if (!attr) {
    if (!carve(&k_attn256<false>, sizeof(WideAttn)) || !carve(&k_attn256<true>, sizeof(WideAttn))) return 1;
    attr = true;
  }
  // every split through the matrix-pipe kernel file (kivi_decode_wide.hip) unless FLAGROT_KIVI_WIDE_PLAIN=1 (read at
  // every call) asks for the plain kernel of this file
  const char* env = std::getenv("FLAGROT_KIVI_WIDE_PLAIN");
  if (env != nullptr && env[0] == '1') {
    const auto kern = f8 ? k_attn256<true> : k_attn256<false>;
    hipLaunchKernelGGL(kern, dim3(B, Hkv, NS + 1), dim3(256), sizeof(WideAttn), st, static_cast<const uint16_t*>(q), q_rs,
                       static_cast<const uint8_t*>(pool), static_cast<const int*>(bt), bt_rs, static_cast<const int*>(cached),
                       kv_start, Hkv, G, NS, chunk, qscale, static_cast<const uint16_t*>(ring), static_cast<const int*>(tail_len),
                       static_cast<const int*>(tail_idx), T, static_cast<float*>(opart), static_cast<float*>(ml));
    if (hipPeekAtLastError() != hipSuccess) return 1;
  } else {
    const int rc = attn_pages256_launch(G, q, q_rs, pool, bt, bt_rs, cached, kv_start, B, Hkv, NS, chunk, qscale, ring, tail_len,
                                        tail_idx, T, opart, ml, f8, st);
    if (rc) return rc;
  }
  hipLaunchKernelGGL(k_merge_parts<D2>, dim3(B, Hkv * G), dim3(MERGE_SLICES * 64), 0, st, static_cast<const float*>(opart), static_cast<const float*>(ml),
                     Hkv, G, NS, static_cast<uint16_t*>(out), out_rs);
  return hipPeekAtLastError() == hipSuccess ? 0 : 1;
}

}  // namespace frkv
