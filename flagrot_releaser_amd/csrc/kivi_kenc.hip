// Key group encoder of the KIVI-style pages at head dim 128 (NH = 1) and 256 (NH = 2): one workgroup of eight wavefronts
// per (32-token group, KV head).  Page layouts: kivi_write.hip (128) and kivi_wide.hip (256).  Compiled with
// -ffp-contract=off: the quantiser rounds every operation on its own (integrations/vllm_flagrot/csrc/kivi.cu:94-128); the
// decision rule is kivi.cu:344-663 (sums in fp32, order free: H32 where its error is strictly smaller, whole head where
// it is strictly smaller than the combination of the sub-vector picks).
//
// What bounds it: vector issue (some 1350 instructions a wavefront: ranges, codes, transforms) and the projections of the
// group's 32 rows and of their three candidates' errors on the NQ calibration queries, 4 x 32 x NQ x D multiply-adds, one
// after the other: FP32 matrix instructions and vector instructions do not run beside each other on a SIMD (two
// workgroups on a CU: 45 k cycles, one 29 k, of which 8 k matrix).  The products run on the matrix pipe in fp32
// (v_mfma_f32_16x16x4_f32: tokens x queries, no precision given up).  A wavefront takes 16 tokens x 16 of 64 queries of ALL
// four matrices -- errors as stored, H32, whole head, and the rows themselves -- with one accumulator per sub-vector, so
// the weights, the costs and the combination of the picks of a (token, query) pair are in one lane and nothing but the
// wavefronts' sums goes through LDS.  More than 64 queries: the products are formed again once the choices are known.  The
// queries are read straight from L2 (a lane's 16 bytes are four k-steps of one query).
//
// Prompt of 4133 tokens x 8 heads, FP8 meta / 16 groups x 8 heads / 256-d heads, 9 groups x 4 (us): a wavefront per (matrix, 32
// queries) with weights and shares exchanged through LDS and IEEE quotients 62.3 / 15.7 / 26.6; this form 46.5 / 11.4 / 20.8.
#include <type_traits>

#include "fr_common.hpp"
#include "kivi_launch.hpp"
#include "kivi_quant.hpp"

namespace frkv {
using namespace fr;
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <int NH, bool F8> struct KPage {                  // where a chunk keeps what
  static constexpr int D = 128 * NH, NV = 4 * NH;
  static constexpr long long CHUNK = F8 ? 10 * D : 12 * D + 16;
  static constexpr int KM = 4 * D;
};

constexpr int QCHUNK = 64;                                 // queries per pass of the workgroup
template <int NH> struct KEnc {
  static constexpr int D = 128 * NH, NV = 4 * NH, LD = D + 4;   // padded rows: 16 rows of a 128-bit read hit 64 banks
  static constexpr int SUMS = 2 * NV + 1;                  // as stored [NV] | H32 [NV] | whole head
  float mat[4][32][LD];                                    // errors as stored | H32 | whole head | the rows
  float par[3][3][D];                                      // per candidate (min, scale, 1 / scale) per channel
  float red[8][SUMS], base[8];                             // per wavefront
  int odd;                                                 // a scale outside the range where its reciprocal decides
  long long slot[32];                                      // page slots of the tokens
};
// the ranges of the eight wavefronts ([8][3][2][D]) lie where the errors go afterwards
static_assert(8 * 3 * 2 * 128 <= 3 * 32 * KEnc<1>::LD && 8 * 3 * 2 * 256 <= 3 * 32 * KEnc<2>::LD, "ranges fit the error rows");

template <int NH, int C> DEVI void rebase(float (&y)[NH][4], int l32) {   // 0 as stored, 1 H32, 2 whole head (involutions)
  if constexpr (C == 1) {
#pragma unroll
    for (int s = 0; s < NH; ++s) fwht<32>(y[s], l32);
  }
  if constexpr (C == 2) {
    if constexpr (NH == 1) fwht<128>(y[0], l32);
    else h256(y, l32);
  }
}
// lanes 0 .. 31: op(a, a of the lane 32 on), lanes 32 .. 63: the same of b
template <class F> DEVI float fold32(float a, float b, F op) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_int(a), __float_as_int(b), false, false);
  return op(__int_as_float(r[0]), __int_as_float(r[1]));
}
// rows of 16 lanes: even rows get a summed over the pair of rows, odd rows b
DEVI float fold16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_int(a), __float_as_int(b), false, false);
  return __int_as_float(r[0]) + __int_as_float(r[1]);
}
DEVI float row_sum(float v) {                              // over the lane's row of 16
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xF, 0xF, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xF, 0xF, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x122, 0xF, 0xF, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x121, 0xF, 0xF, true));
  return v;
}

template <int NH, bool F8>
__global__ void __launch_bounds__(512, NH == 1 ? 4 : 2)
k_k_encode(const uint16_t* __restrict__ src, long long src_rs, const uint16_t* __restrict__ src2, long long src2_rs,
           const long long* __restrict__ sidx, const long long* __restrict__ dslot, int Hkv, const float* __restrict__ qs,
           const float* __restrict__ lz, int NQ, float qsc, uint8_t* __restrict__ pool, int ident,
           const int* __restrict__ kfix) {
  using S = KEnc<NH>;
  using PG = KPage<NH, F8>;
  constexpr int D = S::D, NV = S::NV, TOK = 2;             // tokens per half wave
  extern __shared__ __align__(16) uint8_t lds[];
  S& L = *reinterpret_cast<S*>(lds);
  const int item = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, wv = tid >> 6, lane = tid & 63, l32 = tid & 31, hw = tid >> 5;
  const long long* si = sidx + static_cast<long long>(item) * 32;
  const long long* ds = dslot + static_cast<long long>(item) * 32;
  if (ds[0] < 0) return;
  const uint32_t valid = static_cast<uint32_t>(__ballot(si[l32] != -1));       // bit t: token t belongs to the group
  if (tid == 0) L.odd = 0;
  if (tid < 32) L.slot[tid] = ds[tid];
  // ---- rows and candidates: half wave hw owns tokens 2 hw, 2 hw + 1; lane l channels 128 s + 4 l + i
  float x[TOK][NH][4], y1[TOK][NH][4], y2[TOK][NH][4];
#pragma unroll
  for (int k = 0; k < TOK; ++k) {
    const long long r = si[TOK * hw + k];
    const uint16_t* row = r >= 0 ? src + r * src_rs : r <= -2 ? src2 + (-r - 2) * src2_rs : nullptr;
#pragma unroll
    for (int s = 0; s < NH; ++s) {
      uint32_t w[2] = {0u, 0u};
      if (row != nullptr) {                                // two bytes at a time: rows may start anywhere
        const uint16_t* at = row + static_cast<long long>(h) * D + 128 * s + 4 * l32;
        w[0] = at[0] | (static_cast<uint32_t>(at[1]) << 16);
        w[1] = at[2] | (static_cast<uint32_t>(at[3]) << 16);
      }
      x[k][s][0] = bf16_lo(w[0]); x[k][s][1] = bf16_hi(w[0]); x[k][s][2] = bf16_lo(w[1]); x[k][s][3] = bf16_hi(w[1]);
    }
#pragma unroll
    for (int s = 0; s < NH; ++s) {
#pragma unroll
      for (int i = 0; i < 4; ++i) { y1[k][s][i] = x[k][s][i]; y2[k][s][i] = x[k][s][i]; }
      *reinterpret_cast<float4*>(&L.mat[3][TOK * hw + k][128 * s + 4 * l32]) = make_float4(x[k][s][0], x[k][s][1], x[k][s][2], x[k][s][3]);
    }
    rebase<NH, 1>(y1[k], l32);
    rebase<NH, 2>(y2[k], l32);
  }
  // ---- ranges over the valid tokens: per wavefront (lanes 0 .. 31 minima, 32 .. 63 negated maxima), then one thread per
  // (candidate, channel)
  float* range = &L.mat[0][0][0];
  {
    const bool in[TOK] = {((valid >> (TOK * hw)) & 1u) != 0, ((valid >> (TOK * hw + 1)) & 1u) != 0};
    const bool full = valid == ~0u;
    auto put = [&](int c, const float (&y)[TOK][NH][4]) {
#pragma unroll
      for (int s = 0; s < NH; ++s) {
        float lo[4], hi[4], m[4];
        if (full) {
#pragma unroll
          for (int i = 0; i < 4; ++i) { lo[i] = fminf(y[0][s][i], y[1][s][i]); hi[i] = fminf(-y[0][s][i], -y[1][s][i]); }
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            lo[i] = fminf(in[0] ? y[0][s][i] : INFINITY, in[1] ? y[1][s][i] : INFINITY);
            hi[i] = fminf(in[0] ? -y[0][s][i] : INFINITY, in[1] ? -y[1][s][i] : INFINITY);
          }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) m[i] = fold32(lo[i], hi[i], [](float a, float b) { return fminf(a, b); });
        *reinterpret_cast<float4*>(range + ((wv * 3 + c) * 2 + (lane >> 5)) * D + 128 * s + 4 * l32) = make_float4(m[0], m[1], m[2], m[3]);
      }
    };
    put(0, x);
    put(1, y1);
    put(2, y2);
  }
  __syncthreads();
  for (int e = tid; e < 3 * D; e += 512) {
    const int c = e / D, ch = e % D;
    float mn = INFINITY, mx = INFINITY;
#pragma unroll
    for (int w = 0; w < 8; ++w) {
      mn = fminf(mn, range[((w * 3 + c) * 2) * D + ch]);
      mx = fminf(mx, range[((w * 3 + c) * 2 + 1) * D + ch]);
    }
    float s = kv_scale(mn, -mx);
    kv_params<F8>(mn, s);
    const float d = s == 0.f ? 1.f : s;
    if (!(d > 1e-30f && d < 1e30f)) L.odd = 1;
    L.par[c][0][ch] = mn;
    L.par[c][1][ch] = s;
    L.par[c][2][ch] = __builtin_amdgcn_rcpf(d);
  }
  __syncthreads();
  // ---- codes of all three candidates (two bits each) and, for a choice, their errors in the original basis
  const bool choose = !ident && kfix == nullptr && NQ > 0, odd = L.odd != 0;
  uint32_t codes[3][TOK];                                  // per token: channel (s, i) at bit 8 s + 2 i
  auto encode = [&](auto cand, float (&y)[TOK][NH][4]) {
    constexpr int C = decltype(cand)::value;
#pragma unroll
    for (int k = 0; k < TOK; ++k) {
      uint32_t bits = 0;
#pragma unroll
      for (int s = 0; s < NH; ++s) {
        const float4 mn4 = *reinterpret_cast<const float4*>(&L.par[C][0][128 * s + 4 * l32]);
        const float4 sc4 = *reinterpret_cast<const float4*>(&L.par[C][1][128 * s + 4 * l32]);
        const float4 rc4 = *reinterpret_cast<const float4*>(&L.par[C][2][128 * s + 4 * l32]);
        const float mn[4] = {mn4.x, mn4.y, mn4.z, mn4.w}, sc[4] = {sc4.x, sc4.y, sc4.z, sc4.w}, rc[4] = {rc4.x, rc4.y, rc4.z, rc4.w};
        // the rounding of (y - min) x reciprocal is that of the IEEE quotient unless it lies near a half (kv_codes)
        float n[4], worst = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float q = fminf(fmaxf((y[k][s][i] - mn[i]) * rc[i], 0.f), 3.f);
          n[i] = rintf(q);
          worst = fmaxf(worst, fabsf(q - n[i]));
        }
        if (!(worst < KV_SURE) || odd) {
#pragma unroll
          for (int i = 0; i < 4; ++i) n[i] = static_cast<float>(kv_code(y[k][s][i], mn[i], sc[i]));
        }
        bits |= static_cast<uint32_t>(static_cast<int>(n[0] + 4.f * n[1] + (16.f * n[2] + 64.f * n[3]))) << (8 * s);
#pragma unroll
        for (int i = 0; i < 4; ++i) y[k][s][i] = n[i] * sc[i] + mn[i];
      }
      codes[C][k] = bits;
      __builtin_amdgcn_sched_barrier(0);
      if (choose) {
        rebase<NH, C>(y[k], l32);
#pragma unroll
        for (int s = 0; s < NH; ++s)
          *reinterpret_cast<float4*>(&L.mat[C][TOK * hw + k][128 * s + 4 * l32]) =
              make_float4(y[k][s][0] - x[k][s][0], y[k][s][1] - x[k][s][1], y[k][s][2] - x[k][s][2], y[k][s][3] - x[k][s][3]);
      }
    }
  };
  {
    float y0[TOK][NH][4];
#pragma unroll
    for (int k = 0; k < TOK; ++k)
#pragma unroll
      for (int s = 0; s < NH; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i) y0[k][s][i] = x[k][s][i];
    encode(std::integral_constant<int, 0>{}, y0);
    encode(std::integral_constant<int, 1>{}, y1);
    encode(std::integral_constant<int, 2>{}, y2);
  }
  if (choose && valid != ~0u) {                            // tokens outside the group count nothing
#pragma unroll
    for (int k = 0; k < TOK; ++k)
      if (!((valid >> (TOK * hw + k)) & 1u))
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int s = 0; s < NH; ++s)
            *reinterpret_cast<float4*>(&L.mat[c][TOK * hw + k][128 * s + 4 * l32]) = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  uint32_t pick = 0;                                       // bit j: sub-vector j is H32
  bool whole = false;
  if (!ident && kfix != nullptr) {
    pick = static_cast<uint32_t>(kfix[h]) & ((1u << NV) - 1u);
    whole = (kfix[h] >> 16) & 1;
  }
  if (choose) {
    const int l16 = lane & 15, quad = lane >> 4, tok0 = 16 * (wv & 1), query0 = 16 * (wv >> 1);
    const float* qh = qs + static_cast<long long>(h) * NQ * D;
    const float* mrow = &L.mat[0][tok0 + l16][4 * quad];
    float cost[2 * NV + 1], base = 0.f;                    // as stored [NV] | H32 [NV] | whole head
#pragma unroll
    for (int j = 0; j <= 2 * NV; ++j) cost[j] = 0.f;
    // up to 64 queries: one round does it all; else the rounds of the choices, then those of the combination
    const int chunks = (NQ + QCHUNK - 1) / QCHUNK, rounds = chunks == 1 ? 1 : 2 * chunks;
    for (int rd = 0; rd < rounds; ++rd) {
      const int query = (rd % chunks) * QCHUNK + query0 + l16;
      const bool live = query < NQ;
      const float* qrow = qh + static_cast<long long>(min(query, NQ - 1)) * D + 4 * quad;
      const float lzq = lz[static_cast<long long>(h) * NQ + min(query, NQ - 1)];
      float4 qf[2];                                        // one k-step in use, one on its way
      qf[0] = *reinterpret_cast<const float4*>(qrow);
      __builtin_amdgcn_sched_barrier(0);
      if (rd == 0) __syncthreads();                        // the matrices
      // products of the wavefront's 16 tokens and 16 queries; k-step (s, i): channel 16 s + 4 quad + i
      f32x4 acc[2 * NV], accw = {0.f, 0.f, 0.f, 0.f}, accx = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 2 * NV; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 2 * NV; ++s) {
        if (s + 1 < 2 * NV) qf[(s + 1) & 1] = *reinterpret_cast<const float4*>(qrow + 16 * (s + 1));
        float4 a[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) a[m] = *reinterpret_cast<const float4*>(mrow + m * 32 * S::LD + 16 * s);
        const float4 bq = qf[s & 1];
        const float b[4] = {bq.x, bq.y, bq.z, bq.w};
        const float am[4][4] = {{a[0].x, a[0].y, a[0].z, a[0].w}, {a[1].x, a[1].y, a[1].z, a[1].w},
                                {a[2].x, a[2].y, a[2].z, a[2].w}, {a[3].x, a[3].y, a[3].z, a[3].w}};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          acc[s >> 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(am[0][i], b[i], acc[s >> 1], 0, 0, 0);
          acc[NV + (s >> 1)] = __builtin_amdgcn_mfma_f32_16x16x4f32(am[1][i], b[i], acc[NV + (s >> 1)], 0, 0, 0);
          accw = __builtin_amdgcn_mfma_f32_16x16x4f32(am[2][i], b[i], accw, 0, 0, 0);
          accx = __builtin_amdgcn_mfma_f32_16x16x4f32(am[3][i], b[i], accx, 0, 0, 0);
        }
      }
      // accumulator r of a lane: token tok0 + 4 quad + r, the lane's query; all products of the pair are in this lane
      float w[4];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        w[r] = live && ((valid >> (tok0 + 4 * quad + r)) & 1u) ? fminf(expf(qsc * accx[r] - lzq), 1.f) : 0.f;
      if (rd < chunks) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
#pragma unroll
          for (int j = 0; j < 2 * NV; ++j) cost[j] = fmaf(w[r] * acc[j][r], acc[j][r], cost[j]);
          cost[2 * NV] = fmaf(w[r] * accw[r], accw[r], cost[2 * NV]);
        }
      }
      if (rd == chunks - 1) {                              // the sub-vector choices: as stored on ties
        // sums over the wavefront: sums of pairs of lanes halve the number of registers twice (row t of 16 lanes keeps
        // sum 4 v + 2 (t & 1) + (t >> 1)), then within the rows
        constexpr int N = 2 * NV + 1;
        auto plus = [](float a, float b) { return a + b; };
#pragma unroll
        for (int v = 0; v < (N + 3) / 4; ++v) {
          const float lo = fold32(cost[4 * v], 4 * v + 1 < N ? cost[4 * v + 1] : 0.f, plus);
          const float hi = 4 * v + 2 < N ? fold32(cost[4 * v + 2], cost[4 * v + 3], plus) : 0.f;
          const float sum = row_sum(fold16(lo, hi));
          const int at = 4 * v + 2 * (quad & 1) + (quad >> 1);
          if (l16 == 0 && at < N) L.red[wv][at] = sum;
        }
        __syncthreads();
        float mine = 0.f, other = 0.f;                     // lane j: sub-vector j as stored and H32
        const int j = l32 & (NV - 1);
#pragma unroll
        for (int i = 0; i < 8; ++i) { mine += L.red[i][j]; other += L.red[i][NV + j]; }
        pick = static_cast<uint32_t>(__ballot(other < mine)) & ((1u << NV) - 1u);
      }
      if (rounds == 1 || rd >= chunks) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float p = 0.f;
#pragma unroll
          for (int j = 0; j < NV; ++j) p += (pick >> j) & 1u ? acc[NV + j][r] : acc[j][r];
          base = fmaf(w[r] * p, p, base);
        }
      }
    }
    base = row_sum(fold16(fold32(base, base, [](float a, float b) { return a + b; }), 0.f));
    if (lane == 0) L.base[wv] = base;
    __syncthreads();
    float all = 0.f, mixed = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) { all += L.red[i][2 * NV]; mixed += L.base[i]; }
    whole = all < mixed;                                   // the combination on ties
  }
  // ---- codes of the valid tokens in the chosen bases
#pragma unroll
  for (int k = 0; k < TOK; ++k) {
    const int t = TOK * hw + k;
    if (!((valid >> t) & 1u)) continue;
    const long long slot = L.slot[t];
    uint8_t* chunk = pool + ((slot / 16) * Hkv + h) * PG::CHUNK;
#pragma unroll
    for (int s = 0; s < NH; ++s) {
      // (masks: a choice between array elements would put the array into scratch memory)
      const uint32_t rot = 0u - ((pick >> (4 * s + (l32 >> 3))) & 1u), all = whole ? ~0u : 0u;
      const uint32_t four = ((codes[2][k] & all) | (~all & ((codes[1][k] & rot) | (codes[0][k] & ~rot)))) >> (8 * s);
      uint32_t word = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int ci = (4 * l32 + i) & 15;
        word |= ((four >> (2 * i)) & 3u) << (2 * (ci >> 1) + 16 * (ci & 1));
      }
      word |= __shfl_xor(word, 1, 32);
      word |= __shfl_xor(word, 2, 32);
      if ((l32 & 3) == 0) reinterpret_cast<uint32_t*>(chunk + (slot % 16) * (D / 4))[8 * s + (l32 >> 2)] = word;
    }
  }
  // ---- meta of all 32 cells: cell i holds channels [NV i, NV i + NV)
  if (tid < D) {
    const int c = tid, cell = c / NV, at_slot = c % NV;
    const int cand = whole ? 2 : (pick >> (c >> 5)) & 1u;
    const long long slot = L.slot[cell];
    if (slot >= 0) {
      uint8_t* chunk = pool + ((slot / 16) * Hkv + h) * PG::CHUNK + PG::KM;
      const float mn = L.par[cand][0][c], sc = L.par[cand][1][c];
      if (F8) {                                            // flags at slot 0 of cells 0 .. NV
        const bool neg = at_slot == 0 && (cell < NV ? (!whole && ((pick >> cell) & 1u)) : (cell == NV && whole));
        uint8_t* at = chunk + (slot % 16) * (2 * NV) + 2 * at_slot;
        uint32_t sb = e4m3_bits(sc) | (neg ? 0x80u : 0u);
        if (at_slot == NV - 1) sb |= at[0] & 0x80u;        // the value row's whole-head flag lives here
        *reinterpret_cast<uint16_t*>(at) = static_cast<uint16_t>(sb | (e4m3_bits(mn) << 8));
      } else {                                             // flags at channels 0 .. NV
        const bool neg = c < NV ? (!whole && ((pick >> c) & 1u)) : (c == NV && whole);
        const uint32_t sb = (f16_bits_rn(sc) & 0x7FFFu) | (neg ? 0x8000u : 0u);
        reinterpret_cast<uint32_t*>(chunk + (slot % 16) * (4 * NV))[at_slot] = sb | (f16_bits_rn(mn) << 16);
      }
    }
  }
}

template <int NH, bool F8> int launch(const void* src, long long src_rs, const void* src2, long long src2_rs, const long long* sidx,
                                      const long long* dslot, int N, int Hkv, const float* qs, const float* lz, int NQ,
                                      float qsc, uint8_t* pool, int ident, const int* kfix, hipStream_t st) {
  const auto kern = &k_k_encode<NH, F8>;
  static const hipError_t set = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                    static_cast<int>(sizeof(KEnc<NH>)));
  if (set != hipSuccess) return 1;
  hipLaunchKernelGGL(kern, dim3(N, Hkv), dim3(512), sizeof(KEnc<NH>), st, static_cast<const uint16_t*>(src), src_rs,
                     static_cast<const uint16_t*>(src2), src2_rs, sidx, dslot, Hkv, qs, lz, NQ, qsc, pool, ident, kfix);
  return hipPeekAtLastError() == hipSuccess ? 0 : 1;
}

}  // namespace

int k_encode_launch(int D, const void* src, long long src_rs, const void* src2, long long src2_rs, const long long* sidx,
                    const long long* dslot, int N, int Hkv, const float* qs, const float* lz, int NQ, float qsc,
                    uint8_t* pool, int ident, const int* kfix, int f8, hipStream_t st) {
  const auto go = D == 256 ? (f8 ? &launch<2, true> : &launch<2, false>) : (f8 ? &launch<1, true> : &launch<1, false>);
  return go(src, src_rs, src2, src2_rs, sidx, dslot, N, Hkv, qs, lz, NQ, qsc, pool, ident, kfix, st);
}

}  // namespace frkv
