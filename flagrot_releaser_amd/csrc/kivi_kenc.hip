// Key group encoder of the KIVI-style pages at head dim 128 (NH = 1) and 256 (NH = 2): one workgroup of eight wavefronts
// per (32-token group, KV head).  Page layouts: kivi_write.hip (128) and kivi_wide.hip (256).  Compiled with
// -ffp-contract=off: the quantiser rounds every operation on its own (integrations/vllm_flagrot/csrc/kivi.cu:94-128); the
// decision rule is kivi.cu:344-663 (sums in fp32, order free: H32 where its error is strictly smaller, whole head where
// it is strictly smaller than the combination of the sub-vector picks).
//
// What bounds it: the projections of the group's 32 rows and of their three candidates' errors on the NQ calibration
// queries, 4 x 32 x NQ x D multiply-adds, and for the single group that a decode step completes the chain of phases.
// They run on the matrix pipe in fp32 (v_mfma_f32_32x32x2_f32: tokens x queries, no precision given up): wavefront
// (role, tile) multiplies one of the four matrices -- errors as stored, H32, whole head, and the rows themselves -- with
// 32 of 64 queries, keeping one accumulator per sub-vector, so that both the sub-vector choices and their combination
// come out of ONE product; the weights and the H32 share of the combination change wavefronts through LDS.  More than 64
// queries: the products are formed again once the choices are known.  The queries are read straight from L2 (a lane's
// 16 bytes are four k-steps of one query).
//
// The vector form before it (a thread per (token, query), operands from LDS, every product twice): a prompt of 4133
// tokens x 8 heads 257 us, one group per head 81 us; this form 63 and 17 us.
#include <type_traits>

#include "fr_common.hpp"
#include "kivi_launch.hpp"
#include "kivi_quant.hpp"

namespace frkv {
using namespace fr;
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

template <int NH, bool F8> struct KPage {                  // where a chunk keeps what
  static constexpr int D = 128 * NH, NV = 4 * NH;
  static constexpr long long CHUNK = F8 ? 10 * D : 12 * D + 16;
  static constexpr int KM = 4 * D;
};

constexpr int QTILE = 32, QCHUNK = 64;                     // queries per wavefront tile, per pass of the workgroup
template <int NH> struct KEnc {
  static constexpr int D = 128 * NH, NV = 4 * NH, LD = D + 4;   // padded rows: 16 rows of a 128-bit read hit 64 banks
  float mat[4][32][LD];                                    // errors as stored | H32 | whole head | the rows
  float par[3][2][D];                                      // per candidate (min, scale) per channel
  float swap[2][16][64];                                   // per query tile: weights, later H32's share of the combination
  float red[2][2 * NV + 2];                                // per query tile: as stored [NV] | H32 [NV] | whole | base
  float lz[QCHUNK];
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
DEVI float wave_sum(float v) {
#pragma unroll
  for (int m = 1; m < 32; m <<= 1) v += hx(v, m);
  return v + xor32(v);
}

template <int NH, bool F8>
__global__ void __launch_bounds__(512, NH == 1 ? 4 : 2)
k_k_encode(const uint16_t* __restrict__ src, long long src_rs, const uint16_t* __restrict__ src2, long long src2_rs,
           const long long* __restrict__ sidx, const long long* __restrict__ dslot, int Hkv, const float* __restrict__ qs,
           const float* __restrict__ lz, int NQ, float qsc, uint8_t* __restrict__ pool, int ident,
           const int* __restrict__ kfix) {
  using S = KEnc<NH>;
  using PG = KPage<NH, F8>;
  constexpr int D = S::D, NV = S::NV, LD = S::LD, TOK = 2;  // tokens per half wave
  extern __shared__ __align__(16) uint8_t lds[];
  S& L = *reinterpret_cast<S*>(lds);
  const int item = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, wv = tid >> 6, lane = tid & 63, l32 = tid & 31, hw = tid >> 5;
  const long long* si = sidx + static_cast<long long>(item) * 32;
  const long long* ds = dslot + static_cast<long long>(item) * 32;
  if (ds[0] < 0) return;
  const uint32_t valid = static_cast<uint32_t>(__ballot(si[l32] != -1));       // bit t: token t belongs to the group
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
  // ---- ranges over the valid tokens: per half wave, per wavefront, then one thread per (candidate, channel)
  float* range = &L.mat[0][0][0];
  {
    auto put = [&](int c, const float (&y)[TOK][NH][4]) {
#pragma unroll
      for (int s = 0; s < NH; ++s) {
        float lo[4], hi[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          lo[i] = INFINITY; hi[i] = -INFINITY;
#pragma unroll
          for (int k = 0; k < TOK; ++k)
            if ((valid >> (TOK * hw + k)) & 1u) { lo[i] = fminf(lo[i], y[k][s][i]); hi[i] = fmaxf(hi[i], y[k][s][i]); }
          lo[i] = fminf(lo[i], xor32(lo[i]));
          hi[i] = fmaxf(hi[i], xor32(hi[i]));
        }
        if (lane < 32) {
          float* at = range + ((wv * 3 + c) * 2) * D + 128 * s + 4 * l32;
          *reinterpret_cast<float4*>(at) = make_float4(lo[0], lo[1], lo[2], lo[3]);
          *reinterpret_cast<float4*>(at + D) = make_float4(hi[0], hi[1], hi[2], hi[3]);
        }
      }
    };
    put(0, x);
    put(1, y1);
    put(2, y2);
  }
  __syncthreads();
  for (int e = tid; e < 3 * D; e += 512) {
    const int c = e / D, ch = e % D;
    float mn = INFINITY, mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < 8; ++w) {
      mn = fminf(mn, range[((w * 3 + c) * 2) * D + ch]);
      mx = fmaxf(mx, range[((w * 3 + c) * 2 + 1) * D + ch]);
    }
    float s = kv_scale(mn, mx);
    kv_params<F8>(mn, s);
    L.par[c][0][ch] = mn;
    L.par[c][1][ch] = s;
  }
  __syncthreads();
  // ---- codes of all three candidates (two bits each) and, for a choice, their errors in the original basis
  const bool choose = !ident && kfix == nullptr && NQ > 0;
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
        const float mn[4] = {mn4.x, mn4.y, mn4.z, mn4.w}, sc[4] = {sc4.x, sc4.y, sc4.z, sc4.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int code = kv_code(y[k][s][i], mn[i], sc[i]);
          bits |= static_cast<uint32_t>(code & 3) << (8 * s + 2 * i);
          y[k][s][i] = kv_rec(code, mn[i], sc[i]);
        }
      }
      codes[C][k] = bits;
      __builtin_amdgcn_sched_barrier(0);
      if (choose) {
        rebase<NH, C>(y[k], l32);
        const bool v = (valid >> (TOK * hw + k)) & 1u;     // tokens outside the group count nothing
#pragma unroll
        for (int s = 0; s < NH; ++s)
          *reinterpret_cast<float4*>(&L.mat[C][TOK * hw + k][128 * s + 4 * l32]) =
              make_float4(v ? y[k][s][0] - x[k][s][0] : 0.f, v ? y[k][s][1] - x[k][s][1] : 0.f,
                          v ? y[k][s][2] - x[k][s][2] : 0.f, v ? y[k][s][3] - x[k][s][3] : 0.f);
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
  uint32_t pick = 0;                                       // bit j: sub-vector j is H32
  bool whole = false;
  if (!ident && kfix != nullptr) {
    pick = static_cast<uint32_t>(kfix[h]) & ((1u << NV) - 1u);
    whole = (kfix[h] >> 16) & 1;
  }
  if (choose) {
    const int role = wv >> 1, tile = wv & 1, half = lane >> 5;
    const float* qh = qs + static_cast<long long>(h) * NQ * D;
    const float* mrow = &L.mat[role][l32][4 * half];
    float cost[NV];                                        // roles 0, 1: per sub-vector; role 2: [0] = whole head
    float base = 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j) cost[j] = 0.f;
    // up to 64 queries: one round does it all; else the rounds of the choices, then those of the combination
    const int chunks = (NQ + QCHUNK - 1) / QCHUNK, rounds = chunks == 1 ? 1 : 2 * chunks;
    for (int rd = 0; rd < rounds; ++rd) {
      const int q0 = (rd % chunks) * QCHUNK;
      if (tid < QCHUNK) L.lz[tid] = q0 + tid < NQ ? lz[static_cast<long long>(h) * NQ + q0 + tid] : 0.f;
      __syncthreads();                                     // the matrices (first round); swap is free again
      // projections per sub-vector; k-step (j, s): channels 32 j + 8 s + 4 half + i of the lane's row and query
      f32x16 acc[NV];
      const float* qrow = qh + static_cast<long long>(min(q0 + QTILE * tile + l32, NQ - 1)) * D + 4 * half;
      float4 qf[2][2];                                     // two k-steps in use, two on their way
#pragma unroll
      for (int s = 0; s < 2; ++s) qf[0][s] = *reinterpret_cast<const float4*>(qrow + 8 * s);
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        f32x16 a = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          if (2 * j + p + 1 < 2 * NV) {
#pragma unroll
            for (int s = 0; s < 2; ++s) qf[p ^ 1][s] = *reinterpret_cast<const float4*>(qrow + 32 * j + 16 * (p + 1) + 8 * s);
          }
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            const float4 af = *reinterpret_cast<const float4*>(mrow + 32 * j + 16 * p + 8 * s);
            const float4 bf = qf[p][s];
            a = __builtin_amdgcn_mfma_f32_32x32x2f32(af.x, bf.x, a, 0, 0, 0);
            a = __builtin_amdgcn_mfma_f32_32x32x2f32(af.y, bf.y, a, 0, 0, 0);
            a = __builtin_amdgcn_mfma_f32_32x32x2f32(af.z, bf.z, a, 0, 0, 0);
            a = __builtin_amdgcn_mfma_f32_32x32x2f32(af.w, bf.w, a, 0, 0, 0);
          }
          __builtin_amdgcn_sched_barrier(0);               // (all requests at once would not fit the registers)
        }
        acc[j] = a;
      }
      // the rows' wavefronts turn their logits into weights (accumulator r of a lane: token (r & 3) + 8 (r >> 2) +
      // 4 half, query l32 of the tile); every wavefront of the tile takes them
      if (role == 3) {
        const float lzq = L.lz[QTILE * tile + l32];
        const bool live = q0 + QTILE * tile + l32 < NQ;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          float lg = 0.f;
#pragma unroll
          for (int j = 0; j < NV; ++j) lg += acc[j][r];
          const int t = (r & 3) + 8 * (r >> 2) + 4 * half;
          L.swap[tile][r][lane] = live && ((valid >> t) & 1u) ? fminf(expf(qsc * lg - lzq), 1.f) : 0.f;
        }
      }
      __syncthreads();
      float w[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) w[r] = L.swap[tile][r][lane];
      if (rd < chunks) {
        if (role < 2) {
#pragma unroll
          for (int j = 0; j < NV; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) cost[j] += w[r] * acc[j][r] * acc[j][r];
        } else if (role == 2) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            float p = 0.f;
#pragma unroll
            for (int j = 0; j < NV; ++j) p += acc[j][r];
            cost[0] += w[r] * p * p;
          }
        }
      }
      if (rd == chunks - 1) {                              // the sub-vector choices: as stored on ties
#pragma unroll
        for (int j = 0; j < NV; ++j) cost[j] = wave_sum(cost[j]);
        if (lane == 0) {
          if (role < 2)
#pragma unroll
            for (int j = 0; j < NV; ++j) L.red[tile][NV * role + j] = cost[j];
          if (role == 2) L.red[tile][2 * NV] = cost[0];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < NV; ++j)
          if (L.red[0][NV + j] + L.red[1][NV + j] < L.red[0][j] + L.red[1][j]) pick |= 1u << j;
      }
      __syncthreads();                                     // every wavefront has its weights
      if (rounds == 1 || rd >= chunks) {                   // H32's share of the combination to the wavefront of the rest
        if (role == 1)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            float p = 0.f;
#pragma unroll
            for (int j = 0; j < NV; ++j) p += (pick >> j) & 1u ? acc[j][r] : 0.f;
            L.swap[tile][r][lane] = p;
          }
        __syncthreads();
        if (role == 0)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            float p = L.swap[tile][r][lane];
#pragma unroll
            for (int j = 0; j < NV; ++j) p += (pick >> j) & 1u ? 0.f : acc[j][r];
            base += w[r] * p * p;
          }
      }
    }
    if (role == 0) {
      base = wave_sum(base);
      if (lane == 0) L.red[tile][2 * NV + 1] = base;
    }
    __syncthreads();
    whole = L.red[0][2 * NV] + L.red[1][2 * NV] < L.red[0][2 * NV + 1] + L.red[1][2 * NV + 1];   // base on ties
  }
  // ---- codes of the valid tokens in the chosen bases
#pragma unroll
  for (int k = 0; k < TOK; ++k) {
    const int t = TOK * hw + k;
    if (!((valid >> t) & 1u)) continue;
    const long long slot = ds[t];
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
    const long long slot = ds[cell];
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
