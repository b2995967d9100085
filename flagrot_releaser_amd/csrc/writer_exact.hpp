// The selecting writer's choice for one (token, KV head), evaluated exactly by a workgroup of 2 D threads: every product
// and sum rounded on its own, in the order of kernels/codebook_ref.py:119-236 (include from -ffp-contract=off units only).
//   candidates   wavefront 0: as is, 1: H32 of every 32-group, 2: whole-head Hadamard, 3: the value row
//   local forms  one thread per (candidate, output channel): its chain of 32 products, the tree over the half wave
//   head forms   wavefront b: the block sums of input channels [32 b, 32 b + 32) for all output channels
//   fold         wavefront 0: base, 1: whole head: block sums in block order, then the halving tree
// C_q^T (64 KB per head, 256 KB for 256-d heads) is used once per token, so it does not go through LDS: every thread asks
// for its own 96 or 160 numbers at the start, all in flight together, while the candidates are formed.
#pragma once
#include "fr_launch.hpp"
#include "writer_rows.hpp"

namespace fr {

template <int D>
struct alignas(16) StepSmem {
  float err[3][D];                                 // error vectors of the candidates
  uint32_t code[4][64], word[4][64];               // per lane: four codes (a byte each), scale word; 3: the value row
  float local[2][D / 32];
  float block[D / 32][2][D];
  float head[2];
};

// The thread's numbers of C_q^T (CT[k][i] = C_q[i][k]): the column of its local block, its outputs' rows of the wavefront's
// block.  Loaded once for all tokens of the workgroup.
template <int D>
struct CqRegs {
  float cl[32], cf[32][D / 64];
  DEVI void load(const float* CT) {
    constexpr int O = D / 64;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, out = tid % D, g = out >> 5;
    const float* lcol = CT + static_cast<size_t>(32 * g) * D + out;
    const float* frow = CT + static_cast<size_t>(32 * wv) * D + O * lane;
#pragma unroll
    for (int k = 0; k < 32; ++k) cl[k] = lcol[k * D];
#pragma unroll
    for (int k = 0; k < 32; ++k) {
      if constexpr (O == 4) {
        const float4 c = *reinterpret_cast<const float4*>(frow + k * D);
        cf[k][0] = c.x; cf[k][1] = c.y; cf[k][2] = c.z; cf[k][3] = c.w;
      } else {
        const float2 c = *reinterpret_cast<const float2*>(frow + k * D);
        cf[k][0] = c.x; cf[k][1] = c.y;
      }
    }
  }
};

// One token whose slot is not negative, to its page.  FRESH: the numbers of C_q^T are asked for here, behind the rows and
// before the candidates, and the value codes are stored too (field by field).  Every thread of the workgroup calls it; the
// caller puts a barrier between two calls.
template <int QM, int P, int D, bool FRESH>
DEVI void k2_exact_token(const K2WriteParams& p, StepSmem<D>& S, CqRegs<D>& C, int h, int t, long long slot) {
  using L = Lay<QM, P>;
  constexpr int NB = D / 32, O = D / 64;           // column blocks = wavefronts; output channels per lane
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31;
  const bool do_k = p.passes & 1, do_v = p.passes & 2;
  const int half = D == 256 ? lane >> 5 : 0, d0 = 128 * half + 4 * l32;
  float x[4] = {0.f, 0.f, 0.f, 0.f};
  if (wv < 4) {
    load_row(p.kv, static_cast<long long>(t) * p.kv_ts + static_cast<long long>(wv == 3 ? p.Hkv + h : h) * D + d0, x);
    if (p.kmu != nullptr && wv < 3) {
      const float4 m = *reinterpret_cast<const float4*>(p.kmu + h * D + d0);
      x[0] = x[0] - m.x; x[1] = x[1] - m.y; x[2] = x[2] - m.z; x[3] = x[3] - m.w;
    }
  }
  const int cand = tid / D, out = tid % D, g = out >> 5;
  if (FRESH && do_k) C.load(p.CT + static_cast<size_t>(h) * D * D);
  __builtin_amdgcn_sched_barrier(0);               // all of them asked for before the candidates are formed
  uint8_t* chunk = p.pool + ((slot / P) * (p.Hkv * (D / 128)) + h * (D / 128) + half) * L::CHUNK;
  const int pos = static_cast<int>(slot % P);
  if ((wv < 3 && do_k) || (wv == 3 && do_v)) {
    float y[4] = {x[0], x[1], x[2], x[3]}, q[4], e[4];
    if (wv == 1) fwht<32>(y, l32);
    if (wv == 2) head_transform<D>(y, lane);
    S.word[wv][lane] = quant_group<QM, true>(y, q, e);
    uint32_t code[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) code[i] = code_bits(q[i], QM == QM_SYM4);
    if (wv < 3) {
      if (wv == 1) fwht<32>(e, l32);
      if (wv == 2) head_transform<D>(e, lane);
#pragma unroll
      for (int i = 0; i < 4; ++i) e[i] = e[i] - x[i];
      *reinterpret_cast<float4*>(&S.err[wv][d0]) = make_float4(e[0], e[1], e[2], e[3]);
      S.code[wv][lane] = code[0] | (code[1] << 8) | (code[2] << 16) | (code[3] << 24);
    } else if (FRESH && (D == 256 || lane < 32)) {
      store_v_codes<QM, P>(chunk, pos, code, l32);
    }
  }
  __syncthreads();
  bool key_full = false;
  if (do_k) {
    {
      float u;
#pragma unroll
      for (int k4 = 0; k4 < 8; ++k4) {
        const float4 e4 = *reinterpret_cast<const float4*>(&S.err[cand][32 * g + 4 * k4]);
        const float e[4] = {e4.x, e4.y, e4.z, e4.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float pr = C.cl[4 * k4 + i] * e[i];
          u = 4 * k4 + i == 0 ? pr : u + pr;
        }
      }
      const float form = tree32_lanes(S.err[cand][out] * u);
      if (l32 == 0) S.local[cand][g] = form;
    }
    __syncthreads();
    {
      const float* eb = S.err[S.local[1][wv] < S.local[0][wv] ? 1 : 0] + 32 * wv;     // strict: ties keep the identity
      const float* ef = S.err[2] + 32 * wv;
      float ub[O], uf[O];
#pragma unroll
      for (int k4 = 0; k4 < 8; ++k4) {
        const float4 b4 = *reinterpret_cast<const float4*>(eb + 4 * k4), f4 = *reinterpret_cast<const float4*>(ef + 4 * k4);
        const float b[4] = {b4.x, b4.y, b4.z, b4.w}, f[4] = {f4.x, f4.y, f4.z, f4.w};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int o = 0; o < O; ++o) {
            const float pb = C.cf[4 * k4 + i][o] * b[i], pf = C.cf[4 * k4 + i][o] * f[i];
            ub[o] = 4 * k4 + i == 0 ? pb : ub[o] + pb;
            uf[o] = 4 * k4 + i == 0 ? pf : uf[o] + pf;
          }
      }
#pragma unroll
      for (int o = 0; o < O; ++o) { S.block[wv][0][O * lane + o] = ub[o]; S.block[wv][1][O * lane + o] = uf[o]; }
    }
    __syncthreads();
    if (wv < 2) {
      float v[O];
#pragma unroll
      for (int m = 0; m < O; ++m) {
        const int i = lane + 64 * m;
        float s = S.block[0][wv][i];
#pragma unroll
        for (int b = 1; b < NB; ++b) s = s + S.block[b][wv][i];
        const int c = wv == 1 ? 2 : (S.local[1][i >> 5] < S.local[0][i >> 5] ? 1 : 0);
        v[m] = S.err[c][i] * s;
      }
      float r;                                     // the halving tree: channels 128 apart (D = 256), 64, 32, ..
      if constexpr (O == 4) r = (v[0] + v[2]) + (v[1] + v[3]);
      else r = v[0] + v[1];
      r = tree32_lanes(r + xor32(r));
      if (lane == 0) S.head[wv] = r;
    }
    __syncthreads();
    key_full = S.head[1] < S.head[0];
  }
  if (D == 128 && lane >= 32) return;
  const int kg = d0 >> 5;                          // the lane's 32-group
  if (wv == 0 && do_k) {
    const bool use_h = S.local[1][kg] < S.local[0][kg];
    const int c = key_full ? 2 : use_h ? 1 : 0;
    const uint32_t pack = S.code[c][lane];
    const uint32_t code[4] = {pack & 0xFFu, (pack >> 8) & 0xFFu, (pack >> 16) & 0xFFu, pack >> 24};
    store_row<QM, P>(chunk, pos, false, code, S.word[c][lane] | (c == 1 ? 0x8000u : 0u), l32, false);
    if (!do_v && lane == 0) {   // key-only pass: own bit 15 of the token's group-0 V scale word
      const int off = L::VS_OFF + (8 * (pos >> 3) + vs_slot8(pos)) * 2;
      uint32_t* wp = reinterpret_cast<uint32_t*>(chunk + (off & ~3));
      const uint32_t bit = 0x8000u << ((off & 2) * 8);
      if (key_full) atomicOr(wp, bit); else atomicAnd(wp, ~bit);
    }
  }
  if (wv == 1 && do_v)
    store_v_word<QM, P>(chunk, pos, S.word[3][lane] | (kg == 0 && key_full ? 0x8000u : 0u), l32, !do_k);
}

}  // namespace fr
