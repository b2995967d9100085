// Selecting writer of a prompt: the same bytes as the exact evaluation (writer_exact.hpp) at a fraction of its vector
// instructions.  The quadratic forms d^T C d of the candidates' error vectors are ESTIMATED on the matrix pipe, and a
// choice is taken from the estimates only where it cannot differ from the choice of the exactly ordered FP32 evaluation;
// every other token is evaluated exactly at the end of its workgroup.
//
// Estimate: C and d are split into two BF16 terms each (C = H + L + R, d = h + l + r with |L| <= 2^-8 |C|,
// |R| <= 2^-16 |C|, the same for d); L l + H l + L h and then H h accumulate in FP32, the outer product takes h + l (exact
// in FP32).  A fifth product gives S~ = |h|^T |H| |h|.  With S = |d|^T |C| |d| and u = 2^-24:
//   left out        R d, H r and r of the outer product: 3 x 2^-16 S (and terms of 2^-24 S)
//   rounding        of H h: <= 128 (256) products and sums inside the matrix pipe, each taken as accurate to 2 u, whatever
//                   their order; the small products come first, so theirs are relative to sums of 2^-7 S: 6 (12) u S; a
//                   16-term dot and 8 more sums: 24 u S
//   the reference   sums of <= 39 terms, one product, a tree of depth 8: 48 u S
//   S               <= (1 - 2^-8)^-3 S~ = 1.012 S~
// (Measured for H h: sums of 128 / 256 products through one accumulator are off by at most 8.7 / 13.3 u S, the worst over
// normal, cancelling, equal-signed, 2^+-24 spread, falling and rising operands, 2 M sums each: of the 256 / 512 u S above.)
// together 6.69e-5 S~ (128-d) and 8.27e-5 S~ (256-d).  The screen uses b = kappa S~ + 2^-100 with kappa = 1.15 x that:
// candidate a beats candidate c for certain when e~_a + b_a < e~_c - b_c.  Infinities and NaN leave every comparison
// undecided.
//
// Workgroup = (KV head, tile of tokens), D / 32 wavefronts; wavefront w keeps rows 32 w .. 32 w + 31 of C in registers as
// matrix A operands, its K blocks in the order that begins at its own diagonal block (the local forms use the first two).
// A step takes 16 tokens: candidates in registers (a token on D / 4 lanes, two tokens each), the three error vectors of
// every token as columns of two BF16 matrices in LDS; the base candidate's column of the head form is put together by
// address, block by block.
// Bound by the candidates: three quantisations and five transforms a row, some 800 vector instructions per pair of tokens;
// the matrix pipe takes 1600 cycles a step and wavefront.  Prompt of 8192 tokens x 8 heads of 128 on 4-bit pages 159 ->
// 90 us (before: the forms in FP32 on the matrix pipe, C read from L2 at every step); 2048 tokens x 4 heads of 256 on
// 2-bit pages 241 -> 44 us (before: exact only).
#include <cstdlib>

#include "writer_exact.hpp"

namespace fr {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int SCR_TOK = 16;                   // tokens per step
constexpr int SCR_MAXTILE = 128;              // tokens per workgroup at most (fallback list)

DEVI uint32_t bf16_pair(float a, float b) {
  const f32x2 v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
// two BF16 terms of four numbers
DEVI void split4(const float (&v)[4], uint2& hi, uint2& lo) {
  hi.x = bf16_pair(v[0], v[1]); hi.y = bf16_pair(v[2], v[3]);
  lo.x = bf16_pair(v[0] - bf16_lo(hi.x), v[1] - bf16_hi(hi.x));
  lo.y = bf16_pair(v[2] - bf16_lo(hi.y), v[3] - bf16_hi(hi.y));
}
DEVI f32x16 mfma(const uint4& a, const uint4& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
DEVI uint4 magnitude(const uint4& a, uint32_t nosign) {
  return make_uint4(a.x & nosign, a.y & nosign, a.z & nosign, a.w & nosign);
}

template <int D>
struct ScreenSmem {
  static constexpr int ROW = D + 8;                       // bf16 of a column: 16 bytes of padding
  union {
    struct {
      alignas(16) uint16_t hi[3 * SCR_TOK][ROW];          // column c * 16 + t: error vector of candidate c of token t
      alignas(16) uint16_t lo[3 * SCR_TOK][ROW];
    };
    StepSmem<D> exact;
  };
  uint32_t code[3][SCR_TOK][D / 4];                       // four codes of a lane
  uint16_t word[4][SCR_TOK][D / 32];                      // scale words of the candidates and of the value row
  alignas(16) uint8_t vcode[SCR_TOK][D];
  uint8_t choice[SCR_TOK][D / 32];                        // 0 as is, 1 H32, 2 undecided
  float form[2][D / 32][2 * SCR_TOK];                     // [form | S~][row block][column: base of 16 tokens, whole head of 16]
  long long slot[SCR_TOK];
  VRuns<SCR_TOK> runs;
  int fb[SCR_MAXTILE], nfb;
};

template <int QM, int P, int D, int TURNS>
__global__ void __launch_bounds__(2 * D, D == 128 ? 3 : 2) k_k2_screen(const K2WriteParams p, int tile, float kappa) {
  using L = Lay<QM, P>;
  constexpr int LU = D / 4, NB = D / 32, KB = D / 16;     // lanes of a token, 32-blocks, K blocks of the matrix product
  __shared__ ScreenSmem<D> S;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, kq = lane >> 5;
  const int unit = tid / LU, lu = tid % LU, d0 = 4 * lu, g = lu >> 3, half = D == 256 ? kq : 0;
  const int h = blockIdx.x, t_lo = blockIdx.y * tile, t_hi = min(p.T, t_lo + tile);
  const bool do_v = p.passes & 2;
  constexpr float TINY = 7.888609052210118e-31f;          // 2^-100
  // ---- A operands: row 32 wv + l32 of C^T (the form is the same), K block (2 wv + i) mod KB
  uint4 ah[KB], al[KB];
  {
    const float* row = p.CT + static_cast<size_t>(h) * D * D + static_cast<size_t>(32 * wv + l32) * D;
#pragma unroll
    for (int i = 0; i < KB; ++i) {
      const float* c = row + 16 * ((2 * wv + i) & (KB - 1)) + 8 * kq;
      const float4 c0 = *reinterpret_cast<const float4*>(c), c1 = *reinterpret_cast<const float4*>(c + 4);
      const float a[4] = {c0.x, c0.y, c0.z, c0.w}, b[4] = {c1.x, c1.y, c1.z, c1.w};
      uint2 h0, l0, h1, l1;
      split4(a, h0, l0);
      split4(b, h1, l1);
      ah[i] = make_uint4(h0.x, h0.y, h1.x, h1.y);
      al[i] = make_uint4(l0.x, l0.y, l1.x, l1.y);
    }
  }
  if (tid == 0) S.nfb = 0;

  for (int tb0 = t_lo; tb0 < t_hi; tb0 += SCR_TOK) {
    uint32_t nosign = 0x7FFF7FFFu;
    asm volatile("" : "+s"(nosign));            // (the magnitudes of C are not hoisted out of the loop into registers)
    // ---- P1: candidates and value rows of the unit's two tokens; a workgroup of eight tokens has one each (and the other
    // eight columns hold whatever was there: a column is its token's alone)
    // (a loop, not two copies: with the copies 24 registers spill, 108 -> 105 us; a loop over the candidates too: 112)
    if (TURNS == 1 && lu == 0) S.slot[unit + SCR_TOK / 2] = -1;
#pragma unroll 1
    for (int u = 0; u < TURNS; ++u) {
      const int tk = TURNS * unit + u, t = tb0 + tk;
      long long slot = -1;
      if (t < t_hi) slot = p.slots[static_cast<long long>(t) * (p.slot_ph ? p.Hkv : 1) + (p.slot_ph ? h : 0)];
      if (lu == 0) S.slot[tk] = slot;
      float x[4] = {0.f, 0.f, 0.f, 0.f}, v[4] = {0.f, 0.f, 0.f, 0.f};
      if (slot >= 0) {
        const long long at = static_cast<long long>(t) * p.kv_ts + d0;
        load_row(p.kv, at + static_cast<long long>(h) * D, x);
        if (do_v) load_row(p.kv, at + static_cast<long long>(p.Hkv + h) * D, v);
        if (p.kmu != nullptr) {
          const float4 m = *reinterpret_cast<const float4*>(p.kmu + h * D + d0);
          x[0] = x[0] - m.x; x[1] = x[1] - m.y; x[2] = x[2] - m.z; x[3] = x[3] - m.w;
        }
      }
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        float y[4] = {x[0], x[1], x[2], x[3]}, q[4], e[4];
        if (c == 1) fwht<32>(y, l32);
        if (c == 2) head_transform<D>(y, lane);
        const uint32_t w = quant_group<QM, true>(y, q, e);
        if (c == 1) fwht<32>(e, l32);
        if (c == 2) head_transform<D>(e, lane);
#pragma unroll
        for (int i = 0; i < 4; ++i) e[i] = e[i] - x[i];
        uint2 hi, lo;
        split4(e, hi, lo);
        *reinterpret_cast<uint2*>(&S.hi[c * SCR_TOK + tk][d0]) = hi;
        *reinterpret_cast<uint2*>(&S.lo[c * SCR_TOK + tk][d0]) = lo;
        uint32_t pack = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) pack |= code_bits(q[i], QM == QM_SYM4) << (8 * i);
        S.code[c][tk][lu] = pack;
        if ((lu & 7) == 0) S.word[c][tk][g] = static_cast<uint16_t>(w);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (do_v) {
        float q[4], deq[4];
        const uint32_t w = quant_group<QM, false>(v, q, deq);
        uint32_t pack = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) pack |= code_bits(q[i], QM == QM_SYM4) << (8 * i);
        *reinterpret_cast<uint32_t*>(&S.vcode[tk][d0]) = pack;
        if ((lu & 7) == 0) S.word[3][tk][g] = static_cast<uint16_t>(w);
      }
    }
    __syncthreads();
    // ---- P2: local forms of block wv; columns: as is of 16 tokens, H32 of 16 tokens
    {
      f32x16 acc, mag;
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] = mag[i] = 0.f;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint4 bh = *reinterpret_cast<const uint4*>(&S.hi[l32][32 * wv + 16 * i + 8 * kq]);
        const uint4 bl = *reinterpret_cast<const uint4*>(&S.lo[l32][32 * wv + 16 * i + 8 * kq]);
        acc = mfma(al[i], bl, acc);
        acc = mfma(ah[i], bl, acc);
        acc = mfma(al[i], bh, acc);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint4 bh = *reinterpret_cast<const uint4*>(&S.hi[l32][32 * wv + 16 * i + 8 * kq]);
        acc = mfma(ah[i], bh, acc);
        mag = mfma(magnitude(ah[i], nosign), magnitude(bh, nosign), mag);
      }
      float f = 0.f, s = 0.f;
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {          // rows 8 q4 + 4 kq + r of the block
        const uint2 dh = *reinterpret_cast<const uint2*>(&S.hi[l32][32 * wv + 8 * q4 + 4 * kq]);
        const uint2 dl = *reinterpret_cast<const uint2*>(&S.lo[l32][32 * wv + 8 * q4 + 4 * kq]);
        const float hv[4] = {bf16_lo(dh.x), bf16_hi(dh.x), bf16_lo(dh.y), bf16_hi(dh.y)};
        const float lv[4] = {bf16_lo(dl.x), bf16_hi(dl.x), bf16_lo(dl.y), bf16_hi(dl.y)};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          f = __builtin_fmaf(hv[r] + lv[r], acc[4 * q4 + r], f);
          s = __builtin_fmaf(fabsf(hv[r]), mag[4 * q4 + r], s);
        }
      }
      f += xor32(f); s += xor32(s);
      const float b = kappa * s + TINY, fo = hx(f, 16), bo = hx(b, 16);
      // the reference takes H32 iff its value is strictly smaller
      if (lane < SCR_TOK) S.choice[lane][wv] = fo + bo < f - b ? 1 : fo - bo > f + b ? 0 : 2;
    }
    if (do_v && wv == NB - 1) v_runs<SCR_TOK>(S.slot, S.runs);
    __syncthreads();
    // ---- P3: head forms of row block wv; columns: base of 16 tokens, whole head of 16 tokens
    {
      f32x16 acc, mag;
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] = mag[i] = 0.f;
      const int tok = l32 & 15;
      const bool whole = l32 >= 16;
      const int c0 = whole ? 2 * SCR_TOK + tok : tok;
#pragma unroll
      for (int i = 0; i < 2 * KB; i += 2) {         // the three small products of all blocks, then the large one
        const int blk = (wv + (i % KB) / 2) & (NB - 1);
        const int col = c0 + (!whole && S.choice[tok][blk] == 1 ? SCR_TOK : 0);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const uint4 bh = *reinterpret_cast<const uint4*>(&S.hi[col][32 * blk + 16 * j + 8 * kq]);
          if (i < KB) {
            const uint4 bl = *reinterpret_cast<const uint4*>(&S.lo[col][32 * blk + 16 * j + 8 * kq]);
            acc = mfma(al[i % KB + j], bl, acc);
            acc = mfma(ah[i % KB + j], bl, acc);
            acc = mfma(al[i % KB + j], bh, acc);
          } else {
            acc = mfma(ah[i % KB + j], bh, acc);
            mag = mfma(magnitude(ah[i % KB + j], nosign), magnitude(bh, nosign), mag);
          }
          if (j == 1) __builtin_amdgcn_sched_barrier(0);
        }
      }
      const int col = c0 + (!whole && S.choice[tok][wv] == 1 ? SCR_TOK : 0);
      float f = 0.f, s = 0.f;
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const uint2 dh = *reinterpret_cast<const uint2*>(&S.hi[col][32 * wv + 8 * q4 + 4 * kq]);
        const uint2 dl = *reinterpret_cast<const uint2*>(&S.lo[col][32 * wv + 8 * q4 + 4 * kq]);
        const float hv[4] = {bf16_lo(dh.x), bf16_hi(dh.x), bf16_lo(dh.y), bf16_hi(dh.y)};
        const float lv[4] = {bf16_lo(dl.x), bf16_hi(dl.x), bf16_lo(dl.y), bf16_hi(dl.y)};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          f = __builtin_fmaf(hv[r] + lv[r], acc[4 * q4 + r], f);
          s = __builtin_fmaf(fabsf(hv[r]), mag[4 * q4 + r], s);
        }
      }
      f += xor32(f); s += xor32(s);
      if (kq == 0) { S.form[0][wv][l32] = f; S.form[1][wv][l32] = s; }
    }
    // value codes of all the step's tokens, run by run
    if (do_v) {
      constexpr int NWORD = (QM == QM_ASYM2 ? 64 : 128) * (D / 128), AT_ONCE = 2 * D / NWORD;
      const int n = S.runs.n, j = tid % NWORD, s = j / (NWORD / (D / 128));
      for (int r = tid / NWORD; r < n; r += AT_ONCE) {
        const long long first = S.runs.first[r];
        store_v_words<QM, P>(p.pool + ((first / P) * (p.Hkv * (D / 128)) + h * (D / 128) + s) * L::CHUNK,
                             static_cast<int>(first % P) >> 3, j % (NWORD / (D / 128)), &S.vcode[0][128 * s], D, S.runs.map[r]);
      }
    }
    __syncthreads();
    // ---- P4: base against whole head; the rows of the decided tokens into their pages
#pragma unroll 1
    for (int u = 0; u < TURNS; ++u) {
      const int tk = TURNS * unit + u;
      const long long slot = S.slot[tk];
      float e[2], b[2];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        float f = 0.f, s = 0.f;
#pragma unroll
        for (int w = 0; w < NB; ++w) { f += S.form[0][w][16 * c + tk]; s += S.form[1][w][16 * c + tk]; }
        e[c] = f;
        b[c] = kappa * s + TINY;
      }
      int dec = e[1] + b[1] < e[0] - b[0] ? 1 : e[1] - b[1] > e[0] + b[0] ? 0 : 2;
#pragma unroll
      for (int w = 0; w < NB / 4; ++w)
        if (reinterpret_cast<const uint32_t*>(&S.choice[tk][0])[w] & 0x02020202u) dec = 2;
      if (slot < 0) continue;
      if (dec == 2) {
        if (lu == 0) S.fb[atomicAdd(&S.nfb, 1)] = tb0 + tk;
        continue;
      }
      const int c = dec == 1 ? 2 : S.choice[tk][g];
      uint8_t* chunk = p.pool + ((slot / P) * (p.Hkv * (D / 128)) + h * (D / 128) + half) * L::CHUNK;
      const int pos = static_cast<int>(slot % P);
      const uint32_t pack = S.code[c][tk][lu];
      const uint32_t code[4] = {pack & 0xFFu, (pack >> 8) & 0xFFu, (pack >> 16) & 0xFFu, pack >> 24};
      store_row<QM, P>(chunk, pos, false, code, S.word[c][tk][g] | (c == 1 ? 0x8000u : 0u), l32, false);
      if (do_v) {
        store_v_word<QM, P>(chunk, pos, S.word[3][tk][g] | (g == 0 && dec == 1 ? 0x8000u : 0u), l32, false);
      } else if (lu == 0) {
        const int off = L::VS_OFF + (8 * (pos >> 3) + vs_slot8(pos)) * 2;
        uint32_t* wp = reinterpret_cast<uint32_t*>(chunk + (off & ~3));
        const uint32_t bit = 0x8000u << ((off & 2) * 8);
        if (dec == 1) atomicOr(wp, bit); else atomicAnd(wp, ~bit);
      }
    }
    // (the next step's P1 rewrites what P2 and P3 read, behind the barrier above; codes and words are a unit's own; choices
    //  and runs are rewritten behind the next barrier, forms behind the one after)
  }
  // ---- the tokens the screen could not decide
  __syncthreads();
  const int nfb = S.nfb;
  if (nfb == 0) return;
  CqRegs<D> C;
  C.load(p.CT + static_cast<size_t>(h) * D * D);
  for (int i = 0; i < nfb; ++i) {
    const int t = S.fb[i];
    k2_exact_token<QM, P, D, false>(p, S.exact, C, h, t, p.slots[static_cast<long long>(t) * (p.slot_ph ? p.Hkv : 1) + (p.slot_ph ? h : 0)]);
    __syncthreads();
  }
}

// tokens of a workgroup
template <int D>
int tile_tokens(long long T, int Hkv) {
  // Steps per workgroup: all workgroups resident at once (3 per CU at head dim 128, 1 at 256) as far as the list of undecided
  // tokens allows; from five steps on, 128-d heads take workgroups of two, which the dispatcher spreads evenly (8 heads of
  // 128, us for 1 / 2 / 4 / 6 / 8 steps: 8192 tokens 94 / 91 / 101 / 97 / 106, 6000 tokens 70 / 68 / 66 / 79 / 100; 4 heads of
  // 256, 8192 tokens 187 / 166 / 139 / 188 / 131).
  constexpr long long RESIDENT = D == 128 ? 768 : 256;
  const long long steps = (T + SCR_TOK - 1) / SCR_TOK, fit = (steps * Hkv + RESIDENT - 1) / RESIDENT;
  const long long per = D == 128 && fit > 4 ? 2 : fit < SCR_MAXTILE / SCR_TOK ? fit : SCR_MAXTILE / SCR_TOK;
  // Short prompts, half a step a workgroup where that leaves every CU one at most: the candidates of one token instead of two
  // in a row (us, whole / half steps: 8 heads of 128, 130 tokens 18.2 / 15.6, 260 17.9 / 17.3, 520 19.9 / 21.0; 4 heads of 256,
  // 260 tokens 31.2 / 25.9, 400 31.7 / 25.5, 520 33.6 / 37.6).
  const bool half = (T + SCR_TOK / 2 - 1) / (SCR_TOK / 2) * Hkv <= 256;
  return half ? SCR_TOK / 2 : SCR_TOK * static_cast<int>(per);
}
template <int QM, int P, int D>
int screen(const K2WriteParams& p, float kappa, hipStream_t st) {
  const int tile = tile_tokens<D>(p.T, p.Hkv);
  const dim3 grid(p.Hkv, (p.T + tile - 1) / tile);
  // (A kernel of its own for the half steps: with the number of turns as a value both lose, 8192 tokens 95.1 -> 99.5 us.)
  if (tile < SCR_TOK) hipLaunchKernelGGL((k_k2_screen<QM, P, D, 1>), grid, dim3(2 * D), 0, st, p, tile, kappa);
  else hipLaunchKernelGGL((k_k2_screen<QM, P, D, 2>), grid, dim3(2 * D), 0, st, p, tile, kappa);
  return hipPeekAtLastError() == hipSuccess ? 0 : -1;
}
template <int QM>
int screen_qm(const K2WriteParams& p, bool all_exact, hipStream_t st) {
  static const float scale = getenv("FLAGROT_W3_KAPPA") != nullptr ? static_cast<float>(atof(getenv("FLAGROT_W3_KAPPA"))) : 1.f;
  const float kappa = all_exact ? 1e30f : scale * (p.hd == 256 ? 9.5e-5f : 7.7e-5f);
  if (p.page != 16 && p.page != 32) return -5;
  if (p.hd == 256) return p.page == 16 ? screen<QM, 16, 256>(p, kappa, st) : screen<QM, 32, 256>(p, kappa, st);
  return p.page == 16 ? screen<QM, 16, 128>(p, kappa, st) : screen<QM, 32, 128>(p, kappa, st);
}

}  // namespace

int k2_screen_launch(int kind, const K2WriteParams& p, bool all_exact, hipStream_t st) {
  switch (kind) {
    case KIND_KONLY: return screen_qm<QM_SYM4>(p, all_exact, st);
    case KIND_KONLYA: return screen_qm<QM_ASYM4>(p, all_exact, st);
    case KIND_KONLYA2: return screen_qm<QM_ASYM2>(p, all_exact, st);
  }
  return -4;
}
int k2_screen_tokens(long long T, int Hkv, int hd) { return hd == 256 ? tile_tokens<256>(T, Hkv) : tile_tokens<128>(T, Hkv); }
int k2_screen_lds_bytes(int hd) { return static_cast<int>(hd == 256 ? sizeof(ScreenSmem<256>) : sizeof(ScreenSmem<128>)); }

}  // namespace fr
