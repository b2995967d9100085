// Pieces of the 256-row prefill kernels, shared by the kernel that converts page words between its matrix instructions (k_mq8,
// mq_prefill.hip) and by the pair that converts them once for all tiles of a request (mq_images.hip).
#pragma once
#include "mq_tiles.hpp"

namespace frmq {

// Raw page words of a thread's tile entry, one register set for both groups (a set per group would let the compiler
// reuse the other group's registers for LDS operands and guard them with waits on outstanding fetches):
//   group A  w[0] = K code words of (token, tg) (INT2: .x .y), w[1].xy = the token's four K scale words,
//            w[1].z = the token's group-0 V scale word (whole-head flag of key-only pages)
//   group B  w[0] = V^T entry (e, c8) of a page, w[1], w[2] = V scale words of the entry's run (eight tokens) in its
//            two groups: t0 t2 | t4 t6 | t1 t3 | t5 t7
struct Raw8 {
  u32x4 w[3];
};

// A wavefront of the group fetches one page of the block (page = its index in the group): the page base is
// wave-uniform, the lane adds a 32-bit offset.  Lane = (token pos = lane >> 2, quarter tg) for the K words.
template <int QM, bool K2>
DEVI void load_k8(Raw8& R, const Params& p, const int* pg, int h, int kb, int kend, int t256) {
  using F = Fmt<QM>;
  const uint32_t lane = t256 & 63, pos = lane >> 2, tg = lane & 3u;
  const int pgi = __builtin_amdgcn_readfirstlane(t256 >> 6);
  const int j0 = kb * BN + PAGE * pgi;
  if (j0 + static_cast<int>(pos) < kend) {
    const int page = __builtin_amdgcn_readfirstlane(pg[pgi]);
    const uint8_t* ch = p.pool + static_cast<long long>(page) * p.page_stride + static_cast<long long>(h) * F::CHUNK;
    if constexpr (QM == QM_ASYM2) {
      const u32x2 c = gload<u32x2>(ch + (32u * (pos ^ ((pos >> 1) & 2u)) + 8u * tg));
      R.w[0] = u32x4{c.x, c.y, 0u, 0u};
    } else {
      R.w[0] = gload<u32x4>(ch + 16u * lane);
    }
    const u32x2 ks = gload<u32x2>(ch + (F::KS_OFF + 8u * pos));
    R.w[1].x = ks.x; R.w[1].y = ks.y;
    if constexpr (K2) R.w[1].z = gload<uint16_t>(ch + (F::VS_OFF + (8u * (pos >> 3) + static_cast<uint32_t>(vs_slot8(pos))) * 2u));
  }
}
template <int QM>
DEVI void load_v8(Raw8& R, const Params& p, const int* pg, int h, int kb, int kend, int t256) {
  using F = Fmt<QM>;
  const uint32_t lane = t256 & 63, g = lane >> 5, c8 = lane & 1u;      // entry e = lane >> 1: its dims lie in groups g, g + 2
  const int pgi = __builtin_amdgcn_readfirstlane(t256 >> 6);
  const int j0 = kb * BN + PAGE * pgi;
  if (j0 < kend) {
    const int page = __builtin_amdgcn_readfirstlane(pg[pgi]);
    const uint8_t* ch = p.pool + static_cast<long long>(page) * p.page_stride + static_cast<long long>(h) * F::CHUNK;
    if constexpr (QM == QM_ASYM2) {
      const u32x2 c = gload<u32x2>(ch + (F::V_OFF + 8u * lane));
      R.w[0] = u32x4{c.x, c.y, 0u, 0u};
    } else {
      R.w[0] = gload<u32x4>(ch + (F::V_OFF + 16u * lane));
    }
    R.w[1] = gload<u32x4>(ch + (F::VS_OFF + (g * PAGE + 8u * c8) * 2u));
    R.w[2] = gload<u32x4>(ch + (F::VS_OFF + ((g + 2u) * PAGE + 8u * c8) * 2u));
  }
}

// V^T tile entry: the scale / zero point pairs of the entry's run come from the thread's own scale words, in the run
// order (t0,t4) (t1,t5) (t2,t6) (t3,t7); tokens at or beyond kend get scale 0
template <int QM, class At = Padded>
DEVI void convert_v8(uint8_t* vt, const Raw8& R, int kb, int kend, const Consts& cst, int t256) {
  using F = Fmt<QM>;
  const int pgi = t256 >> 6, e = (t256 & 63) >> 1, c8 = t256 & 1, run = 2 * pgi + c8;
  const bool have = kb * BN + PAGE * pgi < kend;
  const bool ragged = kb * BN + BN > kend;                         // uniform: only the last block of an item
  uint32_t w[4] = {0u, 0u, 0u, 0u};
  if (have) {
    if constexpr (QM == QM_ASYM2) {
      w[0] = R.w[0].x; w[1] = R.w[0].x >> 4; w[2] = R.w[0].y; w[3] = R.w[0].y >> 4;
    } else {
      w[0] = R.w[0].x; w[1] = R.w[0].y; w[2] = R.w[0].z; w[3] = R.w[0].w;
    }
  }
  uint32_t sc[2][4], nz[2][4];
#pragma unroll
  for (int gg = 0; gg < 2; ++gg) {
    const u32x4 v = R.w[1 + gg];
    const uint32_t pr[4] = {__builtin_amdgcn_perm(v.y, v.x, 0x05040100u), __builtin_amdgcn_perm(v.w, v.z, 0x05040100u),
                            __builtin_amdgcn_perm(v.y, v.x, 0x07060302u), __builtin_amdgcn_perm(v.w, v.z, 0x07060302u)};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sc[gg][i] = have ? pr[i] & 0x7FFF7FFFu : 0u;
      nz[gg][i] = (pr[i] & (F::ZM * 0x10001u)) | 0xE400E400u;
    }
  }
  if (ragged) {
    const int t0 = kb * BN + 8 * run;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t m = (t0 + i < kend ? 0xFFFFu : 0u) | (t0 + i + 4 < kend ? 0xFFFF0000u : 0u);
      sc[0][i] &= m; sc[1][i] &= m;
    }
  }
#pragma unroll
  for (int sub = 0; sub < 4; ++sub) {
    const int d = 64 * (sub >> 1) + 16 * (e >> 3) + 8 * (sub & 1) + (e & 7);   // group d >> 5 = 2 (sub >> 1) + (e >> 4)
    uint32_t x[4];
    Unpack<QM>::run(w[sub], nz[sub >> 1], cst, x);
    *reinterpret_cast<u32x4*>(vt + At::v(d, run)) =
        u32x4{pk_mul(x[0], sc[sub >> 1][0]), pk_mul(x[1], sc[sub >> 1][1]), pk_mul(x[2], sc[sub >> 1][2]), pk_mul(x[3], sc[sub >> 1][3])};
  }
}

// lane = row, lanes l and l + 32 hold the two halves of its 64 keys; sacc = score - reference.  full: no key of the
// block is masked for any row of the wavefront.
DEVI void softmax8(f32x16 (&sacc)[2], u32x4 (&pb)[4], f32x16 (&o)[4], float& ref, float& lrow, bool full, int kb, int lim,
                   int kmin, int hh) {
  if (!full) {
    const int jb = kb * BN;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int j = jb + 32 * kt + token_of_acc(i, hh);
        if (!(j <= lim && j >= kmin)) sacc[kt][i] = -INFINITY;
      }
  }
  float mx = -INFINITY;
#pragma unroll
  for (int kt = 0; kt < 2; ++kt)
#pragma unroll
    for (int i = 0; i < 16; ++i) mx = fmaxf(mx, sacc[kt][i]);
  mx = max_halves(mx);
  const bool bump = (mx > 8.f || ref == -INFINITY) && mx != -INFINITY;
  if (__any(bump)) {                                     // rare after the first blocks: move the reference to the row maximum
    const float delta = bump ? mx : 0.f;
    const float alpha = ref == -INFINITY ? 0.f : fexp2(-delta);   // no reference yet: O and l are still zero
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i) sacc[kt][i] -= delta;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[db][i] *= alpha;
    lrow *= alpha;
    if (bump) ref = (ref == -INFINITY ? 0.f : ref) + delta;
  }
  typedef _Float16 h2v __attribute__((ext_vector_type(2)));
  const h2v ones = {static_cast<_Float16>(1.f), static_cast<_Float16>(1.f)};
  float s4[4] = {0.f, 0.f, 0.f, 0.f};                   // the sum of what the value product uses
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {      // ks = 2 kt + s
    const int kt = ks >> 1, s2 = ks & 1;
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = pack_h2_rn(fexp2(sacc[kt][8 * s2 + 2 * j]), fexp2(sacc[kt][8 * s2 + 2 * j + 1]));
#pragma unroll
    for (int j = 0; j < 4; ++j) s4[j] = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2v, w[j]), ones, s4[j], false);
    pb[ks] = u32x4{w[0], w[1], w[2], w[3]};
  }
  lrow += (s4[0] + s4[1]) + (s4[2] + s4[3]);
}

}  // namespace frmq
