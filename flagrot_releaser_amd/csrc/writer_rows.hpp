// Row helpers shared by the selecting writers: loads, the halving trees of the weighted error sums.
#pragma once
#include "fr_common.hpp"

namespace fr {

DEVI void load_row(const void* kv, long long off, float (&x)[4]) {
  const uint2 raw = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(kv) + off);
  x[0] = bf16_lo(raw.x); x[1] = bf16_hi(raw.x); x[2] = bf16_lo(raw.y); x[3] = bf16_hi(raw.y);
}

DEVI float tree128(const float (&p)[4]) {  // halving tree of a 128-vector, 4 consecutive elements per lane
  float v[4] = {p[0], p[1], p[2], p[3]};
#pragma unroll
  for (int o = 16; o > 0; o >>= 1)
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = v[i] + hx(v[i], o);
  return (v[0] + v[2]) + (v[1] + v[3]);
}
DEVI float tree32(const float (&p)[4]) {  // the same over the 32 elements held by 8 lanes
  float v[4] = {p[0], p[1], p[2], p[3]};
#pragma unroll
  for (int o = 4; o > 0; o >>= 1)
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = v[i] + hx(v[i], o);
  return (v[0] + v[2]) + (v[1] + v[3]);
}
DEVI float tree32_lanes(float v) {        // the same tree, one element per lane of a half wave
#pragma unroll
  for (int o = 16; o > 0; o >>= 1) v = v + hx(v, o);
  return v;
}

// orthonormal H_D of a row held by the wavefront (D = 256: lane = dims 4 lane + i; D = 128: both half waves hold it)
template <int D>
DEVI void head_transform(float (&y)[4], int lane) {
  if constexpr (D == 128) {
    fwht<128>(y, lane & 31);
  } else {
    butterflies<128>(y, lane & 31);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float o = xor32(y[i]);
      y[i] = (lane >= 32 ? o - y[i] : y[i] + o) * 0.0625f;
    }
  }
}

// ---- value codes of up to 64 tokens, word by word
// The eight tokens of an aligned run of slots share V^T words.  VRuns: the n runs that the N tokens (slots in LDS, negative:
// none) touch, of each the first slot and, a byte per position, which token holds it (0xFF: none of these).
template <int N>
struct VRuns {
  long long first[N];
  unsigned long long map[N];
  int n;
};
template <int N>
DEVI void v_runs(const long long* slot, VRuns<N>& r) {        // called by one whole wavefront; the caller's barrier follows
  // lane = (token i = lane mod N, a share of the tokens it is compared with); the shares of a token are N lanes apart.  The
  // workgroup waits for this wavefront: with every comparison of a token in one lane, in 64-bit words, it took 3.3 k cycles
  // of a step of 16 tokens (screened writer, 8192 tokens x 4 heads of 256: 152 -> 138 us, x 8 heads of 128: 102 -> 100).
  constexpr int PER = N * N / 64;
  static_assert(N == 8 || N == 16, "whole shares, 64 lanes");
  const int lane = threadIdx.x & 63, i = lane % N, j0 = lane / N * PER;
  const long long s = slot[i], run = s & ~7LL;
  uint32_t lo = ~0u, hi = ~0u;                                // the map, positions 0 .. 3 and 4 .. 7 of the run
  uint32_t later = s < 0 ? 1u : 0u;                           // an earlier token is in the run (or there is none)
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int j = j0 + k;
    const long long o = slot[j];
    if (o < 0 || (o & ~7LL) != run) continue;
    if (j < i) later = 1u;
    const int b = 8 * static_cast<int>(o & 3);
    const uint32_t keep = ~(0xFFu << b), put = static_cast<uint32_t>(j) << b;
    if (o & 4) hi = (hi & keep) | put; else lo = (lo & keep) | put;
  }
#pragma unroll
  for (int m = N; m < 64; m <<= 1) {                          // a position that two tokens name is the later one's
    const bool upper = (lane & m) != 0;
    const uint32_t l = __shfl_xor(lo, m, 64), h = __shfl_xor(hi, m, 64);
    const uint32_t l1 = upper ? lo : l, h1 = upper ? hi : h;
    const uint32_t ml = ((l1 >> 7) & 0x01010101u) * 0xFFu, mh = ((h1 >> 7) & 0x01010101u) * 0xFFu;   // 0xFF: not set there
    lo = (ml & (upper ? l : lo)) | (~ml & l1);
    hi = (mh & (upper ? h : hi)) | (~mh & h1);
    later |= __shfl_xor(later, m, 64);
  }
  const bool leads = lane < N && later == 0u;
  const unsigned long long who = __ballot(leads);
  if (leads) {
    const int at = __popcll(who & ((1ull << lane) - 1));
    r.first[at] = run;
    r.map[at] = lo | (static_cast<unsigned long long>(hi) << 32);
  }
  if (lane == 0) r.n = __popcll(who);
}
// word j of a run: whole if the tokens at hand hold all eight positions, else merged (other tokens may be stored at the
// same time).  codes[token * stride + dim]
template <int QM, int P>
DEVI void store_v_words(uint8_t* chunk, int c8, int j, const uint8_t* codes, int stride, unsigned long long map) {
  using L = Lay<QM, P>;
  uint32_t wd = 0, mask = 0;
  if constexpr (QM == QM_ASYM2) {
    const int e = j >> 1, m = j & 1, dd = 64 * m + 16 * (e >> 3) + (e & 7);
#pragma unroll
    for (int tk = 0; tk < 8; ++tk) {
      const int at = static_cast<int>(map >> (8 * tk)) & 0xFF, sh = 8 * (tk >> 1) + 2 * (tk & 1);
      if (at == 0xFF) continue;
      const uint8_t* c = codes + at * stride + dd;
      wd |= (static_cast<uint32_t>(c[0]) | (static_cast<uint32_t>(c[8]) << 4)) << sh;
      mask |= 0x33u << sh;
    }
    uint32_t* wp = reinterpret_cast<uint32_t*>(chunk + L::V_OFF + (e * (P / 8) + c8) * 8 + 4 * m);
    if (mask == ~0u) *wp = wd;
    else { atomicAnd(wp, ~mask); atomicOr(wp, wd); }
  } else {
    const int e = j >> 2, sub = j & 3, dd = 64 * (sub >> 1) + 16 * (e >> 3) + 8 * (sub & 1) + (e & 7);
#pragma unroll
    for (int tk = 0; tk < 8; ++tk) {
      const int at = static_cast<int>(map >> (8 * tk)) & 0xFF;
      if (at == 0xFF) continue;
      uint32_t m, b;
      place4<QM>(codes[at * stride + dd], (tk & 1) != 0, tk >> 1, m, b);
      wd |= b;
      mask |= m;
    }
    uint32_t* wp = reinterpret_cast<uint32_t*>(chunk + L::V_OFF + (e * (P / 8) + c8) * 16 + 4 * sub);
    if (mask == ~0u) *wp = wd;
    else { atomicAnd(wp, ~mask); atomicOr(wp, wd); }
  }
}

}  // namespace fr
