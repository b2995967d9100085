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

}  // namespace fr
