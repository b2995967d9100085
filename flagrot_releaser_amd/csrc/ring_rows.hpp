// One quad (four channels) of the BF16 rows a request keeps beside its pages: what ring.hip launches by itself, and what the
// writers of a decode step do in workgroups of their own behind those of the pages (ring_quads of them).
#pragma once
#include "fr_common.hpp"
#include "fr_launch.hpp"

namespace fr {

DEVI uint32_t bf16_row_rn(float f) { return f != f ? 0x7FC0u : bf16_rn(f); }      // (the rounding alone may lose a NaN)

inline __host__ __device__ long long ring_quads(const RingRowsParams& p) { return static_cast<long long>(p.rows) * (p.width / 4); }

DEVI void ring_quad(const RingRowsParams& p, long long at) {
  const int quads = p.width / 4;                           // of one row: K heads, then V heads
  if (at >= ring_quads(p)) return;
  const int r = static_cast<int>(at / quads), c = 4 * static_cast<int>(at % quads);
  int t = r;
  long long slot;
  if (p.dest != nullptr) slot = p.dest[r];
  else {                                                   // the leading sinks of the chunk, then the rows of its window
    t = r < p.sinks ? r : p.win0 + (r - p.sinks);
    const int pos = p.start + t;
    slot = p.base + (pos < p.S ? pos : p.S + (pos - p.S) % p.W);
  }
  if (slot < 0 || slot >= p.ring_rows) return;
  uint2 raw = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(p.kv) + static_cast<long long>(t) * p.kv_ts + c);
  if (p.kmu != nullptr && c < p.width / 2) {
    const float4 m = *reinterpret_cast<const float4*>(p.kmu + c);
    raw.x = bf16_row_rn(bf16_lo(raw.x) - m.x) | (bf16_row_rn(bf16_hi(raw.x) - m.y) << 16);
    raw.y = bf16_row_rn(bf16_lo(raw.y) - m.z) | (bf16_row_rn(bf16_hi(raw.y) - m.w) << 16);
  }
  *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p.ring) + slot * p.width + c) = raw;
}

}  // namespace fr
