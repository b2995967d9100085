// Split merge of the KIVI-style decode attention (both head dims): workgroup = (sequence, query head).  The NS + 1
// partials of the query head's (sequence, KV head) are dealt to MERGE_SLICES slices of D / 4 threads, four channels a
// thread; a slice requests the (maximum, sum) pairs and its channels of eight partials together, so a call with up to 64
// partials is ONE memory round trip, and the slices meet in LDS.  One thread per channel over all partials, eight at a time,
// is a round trip of 2.5 us for every eight (head dim 256, 1 sequence x 24 query heads, 51 partials: 19.6 us, this form 4.4;
// head dim 128, 1 x 32 heads, 26 partials 9.9, now 4.1; 16 x 64 heads, 8 partials 4.7 both).  Semantics:
// integrations/vllm_flagrot/csrc/kivi.cu:1908-1931.
#pragma once
#include "fr_common.hpp"

namespace frkv {
using namespace fr;

constexpr int MERGE_SLICES = 8;
template <int D>
__global__ void __launch_bounds__(MERGE_SLICES * D / 4) k_merge_parts(const float* __restrict__ opart, const float* __restrict__ ml,
                                                                      int Hkv, int G, int NS, uint16_t* __restrict__ out,
                                                                      long long out_rs) {
  constexpr int LANES = D / 4;                              // of a slice, four channels each
  __shared__ float2 ms[MERGE_SLICES];
  __shared__ float4 part[MERGE_SLICES][LANES];
  const int b = blockIdx.x, hq = blockIdx.y, h = hq / G, g = hq % G, slice = threadIdx.x / LANES, lane = threadIdx.x % LANES;
  const long long p0 = (static_cast<long long>(b) * Hkv + h) * (NS + 1);
  float M = -INFINITY, L = 0.f;
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int s0 = slice; s0 <= NS; s0 += 8 * MERGE_SLICES) {
    float2 st[8];
    float4 x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {      // past the last partial: the slice's first one again, skipped below
      const bool in = s0 + i * MERGE_SLICES <= NS;
      const long long at = (p0 + (in ? s0 + i * MERGE_SLICES : s0)) * G + g;
      __builtin_memcpy(&st[i], ml + at * 2, sizeof(float2));       // (ml may start at any float; opart is written 16 bytes at a time)
      x[i] = *reinterpret_cast<const float4*>(opart + at * D + 4 * lane);
      if (!in) st[i].x = -INFINITY;
    }
    float top = M;
#pragma unroll
    for (int i = 0; i < 8; ++i) top = fmaxf(top, st[i].x);
    if (top == -INFINITY) continue;                       // nothing but empty partials so far
    const float keep = M == -INFINITY ? 0.f : exp2f(M - top);
    L *= keep; o.x *= keep; o.y *= keep; o.z *= keep; o.w *= keep; M = top;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (st[i].x == -INFINITY) continue;
      const float f = exp2f(st[i].x - M);
      L += f * st[i].y;
      o.x += f * x[i].x; o.y += f * x[i].y; o.z += f * x[i].z; o.w += f * x[i].w;
    }
  }
  if (lane == 0) ms[slice] = make_float2(M, L);
  part[slice][lane] = o;
  __syncthreads();
  if (threadIdx.x >= LANES) return;
  float top = -INFINITY;
#pragma unroll
  for (int s = 0; s < MERGE_SLICES; ++s) top = fmaxf(top, ms[s].x);
  float total = 0.f;
  o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int s = 0; s < MERGE_SLICES; ++s) {
    if (ms[s].x == -INFINITY) continue;
    const float f = exp2f(ms[s].x - top);
    const float4 x = part[s][lane];
    total += f * ms[s].y;
    o.x += f * x.x; o.y += f * x.y; o.z += f * x.z; o.w += f * x.w;
  }
  const float inv = total > 0.f ? 1.f / total : 0.f;
  uint16_t* dst = out + static_cast<long long>(b) * out_rs + static_cast<long long>(hq) * D + 4 * lane;
  const uint32_t r[4] = {bf16_rn(o.x * inv), bf16_rn(o.y * inv), bf16_rn(o.z * inv), bf16_rn(o.w * inv)};
#pragma unroll
  for (int i = 0; i < 4; ++i) dst[i] = static_cast<uint16_t>(r[i]);       // (output rows may start anywhere)
}

}  // namespace frkv
