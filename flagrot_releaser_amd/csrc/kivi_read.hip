// KIVI-style pages back to rows, head dim 128 and 256: one workgroup per (32-token group, KV head), keys and values in the
// basis the writers were given.  Page layouts: kivi_write.hip (128) and kivi_wide.hip (256).  Compiled with
// -ffp-contract=off: transforms in the association of the writers.
//
// A lane owns eight channels of a row (16 bytes of BF16), so a sub-vector lies on four lanes and a rotation exchanges
// twice between neighbours instead of three times; code x step is exact, so that and the minimum are one instruction.  The
// KV heads of a group are neighbours in dispatch order: together they write whole tokens (2 KB and more in one piece).
// Bound by vector issue (20.1 M instructions a launch of 32640 tokens x 8 heads: 81 k of a SIMD's 82 k cycles) and as much by
// its 24 MB in and 134 MB out: kernel 41 -> 34 us (4.6 TB/s, what a large copy reaches), the call on cold pages 59 -> 50 us
// (before: four channels a lane, 2-byte stores, heads outermost).
#include "fr_common.hpp"
#include "kivi_launch.hpp"
#include "kivi_quant.hpp"

namespace frkv {
using namespace fr;
namespace {

template <int D, bool F8> struct Page {
  static constexpr int NV = D / 32, META = F8 ? 2 : 4;     // sub-vectors; bytes of a (step, minimum) pair
  static constexpr int KM = 4 * D, VC = KM + NV * META * 16, VM = VC + 4 * D, VF = 12 * D;
  static constexpr long long CHUNK = F8 ? 10 * D : 12 * D + 16;
};
static_assert(Page<128, false>::VC == 768 && Page<128, true>::VC == 640 && Page<256, false>::VM == 2560 && Page<256, true>::VM == 2304, "layout");

template <bool F8> DEVI void pair_at(const uint8_t* at, float& s, float& mn, bool& flag) {
  if (F8) { flag = at[0] >> 7; s = e4m3_value(at[0] & 0x7Fu); mn = e4m3_value(at[1]); }
  else {
    const uint32_t w = *reinterpret_cast<const uint32_t*>(at);
    flag = (w >> 15) & 1u; s = f16_value(w & 0x7FFFu); mn = f16_value(w >> 16);
  }
}
// Sylvester stages: the three inside the lane and lanes 1, 2 apart (H32); lanes 4, 8 (16) apart on top (H128 / H256)
DEVI void stage(float (&y)[8], int lane, int lm) {
  const uint32_t flip = (lane & lm) ? 0x80000000u : 0u;
#pragma unroll
  for (int i = 0; i < 8; ++i) y[i] = hx(y[i], lm) + __uint_as_float(__float_as_uint(y[i]) ^ flip);
}
DEVI void stages32(float (&y)[8], int lane) {
#pragma unroll
  for (int d = 1; d < 8; d <<= 1)
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (!(i & d)) {
        const float a = y[i], b = y[i + d];
        y[i] = a + b;
        y[i + d] = a - b;
      }
  stage(y, lane, 1);
  stage(y, lane, 2);
}
template <int D> DEVI void stages_head(float (&y)[8], int lane) {
  stage(y, lane, 4);
  stage(y, lane, 8);
  if constexpr (D == 256) stage(y, lane, 16);
}
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
// (rows may begin at any element: no alignment is promised to the stores)
DEVI void put(uint16_t* at, const float (&x)[8]) {
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x2 v = {x[2 * i], x[2 * i + 1]};
    w[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
  }
  __builtin_memcpy(at, w, 16);
}
DEVI void put(float* at, const float (&x)[8]) { __builtin_memcpy(at, x, 32); }

template <typename OT, int D, bool F8>
__global__ void __launch_bounds__(256) k_read_pages(const uint8_t* __restrict__ pool, const int* __restrict__ bt, int g0,
                                                    int Hkv, int nvalid, OT* __restrict__ ok, OT* __restrict__ ov) {
  using PG = Page<D, F8>;
  constexpr int LR = D / 8, NV = PG::NV;                   // lanes of a row
  constexpr float CD = D == 256 ? 0.0625f : kC128;
  const int h = blockIdx.x % Hkv, gi = blockIdx.x / Hkv, lr = threadIdx.x % LR, lane = threadIdx.x & 31, g = g0 + gi;
  const uint8_t* chA = pool + (static_cast<long long>(bt[2 * g]) * Hkv + h) * PG::CHUNK;
  const uint8_t* chB = pool + (static_cast<long long>(bt[2 * g + 1]) * Hkv + h) * PG::CHUNK;
  bool kH = false, kF;                                     // the lane's sub-vector is H32, the group's keys are whole-head
  float ks[8], kmn[8];
  {
    const int j = lr >> 2;
    if (F8) { kH = chA[PG::KM + j * NV * 2] >> 7; kF = chA[PG::KM + NV * NV * 2] >> 7; }
    else {
      kH = (reinterpret_cast<const uint32_t*>(chA + PG::KM)[j] >> 15) & 1u;
      kF = (reinterpret_cast<const uint32_t*>(chA + PG::KM)[NV] >> 15) & 1u;
    }
    bool fl;
#pragma unroll
    for (int i = 0; i < 8; ++i) {                          // channel 8 lr + i: cell (channel / NV), slot channel % NV
      const int c = 8 * lr + i, cell = c / NV;
      pair_at<F8>((cell < 16 ? chA : chB) + PG::KM + ((cell & 15) * NV + c % NV) * PG::META, ks[i], kmn[i], fl);
    }
  }
  const bool rotate = __any(kH);                           // (kF: the same for the workgroup)
#pragma unroll 2
  for (int t = threadIdx.x / LR; t < 32; t += 256 / LR) {
    const long long o = static_cast<long long>(gi) * 32 + t;
    const uint8_t* ch = t < 16 ? chA : chB;
    const int cell = t & 15;
    const uint32_t kw = reinterpret_cast<const uint32_t*>(ch + cell * (D / 4))[lr >> 1] >> (8 * (lr & 1));
    const uint32_t vw = *reinterpret_cast<const uint16_t*>(ch + PG::VC + cell * (D / 4) + 2 * lr);
    float vs, vmn;
    bool vH;
    pair_at<F8>(ch + PG::VM + (cell * NV + (lr >> 2)) * PG::META, vs, vmn, vH);
    const bool vF = F8 ? (ch[PG::KM + cell * NV * 2 + 2 * (NV - 1)] >> 7) != 0 : ch[PG::VF + cell] != 0;
    {
      float x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = __builtin_fmaf(static_cast<float>((kw >> (2 * (i >> 1) + 16 * (i & 1))) & 3u), ks[i], kmn[i]);
      if (kF) {
        stages32(x, lane);
        stages_head<D>(x, lane);
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = x[i] * CD;
      } else if (rotate) {
        float y[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] = x[i];
        stages32(y, lane);
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = kH ? y[i] * kC32 : x[i];
      }
      if (o < nvalid) put(ok + (o * Hkv + h) * D + 8 * lr, x);
    }
    {
      float x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = __builtin_fmaf(static_cast<float>((vw >> (2 * i)) & 3u), vs, vmn);
      if (__any(vH || vF)) {                               // the rows of a wavefront have flags of their own
        float y[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] = x[i];
        stages32(y, lane);
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = vH && !vF ? y[i] * kC32 : x[i];
        if (__any(vF)) {
          stages_head<D>(y, lane);
#pragma unroll
          for (int i = 0; i < 8; ++i) x[i] = vF ? y[i] * CD : x[i];
        }
      }
      if (o < nvalid) put(ov + (o * Hkv + h) * D + 8 * lr, x);
    }
  }
}

template <int D, bool F8>
void read_pages(const uint8_t* pool, const int* bt, int g0, int g1, int nvalid, int Hkv, int fp32, void* ok, void* ov, hipStream_t st) {
  const dim3 grid(static_cast<unsigned>(g1 - g0) * Hkv);
  if (fp32)
    hipLaunchKernelGGL((k_read_pages<float, D, F8>), grid, dim3(256), 0, st, pool, bt, g0, Hkv, nvalid, static_cast<float*>(ok), static_cast<float*>(ov));
  else
    hipLaunchKernelGGL((k_read_pages<uint16_t, D, F8>), grid, dim3(256), 0, st, pool, bt, g0, Hkv, nvalid, static_cast<uint16_t*>(ok), static_cast<uint16_t*>(ov));
}

}  // namespace

int dequant_launch(int D, const uint8_t* pool, const int* bt, int g0, int g1, int nvalid, int Hkv, int fp32, void* ok, void* ov,
                   int f8, hipStream_t st) {
  const auto go = D == 256 ? (f8 ? &read_pages<256, true> : &read_pages<256, false>) : (f8 ? &read_pages<128, true> : &read_pages<128, false>);
  go(pool, bt, g0, g1, nvalid, Hkv, fp32, ok, ov, st);
  return hipPeekAtLastError() == hipSuccess ? 0 : 1;
}

}  // namespace frkv
