// Prefill over pages whose fp16 tiles are made ONCE for all query tiles of a request (head dim 128, 256-row tiles):
// k_tile_images turns every 64-key block of every request into the image of its K and V^T tiles (32 KB, as LDS holds them),
// k_mq_images attends from the images.
//
// k_mq8 (mq_prefill.hip) converts a block for each query tile that reads it: its vector slots are softmax plus conversion,
// 5.3 k cycles a block where the matrix instructions take 2 k.  Here the conversion is a launch of its own, bound by the
// images it writes (138 MB in 34 us), and the attention kernel has nothing between the matrix instructions but the
// softmax: the images go from memory to LDS without passing through registers, two blocks ahead, 3.6 k cycles a block, the
// matrix pipe busy for 57 % of them (k_mq8 40 %).  4 requests x 512 tokens x 64 heads over 16 k on 4-bit key-only pages: 1222
// us, here 2 x (500 + 34) on a cache that repeats, 1418 and 2 x (551 + 37) on new inputs; 1117 TFLOP/s where a large matrix
// product reaches 1170, at a clock of 1.9 GHz (cycles a CU is busy over the dispatch's time; k_mq8 2.2).
#include "mq_launch.hpp"
#include "mq_rows256.hpp"

namespace frmq {
using namespace fr;
namespace {

constexpr int KV = Image::K_BYTES;                     // one tile: K_BYTES = V_BYTES
static_assert(Image::K_BYTES == Image::V_BYTES, "one piece size for both tiles");

// ------------------------------------------------------------------------------------------------ images
// Workgroup = (block record, head of the group); record: (block-table row, block, keys of the request).  A thread has the
// page words of one K and one V^T entry, the four wavefronts a page each; the image is put together in LDS and leaves in
// whole lines.
template <int QM, bool K2>
__global__ void __launch_bounds__(256) k_tile_images(const Params p, const int* __restrict__ recs, int head0, uint8_t* __restrict__ images) {
  __shared__ __align__(16) uint8_t img[Image::BYTES];
  const int* rec = recs + 4 * blockIdx.x;
  const int kb = rec[1], kend = rec[2], h = head0 + blockIdx.y, tid = threadIdx.x;
  const int* pages = p.bt + static_cast<long long>(rec[0]) * p.bt_stride + (BN / PAGE) * kb;
  const Consts cst = make_consts();
  Raw8 rk, rv;
  load_k8<QM, K2>(rk, p, pages, h, kb, kend, tid);
  load_v8<QM>(rv, p, pages, h, kb, kend, tid);
  convert_k_entry<QM, K2, Image>(img, tid, rk.w[0], u32x2{rk.w[1].x, rk.w[1].y}, K2 ? rk.w[1].z : 0u, kb, kend, cst);
  convert_v8<QM, Image>(img + KV, rv, kb, kend, cst, tid);
  __syncthreads();
  u32x4* out = reinterpret_cast<u32x4*>(images + (static_cast<long long>(blockIdx.y) * gridDim.x + blockIdx.x) * Image::BYTES);
#pragma unroll
  for (int i = 0; i < Image::BYTES / 16 / 256; ++i) out[tid + 256 * i] = reinterpret_cast<const u32x4*>(img)[tid + 256 * i];
}

// ------------------------------------------------------------------------------------------------ attention
struct SmemI {
  alignas(16) uint8_t kt[3][KV];                       // K(k) in k mod 3
  alignas(16) uint8_t vt[3][KV];
};
static_assert(256 * QROW <= 6 * KV, "q staging aliases the tiles");

// A matrix slot: O^T += V^T P^T against the V^T image at `vt` (its operands of the first two 16-key steps are in `va` already),
// then the scores minus the row's reference (qk8, mq_prefill.hip) against the K image at `kt`.  One stream of 32 matrix
// instructions, each with the request of the operand that is needed eight instructions later beside it: LDS feeds one
// operand per matrix instruction and SIMD, no more.
DEVI void request_v(const uint8_t* vt, const int (&voff)[4], u32x4 (&va)[2][4]) {
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
#pragma unroll
    for (int db = 0; db < 4; ++db) va[ks][db] = *reinterpret_cast<const u32x4*>(vt + voff[ks] + 32 * db * 128);
}
DEVI void matrix_slot(const uint8_t* vt, const int (&voff)[4], const u32x4 (&va)[2][4], const u32x4 (&pb)[4], f32x16 (&o)[4],
                      const uint8_t* kt, const int (&koff)[8], const u32x4 (&qf)[8], f32x16 (&sacc)[2], const f32x16& init) {
  u32x4 vb[2][4], a0[8], a1[8];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
#pragma unroll
    for (int db = 0; db < 4; ++db) vb[ks][db] = *reinterpret_cast<const u32x4*>(vt + voff[2 + ks] + 32 * db * 128);
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    a0[s] = *reinterpret_cast<const u32x4*>(kt + koff[s]);
    a1[s] = *reinterpret_cast<const u32x4*>(kt + koff[s] + 32 * 256);
  }
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
#pragma unroll
    for (int db = 0; db < 4; ++db)
      o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(as_h8(ks < 2 ? va[ks & 1][db] : vb[ks & 1][db]), as_h8(pb[ks]), o[db], 0, 0, 0);
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    sacc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(as_h8(a0[s]), as_h8(qf[s]), s ? sacc[0] : init, 0, 0, 0);
    sacc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(as_h8(a1[s]), as_h8(qf[s]), s ? sacc[1] : init, 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < 24; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);     // a matrix instruction
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);     // an LDS read
  }
  __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
}

// 1 KB of an image to LDS by one wavefront: lane l's 16 bytes to `dst` + 16 l, without a register in between
DEVI void copy_1k(const uint8_t* src, uint8_t* dst, int lane) {
  __builtin_amdgcn_global_load_lds(reinterpret_cast<const __attribute__((address_space(1))) void*>(reinterpret_cast<uintptr_t>(src + 16 * lane)),
                                   reinterpret_cast<__attribute__((address_space(3))) void*>(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(dst))), 16, 0, 0);
}

// End of a slot, nothing moves across.  Of a matrix slot: this wavefront's reads of LDS have returned (READS), so that what they
// read may be overwritten; of the slot that copy sets are waited for: all but its PENDING newest copies have landed.
template <bool READS, int PENDING> DEVI void slot_end() {
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (READS && PENDING >= 0) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(PENDING < 0 ? 0 : PENDING) : "memory");
  else if constexpr (PENDING >= 0) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(PENDING < 0 ? 0 : PENDING) : "memory");
  else if constexpr (READS) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  else asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Workgroup = (head of the group, work item), 256 rows, eight wavefronts in two groups half a block apart as in k_mq8:
//   slot 2k      group A: O += P(k-1) V(k-1), S = K(k) q      group B: softmax(k-1)
//   slot 2k + 1  group A: softmax(k)                          group B: O += P(k-1) V(k-1), S = K(k) q
// Copy set k is K(k) and V(k-1): what slot 2k is the first to multiply with.  Set k + 2 is requested in slot 2k, whose
// buffers (k + 2 mod 3: K(k-1), V(k-2)) were read last in slot 2k - 1.  The end of slot 2k waits for set k + 1, which leaves
// set k + 2 -- four copies a wavefront -- in flight, so that either group requests the first operands of its next matrix
// slot at the end of its softmax slot: group A in slot 2k + 1 those of V(k), group B in slot 2k those of V(k-1).
// Heads are the grid's fastest index: workgroups go round robin to the eight XCDs, so an XCD's L2 sees few heads and the
// tiles of a request find each other's blocks there.
__global__ void __launch_bounds__(512, 1) k_mq_images(const Params p, const int* __restrict__ tile_block, int nblocks, int head0,
                                                      const uint8_t* __restrict__ images) {
  constexpr int NT = 512, ROWS = 256;
  extern __shared__ __align__(16) uint8_t lds[];
  SmemI& S = *reinterpret_cast<SmemI*>(lds);
  const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int grp = wv >> 2;
  const int item = blockIdx.y, h = head0 + blockIdx.x;
  const Work work(p, item, ROWS);
  const int kb0 = work.block0, nb = work.block1 - work.block0;
  const uint8_t* const first = images + (static_cast<long long>(blockIdx.x) * nblocks + tile_block[p.items[ITEM_INTS * item]] + kb0) * Image::BYTES;

  const int r = 32 * wv + l32;
  const bool rvalid = work.has_row(r);
  const int lim = rvalid ? work.last_key(work.token_of(r)) : -1;
  u32x4 qf[8];
  {
    QRows<NT, ROWS> rows;
    rows.request(p, work, h, D, 0, tid);
    rows.store(lds, work, tid);
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const int dA = 32 * (s >> 1) + 4 * (2 * (s & 1) + hh);
    const u32x2 a = *reinterpret_cast<const u32x2*>(lds + r * QROW + 2 * dA);
    const u32x2 b = *reinterpret_cast<const u32x2*>(lds + r * QROW + 2 * (dA + 16));
    qf[s] = u32x4{(a.x & 0xFFFFu) | (a.y << 16), (b.x & 0xFFFFu) | (b.y << 16),
                  (a.x >> 16) | (a.y & 0xFFFF0000u), (b.x >> 16) | (b.y & 0xFFFF0000u)};
  }
  f32x16 o[4];
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
  float mrow = -INFINITY, lrow = 0.f;                  // mrow: the row's reference
  const int lim_min = -static_cast<int>(wave_max64(-static_cast<float>(rvalid ? lim : -1)));   // exact: key indices < 2^24
  auto is_full = [&](int kb) { return kb * BN >= p.kmin && kb * BN + BN - 1 <= lim_min; };
  f32x16 sacc[2];
  u32x4 pb[4];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) sacc[t][i] = -INFINITY;
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) pb[ks] = u32x4{0u, 0u, 0u, 0u};
  // lane offsets inside a tile of the operand of step s (K: row l32, piece 2 s + hh; V^T: row l32, run 2 ks + hh)
  int koff[8], voff[4];
#pragma unroll
  for (int s = 0; s < 8; ++s) koff[s] = Image::k(l32, 2 * s + hh);
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) voff[ks] = Image::v(l32, 2 * ks + hh);
  // wavefront wv copies the pieces wv and wv + 8 of both tiles
  auto copy_tile = [&](const uint8_t* src, uint8_t* dst) {
    copy_1k(src + 1024 * wv, dst + 1024 * wv, lane);
    copy_1k(src + 1024 * (wv + 8), dst + 1024 * (wv + 8), lane);
  };
  auto copy_set = [&](int k) {                         // K(k) (past the last block: that one again, for nobody) and V(k - 1)
    copy_tile(first + static_cast<long long>(min(k, nb - 1)) * Image::BYTES, S.kt[k % 3]);
    copy_tile(first + static_cast<long long>(k - 1) * Image::BYTES + KV, S.vt[(k - 1) % 3]);
  };
  __syncthreads();                                     // the q staging is no longer read
  // The pipeline starts through harmless work: probabilities 0 against a zeroed V^T tile, scores of -inf.
  for (int i = tid; i < KV / 16; i += NT) reinterpret_cast<u32x4*>(S.vt[2])[i] = u32x4{0u, 0u, 0u, 0u};
  if (nb > 0) {
    copy_tile(first, S.kt[0]);
    slot_end<true, 0>();                               // K(0), the zeros
    copy_set(1);
    auto pin = [&]() {                                 // (the packed probabilities stay in front of the barrier: k_mq8)
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) asm volatile("" : "+v"(pb[ks]));
    };
    f32x16 init;                                       // -reference, what the score accumulators start from
    auto set_init = [&]() {                            // (before the barrier too: no vector work in a matrix slot)
      const float c0 = mrow == -INFINITY ? 0.f : -mrow;
#pragma unroll
      for (int i = 0; i < 16; ++i) init[i] = c0;
      asm volatile("" : "+v"(init));
    };
    set_init();
    u32x4 va[2][4];
    int cur = 0, prev = 2;                             // k mod 3, k - 1 mod 3
    if (grp == 0) {
      request_v(S.vt[2], voff, va);
      for (int k = 0; k < nb; ++k) {
        const bool more = k + 2 <= nb;
        if (more) copy_set(k + 2);
        __builtin_amdgcn_sched_barrier(0);
        matrix_slot(S.vt[prev], voff, va, pb, o, S.kt[cur], koff, qf, sacc, init);
        if (more) slot_end<true, 4>(); else slot_end<true, 0>();
        softmax8(sacc, pb, o, mrow, lrow, is_full(kb0 + k), kb0 + k, lim, p.kmin, hh);
        pin();
        set_init();
        __builtin_amdgcn_sched_barrier(0);
        request_v(S.vt[cur], voff, va);
        slot_end<false, -1>();
        prev = cur; cur = cur == 2 ? 0 : cur + 1;
      }
    } else {
      for (int k = 0; k < nb; ++k) {
        const bool more = k + 2 <= nb;
        if (more) copy_set(k + 2);
        __builtin_amdgcn_sched_barrier(0);
        softmax8(sacc, pb, o, mrow, lrow, is_full(kb0 + k - 1), kb0 + k - 1, lim, p.kmin, hh);
        pin();
        set_init();
        __builtin_amdgcn_sched_barrier(0);
        request_v(S.vt[prev], voff, va);
        if (more) slot_end<false, 4>(); else slot_end<false, 0>();
        matrix_slot(S.vt[prev], voff, va, pb, o, S.kt[cur], koff, qf, sacc, init);
        slot_end<true, -1>();
        prev = cur; cur = cur == 2 ? 0 : cur + 1;
      }
      softmax8(sacc, pb, o, mrow, lrow, is_full(kb0 + nb - 1), kb0 + nb - 1, lim, p.kmin, hh);
      request_v(S.vt[prev], voff, va);
    }
    u32x4 vb[2][4];                                    // the last block's values: V(nb - 1) in `prev`
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int db = 0; db < 4; ++db) vb[ks][db] = *reinterpret_cast<const u32x4*>(S.vt[prev] + voff[2 + ks] + 32 * db * 128);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int db = 0; db < 4; ++db)
        o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(as_h8(ks < 2 ? va[ks & 1][db] : vb[ks & 1][db]), as_h8(pb[ks]), o[db], 0, 0, 0);
  }
  const float l = lrow + __shfl_xor(lrow, 32, 64);
  if (rvalid) {
    const long long base = (static_cast<long long>(item) * p.Hkv + h) * ROWS + r;
    float* op = p.opart + base * D;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4)
        *reinterpret_cast<float4*>(op + 32 * db + 8 * q4 + 4 * hh) =
            make_float4(o[db][4 * q4], o[db][4 * q4 + 1], o[db][4 * q4 + 2], o[db][4 * q4 + 3]);
    if (hh == 0) *reinterpret_cast<float2*>(p.ml + base * 2) = make_float2(mrow, l);
  }
}

}  // namespace

int image_bytes() { return Image::BYTES; }

int images_attn_launch(const Params& p, int nitems, int konly, const int* tile_block, const int* recs, int nblocks, uint8_t* images,
                       int heads, hipStream_t st) {
  static const hipError_t set = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_mq_images), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                    static_cast<int>(sizeof(SmemI)));
  if (set != hipSuccess) return -1;
  const auto make = (konly & 2) ? ((konly & 1) ? k_tile_images<QM_ASYM2, true> : k_tile_images<QM_ASYM2, false>)
                                : ((konly & 1) ? k_tile_images<QM_ASYM4, true> : k_tile_images<QM_ASYM4, false>);
  for (int h0 = 0; h0 < p.Hkv; h0 += heads) {
    const int n = p.Hkv - h0 < heads ? p.Hkv - h0 : heads;
    hipLaunchKernelGGL(make, dim3(nblocks, n), dim3(256), 0, st, p, recs, h0, images);
    if (hipPeekAtLastError() != hipSuccess) return -1;
    hipLaunchKernelGGL(k_mq_images, dim3(n, nitems), dim3(512), sizeof(SmemI), st, p, tile_block, nblocks, h0, images);
    if (hipPeekAtLastError() != hipSuccess) return -1;
  }
  return 0;
}

}  // namespace frmq
