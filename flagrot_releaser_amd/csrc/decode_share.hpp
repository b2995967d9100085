// Split ranges of a batch of uneven sequences (head dim 256 decode): the B * nsplit workgroups of a (KV head, q tile) that the
// plan made for the longest sequence are shared out by the lengths, on the device, since only it knows them.  Every part takes
// at most m units of 64 tokens, m the smallest number (to 1 / 15 of its range) for which the parts of all sequences fit their
// places (p.share), or the plan's own:
// 16 sequences of 2048 ... 8192 tokens planned as 4 x 2048 get parts of at most 1472 instead, on 64 workgroups instead of 46.
// Even lengths give the plan's own ranges.  (Kernel of those 16 sequences, 4 KV heads of 256 in 4-bit pages, 6 query heads
// each: 53.8 -> 43.6 us; bound by two wavefronts per SIMD either way.)
#pragma once
#include "fr_common.hpp"
#include "fr_launch.hpp"

namespace fr {

struct Shares {
  int u, n, first;       // of sequence `lane`: units of 64 tokens, parts, the number of the first part
};
DEVI int ceil_div_units(int a, int m, float r) {                   // a, m <= 2^18, r = 1 / m to a few units: off by one at most
  const int x = a + m - 1;
  int q = static_cast<int>(static_cast<float>(x) * r);
  const int rem = x - q * m;
  q += rem >= m ? 1 : 0;
  return q - (rem < 0 ? 1 : 0);
}
DEVI int share_start(const DecodeParams& p) { return max(p.kv_start, 0) & ~63; }   // tokens below are no part's
DEVI int share_end(const DecodeParams& p, int b) { return min(p.seq_lens[b], p.nsplit * p.chunk); }

// inclusive sum over the lanes up to this one
DEVI int scan_lanes(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);  // from 1, 2, 4, 8 lanes below in the row of 16
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // the sum of the row below into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);  // of the first two rows into rows 2 and 3
  return v;
}

// for whole wavefronts; B <= 64, nsplit >= 2, chunk a multiple of 64, nsplit * chunk <= 2^24 (the launcher's rule).  Every
// workgroup of the launch waits for this: 16 candidates at once, the sequences over the four rows of lanes.
DEVI Shares share_parts(const DecodeParams& p, int lane) {
  Shares s;
  s.u = lane < p.B ? max(0, (share_end(p, lane) - share_start(p) + 63) >> 6) : 0;
  const int all = __builtin_amdgcn_readlane(scan_lanes(s.u), 63);
  // parts of m units: at least all / m of them and fewer than all / m + B, so m lies in [all / S, all / (S - B) + 1], and m of the
  // plan's own size need no more than its places
  const int S = p.share, cap = p.chunk >> 6;
  const int hi = S > p.B ? min(cap, all / (S - p.B) + 1) : cap, lo = min(hi, max(1, (all + S - 1) / S)), step = max(1, (hi - lo + 14) / 15);
  int m = min(hi, lo + step * (lane & 15));                        // candidate lane mod 16; the last one if none fits
  if (hi > lo) {
    const float r = __builtin_amdgcn_rcpf(static_cast<float>(m));
    int count = 0;
#pragma unroll 4
    for (int b = lane >> 4; b < ((p.B + 3) & ~3); b += 4) count += ceil_div_units(__shfl(s.u, b, 64), m, r);
    count += __shfl_xor(count, 16, 64);
    count += __shfl_xor(count, 32, 64);
    const int pick = __ffs(static_cast<int>(__ballot(count <= S) & 0x7FFFu) | 0x8000) - 1;
    m = __builtin_amdgcn_readlane(m, pick);
  } else {
    m = hi;
  }
  s.n = ceil_div_units(s.u, m, __builtin_amdgcn_rcpf(static_cast<float>(m)));
  s.first = scan_lanes(s.n) - s.n;
  return s;
}

// part number `slot` -> its sequence and tokens [lo, hi); false: there is no such part
DEVI bool share_of(const DecodeParams& p, int lane, int slot, int& b, int& lo, int& hi) {
  const Shares s = share_parts(p, lane);
  b = __popcll(__ballot(lane < p.B && s.first <= slot)) - 1;       // (sequences without parts begin where the next one does)
  const int u = __builtin_amdgcn_readlane(s.u, b), n = __builtin_amdgcn_readlane(s.n, b), k = slot - __builtin_amdgcn_readlane(s.first, b);
  if (k >= n) return false;
  const int per = (u + n - 1) / n, end = share_end(p, b);
  lo = max(share_start(p) + 64 * per * k, min(p.kv_start, end));
  hi = min(end, share_start(p) + 64 * per * (k + 1));
  return true;
}

}  // namespace fr
