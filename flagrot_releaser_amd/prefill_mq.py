"""Front end of libflagrot_mq.so (gfx950): multi-query prefill over a prefix that already sits in FlagRot pages.

The calls a step makes, in order (names and arguments as in the reference plugin's module of the same name,
integrations/vllm_flagrot/vllm_flagrot/prefill_mq.py, so code written against it runs unchanged; head dim 128, or 256 with build_plan(D=256)):

  plan = build_plan(reqs, G, Hkv, shift, device)   once per step, shared by all layers: which 64-key blocks each tile of
                                                   query rows reads, cut into work items, as one int32 device buffer
  q16  = prep_q(q, qscale, G, plan.idx, ...)       query rows -> FP16 in the basis the keys are stored in, pre-scaled
  op, ml = attn(q16, pool, bt, plan, G, shift, konly)   one workgroup per (item, KV head): unnormalised partial outputs
  merge(plan, op, ml, G, out=...)                  the items of a tile combined into rows of the layer output
  win_gather(...), bf_merge(...)                   BF16 window / sink rows: gathered, and folded into the page part

The buffer layout is the library's contract: 9 ints per tile, 4 per item, then the output row of every compact row.
Launches are asynchronous on torch's current HIP stream.  Without the library there is no result: nothing here falls back.
"""
from __future__ import annotations

import math
import os
from dataclasses import dataclass

import numpy as np
import torch

from .native import Library, current_stream

D, PAGE, BN = 128, 16, 64
TILE_INTS, ITEM_INTS = 9, 4
# columns of a tile record / an item record (the device code reads them by these positions)
T_BTROW, T_CROW, T_OROW, T_NTOK, T_POS0, T_NKEYS, T_ITEM0, T_NITEMS, T_EXT = range(TILE_INTS)
I_TILE, I_KB0, I_KB1, I_PAD = range(ITEM_INTS)
LOG2E = 1.4426950408889634
ABI = 7
KERNEL = int(os.environ.get("FLAGROT_MQ_KERNEL", "0"))        # 0: pick_kernel per plan
# kernel ids 1 | 2 | 3 are the reference's (64 / 128 / 128 rows per tile); 4 exists on this build only: 256 rows, eight
# wavefronts in two groups that alternate between the matrix and the vector half of a block
KROWS = {1: 64, 2: 128, 3: 128, 4: 256}                       # q rows per tile (= per workgroup)
KCTAS = {1: 4, 2: 2, 3: 2, 4: 1}                              # resident workgroups per CU assumed by the planner

NATIVE = Library("mq", "FLAGROT_MQ_LIB", "frmq_abi_version", ABI, "frmq_last_error", {
    "frmq_last_error": "->s",
    "frmq_smem_bytes": "",
    "frmq_prep_q": "p i l p i i i p p f p i p",
    "frmq_attn": "p p l p l p p i i i i i p p i i p i",
    "frmq_image_bytes": "",
    "frmq_attn_images": "p p l p l p p i p p i i i i i p i p p p i",
    "frmq_merge": "p i p p i i i p l i p l i p",
    "frmq_win_gather": "p i p p p l p l i p p i p",
    "frmq_bf_merge": "i i i p l p p p p p p p p p i i f p l i p",
})
EXPORTS = NATIVE.exports


def lib():
    """the ctypes handle (the library is built first when it is missing or older than its sources)"""
    return NATIVE.dll


def available() -> bool:
    try:
        NATIVE.dll
    except Exception:  # noqa: BLE001
        return False
    return True


def pick_kernel(reqs, G: int) -> int:
    """256-row tiles when some request fills them to three quarters (rows = new tokens x G), else the 128-row kernel."""
    most = max((q1 - q0 for (_, q0, q1, _, _) in reqs), default=0) * G
    return 4 if most >= 192 else 3


_CUS: dict = {}


def num_sms(device) -> int:
    """compute units of `device` (asked once per device)"""
    name = str(device)
    if name not in _CUS:
        _CUS[name] = torch.cuda.get_device_properties(device).multi_processor_count
    return _CUS[name]


@dataclass
class Plan:
    """One step's work list.  `buf` (int32, on the device) holds, back to back: the tile records [ntiles, 9], the item
    records [nitems, 4], the output row of each of the m compact query rows and, with nblocks, every tile's first block record
    [ntiles] and the block records [nblocks, 4] (image_arrays).  A tile record is (block-table row,
    first compact row, first output row, tokens, position of the first token, page keys of the request, first item,
    items, extra visible key or a large negative number); an item record is (tile, first key block, end key block, 0).
    `reqs` keeps the requests in the order their rows were compacted; `rows` is the number of query rows a workgroup of
    kernel `kernel` holds; keys below `kmin` are left to the BF16 sink part."""
    ntiles: int
    nitems: int
    m: int
    buf: torch.Tensor
    reqs: list
    kernel: int = 3
    rows: int = 128
    D: int = 128
    kmin: int = 0
    nblocks: int = 0                # blocks whose tile images key-only pages make first; 0: every tile converts what it reads

    def _span(self, start: int, count: int):
        return self.buf[start:start + count]

    @property
    def tiles(self):
        return self._span(0, self.ntiles * TILE_INTS)

    @property
    def items(self):
        return self._span(self.ntiles * TILE_INTS, self.nitems * ITEM_INTS)

    @property
    def idx(self):
        return self._span(self.ntiles * TILE_INTS + self.nitems * ITEM_INTS, self.m)

    @property
    def tile_block(self):
        """the first block record of every tile"""
        return self._span(self.ntiles * TILE_INTS + self.nitems * ITEM_INTS + self.m, self.ntiles)

    @property
    def block_recs(self):
        return self._span(self.ntiles * (TILE_INTS + 1) + self.nitems * ITEM_INTS + self.m, self.nblocks * BLOCK_INTS)


_W = os.environ.get("FLAGROT_MQ_WAVES")                         # grid target: WAVES x the resident workgroups of the GPU;
WAVES = float(_W) if _W else None                               # unset: split_items searches the number of rounds
MIN_BLOCKS = int(os.environ.get("FLAGROT_MQ_MIN_BLOCKS", "4"))  # >= 4 x 64 keys per work item
NO_EXT = -(1 << 30)


ITEM_OVERHEAD = 12     # blocks: what an item costs besides its key blocks (q staging, first tile, partials, its share of the merge)


def split_items(nb, Hkv: int, slots: int, waves: float | None, min_blocks: int):
    """items per tile.  nb [tiles] = key blocks per tile; slots = resident workgroups of the GPU.  waves given: items of
    about sum(nb) Hkv / (waves slots) blocks.  waves None: the number of rounds (1 .. 8) with the smallest estimated
    makespan rounds x (longest item + ITEM_OVERHEAD), where an item count that leaves the last round partly empty pays
    for the whole round.  Every tile's items have equal length (+- 1 block) and at least min_blocks blocks."""
    nb = np.asarray(nb, dtype=np.int64)
    if nb.size == 0:
        return nb
    total = int(nb.sum()) * Hkv

    def split(bpi):
        n = np.maximum(1, np.rint(nb / max(bpi, 1)).astype(np.int64))
        return np.maximum(1, np.minimum(n, np.maximum(nb // max(min_blocks, 1), 1)))

    if waves is not None:
        return split(max(min_blocks, -(-total // max(int(waves * slots), 1))))
    best = None
    for w in range(1, 9):
        n = split(max(min_blocks, -(-total // (w * slots))))
        rounds = -(-int(n.sum()) * Hkv // slots)
        cost = rounds * (int((-(-nb // n)).max()) + ITEM_OVERHEAD)
        if best is None or cost < best[0]:
            best = (cost, n)
    return best[1]


def plan_arrays(reqs, G: int, Hkv: int, shift: int, ncu: int, kernel: int = KERNEL or 3, waves: float | None = WAVES,
                min_blocks: int = MIN_BLOCKS, ext: dict | None = None):
    """The planner's arithmetic on the host: (tile records int32 [nt, 9], item records int32 [ni, 4], output row per
    compact row int32 [m], query rows per tile).

    A request is (block-table row, q0, q1, L, s): batch rows q0 .. q1 - 1 hold the tokens at positions s .. L - 1.  A
    token at position i reads the page keys j <= i - shift; every token of request r also reads j <= ext[r] when ext
    names r.  Tiles take rows // G consecutive tokens of one request (all G query heads of a token stay together); a
    tile reads keys [0, kend) with kend set by its last token, in 64-key blocks shared out over equal items
    (split_items).  Tiles are emitted longest first, so that the short ones fill the last round of workgroups."""
    rows = KROWS[kernel]
    per_tile = rows // G
    R = np.asarray(list(reqs), dtype=np.int64).reshape(-1, 5)
    bt_row, q0, q1, length, start = (R[:, c] for c in range(5))
    fresh = q1 - q0                                               # new tokens per request
    reach = np.array([ext.get(int(r), NO_EXT) if ext else NO_EXT for r in bt_row], dtype=np.int64)
    keys_of_req = np.maximum(np.maximum(length - shift, reach + 1), 0)
    compact0 = np.cumsum(fresh) - fresh                           # first compact row of each request
    tiles_of_req = -(-fresh // per_tile)
    owner = np.repeat(np.arange(R.shape[0]), tiles_of_req)        # request of every tile
    nth = np.arange(owner.size) - np.repeat(np.cumsum(tiles_of_req) - tiles_of_req, tiles_of_req)
    tok0 = nth * per_tile                                         # first token of the tile inside its request
    ntok = np.minimum(per_tile, fresh[owner] - tok0)
    pos0 = start[owner] + tok0
    kend = np.clip(np.maximum(pos0 + ntok - shift, reach[owner] + 1), 0, keys_of_req[owner])
    blocks = -(-kend // BN)

    by_length = np.argsort(-blocks, kind="stable")
    owner, tok0, ntok, pos0, blocks = (a[by_length] for a in (owner, tok0, ntok, pos0, blocks))
    items_of_tile = split_items(blocks, Hkv, KCTAS[kernel] * ncu, waves, min_blocks)
    first_item = np.cumsum(items_of_tile) - items_of_tile

    T = np.empty((owner.size, TILE_INTS), dtype=np.int32)
    T[:, T_BTROW], T[:, T_CROW], T[:, T_OROW] = bt_row[owner], compact0[owner] + tok0, q0[owner] + tok0
    T[:, T_NTOK], T[:, T_POS0], T[:, T_NKEYS] = ntok, pos0, keys_of_req[owner]
    T[:, T_ITEM0], T[:, T_NITEMS], T[:, T_EXT] = first_item, items_of_tile, reach[owner]

    tile_of_item = np.repeat(np.arange(owner.size), items_of_tile)
    part = np.arange(tile_of_item.size) - first_item[tile_of_item]       # which share of its tile an item is
    nb, ni = blocks[tile_of_item], items_of_tile[tile_of_item]
    I = np.zeros((tile_of_item.size, ITEM_INTS), dtype=np.int32)
    I[:, I_TILE] = tile_of_item
    I[:, I_KB0] = part * nb // ni                                 # shares of nb blocks differ by one block at most
    I[:, I_KB1] = (part + 1) * nb // ni

    out_row = np.repeat(q0 - compact0, fresh) + np.arange(int(fresh.sum()))
    return T, I, out_row.astype(np.int32), rows


BLOCK_INTS = 4
IMAGE = 32768                   # bytes of a block's tile images (one KV head)
# Key-only pages of heavy calls take the images: their conversion (rotations undone per token and block) is paid once per
# request instead of once per query tile, for 32 KB written per block and head and two more launches.  us direct / by images,
# 8 KV heads, 4-bit key-only pages: 4 requests x 16 tiles over 16 k 1345 / 1046 + 72 for the images; 1 x 16 tiles over 8 k
# (17 k reads of a block by a tile and head, 15 per block) 189 / 164; 4 x 6 over 8 k (25 k, 6) 282 / 260; 4 x 16 over 1 k
# (12.5 k, 12) 176 / 138; 8 x 4 over 4 k (17 k, 4) 174 / 168; below: 4 x 8 over 1 k (5 k, 7) 69 / 71, 1 x 8 over 2 k (2 k, 7)
# 42 / 43, 4 x 2 over 1 k (1 k, 2) 27 / 40.  Static pages convert fast enough to lose (1 x 16 over 8 k 155 / 165).
# The same line on 2-bit pages and on ranks of 4 and 2 heads (groups of 4 and 8, 150 plans on it: 1.00 to 1.72 times as fast):
# 2-bit, 8 heads 4 x 16 over 4 k 363 / 302, 1 x 16 over 8 k 168 / 161; 4 heads, 4-bit 2 x 64 over 2 k 389 / 275, 2-bit 2 x 16
# over 8 k 167 / 156; 2 heads, 4-bit 4 x 8 over 12 k 127 / 119, 2-bit 123 / 118.  Where the images have room for some of the heads
# only, several passes may need more rounds of workgroups than one launch for all heads: then the launch stays (4 x 8 over 12 k,
# 32 items x 8 heads in one round, room for 7 heads: 460 / 686, 2-bit 447 / 677).
IMAGE_READS = int(os.environ.get("FLAGROT_MQ_IMAGE_READS", "12000"))            # reads of a block by a tile and KV head
IMAGE_REUSE = float(os.environ.get("FLAGROT_MQ_IMAGE_REUSE", "4"))              # ... per block
IMAGE_BYTES = int(os.environ.get("FLAGROT_MQ_IMAGE_BYTES", str(192 << 20)))     # room for images per call: they stay in the caches


def image_arrays(T, I):
    """Which blocks of which requests the tiles read: (first block record of every tile int32 [nt], block records int32
    [nblocks, 4] = (block-table row, block, page keys of the request, 0)).  Tiles of one request share its blocks."""
    reach = I[T[:, T_ITEM0] + T[:, T_NITEMS] - 1, I_KB1]                                            # blocks a tile reads
    names, owner = np.unique((T[:, T_BTROW].astype(np.int64) << 32) | T[:, T_NKEYS], return_inverse=True)
    blocks = np.zeros(names.size, dtype=np.int64)
    np.maximum.at(blocks, owner, reach)
    first = np.cumsum(blocks) - blocks
    recs = np.zeros((int(blocks.sum()), BLOCK_INTS), dtype=np.int32)
    recs[:, 0], recs[:, 2] = np.repeat(names >> 32, blocks), np.repeat(names & 0xFFFFFFFF, blocks)
    recs[:, 1] = np.arange(len(recs)) - np.repeat(first, blocks)
    return first[owner].astype(np.int32), recs


def image_rounds(nitems: int, Hkv: int, heads: int, ncu: int) -> int:
    """rounds of workgroups (one per CU) of all passes over the images, `heads` KV heads a pass"""
    whole, rest = divmod(Hkv, heads)
    return whole * -(-nitems * heads // ncu) + -(-nitems * rest // ncu)


def heads_per_pass(nitems: int, nblocks: int, Hkv: int, ncu: int) -> int:
    """KV heads per pass over the images: of what IMAGE_BYTES have room for, the number with the fewest rounds of workgroups
    over all passes, the larger one on ties"""
    room = min(Hkv, max(1, IMAGE_BYTES // (nblocks * IMAGE)))
    return min(range(room, 0, -1), key=lambda n: image_rounds(nitems, Hkv, n, ncu))


def image_heads(plan, Hkv: int, ncu: int) -> int:
    return heads_per_pass(plan.nitems, plan.nblocks, Hkv, ncu)


def image_room(size: int, device):
    """memory for the images of a call, or None where the device has none left (a cache of pages may hold all the rest)"""
    try:
        return torch.empty(size, dtype=torch.uint8, device=device)
    except torch.OutOfMemoryError:
        return None


def build_plan(reqs, G: int, Hkv: int, shift: int, device, sink: int = 0, kernel: int | None = None,
               waves: float | None = None, min_blocks: int | None = None, D: int = D, ext: dict | None = None, konly: bool = True) -> Plan:
    """plan_arrays for the GPU `device`, uploaded as one int32 tensor.  sink: keys [0, sink) are masked in the kernel
    (the BF16 sink part covers them); kernel None: pick_kernel.  konly False: the pages are of a static format, which has no use
    for the block records of heavy calls (the plan does for either kind with them; 64 tiles over 16 k: 145 us of host time
    without, 210 with)."""
    assert D in (128, 256), D
    reqs = list(reqs)
    kernel = 3 if D == 256 else kernel or KERNEL or pick_kernel(reqs, G)     # head dim 256: one kernel, 128-row tiles
    T, I, out_row, rows = plan_arrays(reqs, G, Hkv, shift, num_sms(device), kernel, WAVES if waves is None else waves,
                                      MIN_BLOCKS if min_blocks is None else min_blocks, ext)
    parts, nblocks, reads = [T.ravel(), I.ravel(), out_row], 0, int((I[:, I_KB1] - I[:, I_KB0]).sum())
    if konly and kernel == 4 and reads * Hkv >= IMAGE_READS:
        tile_block, recs = image_arrays(T, I)
        n, ncu = len(recs), num_sms(device)
        if (n * IMAGE <= IMAGE_BYTES and reads >= IMAGE_REUSE * n
                and image_rounds(len(I), Hkv, heads_per_pass(len(I), n, Hkv, ncu), ncu) <= image_rounds(len(I), Hkv, Hkv, ncu)):
            parts += [tile_block, recs.ravel()]
            nblocks = n
    packed = torch.from_numpy(np.concatenate(parts))
    return Plan(ntiles=len(T), nitems=len(I), m=len(out_row), buf=packed.to(device), reqs=reqs, kernel=kernel, rows=rows,
                D=D, kmin=int(sink), nblocks=nblocks)


# ------------------------------------------------------------------------------------------------ launches
def _rows_are_heads(t: torch.Tensor, Dh: int) -> bool:
    """[n, H, Dh] with the H rows of a token back to back (the token stride is free)"""
    return t.stride(2) == 1 and t.stride(1) == Dh


def prep_q(q: torch.Tensor, qscale: float, G: int, idx: torch.Tensor | None = None, kfull=None, kmask=None):
    """q [n, Hq, 128] (bf16 or fp32) -> FP16 [m, Hq, 128] ready for `attn`: row c is q[idx[c]] (every row when idx is
    None), taken into the basis its KV head's keys are stored in and multiplied by qscale (softmax scale x log2 e).
    Static formats pass kfull uint8 [Hkv] (1: the whole head is stored as H_128 x / 8) and kmask uint8 [Hkv, 4] (1: that
    32-channel group is stored as orthonormal H32 x)."""
    n, Hq, Dh = q.shape
    assert Dh in (128, 256), "head dim 128 or 256"
    assert q.dtype in (torch.bfloat16, torch.float32) and _rows_are_heads(q, Dh)
    assert idx is None or idx.dtype == torch.int32
    m = n if idx is None else idx.numel()
    q16 = q.new_empty((m, Hq, Dh), dtype=torch.float16)
    NATIVE.run("frmq_prep_q", q, q.dtype == torch.float32, q.stride(0), idx, m, Hq, G, kfull, kmask, float(qscale), q16,
               Dh, current_stream())
    return q16


def attn(q16, pool, bt, plan: Plan, G: int, shift: int, konly: bool, int2: bool = False):
    """The page part of the attention, still split by item: (opart fp32 [items, Hkv, rows, D], unnormalised;
    ml fp32 [items, Hkv, rows, 2] = running maximum in log2 units and sum).  pool uint8 [pages, Hkv, chunk bytes] (at
    head dim 256 a chunk is two 128-d half chunks), bt int32 block table, q16 from prep_q; konly: key-only-rotated page
    kinds; int2: 2-bit codes (80-byte tokens per 128 dims).  Plans with block records: up to IMAGE_BYTES of device memory hold
    the images of their tiles during the call (a captured call's belong to its graph's pool); where they cannot be had, every
    tile converts what it reads."""
    Hkv, Dh = pool.shape[1], q16.shape[2]
    token_bytes = 80 if int2 else 144
    assert Dh == plan.D, (Dh, plan.D)
    assert pool.dtype == torch.uint8 and pool.stride(2) == 1 and pool.stride(1) == token_bytes * PAGE * (Dh // 128)
    assert bt.dtype == torch.int32 and bt.stride(1) == 1
    assert q16.dtype == torch.float16 and q16.is_contiguous() and q16.shape[1] == Hkv * G
    opart = q16.new_empty((plan.nitems, Hkv, plan.rows, Dh), dtype=torch.float32)
    ml = q16.new_empty((plan.nitems, Hkv, plan.rows, 2), dtype=torch.float32)
    heads = image_heads(plan, Hkv, num_sms(q16.device)) if konly and plan.nblocks else 0
    images = image_room(heads * plan.nblocks * IMAGE, q16.device) if heads else None
    if images is not None:
        NATIVE.run("frmq_attn_images", q16, pool, pool.stride(0), bt, bt.stride(0), plan.tiles, plan.items, plan.nitems,
                   plan.tile_block, plan.block_recs, plan.nblocks, Hkv, G, shift, int(konly) + 2 * int(int2), images, heads,
                   opart, ml, current_stream(), plan.kmin)
        return opart, ml
    NATIVE.run("frmq_attn", q16, pool, pool.stride(0), bt, bt.stride(0), plan.tiles, plan.items, plan.nitems, Hkv, G,
               shift, int(konly) + 2 * int(int2), opart, ml, plan.kernel, Dh, current_stream(), plan.kmin)
    return opart, ml


def merge(plan: Plan, opart, ml, G: int, out=None, fp32: bool = False, want_lse: bool = False):
    """Folds the items of every tile together.  fp32 False: bf16 rows written into `out`, a [n, Hq * 128] view of the
    layer output whose row r is batch row r; fp32 True: a new fp32 [m, Hq, 128] tensor in compact row order.  want_lse:
    also the natural-log sum of exponentials per (head, compact row), -inf where a row saw no key.
    Returns (rows written or created, lse or None)."""
    Hkv, Dh = opart.shape[1], opart.shape[3]
    Hq = Hkv * G
    lse = opart.new_empty((Hq, plan.m)) if want_lse else None
    if fp32:
        dst, dst_stride = opart.new_empty((plan.m, Hq, Dh)), Hq * Dh
    else:
        assert out is not None and out.dtype == torch.bfloat16 and out.stride(-1) == 1
        dst, dst_stride = out, out.stride(0)
    NATIVE.run("frmq_merge", plan.tiles, plan.ntiles, opart, ml, Hkv, G, plan.rows, dst, dst_stride, fp32, lse,
               plan.m if want_lse else 0, Dh, current_stream())
    return dst, lse


def ref_partial_lse_merge(parts):
    """torch statement of the merge of partial attentions: parts = [(o [n, H, D], lse [H, n] natural log)], an lse of
    -inf or +inf marks an empty part, and every row has a non-empty one.  fp32 [n, H, D]."""
    logs = []
    for _, lse in parts:
        lse = lse.float().masked_fill(torch.isposinf(lse), -math.inf)
        logs.append(lse.t().unsqueeze(-1))                               # [n, H, 1]
    top = torch.stack(logs).amax(0)
    weights = [torch.exp(lg - top) for lg in logs]
    mix = sum(o.float() * w for (o, _), w in zip(parts, weights))
    return mix / sum(weights)


# ------------------------------------------------------------------------------------------------ BF16 window / sink rows
def win_gather(map_, nk, sinkb, preb, kch, vch, Hkv, D):
    """Collects the K and V rows of the windowed attention call into two new contiguous bf16 [nk, Hkv, D] tensors.
    map_[d] = (source << 32) | row tells where row d comes from: source 0 = sinkb, 1 = preb (both [*, 2 Hkv, D], K heads
    first), 2 = this batch's rows kch / vch ([n, Hkv * D], any row stride)."""
    for src in (sinkb, preb):
        assert src is None or (src.dtype == torch.bfloat16 and src.is_contiguous())
    assert kch.dtype == torch.bfloat16 and kch.stride(-1) == 1 and vch.stride(-1) == 1
    kw = kch.new_empty((nk, Hkv, D))
    vw = kch.new_empty((nk, Hkv, D))
    NATIVE.run("frmq_win_gather", map_, nk, sinkb, preb, kch, kch.stride(0), vch, vch.stride(0), Hkv, kw, vw, D,
               current_stream())
    return kw, vw


def bf_merge(q, idx, o_p, lse_p, o_w, lse_w, sk, row_req, row_pos, sk_len, S, W, scale, out, Hkv):
    """Writes out[idx[c]] for every compact row c: the LSE-weighted mix of up to three parts.  Pages: o_p fp32
    [m, Hq, D] with lse_p [Hq, m].  Window: o_w bf16 [m, Hq, D] with lse_w [Hq, m], or None when W is 0.  Sinks:
    computed here from sk bf16 [requests, S, 2 Hkv, D] (original basis) over the keys j < min(S, sk_len[request]) that
    also satisfy j <= position - W, or None when S is 0.  q [n, Hq, D] are the batch's query rows; row_req / row_pos
    give request and position of each compact row."""
    m, Hq, Dh = o_p.shape
    assert o_p.is_contiguous() and lse_p.is_contiguous() and idx.dtype == torch.int64
    assert _rows_are_heads(q, Dh) and out.stride(-1) == 1
    NATIVE.run("frmq_bf_merge", m, Hq, Hkv, q, q.stride(0), idx, o_p, lse_p, o_w, lse_w, sk, row_req, row_pos, sk_len, S,
               W, float(scale), out, out.stride(0), Dh, current_stream())
