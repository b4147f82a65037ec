"""What parts need from the machine: device, activation dtype, and the matrix product.

Matrix products ``x[M,K] @ w[N,K]^T``:
* float32 weights: the hand-written float kernels always (float operands, products and sums, no
  reduced-precision matrix mode), whatever the activation dtype.  This is the whole float32 path
  and also what keeps a tensor that a checkpoint stores in 32 bits exact in a bfloat16 run.  With float32
  activations whose rows lie in units of 16 bytes: up to 16 rows ops.gemv_f32 on a packed copy, more rows (from 9
  on where there is no such copy) ops.gemm_f32 (f32_plan chooses its tile and groups of K) or, from
  some 20 to 200 rows on, ops.gemm_split (the same products by three exact bfloat16 parts of each float; split_plan);
  everything else ops.gemv_skinny up to 8 rows and ops.gemm_tiled.
* bfloat16 weights, up to 64 rows (decode): the hand-written skinny kernel on the matrix cores that
  streams the weight once (where the width fits its registers: see ops.gemv_mfma_group_limit).  From
  17 rows on, the products that come as partial planes (output and down projection) and, from 33 rows
  on, the gated product run on the kernel whose wavefronts each stream their own stages of K through
  shared memory (ops.gemm_rows): with that many rows the activations cost as much traffic as the
  weights, and its loads never stop for a barrier (see rows_plan and gated_linear).
* bfloat16 weights, 65 to 256 rows, K up to 2048 and few columns (the output projection at the 1B
  width): ops.gemm_rows again, a block for every 64 rows (see mid_rows_ring).
* bfloat16 weights, 65 rows and more, narrow output and long K (the down projection of short
  prompts): partial planes from the hand-written matrix-core kernel (see mid_k_groups).
* bfloat16 weights, many rows (prefill): tiles of 256x256 and their halves (ops.gemm_duo) where their rounds are full enough, and
  with them what stands around a product: the gating of a gated feed-forward, the rotation and the page writes behind q/k/v, a
  gate's product beside gate and up (duo_product, duo_planes, duo_qkv, duo_beside and gated_linear hold the rules and both
  sides' times).  The gate/up product of short prompts whose tiles all run at once is ops.gemm_mfma's (gated_linear).
  Everything else is the library's product (hipBLASLt through torch), as the reference's engine leaves its matrix
  products to its tensor library (crates/burn-lm-llama/src/nn/attention/mha.rs:124-126).  With
  BURN_LM_AMD_FUSED_GATE_UP=1 gate and up run on ops.gemm_mfma for every prompt of 192 rows and more that no rule above takes;
  =0 leaves every product to the library.
"""
from __future__ import annotations

import functools
import os

import torch

from ..csrc import ops
from ..parts.base import Unscaled

SKINNY_MAX_ROWS = 8
MFMA_SKINNY_MAX_ROWS = 64
# The longest K one group of the row-ring product walks before the sum is better cut into partial planes,
# and up to which that product beats the library's at 65 to 256 rows (a block streams its stages of K one
# after another, so its time grows with K while the library's tiles get longer runs): measured at
# widths of 2048, 3072 and 4096.
RING_GROUP_K = 2048
# The shortest K a group keeps when a short K is cut for more blocks.
RING_MIN_GROUP_K = 512
# Numbers of groups that a skinny product's K may be cut into, the longest stretch of K a group gets where a
# finer cut is to be had, and the least share of the compute units that the last round of blocks should keep busy.
GROUP_CHOICES = (1, 2, 3, 4, 6, 8, 12, 16)
GROUP_MAX_K = 4096
GROUP_MIN_FILL = 0.6
# 65 to 256 rows: the longest K at which the row-ring product with a block for every 64 rows still beats the
# library's and the matrix-core kernel's planes (measured: ahead at 1536, 2048 and 2560, behind at 3072 and 4096).
RING_MID_K = 2560
# The longest K at which the fused q/k/v projection on the row ring beats the library's product followed by the
# rotation kernel (ahead at 5120 and below, 20-29 % behind at 8192).
RING_QKV_K = 6144
# The shortest K a group of the matrix-core kernel's partial planes keeps, and the most rows for which a product
# comes as such planes (every group writes a float32 plane of rows x columns that the next norm reads back: measured
# over whole prompts, 2-5 % faster up to 512 tokens and equal beyond).
MFMA_MIN_GROUP_K = 768
MID_PLANES_MAX_ROWS = 512
NARROW_MIN_GROUP_K = 256
# Rows for which the fused gate/up product is used when it is switched on (below, the library is
# ahead by far; above, its better rate on long runs of tiles has made up for the extra pass).
FUSED_GATE_UP_ROWS = (192, 4096)


def rows_plan(N, K, compute_units):
    """(groups of K, columns per block) for a product of 17 to 64 rows that may come as partial
    planes (ops.gemm_rows).  A group spans about RING_GROUP_K of K (measured at the 1B, 3B and 8B layer
    shapes: shorter groups write more planes than they gain, longer ones leave compute units
    idle); 32 columns per block where that gives at most one block per compute unit, else 64;
    and a short K is cut further, down to RING_MIN_GROUP_K, while the blocks still all run at once (a
    second, partial round costs more than the shorter walk along K gains: width 2560, 64 rows, two
    groups 6.8 us, four groups 8.8)."""
    groups = 1
    while groups < 8 and K // (groups * 2) >= RING_GROUP_K:
        groups *= 2
    columns = 32 if -(-N // 32) * groups <= compute_units else 64
    while groups < 8 and K // (groups * 2) >= RING_MIN_GROUP_K and -(-N // columns) * groups * 2 <= compute_units:
        groups *= 2
    return groups, columns


# Tiles of ops.gemm_f32: microseconds for a step of 32 along K of a block that has its compute unit to itself (the loads'
# latency shows), and per step and block where blocks share a unit (the matrix instructions' rate).  Measured with 17 to
# 2,048 rows at [3072, 2048], [2048, 2048], [16384, 2048], [2048, 8192], [5000, 1416].
F32_STEP_US = {(128, 128): (2.33, 2.0), (128, 64): (1.25, 1.0), (64, 128): (1.2, 1.0), (64, 64): (0.7, 0.5)}
F32_SHARE_US = 0.1
JOIN_BF16_WIDTH = 1024     # see Runtime.join_takes
F32_SKINNY_MAX_ROWS = 16
F32_SKINNY_GROUP_K = 2048
LAST_LEVEL_BYTES = 256 << 20      # the cache in front of the memory


def _planes_us(M, N, groups, planes):
    """What partial planes cost their reader: their bytes, and where that is a pass of its own its launch and its result's bytes."""
    return M * N * groups * 4 / 5e6 if planes else 3.0 + M * N * (groups + 1) * 4 / 5e6


@functools.lru_cache(maxsize=4096)      # a length asks for some ten; made anew at every product, each took 2 to 12 us of the host
def f32_plan(M, N, K, compute_units, planes=False, gated=False, added=False):
    """(tile, groups of K, microseconds) of ops.gemm_f32 that a sum of its parts' costs finds fastest: every unit works through
    its share of the blocks, and every plane of partial products is read once by the norm that adds it (planes) or by a pass that does
    (added: for results that have to be whole; few rows of few columns are a handful of blocks that each walk all of K otherwise).
    Against the best tile and groups of the sweep the choice is within 6 % from 250 rows on and within 20 % below."""
    best = None
    for (bm, bn), (alone, shared) in F32_STEP_US.items():
        if gated and bn != 128:
            continue
        tiles = -(-M // bm) * -(-N // (bn // 2 if gated else bn))
        for groups in (1, 2, 4, 8) if (planes or added) and not gated else (1,):
            if groups > 1 and K // groups < 128:
                continue
            steps = -(-K // groups // 32)
            per_unit = -(-tiles * groups // compute_units)
            us = 3.0 + steps * max(alone, per_unit * shared + F32_SHARE_US) + (_planes_us(M, N, groups, planes) if groups > 1 else 0.0)
            if best is None or us < best[2] * 0.999:
                best = ((bm, bn), groups, us)
    return best


# Tiles of ops.gemm_split: microseconds for a step of 32 along K of a block while few units are busy, and while all are (the card's
# power), and a block's first loads and last stores.  Measured on weights that come from memory (ten matrices in turn), 24 to 1,500
# rows, [16384, 2048] gated and not, [2048, 8192], [3072, 2048], [2048, 2048], [5120, 3072], [3072, 8192] in 1 to 8 groups.  The
# choice between both kernels' tiles and groups is within 2 % of the fastest in the mean and never more than 7 % behind what gemm_f32
# alone would take.
SPLIT_STEP_US = {(128, 256): (1.71, 2.3), (128, 128): (0.95, 1.29), (64, 256): (1.07, 1.44), (64, 128): (0.63, 0.82)}
SPLIT_BLOCK_US = 2.5


@functools.lru_cache(maxsize=4096)
def split_plan(M, N, K, compute_units, planes=False, gated=False, added=False):
    """(tile, groups of K, microseconds with the pass that makes the rows' parts) of ops.gemm_split, as f32_plan has them of
    ops.gemm_f32; None where it does not have the sizes."""
    if not ops.split_takes(M, N, K, gated):
        return None
    best = None
    for (bm, bn), (few, all_) in SPLIT_STEP_US.items():
        if gated and bn != 256:
            continue
        tiles = -(-M // bm) * -(-N // (bn // 2 if gated else bn))
        for groups in (1, 2, 4, 8) if (planes or added) and not gated else (1,):
            steps = -(-K // 128 // groups) * 4
            if groups > 1 and (K // groups < 256 or (groups - 1) * steps * 32 >= K):
                continue
            per_unit = -(-tiles * groups // compute_units)
            fill = tiles * groups / (per_unit * compute_units)
            us = 2.0 + per_unit * (SPLIT_BLOCK_US + steps * (few + (all_ - few) * fill)) + (_planes_us(M, N, groups, planes) if groups > 1 else 0.0)
            if best is None or us < best[2] * 0.999:
                best = ((bm, bn), groups, us)
    return best[0], best[1], best[2] + split_rows_us(M, K)


def split_rows_us(M, K):
    """The pass that makes the rows' parts, as fitted together with SPLIT_STEP_US and F32_STEP_US.  By itself, between the kernel that has stored the
    rows and the product, it takes 2.7 / 3.0 / 4.0 / 5.0 / 5.6 / 6.0 us for 17 / 64 / 128 / 200 / 500 / 1,000 rows of 2,048 and 3.3 / 3.9 / 4.7 / 5.5 /
    7.3 / 14 of 8,192; with these in its place the choice falls on the float instructions at 140 to 520 rows of [2048, 2048], [3072, 3072], [1024, 4096]
    and [3072, 2048], where they are 2 to 16 % slower (product, pass and the sum of the planes: 240 rows of [2048, 2048] 27.3 / 29.2, 520 49.8 / 58.0)."""
    return max(3.4, 2.3 + M * K * 10 / 7e6)


# ops.gemm_duo: what half a tile takes of a whole one's time (K = 2048 / 8192, all blocks at once: 22 of 38 us, 73 of 128), and how
# full the rounds of tiles must be for it to be the faster one: for a gated product (against the library's and the gating pass), for
# one round of halves of a plain one or of its planes (see gated_linear, duo_product and duo_planes).
DUO_HALF = 0.57
DUO_GATED_FILL = 0.62
DUO_GATED_LONE_FILL = 0.9
DUO_HALVES_FILL = 0.74
DUO_QKV_FILL = 0.62
DUO_HALVES_K = 8192
DUO_PLANES_FILL = 0.78
DUO_PLANES_K = 6144
DUO_FOURS_FILL = 0.6        # see Runtime.duo_part_planes
DUO_FIVES_FILL = 0.75


@functools.lru_cache(maxsize=4096)
def duo_plan(M, N, compute_units, gated=False, beside=0):
    """(whole tiles, rounds, fill) of ops.gemm_duo: the tiles that do not fill a round run as halves where that is shorter; rounds in
    the time of a whole tile; fill: the share of the rounds' time that works on rows and columns that exist."""
    tiles, tail = ops.gemm_duo_tiles(M, N, gated, beside)
    full, rest = divmod(tiles, compute_units)
    left = compute_units - rest if rest else 0            # units that a last, partial round of whole tiles leaves to the tail
    whole = full + (1 if rest else 0) + DUO_HALF * -(-max(0, tail - left) // compute_units)
    halves = full + DUO_HALF * -(-(2 * rest + tail) // compute_units)
    rounds = min(whole, halves)
    return tiles if whole <= halves else tiles - rest, rounds, M * (N / (32768.0 if gated else 65536.0) + beside / 65536.0) / compute_units / rounds


class FusedProjectionPlan:
    """Launch geometry of a projection that a part fuses with work of its own (Runtime.qkv_plan).
    kernel: "rows" (ops.gemm_rows_qkv_rope's geometry: `rows` rows staged per block, `columns` columns
    per block, weights as the checkpoint stores them) or "packed" (ops.gemv_qkv_rope's: the packed
    copy of the weights, all rows in registers)."""
    __slots__ = ("kernel", "columns", "rows")

    def __init__(self, kernel, columns=0, rows=0):
        self.kernel, self.columns, self.rows = kernel, columns, rows

    def __repr__(self):
        return f"FusedProjectionPlan({self.kernel!r}, columns={self.columns}, rows={self.rows})"

    def __eq__(self, other):
        return isinstance(other, FusedProjectionPlan) and (self.kernel, self.columns, self.rows) == (other.kernel, other.columns, other.rows)


class PackingRoom:
    """The memory that a runtime's float32 matrices may take a second time: an eighth of the device's (36 of 288 GB: every
    matrix of a model of 8 billion weights), and only while as much stays free.  The float32 kernels for few rows that read
    the checkpoint's layout serve the rest, as they serve matrices that have no packed form."""
    SHARE = 8

    def __init__(self, device):
        self.device, self.taken = device, 0

    def grant(self, size):
        free, total = torch.cuda.mem_get_info(self.device)
        free += torch.cuda.memory_reserved(self.device) - torch.cuda.memory_allocated(self.device)     # what torch holds unused
        if self.taken + size > total // self.SHARE or free - size < total // self.SHARE:
            return False
        self.taken += size
        return True

    def give_back(self, size):
        self.taken -= size


class LinearWeight:
    """A bound weight matrix [N, K] and, where the skinny product takes it, its copy packed for that
    product.  The copy is made when a product first asks for it (``packed``): an engine that only ever
    runs prompts and large batches never holds a matrix twice.  ``packable`` says whether there is one to
    be had; ``drop_packed()`` gives its memory back (it is made again on demand).
    room (float32 matrices): what grants the copy its memory.  Without it, or if the allocation fails all the
    same, ``packed`` is None and the matrix stays unpackable, so that every later step, recorded or not, takes the
    same kernels."""

    def __init__(self, w, packable=False, gated=False, packed=None, room=None):
        self.w, self.gated, self.room = w, gated, room
        self.packable = bool(packable) or packed is not None
        self._packed = packed
        self.shape, self.dtype = w.shape, w.dtype

    @property
    def packed(self):
        if self._packed is None and self.packable:
            if torch.cuda.is_current_stream_capturing():
                raise RuntimeError("a weight's packed copy would have to be made while a graph is being recorded; a step "
                                   "of this shape has to run once outside a recording first")
            if self.room is None:
                self._packed = ops.pack_weight(self.w, gated=self.gated)
            else:
                self._pack_within_room()
        return self._packed

    def _pack_within_room(self):
        size = self.w.numel() * self.w.element_size()
        if self.room.grant(size):
            try:
                self._packed = ops.pack_weight(self.w, gated=self.gated)
            except torch.cuda.OutOfMemoryError:
                self.room.give_back(size)
        self.packable = self._packed is not None

    @property
    def is_packed(self):
        return self._packed is not None

    def drop_packed(self):
        if self._packed is not None and self.room is not None:
            self.room.give_back(self.w.numel() * self.w.element_size())
        self._packed = None


class Runtime:
    bound_bytes = 0      # of the matrices bound so far that could stay in the last-level cache (one bound twice counts twice)

    def __init__(self, dtype=torch.bfloat16, device="cuda:0"):
        if dtype not in (torch.bfloat16, torch.float32):
            raise ValueError(f"activation dtype must be bfloat16 or float32, got {dtype}")
        self.dtype = dtype
        self.device = torch.device(device)
        if self.device.type != "cuda":
            raise RuntimeError("burn-lm_amd runs on the GPU only (device 'cuda:N'); there is no CPU path")
        if not torch.cuda.is_available():
            raise RuntimeError("no GPU is visible to this process; burn-lm_amd has no CPU path")
        self.ops = ops
        self._k_groups = {}     # (N, K, M) -> groups of K, as chosen once (see k_groups)
        self._f32_groups = {}   # the same for the float32 products of up to 16 rows (see f32_skinny_groups; more rows: f32_plan)
        self.packing_room = PackingRoom(self.device)
        ops.library()  # fail now, loudly, if the kernel library cannot be had
        ops.arrival_counters(self.device)   # allocated here, before any graph capture can be open
        ops.gemm_mfma_init(self.device)     # likewise: a function attribute is set once per device
        ops.static_scratch_init(self.device)   # likewise: the address of the library's own scratch array
        ops.attn_paged_init(self.device)       # likewise: the shared memory of the generic attention's value tiles
        ops.gemm_rows_init(self.device)        # likewise: the rings of stages of the product for 17 to 64 rows
        self.compute_units = torch.cuda.get_device_properties(self.device).multi_processor_count
        asked = os.environ.get("BURN_LM_AMD_FUSED_GATE_UP")   # "1": wherever it can run, "0": nowhere, unset: where it is ahead
        self.fused_gate_up_rows = FUSED_GATE_UP_ROWS if asked == "1" else (0, -1)
        self.fused_gate_up_measured = asked != "0"
        self.mid_partials = os.environ.get("BURN_LM_AMD_MID_PARTIALS") != "0"   # "0": the library's products instead
        # most rows for which the skinny kernels take the gated product and the partial planes; above,
        # the matrix-core kernels of short prompts do where their tiles fit (settings for measurements:
        # from 33 rows on those are 1-2 % ahead at some shapes and as much behind at others)
        self.skinny_gated_rows = int(os.environ.get("BURN_LM_AMD_SKINNY_GATED_ROWS", MFMA_SKINNY_MAX_ROWS))
        self.skinny_planes_rows = int(os.environ.get("BURN_LM_AMD_SKINNY_PLANES_ROWS", MFMA_SKINNY_MAX_ROWS))
        # "16" or "32": query rows per wavefront of the prefill attention, whatever the step (for measurements)
        self.prefill_queries = int(os.environ.get("BURN_LM_AMD_PREFILL_TILE", "0") or 0)
        # "0": 17 to 64 rows stay on the packed skinny kernels (for measurements)
        self.rows_ring = os.environ.get("BURN_LM_AMD_ROWS_RING") != "0"

    def empty(self, *shape, dtype=None):
        return torch.empty(*shape, dtype=dtype or self.dtype, device=self.device)

    def weight(self, w, gated=False):
        """Prepares a bound matrix for linear(): bfloat16 matrices, and in a float32 run float32 ones, may get a
        packed copy that the skinny product streams (made at the first product of up to 16 rows, or of up to 64
        bfloat16 ones where no other kernel takes them; it doubles the matrix's memory, in float32 within
        PackingRoom's bounds; the plain copy serves everything else).
        gated=True: w is [gate rows; up rows] of a gated feed-forward and will be used through
        gated_linear(); its packed copy pairs each gate row with its up row."""
        w = w.contiguous()
        N, K = w.shape
        size = w.numel() * w.element_size()
        self.bound_bytes += size if size <= LAST_LEVEL_BYTES else 0
        # (a K too long for one group of the skinny product still runs in several, as partial planes; the gated
        # product has no planes)
        packable = w.dtype == torch.bfloat16 and K % 8 == 0 and K >= 8 and (
            ops.gemv_mfma_supported(1, N, K) and N % 16 == 0 if gated else True)
        if w.dtype == torch.float32:
            # the gated product has no planes, so a longer K or an odd number of pairs goes as a plain product and a pass
            packable = self.dtype == torch.float32 and K % 4 == 0
            gated = gated and N % 16 == 0 and K <= F32_SKINNY_GROUP_K
            return LinearWeight(w, packable, gated, room=self.packing_room)
        return LinearWeight(w, packable, gated)

    @property
    def streams_weights(self):
        """Whether a step finds its weights in memory, not in the last-level cache, where the step before would have left them (see GR_ONCE_BYTES of
        gemm_rows.hip)."""
        return self.bound_bytes > LAST_LEVEL_BYTES

    def k_groups(self, N, K, M=1):
        """Into how many groups a skinny product's K is cut: the fewest whose stretch of K is at most
        GROUP_MAX_K (beyond it a wavefront re-reads its activations for every tile) and whose blocks fill
        at least GROUP_MIN_FILL of their last round on the compute units.  Every block streams its stretch
        of the weights at what one unit can bring, so the product takes as long as the unit with the most
        blocks, and a number of blocks just above a multiple of the units leaves most of the chip idle for
        a block's time; few groups of many wavefronts do better than many of few, and every group is a plane
        that the next norm has to add.  Product and norm together, us at 8 rows (blocks x wavefronts in
        brackets): [4096, 14336] in 4 groups (256x7) 25.1, in 8 (512x4) 28.1; [3072, 3072] in 1 (192x6) 9.4,
        in 4 (384x2) 10.2; [2560, 11008] in 3 (240x8) 15.7, in 8 (432x3) 17.6, in 16 (512x2) 19.9; [1536, 6144]
        in 2 (192x6) 9.4, in 8 (384x2) 11.2; [2048, 8192] in 2 (256x8) 11.4, in 3 (192x6) 12.0, in 4 (512x4) 11.3;
        [2048, 2048] in 1 (128x4) 7.1, in 2 (256x2) 6.6; [8192, 8192] in 2 (256x8) 30.7, in 4 (512x4) 29.8."""
        known = self._k_groups.get((N, K, M))
        if known is None:
            known = self._k_groups[(N, K, M)] = self._choose_k_groups(N, K, M)
        return known

    def _choose_k_groups(self, N, K, M):
        best, best_fill = None, -1.0
        for g in GROUP_CHOICES:
            if g > 1 and K // g < RING_MIN_GROUP_K:
                break
            geometry = ops.gemv_mfma_geometry(M, N, K, g)
            if geometry is None or -(-K // g) > GROUP_MAX_K:
                continue
            blocks = geometry[0]
            fill = blocks / (-(-blocks // self.compute_units) * self.compute_units)
            if fill >= GROUP_MIN_FILL:
                return g
            if fill > best_fill:
                best, best_fill = g, fill
        if best is not None:
            return best
        # no grouping within the bounds: the coarsest one the kernel takes
        return next((g for g in (1, 2, 4, 8, 16, 32, 64) if ops.gemv_mfma_geometry(M, N, K, g) is not None), 64)

    def f32_skinny_groups(self, M, N, K, planes):
        """Into how many groups ops.gemv_f32 cuts K: the fewest that it takes and, where the planes may stay apart, whose
        blocks fill at least GROUP_MIN_FILL of a round on the compute units (us at 8 rows, in 1 / 2 / 4 groups: [2048, 2048]
        8.7 / 6.6 / 5.7 with 128 / 256 / 256 blocks; [2048, 8192] in 4 / 8 groups 16.0 / 15.6)."""
        key = (M, N, K, planes)
        known = self._f32_groups.get(key)
        if known is None:
            taken = [(g, ops.gemv_f32_geometry(M, N, K, g)) for g in (1, 2, 4, 8, 16, 32, 64)]
            taken = [(g, geometry[0]) for g, geometry in taken if geometry is not None]
            full = [g for g, blocks in taken if blocks >= GROUP_MIN_FILL * self.compute_units and K // g >= 256]
            known = self._f32_groups[key] = (full[0] if planes and full else taken[0][0]) if taken else 0
        return known

    def _f32_linear(self, x, w, holder, out, planes):
        """The float32 product of operands that ops.f32_rows takes, or None where the older kernels do it."""
        M, K = x.shape
        N = w.shape[0]
        packed = holder.packed if M <= F32_SKINNY_MAX_ROWS and holder is not None and not holder.gated else None
        if packed is not None:
            groups = self.f32_skinny_groups(M, N, K, planes)
            if groups == 1:
                return ops.gemv_f32(x, packed, out if out is not None else torch.empty(M, N, dtype=torch.float32, device=x.device), K)
            if groups:
                parts = ops.gemv_f32(x, packed, torch.empty(groups, M, N, dtype=torch.float32, device=x.device), K)
                if planes:
                    return parts
                if out is None or out.is_contiguous():
                    return ops.sum_planes(parts, out if out is not None else torch.empty(M, N, dtype=torch.float32, device=x.device))
        if M <= SKINNY_MAX_ROWS:
            return None
        added = not planes and (out is None or (out.is_contiguous() and out.data_ptr() % 16 == 0))
        tile, groups, us = f32_plan(M, N, K, self.compute_units, planes, added=added)
        split = split_plan(M, N, K, self.compute_units, planes, added=added)
        by_parts = split is not None and split[2] < us and (out is None or (out.stride(0) % 4 == 0 and out.data_ptr() % 16 == 0))
        if by_parts:
            tile, groups, _ = split
        if out is None:
            out = torch.empty(M, N, dtype=torch.float32, device=x.device) if groups == 1 or added else None
        into = out if groups == 1 else torch.empty(groups, M, N, dtype=torch.float32, device=x.device)
        if by_parts:
            ops.gemm_split(ops.split_rows(x), w, into, tile=tile)
        else:
            ops.gemm_f32(x, w, into, tile=tile)
        return ops.sum_planes(into, out) if groups > 1 and added else into

    def rows_plan(self, N, K):
        """(groups of K, columns per block) for a product of 17 to 64 rows that may come as partial planes."""
        return rows_plan(N, K, self.compute_units)

    def mid_rows_ring(self, M, N, K, planes):
        """65 to 256 rows, K up to 2048, few columns (the output projection of short prompts and of decode
        steps of many sequences at the 1B width): the product of 17 to 64 rows with a block for every 64
        rows, while all its blocks of 32 columns run at once.  Returns the groups of K (two where that
        still gives every block a compute unit and the caller takes partial planes), 0 for another kernel.
        Measured per call at the 1B shape against the library's product: 6.8-7.2 against 9.8 us at 65-128
        rows, 8.0 against 10.8 at 192, 8.9 against 11.1 at 256; at K = 3072 and 4096 (3B, 8B) equal or
        behind, hence the bound on K."""
        if not (self.rows_ring and MFMA_SKINNY_MAX_ROWS < M <= 256 and K <= RING_MID_K):
            return 0
        blocks = self.rows_ring_blocks(M, N)
        if blocks > self.compute_units:
            return 0
        return 2 if planes and K >= 1024 and blocks * 2 <= self.compute_units else 1

    def rows_ring_blocks(self, M, N, columns=32):
        """Blocks of 64 rows and 32 or 64 columns that ops.gemm_rows and ops.gemm_rows_qkv_rope launch."""
        return -(-N // columns) * -(-M // 64)

    def qkv_plan(self, M, N, K):
        """Which fused projection geometry a position encoding should build on for M rows of width K and
        N = all query, key and value columns, or None (project with linear(), then encode).  The encoding
        only has to check that its own kernel exists for the answer; the thresholds live here.
        17 to 64 rows: the row-ring geometry (per call against the packed kernel with two to four row tiles,
        us: width 1536 at 24 / 32 rows 6.4 / 6.7 against 7.4 / 8.0; width 2048 at 17 / 24 / 32 rows 7.0 / 7.0 / 7.4
        against 7.2 / 7.8 / 8.6; width 3072 8.5-9.2 against 16.5-21.8; whole decode steps at batch 17 to 64 of
        the 3B and 8B shapes 2-6 % faster); 33 to 64 rows as two blocks of 32 while both sets run at once (1B
        shape: 7.8-8.2 against 9.3-9.8 us).  65 to 256 rows: a block for every 64
        rows, 32 columns per block while those blocks all run at once, else 64 while there are at most one
        and a half per compute unit (per layer against the library's product and the rotation kernel: 1B
        shape 10 against 14-16 us at 65-128 rows, 13.3 against 21 at 192, 13.6 against 16 at 256; 3B 16-17
        against 18-27 at 65-192, 28.5 against 33 at 256; 8B 21-24.5 against 28-31 at 65-128, 36 against 39
        at 192, 38.5 against 46 at 256).  Up to 16 rows, and whenever the row-ring kernel is not to be
        had: the packed geometry."""
        if self.rows_ring and K <= RING_QKV_K:
            if 16 < M <= MFMA_SKINNY_MAX_ROWS:
                halves = M > 32 and self.rows_ring_blocks(64, N) * 2 <= self.compute_units
                return FusedProjectionPlan("rows", 32, 32 if halves else 64)
            if MFMA_SKINNY_MAX_ROWS < M <= 256:
                if self.rows_ring_blocks(M, N) <= self.compute_units:
                    return FusedProjectionPlan("rows", 32, 64)
                if self.rows_ring_blocks(M, N, 64) * 2 <= self.compute_units * 3:
                    return FusedProjectionPlan("rows", 64, 64)
        if M <= MFMA_SKINNY_MAX_ROWS:
            return FusedProjectionPlan("packed")
        return None

    def mid_planes_plan(self, M, N, K):
        """More than 32 rows, narrow output, long K (the down projection, the output projection of wide models): the
        product as partial planes of the matrix-core kernel over groups of K (the block's next norm sums the
        planes).  -> (groups, tile), or (0, None) for the library's product.  Of the 128x128 and 128x64 tiles
        with eight, four or two groups of at least MFMA_MIN_GROUP_K, the one whose blocks come closest to one
        per compute unit without exceeding that, the larger tile on a tie, and nothing if even that leaves half the
        units idle.  Measured at 128 rows (us, chosen / library): widths 2560, 5120 and 8192 with an inner size of
        11008: 22.4 / 57.6, 37.5 / 60.9, 45.4 / 67.2; width 1536: 14.5 / 21.9; a tie (width 2560, 160 blocks): 128x128
        in eight groups 22.4, 128x64 in four 25.9.  Over whole prompts of 65 to 128 tokens: 6 % faster at the
        Llama-3.2-1B shape, 19 % at 3B, 21 % at 8B (the library's product of few rows and a long K streams the
        weights at a quarter of the memory rate); 2-5 % up to 512 tokens, where two groups still fit; equal beyond."""
        best = (0, None, 0)
        if M > MID_PLANES_MAX_ROWS:
            return 0, None
        for tile, tn in (((128, 128, 4), 128), ((128, 64, 6), 64)):
            tiles = -(-M // 128) * -(-N // tn)
            for g in (8, 4, 2):
                blocks = tiles * g
                if K // g >= MFMA_MIN_GROUP_K and self.compute_units // 2 <= blocks <= self.compute_units and blocks > best[2]:
                    best = (g, tile, blocks)
        return best[0], best[1]

    def narrow_groups(self, M, N, K):
        """Groups of K for a float32 result of at most 64 columns and many rows (a router's logits, the gates of a
        recurrence): its row tiles alone are a handful of blocks, each walking all of K; cut into groups of at least
        NARROW_MIN_GROUP_K the product fills the chip, and a small kernel adds the planes.  1: not worth it."""
        if N > 64 or M <= MFMA_SKINNY_MAX_ROWS:
            return 1
        tiles, groups = -(-M // 128), 1
        while groups < 16 and K // (groups * 2) >= NARROW_MIN_GROUP_K and tiles * groups * 2 <= self.compute_units:
            groups *= 2
        return groups

    def mid_k_groups(self, M, N, K):
        """Groups of K of mid_planes_plan (0: the library's product)."""
        return self.mid_planes_plan(M, N, K)[0]

    def linear(self, x, w, out_dtype=None, out=None, partials=False):
        """x [M,K] @ w[N,K]^T -> [M,N] in out_dtype (default: the activation dtype).  w: a
        LinearWeight from weight(), or a plain tensor.  partials=True allows the result to come as
        float32 [groups, M, N] partial products (the caller hands it to a norm's add, which sums
        them); it is used for narrow outputs in decode."""
        packable, holder = False, None
        if isinstance(w, LinearWeight):
            holder, w = w, w.w
            packable = holder.packable and not holder.gated   # a gated copy has its rows re-ordered
        M, K = x.shape
        N = w.shape[0]
        out_dtype = out_dtype or self.dtype
        planes = partials and out is None       # the result may come as float32 partial planes
        if w.dtype == torch.float32 or x.dtype == torch.float32:
            if out_dtype == torch.float32 and ops.f32_rows(x, w):
                done = self._f32_linear(x, w, holder, out, planes)
                if done is not None:
                    return done
            if out is None:
                out = torch.empty(M, N, dtype=out_dtype, device=x.device)
            if M <= SKINNY_MAX_ROWS and x.dtype == w.dtype == out_dtype == torch.float32 and K % 8 == 0 \
                    and x.stride(0) % 8 == 0:
                return ops.gemv_skinny(x, w, out)
            return ops.gemm_tiled(x, w, out)
        aligned = K % 8 == 0 and x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0
        if (M > MFMA_SKINNY_MAX_ROWS and aligned and x.dtype == w.dtype == torch.bfloat16 and x.stride(1) == 1
                and w.is_contiguous() and out_dtype == torch.bfloat16):
            groups = self.mid_rows_ring(M, N, K, planes=planes)
            if groups > 1:
                return ops.gemm_rows(x, w, torch.empty(groups, M, N, dtype=torch.float32, device=x.device), columns=32)
            if groups == 1:
                return ops.gemm_rows(x, w, out if out is not None else torch.empty(M, N, dtype=out_dtype, device=x.device),
                                     columns=32)
        plain_bf16 = aligned and x.dtype == w.dtype == torch.bfloat16 and x.stride(1) == 1 and w.is_contiguous()
        if planes and self.mid_partials and M > self.skinny_planes_rows and plain_bf16:
            groups, tile = self.mid_planes_plan(M, N, K)
            if groups:
                return ops.gemm_mfma(x, w, torch.empty(groups, M, N, dtype=torch.float32, device=x.device), tile=tile)
        if planes and plain_bf16 and self.duo_planes(M, N, K):
            planes_out = torch.empty(2, M, N, dtype=torch.float32, device=x.device)
            if ops.gemm_duo_takes(x, w, planes_out):
                return ops.gemm_duo(x, w, planes_out, whole=0)
        parts = self.duo_part_planes(M, N, K) if planes and plain_bf16 else None
        if parts is not None:
            planes_out = torch.empty(parts[0], M, N, dtype=torch.float32, device=x.device)
            if ops.gemm_duo_takes(x, w, planes_out):
                return ops.gemm_duo(x, w, planes_out, whole=0, fives=parts[1])
        if (planes and self.rows_ring and 16 < M <= MFMA_SKINNY_MAX_ROWS and plain_bf16
                and (M > 32 or K <= 4096 or -(-N // 32) * 8 <= 3 * self.compute_units)):
            # 17 to 64 rows as partial planes (measured against the packed skinny kernel at the 1B, 3B and 8B
            # shapes: output projection 15-35 % faster at every row count, down projection 25-40 % at K = 8192 of
            # the 1B width, equal to 10 % at the wider ones from 33 rows on).  Up to 32 rows: where K is short or the
            # output narrow (up to 96 blocks of 32 columns on 256 units: widths 1536 and 2560 with inner sizes of
            # 6144 and 11008 at 32 rows 6.2-9.3 us against 8.1-12.0); a wide output with a long K stays with the
            # packed kernel there (equal to 8 % ahead)
            groups, columns = self.rows_plan(N, K)
            if M > 32 and self.mid_partials and -(-N // columns) * groups > self.compute_units:
                # more blocks than compute units even with 64 columns each (a long K under a wide output): the
                # matrix-core kernel's planes where they fill the chip (width 8192, K = 11008, 64 rows: 42.6 against 46.3 us)
                g2, tile = self.mid_planes_plan(M, N, K)
                if g2:
                    return ops.gemm_mfma(x, w, torch.empty(g2, M, N, dtype=torch.float32, device=x.device), tile=tile)
            if groups > 1:
                return ops.gemm_rows(x, w, torch.empty(groups, M, N, dtype=torch.float32, device=x.device), columns=columns, once=self.streams_weights)
        if packable and M <= MFMA_SKINNY_MAX_ROWS and aligned:
            if planes:
                groups = self.k_groups(N, K, M)
                if groups > 1:
                    return ops.gemv_mfma(x, holder.packed, torch.empty(groups, M, N, dtype=torch.float32, device=x.device), K)
            if ops.gemv_mfma_supported(M, N, K):
                if out is None:
                    out = torch.empty(M, N, dtype=out_dtype, device=x.device)
                return ops.gemv_mfma(x, holder.packed, out, K)
        if out is None:
            out = torch.empty(M, N, dtype=out_dtype, device=x.device)
        if (out_dtype == torch.float32 and M > 32 and aligned and x.dtype == w.dtype == torch.bfloat16
                and x.stride(1) == 1 and w.is_contiguous() and out.stride(1) == 1 and N * K * 2 < 1 << 32):
            groups = self.narrow_groups(M, N, K) if out.is_contiguous() else 1
            if groups > 1:
                planes = torch.empty(groups, M, N, dtype=torch.float32, device=x.device)
                return ops.sum_planes(ops.gemm_mfma(x, w, planes, tile=(128, 64, 6)), out)
            tiles = -(-M // 256) * -(-N // 128)
            if planes and M > MID_PLANES_MAX_ROWS and tiles * 2 <= self.compute_units and K >= 2 * MFMA_MIN_GROUP_K:
                # a residual's new start: partial planes fill the chip where the tiles alone leave half of it idle, and
                # the norm behind it adds them (2,048 rows, width 2048, K = 4096: 42.4 us against 57.9)
                return ops.gemm_mfma(x, w, torch.empty(2, M, N, dtype=torch.float32, device=x.device), tile=(256, 128))
            # float32 results (logits) for more rows than one skinny product takes at this width (more than 64,
            # or more than 32 where K is above 2048): the matrix-core kernel with a float output, which reads
            # the weights once.  Measured per call with a vocabulary of 128,256 against the skinny product in
            # chunks of rows (us): width 2048, 65 / 128 / 256 rows: 141 / 156 / 189 against 202 / 230 / 453;
            # width 3072, 33-64 rows: 154-169 against 268-298; width 4096: 233-238 against 329-350, 65-128 rows
            # 240-252 against 509-687; the library's product with a float output: equal to 5 % behind.
            return ops.gemm_mfma(x, w, out, tile=(128, 128, 4) if M <= 128 else (256, 128))
        if packable and aligned and out_dtype == torch.float32:
            # 17 to 32 rows at a K above 4096: the most rows the skinny product does take at a time (16); the
            # weights stream once per chunk, which still beats the plain tiled kernel by far
            chunk = next((c for c in (64, 32, 16) if ops.gemv_mfma_supported(c, N, K)), 0)
            if chunk:
                for r in range(0, M, chunk):
                    ops.gemv_mfma(x[r:r + chunk], holder.packed, out[r:r + chunk], K)
                return out
        if M <= SKINNY_MAX_ROWS and aligned:
            return ops.gemv_skinny(x, w, out)
        if out_dtype == torch.bfloat16:
            if plain_bf16 and self.fused_gate_up_measured and self.duo_product(M, N, K) and ops.gemm_duo_takes(x, w, out):
                return ops.gemm_duo(x, w, out, whole=self.duo_tiles(M, N))
            return torch.matmul(x, w.t(), out=out)
        # float32 logits from bfloat16 operands with many rows: own kernel (float accumulation)
        return ops.gemm_tiled(x, w, out)

    def f32_qkv_packed(self, x, w, M, N, K):
        """The packed copy of a float32 q/k/v projection that ops.gemv_f32_qkv_rope reads, or None where another kernel does it."""
        if not (isinstance(w, LinearWeight) and M <= F32_SKINNY_MAX_ROWS and w.dtype == x.dtype == torch.float32 and not w.gated
                and ops.f32_rows(x, w.w) and self.f32_skinny_groups(M, N, K, False) == 1):
            return None
        return w.packed

    def f32_qkv_split(self, x, w, M, N, K):
        """The tile of ops.gemm_split_qkv_rope for a float32 q/k/v projection of many rows, or None where a product and the kernel that turns
        its results and fills the pages (4 us and 8 bytes an element) are faster: where groups of K are, whose planes have to be added first."""
        if not (M > F32_SKINNY_MAX_ROWS and x.dtype == torch.float32 and ops.f32_rows(x, w)):
            return None
        split = split_plan(M, N, K, self.compute_units)
        if split is None:
            return None
        apart = min(plan(M, N, K, self.compute_units, added=True)[2] for plan in (f32_plan, split_plan))
        return split[0] if split[2] < apart + 4.0 + M * N * 8 / 3.5e6 else None

    def duo_tiles(self, M, N):
        """How many of a product's tiles ops.gemm_duo runs as whole ones."""
        return duo_plan(M, N, self.compute_units)[0]

    def duo_qkv(self, M, N, K):
        """Whether a q/k/v projection of more than 256 rows goes to ops.gemm_duo_qkv_rope, which turns queries and keys and fills the
        pages behind the product instead of a kernel that reads its results and writes them back.  Us, this / the product of before and
        that kernel, in graphs: [3072, 2048] 2,048 / 2,500 / 4,000 rows 32.4 / 38.0, 36.0 / 42.4, 52.1 / 58.1; [5120, 3072] 1,218 /
        2,048 / 3,300 rows 47.9 / 58.4, 71.9 / 73.4, 118 / 129; [6144, 4096] 1,036 / 2,048 / 4,000 rows 57.4 / 65.7, 90.1 / 98.1, 165 /
        184.  Within prompts: 2,048 rows of the 1B shape 36.8 / 29.2 + 8.0 and a launch, 9,681 rows of the 3B shape 225 / 325 +
        50.  Less full rounds are equal or behind:
        [3072, 2048] 3,300 rows (fill 0.60) 54.1 / 50.8, 3,356 (0.615) 53.6 / 51.3, 1,000 (0.32) 28.4 / 27.2; [5120, 3072] 1,150 rows
        (0.62) 50.8 / 49.2, 600 rows (0.32) 46 / 39."""
        return self.fused_gate_up_measured and M > 256 and K <= RING_QKV_K and duo_plan(M, N, self.compute_units)[2] >= DUO_QKV_FILL

    def duo_planes(self, M, N, K):
        """Whether a product of long prompts that may come as planes (the down projection) runs as halves of ops.gemm_duo's tiles over two
        groups of K: where these are at least DUO_PLANES_FILL of one round, and not more.  With the norm that adds the planes, us, this /
        the library, in turn: width 2048, K = 8192, 1,639 / 1,686 / 1,870 / 1,951 / 2,048 rows 69.5 / 72.5, 64.8 / 73.6, 71.1 / 75.5,
        70.7 / 76.5, 76.3 / 75.8 (the library's 128x128 tiles are one full round there; within prompts of the 1B shape 69.3 / 68.4);
        K = 6144 1,638 / 1,750 / 2,048 rows 49.7 / 54.4, 58.7 / 61.3, 64.7 / 63.7; width 3072, K = 8192, 1,045 and 1,280 rows 64.1 / 74.5
        and 71.5 / 77.1; width 4096, K = 14336, 788 and 1,024 rows 111 / 126 and 124 / 136.  With 192 blocks behind: width 2048, K = 8192,
        1,443 and 1,532 rows 64.6 / 59.6 and 68.5 / 60.7; width 4096, K = 14336, 768 rows 117 / 111; and a shorter K gains nothing:
        width 2048, K = 4096, 1,716 and 2,048 rows 39.5 / 39.7 and 42.8 / 41.5, K = 2048 (in a graph) 1,600 and 2,048 rows 29.6 / 27.4 and
        36.3 / 29.9."""
        if not self.fused_gate_up_measured or M <= MID_PLANES_MAX_ROWS or K < DUO_PLANES_K:
            return False
        tiles, tail = ops.gemm_duo_tiles(M, N)
        return DUO_PLANES_FILL * self.compute_units <= 2 * (2 * tiles + tail) <= self.compute_units

    def duo_part_planes(self, M, N, K):
        """(groups of K, fives) with which such a product runs as planes of parts of ops.gemm_duo's tiles, all in one round, or None: halves
        over four groups, or tiles of 160 rows (fives) over four or two; of the first that fits, with a group of at
        least RING_GROUP_K, K from DUO_PLANES_K on, and four groups' blocks on DUO_FOURS_FILL of the units, two groups' on DUO_FIVES_FILL.
        With the norm that adds the planes, us, this / as before (the library where nothing else is said):
        * halves, four groups: width 2048, K = 8192, 675 / 770 / 883 rows 40.4 / 46.7, 42.4 / 48.0, 44.4 / 50.8; K = 16384 657 / 855 / 962 rows
          59 / 78, 69 / 90, 70 / 96; width 3072, K = 8192, 537 / 620 rows 43.9 / 51.2, 44.7 / 52.9; width 1024, K = 8192, 1,240 / 1,389 rows
          35.4 / 42.0, 37.7 / 43.2; width 1536, K = 12288, 845 / 1,132 rows 47.9 / 58.4, 56.0 / 69.6;
        * 160 rows, four groups: width 2048, K = 8192, 1,035 / 1,147 / 1,274 rows 51.2 / 61.7, 52.1 / 60.3, 53.0 / 63.0; K = 16384 74.9 / 104.6,
          74.9 / 103.0, 80.7 / 111.6; width 3072, K = 8192, 646 / 778 rows 49.0 / 57.5, 52.1 / 60.7; width 4096, K = 14336, 524 / 599 rows
          71.4 / 93.8, 72.8 / 98.7;
        * 160 rows, two groups: width 2048, K = 8192, 2,075 / 2,166 / 2,500 rows 77.6 / 84.5, 79.3 / 86.0, 83.4 / 88.1; width 3072, K = 8192, 1,282 /
          1,405 / 1,534 rows 74.6 / 77.9, 74.9 / 81.4, 80.5 / 86.8; width 4096, K = 14336, 1,085 / 1,268 rows 115 / 131, 124 / 139; width 2560,
          K = 11008, 1,554 / 1,915 rows 94.6 / 103.7, 102.2 / 112.7; less full 0.71 of the units, where halves over two groups fit: 74.1 / 68.5;
        * three groups gain nothing: width 1536, K = 6144, 1,749 to 1,985 rows 1.03 of the library's time."""
        if not self.fused_gate_up_measured or M <= MID_PLANES_MAX_ROWS or K < DUO_PLANES_K or self.duo_planes(M, N, K):
            return None
        for rows, groups, fill in ((128, 4, DUO_FOURS_FILL), (160, 4, DUO_FOURS_FILL), (160, 2, DUO_FIVES_FILL)):
            blocks = -(-M // rows) * -(-N // 256) * groups
            if K % (128 * groups) == 0 and K // groups >= RING_GROUP_K and blocks <= self.compute_units \
                    and M * N * groups >= fill * self.compute_units * rows * 256:
                return groups, rows == 160
        return None

    def duo_product(self, M, N, K):
        """Whether a plain bfloat16 product of many rows goes to ops.gemm_duo and not to the library (us, duo / library, in turn):
        * one round of halves, at least DUO_HALVES_FILL of the units busy, K up to DUO_HALVES_K: [2048, 2048] 3,589 and 4,062 rows 31.1 /
          33.6 and 30.6 / 32.9; [5120, 2048] 1,482 and 1,535 rows 28.8 / 31.2 and 27.9 / 30.1; [3072, 3072] 2,387 and 2,661 rows 39.0 /
          42.8 and 39.9 / 42.4; [5120, 3072] 1,400 and 1,488 rows 50.0 / 51.5 and 47.2 / 46.6; [2048, 8192] 3,476 and 4,049 rows 99.9 /
          106.4 and 103.6 / 106.6 (longer K goes either way: [4096, 14336] 1,738 / 1,856 / 1,917 rows 199 / 217, 201 / 196, 208 / 194);
        * whole rounds and a last one of halves, where the library's times jump with the rows: [2048, 2048] 9,078 and 9,510 rows 70 / 66
          and 70 / 79; [5120, 2048] 3,750 / 7,100 / 8,017 rows 70 / 80, 115 / 114, 121 / 149; [3072, 3072] 5,931 and 8,189 rows 98 / 104
          and 106 / 115; [6144, 4096] 2,735 / 4,077 / 5,888 rows 128 / 207, 141 / 153, 216 / 211; [3072, 8192] 5,595 and 7,919 rows
          239 / 232 and 262 / 277; [4096, 14336] 4,983 and 5,448 rows 463 / 426 and 454 / 841; 0.90 of its time over 84 sizes.
        Whole rounds alone, full as they may be, are the library's: [2048, 2048] 8,100 rows 50.8 / 47.5, [3072, 2048] 5,217 rows 48.9 /
        47.1, [6144, 2048] 5,345 and 7,999 rows 97.6 / 93.2 and 147.7 / 138.7, [3072, 3072] 5,326 rows 69.6 / 66.5."""
        if M <= MFMA_SKINNY_MAX_ROWS:
            return False
        whole, rounds, fill = duo_plan(M, N, self.compute_units)
        if rounds <= DUO_HALF:
            return fill >= DUO_HALVES_FILL and K <= DUO_HALVES_K
        tiles = ops.gemm_duo_tiles(M, N)[0]
        return whole < tiles and tiles >= self.compute_units

    # ---- products of few rows that do a neighbouring norm's work (ops.gemv_join, parts/block.py) ----
    def join_takes(self, M, w):
        """Whether the product of M rows with w can add its result to the residual and leave the next norm's rows (join).  Up to eight
        rows: beyond, every block's activations, all of K for few columns, cost more than the norm's kernel (a layer of the 1B shape
        without its attention, us, norms as kernels / joined: 1 row 34.9 / 29.9, 4 rows 36.2 / 31.5, 8 rows 37.6 / 34.1, 16 rows 40.9 /
        40.2; of the 3B shape 50.3 / 44.3, 52.6 / 45.9, 54.3 / 48.3, 59.2 / 68.7).  bfloat16 from JOIN_BF16_WIDTH columns on.  Neither time
        nor error draws that line (a product and its norm apart / joined, us, rows 1 and 8: [64, 176] 4.6 / 2.9, 4.9 / 3.0, [256, 704] 5.2 / 2.9, 5.5 /
        3.1, [512, 1408] 5.6 / 3.1, 6.1 / 3.4, [768, 3072] 5.9 / 3.9, 6.5 / 4.7; three small models joined and apart are equally far from
        64 bits, to 3 in a hundred): the rows are rounded in front of the norm's factor instead of behind it, and the widths below
        are those whose steps are compared, value by value, with an implementation that rounds behind it."""
        return (M <= ops.SCALED_ROWS and isinstance(w, LinearWeight) and not w.gated and w.dtype == self.dtype and w.packable
                and (w.dtype == torch.float32 or w.shape[0] >= JOIN_BF16_WIDTH) and self.join_gains(w.dtype, M, *w.shape) and w.packed is not None)

    def join_gains(self, dtype, M, N, K):
        """Whether gemv_join is the shorter way.  It is not for a long K where a block's columns are no whole 64 bytes of the packed weights (its
        neighbours read the rest of their lines once more), nor in float32 where few columns leave units idle while each block reads all rows'
        K.  A product and the norm's kernel / this, us, rows 1, 4 and 8:
        * bfloat16, blocks of 8, 12 and 16 columns: [2048, 16384] 18.2 / 14.0, 17.7 / 14.6, 18.5 / 16.6; [3072, 8192] 14.8 / 14.1, 15.3 / 14.0, 15.2 /
          15.1; [4096, 16384] 28.9 / 24.9, 29.7 / 25.2, 29.9 / 25.7; [1152, 9216] 9.3 / 8.1, 9.3 / 8.6, 9.8 / 9.9;
        * of 9, 11, 13 and 15: [2304, 6336] 11.3 / 8.9, 11.4 / 9.3, 11.8 / 10.3; [2304, 9216] 12.7 / 13.2, 12.7 / 12.8, 13.0 / 14.0; [2816, 7744] 13.8 /
          12.5, 13.7 / 12.5, 14.3 / 13.6; [2816, 11264] 17.3 / 17.8, 17.9 / 18.3, 17.5 / 19.8; [3840, 10560] 19.4 / 18.5, 19.4 / 19.4, 19.8 / 21.0;
        * of 10 and 14: [2560, 10240] 14.6 / 13.8, 15.1 / 13.3, 14.9 / 14.5; [3584, 9856] 18.5 / 18.6, 19.0 / 18.4, 18.9 / 19.1; [2560, 14080] 17.9 /
          17.0, 18.4 / 18.1, 18.7 / 20.9; [3584, 14336] 23.7 / 23.7, 24.4 / 24.5, 24.5 / 25.8;
        * float32, blocks of 8: [1024, 4096] 8.0 / 7.2, 8.2 / 7.7, 8.3 / 8.6; [768, 4224] 9.2 / 9.2, 9.5 / 10.0, 9.8 / 11.2; [1152, 6336] 16.0 / 11.2, 16.9
          / 11.6, 17.5 / 13.4; [1024, 8192] 11.7 / 12.0, 11.9 / 13.0, 12.0 / 14.6; [1536, 8448] 18.6 / 17.5, 18.9 / 19.7, 19.5 / 20.8; [1792, 14336] 25.9 /
          22.0, 26.3 / 23.9, 26.6 / 28.1; [2048, 11264] 23.6 / 20.8, 23.6 / 22.1, 24.2 / 25.6; [2048, 16384] 32.6 / 26.2, 33.1 / 27.6, 33.4 / 31.8;
        * float32, of 9 to 14: [2560, 2560] 12.1 / 9.2, 12.8 / 9.7, 13.1 / 10.5; [3584, 3584] 15.7 / 12.1, 16.1 / 12.5, 16.3 / 13.5; [2304, 6336] 18.7 /
          20.4, 18.9 / 21.0, 19.3 / 21.0; [3072, 8448] 27.5 / 30.4, 27.2 / 30.4, 27.7 / 32.7; of 16: [4096, 16384] 57.4 / 47.9, 59.1 / 48.9, 59.3 / 51.4."""
        columns = ops.gemv_join_columns(dtype, M, N, K)
        if columns == 0:
            return False
        if dtype == torch.bfloat16:
            return columns % 4 == 0 or K <= (8192 if columns % 2 else 10240)
        if columns > 8:
            return columns == 16 or K <= 4096
        return N >= 2048 or K <= 4 * N or (M <= 4 and (N >= 1536 or K <= 6 * N))

    def join_reads(self, x, w):
        """Whether join takes these rows: of the weights' type, in whole pieces of 16 bytes (an attention's or a gating's own always are)."""
        return x.dtype == w.dtype and x.dim() == 2 and x.stride(1) == 1 and x.stride(0) * x.element_size() % 16 == 0 and x.data_ptr() % 16 == 0

    def join(self, product, h, gamma, eps):
        """h += the product; the rows of an RMS norm with gamma (float32) and eps behind it, Unscaled."""
        x, w = product.x, product.w
        M, (N, K) = x.shape[0], w.shape
        y = torch.empty(M, N, dtype=self.dtype, device=x.device)
        sums = torch.empty(M, N // ops.gemv_join_columns(w.dtype, M, N, K), dtype=torch.float32, device=x.device)
        return Unscaled(ops.gemv_join(x, w.packed, h, gamma, y, sums, K), sums, eps)

    def experts_take(self, x, w):
        """Whether the gated product of stacked experts runs with their weights in its epilogue (ops.gemv_experts): where the packed kernel
        takes the rows.  Elsewhere it is a product and a pass."""
        return (isinstance(w, LinearWeight) and w.gated and w.packable and x.dtype == w.dtype == torch.bfloat16
                and x.shape[0] <= MFMA_SKINNY_MAX_ROWS and bool(ops.gemv_mfma_supported(x.shape[0], *w.shape))
                and x.stride(1) == 1 and x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0)

    def gated_takes_unscaled(self, M, w):
        """Whether gated_linear takes M Unscaled rows: where its packed kernels have them."""
        if not (isinstance(w, LinearWeight) and w.gated and w.packable and M <= ops.SCALED_ROWS and w.dtype == self.dtype):
            return False
        if self.dtype == torch.float32:
            return w.packed is not None
        return M <= self.skinny_gated_rows and bool(ops.gemv_mfma_supported(M, *w.shape))

    def qkv_takes_unscaled(self, M, w, head_dim):
        """The same of a q/k/v projection with rotation in adjacent pairs."""
        if not (isinstance(w, LinearWeight) and not w.gated and w.packable and M <= ops.SCALED_ROWS and w.dtype == self.dtype):
            return False
        N, K = w.shape
        if self.dtype == torch.float32:
            return head_dim % 2 == 0 and self.f32_skinny_groups(M, N, K, False) == 1 and w.packed is not None
        plan = self.qkv_plan(M, N, K)
        return plan is not None and plan.kernel == "packed" and ops.gemv_qkv_rope_supported(M, K, head_dim, 0)

    def _gated_by_library(self, M, K, inner):
        """17 to 64 rows of a gated product that are better left to the library's product and the gating kernel:
        from 33 rows on where K is beyond 4096 (measured at widths 5120 and 8192 with inner sizes of 6144 to 28672:
        6-23 % ahead of the row ring, whose blocks each walk all of K, and of the matrix-core tiles of short
        prompts) or the row ring would take more than two rounds of blocks (width 2560 with an inner size of
        28672: 66.9 against 74.6 us); up to 32 rows where K is beyond what the packed kernel takes and the row
        ring's blocks do not all run at once (width 5120, inner size 11008: 51.6 against 57.7)."""
        if M > 32:
            return K > 4096 or -(-inner // 32) > 2 * self.compute_units
        return K > 4096 and -(-inner // 32) > self.compute_units

    def duo_beside(self, M, inner, n):
        """How many tiles ops.gemm_duo_beside runs as whole ones for a gated product with n plain columns beside it, or None where the
        two run apart.  The gated tiles have to be worth it by themselves, as in gated_linear (a lone round of halves at a wide K as
        well: the two apart are a launch and a pass more), and the columns beside them have to fit into what is left of the last
        round, or into whole tiles where that was of halves (us, together / apart, in a graph; inner size 8192 and a width of columns
        beside it: width 2048, 384 / 700 / 1,300 / 2,166 rows 33 / 40, 47 / 57, 91 / 102, 132 / 151; width 3072, 384 / 700 / 1,300 /
        2,166 rows 55 / 69, 71 / 94, 135 / 156, 205 / 231, with 512 columns 384 / 700 / 1,300 rows 53 / 57, 67 / 79, 118 / 131).
        Halves more behind full rounds are behind: width 2048, 900 / 1,000 / 2,048 rows 69 / 68, 71 / 68, 132 / 128; width 3072
        112 / 102, 117 / 111, 195 / 191, with 512 columns 1,000 and 2,048 rows 101 / 90 and 176 / 164."""
        alone, both = (duo_plan(M, inner, self.compute_units, True, b) for b in (0, n))
        fits = M > 256 and min(alone[2], both[2]) >= DUO_GATED_FILL and both[1] - alone[1] < DUO_HALF - 0.01
        return both[0] if fits else None

    def gated_linear_beside(self, x, w, beside, stacked, activation):
        """(gated_linear(x, w, activation), linear(x, beside)) of two matrices that lie one behind the other in `stacked`: in one
        launch where duo_beside says so."""
        M, inner, n = x.shape[0], w.shape[0] // 2, beside.shape[0]
        if self.fused_gate_up_measured and stacked.dtype == self.dtype == torch.bfloat16 and stacked.numel() < 1 << 31:
            whole = self.duo_beside(M, inner, n)
            if whole is not None:
                out, z = (torch.empty(M, m, dtype=self.dtype, device=x.device) for m in (inner, n))
                if ops.gemm_duo_takes(x, stacked, out, gated=True) and ops.gemm_duo_takes(x, stacked, z):
                    return ops.gemm_duo_beside(x, stacked, out, z, activation=activation, whole=whole)
        return self.gated_linear(x, w, activation=activation), self.linear(x, beside)

    def f32_gated_plan(self, M, inner, K):
        """(whether by parts, tile) of the float32 gated product, or None for few rows, where the plain product's smaller tiles and the
        pass behind it (12 bytes an element) are faster."""
        tile, _, us = f32_plan(M, inner, K, self.compute_units, gated=True)
        split = split_plan(M, inner, K, self.compute_units, gated=True)
        by_parts = split is not None and split[2] < us
        if by_parts:
            tile, _, us = split
        apart = [plan(M, 2 * inner, K, self.compute_units, added=True) for plan in (f32_plan, split_plan)]
        return (by_parts, tile) if us <= min(p[2] for p in apart if p is not None) + 3.0 + M * inner * 12 / 5e6 else None

    def gated_pair(self, x, w, down):
        """linear(gated_linear(x, w), down, partials=True): in float32 the first product leaves its rows as the parts that the second
        reads, where both run by parts."""
        if not isinstance(x, Unscaled) and self.dtype == torch.float32 and x.shape[0] > F32_SKINNY_MAX_ROWS:
            plain, narrow = (v.w if isinstance(v, LinearWeight) else v for v in (w, down))
            M, K = x.shape
            N, inner = narrow.shape
            if plain.shape[0] == 2 * inner and ops.f32_rows(x, plain) and narrow.dtype == torch.float32 and narrow.is_contiguous() and narrow.data_ptr() % 16 == 0:
                gated, split = self.f32_gated_plan(M, inner, K), split_plan(M, N, inner, self.compute_units, planes=True)
                if gated is not None and gated[0] and split is not None and \
                        split[2] - split_rows_us(M, inner) < f32_plan(M, N, inner, self.compute_units, True)[2]:
                    parts = ops.gemm_split_parts(ops.split_rows(x), plain, M, tile=gated[1])
                    shape = (M, N) if split[1] == 1 else (split[1], M, N)
                    return ops.gemm_split(parts, narrow, torch.empty(shape, dtype=torch.float32, device=x.device), tile=split[0])
        return self.linear(self.gated_linear(x, w), down, partials=True)

    def gated_linear(self, x, w, activation="silu"):
        """act(x gate^T) * (x up^T) for w = [gate rows; up rows] ([2I, K]) -> [M, I]; act is silu or
        (activation="gelu_tanh") the tanh form of GELU.  With few rows in bfloat16 the gating is fused
        into the product (weight(w, gated=True) pairs the rows for it); otherwise the product is followed
        by the gating kernel.  x may be Unscaled where gated_takes_unscaled says so."""
        if isinstance(x, Unscaled):
            out = torch.empty(x.y.shape[0], w.shape[0] // 2, dtype=self.dtype, device=x.y.device)
            if self.dtype == torch.float32:
                if activation != "silu":
                    raise ValueError("gated_linear: float32 rows that come unscaled are gated with silu")
                return ops.gemv_f32(x.y, w.packed, out, w.shape[1], gated=True, scale=x.scale)
            return ops.gemv_mfma(x.y, w.packed, out, w.shape[1], gated=True, activation=activation, scale=x.scale)
        M, K = x.shape
        inner = w.shape[0] // 2
        plain = w.w if isinstance(w, LinearWeight) else w
        if activation not in ("silu", "gelu_tanh"):
            raise ValueError(f"gated_linear: activation {activation!r} unknown (silu, gelu_tanh)")
        if plain.dtype == torch.float32 and self.dtype == torch.float32 and activation == "silu" and ops.f32_rows(x, plain):
            if M <= F32_SKINNY_MAX_ROWS:
                packed = w.packed if isinstance(w, LinearWeight) and w.gated else None
                if packed is not None:
                    return ops.gemv_f32(x, packed, torch.empty(M, inner, dtype=torch.float32, device=x.device), K, gated=True)
            else:
                plan = self.f32_gated_plan(M, inner, K)
                if plan is not None:
                    out = torch.empty(M, inner, dtype=torch.float32, device=x.device)
                    if plan[0]:
                        return ops.gemm_split(ops.split_rows(x), plain, out, gated=True, tile=plan[1])
                    return ops.gemm_f32(x, plain, out, gated=True, tile=plan[1])
        silu = activation == "silu"      # the row-ring kernel gates with silu only; the others take the activation
        fusable = (x.dtype == plain.dtype == self.dtype == torch.bfloat16 and K % 8 == 0 and x.stride(1) == 1
                   and x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0 and plain.is_contiguous())
        by_library = 16 < M <= MFMA_SKINNY_MAX_ROWS and self._gated_by_library(M, K, inner)
        if fusable and silu and self.rows_ring and 16 < M <= MFMA_SKINNY_MAX_ROWS and not by_library and (
                M > 32 or -(-inner // 32) <= self.compute_units * (2 if K <= RING_GROUP_K else 1)):
            # 33 to 64 rows (measured against the packed skinny kernel: 4-15 % faster at the 1B and 3B shapes, and
            # at wider ones in place of the library's product, which the packed kernel's registers leave them to);
            # from 17 rows on where the blocks come in one round, or in two where K is short (us at 17 / 24 / 32
            # rows against the packed kernel: width 2048, inner 8192: 14.0 / 14.3 / 14.3 against 16.4 / 17.7 / 18.2;
            # width 1536: 11.8 / 11.9 / 12.0 against 13.3 / 14.1 / 14.6; 3B: 10-15 %)
            return ops.gemm_rows(x, plain, torch.empty(M, inner, dtype=self.dtype, device=x.device), gated=True, once=self.streams_weights)
        if (isinstance(w, LinearWeight) and w.packable and w.gated and x.dtype == torch.bfloat16 and not by_library
                and M <= self.skinny_gated_rows and ops.gemv_mfma_supported(M, w.shape[0], K)
                and x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0):
            out = torch.empty(M, inner, dtype=self.dtype, device=x.device)
            return ops.gemv_mfma(x, w.packed, out, K, gated=True, activation=activation)
        if fusable and self.fused_gate_up_measured and M > MFMA_SKINNY_MAX_ROWS:
            # Short prompts: when all tiles of the product run at once (one block per compute unit,
            # most of the units busy), the fused kernel with a deep ring of stages streams the
            # weights faster than the library product and the gating pass after it (measured at
            # 65 to 320 rows: 5-25 % at widths of 1536 to 3072, 4 % at 4096; with a second round
            # of tiles the library is ahead).  The narrower tile first: it spreads over more units.
            m128 = -(-M // 128)
            for tile, pairs in (((128, 64, 6), 32), ((128, 128, 4), 64)):
                blocks = m128 * -(-inner // pairs)
                if self.compute_units // 4 <= blocks <= self.compute_units:
                    return ops.gemm_mfma(x, plain, torch.empty(M, inner, dtype=self.dtype, device=x.device),
                                         gated=True, tile=tile, activation=activation)
            # Longer prompts: tiles of 256x256, the ones that do not fill a round as halves (ops.gemm_duo), where the rounds are
            # full enough (us against the library's product and the gating pass, inner size 8192: width 2048, 512 / 1,000 / 1,300 /
            # 2,048 / 2,166 / 9,681 rows 31 / 43, 51 / 67, 76 / 97, 100 / 120, 118 / 146, 449 / 625; width 3072, 700 / 2,048 / 9,681
            # rows 69 / 73, 152 / 176, 665 / 863; width 4096, inner size 14336, 400 / 1,300 / 4,096 rows 87 / 94, 262 / 277,
            # 654 / 701; too little is full: that shape with 260 rows 86 / 71).  A lone round of halves at a K beyond RING_GROUP_K has to
            # be nearly full (width 3072 within prompts of 384 and 512 rows: 52 / 50 and equal; width 2048: 34 / 37).
            if M > 256:
                whole, rounds, fill = duo_plan(M, inner, self.compute_units, True)
                enough = DUO_GATED_LONE_FILL if rounds <= DUO_HALF and K > RING_GROUP_K else DUO_GATED_FILL
                out = torch.empty(M, inner, dtype=self.dtype, device=x.device) if fill >= enough else None
                if out is not None and ops.gemm_duo_takes(x, plain, out, gated=True):
                    return ops.gemm_mfma(x, plain, out, gated=True, tile=(256, 256), activation=activation, whole=whole)
            # 256x128 tiles that make one round on at least three quarters of the compute units, with rows
            # that fill their tiles to 85 % and more: measured against the library's product and the gating
            # kernel 11-16 % faster with a full round (512 rows of an inner size of 8192 at widths 2048 and
            # 3072; 900 and 1,024 rows of an inner size of 4096), 6 % with three quarters of one (700 and 768
            # rows, inner 4096); rows that fill their tiles less (320, 520, 600) are equal or 5 % behind, and
            # one and a half rounds and more 15-30 % behind.
            m256 = -(-M // 256)
            blocks = m256 * -(-inner // 64)
            if M > 256 and M * 20 >= m256 * 256 * 17 and self.compute_units * 3 // 4 <= blocks <= self.compute_units:
                return ops.gemm_mfma(x, plain, torch.empty(M, inner, dtype=self.dtype, device=x.device),
                                     gated=True, tile=(256, 128), activation=activation)
            # Long prompts of a width that gemm_duo does not take (no multiple of 128): gemm_mfma's tiles of 256x256 where they come in
            # whole rounds, K up to RING_GROUP_K and 4,096 rows (us against the library's product and the gating pass, in a graph:
            # width 1088, inner size 8192, 1,024 / 2,048 / 4,096 rows 36.9 / 46.4, 70.4 / 86.6, 137 / 158; width 1600 49.4 / 58.2, 98.7 /
            # 110, 187 / 201; width 1984 59.1 / 67.3, 120 / 122, 242 / 229; inner size 4096, 2,048 rows 35.9 / 44.5, 48.3 / 54.3, 58.4 / 63.9).
            if K <= RING_GROUP_K and 256 <= M <= 4096 and (-(-M // 256) * -(-inner // 128)) % self.compute_units == 0:
                return ops.gemm_mfma(x, plain, torch.empty(M, inner, dtype=self.dtype, device=x.device),
                                     gated=True, tile=(256, 256), activation=activation)
        if fusable and self.fused_gate_up_rows[0] <= M <= self.fused_gate_up_rows[1]:
            # the largest tile that still gives every compute unit a block (a tile of n columns holds n / 2 gated pairs)
            m256 = -(-M // 256)
            tile = ((256, 256) if m256 * -(-inner // 128) >= self.compute_units else
                    (256, 128) if m256 * -(-inner // 64) >= self.compute_units else (128, 128))
            return ops.gemm_mfma(x, plain, torch.empty(M, inner, dtype=self.dtype, device=x.device), gated=True, tile=tile, activation=activation)
        gu = self.linear(x, w if isinstance(w, LinearWeight) and not w.gated else plain)
        act = torch.empty(M, inner, dtype=gu.dtype, device=x.device)
        (ops.swiglu if silu else ops.gelu_glu)(gu, act)
        return act
