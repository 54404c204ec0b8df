"""Selection of hand-written gfx950 kernels for CKL kernel specializations.

Each library entry names the CKL kernel body it implements (its contract, from
ckl.decoder_kernels) and how to launch its gfx950 implementation (csrc/kernels/library.hip). A
specialization uses the library kernel only when

  1. its kernel IR, printed canonically, is identical to the contract body lowered with the
     same concrete signature (same shapes, dtypes and constexpr values), and
  2. every launch of it covers exactly the thread domain the library kernel computes
     (for example `linear` must be launched over y = B rows and x >= O columns).

Otherwise the kernel is compiled from its own IR (csrc/runtime/codegen.cpp), and `explain`
says why; a kernel that carries a library kernel's name without its body draws a warning. The
dependency graph is always derived from the CKL body, never from the library kernel; the
reference allows several implementations of one kernel when their observable effects agree
(specs/mlir-layout-aware-gpu-compiler-spec.md:241).
"""
from __future__ import annotations

import warnings
from dataclasses import dataclass
from typing import Callable, Optional

from .decoder_kernels import (add, advance, append_kv, attention_scores, attention_values, embedding, greedy, linear,
                              multiply, rms_apply, rms_stats, rope, silu, softmax, update)
from .frontend.checker import BoundSignature, bind
from .frontend.emitter import lower_kernel
from .frontend.source import Definition, FrontendError
from .types import BufferSpec


# ---------------------------------------------------------------------------- launches
BLOCK = 256
VALUES_BLOCK = 512      # kValuesBlock: attention_values workgroup (one per (b, h))
GREEDY_CHUNK = 4096     # kGreedyChunk: logits per greedy workgroup
GREEDY_ROW_THREADS = 1024   # one workgroup per row of at most 8 float4 per thread (kGreedyRowLoads)


def _cdiv(a: int, b: int) -> int:
    return (a + b - 1) // b


@dataclass(frozen=True)
class Launch:
    grid: int
    constants: tuple
    block: int = BLOCK
    shared: int = 0
    entry: str = ""          # entry point when the family has several (default ckl_<name>)
    # Device workspace the compiled plan gives the kernel: `workspace` bytes of state that reads
    # zero at every launch (zero page, completion counters), and, when `partials` >= 0, a second
    # pointer to `partials` bytes of split-reduction planes (0: a null pointer) that live only
    # until the kernel's readers have run, so the plan may share them between kernels.
    workspace: int = 0
    partials: int = -1
    # (members, Launch): the launch a dispatch takes instead when at least `members` dispatches
    # of the kernel in its block multiply the same first operand (siblings the inferred graph
    # runs as one shared-operand launch); the native prepare step picks it per dispatch, so every
    # run mode launches the same tiling.
    variants: tuple = ()


def _elementwise(count: int, inner: int) -> int:
    return _cdiv(count // 4 if inner % 4 == 0 else count, BLOCK)


def _embedding(shapes, consts, ext):
    (b,), (v, c) = shapes[0], shapes[1]
    return Launch(_elementwise(b * c, c), (b, c, v)) if ext[0] >= c and ext[1:] == (b, 1) else None


def _rms_stats(shapes, consts, ext):
    b, c = shapes[0]
    return Launch(b, (b, c)) if ext[0] >= b and ext[1:] == (1, 1) else None      # one workgroup per row


def _rms_apply(shapes, consts, ext):
    (b, c), (g, _c) = shapes[0], shapes[2]
    layer = consts[4]
    if not (0 <= layer < g) or not (ext[0] >= c and ext[1:] == (b, 1)):
        return None
    return Launch(_elementwise(b * c, c), (b, c, layer))


# Tiling of the linear family (csrc/kernels/library.hip, "linear"): output tiles of 64 columns
# (vector path) or 32*J columns (f32 MFMA path, 32 batch rows per tile), reduction slices of
# k_chunk rows shared by the 4 waves of a workgroup, and k_split slices combined through the
# workspace. A B = 32 f32 GEMV costs 16 MFMA FLOP per weight byte, so the MFMA work is two thirds
# of the HBM time and has to hide under the loads. Measured inside the large decode step on
# MI355X (weights not cached), it does so only with one workgroup (one wave per SIMD) per CU:
# with two or three workgroups per CU the MFMA and load phases of the waves sharing a SIMD stop
# overlapping and a launch costs close to the sum of its MFMA-only and load-only times (gate/up
# 33.6 us at 704 workgroups; 25.0 us on 176 workgroups), and a grid just over the CU count
# doubles. So the MFMA path picks, in the order J = 2, 4, 1, the first tiling whose grid fills at
# least LINEAR_MIN_FILL of LINEAR_TARGET_GROUPS workgroups without exceeding it (splitting K into
# slices of at least LINEAR_MIN_CHUNK rows), else the fullest. Sibling linears that multiply the
# same x (q/k/v, gate/up) then run in the inferred graph as one launch of the same grid in which
# every workgroup serves all of them (ckl_linear_mfma<J>x1_shared<M>, csrc/runtime/runtime.cpp).
# The inferred graph hands the split combine to the consuming chain kernel
# (csrc/runtime/chains.cpp), so splits there cost only their partial planes. The vector path
# (B <= 16, latency-bound) runs one workgroup per (64-column tile, batch row) whose up to 16
# waves take 64 reduction rows each, all loaded in one round trip; it splits only beyond 1024
# rows.
# Three or more siblings (q/k/v) try J = 1 first: each member then contributes 2 KB to a wave's
# stage (6 KB for three), and the grid of the same size splits K into half as many slices, so
# the launch writes half the partial planes and its consumer adds half as many. Measured on the
# large decoder's projections alone (cold weights, in sequence): q/k/v 14.7 us with J = 1 against
# 16.1-16.4 us with J = 2, while a single projection of the same shape is slower with J = 1
# (6.5 us against 7.2 us) and the gate/up pair is no faster with J = 2 (24.2 against 24.4 us).
# Reduction and output widths that are no multiple of 4 take the same kernels (4-byte-aligned vector
# loads; the last lane's columns move back into the row). One thread per output from the kernel's own
# IR, which they took before, re-reads every weight row for each request: norm -> linear -> greedy
# at 32 x 2048 x 32001 took 1643 us against 81 us, an MLP of 61 x 1500 x 4106 908 us against 78 us.
LINEAR_TARGET_GROUPS = 256    # MI355X compute units
LINEAR_EPILOGUE_COLUMN_BYTES = 4 * 16 * 64 * 4   # LDS per weight column of a lane (4 waves x 16 registers)
LINEAR_MIN_FILL = 0.85
LINEAR_MIN_CHUNK = 256
LINEAR_ZERO_PAGE = 256    # kZeroPage: leading workspace bytes that stay zero
LINEAR_VECTOR_ROWS = 16
LINEAR_VECTOR_WAVES = 16      # waves per vector-path workgroup at most (1024 threads)
LINEAR_VECTOR_WAVE_ROWS = 64  # kVectorRows: reduction rows per wave


LINEAR_SHARED_J1_MEMBERS = 3   # siblings from which the MFMA path tries J = 1 first

# At most 16 rows: ckl_linear_mfma16_<J> (16 rows x 16*J columns per wave) reads the weights once,
# the row-parallel kernel once per row, but the latter does not split up to 1024 reduction rows (so
# ordinary launches combine nothing) and fuses with the row ops around it. Measured (us a launch in a
# graph / ordinary, rows = 8, row-parallel -> MFMA): 2048 x 2048 in a 4-layer step 753 -> 262 us a
# step; 2048 x 1024 9.4/10.2 -> 6.2/8.9, 2048 x 512 7.2/8.3 -> 5.4/8.1, 1536 x 768 7.7/8.5 -> 5.4/8.1,
# but 1024 x 1024 6.9/7.0 -> 5.1/8.0 and 512 x 512 5.3/6.0 -> 5.0/7.6: so more reduction rows than the
# row-parallel kernel takes unsplit, and 2 MB of weights (4 rows of 1152 x 64, ordinary, lost 1 us).
# q/k/v groups need both that and 32 MB read for all rows (8 rows of 1024 x 1024, ordinary: a layer
# 46.1 -> 50.6 us). Expanding projections (gate/up, heads) fill the chip row by row and lose their
# fusion: there the weights read again for every row must be worth it (one row: 2048 x 32000 equal;
# 8 rows of 1024 x 8192 76 -> 56 us, of 256 x 32000 71 -> 41; 8 rows of 768 x 2048 48.4 -> 48.9, 2 of
# 512 x 8192 39.8 -> 40.9).
# J = 4 halves the workgroups that share a column; more than 8 splits cost more planes than they
# give (2048 x 1024: 8 splits of J = 2 6.2 us, 16 of J = 4 6.6 us).
LINEAR_MFMA16_MIN_CHUNK = 128
LINEAR_MFMA16_MAX_SPLIT = 8
LINEAR_VECTOR_UNSPLIT = LINEAR_VECTOR_WAVES * LINEAR_VECTOR_WAVE_ROWS


def _mfma_tiling(b: int, i: int, o: int, order, tile_rows: int, min_chunk: int, max_split: int):
    """(J, column tiles, K splits, slice rows) of an MFMA linear: the first J of `order` whose grid
    fills at least LINEAR_MIN_FILL of LINEAR_TARGET_GROUPS without exceeding it, else the fullest."""
    row_tiles = _cdiv(b, tile_rows)
    best = None
    for j in order:
        if j > o:                                  # a lane's j columns are columns of one row
            continue
        tiles = _cdiv(o, tile_rows * j)            # as many lanes hold columns as rows
        split = max(1, min(LINEAR_TARGET_GROUPS // (row_tiles * tiles), i // min_chunk, max_split))
        chunk = _cdiv(_cdiv(i, split), 16) * 16
        split = _cdiv(i, chunk)
        grid = row_tiles * tiles * split
        fill = grid / LINEAR_TARGET_GROUPS if grid <= LINEAR_TARGET_GROUPS else 0.5
        if best is None or fill > best[0]:
            best = (fill, j, tiles, split, chunk)
        if fill >= LINEAR_MIN_FILL:
            return best[1:]
    return best[1:]


def _takes_mfma16(b: int, i: int, o: int, members: int) -> bool:
    """Whether a linear of at most LINEAR_VECTOR_ROWS rows takes the 16-row MFMA kernel (the figures
    are above)."""
    weights = 4 * i * o
    if members >= LINEAR_SHARED_J1_MEMBERS:
        return i > LINEAR_VECTOR_UNSPLIT and b * weights >= 32 << 20
    if o > i:
        return b * weights >= 48 << 20 or (weights >= 8 << 20 and i >= LINEAR_VECTOR_UNSPLIT)
    return i > LINEAR_VECTOR_UNSPLIT and o >= 16 and weights >= 2 << 20


def linear_tiling(b: int, i: int, o: int, members: int = 1) -> dict:
    """Tiling of one linear (`members` = how many sibling linears of this shape multiply the same
    x and run as one shared-operand launch)."""
    block = BLOCK
    if b > LINEAR_VECTOR_ROWS:
        order = (1, 2, 4) if members >= LINEAR_SHARED_J1_MEMBERS else (2, 4, 1)
        j, tiles, split, chunk = _mfma_tiling(b, i, o, order, 32, LINEAR_MIN_CHUNK, LINEAR_TARGET_GROUPS)
        row_tiles = _cdiv(b, 32)
        rows = row_tiles * 32
        shared = j * LINEAR_EPILOGUE_COLUMN_BYTES      # the 4 waves' accumulator tiles, one pass
        entry = f"ckl_linear_mfma{j}x1"
    elif _takes_mfma16(b, i, o, members):
        order = (2, 4) if members >= LINEAR_SHARED_J1_MEMBERS else (4, 2)
        j, tiles, split, chunk = _mfma_tiling(b, i, o, order, 16, LINEAR_MFMA16_MIN_CHUNK, LINEAR_MFMA16_MAX_SPLIT)
        row_tiles, rows = 1, b                            # planes hold the batch rows only
        shared = j * LINEAR_EPILOGUE_COLUMN_BYTES // 4    # 4 accumulator registers a column
        entry = f"ckl_linear_mfma16_{j}x1"
    else:
        tiles = _cdiv(o, 64)
        waves = min(LINEAR_VECTOR_WAVES, _cdiv(i, LINEAR_VECTOR_WAVE_ROWS))
        chunk = LINEAR_VECTOR_WAVE_ROWS                   # rows per wave (kVectorRows)
        split = _cdiv(i, waves * chunk)
        rows, row_tiles = b, b                            # one workgroup per batch row
        shared = 0
        entry = "ckl_linear_rowvec"
        block = 64 * waves
    workspace, partials = LINEAR_ZERO_PAGE, 0
    if split > 1:
        workspace += _cdiv(4 * row_tiles * tiles, 256) * 256
        partials = 4 * split * rows * o
    return dict(grid=row_tiles * split * tiles, tiles=tiles, split=split, chunk=chunk, shared=shared, entry=entry,
                workspace=workspace, partials=partials, block=block)


def _linear(shapes, consts, ext):
    (b, i), (w, _i, o) = shapes[0], shapes[1]
    layer = consts[3]
    if not (0 <= layer < w) or not (ext[0] >= o and ext[1:] == (b, 1)):
        return None
    def launch(t, variants=()):
        return Launch(t["grid"], (b, i, o, layer, t["tiles"], t["split"], t["chunk"], 0), block=t["block"],
                      shared=t["shared"], entry=t["entry"], workspace=t["workspace"], partials=t["partials"],
                      variants=variants)

    t = linear_tiling(b, i, o)
    shared = linear_tiling(b, i, o, LINEAR_SHARED_J1_MEMBERS)
    variants = ((LINEAR_SHARED_J1_MEMBERS, launch(shared)),) if shared != t else ()
    return launch(t, variants)


def _rope(shapes, consts, ext):
    (b, c), (t, r, _two) = shapes[0], shapes[1]
    if c % (2 * r):
        return None
    a = c // (2 * r)
    if not (ext[0] >= r and ext[1:] == (a, b)):
        return None
    unit = 1 if r % 2 else 2      # rope_unit: pairs a thread rotates (two: 128-bit accesses)
    return Launch(_cdiv(b * a * (r // unit), BLOCK), (b, a, r, t))


def _append_kv(shapes, consts, ext):
    (b, c), (l, _b, a, t, d) = shapes[0], shapes[2]
    layer = consts[5]
    if a * d != c or not (0 <= layer < l) or not (ext[0] >= d and ext[1:] == (a, b)):
        return None
    return Launch(_elementwise(b * a * d, d), (l, b, a, t, d, layer))


def _scores(shapes, consts, ext):
    (b, c), (l, _b, a, t, d) = shapes[0], shapes[1]
    layer = consts[5]
    if a * d != c or not (0 <= layer < l) or not (ext[0] >= t and ext[1:] == (a, b)):
        return None
    return Launch(b * a * _cdiv(t, BLOCK), (l, b, a, t, d, layer))


def _softmax(shapes, consts, ext):
    b, a, t = shapes[0]
    if not (ext[0] >= b and ext[1:] == (a, 1)):
        return None
    # One wave per row, or a workgroup: 256 threads, or 1024 on rows so long that the values of few
    # rows are always split, so that no chain wants softmax and values in one workgroup (256 threads
    # stream a row of more than 2048 three times: 16 rows of 8001 19.7 -> 5.4 us).
    row_threads = 64 if t <= 512 else 1024 if t > SOFTMAX_WIDE_ROW and b * a <= VALUES_SPLIT_HEADS else 256
    block = max(BLOCK, row_threads)
    return Launch(_cdiv(b * a, block // row_threads), (b, a, t, row_threads), block=block)


# Long contexts of few requests: a workgroup per (b, h) row leaves most of the chip idle, and one
# workgroup streams only ~50 GB/s. The rows are then cut into slices (ckl_attention_values_split),
# and the chain that needs a whole row in one workgroup becomes two launches (rope -> append_kv ->
# scores, softmax -> values). At least 512 KB of values a row pay for that once about half the capacity
# is in use, and 16 KB more of them for every (b, h) row (attention layer at the end of the capacity,
# chain -> split, graph us: 16 rows of 8192 x 128 196 -> 66, of 1040 x 128 59 -> 52 (row 520 51 -> 50, row
# 100 41 -> 47), of 700 x 128 46 -> 50 and of 512 x 128 43 -> 49 as three launches; 64 rows of 1040 x 128
# 64 -> 59, but at row 520 53.5 -> 54.5; 128 rows of 2048 x 128 88 -> 90 as three launches).
# About VALUES_SPLIT_GROUPS workgroups, but 16 slices or one per 128 KB (8 rows of 8192 x 64: 16 slices
# 34.5, 64 37.4, 128 44.3 us: the last workgroup adds them; 4 rows of 8192 x 128: 16 41.0, 32 38.4).
# One workgroup of 512 threads per compute unit (attention layer, us, 16 rows of 8192 x 128 / 64 rows of
# 4096 x 64: 512 of 256 threads 72.1 / 72.3, 512 of 512 71.5 / 72.3, 384 of 512 68.7 / 72.7, 256 of 512
# 67.4 / 70.2, 192 of 512 68.2 / 71.4; 256 of 256 69.8 / 72.5).
VALUES_SPLIT_HEADS = 64
VALUES_SPLIT_BYTES = 1 << 19
VALUES_SPLIT_HEAD_BYTES = 1 << 14
VALUES_SPLIT_GROUPS = 256
SOFTMAX_WIDE_ROW = 6144


def _values_slices(heads: int, t: int, d: int) -> int:
    """Slices per (b, h) row of the values' sum (1: one workgroup a row)."""
    if heads > VALUES_SPLIT_HEADS or d % 4 or d > 256:
        return 1
    if t <= SOFTMAX_WIDE_ROW and 4 * t * d < max(VALUES_SPLIT_BYTES, heads * VALUES_SPLIT_HEAD_BYTES):
        return 1
    return max(1, min(_cdiv(VALUES_SPLIT_GROUPS, heads), max(16, 4 * t * d >> 17), t // 64))


def _values(shapes, consts, ext):
    (b, a, t), (l, _b, _a, _t, d), (_b2, c) = shapes[0], shapes[1], shapes[3]
    layer = consts[4]
    if a * d != c or not (0 <= layer < l) or not (ext[0] >= d and ext[1:] == (a, b)):
        return None
    # Enough row groups to keep ~8 rows in flight per lane over the whole capacity, at least one
    # wave, at most VALUES_BLOCK threads; D/4 lanes own a row.
    width = d // 4 if d % 4 == 0 and d <= 256 else 64
    block = 64
    while block < VALUES_BLOCK and (block // width) * 8 < t:
        block *= 2
    slices = _values_slices(b * a, t, d)
    if slices > 1:
        return Launch(b * a * slices, (l, b, a, t, d, layer, slices), block=VALUES_BLOCK, entry="ckl_attention_values_split",
                      workspace=_cdiv(4 * b * a, 256) * 256, partials=4 * b * a * slices * d)
    return Launch(b * a, (l, b, a, t, d, layer), block=block)


def _binary(shapes, consts, ext):
    (b, c) = shapes[0]
    return Launch(_elementwise(b * c, c), (b * c,)) if ext[0] >= c and ext[1:] == (b, 1) else None


def _unary(shapes, consts, ext):
    (b, c) = shapes[0]
    return Launch(_elementwise(b * c, c), (b * c,)) if ext[0] >= c and ext[1:] == (b, 1) else None


def _greedy(shapes, consts, ext):
    (b, v), (t, _b) = shapes[0], shapes[2]
    if not (ext[0] >= b and ext[1:] == (1, 1)):
        return None
    workspace = _cdiv(12 * b + 4, 256) * 256       # keys, counters, row count (greedy -> advance chain)
    if GREEDY_CHUNK < v <= 8 * 4 * GREEDY_ROW_THREADS and v % 4 == 0:
        return Launch(b, (b, v, t, 1), block=GREEDY_ROW_THREADS, workspace=workspace)
    chunks = _cdiv(v, GREEDY_CHUNK)
    return Launch(b * chunks, (b, v, t, chunks), workspace=workspace)


def _advance(shapes, consts, ext):
    return Launch(1, (), block=64) if ext == (1, 1, 1) else None


def _update(shapes, consts, ext):
    (n,) = shapes[0]
    return Launch(_elementwise(n, n), (n,)) if ext[0] >= n and ext[1:] == (1, 1) else None


@dataclass(frozen=True)
class LibraryKernel:
    name: str
    contract: Definition
    launch: Callable
    groupable: bool = False

    @property
    def entry_point(self) -> str:
        return f"ckl_{self.name}"


LIBRARY = (
    LibraryKernel("embedding", embedding, _embedding),
    LibraryKernel("rms_stats", rms_stats, _rms_stats),
    LibraryKernel("rms_apply", rms_apply, _rms_apply),
    LibraryKernel("linear", linear, _linear, groupable=True),
    LibraryKernel("rope", rope, _rope, groupable=True),
    LibraryKernel("append_kv", append_kv, _append_kv),
    LibraryKernel("attention_scores", attention_scores, _scores),
    LibraryKernel("softmax", softmax, _softmax),
    LibraryKernel("attention_values", attention_values, _values),
    LibraryKernel("add", add, _binary),
    LibraryKernel("silu", silu, _unary),
    LibraryKernel("multiply", multiply, _binary),
    LibraryKernel("greedy", greedy, _greedy),
    LibraryKernel("advance", advance, _advance),
    LibraryKernel("update", update, _update),
)


def _rebind(contract: Definition, signature: BoundSignature) -> Optional[BoundSignature]:
    names = [a.arg for a in contract.tree.args.args]
    if len(names) != len(signature.parameters):
        return None
    runtime = {n: p.dtype for n, p in zip(names, signature.parameters) if not p.is_constant}
    constants = {n: p.value for n, p in zip(names, signature.parameters) if p.is_constant}
    try:
        return bind(contract, runtime, constants)
    except FrontendError:
        return None


@dataclass(frozen=True)
class Selection:
    symbol: str
    kernel: LibraryKernel
    launch: Launch


class LibraryNameWarning(UserWarning):
    """A kernel named like a library kernel is compiled from its own body instead."""


def explain(lowered) -> dict:
    """Per kernel symbol of `lowered`: ("library", entry point) when a library kernel serves it,
    ("jit", reason) otherwise."""
    report = {}
    for spec, text, extents in zip(lowered.specializations, lowered.kernels, lowered.extents):
        report[spec.symbol] = ("jit", "no library kernel has this body")
        for entry in LIBRARY:
            bound = _rebind(entry.contract, spec.signature)
            if bound is None or lower_kernel(entry.contract, bound) != text:
                continue
            shapes = [p.dtype.shape if isinstance(p.dtype, BufferSpec) else None for p in spec.signature.parameters]
            consts = [p.value if p.is_constant else None for p in spec.signature.parameters]
            launches = {entry.launch(shapes, consts, ext) for ext in extents}
            if len(launches) == 1 and None not in launches:
                launch = launches.pop()
                report[spec.symbol] = ("library", Selection(spec.symbol, entry, launch))
            else:
                report[spec.symbol] = ("jit", f"body of library kernel {entry.name}, but launched over threads "
                                              f"{sorted(extents)} that its gfx950 kernel does not cover")
            break
        kind, detail = report[spec.symbol]
        named = spec.definition.name if spec.definition is not None else ""
        if kind == "jit" and any(entry.name == named for entry in LIBRARY):
            warnings.warn(f"kernel '{named}' ({spec.symbol}) is compiled from its own IR: {detail}", LibraryNameWarning,
                          stacklevel=3)
    return report


def select(lowered) -> dict:
    """Map kernel symbols of `lowered` to library selections (unselected kernels are JIT-compiled)."""
    return {symbol: detail for symbol, (kind, detail) in explain(lowered).items() if kind == "library"}


def selection_attribute(selections: dict, artifact: str) -> str:
    """Module attribute text `ckl.hip.selection = {...}` consumed by the native prepare step."""
    entries = []
    for symbol, s in sorted(selections.items()):
        fields = [f'artifact = "{artifact}"', f"block = array<i64: {s.launch.block}, 1, 1>",
                  "constants = [" + ", ".join(f"{int(c)} : i32" for c in s.launch.constants) + "]",
                  f'entry_point = "{s.launch.entry or s.kernel.entry_point}"', f"grid = array<i64: {s.launch.grid}, 1, 1>",
                  f'implementation = "ckl.hip.library.{s.kernel.name}"', f"shared_memory = {s.launch.shared} : i64"]
        if s.launch.workspace:
            fields.append(f"workspace = {s.launch.workspace} : i64")
        if s.launch.partials >= 0:
            fields.append(f"partials = {s.launch.partials} : i64")
        if s.launch.variants:
            variants = []
            for members, v in s.launch.variants:
                variant = [f"block = array<i64: {v.block}, 1, 1>",
                           "constants = [" + ", ".join(f"{int(c)} : i32" for c in v.constants) + "]",
                           f'entry_point = "{v.entry or s.kernel.entry_point}"', f"grid = array<i64: {v.grid}, 1, 1>",
                           f"members = {members} : i64", f"shared_memory = {v.shared} : i64",
                           f"workspace = {v.workspace} : i64", f"partials = {v.partials} : i64"]
                variants.append("{" + ", ".join(variant) + "}")
            fields.append("variants = [" + ", ".join(variants) + "]")
        if s.kernel.groupable:
            fields.append(f'group = "{s.kernel.name}"')
        entries.append(f"{symbol} = {{{', '.join(sorted(fields))}}}")
    return "ckl.hip.selection = {" + ", ".join(entries) + "}"
