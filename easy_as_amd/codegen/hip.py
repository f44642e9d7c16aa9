"""eas IR -> gfx950 HIP C++ (the backend's code generator).

``ir_to_hip(ir)`` returns a :class:`Lowered` with the source, the reference's
``(block_size, launch_mode)`` pair (reference contract: ``ir_to_msl`` at
``eas/codegen/msl.py:353``) and a :class:`Geometry` telling the runtime how a
reference-level launch (programs / threadgroups) maps onto HIP workgroups.

Execution model on MI355X (CDNA4, wave64):

* **spmd** (``mk.arange``): the reference runs one program per Metal thread,
  walking its BLOCK lanes serially (``msl.py:98-350``).  Here a program is
  spread across ``T`` threads; each thread owns ``LPT`` lanes in chunks of
  ``VEC`` consecutive lanes (4 x f32 / 8 x f16 = 16 bytes) so lane-contiguous
  accesses become ``global_load_dwordx4`` / ``global_store_dwordx4``.  A
  16-byte group takes the vector path only when all its lanes are unmasked,
  its offsets are consecutive and its address is 16-byte aligned; any other
  group uses masked scalar accesses, so every kernel keeps the reference's
  per-lane semantics (masked load -> 0, masked store -> no write).  Small
  programs are packed ``PPW`` per workgroup.  ``alloc_tg`` stays private per
  program, and a ``__syncthreads`` is inserted between memory accesses that
  one Metal thread did in order but that now run on different threads.
* **thread** (``mk.tid``): one threadgroup = one workgroup of BLOCK threads,
  ``alloc_tg`` = LDS, ``barrier`` = ``__syncthreads``.  ``lane_id``/``sg_id``
  describe 32-lane virtual simdgroups (``threadIdx.x % 32`` / ``/ 32``).
  Metal's non-uniform ``dispatchThreads`` is emulated by a hidden
  ``__eas_nthreads`` argument: threads past it have no side effects.

Float semantics: kernels are compiled with ``-ffp-contract=off`` so FMAs come
only from the IR (``fma`` op); float literals are printed as the reference
prints them (``repr(v) + 'f'``, ``msl.py:25-34``) so both compilers round the
same decimal.
"""

from __future__ import annotations

import math
import os
from dataclasses import dataclass, field, replace
from typing import Any, Iterable

from ..ir import DType, IRModule, Inst, ValueRef

# ---------------------------------------------------------------------------
# results
# ---------------------------------------------------------------------------


@dataclass(frozen=True)
class Geometry:
    """How the runtime turns a reference-level launch into a HIP dispatch.

    kind ``spmd``: logical grid = programs; physical grid.x =
    ceil(programs.x / (ppw * unroll)) * split, block = ``wg_size``; hidden arg =
    programs.x.  ``split`` > 1 spreads each program's lanes over that many
    workgroups (then ``ppw`` is 1).
    kind ``thread``: logical = threadgroups of ``block_size`` threads (or a 1-D
    thread count); hidden arg = number of live threads along x.
    A thread kernel's ``params["gemm"]`` is the geometry of the GEMM that computes the same for a
    launch by whole threadgroups.
    kind ``gemm``: a lifted matmul; ``params`` describe its own tiling.
    """

    kind: str
    entry: str
    block_size: int
    wg_size: int
    programs_per_wg: int = 1
    unroll: int = 1
    params: dict[str, Any] = field(default_factory=dict)
    split: int = 1


@dataclass(frozen=True)
class Lowered:
    src: str
    block_size: int
    launch_mode: str
    geometry: Geometry


# ---------------------------------------------------------------------------
# shared helpers
# ---------------------------------------------------------------------------

_CTYPE = {DType.F32: "float", DType.F16: "_Float16", DType.BF16: "__bf16", DType.U32: "uint32_t", DType.BOOL: "bool"}

PRELUDE = """\
// Generated by easy_as_amd.codegen.hip for gfx950 (CDNA4, wave64).
#pragma clang fp contract(off)
typedef unsigned int uint32_t;
typedef unsigned long long uint64_t;
typedef float eas_f32x4 __attribute__((ext_vector_type(4)));
typedef float eas_f32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 eas_f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 eas_f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 eas_f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 eas_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 eas_bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 eas_bf16x2 __attribute__((ext_vector_type(2)));
static __device__ __forceinline__ uint32_t eas_f2u(float x) {
  // saturating float -> u32 (NaN -> 0): a defined result for every input
  return x != x ? 0u : (x <= 0.0f ? 0u : (x >= 4294967296.0f ? 0xffffffffu : (uint32_t)x));
}
"""

# Added to sources that use an fma on 16-bit values (see ``with_helpers``).
FMA16_HELPERS = """// 16-bit fma: the exact x*y+z rounded to binary32, then to the 16-bit type (two roundings).
// The empty asm keeps the compiler from merging the pair into v_fma_mixlo_f16, which
// rounds the exact value to binary16 once and so differs on some inputs.
static __device__ __forceinline__ _Float16 eas_fma_f16(_Float16 x, _Float16 y, _Float16 z) {
  float f = __builtin_fmaf((float)x, (float)y, (float)z);
  __asm__ volatile("" : "+v"(f));
  return (_Float16)f;
}
static __device__ __forceinline__ __bf16 eas_fma_bf16(__bf16 x, __bf16 y, __bf16 z) {
  float f = __builtin_fmaf((float)x, (float)y, (float)z);
  __asm__ volatile("" : "+v"(f));
  return (__bf16)f;
}
"""


# Added to sources that convert to a 16-bit type (see ``with_helpers``).
CVT16_HELPERS = """// Conversion to a 16-bit type of a value already rounded to binary32.  The empty asm keeps the
// compiler from folding the instruction that produced the value into the conversion: a
// v_fma_mixlo_f16 / v_mad_mixlo_f16 rounds the exact product or sum to binary16 once, which
// differs on some inputs from rounding to binary32 first.
static __device__ __forceinline__ _Float16 eas_f32_to_f16(float f) {
  __asm__ volatile("" : "+v"(f));
  return (_Float16)f;
}
static __device__ __forceinline__ __bf16 eas_f32_to_bf16(float f) {
  __asm__ volatile("" : "+v"(f));
  return (__bf16)f;
}
"""


def with_helpers(lines: list[str]) -> str:
    """The emitted lines as one source, with the 16-bit fma and conversion helpers after the
    prelude when the kernel calls them."""
    src = "\n".join(lines) + "\n"
    extra = ""
    if "eas_fma_f16(" in src or "eas_fma_bf16(" in src:
        extra += FMA16_HELPERS
    if "eas_f32_to_f16(" in src or "eas_f32_to_bf16(" in src:
        extra += CVT16_HELPERS
    return src.replace(PRELUDE, PRELUDE + extra, 1) if extra else src


def ctype(dt: DType) -> str:
    try:
        return _CTYPE[dt]
    except KeyError:
        raise ValueError(f"unsupported dtype for HIP codegen: {dt}") from None


def literal(value: Any, dt: DType) -> str:
    """C++ literal for an IR const of dtype ``dt``."""
    if dt == DType.BOOL:
        return "true" if value else "false"
    if dt == DType.U32:
        v = int(value)
        if v < 0:
            raise ValueError("negative constants not supported")
        return f"{v}u" if v < (1 << 32) else f"((uint32_t){v}ull)"
    if dt in (DType.F32, DType.F16, DType.BF16):
        f = float(value)
        if math.isnan(f):
            text = '__builtin_nanf("")'
        elif math.isinf(f):
            text = "__builtin_inff()" if f > 0 else "(-__builtin_inff())"
        else:
            text = (repr(f) if isinstance(value, float) else f"{int(value)}.0") + "f"
        return text if dt == DType.F32 else f"(({_CTYPE[dt]}){text})"
    raise ValueError(f"unsupported const dtype: {dt}")


def zero(dt: DType) -> str:
    return {DType.F32: "0.0f", DType.F16: "((_Float16)0.0f)", DType.BF16: "((__bf16)0.0f)", DType.U32: "0u",
            DType.BOOL: "false"}[dt]


def cast_expr(x: str, src: DType, dst: DType) -> str:
    """Value-converting cast with defined results for every input."""
    if src == dst:
        return x
    if dst == DType.BOOL:
        return f"({x} != {zero(src)})"
    if src == DType.BOOL:
        return f"({x} ? {literal(1.0 if dst != DType.U32 else 1, dst)} : {zero(dst)})"
    if dst == DType.U32:
        return f"eas_f2u((float)({x}))"
    if dst in (DType.F16, DType.BF16):
        # through binary32 (exact from f16/bf16; u32 rounds to binary32 first), then one
        # rounding to the 16-bit type that the compiler may not merge with the producer
        helper = "eas_f32_to_f16" if dst == DType.F16 else "eas_f32_to_bf16"
        return f"{helper}({x})" if src == DType.F32 else f"{helper}((float)({x}))"
    return f"(({ctype(dst)})({x}))"


def binop_expr(op: str, dt: DType, x: str, y: str) -> str:
    """``x op y`` for operands of dtype ``dt``.  bf16 arithmetic runs in f32 and
    rounds once to bf16: f32's 24 bits are at least 2 * 8 + 2, so the sum or
    product of two bf16 values rounded to f32 and then to bf16 is the correctly
    rounded bf16 result."""
    if dt == DType.BF16 and op in ("add", "mul", "lt"):
        e = f"(float){x} {_BINOP[op]} (float){y}"
        return f"({e})" if op == "lt" else f"((__bf16)({e}))"
    return f"{x} {_BINOP[op]} {y}"


def infer_block_and_mode(ir: IRModule) -> tuple[int, str]:
    """``arange`` sizes -> ("spmd", BLOCK); ``tid`` sizes -> ("thread", BLOCK).

    Mixing the two, or two different sizes of one, is an error
    (reference ``msl.py:59-95``).
    """
    ar = {int(i.args[1]) for i in ir.insts if i.op == "arange"}
    td = {int(i.args[1]) for i in ir.insts if i.op == "tid"}
    if len(ar) > 1:
        raise ValueError("multiple arange sizes not supported")
    if len(td) > 1:
        raise ValueError("multiple tid sizes not supported")
    if ar and td:
        raise ValueError("kernel must not mix mk.arange(...) and mk.tid(...)")
    if ar:
        return ar.pop(), "spmd"
    if td:
        return td.pop(), "thread"
    raise ValueError("kernel must use mk.arange(0, BLOCK) (spmd) or mk.tid(0, BLOCK) (thread) to define BLOCK")


class _Module:
    """Per-IR facts shared by both emitters."""

    def __init__(self, ir: IRModule) -> None:
        self.ir = ir
        self.defs: dict[int, Inst] = {}
        self.arg_name: dict[int, str] = {}
        self.tg_ids: set[int] = set()
        self.uses: dict[int, int] = {}
        for inst in ir.insts:
            if inst.out is not None:
                self.defs[inst.out.id] = inst
            if inst.op == "arg":
                self.arg_name[inst.out.id] = str(inst.args[0])
            elif inst.op == "alloc_tg":
                self.tg_ids.add(inst.out.id)
            for a in inst.args:
                if isinstance(a, ValueRef):
                    self.uses[a.id] = self.uses.get(a.id, 0) + 1
        self.written = {
            self.arg_name[i.args[0].id]
            for i in ir.insts
            if i.op in ("store", "mma_store") and i.args[0].id in self.arg_name
        }

    def name(self, ref: ValueRef) -> str:
        return self.arg_name.get(ref.id, f"v{ref.id}")

    def const(self, ref: ValueRef) -> Any:
        d = self.defs.get(ref.id)
        return d.args[0] if d is not None and d.op == "const" else None

    def is_true(self, ref: ValueRef) -> bool:
        return self.const(ref) is True

    def params(self, hidden: Iterable[str]) -> str:
        ps = []
        for arg in self.ir.args:
            if arg.kind == "buffer":
                const = "" if arg.name in self.written else "const "
                ps.append(f"{const}{ctype(arg.dtype)}* __restrict__ {arg.name}")
            else:
                ps.append(f"const {ctype(arg.dtype)} {arg.name}")
        ps.extend(f"const uint32_t {h}" for h in hidden)
        return ",\n    ".join(ps)


def _env_int(name: str, default: int) -> int:
    v = os.environ.get(name, "").strip()
    return int(v) if v else default


_BINOP = {"add": "+", "mul": "*", "floordiv": "/", "mod": "%", "lt": "<", "and": "&&", "or": "||"}

# ---------------------------------------------------------------------------
# SPMD emitter
# ---------------------------------------------------------------------------

_SPMD_FORBIDDEN = {"tid", "local_id", "lane_id", "sg_id", "dot", "mma_zero", "mma", "mma_store"}


def _has_dense_store(ir: IRModule) -> bool:
    """True if some global store writes a multi-lane value under a mask that depends
    on indices only (not on loaded data): a dense output stream."""
    tg = {i.out.id for i in ir.insts if i.op == "alloc_tg" and i.out is not None}
    tainted: set[int] = set()
    for inst in ir.insts:
        if inst.out is None:
            continue
        if inst.op == "load" or any(getattr(x, "id", None) in tainted for x in inst.args):
            tainted.add(inst.out.id)
    for inst in ir.insts:
        if inst.op == "store":
            buf, off, val, mask = inst.args
            if buf.id not in tg and max(off.lanes, val.lanes) > 1 and mask.id not in tainted:
                return True
    return False


class _SpmdEmitter:
    """Programs of BLOCK lanes.  ``thread_mode``: ``ir`` is a thread-mode kernel in program-of-lanes
    form (``thread_lanes.as_lanes``): one program per threadgroup, the live thread count an argument
    of the IR, and the launch and geometry those of a thread-mode kernel."""

    def __init__(self, ir: IRModule, block: int, thread_mode: bool = False) -> None:
        self.thread_mode = thread_mode
        for inst in ir.insts:
            if inst.op in _SPMD_FORBIDDEN:
                raise ValueError(f"op {inst.op!r} is not supported in spmd mode (use mk.tid for thread-level kernels)")
        self.m = _Module(ir)
        self.ir = ir
        self.block = block
        widths = [2 if a.dtype in (DType.F16, DType.BF16) else 4 for a in ir.args if a.kind == "buffer"] or [4]
        vec = 16 // max(widths)
        while vec > 1 and block % vec:
            vec //= 2
        # Lanes per thread, measured on MI355X (N = 2^28 f32): kernels that write a
        # dense output stream run best with one 16-byte vector per thread (write-only
        # 84 %, copy 81 %, fma 79 % of HBM, add unchanged at 81-82 %); kernels that
        # only read (or store sparsely, under data-dependent masks) keep 64 bytes per
        # thread in flight (read-only 88 % vs 84 %).  Fewer when BLOCK does not allow it.
        default_bytes = 16 if _has_dense_store(ir) else 64
        lanes_per_thread = _env_int("EAS_HIP_SPMD_LPT", default_bytes // max(widths))
        while lanes_per_thread > vec and (lanes_per_thread % vec or block % lanes_per_thread):
            lanes_per_thread //= 2
        if lanes_per_thread % vec or block % lanes_per_thread:
            lanes_per_thread = vec
        while block // lanes_per_thread > 1024:
            lanes_per_thread *= 2
            if block % lanes_per_thread:
                raise ValueError(f"spmd BLOCK={block} cannot be mapped onto <= 1024 threads")
        self.vec = vec
        self.lpt = lanes_per_thread
        self.T = block // lanes_per_thread
        self.sync_before = self.plan_syncs()
        # A program's lanes may be spread over several workgroups when nothing in it orders
        # one lane's memory accesses after another's: no threadgroup memory, no barrier and no
        # store/load hazard on a buffer (each of those needs the program in one workgroup).
        splittable = not self.sync_before and not any(i.op in ("alloc_tg", "barrier") for i in ir.insts)
        target_wg = _env_int("EAS_HIP_SPMD_WG", 0) or self.default_wg_threads(default_bytes)
        if target_wg < 1 or target_wg > 1024 or target_wg & (target_wg - 1):
            raise ValueError(f"EAS_HIP_SPMD_WG must be a power of two in [1, 1024], got {target_wg}")
        if self.T > target_wg and splittable and self.T % target_wg == 0:
            # the program's T threads over T / target_wg workgroups (a split must cover every
            # thread: a BLOCK whose thread count the workgroup size does not divide keeps its
            # program in one workgroup)
            self.split, self.ppw, self.wg = self.T // target_wg, 1, target_wg
        else:
            self.split = 1
            self.ppw = max(1, target_wg // self.T)
            self.wg = self.T * self.ppw
        self.unroll = max(1, _env_int("EAS_HIP_SPMD_UNROLL", 1))
        # Streaming (nt) global loads/stores: +5-7% HBM bandwidth on MI355X for SPMD kernels.
        self.nontemporal = _env_int("EAS_HIP_SPMD_NT", 1) != 0
        self.lines: list[str] = []

    def default_wg_threads(self, bytes_per_thread: int) -> int:
        """Threads per workgroup for this kernel, from its number of HBM streams.

        Measured on MI355X at N = 2^28 f32 with 16 bytes per lane (one workgroup per
        chunk, every chunk of every stream ``threads * 16`` bytes): the fewer bytes a
        workgroup moves per stream the better HBM serves the mix of streams (add: 512 B
        7.08 TB/s, 1 KiB 6.67, 4 KiB 6.45), until the command processor's dispatch rate
        of about 4.7 workgroups per ns caps the launch (copy at 512 B per stream: 4.8
        TB/s, at 1 KiB 6.68; fill at 1 KiB 4.8, at 4 KiB 6.82).  So a kernel with one
        stream takes 4 KiB per workgroup, two streams 1 KiB, three or more 512 B
        (add, fma: 32 threads, half a wave).  Kernels without a dense output stream
        keep 256 threads of ``bytes_per_thread``."""
        if bytes_per_thread != 16:
            return 256
        streams = sum(1 for i in self.ir.insts if i.op in ("load", "store")
                      and i.args[0].id not in self.m.tg_ids and i.args[1].lanes > 1)
        per_stream = 4096 if streams <= 1 else (1024 if streams == 2 else 512)
        return per_stream // 16

    # -- lane access -------------------------------------------------------
    def lane_index(self, j: int) -> str:
        """Global lane index (within the program) of this thread's element j."""
        r, e = divmod(j, self.vec)
        off = r * self.T * self.vec + e
        return f"(__lbase + {off}u)" if off else "__lbase"

    def at(self, ref: ValueRef, j: int) -> str:
        n = self.m.name(ref)
        return n if ref.lanes == 1 else f"{n}[{j}]"

    def elems(self, out: ValueRef) -> range:
        return range(self.lpt if out.lanes > 1 else 1)

    def decl(self, out: ValueRef) -> str:
        ty = ctype(out.dtype)
        return f"{ty} v{out.id}[{self.lpt}]" if out.lanes > 1 else f"{ty} v{out.id}"

    def assign(self, out: ValueRef, j: int) -> str:
        return f"v{out.id}[{j}]" if out.lanes > 1 else f"v{out.id}"

    # -- memory --------------------------------------------------------------
    def buf_expr(self, ref: ValueRef) -> str:
        if ref.id in self.m.tg_ids:
            return f"v{ref.id}[__slot]" if self.ppw > 1 else f"v{ref.id}"
        return self.m.name(ref)

    def emit_load(self, inst: Inst, ind: str, live: str | None) -> None:
        out = inst.out
        buf, off, mask = inst.args
        b = self.buf_expr(buf)
        ty = ctype(out.dtype)
        self.lines.append(f"{ind}{self.decl(out)};")
        is_tg = buf.id in self.m.tg_ids

        def masked(j: int) -> str:
            conds = [] if self.m.is_true(mask) else [self.at(mask, j)]
            if live:
                conds.append(live)
            return " && ".join(conds)

        if out.lanes == 1:
            cond = masked(0)
            if cond:
                self.lines.append(f"{ind}{self.assign(out, 0)} = {zero(out.dtype)};")
                self.lines.append(f"{ind}if ({cond}) {self.assign(out, 0)} = {b}[{self.at(off, 0)}];")
            else:
                self.lines.append(f"{ind}{self.assign(out, 0)} = {b}[{self.at(off, 0)}];")
            return
        vbytes = self.vec * (2 if out.dtype in (DType.F16, DType.BF16) else 4)
        vty = _vec_type(out.dtype, self.vec)
        for g in range(self.lpt // self.vec):
            j0 = g * self.vec
            js = range(j0, j0 + self.vec)
            conds = [c for c in (masked(j) for j in js) if c]
            conds += [f"{self.at(off, j)} == {self.at(off, j0)} + {j - j0}u" for j in js if j != j0]
            if vty is not None and not is_tg:
                p = f"__p{out.id}_{g}"
                self.lines.append(f"{ind}const {ty}* {p} = {b} + {self.at(off, j0)};")
                conds.append(f"(((uint64_t){p}) & {vbytes - 1}ull) == 0ull")
                load = (f"__builtin_nontemporal_load((const {vty}*){p})" if self.nontemporal
                        else f"*(const {vty}*){p}")
                self.lines.append(f"{ind}if ({' && '.join(conds) or 'true'}) {{")
                t = f"__t{out.id}_{g}"
                self.lines.append(f"{ind}  const {vty} {t} = {load};")
                for e, j in enumerate(js):
                    self.lines.append(f"{ind}  v{out.id}[{j}] = {t}[{e}];")
                self.lines.append(f"{ind}}} else {{")
                inner = ind + "  "
            else:
                inner = ind
            for j in js:
                c = masked(j)
                src = f"{b}[{self.at(off, j)}]"
                if c:
                    self.lines.append(f"{inner}v{out.id}[{j}] = ({c}) ? {src} : {zero(out.dtype)};")
                else:
                    self.lines.append(f"{inner}v{out.id}[{j}] = {src};")
            if vty is not None and not is_tg:
                self.lines.append(f"{ind}}}")

    def emit_store(self, inst: Inst, ind: str, live: str | None) -> None:
        buf, off, val, mask = inst.args
        b = self.buf_expr(buf)
        is_tg = buf.id in self.m.tg_ids

        def masked(j: int) -> str:
            conds = [] if self.m.is_true(mask) else [self.at(mask, j)]
            if live:
                conds.append(live)
            return " && ".join(conds)

        if off.lanes == 1:
            # A program-uniform store: one thread of the program performs it.
            conds = ["__t == 0u"] + ([masked(0)] if masked(0) else [])
            self.lines.append(f"{ind}if ({' && '.join(conds)}) {b}[{self.at(off, 0)}] = {self.at(val, 0)};")
            return
        dt = buf.dtype
        vbytes = self.vec * (2 if dt in (DType.F16, DType.BF16) else 4)
        vty = _vec_type(dt, self.vec)
        for g in range(self.lpt // self.vec):
            j0 = g * self.vec
            js = range(j0, j0 + self.vec)
            if vty is not None and not is_tg:
                conds = [c for c in (masked(j) for j in js) if c]
                conds += [f"{self.at(off, j)} == {self.at(off, j0)} + {j - j0}u" for j in js if j != j0]
                p = f"__q{g}_{len(self.lines)}"  # unique by position: the text is the same in every process
                self.lines.append(f"{ind}{ctype(dt)}* {p} = {b} + {self.at(off, j0)};")
                conds.append(f"(((uint64_t){p}) & {vbytes - 1}ull) == 0ull")
                vals = ", ".join(self.at(val, j) for j in js)
                self.lines.append(f"{ind}if ({' && '.join(conds)}) {{")
                if self.nontemporal:
                    self.lines.append(f"{ind}  __builtin_nontemporal_store(({vty}){{{vals}}}, ({vty}*){p});")
                else:
                    self.lines.append(f"{ind}  *({vty}*){p} = ({vty}){{{vals}}};")
                self.lines.append(f"{ind}}} else {{")
                inner = ind + "  "
            else:
                inner = ind
            for j in js:
                c = masked(j)
                st = f"{b}[{self.at(off, j)}] = {self.at(val, j)};"
                self.lines.append(f"{inner}if ({c}) {st}" if c else f"{inner}{st}")
            if vty is not None and not is_tg:
                self.lines.append(f"{ind}}}")

    # -- hazards ---------------------------------------------------------------
    def plan_syncs(self) -> set[int]:
        """Indices of instructions that need a ``__syncthreads`` before them.

        One Metal thread executed the whole program in order; here its lanes
        run on ``T`` threads.  A store followed by any later access of the same
        buffer (or a load followed by a store) needs a workgroup barrier in
        between unless an explicit ``barrier`` already separates them.
        """
        need: set[int] = set()
        if self.T == 1:
            return need
        written: set[int] = set()
        read: set[int] = set()
        for idx, inst in enumerate(self.ir.insts):
            if inst.op == "barrier":
                written.clear()
                read.clear()
                continue
            if inst.op == "load":
                key = inst.args[0].id
                if key in written:
                    need.add(idx)
                    written.clear()
                    read.clear()
                read.add(key)
            elif inst.op == "store":
                key = inst.args[0].id
                if key in written or key in read:
                    need.add(idx)
                    written.clear()
                    read.clear()
                written.add(key)
        return need

    # -- main ----------------------------------------------------------------------
    def emit(self) -> Lowered:
        ir = self.ir
        sync_before = self.sync_before
        has_barrier = any(i.op == "barrier" for i in ir.insts) or bool(sync_before)
        live = "__plive" if has_barrier else None
        L = self.lines
        L.append(PRELUDE)
        L.append(f'extern "C" __global__ void __launch_bounds__({self.wg}) {ir.name}(')
        L.append(f"    {self.m.params([] if self.thread_mode else ['__eas_nprog'])}) {{")
        if self.thread_mode:  # one program per threadgroup: those holding at least one live thread
            b = self.block
            L.append(f"  const uint32_t __eas_nprog = __eas_nthreads / {b}u + (__eas_nthreads % {b}u != 0u ? 1u : 0u);")
        for inst in ir.insts:
            if inst.op == "alloc_tg":
                size = int(inst.args[0])
                dims = f"[{self.ppw}][{size}]" if self.ppw > 1 else f"[{size}]"
                L.append(f"  __shared__ {ctype(inst.out.dtype)} v{inst.out.id}{dims};")
        # __t: this thread's index among the T threads of its program (lanes __t*VEC onwards);
        # __slot: which of the workgroup's packed programs it serves; __wgi: the workgroup's
        # index among the launch's program groups (workgroups that share a split program
        # have the same one)
        if self.split > 1:
            L.append("  const uint32_t __slot = 0u;")
            L.append(f"  const uint32_t __t = (blockIdx.x % {self.split}u) * {self.wg}u + threadIdx.x;")
            L.append(f"  const uint32_t __wgi = blockIdx.x / {self.split}u;")
        elif self.ppw > 1:
            L.append(f"  const uint32_t __slot = threadIdx.x / {self.T}u;")
            L.append(f"  const uint32_t __t = threadIdx.x % {self.T}u;")
            L.append("  const uint32_t __wgi = blockIdx.x;")
        else:
            L.append("  const uint32_t __slot = 0u;")
            L.append("  const uint32_t __t = threadIdx.x;")
            L.append("  const uint32_t __wgi = blockIdx.x;")
        L.append(f"  const uint32_t __lbase = __t * {self.vec}u;")
        L.append("  #pragma unroll")
        L.append(f"  for (uint32_t __u = 0; __u < {self.unroll}u; ++__u) {{")
        L.append(f"  const uint32_t __pid = (__wgi * {self.unroll}u + __u) * {self.ppw}u + __slot;")
        if live:
            L.append("  const bool __plive = __pid < __eas_nprog;")
        else:
            L.append("  if (__pid < __eas_nprog) {")
        ind = "  "
        for idx, inst in enumerate(ir.insts):
            if idx in sync_before:
                L.append(f"{ind}__syncthreads();")
            self.emit_inst(inst, ind, live)
        if not live:
            L.append("  }")
        L.append("  }")
        L.append("}")
        mode = "thread" if self.thread_mode else "spmd"
        geo = Geometry(mode, ir.name, self.block, self.wg, self.ppw, self.unroll,
                       {"vec": self.vec, "lanes_per_thread": self.lpt, "threads_per_program": self.T,
                        "nontemporal": self.nontemporal, "lanes": True}, split=self.split)
        return Lowered(with_helpers(L), self.block, mode, geo)

    def emit_inst(self, inst: Inst, ind: str, live: str | None) -> None:
        op, out, a = inst.op, inst.out, inst.args
        L = self.lines
        if op in ("arg", "alloc_tg"):
            return
        if op == "const":
            L.append(f"{ind}const {ctype(out.dtype)} v{out.id} = {literal(a[0], out.dtype)};")
        elif op in ("program_id", "thread_id"):
            # SPMD programs are the reference's Metal threads: thread_id == program_id.
            src = {0: "__pid", 1: "blockIdx.y", 2: "blockIdx.z"}[int(a[0])]
            L.append(f"{ind}const uint32_t v{out.id} = {src};")
        elif op == "arange":
            start = int(a[0])
            L.append(f"{ind}{self.decl(out)};")
            for j in range(self.lpt):
                L.append(f"{ind}v{out.id}[{j}] = {start}u + {self.lane_index(j)};")
        elif op in _BINOP:
            L.append(f"{ind}{self.decl(out)};")
            for j in self.elems(out):
                L.append(f"{ind}{self.assign(out, j)} = {binop_expr(op, a[0].dtype, self.at(a[0], j), self.at(a[1], j))};")
        elif op == "not":
            L.append(f"{ind}{self.decl(out)};")
            for j in self.elems(out):
                L.append(f"{ind}{self.assign(out, j)} = !{self.at(a[0], j)};")
        elif op == "where":
            L.append(f"{ind}{self.decl(out)};")
            for j in self.elems(out):
                L.append(f"{ind}{self.assign(out, j)} = {self.at(a[0], j)} ? {self.at(a[1], j)} : {self.at(a[2], j)};")
        elif op == "cast":
            src = a[0]
            L.append(f"{ind}{self.decl(out)};")
            for j in self.elems(out):
                L.append(f"{ind}{self.assign(out, j)} = {cast_expr(self.at(src, j), src.dtype, out.dtype)};")
        elif op == "fma":
            L.append(f"{ind}{self.decl(out)};")
            for j in self.elems(out):
                L.append(f"{ind}{self.assign(out, j)} = {fma_expr(out.dtype, *(self.at(x, j) for x in a))};")
        elif op == "load":
            self.emit_load(inst, ind, live)
        elif op == "store":
            self.emit_store(inst, ind, live)
        elif op == "barrier":
            L.append(f"{ind}__syncthreads();")
        else:
            raise ValueError(f"unsupported op in spmd codegen: {op!r}")


def _vec_type(dt: DType, vec: int) -> str | None:
    if dt == DType.F32:
        return {4: "eas_f32x4", 2: "eas_f32x2"}.get(vec)
    if dt == DType.F16:
        return {8: "eas_f16x8", 4: "eas_f16x4", 2: "eas_f16x2"}.get(vec)
    if dt == DType.BF16:
        return {8: "eas_bf16x8", 4: "eas_bf16x4", 2: "eas_bf16x2"}.get(vec)
    return None


def fma_expr(dt: DType, x: str, y: str, z: str) -> str:
    """``fma(x, y, z)`` with one binary32 rounding; on f16 (bf16) values the reference's
    ``half(fma((float)x, (float)y, (float)z))`` (``msl.py:291-294``): fma in binary32, then
    a second rounding to the 16-bit type."""
    if dt == DType.F16:
        return f"eas_fma_f16({x}, {y}, {z})"
    if dt == DType.BF16:
        return f"eas_fma_bf16({x}, {y}, {z})"
    return f"__builtin_fmaf({x}, {y}, {z})"


# ---------------------------------------------------------------------------
# thread-mode emitter
# ---------------------------------------------------------------------------


class _ThreadEmitter:
    def __init__(self, ir: IRModule, block: int) -> None:
        if block > 1024:
            raise ValueError(f"thread-mode BLOCK={block} exceeds 1024 threads per workgroup")
        self.ir = ir
        self.m = _Module(ir)
        self.block = block
        self.lines: list[str] = []
        ops = {i.op for i in ir.insts}
        # Barriers (and LDS / simdgroup cooperation) forbid per-thread early exits.
        self.cooperative = bool(ops & {"barrier", "alloc_tg", "mma_zero", "mma", "mma_store"})
        self.live = "__live" if self.cooperative else None
        self.skip: set[int] = set()
        self.fused_dots: dict[int, list[Inst]] = {}
        self.inline_bool: dict[int, str] = {}

    # -- expressions -----------------------------------------------------------
    def n(self, ref: ValueRef) -> str:
        return self.inline_bool.get(ref.id) or self.m.name(ref)

    def guard(self, mask: ValueRef, known_true: set[int]) -> str | None:
        conds = []
        if not (self.m.is_true(mask) or mask.id in known_true):
            conds.append(self.n(mask))
        if self.live:
            conds.append(self.live)
        return " && ".join(conds) if conds else None

    def elem(self, buf: ValueRef, idx: str) -> str:
        e = f"{self.m.name(buf)}[{idx}]"
        return f"(float){e}" if buf.dtype in (DType.F16, DType.BF16) else e

    # -- analyses -------------------------------------------------------------
    def plan_inline_bools(self) -> None:
        """Fold single-use boolean trees that feed masks into one C expression."""
        m = self.m

        def build(ref: ValueRef) -> str | None:
            if ref.dtype != DType.BOOL or m.uses.get(ref.id, 0) != 1:
                return None
            d = m.defs.get(ref.id)
            if d is None:
                return None
            if d.op == "lt":
                return f"({binop_expr('lt', d.args[0].dtype, m.name(d.args[0]), m.name(d.args[1]))})"
            if d.op in ("and", "or"):
                parts = [build(x) or m.name(x) for x in d.args]
                return f"({parts[0]} {_BINOP[d.op]} {parts[1]})"
            if d.op == "not":
                return f"(!{build(d.args[0]) or m.name(d.args[0])})"
            return None

        for inst in self.ir.insts:
            if inst.op not in ("load", "store"):
                continue
            mask = inst.args[2] if inst.op == "load" else inst.args[3]
            if m.is_true(mask):
                continue
            expr = build(mask)
            if expr is not None:
                self.inline_bool[mask.id] = expr
                stack = [mask]
                while stack:
                    r = stack.pop()
                    if r.dtype != DType.BOOL or m.uses.get(r.id, 0) != 1:
                        continue
                    d = m.defs.get(r.id)
                    if d is None or d.op not in ("lt", "and", "or", "not"):
                        continue
                    self.skip.add(r.id)
                    stack.extend(x for x in d.args if isinstance(x, ValueRef))

    def plan_tn4(self) -> None:
        """Group 4 dots sharing A/K/strides whose B bases are base+0..3 (one
        16-byte B read per k instead of four scalar reads)."""
        m = self.m
        insts = self.ir.insts
        taken: set[int] = set()

        def split(ref: ValueRef) -> tuple[int, int]:
            d = m.defs.get(ref.id)
            if d is not None and d.op == "add":
                x, y = d.args
                cx, cy = m.const(x), m.const(y)
                if isinstance(cy, int) and not isinstance(cy, bool) and cx is None:
                    return x.id, cy
                if isinstance(cx, int) and not isinstance(cx, bool) and cy is None:
                    return y.id, cx
            return ref.id, 0

        for i, inst in enumerate(insts):
            if inst.op != "dot" or id(inst) in taken:
                continue
            a_buf, a_base, a_st, b_buf, b_base, b_st, k = inst.args
            sig = (a_buf.id, a_base.id, a_st.id, b_buf.id, b_st.id, k.id)
            base, off = split(b_base)
            if off != 0:
                continue
            found = {0: inst}
            for j in range(i + 1, min(len(insts), i + 96)):
                other = insts[j]
                if other.op in ("store", "barrier", "mma", "mma_store"):
                    break
                if other.op != "dot" or id(other) in taken:
                    continue
                oa = other.args
                if (oa[0].id, oa[1].id, oa[2].id, oa[3].id, oa[5].id, oa[6].id) != sig:
                    continue
                ob, oo = split(oa[4])
                if ob == base and oo in (1, 2, 3) and oo not in found:
                    found[oo] = other
                    if len(found) == 4:
                        break
            if len(found) == 4:
                group = [found[o] for o in range(4)]
                for g in group:
                    taken.add(id(g))
                self.fused_dots[id(inst)] = group
                for g in group[1:]:
                    self.skip.add(g.out.id)

    # -- emission -----------------------------------------------------------------
    def emit(self) -> Lowered:
        ir, m, L = self.ir, self.m, self.lines
        self.plan_inline_bools()
        self.plan_tn4()
        stores = [i for i in ir.insts if i.op == "store"]
        early = None
        if not self.cooperative and len(stores) == 1 and not m.is_true(stores[0].args[3]):
            early = stores[0].args[3]
        L.append(PRELUDE)
        L.append(f'extern "C" __global__ void __launch_bounds__({self.block}) {ir.name}(')
        L.append(f"    {m.params(['__eas_nthreads'])}) {{")
        for inst in ir.insts:
            if inst.op == "alloc_tg":
                L.append(f"  __shared__ __attribute__((aligned(16))) {ctype(inst.out.dtype)} v{inst.out.id}[{int(inst.args[0])}];")
        L.append(f"  const uint32_t __gid = blockIdx.x * {self.block}u + threadIdx.x;")
        if self.cooperative:
            L.append("  const bool __live = __gid < __eas_nthreads;")
        else:
            L.append("  if (__gid >= __eas_nthreads) return;")
        order = list(ir.insts)
        known_true: set[int] = set()
        if early is not None:
            # Hoist the store mask's dependencies, exit threads whose single store
            # is masked off, then run everything else unguarded where the mask
            # is the same value (reference: early return, msl.py:681-688).
            deps = self.deps_of(early)
            first = [i for i in order if i.out is not None and i.out.id in deps]
            rest = [i for i in order if not (i.out is not None and i.out.id in deps)]
            for inst in first:
                self.emit_inst(inst, "  ", known_true)
            L.append(f"  if (!{self.n(early)}) return;")
            known_true.add(early.id)
            order = rest
        for inst in order:
            self.emit_inst(inst, "  ", known_true)
        L.append("}")
        geo = Geometry("thread", ir.name, self.block, self.block)
        return Lowered(with_helpers(L), self.block, "thread", geo)

    def deps_of(self, ref: ValueRef) -> set[int]:
        seen: set[int] = set()
        stack = [ref.id]
        while stack:
            v = stack.pop()
            if v in seen:
                continue
            seen.add(v)
            d = self.m.defs.get(v)
            if d is not None:
                stack.extend(a.id for a in d.args if isinstance(a, ValueRef))
        return seen

    def emit_inst(self, inst: Inst, ind: str, known_true: set[int]) -> None:
        op, out, a = inst.op, inst.out, inst.args
        m, L = self.m, self.lines
        if op in ("arg", "alloc_tg"):
            return
        if out is not None and (out.id in self.skip or (m.uses.get(out.id, 0) == 0 and op not in ("dot",))):
            if op != "dot" or out.id in self.skip:
                return
        if op == "const":
            L.append(f"{ind}const {ctype(out.dtype)} v{out.id} = {literal(a[0], out.dtype)};")
        elif op == "program_id":
            L.append(f"{ind}const uint32_t v{out.id} = blockIdx.{'xyz'[int(a[0])]};")
        elif op == "thread_id":
            src = {0: "__gid", 1: "blockIdx.y", 2: "blockIdx.z"}[int(a[0])]
            L.append(f"{ind}const uint32_t v{out.id} = {src};")
        elif op == "local_id":
            L.append(f"{ind}const uint32_t v{out.id} = {'threadIdx.x' if int(a[0]) == 0 else '0u'};")
        elif op == "tid":
            start = int(a[0])
            L.append(f"{ind}const uint32_t v{out.id} = {f'{start}u + ' if start else ''}threadIdx.x;")
        elif op == "lane_id":
            L.append(f"{ind}const uint32_t v{out.id} = threadIdx.x & 31u;")
        elif op == "sg_id":
            L.append(f"{ind}const uint32_t v{out.id} = threadIdx.x >> 5;")
        elif op == "arange":
            raise ValueError("arange is not supported in thread mode codegen; use mk.tid(...) for thread-level kernels")
        elif op in _BINOP:
            L.append(f"{ind}const {ctype(out.dtype)} v{out.id} = {binop_expr(op, a[0].dtype, self.n(a[0]), self.n(a[1]))};")
        elif op == "not":
            L.append(f"{ind}const bool v{out.id} = !{self.n(a[0])};")
        elif op == "where":
            L.append(f"{ind}const {ctype(out.dtype)} v{out.id} = {self.n(a[0])} ? {self.n(a[1])} : {self.n(a[2])};")
        elif op == "cast":
            L.append(f"{ind}const {ctype(out.dtype)} v{out.id} = {cast_expr(self.n(a[0]), a[0].dtype, out.dtype)};")
        elif op == "fma":
            L.append(f"{ind}const {ctype(out.dtype)} v{out.id} = {fma_expr(out.dtype, *(self.n(x) for x in a))};")
        elif op == "load":
            buf, off, mask = a
            g = self.guard(mask, known_true)
            src = f"{m.name(buf)}[{self.n(off)}]"
            if g:
                L.append(f"{ind}{ctype(out.dtype)} v{out.id} = {zero(out.dtype)};")
                L.append(f"{ind}if ({g}) {{ v{out.id} = {src}; }}")
            else:
                L.append(f"{ind}const {ctype(out.dtype)} v{out.id} = {src};")
        elif op == "store":
            buf, off, val, mask = a
            g = self.guard(mask, known_true)
            st = f"{m.name(buf)}[{self.n(off)}] = {self.n(val)};"
            L.append(f"{ind}if ({g}) {{ {st} }}" if g else f"{ind}{st}")
        elif op == "barrier":
            L.append(f"{ind}__syncthreads();")
        elif op == "dot":
            group = self.fused_dots.get(id(inst))
            if group is not None:
                self.emit_dot_tn4(group, ind)
            else:
                self.emit_dot(inst, ind)
        elif op == "mma_zero":
            L.append(f"{ind}float v{out.id}_0 = 0.0f, v{out.id}_1 = 0.0f;")
        elif op == "mma":
            self.emit_mma(inst, ind)
        elif op == "mma_store":
            c, base, stride, frag = a
            f = self.m.name(frag)
            row = f"({self.n(base)} + (threadIdx.x & 31u) / 4u * {self.n(stride)} + (threadIdx.x & 3u) * 2u)"
            cond = f"if ({self.live}) " if self.live else ""
            L.append(f"{ind}{cond}{{ const uint32_t __o = {row}; {m.name(c)}[__o] = {f}_0; {m.name(c)}[__o + 1u] = {f}_1; }}")
        else:
            raise ValueError(f"unsupported op: {op}")

    def dot_bound(self, k: ValueRef) -> str:
        kb = self.n(k)
        return f"({self.live} ? {kb} : 0u)" if self.live else kb

    def emit_dot(self, inst: Inst, ind: str) -> None:
        a_buf, a_base, a_st, b_buf, b_base, b_st, k = inst.args
        o = inst.out.id
        L = self.lines
        L.append(f"{ind}float v{o} = 0.0f;")
        L.append(f"{ind}{{ uint32_t __ai = {self.n(a_base)}, __bi = {self.n(b_base)};")
        kc = self.m.const(k)
        if isinstance(kc, int) and 1 <= kc <= 32:
            L.append(f"{ind}  #pragma unroll")
        L.append(f"{ind}  for (uint32_t k{o} = 0; k{o} < {self.dot_bound(k)}; ++k{o}) {{")
        L.append(f"{ind}    v{o} = __builtin_fmaf({self.elem(a_buf, '__ai')}, {self.elem(b_buf, '__bi')}, v{o});")
        L.append(f"{ind}    __ai += {self.n(a_st)}; __bi += {self.n(b_st)};")
        L.append(f"{ind}  }} }}")

    def emit_dot_tn4(self, group: list[Inst], ind: str) -> None:
        a_buf, a_base, a_st, b_buf, b_base, b_st, k = group[0].args
        outs = [g.out.id for g in group]
        o = outs[0]
        L = self.lines
        bname = self.m.name(b_buf)
        vty = {DType.F32: "eas_f32x4", DType.F16: "eas_f16x4", DType.BF16: "eas_bf16x4"}[b_buf.dtype]
        bty = ctype(b_buf.dtype)
        L.append(f"{ind}float {', '.join(f'v{x} = 0.0f' for x in outs)};")
        L.append(f"{ind}{{ uint32_t __ai = {self.n(a_base)}, __bi = {self.n(b_base)};")
        kc = self.m.const(k)
        if isinstance(kc, int) and 1 <= kc <= 32:
            L.append(f"{ind}  #pragma unroll")
        L.append(f"{ind}  for (uint32_t k{o} = 0; k{o} < {self.dot_bound(k)}; ++k{o}) {{")
        L.append(f"{ind}    const float __a = {self.elem(a_buf, '__ai')};")
        L.append(f"{ind}    const {bty}* __bp = {bname} + __bi;")
        align = 15 if b_buf.dtype == DType.F32 else 7
        L.append(f"{ind}    if ((((uint64_t)__bp) & {align}ull) == 0ull) {{")
        L.append(f"{ind}      const {vty} __b = *(const {vty}*)__bp;")
        for e, x in enumerate(outs):
            L.append(f"{ind}      v{x} = __builtin_fmaf(__a, (float)__b[{e}], v{x});")
        L.append(f"{ind}    }} else {{")
        for e, x in enumerate(outs):
            L.append(f"{ind}      v{x} = __builtin_fmaf(__a, (float)__bp[{e}], v{x});")
        L.append(f"{ind}    }}")
        L.append(f"{ind}    __ai += {self.n(a_st)}; __bi += {self.n(b_st)};")
        L.append(f"{ind}  }} }}")

    def emit_mma(self, inst: Inst, ind: str) -> None:
        """Literal 8x8x8 simdgroup MMA: lane l of the 32-lane simdgroup owns C
        elements (l/4, 2*(l%4)) and (l/4, 2*(l%4)+1) and accumulates them with
        f32 fmas over k ascending."""
        a_buf, a_base, a_st, b_buf, b_base, b_st, acc = inst.args
        o = inst.out.id
        acc_n = self.m.name(acc)
        L = self.lines
        live = self.live or "true"
        L.append(f"{ind}float v{o}_0 = {acc_n}_0, v{o}_1 = {acc_n}_1;")
        L.append(f"{ind}{{ const uint32_t __r = (threadIdx.x & 31u) >> 2, __c = (threadIdx.x & 3u) * 2u;")
        L.append(f"{ind}  const uint32_t __ar = {self.n(a_base)} + __r * {self.n(a_st)};")
        L.append(f"{ind}  #pragma unroll")
        L.append(f"{ind}  for (uint32_t __k = 0; __k < 8u; ++__k) {{")
        L.append(f"{ind}    const uint32_t __br = {self.n(b_base)} + __k * {self.n(b_st)} + __c;")
        L.append(f"{ind}    const float __a = {live} ? {self.elem(a_buf, '__ar + __k')} : 0.0f;")
        L.append(f"{ind}    v{o}_0 = __builtin_fmaf(__a, {live} ? {self.elem(b_buf, '__br')} : 0.0f, v{o}_0);")
        L.append(f"{ind}    v{o}_1 = __builtin_fmaf(__a, {live} ? {self.elem(b_buf, '__br + 1u')} : 0.0f, v{o}_1);")
        L.append(f"{ind}  }} }}")


# ---------------------------------------------------------------------------
# entry point
# ---------------------------------------------------------------------------


_ARG_LAYOUT = {DType.U32: 4, DType.F32: 4, DType.F16: 2, DType.BF16: 2, DType.BOOL: 1}


def kernarg_offsets(ir: IRModule) -> list[int]:
    """Byte offset of each of a kernel's own arguments in the packed argument blob, in IR
    order, each at its natural alignment (buffers are 8-byte pointers), as the native launch
    packs them."""
    offs, off = [], 0
    for arg in ir.args:
        size = 8 if arg.kind == "buffer" else _ARG_LAYOUT[arg.dtype]
        off = -(-off // size) * size
        offs.append(off)
        off += size
    return offs


def kernarg_bytes(ir: IRModule) -> int:
    """Packed size of a kernel's own arguments (``kernarg_offsets``' layout)."""
    if not ir.args:
        return 0
    last = ir.args[-1]
    return kernarg_offsets(ir)[-1] + (8 if last.kind == "buffer" else _ARG_LAYOUT[last.dtype])


# entry points of a lifted GEMM, by their bit in the eas-gemm line's entry mask (eas_hip_gemm_entry)
GEMM_ENTRY_BITS = (("pp_entry", 1), ("t128_entry", 2), ("t128x256_entry", 3), ("t128x64_entry", 4),
                   ("t64_entry", 5))


def gemm_marker(ir: IRModule, geo: Geometry) -> str:
    """The ``// eas-gemm:`` line of a lifted GEMM: what its launch plan needs, for
    ``eas_hip_gemm_shape_parse`` in the C ABI (the same inputs ``gemm_lift.plan_gemm``
    reads from the geometry and the runtime arguments)."""
    from .gemm_lift import SKINNY_CUT, WIDE_M

    p = geo.params
    offs = kernarg_offsets(ir)
    pos = {a.name: i for i, a in enumerate(ir.args)}

    def scalar(name: str | None) -> str:
        if name is None:
            return ""
        arg = ir.args[pos[name]]
        assert arg.kind == "scalar" and arg.dtype == DType.U32, f"GEMM size argument {name!r} must be a u32 scalar"
        return str(offs[pos[name]])

    def elem(name: str) -> int:
        return 2 if ir.args[pos[name]].dtype in (DType.F16, DType.BF16) else 4

    mask = 1
    for key, bit in GEMM_ENTRY_BITS:
        if p.get(key):
            assert p[key] == geo.entry + {1: "__pp", 2: "__t128", 3: "__t128x256", 4: "__t128x64",
                                          5: "__t64x64"}[bit], p[key]
            mask |= 1 << bit
    items = [("entry", geo.entry), ("entries", mask), ("K", p["K"]), ("tm", p["TM"]), ("tn", p["TN"]),
             ("row_axis", p["row_axis"]), ("bm", p["BM"]), ("bn", p["BN"]), ("threads", p["threads"]),
             ("pp_threads", p["pp_threads"]), ("t128_threads", p["t128_threads"]),
             ("skinny_m", p["skinny_m"]), ("skinny_n", p["skinny_n"]), ("skinny_cut", SKINNY_CUT),
             ("wide_m", WIDE_M), ("f32", int(bool(p.get("f32")))),
             ("col_masked", int(bool(p.get("col_masked", True)))), ("m", scalar(p.get("m_sym"))),
             ("ldb", scalar(p["n_sym"])), ("row_base", scalar(p.get("row_base"))),
             ("col_base", scalar(p.get("col_base"))), ("a", pos[p["a"]]), ("b", pos[p["b"]]), ("c", pos[p["c"]]),
             ("a_off", offs[pos[p["a"]]]), ("b_off", offs[pos[p["b"]]]), ("a_elem", elem(p["a"])),
             ("b_elem", elem(p["b"])), ("c_elem", elem(p["c"]))]
    return "// eas-gemm: " + " ".join(f"{k}={v}" for k, v in items if v != "") + "\n"


def launch_marker(ir: IRModule, geo: Geometry) -> str:
    """The ``// eas-launch:`` line the native layer reads a kernel's launch shape from
    (``eas_hip_launch_shape_parse`` in the C ABI), and a lifted GEMM's ``// eas-gemm:`` line."""
    hidden = 4 if geo.kind == "gemm" else 1
    ppw = geo.programs_per_wg * geo.unroll if geo.kind in ("spmd", "thread") else 1
    line = (f"// eas-launch: kind={geo.kind} block={geo.block_size} wg={geo.wg_size} ppw={ppw} "
            f"split={geo.split} args={kernarg_bytes(ir)} hidden={hidden}\n")
    gemm = geo if geo.kind == "gemm" else geo.params.get("gemm")
    return line + gemm_marker(ir, gemm) if gemm is not None else line


def ir_to_hip(ir: IRModule) -> Lowered:
    """Lower verified, optimised IR to gfx950 HIP C++.  The source starts with the
    kernel's launch shape (``launch_marker``)."""
    block, mode = infer_block_and_mode(ir)
    if mode == "spmd":
        low = _SpmdEmitter(ir, block).emit()
    else:
        from .gemm_lift import try_lift, try_lift_chain
        from .thread_lanes import as_lanes

        low = try_lift(ir, block)
        if low is None:
            lanes = as_lanes(ir, block)
            low = _SpmdEmitter(lanes, block, thread_mode=True).emit() if lanes is not None else \
                _ThreadEmitter(ir, block).emit()
            mm = try_lift_chain(ir, block)
            if mm is not None:  # the same source, launch shape and entry, with the GEMM's entries after it
                geo = replace(low.geometry, params={**low.geometry.params, "gemm": mm.geometry})
                low = Lowered(low.src + mm.src.replace(PRELUDE, "", 1), low.block_size, low.launch_mode, geo)
    return Lowered(launch_marker(ir, low.geometry) + low.src, low.block_size, low.launch_mode, low.geometry)
