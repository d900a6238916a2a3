"""Straight-line kernels for an arbitrary uniform-1d plan (used by ``cuequivariance_amd/jit.py`` at first use).

The table-driven executor (``csrc/uniform1d.hip``) interprets the path table per output element; for plans outside the
two generated families (channel-wise products, symmetric contractions) - second derivatives, spherical harmonics,
flattened fully connected products - this generator bakes the table into the instruction stream instead.  One kernel per
output buffer: a wavefront owns 64 channels of one output row (a lane owns a whole row when there is no channel mode; where
the rows are few and their lists long, up to 16 wavefronts of a block share a row's list, ``row_parts`` in ``cw_common.h``), walks the batch elements that map to the row (the row
itself for a batched output, its CSR range for an indexed one), loads every input segment the output's paths read once
per batch element and evaluates the paths as fused multiply-adds into one accumulator per output segment.

The call shapes the generated ``run`` accepts: every tensor in the math type, outputs batched or indexed (with the CSR
grouping), inputs shared / batched / indexed; a scalar-segment output (``buffer_dim`` 0) fed by channel-carrying inputs
only when the extent fits one wavefront.  Anything else is declined and the table-driven kernels run.
"""

from __future__ import annotations

import re
from collections import defaultdict

from ..tables import U1dTables
from .channelwise import _lit, io_type

MAX_TERMS = 40000  # beyond this the translation unit takes minutes to compile: left to the table-driven kernels


def output_terms(t: U1dTables):
    """{output buffer: [(output segment, ((input buffer, segment), ...), coefficient)]} over all operations."""
    terms = defaultdict(list)
    nin = t.num_inputs
    for o in range(len(t.num_operands)):
        bufs, paths = t.operation(o)
        out_pos = [s for s, b in enumerate(bufs) if b >= nin]
        assert len(out_pos) == 1
        out_pos = out_pos[0]
        for idx, c in paths:
            if c == 0.0:
                continue
            ins = tuple((bufs[s], idx[s]) for s in range(len(bufs)) if s != out_pos)
            terms[bufs[out_pos]].append((idx[out_pos], ins, c))
    return terms


def supported(t: U1dTables) -> bool:
    return 0 < sum(len(v) for v in output_terms(t).values()) <= MAX_TERMS


FOLD = 8  # segments of the output that meet in LDS at a time (16 wavefronts, float64: 64 KB)


UNBOUND = 4  # wavefronts of a block that bound nothing: each may have all registers of its SIMD


def _most_parts(values: int, terms: int, T: str) -> int:
    """Most wavefronts to try for the list of an output row.  Sixteen leave a wavefront 128 registers, eight 256, and a kernel that needs
    more spills in every launch, a batched output's too.  What it needs is up to the compiler, which keeps products of operands
    beside the ``values`` (inputs read once per batch element and sums): this is a guess that saves compiling twice, ``fewer_parts`` has the last
    word.  (Registers of second derivatives, float: channel-wise product, 78 values and 116 terms, 65; 193 and 706, 167 - product
    basis, 28 and 268, 86; 37 and 361, 157; 39 and 1 137, 246; 56 and 1 531, 279.  All gradients of that basis's gradients, 64 ch
    l <= 2 -> l <= 1, us with sixteen wavefronts wherever the values fit / as here: float 451 rows 77 / 51, 20 000 rows
    2 543 / 1 247; float64 3 000 rows 3 918 / 512.)"""
    registers = (values + max(0, terms - 4 * values) // 4) * (2 if T == "double" else 1) + 30
    return 16 if registers <= 110 else 8 if registers <= 320 else UNBOUND


REPORT_FLAG = "-Rpass-analysis=kernel-resource-usage"


def fewer_parts(parts: dict, report: str):
    """``parts`` ({output buffer: most wavefronts that share a list}) after a look at what the compiler says of the unit emitted with them
    (``REPORT_FLAG``): half as many where a kernel spills registers, ``UNBOUND`` where it says nothing; ``None`` when they may stay."""
    spilled, kernel = {}, None
    for line in report.splitlines():
        if (m := re.search(r"Function Name: \S*out(\d+)_kernel", line)) is not None:
            kernel = int(m.group(1))
        elif kernel is not None and (m := re.search(r"ScratchSize \[bytes/lane\]: (\d+)", line)) is not None:
            spilled[kernel] = int(m.group(1)) > 0
    fewer = {ob: n if n <= UNBOUND or spilled.get(ob) is False else n // 2 if ob in spilled else UNBOUND for ob, n in parts.items()}
    return None if fewer == parts else fewer


def parts_of(t: U1dTables, T: str) -> dict:
    """{output buffer: most wavefronts that share the list of one of its rows}, before the compiler was asked."""
    terms = output_terms(t)

    def values(tl):
        return len({bs for _, ins, _ in tl for bs in ins}) + len({oseg for oseg, _, _ in tl})

    return {ob: _most_parts(values(terms.get(ob, [])), len(terms.get(ob, [])), T) if t.operand_extent > 1 else 1
            for ob in range(t.num_inputs, t.num_inputs + t.num_outputs)}


def emit_unit(t: U1dTables, T: str, name: str, table_hash: int, io=None, parts=None) -> str:
    """``io``: element type of the buffers when it is not the arithmetic type ``T`` ("bf16" / "f16" with ``T`` = float).  ``parts``: of
    ``parts_of``, or what ``fewer_parts`` made of it."""
    TI, io_code, tag = io_type(T, io)
    E = t.operand_extent
    nin, nout = t.num_inputs, t.num_outputs
    nch = (E + 63) // 64
    terms = output_terms(t)
    addressing = {b: t.segment_addressing(b) for b in range(nin + nout) if t.buffer_dim[b]}

    def at(b, s):  # element (segment s, channel uu) of a row of buffer b, under the buffer's layout
        base, stride = addressing[b][s]
        return f"{base} + uu" if stride == 1 else f"{base} + uu * {stride}"

    L = []
    A = L.append
    A("// GENERATED by cuequivariance_amd/codegen/general.py - do not edit.")
    A(f"// uniform-1d plan '{name}': extent {E}, {nin} inputs, {nout} outputs, {sum(len(v) for v in terms.values())} paths, math {T}" + (f", buffers of {tag}" if io else ""))
    A('#include "cw_common.h"')
    A("")
    A("namespace cueq {")
    A(f"namespace g_{name}" + (f"_{tag}" if io else "") + " {")
    A(f"using TI = {TI};  // element type of the buffers")
    A("")
    A("// the inputs of one call (pointer, index tensor, batch mode), passed to the kernels by value")
    A("struct InBuf { const void* data; const void* index; int32_t mode; int32_t idx64; };")
    A(f"struct InTable {{ InBuf b[{max(nin, 1)}]; }};")
    A("")
    most_parts = parts_of(t, T) if parts is None else parts
    for ob in range(nin, nin + nout):
        tl = terms.get(ob, [])
        used = sorted({bs for _, ins, _ in tl for bs in ins})
        used_bufs = sorted({b for b, _ in used})
        out_dim, out_nseg = t.buffer_dim[ob], t.buffer_num_segments[ob]
        out_width = out_nseg * (E if out_dim else 1)
        by_seg = defaultdict(list)
        for oseg, ins, c in tl:
            by_seg[oseg].append((ins, c))
        A(f"// output buffer {ob}: {len(tl)} paths into {len(by_seg)} of {out_nseg} segments")
        most = most_parts[ob]
        A(f"__global__ void __launch_bounds__({64 * most}) out{ob}_kernel(const InTable tab, TI* __restrict__ out, int64_t rows, "
          "const int64_t* __restrict__ csr_offsets, const int64_t* __restrict__ csr_perm) {")
        if most > 1:
            A(f"  extern __shared__ __align__(16) unsigned char fold_shared[];  // (blocks of one wavefront have none)")
            A("  const int lane = threadIdx.x & 63, nparts = blockDim.x >> 6, part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);")
        else:
            A("  const int lane = threadIdx.x;")
        if E == 1:  # no channel mode: a lane per output row
            A("  const int64_t r = static_cast<int64_t>(blockIdx.x) * 64 + lane;")
            A("  if (r >= rows) return;")
            A("  constexpr bool active = true; constexpr int uu = 0;")
        else:
            A(f"  const int64_t r = static_cast<int64_t>(blockIdx.x) / {nch};")
            A(f"  const int ch = static_cast<int>(static_cast<int64_t>(blockIdx.x) - r * {nch});")
            A("  if (r >= rows) return;")
            A(f"  const int u = ch * 64 + lane; const bool active = u < {E}; const int uu = active ? u : 0;")
        # a scalar output contracts the channel mode of the paths that carry it; paths of scalars only contribute once
        # and are kept in accumulators of their own (sacc), outside the sum over lanes
        contracting = (not out_dim) and E > 1 and any(t.buffer_dim[b] for b in used_bufs)

        def is_scalar_path(ins):
            return contracting and not any(t.buffer_dim[b] for b, _ in ins)

        for s in sorted(by_seg):
            A(f"  {T} acc{s} = 0;")
            if any(is_scalar_path(ins) for ins, _ in by_seg[s]):
                A(f"  {T} sacc{s} = 0;")
        A("  int64_t z0 = r, z1 = r + 1;")
        A("  if (csr_offsets) { z0 = csr_offsets[r]; z1 = csr_offsets[r + 1]; }")
        if most > 1:
            A("  if (nparts > 1) {  // (a power of two)")
            A("    const int64_t first = z0, count = z1 - z0;")
            A("    const int shift = 31 - __builtin_clz(nparts);")
            A("    z0 = first + ((count * part) >> shift); z1 = first + ((count * (part + 1)) >> shift);")
            A("  }")
        A("  for (int64_t zz = z0; zz < z1; ++zz) {")
        A("    const int64_t z = csr_perm ? csr_perm[zz] : zz;")
        for b in used_bufs:
            width = t.buffer_num_segments[b] * (E if t.buffer_dim[b] else 1)
            A(f"    const int64_t row{b} = tab.b[{b}].mode == CUEQ_BATCH_INDEXED ? load_index(tab.b[{b}].index, tab.b[{b}].idx64, z) : "
              f"(tab.b[{b}].mode == CUEQ_BATCH_BATCHED ? z : 0);")
            A(f"    const TI* __restrict__ p{b} = static_cast<const TI*>(tab.b[{b}].data) + row{b} * {width}ll;")
        for b, s in used:
            A(f"    const {T} v{b}_{s} = io_ld(p{b} + ({at(b, s)}));" if t.buffer_dim[b] else f"    const {T} v{b}_{s} = io_ld(p{b} + {s});")
        for oseg in sorted(by_seg):
            for ins, c in by_seg[oseg]:
                acc = f"sacc{oseg}" if is_scalar_path(ins) else f"acc{oseg}"
                if not ins:
                    A(f"    {acc} += {_lit(c, T)};")
                elif len(ins) == 1:
                    A(f"    {acc} = fma({_lit(c, T)}, v{ins[0][0]}_{ins[0][1]}, {acc});")
                else:
                    prod = " * ".join(f"v{b}_{s}" for b, s in ins[1:])
                    A(f"    {acc} = fma({_lit(c, T)} * v{ins[0][0]}_{ins[0][1]}, {prod}, {acc});")
        A("  }")
        A(f"  TI* __restrict__ op = out + r * {out_width}ll;")
        if contracting:  # scalar output segments: the channel mode is contracted (one wavefront covers it)
            for s in sorted(by_seg):
                A(f"  acc{s} = wave_sum(active ? acc{s} : {T}(0));")
                if any(is_scalar_path(ins) for ins, _ in by_seg[s]):
                    A(f"  acc{s} += sacc{s};")
        mine = "active" if out_dim else ("lane == 0" if E > 1 else "true")
        place = (lambda s: at(ob, s)) if out_dim else str
        if most > 1:
            # the parts' sums meet in LDS, FOLD segments at a time; the wavefronts share the segments and add the parts in order
            A("  if (nparts > 1) {")
            A(f"    {T}* s_fold = reinterpret_cast<{T}*>(fold_shared);")
            filled = sorted(by_seg)
            held = min(FOLD, len(filled))  # of every part
            for c0 in range(0, len(filled), FOLD):
                if c0:
                    A("    __syncthreads();")
                for n, s in enumerate(filled[c0: c0 + FOLD]):
                    A(f"    s_fold[(part * {held} + {n}) * 64 + lane] = acc{s};")
                A("    __syncthreads();")
                for n, s in enumerate(filled[c0: c0 + FOLD]):
                    A(f"    if (part == ({n} & (nparts - 1))) {{ const {T} sum = fold_sum_of(nparts, s_fold + {n * 64} + lane, {held * 64}); "
                      f"if ({mine}) io_st(sum, op + ({place(s)})); }}")
            empty = [s for s in range(out_nseg) if s not in by_seg]
            if empty:
                A(f"    if (part == 0 && {mine}) {{")
                for s in empty:
                    A(f"      io_st({T}(0), op + ({place(s)}));")
                A("    }")
            A("    return;")
            A("  }")
        A(f"  if ({mine}) {{")
        for s in range(out_nseg):
            A("    io_st(" + (f"acc{s}" if s in by_seg else f"{T}(0)") + f", op + ({place(s)}));")
        A("  }")
        A("}")
        A("")
    A("static int run(const SpecCall& c) {")
    A("  const cueq_u1d_buffer* b = c.buffers;")
    A(f"  if (common_dtype(b, {nin + nout}) != {io_code}) return CUEQ_ERR_UNSUPPORTED;")
    for ob in range(nin, nin + nout):
        A(f"  if (b[{ob}].batch_dim == CUEQ_BATCH_SHARED) return CUEQ_ERR_UNSUPPORTED;")
        A(f"  if (b[{ob}].batch_dim == CUEQ_BATCH_INDEXED && (!b[{ob}].csr_offsets || (!b[{ob}].csr_perm && c.batch > 0))) return CUEQ_ERR_UNSUPPORTED;")
        used_bufs = sorted({bb for _, ins, _ in terms.get(ob, []) for bb, _ in ins})
        if not t.buffer_dim[ob] and any(t.buffer_dim[bb] for bb in used_bufs) and E > 64:
            A("  return CUEQ_ERR_UNSUPPORTED;  // a scalar output that contracts more than one wavefront of channels")
    A("  InTable tab;")
    A(f"  for (int i = 0; i < {nin}; ++i) tab.b[i] = InBuf{{b[i].data, b[i].index, b[i].batch_dim, b[i].index_is_64}};")
    A(f'  KernelTimer timer("{name}_{tag}", c.stream);')
    for ob in range(nin, nin + nout):
        A("  {")
        A(f"    const int64_t rows = b[{ob}].rows;")
        A(f"    const bool idx = b[{ob}].batch_dim == CUEQ_BATCH_INDEXED;")
        A(f"    const int64_t grid = {'(rows + 63) / 64' if E == 1 else f'rows * {nch}'};")
        A('    CUEQ_REQUIRE(grid < (int64_t(1) << 31), CUEQ_ERR_TOO_LARGE, "too many output rows for one launch");')
        A("    if (rows > 0) {")
        if most_parts[ob] > 1:
            A(f"      const int nparts = idx ? row_parts(grid, c.batch, rows, {most_parts[ob]}) : 1;")
            held = min(FOLD, len({seg for seg, _, _ in terms.get(ob, [])}))
            A(f"      const unsigned shared = nparts > 1 ? nparts * {held * 64}u * sizeof({T}) : 0u;")
        else:
            A("      constexpr int nparts = 1; constexpr unsigned shared = 0;")
        A(f"      hipLaunchKernelGGL(out{ob}_kernel, dim3(static_cast<unsigned>(grid)), dim3(64 * nparts), shared, c.stream, tab, static_cast<TI*>(b[{ob}].data), rows,")
        A(f"                         idx ? b[{ob}].csr_offsets : nullptr, idx ? b[{ob}].csr_perm : nullptr);")
        A("      CUEQ_CHECK_HIP(hipGetLastError());")
        A("    }")
        A("  }")
    A("  return CUEQ_OK;")
    A("}")
    A("")
    A(f'static const U1dSpec spec = {{0x{table_hash:016x}ull, "{name}_{tag}", run, nullptr, {io_code}}};')
    A("static SpecRegistrar reg(&spec);")
    A("")
    A("}  // namespace")
    A("}  // namespace cueq")
    return "\n".join(L) + "\n"
