"""Sources of mapped reductions: an elementwise group reduced without storing it.

The mapped array is split at its reduced axes into (outer, reduced, inner).
Three kernels: rows (the reduced axes are the last ones, inner = 1), columns
(they are adjacent and inner > 1) and any (the rest: one element per lane
through index arithmetic). Values, identities and combinations are those of
the elementwise sources (_hip_lowering.py); only the order of a sum depends on
the kernel, and it is fixed for a shape, so results repeat bit for bit.
"""

from math import gcd, prod

from . import _hip_lowering as source_

VECTOR = source_.VECTOR
BLOCK = source_.BLOCK
CHUNK = source_.REDUCE_CHUNK
WAVES = BLOCK // 64
# Between the loads of a batch and their use: without it the compiler sinks
# each load to its use and one is in flight at a time.
FENCE = "__builtin_amdgcn_sched_barrier(0);"
COMPUTE_UNITS = 256  # of the gfx950 parts these sources are compiled for
MOST_WORKGROUPS = 2**24 - 1  # of BLOCK threads: a launch takes fewer than 2^32


class MapReduce(tuple):
    """Payload of a mapped reduction: (source, count, chunks), the kernel, the
    outputs and the partials of each output; as attributes its grid and the
    shape of the partials, whose axis 1 is still to be reduced."""

    def __new__(cls, source, count, chunks, grid, partials):
        self = super().__new__(cls, (source, count, chunks))
        self.grid, self.partials = grid, partials
        return self


def row_lanes(outer, reduced):
    """Lanes that share one row of a contiguous row reduction: about 16
    elements (four vector loads) each, inside a wave, so that short rows share
    waves and need no barrier; a whole workgroup for rows of several chunks,
    and where there are too few rows to give every compute unit 16 waves. The
    rule of hp_reduce's rows (reduce.hip, row_lanes), whose sums are bit for
    bit those of this kernel."""
    lanes = 1
    while lanes < 64 and lanes * 16 < reduced:
        lanes *= 2
    if lanes == 64 and (outer < 4096 or reduced > CHUNK):
        return BLOCK
    return lanes


class _Mapped:
    """The mapped array: how its leaves are read and its element computed."""

    def __init__(self, shape, axes, leaves, nodes, operation, acc_dtype):
        self.shape, self.axes, self.leaves, self.nodes = tuple(shape), tuple(axes), leaves, nodes
        self.operation, self.acc_dtype = operation, acc_dtype
        self.acc = source_.ctype(acc_dtype)
        self.identity = source_._identity(operation, acc_dtype)
        params, _, _ = source_._body(self.shape, leaves, nodes)
        self.params = ", ".join([*params, f"{self.acc}* __restrict__ out"])
        self.outer = prod(self.shape[: self.axes[0]]) if self.axes else prod(self.shape)
        self.reduced = prod(self.shape[d] for d in self.axes)
        self.inner = prod(self.shape[self.axes[-1] + 1 :]) if self.axes else 1
        self.access = [None if leaf.scalar else self._access(leaf) for leaf in leaves]

    def adjacent(self):
        return bool(self.axes) and self.axes == tuple(range(self.axes[0], self.axes[-1] + 1)) and prod(self.shape) > 0

    def _access(self, leaf):
        """'full' (the element's own index), 'outer', 'reduced' or 'inner' (the
        leaf varies along that part only), 'one', or 'any' (the flat index)."""
        if leaf.shape == self.shape:
            return "full"
        rank = len(self.shape)
        padded = (1,) * (rank - len(leaf.shape)) + leaf.shape
        if prod(padded) == 1:
            return "one"
        if self.adjacent():
            first, last = self.axes[0], self.axes[-1]
            parts = {"outer": range(first), "reduced": self.axes, "inner": range(last + 1, rank)}
            for name, part in parts.items():
                if all(padded[d] == (self.shape[d] if d in part else 1) for d in range(rank)):
                    return name
        return "any"

    def reads(self, *kinds):
        """(index, C type) of the leaves read in one of these ways."""
        return [(k, source_.ctype(self.leaves[k].dtype)) for k, a in enumerate(self.access) if a in kinds]

    def bytes_read(self):
        """Of the leaves that every element reads anew."""
        return prod(self.shape) * sum(self.leaves[k].dtype.itemsize for k, _ in self.reads("full", "any"))

    def combine(self, left, right):
        return source_._combine(self.operation, self.acc_dtype, left, right)

    def _lambda(self, name, given):
        """The mapped element at flat index i as a device lambda; the leaves in
        ``given`` are its arguments, the others are read through i."""

        def leaf_value(k):
            if k in given:
                return f"a{k}"
            return f"x{k}[{source_._broadcast_offset(self.shape, self.leaves[k].shape, 'i')}]"

        _, lines, result = source_._body(self.shape, self.leaves, self.nodes, leaf_value=leaf_value)
        boolean = bool(self.nodes) and self.nodes[-1][3].kind == "b"
        value = f"({result} != 0)" if boolean else result
        arguments = "".join(f", const {source_.ctype(self.leaves[k].dtype)} a{k}" for k in given)
        body = "\n    ".join(lines)
        return f"""const auto {name} = [&](const long long i{arguments}) -> {self.acc} {{
    {body}
    return ({self.acc})({value});
  }};"""

    def lambdas(self, *kinds):
        """`mapped(i, leaves read in one of `kinds`)` and `element(i)`."""
        given = [k for k, _ in self.reads(*kinds)]
        return self._lambda("mapped", given) + "\n  " + self._lambda("element", []), given

    def kernel(self, body, workgroups=0):
        """The kernel of `body`; with more `workgroups` than a launch takes, the
        body (for workgroup `at`) in a loop over them."""
        loop, close = "const unsigned at = blockIdx.x;", ""
        if workgroups > MOST_WORKGROUPS:
            loop = f"for (unsigned at = blockIdx.x; at < {workgroups}U; at += gridDim.x) {{"
            close = "__syncthreads();  // the next one writes the same LDS\n}"
        return f"""{source_._PRELUDE}
extern "C" __global__ __launch_bounds__({BLOCK}) void pacho_map_reduce({self.params}) {{
{loop}
{body}
{close}
}}
"""


def map_reduce_source(shape, axes, leaves, nodes, operation, acc_dtype):
    """The kernel and launch geometry of a mapped reduction, as a MapReduce."""
    mapped = _Mapped(shape, axes, leaves, nodes, operation, acc_dtype)
    if mapped.adjacent() and mapped.inner == 1:
        return _rows(mapped)
    if mapped.adjacent():
        return _columns(mapped)
    return _any(mapped)


def _lines(lines, indent):
    return ("\n" + " " * indent).join(lines)


def _rows(m):
    """Lanes of a row (or of a CHUNK piece of one) take VECTOR consecutive
    elements per step, four steps in flight; the four elements combine in
    pairs, then with the lane's accumulator; lanes meet in a butterfly and
    waves in LDS. Bound by HBM: full leaves are read in 16-byte loads at
    element alignment, with the nontemporal hint where a wave reads whole
    lines of one row (16384 x 4000 float32: 45 against 50 us; `stream` below
    for 8-byte elements) and without it where rows share lines (1200000 x 49:
    45 against 73 us). Max of x * x over
    the rows of 65536 x 4001 float32: 170 us (6.2 TB/s). With an element per
    lane and load and a workgroup per row, the max over rows took 107 us at
    16384 x 4000 and 47 us at 68848 x 49; now 45 and 6 us."""
    chunks = max(1, -(-m.reduced // CHUNK))
    lanes = row_lanes(m.outer, m.reduced)
    lambdas, given = m.lambdas("full", "reduced", "outer", "one")
    vectors = m.reads("full", "reduced")
    constants = [f"const {t} s{k} = x{k}[{'o' if m.access[k] == 'outer' else '0'}];" for k, t in m.reads("outer", "one")]
    stride, in_flight = lanes * VECTOR, 4

    def stream(k):
        # reduce.hip, streams(): of 8-byte leaves only those beyond the last
        # cache whose rows start on lines.
        size = m.leaves[k].dtype.itemsize
        far = prod(m.leaves[k].shape) * size > 256_000_000 and m.reduced * size % 128 == 0
        return "true" if lanes >= 64 and (size < 8 or far) else "false"

    def declare(u):
        return [f"{t} l{u}_{k}[{VECTOR}];" for k, t in vectors]

    def load(u):
        index = {"full": f"first + r + {u * stride}", "reduced": f"r + {u * stride}"}
        return [f"pacho_loadu<{stream(k)}>(x{k} + ({index[m.access[k]]}), l{u}_{k});" for k, t in vectors]

    def fold(u):
        def value(e):
            arguments = "".join(f", l{u}_{k}[{e}]" if m.access[k] in ("full", "reduced") else f", s{k}" for k in given)
            return f"const {m.acc} t{e} = mapped(first + r + {u * stride + e}{arguments});"

        pairs = [f"const {m.acc} low = {m.combine('t0', 't1')}, high = {m.combine('t2', 't3')};"]
        total = [f"const {m.acc} four = {m.combine('low', 'high')};", f"acc = {m.combine('acc', 'four')};"]
        return ["{", *("  " + line for line in [value(e) for e in range(VECTOR)] + pairs + total), "}"]

    def whole(u):
        return f"r + {u * stride + VECTOR} <= end"

    if lanes == BLOCK:
        finish = f"""if ((threadIdx.x & 63) == 0) partial[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {{
    {m.acc} total = partial[0];
    for (int w = 1; w < {WAVES}; ++w) total = {m.combine("total", "partial[w]")};
    out[g] = total;
  }}"""
    else:
        finish = f"if (lane == 0 && g < {m.outer}LL) out[g] = acc;"
    body = f"""  __shared__ {m.acc} partial[{WAVES}];
  {lambdas}
  const int lane = threadIdx.x % {lanes};
  const long long g = (long long)blockIdx.x * {BLOCK // lanes} + threadIdx.x / {lanes};
  const long long o = g / {chunks}LL, chunk = g % {chunks}LL;
  const long long first = o * {m.reduced}LL;
  const long long begin = chunk * {CHUNK}LL;
  const long long end = begin + {CHUNK}LL < {m.reduced}LL ? begin + {CHUNK}LL : {m.reduced}LL;
  {m.acc} acc = {m.identity};
  if (g < {m.outer * chunks}LL) {{
    {_lines(constants, 4)}
    long long r = begin + lane * {VECTOR};
    for (; r + {(in_flight - 1) * stride + VECTOR} <= end; r += {in_flight * stride}) {{
      {_lines([line for u in range(in_flight) for line in declare(u) + load(u)], 6)}
      {FENCE}
      {_lines([line for u in range(in_flight) for line in fold(u)], 6)}
    }}
    {{  // the groups left over, all loaded before the first is folded
      {_lines([line for u in range(in_flight - 1) for line in declare(u)], 6)}
      {_lines([f"if ({whole(u)}) {{ {' '.join(load(u))} }}" for u in range(in_flight - 1)], 6)}
      {FENCE}
      {_lines([line for u in range(in_flight - 1) for line in [f"if ({whole(u)})", *fold(u)]], 6)}
      while (r + {VECTOR} <= end) r += {stride};
    }}
    for (; r < end; ++r) {{  // one lane's last, partial group
      const {m.acc} value = element(first + r);
      acc = {m.combine("acc", "value")};
    }}
  }}
#pragma unroll
  for (int offset = 1; offset < {min(lanes, 64)}; offset <<= 1) {{
    const {m.acc} other = __shfl_xor(acc, offset, 64);
    acc = {m.combine("acc", "other")};
  }}
  {finish}"""
    return MapReduce(m.kernel(body), m.outer, chunks, -(-m.outer * chunks // (BLOCK // lanes)), (m.outer, chunks))


# Partials of a column reduction: workgroups aimed for per compute unit, rows
# a thread folds at least, and the most bytes of partials.
GROUPS_PER_CU = 2
LEAST_ROWS = 16
MOST_PARTIAL_BYTES = 8 << 20
# A reduction of at most so many bytes and rows does without partials.
ONE_LAUNCH_BYTES = 16 << 20
ONE_LAUNCH_ROWS = 8192


def _column_plan(outer, reduced, inner, width, acc_bytes, unit=1, read=None):
    """(groups of `width` columns a workgroup spans, column blocks, rows per
    step, rows per chunk, chunks). Of the ways to cut a row into equal blocks
    of at least 16 groups (256 bytes of 4-byte columns), a multiple of `unit`,
    the one that leaves the fewest threads without a column, the widest of
    equals. Where that would leave partials of an array of few rows and bytes
    (`read`, None for an array of any size), blocks of a few columns take all
    rows in one launch instead: its lines come from the caches when neighbours
    read them again, and a second launch costs more than that (float32, us a
    call with partials / without: 300 x 17 15.5 / 7.4, 1000 x 1001 17.1 / 8.3,
    8000 x 64 16.5 / 8.0, 4000 x 1024 17.0 / 8.3; past the limits 4000 x 4096
    17.6 / 19.0, 8000 x 1001 17.0 / 17.2). The fewer the rows the wider the
    blocks, about 16 rows a thread, from 16 bytes of columns on."""
    groups = -(-inner // width)
    best, fewest = None, -(-groups // BLOCK)
    for blocks in range(fewest, min(max(fewest, groups // 16), fewest + 32) + 1):
        across = -(-(-(-groups // blocks)) // unit) * unit
        used = groups * (BLOCK // across) / (-(-groups // across) * BLOCK)
        if best is None or used > best[0] + 0.02:
            best = used, across
    across = best[1]
    blocks, step = -(-groups // across), BLOCK // across
    chunks = max(1, COMPUTE_UNITS * GROUPS_PER_CU // (outer * blocks))
    chunks = min(chunks, max(1, MOST_PARTIAL_BYTES // (outer * inner * acc_bytes)))
    rows = max(-(-reduced // chunks), LEAST_ROWS * step)
    rows = -(-rows // step) * step
    chunks = -(-reduced // rows)
    if chunks > 1 and reduced <= ONE_LAUNCH_ROWS and read is not None and read <= ONE_LAUNCH_BYTES:
        least = -(-16 // (width * acc_bytes))
        across = min(groups, max(least, min(8, LEAST_ROWS * BLOCK // reduced)))
        step = BLOCK // across
        return across, -(-groups // across), step, -(-reduced // step) * step, 1
    return across, blocks, step, rows, chunks


def _folded_rows(m, width):
    """Rows that the column kernel takes as one long row, so that every long
    row starts at the same place of a 128-byte line (of a 16-byte vector for
    fewer rows), and whether it is the line; 1 where rows are whole vectors,
    where a leaf varies along the rows, where too few long rows would be left
    for each of their columns' own partial, or where one launch of single
    columns does it without partials."""
    if m.inner % width == 0 or m.reads("reduced"):
        return 1, False
    if _column_plan(m.outer, m.reduced, m.inner, 1, m.acc_dtype.itemsize, read=m.bytes_read())[4] == 1:
        return 1, False
    for period, least in ((8 * width, 64), (width, 16)):
        rows = period // gcd(m.inner, period)
        if m.reduced >= least * rows and m.outer * rows * m.inner * m.acc_dtype.itemsize <= MOST_PARTIAL_BYTES:
            return rows, period > width
    return 1, False


# Batches of a float sum that may join one accumulator one after the other.
LONGEST_CHAIN = 4


def _cascade(m, width, levels):
    """Sources that declare, add to and close `levels` partial sums of `carry`s:
    level l holds the sum of 2^l of them and is full where bit l of their count
    is set, so that every sum is of two of the same size. A chain of them adds
    an error of its length's root: 4095 rows of 524288 float32 columns, 512
    batches in one chain, had 7 times the error of lanes that meet in a tree
    (squares of normal values, rms), and with levels 0.93 times (300 to 262144
    rows: 0.91 to 1.10, which the sample does not tell apart). The count is the
    same for all threads of a wave that still add, so the branches cost a
    scalar test each: 4095 x 262144 float32 took 672 us in one chain and 648
    with levels, 100003 x 1025 68.4 and 68.1, 65536 x 4096 167 and 165."""
    if not levels:
        return [], [], []
    each = f"_Pragma(\"unroll\") for (int v = 0; v < {width}; ++v)"
    declare = [f"{m.acc} carry[{width}], level[{levels}][{width}];", "unsigned count = 0;"]
    join, close = [], ["}" * (levels - 1)]
    for l in range(levels):
        keep = f"{each} level[{l}][v] = carry[v];"
        if l == levels - 1:
            join.append(keep)
        else:
            add = f"{each} carry[v] = {m.combine(f'level[{l}][v]', 'carry[v]')};"
            join += [f"if (!(count & {1 << l}U)) {{ {keep} }} else {{", f"  {add}"]
    join += [*close, "++count;"]
    close = [f"if (count & {1 << l}U) {{ {each} acc[v] = {m.combine('acc[v]', f'level[{l}][v]')}; }}" for l in range(levels)]
    return declare, join, close


def _columns(m):
    """A workgroup owns a block of columns and a chunk of rows; a thread reads
    `width` adjacent columns of every step-th row, eight rows (16 of one
    column) in flight. Each batch folds on its own, in pairs; the batches of a
    float sum then meet in pairs too (_cascade), those of other reductions in
    one accumulator; the rows of a step meet in LDS in a fixed tree. Leaves
    that vary along inner only are read once. Bound by HBM: where rows are whole vectors a thread takes 16 bytes
    with the nontemporal hint (100003 x 1024 float32: 67 us, 6.1 TB/s, against
    78 us without the hint). Other rows are folded (_folded_rows): 32 rows of
    1025 float32 are one row of 32800 columns that starts on a line, whose
    partials are 32 rows of the result's partials, and the last, cut long row
    goes element by element: the sum of squares of 100003 x 1025 float32 88 us
    by single columns, 73 with long rows that start on 16 bytes, 67 on lines.
    Where that does not serve, a thread takes one column without the hint. Workgroups are renumbered so that an XCD
    (ids i % 8) owns neighbouring column blocks, which share lines. With a
    lane per row of one column and 64 lines per wave access, the mean square
    over axis 0 of 100003 x 1025 took 1062 us."""
    wide = max([m.acc_dtype.itemsize, *(leaf.dtype.itemsize for leaf in m.leaves if not leaf.scalar)]) == 8
    width, batch = 2 if wide else 4, 8
    stream = "true"
    folded, lines_whole = _folded_rows(m, width)
    if folded == 1 and m.inner % width:
        width, batch, stream = 1, 16, "false"
    inner, total = folded * m.inner, m.reduced * m.inner
    reduced = -(-m.reduced // folded)
    across, blocks, step, rows, chunks = _column_plan(
        m.outer, reduced, inner, width, m.acc_dtype.itemsize, 8 if lines_whole else 1,
        m.bytes_read() if folded == 1 else None,
    )
    grid = m.outer * chunks * blocks
    lambdas, given = m.lambdas("full", "reduced", "outer", "inner", "one")
    constants = [f"const {t} s{k} = x{k}[{'o' if m.access[k] == 'outer' else '0'}];" for k, t in m.reads("outer", "one")]
    for k, t in m.reads("inner"):
        each = f"_Pragma(\"unroll\") for (int v = 0; v < {width}; ++v) c{k}[v] = x{k}[(col + v) % {m.inner}LL];"
        constants.append(f"{t} c{k}[{width}]; " + (each if folded > 1 else f"pacho_loadu<false>(x{k} + col, c{k});"))

    def loads(j):
        at = f"first + r * {inner}LL + {j * step * inner}LL"
        lines = [f"{t} l{j}_{k}[{width}]; pacho_loadu<{stream}>(x{k} + ({at}), l{j}_{k});" for k, t in m.reads("full")]
        return lines + [f"const {t} l{j}_{k} = x{k}[r + {j * step}];" for k, t in m.reads("reduced")]

    def value(j, v):
        names = {"full": f"l{j}_%d[{v}]", "reduced": f"l{j}_%d", "inner": f"c%d[{v}]"}
        arguments = "".join(", " + names.get(m.access[k], "s%d") % k for k in given)
        return f"mapped(first + r * {inner}LL + {j * step * inner + v}LL{arguments})"

    most = -(-rows // (batch * step))  # batches of a thread
    levels = most.bit_length() if m.operation == "sum" and m.acc_dtype.kind == "f" and most > LONGEST_CHAIN else 0

    def within(j):
        return f"r + {j * step} < whole"

    def left_over():
        """The loads of a batch that is not full."""
        lines = []
        for j in range(batch - 1):
            lines += [f"{t} l{j}_{k}[{width}] = {{}};" for k, t in m.reads("full")] + [f"{t} l{j}_{k} = {{}};" for k, t in m.reads("reduced")]
            at = f"first + r * {inner}LL + {j * step * inner}LL"
            some = [f"pacho_loadu<{stream}>(x{k} + ({at}), l{j}_{k});" for k, _ in m.reads("full")]
            some += [f"l{j}_{k} = x{k}[r + {j * step}];" for k, _ in m.reads("reduced")]
            lines.append(f"if ({within(j)}) {{ {' '.join(some)} }}")
        return lines

    def fold(count, into="acc"):
        full = count == batch
        lines = []
        for v in range(width):
            some = (value(j, v) if full else f"{within(j)} ? {value(j, v)} : {m.identity}" for j in range(count))
            lines += ["{", *(f"  {m.acc} some{j} = {one};" for j, one in enumerate(some))]
            apart = 1
            while apart < count:
                for j in range(0, count - apart, 2 * apart):
                    lines.append(f"  some{j} = {m.combine(f'some{j}', f'some{j + apart}')};")
                apart *= 2
            joined = m.combine(f"acc[{v}]", "some0") if into == "acc" else "some0"
            lines += [f"  {into}[{v}] = {joined};", "}"]
        return lines

    declare, join, close = _cascade(m, width, levels)
    tree = f"""
  for (int n = {step}; n > 1;) {{
    const int half = (n + 1) / 2;
#pragma unroll
    for (int v = 0; v < {width}; ++v) partial[threadIdx.x * {width} + v] = acc[v];
    __syncthreads();
    if (row < n - half) {{
#pragma unroll
      for (int v = 0; v < {width}; ++v) {{
        const {m.acc} other = partial[(threadIdx.x + half * {across}) * {width} + v];
        acc[v] = {m.combine("acc[v]", "other")};
      }}
    }}
    __syncthreads();
    n = half;
  }}""" if step > 1 else ""
    body = f"""  __shared__ {m.acc} partial[{BLOCK * width if step > 1 else 1}];
  {lambdas}
  const unsigned id = at < {grid // 8 * 8}U ? at % 8 * {grid // 8}U + at / 8 : at;
  const unsigned block = id % {blocks}U, chunk = id / {blocks}U % {chunks}U;
  const long long o = id / {blocks * chunks}U;
  const int row = threadIdx.x / {across};
  const long long col = (block * {across}LL + threadIdx.x % {across}) * {width};
  const bool active = row < {step} && col < {inner}LL;
  const long long first = o * {total}LL + col;
  const long long begin = chunk * {rows}LL;
  const long long end = begin + {rows}LL < {reduced}LL ? begin + {rows}LL : {reduced}LL;
  // Rows that hold all of this thread's columns: all but the last of folded ones.
  const long long full = ({total}LL - col - {width} + {inner}LL) / {inner}LL, whole = full < end ? full : end;
  {m.acc} acc[{width}];
#pragma unroll
  for (int v = 0; v < {width}; ++v) acc[v] = {m.identity};
  if (active) {{
    {_lines(constants + declare, 4)}
    long long r = begin + row;
    for (; r + {(batch - 1) * step} < whole; r += {batch * step}) {{
      {_lines([line for j in range(batch) for line in loads(j)], 6)}
      {FENCE}
      {_lines(fold(batch, "carry") + join if levels else fold(batch), 6)}
    }}
    if (r < whole) {{  // the rows left over, as one batch
      {_lines(left_over(), 6)}
      {FENCE}
      {_lines(fold(batch - 1, "carry") + join if levels else fold(batch - 1), 6)}
      while (r < whole) r += {step};
    }}
    if (r < end) {{
      for (int v = 0; v < {width}; ++v) {{
        if (r * {inner}LL + col + v < {total}LL) {{
          const {m.acc} value = element(first + r * {inner}LL + v);
          acc[v] = {m.combine("acc[v]", "value")};
        }}
      }}
    }}
    {_lines(close, 4)}
  }}{tree}
  if (active && row == 0) {{
    for (int v = 0; v < {width}; ++v) out[(o * {chunks}LL + chunk) * {inner}LL + col + v] = acc[v];
  }}"""
    return MapReduce(
        m.kernel(body, grid), m.outer * m.inner, chunks * folded, min(grid, MOST_WORKGROUPS),
        (m.outer, chunks * folded, m.inner),
    )


def _any(m):
    """Reduced axes that are not adjacent, none, or an empty array: a workgroup
    per (output, CHUNK of its elements), one element per lane."""
    index, count, reduced = source_._reduction_index(m.shape, m.axes)
    chunks = max(1, -(-reduced // CHUNK))
    body = f"""  __shared__ {m.acc} partial[{WAVES}];
  {m._lambda("element", [])}
  const long long g = at;
  const long long o = g / {chunks}LL, chunk = g % {chunks}LL;
  const long long begin = chunk * {CHUNK}LL;
  const long long end = begin + {CHUNK}LL < {reduced}LL ? begin + {CHUNK}LL : {reduced}LL;
  {m.acc} acc = {m.identity};
  for (long long r = begin + threadIdx.x; r < end; r += {BLOCK}) {{
    const {m.acc} value = element({index});
    acc = {m.combine("acc", "value")};
  }}
#pragma unroll
  for (int offset = 1; offset < 64; offset <<= 1) {{
    const {m.acc} other = __shfl_xor(acc, offset, 64);
    acc = {m.combine("acc", "other")};
  }}
  if ((threadIdx.x & 63) == 0) partial[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {{
    {m.acc} total = partial[0];
    for (int w = 1; w < {WAVES}; ++w) total = {m.combine("total", "partial[w]")};
    out[g] = total;
  }}"""
    grid = count * chunks
    return MapReduce(m.kernel(body, grid), count, chunks, min(grid, MOST_WORKGROUPS), (count, chunks))
