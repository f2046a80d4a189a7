"""Launches of a compiled plan: its steps regrouped so that the device reads
and starts less, with the same values.

The compiler's steps (what ``explain()`` reports) say what is computed; this
module decides which of them share a kernel. Every elementwise node keeps its
own rounding and every element the same expression, so the results of a
regrouped plan are those of its steps, except that a row reduction inside a
row program may add in another fixed order. In turn:

1. rows: consecutive steps over the same rows (reductions along the last axes,
   elementwise steps that read their results back along the row) become one
   kernel that holds the row in registers: softmax reads its input once and
   writes its result once, where four steps moved six arrays (16384 x 4000
   float32: 264 -> 100 us);
2. inlining: an elementwise value that only other elementwise groups read is
   recomputed in each of them where that moves fewer bytes than writing it and
   reading it back (column standardisation of 100003 x 1025 float32:
   479 -> 404 us), or where it is a single element;
3. merging: independent elementwise steps become ranges of one launch's
   workgroups (the four weight updates of an SGD step, the two vector updates
   of a conjugate gradient iteration: about 5 us for each launch saved).
"""

from math import prod
from typing import Any, NamedTuple

import numpy as np

from . import _hip_lowering as source_
from ._compiler import ELEMENTWISE, Step
from ._hip_map_reduce import CHUNK, COMPUTE_UNITS, WAVES, row_lanes

# Operations cheap enough to repeat in every reader of a value.
CHEAP = frozenset(
    "add subtract multiply negative positive absolute where cast equal not_equal less less_equal greater "
    "greater_equal isfinite".split()
)
MOST_REPEATED = 4  # nodes of an inlined value
MOST_MERGED = 8  # outputs of a merged launch
MOST_ARGUMENTS = 256  # operands of its members together: far below what a packed launch takes
SMALL = 1 << 16  # elements up to which a step may run later than the plan has it
MOST_REGISTERS = 160  # 32-bit registers of row values per lane
# By operation and whether it is in float32 or wider. What one element adds to
# the time of a lane that has its SIMD to itself, in us (the rest: next to
# nothing), fitted to rows of 4000 to 16384 elements.
LANE_TIME = {
    ("power", 4): 0.55, ("sin", 4): 0.1, ("cos", 4): 0.1, ("tanh", 4): 0.1,
    ("power", 8): 0.55, ("tanh", 8): 0.33, ("sin", 8): 0.2, ("cos", 8): 0.2, ("log", 8): 0.2, ("exp", 8): 0.05,
}
LAUNCH_TIME = 4.0  # us that a launch less saves a call
# Elements that fit the compiler's limit on a lane's unrolled code; past it the
# row goes to scratch memory (sin over 16384 x 16384 float32: 531 us in steps,
# 1183 in a program of 64 elements a lane; 56 still fit).
MOST_UNROLLED = {
    ("sin", 4): 56, ("cos", 4): 56, ("tanh", 4): 192,
    ("sin", 8): 64, ("cos", 8): 64, ("power", 8): 64, ("tanh", 8): 96, ("log", 8): 192,
}


class Launch(NamedTuple):
    """Several steps in one kernel: the nodes it stores, the values it reads."""

    nodes: tuple
    args: tuple
    payload: Any


class _Kernel(NamedTuple):
    source: str
    name: str
    grid: int


def arrange(lowering, steps, outputs):
    """The plan's launches in order: Step objects as they came, or with another
    payload, and Launch objects."""
    kept = {id(node) for node in outputs}
    return _merge(_inline(lowering, _rows(list(steps), kept), kept))


def _stored(launch):
    return launch.nodes if isinstance(launch, Launch) else (launch.node,)


def _collect(root, stored):
    """(group in dependency order, leaves) of the elementwise value `root`:
    nodes down to inputs, scalars and the values in `stored` (ids)."""
    group, leaves, seen = [], [], set()

    def visit(node, first):
        if id(node) in seen:
            return
        seen.add(id(node))
        if node.op in ELEMENTWISE and (first or id(node) not in stored):
            for child in node.inputs:
                visit(child, False)
            group.append(node)
        else:
            leaves.append(node)

    visit(root, True)
    return group, leaves


# ---- 1: row programs -----------------------------------------------------------


class _RowSpace:
    """Rows of `shape` along its last axes: (outer, reduced)."""

    def __init__(self, shape, axes):
        self.shape, self.axes = tuple(shape), tuple(axes)
        self.outer, self.reduced = prod(self.shape[: axes[0]]), prod(self.shape[axes[0] :])

    def access(self, shape):
        """How (o, r) reads an array of `shape`: 'full', 'outer', 'reduced', 'one', or None."""
        shape = tuple(shape)
        if len(shape) > len(self.shape):
            return None
        padded = (1,) * (len(self.shape) - len(shape)) + shape
        first = self.axes[0]
        head, tail = padded[:first], padded[first:]
        row, column = self.shape[:first], self.shape[first:]
        ones = all(d == 1 for d in head), all(d == 1 for d in tail)
        if all(ones):
            return "one"
        if head == row and tail == column:
            return "full"
        if head == row and ones[1]:
            return "outer"
        if ones[0] and tail == column:
            return "reduced"
        return None

    @classmethod
    def of(cls, step):
        """The rows that a reduction step reduces, or None."""
        if step.kind not in ("reduce", "map_reduce"):
            return None
        node = step.node
        shape, axes = tuple(node.inputs[0].shape), tuple(node.attrs["axes"])
        trailing = axes and axes == tuple(range(axes[0], len(shape)))
        if not trailing or prod(shape) == 0 or node.dtype.kind == "b" or prod(shape) > 2**31 - 1:
            return None
        space = cls(shape, axes)
        return space if space.reduced > 1 else None


def _rows(steps, kept):
    """Replace runs of steps over the same rows by row programs."""
    result, i = [], 0
    while i < len(steps):
        best = None
        for space in _spaces(steps, i):
            end = i
            while end < len(steps) and _joins(steps, i, end, space):
                end += 1
            while end > i + 1:
                program = _row_program(steps, i, end, space, kept)
                if program is not None:
                    best = (end, program) if best is None or end > best[0] else best
                    break
                end -= 1
        if best is None:
            result.append(steps[i])
            i += 1
        else:
            result.append(best[1])
            i = best[0]
    return result


def _spaces(steps, i):
    """Row spaces that a run starting at step i could have: that of the first
    reduction at or shortly after it."""
    for step in steps[i : i + 3]:
        space = _RowSpace.of(step)
        if space is not None:
            return [space]
    return []


def _joins(steps, begin, end, space):
    """Whether steps[end] can run in the row program of steps[begin:end]."""
    step = steps[end]
    inside = {id(s.node) for s in steps[begin:end]}
    if step.kind in ("reduce", "map_reduce"):
        own = _RowSpace.of(step)
        if own is None or (own.shape, own.axes) != (space.shape, space.axes):
            return False
    elif step.kind != "fused" or space.access(step.node.shape) not in ("full", "outer"):
        return False
    for arg in step.args:
        access = "one" if arg.op == "scalar" and not arg.shape else space.access(arg.shape)
        # A result of this run is only known along its own row.
        if access is None or (id(arg) in inside and access not in ("full", "outer")):
            return False
    return True


def _lanes(space):
    lanes = row_lanes(space.outer, space.reduced)
    return lanes if lanes < 64 or space.reduced <= 2048 and lanes == 64 else source_.BLOCK


def _row_program(steps, begin, end, space, kept):
    """The Launch of steps[begin:end], or None where it would not save a pass
    over the rows or they do not fit the registers."""
    run = steps[begin:end]
    inside = {id(s.node): s for s in run}
    reductions = [s for s in run if s.kind != "fused"]
    full = [s for s in run if s.kind == "fused" and space.access(s.node.shape) == "full"]
    if not reductions or len(reductions) + len(full) < 2:
        return None
    later = {id(a) for s in steps[end:] for a in s.args}
    outputs = [s.node for s in run if id(s.node) in kept or id(s.node) in later]
    args = []
    for step in run:
        for arg in step.args:
            if id(arg) not in inside and all(arg is not a for a in args):
                args.append(arg)
    leaves = [source_._leaf_of(a) for a in args]
    access = [None if leaf.scalar else space.access(leaf.shape) for leaf in leaves]
    lanes = _lanes(space)
    groups = -(-space.reduced // (lanes * source_.VECTOR))
    words = [max(1, leaf.dtype.itemsize // 4) for leaf, a in zip(leaves, access) if a in ("full", "reduced")]
    words += [max(1, s.node.dtype.itemsize // 4) for s in full if any(s.node is a for t in run for a in t.args)]
    if groups * source_.VECTOR * sum(words) > MOST_REGISTERS:
        return None
    if sum(a == "full" for a in access) > 4:
        return None
    grid = -(-space.outer // (source_.BLOCK // lanes))
    if not _serves(run, {id(a) for a in args} | set(inside), space, groups * source_.VECTOR, grid):
        return None
    source = _row_source(run, inside, outputs, args, leaves, access, space, lanes, groups)
    return Launch(tuple(outputs), tuple(args), _Kernel(source, "pacho_rows", grid))


def _serves(run, stored, space, elements, grid):
    """Whether a program of `elements` a lane and `grid` workgroups is as fast
    as its steps. Few long rows leave most of the chip to the steps alone, whose
    lanes take 16 elements each: with operations that keep a lane busy that is
    worth more than the launches (x ** 1.7 and its maximum over 4 x 8192
    float32, alone: 31.4 us against 27.4; tanh over 4 x 8192 float64 27.3
    against 24.6, over 4 x 4000 22.5 against 23.4). The gap closes as workgroups
    share compute units, at four of them altogether (1024 x 8192 float64, power:
    59.7 against 64.1)."""
    time = 0.0
    for step in run:
        fused = step.kind == "fused"
        root = step.node if fused else step.node.inputs[0]
        if (fused and space.access(root.shape) != "full") or (not fused and id(root) in stored):
            continue
        group, _ = _collect(root, stored - {id(root)})
        kinds = [(node.op, 4 if node.dtype == np.float32 else 8) for node in group]
        if sum(elements / MOST_UNROLLED[kind] for kind in kinds if kind in MOST_UNROLLED) > 1:
            return False
        time += sum(LANE_TIME.get(kind, 0.0) for kind in kinds)
    launches = len(run) - 1 + sum(step.kind != "fused" and space.reduced > CHUNK for step in run)
    idle = max(0.0, 1 - grid / (4 * COMPUTE_UNITS))
    more = elements - source_.ELEMENTS_PER_THREAD * source_.VECTOR
    return time * more * idle <= LAUNCH_TIME * launches


def _row_source(run, inside, outputs, args, leaves, access, space, lanes, groups):
    """One pass: a lane loads its groups of VECTOR consecutive elements (the
    order of the row reductions: group g of a lane starts at (g * lanes + lane)
    * VECTOR), all leaves before the first use, then every step runs over them
    in turn. Row results are held by every lane of the row."""
    vector, block = source_.VECTOR, source_.BLOCK
    ctype = source_.ctype
    position = {id(a): k for k, a in enumerate(args)}
    number = {id(s.node): j for j, s in enumerate(run)}
    whole = space.reduced // (lanes * vector)  # groups that every lane has whole
    params = [f"{ctype(l.dtype)} x{k}" if l.scalar else f"const {ctype(l.dtype)}* __restrict__ x{k}" for k, l in enumerate(leaves)]
    params += [f"{ctype(node.dtype)}* __restrict__ out{j}" for j, node in enumerate(outputs)]
    lines = []
    for k, (leaf, a) in enumerate(zip(leaves, access)):
        t = ctype(leaf.dtype)
        if a in ("full", "reduced"):
            at = "first + r" if a == "full" else "r"
            lines.append(f"{t} l{k}[{groups}][{vector}];")
            lines.append(
                f"_Pragma(\"unroll\") for (int g = 0; g < {groups}; ++g) {{ const int r = (g * {lanes} + lane) * {vector}; "
                f"if (g < {whole} || r + {vector} <= {space.reduced}) pacho_loadu<false>(x{k} + {at}, l{k}[g]); "
                f"else {{ _Pragma(\"unroll\") for (int e = 0; e < {vector}; ++e) l{k}[g][e] = r + e < {space.reduced} ? x{k}[{at} + e] : ({t})0; }} }}"
            )
        elif a in ("outer", "one"):
            lines.append(f"const {t} s{k} = x{k}[{'o' if a == 'outer' else '0'}];")
    lines.append("__builtin_amdgcn_sched_barrier(0);")

    def value_of(node):
        """Expression of a leaf's or an earlier step's value at element (g, e)."""
        if id(node) in position:
            k = position[id(node)]
            if leaves[k].scalar:
                return f"x{k}"
            return f"l{k}[g][e]" if access[k] in ("full", "reduced") else f"s{k}"
        j = number[id(node)]
        return f"q{j}[g][e]" if space.access(node.shape) == "full" else f"q{j}"

    def expression(root, is_root_stored):
        """Lines and symbol of the elementwise value `root`."""
        if id(root) in position or (id(root) in number and not is_root_stored):
            return [], value_of(root)
        group, group_leaves = _collect(root, (set(position) | set(number)) - {id(root)})
        specs, nodes = source_._graph(group, group_leaves)
        names = [value_of(leaf) for leaf in group_leaves]
        plain = [source_._Leaf(False, spec.dtype, spec.shape) for spec in specs]
        _, body, symbol = source_._body(space.shape, plain, nodes, leaf_value=lambda k: names[k])
        return body, symbol

    for j, step in enumerate(run):
        node, t = step.node, ctype(step.node.dtype)
        stored = [i for i, out in enumerate(outputs) if out is node]
        if step.kind == "fused":
            body, symbol = expression(node, True)
            if space.access(node.shape) == "full":
                lines.append(f"{t} q{j}[{groups}][{vector}];")
                lines.append(f"_Pragma(\"unroll\") for (int g = 0; g < {groups}; ++g) _Pragma(\"unroll\") for (int e = 0; e < {vector}; ++e) {{")
                lines += ["  " + line for line in body] + [f"  q{j}[g][e] = {symbol};", "}"]
                for i in stored:
                    lines.append(
                        f"if (mine) {{ _Pragma(\"unroll\") for (int g = 0; g < {groups}; ++g) {{ const int r = (g * {lanes} + lane) * {vector}; "
                        f"if (g < {whole} || r + {vector} <= {space.reduced}) pacho_storeu(out{i} + first + r, q{j}[g]); "
                        f"else {{ _Pragma(\"unroll\") for (int e = 0; e < {vector}; ++e) if (r + e < {space.reduced}) out{i}[first + r + e] = q{j}[g][e]; }} }} }}"
                    )
            else:
                lines += [f"{t} q{j};", "{", *("  " + line for line in body), f"  q{j} = {symbol};", "}"]
                lines += [f"if (mine && lane == 0) out{i}[o] = q{j};" for i in stored]
            continue
        operation = node.attrs.get("operation", "sum")
        dtype = node.dtype

        def combine(left, right):
            return source_._combine(operation, dtype, left, right)

        root = node.inputs[0]
        body, symbol = expression(root, False)
        boolean = root.dtype.kind == "b"
        symbol = f"({symbol} != 0)" if boolean else symbol
        lines.append(f"{t} q{j} = {source_._identity(operation, dtype)};")
        lines.append(f"_Pragma(\"unroll\") for (int g = 0; g < {groups}; ++g) {{")
        lines.append(f"  {t} t[{vector}];")
        lines.append(f"  _Pragma(\"unroll\") for (int e = 0; e < {vector}; ++e) {{")
        lines += ["    " + line for line in body] + [f"    t[e] = ({t})({symbol});", "  }"]
        lines.append(f"  const int r = (g * {lanes} + lane) * {vector};")
        lines.append(f"  if (g < {whole} || r + {vector} <= {space.reduced}) {{")
        lines.append(f"    const {t} low = {combine('t[0]', 't[1]')}, high = {combine('t[2]', 't[3]')};")
        lines.append(f"    const {t} four = {combine('low', 'high')};")
        lines.append(f"    q{j} = {combine(f'q{j}', 'four')};")
        lines.append("  } else {")
        lines.append(f"    _Pragma(\"unroll\") for (int e = 0; e < {vector}; ++e) if (r + e < {space.reduced}) q{j} = {combine(f'q{j}', 't[e]')};")
        lines.append("  }")
        lines.append("}")
        lines.append(f"_Pragma(\"unroll\") for (int offset = 1; offset < {min(lanes, 64)}; offset <<= 1) {{")
        lines.append(f"  const {t} other = __shfl_xor(q{j}, offset, 64);")
        lines.append(f"  q{j} = {combine(f'q{j}', 'other')};")
        lines.append("}")
        if lanes == block:
            lines.append("{")
            lines.append(f"  __shared__ {t} partial[{WAVES}];")
            lines.append(f"  if ((threadIdx.x & 63) == 0) partial[threadIdx.x >> 6] = q{j};")
            lines.append("  __syncthreads();")
            lines.append(f"  q{j} = partial[0];")
            lines.append(f"  _Pragma(\"unroll\") for (int w = 1; w < {WAVES}; ++w) q{j} = {combine(f'q{j}', 'partial[w]')};")
            lines.append("}")
        lines += [f"if (mine && lane == 0) out{i}[o] = q{j};" for i in stored]
    body = "\n  ".join(lines)
    return f"""{source_._PRELUDE}
extern "C" __global__ __launch_bounds__({block}) void pacho_rows({", ".join(params)}) {{
  const int lane = threadIdx.x % {lanes};
  const long long row = (long long)blockIdx.x * {block // lanes} + threadIdx.x / {lanes};
  const bool mine = row < {space.outer}LL;
  const long long o = mine ? row : {space.outer - 1}LL;  // spare lanes repeat the last row and store nothing
  const long long first = o * {space.reduced}LL;
  {body}
}}
"""


# ---- 2: inlining ---------------------------------------------------------------


def _inline(lowering, launches, kept):
    """Drop the steps whose values are better recomputed by their readers."""
    readers = {}
    for launch in launches:
        for arg in launch.args:
            readers.setdefault(id(arg), []).append(launch)
    dropped = set()
    for launch in launches:
        if isinstance(launch, Launch) or launch.kind != "fused" or id(launch.node) in kept:
            continue
        if _worth_repeating(launch, readers.get(id(launch.node), []), dropped):
            dropped.add(id(launch.node))
    if not dropped:
        return launches
    stored = {id(node) for launch in launches for node in _stored(launch)} - dropped
    result = []
    for launch in launches:
        if not isinstance(launch, Launch) and id(launch.node) in dropped:
            continue
        if any(id(arg) in dropped for arg in launch.args):
            root = launch.node if launch.kind == "fused" else launch.node.inputs[0]
            group, leaves = _collect(root, stored)
            prepare = lowering.prepare_fused if launch.kind == "fused" else lowering.prepare_map_reduce
            args, payload = prepare(launch.node, group, leaves)
            launch = Step(launch.node, launch.kind, tuple(args), payload)
        result.append(launch)
    return result


def _worth_repeating(step, readers, dropped):
    """Whether every reader of `step` can compute its value itself for less."""
    if not readers or any(isinstance(r, Launch) or r.kind not in ("fused", "map_reduce") for r in readers):
        return False
    # A bare reduction of the stored value has its own kernel and order.
    if any(r.kind == "map_reduce" and r.node.inputs[0] is step.node for r in readers):
        return False
    if any(id(arg) in dropped for arg in step.args):
        return False
    group, leaves = _collect(step.node, {id(arg) for arg in step.args})
    if len(group) > MOST_REPEATED:
        return False
    size = prod(step.node.shape)
    if size == 1:
        return all(node.op in CHEAP or node.op in ("true_divide", "divide") for node in group)
    if any(node.op not in CHEAP for node in group):
        return False

    def bytes_of(node):
        return 0 if node.op == "scalar" else prod(node.shape) * node.dtype.itemsize

    own = size * step.node.dtype.itemsize
    read = sum(bytes_of(leaf) for leaf in leaves)
    stored_cost = read + own + len(readers) * own
    inline_cost = sum(sum(bytes_of(leaf) for leaf in leaves if all(leaf is not a for a in r.args)) for r in readers)
    return inline_cost < stored_cost


# ---- 3: merging ----------------------------------------------------------------


def _merge(launches):
    """Join independent elementwise steps into launches of several outputs. A
    launch stands where its last member stood, after the steps between; only
    small members wait like that, large ones join their direct neighbours."""
    result, at = [], 0
    while at < len(launches):
        members, last = [launches[at]], at
        if _is_fused(launches[at]):
            for i in range(at + 1, len(launches)):
                later = launches[i]
                stored = {id(s.node) for s in members}
                if len(members) == MOST_MERGED or any(id(arg) in stored for arg in later.args):
                    break
                small = all(prod(s.node.shape) <= SMALL for s in members)
                operands = sum(len(s.args) for s in members) + len(later.args)
                if _is_fused(later) and (small or last == i - 1) and operands <= MOST_ARGUMENTS:
                    members.append(later)
                    last = i
                elif not small:
                    break
        result += [s for s in launches[at : last + 1] if all(s is not m for m in members)]
        result.append(members[0] if len(members) == 1 else _merged(members))
        at = last + 1
    return result


def _is_fused(launch):
    return not isinstance(launch, Launch) and launch.kind == "fused" and prod(launch.node.shape) > 0


def _merged(members):
    """One kernel whose workgroups are dealt out to the members in turn."""
    parts, params, args, names, grid = [], [], [], {}, 0
    for j, step in enumerate(members):
        group, leaves = _collect(step.node, {id(arg) for arg in step.args})
        specs, nodes = source_._graph(group, leaves)
        mapping = []
        for leaf, spec in zip(leaves, specs):
            if id(leaf) not in names:
                names[id(leaf)] = f"a{len(args)}"
                t = source_.ctype(spec.dtype)
                params.append(f"{t} a{len(args)}" if spec.scalar else f"const {t}* __restrict__ a{len(args)}")
                args.append(leaf)
            mapping.append(names[id(leaf)])
        body, own_params, blocks = source_.elementwise_body(step.node.shape, specs, nodes, np.dtype(step.node.dtype))
        parts.append((j, body, own_params, mapping, blocks, source_.ctype(step.node.dtype)))
        grid += blocks
    functions, calls, at = [], [], 0
    for j, body, own_params, mapping, blocks, t in parts:
        functions.append(
            f"__device__ __forceinline__ void part{j}(const unsigned block, {', '.join(own_params)}) {{\n{body}\n}}\n"
        )
        test = f"if (blockIdx.x < {at + blocks}U)" if j < len(parts) - 1 else ""
        calls.append(f"{test} {{ part{j}(blockIdx.x - {at}U, {', '.join([*mapping, f'out{j}'])}); return; }}")
        params.append(f"{t}* __restrict__ out{j}")
        at += blocks
    source = f"""{source_._PRELUDE}
{"".join(functions)}
extern "C" __global__ __launch_bounds__({source_.BLOCK}) void pacho_merged({", ".join(params)}) {{
  {(chr(10) + "  ").join(calls)}
}}
"""
    return Launch(tuple(s.node for s in members), tuple(args), _Kernel(source, "pacho_merged", grid))
