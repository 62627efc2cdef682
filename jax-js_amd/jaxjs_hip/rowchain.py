"""Chains of Kernels over the same rows, run as one launch (`rows.hip.inc`).

The front-end's fusion boundaries (src/frontend/jit.ts:572-789) leave a softmax, a layer normalisation or an argmax as
three to five Kernels that read the same `[R, C]` rows: reductions along a row, maps over the rows that use the
reductions' results, maps of the per-row results.  `RowChain` is such a run of Kernels; `collect_chain` finds one in a
list of dispatches, `gen_rows` writes its source.  Every intermediate keeps the storage type it has between separate
launches, so results differ from theirs by nothing but the order of a reduction's terms.
"""

from __future__ import annotations

from dataclasses import dataclass, field
from typing import Dict, List, Optional, Sequence, Tuple

from .alu import AluExp, AluOp, DType, Kernel, byteWidth
from .codegen import CTYPE, SOURCE_OPTION, STORAGE_CTYPE, _fits_i32, const_literal
from .composite import Composite
from .kernelgen import IDENT, KernelSource, LaunchStep, _Body, _lane_accumulate, _prelude, _reduce_text, fill, template
from . import tuner

MAX_LANES = 1024


# ---- index forms -----------------------------------------------------------------------------------------------------
# An index over the symbols gidx in [0, R) and ridx in [0, C) as a sum of multiples of floor(symbol / a):
# {(symbol, a): factor} with the constant under None.  `x % b` is x - b * floor(x / b), so two ways of unravelling and
# ravelling the same position come out as the same sum, which the term-by-term simplifier does not see.

Form = Dict[Optional[Tuple[str, int]], int]


def _tidy(f: Form, extent: Dict[str, int]) -> Form:
    return {k: v for k, v in f.items() if v and (k is None or k[1] < extent[k[0]])}  # floor(s / a) is 0 for a >= extent


def _bounds(f: Form, extent: Dict[str, int]) -> Tuple[int, int]:
    lo = hi = f.get(None, 0)
    for k, v in f.items():
        if k is not None:
            top = v * ((extent[k[0]] - 1) // k[1])
            lo, hi = lo + min(top, 0), hi + max(top, 0)
    return lo, hi


def _divide(f: Form, d: int, extent: Dict[str, int]) -> Optional[Form]:
    """floor(f / d) for f >= 0, where it is such a sum again."""
    out = {k: v // d for k, v in f.items() if v % d == 0}
    rest = {k: v for k, v in f.items() if v % d}
    lo, hi = _bounds(rest, extent)
    if 0 <= lo and hi < d:
        return out
    # one term g * floor(s / a) with g | d, the others below g: its quotient is floor(s / (a * d / g))
    for k, g in sorted(((k, v) for k, v in rest.items() if k is not None and v > 0), key=lambda kv: -kv[1]):
        lo, hi = _bounds({q: v for q, v in rest.items() if q != k}, extent)
        if d % g == 0 and 0 <= lo and hi < g:
            at = (k[0], k[1] * (d // g))
            out[at] = out.get(at, 0) + 1
            return _tidy(out, extent)
    return None


def index_form(e: AluExp, extent: Dict[str, int]) -> Optional[Form]:
    """The form of an int32 index expression over the two symbols, or None where it has none."""
    if e.op == AluOp.Const:
        return {None: int(e.arg)} if e.arg else {}
    if e.op == AluOp.Special:
        return _tidy({(e.arg[0], 1): 1}, extent) if e.arg[0] in extent else None
    if e.dtype != DType.Int32 or e.op not in (AluOp.Add, AluOp.Sub, AluOp.Mul, AluOp.Idiv, AluOp.Mod) or not _fits_i32(e):
        return None
    a, b = index_form(e.src[0], extent), index_form(e.src[1], extent)
    if a is None or b is None:
        return None
    if e.op in (AluOp.Add, AluOp.Sub):
        s = 1 if e.op == AluOp.Add else -1
        return _tidy({k: a.get(k, 0) + s * b.get(k, 0) for k in {**a, **b}}, extent)
    if e.op == AluOp.Mul:
        if set(a) <= {None}:
            a, b = b, a
        return _tidy({k: v * b.get(None, 0) for k, v in a.items()}, extent) if set(b) <= {None} else None
    d = b.get(None, 0)
    if set(b) - {None} or d <= 0 or e.src[0].min < 0:
        return None
    q = _divide(a, d, extent)
    if q is None or e.op == AluOp.Idiv:
        return q
    return _tidy({k: a.get(k, 0) - d * q.get(k, 0) for k in {**a, **q}}, extent)


# ---- chains ----------------------------------------------------------------------------------------------------------

@dataclass
class Stage:
    """One Kernel of a chain: "reduce" folds a row, "map" gives a value per element, "scalar" one per row.  `refs[gid]` is
    ("in", k) for the chain's k-th input or ("stage", j) for an earlier stage's result."""

    kernel: Kernel
    kind: str
    refs: List[Tuple[str, int]]
    exp: AluExp
    epilogue: Optional[AluExp] = None
    full: set = field(default_factory=set)     # id(load node) read at the element's own position
    scalar: set = field(default_factory=set)   # id(load node) read at the row's own position


@dataclass
class RowChain(Composite):
    R: int
    C: int
    stages: List[Stage]
    inputs: List[int]        # caller's buffer ids, in parameter order
    outputs: List[int]       # stages whose results are stored, in parameter order
    name: str = "rows"

    def key(self) -> tuple:
        return ("rows", self.R, self.C, tuple((s.kernel.key(), tuple(s.refs)) for s in self.stages), tuple(self.outputs))

    def output_bytes(self) -> List[int]:
        return [self.stages[j].kernel.bytes for j in self.outputs]

    def generate(self, numerics: str) -> KernelSource:
        return gen_rows(self, numerics)

    def extents(self) -> List[int]:
        return [self.R, self.C]

    def label(self):
        return "Rows", [("kernels", str(len(self.stages))), ("size", str(self.R * self.C))]


def lower_stage(kernel: Kernel, R: int, C: int) -> Optional[Stage]:
    """`kernel` as a stage of a chain over [R, C], its index expressions in terms of the row (gidx) and the position in
    the row (ridx); None when it does not have that shape."""
    re = kernel.reduction
    extent = {"gidx": R, "ridx": C}
    row, col = AluExp.special(DType.Int32, "gidx", R), AluExp.special(DType.Int32, "ridx", C)
    if re is not None:
        if kernel.size != R or re.size != C:
            return None
        kind, sub = "reduce", {"gidx": row, "ridx": col}
    elif kernel.size == R * C and C > 1:
        kind, sub = "map", {"gidx": AluExp.add(AluExp.mul(row, AluExp.i32(C)), col)}
    elif kernel.size == R:
        kind, sub = "scalar", {"gidx": row}
    else:
        return None
    exp = kernel.exp
    if re is not None and exp.dtype != re.dtype:
        exp = AluExp.cast(re.dtype, exp)

    def lower(e: AluExp, s) -> AluExp:
        return e.substitute(s).rewriteGlobalViews().reduceExactIndex().simplify()

    st = Stage(kernel, kind, [], lower(exp, sub), lower(re.epilogue, {"gidx": row}) if re is not None else None)
    for e in (st.exp, st.epilogue):
        if e is None:
            continue
        for n in e.collect(lambda x: x.op == AluOp.GlobalIndex):
            f = index_form(n.src[0], extent)
            if f == _tidy({("gidx", 1): C, ("ridx", 1): 1}, extent) and e is st.exp and n.arg[1] == R * C:
                st.full.add(id(n))
            elif f == _tidy({("gidx", 1): 1}, extent) and n.arg[1] == R:
                st.scalar.add(id(n))
    return st


def _loads(st: Stage) -> List[AluExp]:
    return [n for e in (st.exp, st.epilogue) if e is not None for n in e.collect(lambda x: x.op == AluOp.GlobalIndex)]


def collect_chain(units: Sequence[tuple], first: int, wanted) -> Optional[Tuple[RowChain, int]]:
    """The longest chain that starts with dispatch `first` of `units` ((kernel, input ids, output id) each, kernel None for
    anything else) and takes the dispatches that follow it without a gap: (chain, number of dispatches), or None below two.
    `wanted(output id, last)` says whether anything past dispatch `last` still reads that result."""
    def shape_of():
        k = units[first][0]
        if k is None:
            return None
        if k.reduction is not None:
            return k.size, k.reduction.size
        nxt = units[first + 1] if first + 1 < len(units) else None  # a map first: the reduction behind it gives the rows
        if nxt is None or nxt[0] is None or nxt[0].reduction is None or units[first][2] not in nxt[1]:
            return None
        R, C = nxt[0].size, nxt[0].reduction.size
        return (R, C) if k.size == R * C else None

    shape = shape_of()
    if shape is None:
        return None
    R, C = shape
    if R < 1 or C < 2 or R * C >= (1 << 31):
        return None
    stages: List[Stage] = []
    inputs: List[int] = []
    made: Dict[int, int] = {}
    read_full = set()  # buffers the chain holds as rows: a new stage has to share one of them
    ids: List[int] = []
    at = first
    while at < len(units):
        k, ins, out = units[at]
        if k is None or k.size == 0:
            break
        st = lower_stage(k, R, C)
        if st is None or (k.reduction is not None and k.reduction.dtype in (DType.Float64,)) or k.dtype == DType.Float64:
            break
        ok, touched, fulls = True, set(), set()
        for n in _loads(st):
            buf = ins[n.arg[0]]
            touched.add(buf)
            if n.dtype == DType.Float64:
                ok = False
            if buf in made:  # an earlier stage's result: only in the place where this lane holds it
                kind = stages[made[buf]].kind
                ok = ok and (id(n) in st.full if kind == "map" else id(n) in st.scalar)
            elif id(n) in st.full:
                fulls.add(buf)
        if not ok or (stages and not (touched & (set(made) | read_full))):
            break
        if not stages and k.reduction is not None and not fulls:
            break  # nothing runs along the row: not a row reduction
        for buf in ins:
            if buf in made:
                st.refs.append(("stage", made[buf]))
            else:
                if buf not in inputs:
                    inputs.append(buf)
                st.refs.append(("in", inputs.index(buf)))
        read_full |= fulls
        made[out] = len(stages)
        stages.append(st)
        ids.append(out)
        at += 1
        if len(inputs) > 24 or len(stages) >= 16:
            break
    # shorten until it ends where the registers suffice and at least two dispatches become one
    while len(stages) >= 2:
        last = first + len(stages) - 1
        outs = [j for j, o in enumerate(ids[:len(stages)]) if wanted(o, last)]
        used = [i for i, b in enumerate(inputs) if any(("in", i) == r for s in stages for r in s.refs)]
        chain = RowChain(R, C, [Stage(s.kernel, s.kind, [("in", used.index(r[1])) if r[0] == "in" else r for r in s.refs], s.exp, s.epilogue,
                                      s.full, s.scalar) for s in stages], [inputs[i] for i in used], outs)
        if outs and any(s.kind == "reduce" for s in stages) and plan_rows(chain) is not None:
            return chain, len(stages)
        stages.pop()
    return None


# ---- launch shape and source -----------------------------------------------------------------------------------------

def _types(chain: RowChain) -> List[Optional[DType]]:
    used: List[Optional[DType]] = [None] * len(chain.inputs)
    for st in chain.stages:
        for n in _loads(st):
            kind, k = st.refs[n.arg[0]]
            if kind == "in":
                used[k] = n.dtype
    return used


def _rows_held(chain: RowChain) -> Tuple[Dict[int, int], Dict[int, int]]:
    """(input -> last stage that reads it as a row, map stage -> last stage that reads it)."""
    rows: Dict[int, int] = {}
    maps: Dict[int, int] = {}
    for j, st in enumerate(chain.stages):
        if st.kind == "map":
            maps.setdefault(j, j)
        for n in _loads(st):
            kind, k = st.refs[n.arg[0]]
            if kind == "in" and id(n) in st.full:
                rows[k] = j
            elif kind == "stage" and chain.stages[k].kind == "map":
                maps[k] = j
    return rows, maps


def plan_rows(chain: RowChain) -> Optional[dict]:
    """Vector width, lanes per row and iterations; None when a row does not fit the registers of one workgroup."""
    types = _types(chain)
    rows, maps = _rows_held(chain)
    sizes = [byteWidth(types[k]) for k in rows] + [byteWidth(chain.stages[j].kernel.dtype) for j in maps]
    V = 16 // min(sizes)
    while chain.C % V:
        V //= 2
    groups = chain.C // V
    # About 16 float32 (32 float16) elements per lane: enough loads in flight per lane to cover HBM latency with a
    # handful of waves per SIMD, few enough that the arrays do not cut into those waves; and at least 64 bytes of a row
    # per load, or narrow rows are fetched line by line several times over.  With few rows the lanes are
    # spread wider, down to one group each, since the launch then waits on latency and not on bandwidth.
    per_lane = max(16, 64 // min(sizes))
    T = 4
    while T < MAX_LANES and T < groups and (T * per_lane < chain.C or T * V * min(sizes) < 64 or chain.R * T < tuner.CU_COUNT * 256):
        T *= 2
    iters = -(-groups // T)
    # registers the rows and intermediates take between two stages (inside one, what dies makes room for what is born)
    held = [(byteWidth(types[k]), -1, last) for k, last in rows.items()] + \
           [(byteWidth(chain.stages[m].kernel.dtype), m, last) for m, last in maps.items()]
    peak = max(sum(b for b, born, last in held if born < j <= last) for j in range(len(chain.stages) + 1))
    if peak * iters * V > (88 * 4 if T == MAX_LANES else 160 * 4):
        return None
    block = max(T, 64 if chain.R * T <= tuner.CU_COUNT * 256 else 256)
    full = sum(1 for i in range(iters) if (i + 1) * T * V <= chain.C)
    return dict(V=V, T=T, iters=iters, full=full, block=block, grid=-(-chain.R * T // block))


def _fold_text(op: AluOp, dtype: DType, halves: bool) -> str:
    """One step of a fold.  float32 maxima and minima are the instruction that lets a NaN through (`jh_row_max`); where a
    chain has float16 values this compiler's instruction selection can fail on it, and the select around `fmax` stays."""
    if dtype == DType.Float32 and op in (AluOp.Max, AluOp.Min) and not halves:
        return f"jh_row_{'max' if op == AluOp.Max else 'min'}(a, b)"
    return _reduce_text(op, dtype)


@dataclass
class RowText:
    """A chain as source text: `machinery` in front of the kernel, `loads` of the rows and `stages` inside it.  They use the names t
    (lane of the row), gidx (row), live (whether it is stored), at (its first element) and put (its first element in the
    outputs); inputs are in_name{i}, outputs out{stage}."""
    machinery: str
    loads: str
    stages: str
    params: List[str]
    need: Dict[int, int]
    halves: bool


def row_text(chain: RowChain, p: dict, numerics: str, in_name: str = "in", local: Optional[int] = None) -> RowText:
    """The chain as text under plan `p` (vector width V, lanes T, iterations).  Input `local`, read as rows only, is no
    parameter: its row starts at the pointer `jh_row`."""
    V, T = p["V"], p["T"]
    types = _types(chain)
    rows, _ = _rows_held(chain)
    params = [f"const {STORAGE_CTYPE[d or DType.Float32]}* __restrict__ {in_name}{k}" for k, d in enumerate(types) if k != local]
    params += [f"{STORAGE_CTYPE[chain.stages[j].kernel.dtype]}* __restrict__ out{j}" for j in chain.outputs]
    halves = any(d == DType.Float16 for d in types) or any(
        e is not None and e.collect(lambda n: n.dtype == DType.Float16) for s in chain.stages for e in (s.exp, s.epilogue))
    loop = ["#pragma unroll", "  for (int i = 0; i < JH_ITER; ++i) {", "    const int c0 = (i * JH_T + t) * JH_V;", "    if (i < JH_FULL || c0 < JH_WIDTH) {"]
    end = ["    }", "  }"]
    loads: List[str] = []
    for k in rows:
        ct = STORAGE_CTYPE[types[k]]
        loads.append(f"  jh_pack<{ct}, JH_V> x{k}[JH_ITER];")
    if rows:
        loads += loop
        for k in rows:
            ct = STORAGE_CTYPE[types[k]]
            # rows that this launch reads once and that are many: past the caches (see jh_vload_nt)
            kind = "jh_vload_nt" if chain.R * chain.C >= (1 << 22) else "jh_vload"
            base = f"{in_name}{k} + at" if k != local else "jh_row"
            loads.append(f"      x{k}[i] = {kind}<{ct}, JH_V>({base} + c0);")
        loads += end
    text: List[str] = []
    folds: Dict[tuple, str] = {}   # a fold that an earlier stage has done already
    n_folds = 0
    for j, st in enumerate(chain.stages):
        args = [f"{in_name}{k}" if kind == "in" else "nullptr" for kind, k in st.refs]
        over: Dict[int, str] = {}
        for n in _loads(st):
            kind, k = st.refs[n.arg[0]]
            if kind == "stage":
                over[id(n)] = f"y{k}[i].v[lane]" if chain.stages[k].kind == "map" else f"y{k}"
            elif id(n) in st.full:
                over[id(n)] = f"x{k}[i].v[lane]"
        out_t = STORAGE_CTYPE[st.kernel.dtype]
        stored = j in chain.outputs
        if st.kind in ("map", "reduce"):
            classes = {i: c for i, c in tuner.classify_loads(st.exp, "ridx", V).items() if i not in over}
            body = _Body(st.exp, args, IDENT, "ridx", "c0", V, classes, numerics, "      ", f"{j}_")
            hoisted, lane_loads = body.hoisted()
            body.indent = "        "
            lane_loads = {**lane_loads, **over}
        if st.kind == "map":
            lane_body, value = body.lanes(lane_loads)
            text.append(f"  jh_pack<{out_t}, JH_V> y{j}[JH_ITER];")
            text += loop + [hoisted, "#pragma unroll", "      for (int lane = 0; lane < JH_V; ++lane) {", "        const int ridx = c0 + lane;", "        (void)ridx;",
                            lane_body, f"        y{j}[i].v[lane] = ({out_t})({value});", "      }"]
            if stored:
                text.append(f"      if (live) jh_vstore<{out_t}, JH_V>(out{j} + put + c0, y{j}[i]);")
            text += end
            continue
        if st.kind == "reduce":
            re = st.kernel.reduction
            acc_t = CTYPE[re.dtype]
            what = (st.exp, re.op, re.dtype, tuple(st.refs[n.arg[0]] for n in st.exp.collect(lambda x: x.op == AluOp.GlobalIndex)))
            if what not in folds:
                lane_body, value = _lane_accumulate(body, lane_loads, st.exp, re, acc_t, f"a{j}")
                value = value.replace("JH_REDUCE(", f"jh_op{j}(", 1) if value.startswith("JH_REDUCE(") else value
                text.append(f"  const auto jh_op{j} = [](const {acc_t} a, const {acc_t} b) {{ return ({acc_t})({_fold_text(re.op, re.dtype, halves)}); }};")
                text.append(f"  {acc_t} a{j} = {const_literal(re.dtype, re.identity)};")
                text += loop + [hoisted, "#pragma unroll", "      for (int lane = 0; lane < JH_V; ++lane) {", "        const int ridx = c0 + lane;", "        (void)ridx;",
                                lane_body, f"        a{j} = {value};", "      }"] + end
                text.append(f"  a{j} = jh_row_fold(a{j}, jh_op{j}, JH_SLOTS({n_folds}, {acc_t}));")
                folds[what] = f"a{j}"
                n_folds += 1
            exp, names = st.epilogue, {"gidx": "gidx", "acc": folds[what]}
        else:
            exp, names = st.exp, {"gidx": "gidx"}
        one = _Body(exp, args, names, "gidx", "gidx", 1, {}, numerics, "  ", f"e{j}_")
        scalar_body, value = one.lanes({i: t for i, t in over.items()})
        text += [scalar_body, f"  const {out_t} y{j} = ({out_t})({value});"]
        if stored:
            text.append(f"  if (live && t == 0) out{j}[gidx] = y{j};")
    machinery = fill(template("row_fold.hip.inc"), dict(C=chain.C, V=V, T=T, ITER=p["iters"], FULL=p["full"], REDUCTIONS=n_folds))
    need: Dict[int, int] = {}
    for st in chain.stages:
        for n in _loads(st):
            kind, k = st.refs[n.arg[0]]
            if kind == "in" and k != local:
                need[k] = max(need.get(k, 0), n.arg[1] * byteWidth(n.dtype))
    return RowText(machinery, "\n".join(loads), "\n".join(x for x in text if x), params, need, halves)


def gen_rows(chain: RowChain, numerics: str, name: str = "jh_rows") -> KernelSource:
    p = plan_rows(chain)
    r = row_text(chain, p, numerics)
    src = (SOURCE_OPTION + "-fno-slp-vectorize\n" if r.halves else "") + _prelude(numerics) + r.machinery + fill(template("rows.hip.inc"), dict(
        R=chain.R, BLOCK=p["block"], NAME=name, PARAMS=", ".join(r.params), LOADS=r.loads, STAGES=r.stages))
    step = LaunchStep(name, (p["grid"], 1, 1), (p["block"], 1, 1), 0, [("in", k) for k in range(len(_types(chain)))] + [("out", i) for i in range(len(chain.outputs))])
    return KernelSource([src], [step], [], "rows", r.need, dict(p, R=chain.R, C=chain.C, kernels=len(chain.stages)))
