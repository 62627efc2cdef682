"""Contractions whose operands are read through windows, pads, strides or flips: those operands are laid out as matrices first.

A convolution reaches a backend as one reduce Kernel over a view of its image (src/frontend/convolution.ts), in which every
element of a patch is found by its own index expression.  The general product templates evaluate that expression for every
element of every tile, with one load behind it: 50 to 100 ns per element of k, whatever else the tile does, and the reductions
by rows or columns for every product.  Here the elements are gathered once, by all CUs (`layout.hip.inc`), into matrices whose
rows run along k, padded by zeros to whole groups, and the product reads plain operands, for which it has direct loads and
slices of k.  microseconds, with the layouts: float16 2 x [172, 42, 42] by 56 x 3 x 3, stride 2, 123 -> 12, [256, 45, 45] by 24 x 5 x 5 470 ->
41; float32 cotangents of filters 9 x [43, 37, 37] by 54 x 5 x 5 1484 -> 90, 4 x [192, 50, 50] by 192 x 3 x 3 616 -> 120; of images
5 x [40, 41, 41] by 213 x 5 x 5, stride 2, 549 -> 140.  Over 300 convolutions and cotangents drawn (1 to 32 images of 7 to 56, 16 to 256
channels, windows of 1, 3 and 5, strides of 1 and 2, both types) 2.16 times as fast in the mean.
"""

from __future__ import annotations

from typing import List, Optional, Sequence, Tuple

from . import tuner
from .alu import AluExp, AluOp, AluVar, DType, Kernel, Reduction, byteWidth
from .codegen import STORAGE_CTYPE, HipExpCodegen, strip_parens
from .composite import Composite
from .gemm import few_plan
from .kernelgen import KernelSource, LaunchStep, _prelude, fill, generate, template
from .shape import ShapeTracker, prod, unravelAlu

PACK_BYTES = 1 << 30  # of both matrices


class Layout:
    """Elements of a view as a matrix of `rows` (its axes but the last) along k, with zeros behind its last axis up to `K`."""

    def __init__(self, dtype: DType, st, K: int):
        self.dtype, self.st, self.rows, self.K = dtype, st, list(st.shape[:-1]), K

    @property
    def bytes(self) -> int:
        return prod(self.rows) * self.K * byteWidth(self.dtype)

    def place(self):
        """(mask or None, load) of element (row, k), or None where its expression has another form or is not a 32-bit number (a plain
        operand may lie anywhere in its buffer: the templates find its rows by 64-bit strides)."""
        row = AluExp.special(DType.Int32, "row", max(prod(self.rows), 1))
        at = [u.simplify() for u in unravelAlu(self.rows, row)] + [AluExp.special(DType.Int32, "k", self.st.shape[-1])]
        e = AluExp.globalView(self.dtype, 0, self.st, at).rewriteGlobalViews().reduceExactIndex().simplify()
        cond = None
        if e.op == AluOp.Where and e.src[2].op == AluOp.Const and float(e.src[2].arg) == 0.0:
            cond, e = e.src[0], e.src[1]
        return (cond, e) if e.op == AluOp.GlobalIndex and e.src[0].min >= -(1 << 31) and e.src[0].max < 1 << 31 else None


class Layouts(Composite):
    """The operands of a contraction, laid out by one launch."""

    def __init__(self, layouts: Sequence[Layout], inputs: Sequence[int]):
        self.layouts, self.inputs = list(layouts), list(inputs)

    def key(self) -> tuple:
        return ("layouts", tuple((x.dtype, x.st.key(), x.K) for x in self.layouts))

    def output_bytes(self) -> List[int]:
        return [x.bytes for x in self.layouts]

    def extents(self) -> List[int]:
        return [sum(x.bytes // byteWidth(x.dtype) for x in self.layouts)]

    def label(self):
        return "Layouts", [("operands", str(len(self.layouts))), ("size", str(self.extents()[0]))]

    def generate(self, numerics: str) -> KernelSource:
        bodies, params, args, calls, need, first = [], [], [], [], {}, 0
        for i, x in enumerate(self.layouts):
            cond, load = x.place()
            cg = HipExpCodegen(["in"], {"row": "row", "k": "k"}, "  ", prefix="p", numerics=numerics)
            cg.countReferences(load.src[0])
            if cond is not None:
                cg.countReferences(cond)
            index = strip_parens(cg.run(load.src[0]))
            inside = " && ".join(([f"k < {x.st.shape[-1]}"] if x.K != x.st.shape[-1] else []) + ([f"({strip_parens(cg.run(cond))})"] if cond is not None else [])) or "true"
            rows, elem = prod(x.rows), STORAGE_CTYPE[x.dtype]
            V = 16 // byteWidth(x.dtype)
            groups = x.K // V
            # parts of a row so that as few of 256 lanes as can be have nothing to do
            parts = max(range(-(-groups // 256), -(-groups // 256) + 4), key=lambda n: (256 // -(-groups // n) * -(-groups // n)) * groups / (n * -(-groups // n)))
            lanes = -(-groups // parts)
            together = 256 // lanes
            per = max(1, min(LAYOUT_ROWS, rows // together * parts // LAYOUT_BLOCKS))
            bodies.append(fill(template("layout.hip.inc"), dict(SPACE=f"jh_{i}", ROWS=rows, K=x.K, V=V, PER=per, LANES=lanes, PARTS=parts, ELEM=elem,
                                                                LINES="\n".join(cg.take_lines()), INSIDE=inside, INDEX=index)))
            params += [f"const {elem}* __restrict__ in{i}", f"{elem}* __restrict__ out{i}"]
            args += [("in", i), ("out", i)]
            blocks = -(-rows // (together * per)) * parts
            calls.append(f"  {'else ' if i else ''}{f'if (block < {first + blocks}) ' if i + 1 < len(self.layouts) else ''}jh_{i}::jh_layout(in{i}, out{i}, block{f' - {first}' if first else ''});")
            need[i] = load.arg[1] * byteWidth(x.dtype)
            first += blocks
        src = _prelude(numerics) + "".join(bodies) + (
            f"extern \"C\" __global__ __launch_bounds__(256) void jh_layouts({', '.join(params)}) {{\n  const int block = (int)blockIdx.x;\n" + "\n".join(calls) + "\n}\n")
        return KernelSource([src], [LaunchStep("jh_layouts", (first, 1, 1), (256, 1, 1), 0, args)], [], "layouts", need, dict(parts=len(self.layouts), grid=first))


LAYOUT_ROWS = 16      # of a lane
LAYOUT_BLOCKS = 2048  # workgroups below which a lane takes fewer rows


def _walk(shape, last=None):
    return [u.simplify() for u in unravelAlu(shape, AluVar.gidx)] + ([last] if last is not None else [])


class Packed:
    """`layouts`: (`Layout`, argument of the contraction that it reads, argument of `product` that it writes); `product` takes the
    contraction's arguments, those of the layouts in place of what nothing else reads or behind the others."""

    def __init__(self, layouts: List[Tuple[Layout, int, int]], product: Kernel):
        self.layouts, self.product = layouts, product
        self.options = {}  # that the product is prepared with, beside its own
        self.instead: Optional[Kernel] = None  # the contraction that would run otherwise


def _operands(kernel: Kernel):
    """Both GlobalViews of a sum of products over float16 or float32 views in their plain order, or None."""
    re = kernel.reduction
    if re is None or re.op != AluOp.Add or re.dtype != DType.Float32 or kernel.size == 0 or re.size == 0:
        return None
    root = tuner._strip_float_casts(kernel.exp)
    if root.op != AluOp.Mul:
        return None
    views = [tuner._strip_float_casts(s) for s in root.src]
    if any(v.op != AluOp.GlobalView for v in views) or views[0].dtype != views[1].dtype or views[0].dtype not in (DType.Float16, DType.Float32):
        return None
    shape = list(views[0].arg[1].shape)
    if list(views[1].arg[1].shape) != shape or len(shape) < 2 or shape[-1] != re.size or prod(shape[:-1]) != kernel.size:
        return None
    walk = _walk(shape[:-1], AluVar.ridx)
    if any(len(v.src) != len(walk) or any(x.simplify() is not y for x, y in zip(v.src, walk)) for v in views):
        return None
    return views, shape


def _plain(st) -> bool:
    """Whether the general templates read this view by vectors: one strided view, or one whose k axis comes in whole runs."""
    f = tuner._flatten_k_split(st)
    return f is not None and f[0].mask is None and min(f[0].strides) >= 0 and (not f[1] or (f[0].strides[-1] == 1 and f[1] % 64 == 0 and f[2] % 8 == 0 and f[2] > 0))


def _grouped(st, vec: int) -> bool:
    """Whether the templates with direct loads read the view as it stands: rows along k that start on the 16-byte grid."""
    v = st.views[0]
    return len(st.views) == 1 and v.strides[-1] == 1 and not any(x % vec for x in (v.offset, *v.strides[:-1]))


def pack(kernel: Kernel) -> Optional[Packed]:
    """The contraction with its gathered operands laid out, or None where it has none (or is no contraction)."""
    found = _packed(kernel, 4)
    if found is None or kernel.reduction.size < 512 or found.layouts[0][0].dtype != DType.Float32:
        return found
    # one float32 product, and not one for every image: up to eight slices of the axis have to be whole 16-byte groups
    return found if tuner.match_gemm(found.product)["batch"] else _packed(kernel, 32)


def _packed(kernel: Kernel, group32: int) -> Optional[Packed]:
    found = _operands(kernel)
    if found is None:
        return None
    views, shape = found
    gathered = [not _plain(v.arg[1]) for v in views]
    if not any(gathered):
        return None
    half = views[0].dtype == DType.Float16
    K = shape[-1]
    # whole 16-byte groups, or slabs and slices of a long axis that are whole slabs
    group = group32 if not half else 64 if K < 2048 else 128 if K < 4096 else 256
    K_pad = -(-K // group) * group
    layouts, replaced, nargs, total = [], {}, kernel.nargs, 0
    reads = [n.arg[0] for e in (kernel.exp, kernel.reduction.epilogue) for n in e.collect(lambda n: n.op in (AluOp.GlobalIndex, AluOp.GlobalView))]
    for v, g in zip(views, gathered):
        if id(v) in replaced or (not g and K_pad == K and _grouped(v.arg[1], 8 if half else 4)):
            continue
        gid, st = v.arg
        outer = st.views[-1]
        kept = [d for d in range(len(shape) - 1) if shape[d] > 1 and (outer.strides[d] != 0 or (outer.mask is not None and tuple(outer.mask[d]) != (0, shape[d])))]
        rows = [shape[d] for d in kept]
        total += prod(rows) * K_pad * byteWidth(v.dtype)
        if total > PACK_BYTES:
            return None
        layout = Layout(v.dtype, st.shrink([(0, n if d in kept or d == len(shape) - 1 else 1) for d, n in enumerate(shape)]).reshape(rows + [K]).simplify(), K_pad)
        if layout.place() is None:
            return None
        to = gid if reads.count(gid) == 1 else nargs
        nargs += to == nargs
        layouts.append((layout, gid, to))
        dense = ShapeTracker.fromShape(rows + [K_pad]).reshape([n if d in kept else 1 for d, n in enumerate(shape[:-1])] + [K_pad]).expand(shape[:-1] + [K_pad])
        replaced[id(v)] = AluExp.globalView(v.dtype, to, dense, _walk(shape[:-1], AluVar.ridx))
    re = kernel.reduction
    product = Kernel(nargs, kernel.size, kernel.exp.rewrite(lambda n: replaced.get(id(n))), Reduction(re.dtype, re.op, K_pad, re.epilogue))
    return Packed(layouts, product) if tuner.match_gemm(product) is not None else None


def _us_gathered(kernel: Kernel) -> float:
    """Estimated time of the contraction as it stands, in microseconds; 0 where it has a kernel of its own that this does not replace.

    A fit to 180 Kernels of drawn convolutions.  The templates' time is their walk over k, by how many operands have vector loads,
    and goes on with the workgroups of a CU, which hide each other's loads in part; that of the reductions by rows and columns is the
    products, 0.3 to 1.7 million a microsecond where windows are walked and eight where both operands come in vectors.  An image whose windows' rows come
    in whole groups of four or eight has vector loads too, for a walk of 6 to 10 ns an element of k in float16 and 37 in float32 (94 convolutions with windows of 4 to 16: float16 [6, 20, 28, 28] to 461, 4 x 4, stride 4, 6.1 us, laid
    out 8.2; 171 to 299 channels of 60 x 60, 4 x 4, 20.6 and 35.9; [2, 388, 40, 40] to 65, stride 2, 11.7 and 29.0)."""
    t = tuner.tuneHip(kernel)
    K = kernel.reduction.size
    if t.klass != "gemm":
        loads = tuner._load_nodes(t.exp)
        half = byteWidth(loads[0].dtype) == 2
        vectors = all(str((t.vector_loads or {}).get(id(n), "")).startswith("vector") for n in loads)
        runs = all(w.mask is None for v in _operands(kernel)[0] for w in v.arg[1].views) and all(v.arg[1].views[0].strides[-1] == 1 for v in _operands(kernel)[0])
        rate = 8e6 if vectors else 4e6 if K <= 64 else 2.5e6 if runs or K <= 128 else 0.65e6 if half else 1.0e6  # products a microsecond
        return 3.0 + kernel.size * K / rate
    g = t.gemm
    if not (g.get("a_gather") or g.get("b_gather")):
        return 0.0
    info = generate(kernel).info
    if info.get("conv") or info.get("few") or info.get("wgrad"):
        return 0.0
    half = g["dtype"] == DType.Float16
    split = int(info.get("splitk", 1))
    rounds = max(1.0, info["tiles"] * split / tuner.CU_COUNT) ** 0.5  # workgroups that share a CU hide each other's loads
    single = sum(x == "element" for x in info.get("gather", {}).values())  # operands without vector loads
    per_k = (0.045 + 0.0275 * single + (0.03 if g.get("a_loose") or g.get("b_loose") else 0.0)) if half else 0.05 + 0.01 * single
    fold = 2.0 if split > 1 else 0.0
    us = max(3.0, per_k * K / split * rounds - 1.0) + fold
    gather = info.get("gather", {})
    if gather.get("a") == "none" and gather.get("b") in ("k4", "k8"):
        area = info["BM"] * info["BN"] / 4096
        us = min(us, (4.7 + (0.0063 + 0.0036 * (area - 1)) * K / split * rounds if half else 3.4 + 0.0373 * K / split * rounds) + fold)
    return us


def _us_packed(packed: Packed, sums_stay: bool) -> float:
    """Estimated time of the layouts' launch and the product, in microseconds, fitted to the same Kernels: two launches, 0.5 to 0.6
    million elements laid out a microsecond (1.2 TB/s in float16, 2 in float32), and the product's walk over k.  `sums_stay`: a
    float32 contraction that a reduction by rows or columns computes stays with one, whose many short sums lose less than
    the one of a matrix instruction's accumulator (relative error against 64 bits 1.4e-7 and 5.5e-7 over k = 30250).  Vectors of four make
    a lane's sum four times as long, so a row gets up to four times as many lanes (9 x [28, 18, 18] by 25 x 5 x 5, stride 2, 1.32e-7
    as it stands, 1.32e-7 laid out, 0.96e-7 with the lanes; 26, 10.4 and 11 us), and one that has them all and a longer axis is left as it is.

    Other products of 2 to 31 rows or columns, which go to the reductions by rows as a rule, go to the matrix cores where that is estimated to
    be faster: the reductions read the other operand once for each of those rows.  float16 16 x [64, 38, 38] to 24 channels, 3 x 3,
    108 us there and 32 in tiles, 22 x [18, 26, 26] to 28, stride 2, 96 and 27, 25 x [64, 17, 17] to 27, stride 2, 84 and 33; but 3 x [59, 11, 11] to
    23 8.9 and 9.9."""
    product = packed.product
    t, K = tuner.tuneHip(product), product.reduction.size
    half = packed.layouts[0][0].dtype == DType.Float16
    us = 7.0 + sum(x.bytes // byteWidth(x.dtype) for x, _gid, _to in packed.layouts) / (6e5 if half else 5e5)
    if sums_stay:
        packed.options = dict(allow_gemm=False)
        s = tuner.tuneHip(product, allow_gemm=False)
        if s.klass != "reduce_row":
            return float("inf")
        lanes = s.params["T"]
        if lanes < 256 and K >= 8 * lanes:
            lanes = packed.options["row_lanes"] = min(256, 4 * lanes)
        if K > 32 * lanes:
            return float("inf")
        return us + product.size * K / 3e6
    sums = product.size * K / (5e6 if half else 3e6) if t.klass != "gemm" else None
    if sums is not None:
        t = tuner.tuneHip(product, thin_rows=True)
        if t.klass != "gemm":
            return us + sums
    g, side = t.gemm, 128 if half else 64
    if few_plan(t) is not None:
        walk = K * (0.005 if half else 0.008)
    else:
        tiles = -(-g["M"] // side) * -(-g["N"] // side) * prod([b[0] for b in g["batch"]])
        slices = max(1, min(8, tuner.CU_COUNT // tiles, K // 512)) if half or not g["batch"] else 1
        walk = K / slices * (0.0065 if half else 0.0165) * max(1.0, tiles / tuner.CU_COUNT) + (3.0 if slices > 1 else 0.0)
    if sums is not None and sums <= walk:
        return us + sums
    packed.options = dict(thin_rows=True) if sums is not None else {}
    return us + walk


def packs(kernel: Kernel, spared: float = 0.0, instead: Optional[Kernel] = None) -> Optional[Packed]:
    """As `pack`, where that is estimated to be the faster side by a tenth; `instead`: the contraction that would run otherwise, if
    that is another one, and `spared`: microseconds of a launch that comes with it.

    The tenth keeps what is about the same where it was.  Convolutions with a patch template or bands of their own stay with them
    (8 x [192, 45, 45] by 128 x 3 x 3 float16: 31 us there, 74 laid out), and so do short k axes (float16 [59, 45, 45] by 36 x 1 x 1,
    stride 2: 6.0 and 9.0) and many tiles behind vector loads (float32 19 x [192, 25, 25] by 60 x 3 x 3 52 and 75)."""
    found = pack(kernel)
    if found is None:
        return None
    found.instead = instead = instead or kernel
    before = _us_gathered(instead)
    sums_stay = instead.reduction.size > 64 and found.layouts[0][0].dtype == DType.Float32 and tuner.tuneHip(instead).klass != "gemm"
    return found if before and _us_packed(found, sums_stay) < 0.9 * (before + spared) else None
