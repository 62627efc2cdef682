"""How a jit program runs on the `hip` backend: its dispatches as one list of native launches.

A `JitProgram` (src/frontend/jit.ts:111-162) is a fixed list of allocations, dispatches and releases.  `Schedule` prepares
it once: neighbouring Kernels over the same rows become one launch (`rowchain.py`), every intermediate gets a place in one
workspace that is taken from the backend's pool for the call (places are used again as soon as their buffer is dead), and
the launches of all steps go to the stream in one native call (`jh_launch_list`).  Per call the host looks up the input
slots, allocates the output slots and makes that call; dispatching step by step cost 6 us of host time per launch, which
is more than most launches of a small program take on the device.
"""

from __future__ import annotations

import ctypes
import threading
from typing import Any, Dict, List, Optional, Sequence, Tuple

from . import tracing
from .alu import AluExp, AluOp, AluVar, DType, Kernel, Reduction, byteWidth
from .attentioncache import join_cache
from .composite import MAPS_MOST, WEIGHTS_MOST, Maps, Weights, joins_maps
from .errors import DeviceMemoryError, SlotError
from .gemm import is_direct_product, is_sliced_product
from .kernelgen import generate
from .patches import Layouts, Packed, packs
from .routine import Routine, Routines
from .rowchain import RowChain, _tidy, collect_chain, index_form
from .rowproduct import join_behind, join_rows
from .runtime import LAUNCH_ARGS, LaunchRef, LaunchStepC, check
from .shape import prod, unravelAlu
from .tuner import match_gemm
from .wgradgen import is_filter_cotangent


class Unit:
    """One dispatch of the schedule: an executable (of `source`, prepared with `options`), the buffer ids it reads and the ones
    it writes."""

    def __init__(self, source, inputs: Sequence[int], outputs: Sequence[int], **options):
        self.source, self.inputs, self.outputs, self.options = source, list(inputs), list(outputs), options
        self.exe = None
        self.early: Optional[int] = None  # the buffer that holds what this unit's first step would make (see `Weights`)
        self.sizes: Dict[int, int] = {}   # bytes of the outputs that are buffers of the schedule and not of the program


_LONG_OPS = (AluOp.Erf, AluOp.Erfc, AluOp.Sin, AluOp.Cos, AluOp.Asin, AluOp.Atan)  # dozens of instructions each


def join_epilogue(product: Kernel, buffer: int, following: Kernel, inputs: Sequence[int]) -> Optional[Kernel]:
    """The contraction `product`, which writes `buffer`, with the elementwise `following` (reading `inputs`) as the rest of
    its epilogue, or None.  `following` has to read nothing but `buffer`, each element at its own position.  The product's
    value keeps the type it was stored in, so results keep their bits.

    A value that is used more than once ends the front-end's fusion (src/frontend/jit.ts:572-789): gelu behind a linear
    layer was a launch of its own that read and wrote the whole activation again (float16 [8192, 3072]: 24 us).

    Where the epilogue is long it stays a launch of its own behind float16 tiles: a tile's few threads have it in front of
    them when the product is done, and the product is quick (512 x 512 x 512, x erfc(x): 13.5 us joined, 8.7 in two
    launches; sine 12.8 and 8.6; arc tangent 10.5 and 8.4; 8192 x 3072 x 768 78 and 73).  exp and log are short enough
    (tanh, mish), float32 products long enough (1024 x 1024 x 1024: 35.4 and 33.8, 8000 x 1000 x 100 43 and 47), and a
    short k axis or the kernel for few rows leaves room (2048 x 2048 x 64 12.7 and 15.5, 8 x 3072 x 768 5.7 and 8.7)."""
    re = product.reduction
    if re is None or following.reduction is not None or following.size != product.size or product.size == 0:
        return None
    gidx = AluExp.special(DType.Int32, "gidx", product.size)
    exp = following.exp.substitute({"gidx": gidx}).rewriteGlobalViews().reduceExactIndex().simplify()
    loads = exp.collect(lambda n: n.op == AluOp.GlobalIndex)
    own = _tidy({("gidx", 1): 1}, {"gidx": product.size})
    if not loads or any(inputs[n.arg[0]] != buffer or n.dtype != re.epilogue.dtype or index_form(n.src[0], {"gidx": product.size}) != own for n in loads):
        return None
    g = match_gemm(product)
    if g is None:
        return None
    if g["dtype"] == DType.Float16 and g["K"] >= 256 and exp.collect(lambda n: n.op in _LONG_OPS):
        plan = generate(product)
        if plan.klass.startswith("gemm") and not plan.info.get("few"):
            return None
    exp = exp.rewrite(lambda n: re.epilogue if n.op == AluOp.GlobalIndex else None)
    return Kernel(product.nargs, product.size, product.exp_raw, Reduction(re.dtype, re.op, re.size, exp))


def join_transposed(product: Kernel, buffer: int, following: Kernel, inputs: Sequence[int], layouts: bool) -> Tuple[Optional[Kernel], Optional[Packed]]:
    """The filter cotangent `product`, which writes `buffer`, with its outputs in the order in which the elementwise `following`
    (reading `inputs`) reads them, and that Kernel as the rest of its epilogue, where a kernel of its own takes it then or, with
    `layouts`, its operands are laid out (which comes with it); or None twice.

    The transpose rule of a convolution leaves the filter's cotangent with its channels exchanged, and puts them right by a
    copy ([64, 64, 3, 3]: a launch of 4.7 us; the product's last launch writes one order as fast as the other)."""
    re = product.reduction
    if re is None or following.reduction is not None or following.size != product.size or product.size == 0:
        return None, None
    reads = following.exp.collect(lambda n: n.op == AluOp.GlobalView)
    if not reads or any(inputs[n.arg[0]] != buffer or n.dtype != re.epilogue.dtype or n.arg[1] is not reads[0].arg[1] for n in reads):
        return None, None
    inside = set(id(n) for r in reads for s in r.src for n in s.collect(lambda n: n.op == AluOp.Special))
    if following.exp.collect(lambda n: n.op == AluOp.GlobalIndex or (n.op == AluOp.Special and id(n) not in inside)) \
            or re.epilogue.collect(lambda n: n.op in (AluOp.GlobalIndex, AluOp.GlobalView) or (n.op == AluOp.Special and n.arg[0] == "gidx")):
        return None, None
    views = product.exp.collect(lambda n: n.op == AluOp.GlobalView)
    st = reads[0].arg[1]
    shape = list(views[0].arg[1].shape[:-1]) if views else []
    if len(st.views) != 1 or st.views[0].mask is not None or st.views[0].offset != 0 or any(list(v.arg[1].shape[:-1]) != shape for v in views) \
            or sorted(st.shape) != sorted(shape) or prod(shape) != product.size:
        return None, None
    # axis k of the result is the product's axis with that stride (any that is left, of length one); the walks of both Kernels have to be the plain ones
    strides = [prod(shape[i + 1:]) for i in range(len(shape))]
    order: List[int] = []
    for n, s in zip(st.shape, st.views[0].strides):
        order.append(next((i for i, m in enumerate(shape) if i not in order and m == n and (n == 1 or strides[i] == s)), -1))
    if -1 in order:
        return None, None
    walk = lambda dims: [u.simplify() for u in unravelAlu(dims, AluVar.gidx)]  # noqa: E731
    if any(list(r.src) != walk(st.shape) for r in reads) or any(list(v.src) != walk(shape) + [AluVar.ridx] for v in views):
        return None, None
    exp = product.exp.rewrite(lambda n: AluExp.globalView(n.dtype, n.arg[0], n.arg[1].permute(order + [len(order)]), walk(st.shape) + [AluVar.ridx])
                              if n.op == AluOp.GlobalView else None)
    epilogue = following.exp.rewrite(lambda n: re.epilogue if n.op == AluOp.GlobalView else None)
    joined = Kernel(product.nargs, product.size, exp, Reduction(re.dtype, re.op, re.size, epilogue))
    if is_filter_cotangent(joined):
        return joined, None
    packed = packs(joined, COPY_US, product) if layouts else None
    return (joined, packed) if packed is not None else (None, None)


class _Dispatch:
    """One dispatch of a program: `kernel` or `routine`, and buffer ids."""

    def __init__(self, kernel, routine, inputs, output, outputs, packed=None):
        self.kernel, self.routine, self.inputs, self.output, self.outputs = kernel, routine, inputs, output, outputs
        self.packed = packed  # `kernel` with its operands laid out, where that is why it was made of two


COPY_US = 3.0  # the copy that `join_transposed` spares


def plan_dispatches(prog, layouts: bool = True) -> List[_Dispatch]:
    """The program's dispatches, elementwise Kernels behind a contraction joined to it where nothing else reads its result."""
    made = [_Dispatch(s.kernel, s.routine, s.inputs, s.output, s.outputs) for s in prog.steps if s.kind == "execute"]
    reads: Dict[int, int] = {}
    for d in made:
        for i in set(d.inputs):
            reads[i] = reads.get(i, 0) + 1
    kept = set(prog.outputs)
    rotated = before_rotations(made)
    out: List[_Dispatch] = []
    for d in made:
        before = out[-1] if out else None
        if before is not None and before.kernel is not None and d.kernel is not None and before.output in d.inputs \
                and reads[before.output] == 1 and before.output not in kept:
            joined, packed = join_epilogue(before.kernel, before.output, d.kernel, d.inputs), None
            if joined is None:
                joined, packed = join_transposed(before.kernel, before.output, d.kernel, d.inputs, layouts and d.output not in rotated)
            elif before.packed is not None:  # two joined for the sake of layouts: a third only if they stay
                packed = packs(joined, COPY_US, before.packed.instead)
                joined = joined if packed is not None else None
            if joined is not None:
                out[-1] = _Dispatch(joined, None, before.inputs, d.output, d.outputs, packed)
                continue
        out.append(d)
    return out


def adjacent_maps(steps: Sequence[_Dispatch], k: int, view) -> int:
    """How many dispatches from `k` on are elementwise Kernels that run side by side in one launch (see `Maps`), whose arguments
    a step of a launch list takes."""
    n, args, written = 0, 0, set()
    while n < MAPS_MOST and k + n < len(steps):
        d = steps[k + n]
        if d.kernel is None or not joins_maps(d.kernel) or written & set(d.inputs) or args + d.kernel.nargs + 1 > LAUNCH_ARGS:
            break
        if n and collect_chain(view, k + n, lambda o, last: True) is not None:
            break  # the first of Kernels over the same rows
        written.add(d.output)
        args += d.kernel.nargs + 1
        n += 1
    return n


def before_rotations(steps: Sequence[_Dispatch]) -> set:
    """The buffers that a JacobiEigh's matrix is made from.  Which sign and place an eigenvector gets from the rotations hangs on the
    last bits of the matrix, so the products in front keep the order of sums that their Kernels have one by one (an SVD of
    1024 x 128 returned negated vectors where its Gram matrix had another)."""
    found: set = set()
    for s in reversed(steps):
        written = [s.output] if s.routine is None else s.outputs
        if (s.routine is not None and s.routine.name == Routines.JacobiEigh) or any(o in found for o in written):
            found.update(s.inputs)
    return found


def plan_units(prog, layouts: bool = True) -> List[Unit]:
    """The program's dispatches with runs of Kernels over the same rows joined.  `layouts`: operands may be laid out as matrices."""
    steps = plan_dispatches(prog, layouts)
    rotated = before_rotations(steps)
    last_read: Dict[int, int] = {}
    for k, s in enumerate(steps):
        for i in s.inputs:
            last_read[i] = k
    kept = set(prog.outputs)
    view = [(s.kernel, s.inputs, s.output) if s.routine is None else (None, s.inputs, -1) for s in steps]
    units: List[Unit] = []
    fresh = max([prog.nargs - 1, *(i for s in prog.steps if s.kind == "malloc" for i in [s.output]), *(i for s in steps for i in s.inputs)]) + 1
    k = 0
    while k < len(steps):
        s = steps[k]
        found = collect_chain(view, k, lambda o, last: o in kept or last_read.get(o, -1) > last)
        if found is not None:
            chain, n = found
            before = steps[k - 1] if units and units[-1].outputs == [steps[k - 1].output] and isinstance(units[-1].source, Kernel) else None
            if before is not None and before.output not in kept and last_read.get(before.output, -1) < k + n:
                joined = join_behind(before.kernel, before.inputs, before.output, chain)
                if joined is not None:
                    units[-1] = Unit(joined, joined.inputs, [steps[k + j].output for j in chain.outputs])
                    k += n
                    continue
            units.append(Unit(chain, chain.inputs, [steps[k + j].output for j in chain.outputs]))
            k += n
            continue
        together = adjacent_maps(steps, k, view)
        if together > 1:
            run = steps[k:k + together]
            ids = [i for d in run for i in d.inputs]
            units.append(Unit(Maps([d.kernel for d in run], ids), ids, [d.output for d in run]))
            k += together
            continue
        cached = join_cache(units[-1].source, units[-1].outputs, s.routine, s.inputs) if s.routine is not None and units and isinstance(units[-1].source, Maps) else None
        if cached is not None:
            joined, at = cached
            maps, made = units[-1].source.kernels, units.pop().outputs
            rest = [i for i in range(len(maps)) if i not in at]
            before = steps[k - len(maps):k]
            if rest:
                ids = [i for r in rest for i in before[r].inputs]
                units.append(Unit(maps[rest[0]] if len(rest) == 1 else Maps([maps[r] for r in rest], ids), ids, [made[r] for r in rest]))
            units.append(Unit(joined, joined.inputs, s.outputs + [made[i] for i in at]))
            k += 1
            continue
        product = None
        if s.routine is None and units and isinstance(units[-1].source, RowChain) and len(units[-1].outputs) == 1:
            rows = units[-1].outputs[0]
            if rows in s.inputs and rows not in kept and last_read[rows] == k:
                product = join_rows(units[-1].source, rows, s.kernel, s.inputs)
        if product is not None:
            units[-1] = Unit(product, product.inputs, [s.output])
            k += 1
            continue
        if s.routine is not None:
            units.append(Unit(s.routine, s.inputs, s.outputs))
        elif is_filter_cotangent(s.kernel):
            units.append(Unit(s.kernel, s.inputs, [s.output], filter_bands=True))
        else:
            kernel, inputs = s.kernel, list(s.inputs)
            packed = (s.packed or packs(kernel)) if layouts and s.output not in rotated else None
            if packed is not None:
                kernel, made = packed.product, []
                reads = [inputs[gid] for _layout, gid, _to in packed.layouts]
                inputs += [-1] * (kernel.nargs - len(inputs))
                for layout, _gid, to in packed.layouts:
                    inputs[to] = fresh
                    made.append(fresh)
                    fresh += 1
                units.append(Unit(Layouts([layout for layout, _gid, _to in packed.layouts], reads), reads, made))
                units[-1].sizes = {to: layout.bytes for to, (layout, _gid, _to) in zip(made, packed.layouts)}
            options = packed.options if packed is not None else {}
            if not options and s.output not in rotated:
                options = dict(direct_f32=True) if is_direct_product(kernel) else dict(sliced_f16=True) if is_sliced_product(kernel) else {}
            units.append(Unit(kernel, inputs, [s.output], **options))
        k += 1
    return units


_ALIGN = 256


def place_intermediates(units: Sequence[Unit], sizes: Dict[int, int], keep) -> Dict[int, int]:
    """Byte offsets of the buffers that live only inside the program, and the workspace's size under -1: each buffer takes
    the lowest gap that is free from its first write to its last use."""
    first: Dict[int, int] = {}
    last: Dict[int, int] = {}
    for k, u in enumerate(units):
        for b in u.outputs:
            first.setdefault(b, k)
            last[b] = k
        for b in u.inputs + ([u.early] if u.early is not None else []):
            if b in first:
                last[b] = k
    placed: Dict[int, int] = {-1: 0}
    for b in sorted((b for b in first if b not in keep), key=lambda b: (first[b], -sizes[b])):
        need = (sizes[b] + _ALIGN - 1) // _ALIGN * _ALIGN
        busy = sorted((placed[o], placed[o] + (sizes[o] + _ALIGN - 1) // _ALIGN * _ALIGN) for o in placed
                      if o >= 0 and first[o] <= last[b] and first[b] <= last[o])
        at = 0
        for lo, hi in busy:
            if at + need <= lo:
                break
            at = max(at, hi)
        placed[b] = at
        placed[-1] = max(placed[-1], at + need)
    return placed


class Schedule:
    """A jit program prepared for one backend.

    Operands that are laid out as matrices are memory that a program does without as well (up to 1 GiB a contraction): a call for which
    the device has no room runs by a second schedule that lays out none, and so do later ones."""

    def __init__(self, backend, prog, layouts: bool = True):
        from .jit import jitCompile
        from .rewrite import fuse_attention

        self.source = prog  # its expressions, which name it in the backend's cache, live as long as the schedule
        fused = fuse_attention(prog.jaxpr, prog.consts) if prog.jaxpr is not None else None
        if fused is not None:
            prog = jitCompile(fused, prog.consts, backend.maxArgs)
        self.backend, self.prog = backend, prog
        self.units = plan_units(prog, layouts)
        self.laid_out = any(isinstance(u.source, Layouts) for u in self.units)
        self._lean: Optional[Schedule] = None
        self._no_room = False  # for its layouts, in an earlier call
        self._sizes = {s.output: s.size for s in prog.steps if s.kind == "malloc"}
        for u in self.units:
            self._sizes.update(u.sizes)
        self._made = list(dict.fromkeys(o for o in prog.outputs if o >= prog.nargs))
        self._increfs = [s.output for s in prog.steps if s.kind == "incref"]
        self._lock = threading.Lock()
        pinned = []
        try:  # a unit that is prepared here must not push out one that was prepared before it
            for u in self.units:
                try:
                    u.exe = backend.prepareSync(u.source, **u.options)
                except DeviceMemoryError:  # of the executable's own workspace
                    if not u.options:
                        raise
                    u.options = {}
                    u.exe = backend.prepareSync(u.source)
                backend.pin(u.exe)
                pinned.append(u.exe)
            for u in self._weights():
                u.exe = backend.prepareSync(u.source)
                backend.pin(u.exe)
                pinned.append(u.exe)
                self.units.insert(0, u)
            self._work = place_intermediates(self.units, self._sizes, set(self._made))
            self._bind()
        finally:
            for exe in pinned:
                backend.unpin(exe)

    def _weights(self) -> List[Unit]:
        """Launches that lay out the weights of several units, which read them from the program's inputs, into buffers of the call."""
        found = [u for u in self.units if isinstance(u.source, Kernel) and u.source.size and u.exe.data.ks.early is not None
                 and u.inputs[u.exe.data.ks.early.gid] < self.prog.nargs]
        out = []
        for at in range(0, len(found), WEIGHTS_MOST):
            group = found[at:at + WEIGHTS_MOST]
            if len(group) < 2:
                continue
            sources = [u.exe.data.ks for u in group]
            for u, ks in zip(group, sources):
                u.early = max([*self._sizes, self.prog.nargs - 1, *(i for v in self.units for i in v.inputs + v.outputs)]) + 1
                self._sizes[u.early] = ks.early.bytes
            ids = [u.inputs[ks.early.gid] for u, ks in zip(group, sources)]
            out.append(Unit(Weights([u.source for u in group], sources, ids), ids, [u.early for u in group]))
        return out

    def _bind(self) -> None:
        """The native launch list.  Buffer table: inputs, outputs made here, workspace."""
        self._releases = self.backend._releases
        n = self.prog.nargs
        table = {i: i for i in range(n)}
        table.update({o: n + k for k, o in enumerate(self._made)})
        self._workspace = n + len(self._made)
        self._need: Dict[int, int] = {}
        steps, refs = [], []
        for u in self.units:
            prep = u.exe.data
            if prep.released:
                raise ValueError("executable was released (evicted from the backend's cache): prepare it again")
            if isinstance(u.source, Kernel) and u.source.size == 0:
                continue
            needs = dict(prep.ks.min_input_bytes)
            if isinstance(u.source, Routine):
                t = u.source.type
                needs = {i: needs.get(i, prod(s) * byteWidth(d)) for i, (s, d) in enumerate(zip(t.inputShapes, t.inputDtypes))}
            for gid, need in needs.items():
                b = u.inputs[gid]
                if b < n:
                    self._need[b] = max(self._need.get(b, 0), need)
                elif self._sizes[b] < need:
                    raise ValueError(f"buffer {b} holds {self._sizes[b]} bytes, its reader addresses {need}")
            for k, (step, fn) in enumerate(zip(prep.ks.steps, prep.functions)):
                if k == 0 and u.early is not None:
                    continue
                c = LaunchStepC(fn, (ctypes.c_uint32 * 3)(*step.grid), (ctypes.c_uint32 * 3)(*step.block), step.shared, len(step.args))
                steps.append(c)
                for kind, i in step.args:
                    if kind in ("in", "out") or (kind, i) == ("scratch", 0) and u.early is not None:
                        b = u.inputs[i] if kind == "in" else u.outputs[i] if kind == "out" else u.early
                        refs.append(LaunchRef(0, table[b]) if b in table else LaunchRef(self._work[b], self._workspace))
                    else:
                        refs.append(LaunchRef(prep.scratch[i] if kind == "scratch" else int(i), -1))
        self._n_steps = len(steps)
        self._steps = (LaunchStepC * max(len(steps), 1))(*steps)
        self._refs = (LaunchRef * max(len(refs), 1))(*refs)
        self._buffers = (ctypes.c_uint64 * (self._workspace + 1))()
        self._inputs = [(i, self._need.get(i, 0)) for i in range(n)]
        self._zeroed = any(u.exe.data.ks.zeroed_scratch for u in self.units)

    def size_of(self, buffer: int) -> int:
        """Bytes of a buffer that a unit writes, of the program's or of the schedule's own."""
        return self._sizes[buffer]

    def live(self) -> bool:
        """False once an executable of the schedule was released (evicted from the backend's cache)."""
        if self._releases != self.backend._releases:
            if any(u.exe.data.released for u in self.units):
                return False
            self._releases = self.backend._releases
        return True

    def without_layouts(self) -> "Schedule":
        if self._lean is None or not self._lean.live():
            self._lean = Schedule(self.backend, self.source, layouts=False)
        return self._lean

    def _gives_way(self, error: BaseException) -> bool:
        """Whether `error` is that the device has no room, with layouts in the schedule: this call and later ones do without."""
        if not self.laid_out or not isinstance(error, DeviceMemoryError):
            return False
        self._no_room = True
        return True

    def run(self, inputs: Sequence[int]) -> List[int]:
        if self._no_room:
            return self.without_layouts().run(inputs)
        be, prog = self.backend, self.prog
        if len(inputs) != prog.nargs:
            raise ValueError(f"jit program takes {prog.nargs} inputs, got {len(inputs)}")
        if not self.live():
            raise ValueError("executable was released (evicted from the backend's cache): prepare the program again")
        if be.trace is not None or (tracing.isTracing() and not be.capturing):
            return self._run_by_unit(inputs)
        slots = be._slots
        made: List[int] = []
        space = 0
        try:
            for o in self._made:
                made.append(be.malloc(self._sizes[o]))
            space = be._alloc(self._work[-1])
            with self._lock:
                buf = self._buffers
                for i, need in self._inputs:
                    s = slots.get(inputs[i])
                    if s is None:
                        raise SlotError(inputs[i])
                    if s["size"] < need:
                        raise ValueError(f"input {i} holds {s['size']} bytes, the program addresses {need}")
                    buf[i] = s["ptr"]
                for k, m in enumerate(made):
                    buf[prog.nargs + k] = slots[m]["ptr"]
                buf[self._workspace] = space
                rc = be.dev.lib.jh_launch_list(self._steps, self._n_steps, self._refs, buf)
                if rc:
                    if self._zeroed and not be.capturing:
                        for u in self.units:
                            u.exe.data.rezero(be.dev)
                    check(rc, "jh_launch_list")
        except BaseException as e:
            for m in made:
                be.decRef(m)
            if not self._gives_way(e):
                raise
            return self.without_layouts().run(inputs)  # (nothing was launched, and the workspace not allocated)
        finally:
            be._release(space, self._work[-1])  # a later owner's work is queued behind this program's on the one stream
        scope = dict(zip(self._made, made))
        for o in self._increfs:
            be.incRef(scope[o] if o in scope else inputs[o])
        return [scope[o] if o in scope else inputs[o] for o in prog.outputs]

    def _run_by_unit(self, inputs: Sequence[int]) -> List[int]:
        """The same dispatches one at a time, for per-dispatch timestamps."""
        be, prog = self.backend, self.prog
        scope = dict(enumerate(inputs))
        made: Dict[int, int] = {}
        try:
            for u in self.units:
                for o in u.outputs:
                    scope[o] = made[o] = be.malloc(self._sizes[o])
                be.dispatch(u.exe, [scope[i] for i in u.inputs], [scope[o] for o in u.outputs])
        except BaseException as e:
            for s in made.values():
                be.decRef(s)
            if not self._gives_way(e):
                raise
            return self.without_layouts().run(inputs)
        for o, s in made.items():
            if o not in self._made:
                be.decRef(s)
        for o in self._increfs:
            be.incRef(scope[o])
        return [scope[o] for o in prog.outputs]


class PreparedProgram(dict):
    """What `JitProgram.prepare` hands out for the `hip` backend: the schedule, and under a step's index the executable of
    that step alone, prepared when it is asked for."""

    def __init__(self, backend, prog):
        super().__init__()
        self.prog, self.schedule = prog, backend.scheduleProgram(prog)

    def __missing__(self, k: int) -> Any:
        s = self.prog.steps[k]
        if s.kind != "execute":
            raise KeyError(k)
        self[k] = exe = self.schedule.backend.prepareSync(s.kernel if s.routine is None else s.routine)
        return exe
