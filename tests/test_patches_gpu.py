"""Convolutions and their cotangents whose operands are laid out in front of the product, against float64 on the CPU.

Sizes are at the edges of the layouts: k axes that end inside a 16-byte group, a slab and a slice, rows that do not divide over
a workgroup's lanes, more groups of k than a workgroup has lanes, windows that hang over all sides, strides and dilations,
channels below and above the matrix tiles, operands that are read twice or by the epilogue too."""
import numpy as np
import pytest
import torch

from jaxjs_hip import DType
from jaxjs_hip import jit as J
from jaxjs_hip.convolution import ConvParams
from jaxjs_hip.jit import ShapedArray
from jaxjs_hip.patches import Layouts
from jaxjs_hip.schedule import plan_units

from gpu_util import WARM_ONLY, backend, compile_units

CASES = [  # dtype, batch, channels in and out, size, window, stride, padding, dilation
    ("f32", 2, 41, 50, 16, 3, 1, 1, 1),
    ("f32", 3, 20, 33, 21, 5, 2, 2, 1),
    ("f32", 1, 37, 64, 19, 3, 1, 2, 2),
    ("f32", 4, 130, 35, 9, 3, 1, 1, 1),
    ("f32", 5, 35, 64, 25, 1, 1, 0, 1),
    ("f32", 2, 17, 23, 30, 3, 1, 1, 1),
    ("f16", 2, 172, 56, 20, 3, 2, 1, 1),
    ("f16", 3, 41, 129, 13, 5, 2, 2, 1),
    ("f16", 1, 90, 40, 17, 5, 1, 2, 1),
    ("f16", 6, 45, 70, 11, 1, 1, 0, 1),
    ("f16", 2, 26, 44, 21, 3, 1, 1, 1),
]
NP = dict(f32=np.float32, f16=np.float16)


def programs(dtype, B, C, O, S, W, stride, pad, dilation):
    p = ConvParams(0, [stride] * 2, [(pad, pad)] * 2, [1, 1], [dilation] * 2)
    xs, ws = (B, C, S, S), (O, C, W, W)
    out = (S + 2 * pad - dilation * (W - 1) - 1) // stride + 1
    d = dict(f32=DType.Float32, f16=DType.Float16)[dtype]
    x, w, ct = ShapedArray(xs, d), ShapedArray(ws, d), ShapedArray((B, O, out, out), d)
    return dict(forward=(J.jit(lambda x, w: J.conv(x, w, p), [x, w]), (xs, ws)),
                image=(J.jit(lambda ct, w: J.convTransposeLhs(ct, w, list(xs), p), [ct, w]), ((B, O, out, out), ws)),
                filter=(J.jit(lambda x, ct: J.convTransposeRhs(x, ct, list(ws), p), [x, ct]), (xs, (B, O, out, out)))), (xs, ws, (B, O, out, out))


def warm(progs):
    if WARM_ONLY:
        for prog in progs:
            compile_units(prog)
        pytest.skip("warm-up run: compiled only")


def expected(which, args, shapes, stride, pad, dilation):
    xs, ws, _ = shapes
    t = [torch.from_numpy(a.astype(np.float64)) for a in args]
    kw = dict(stride=stride, padding=pad, dilation=dilation)
    if which == "forward":
        return torch.nn.functional.conv2d(t[0], t[1], **kw).numpy()
    if which == "image":
        return torch.nn.grad.conv2d_input(list(xs), t[1], t[0], **kw).numpy()
    return torch.nn.grad.conv2d_weight(t[0], list(ws), t[1], **kw).numpy()


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=str)
def test_laid_out_operands_give_the_convolution(case):
    dtype, stride, pad, dilation = case[0], *case[6:]
    made, shapes = programs(*case)
    warm(prog for prog, _operands in made.values())
    be = backend()
    rng = np.random.default_rng(len(str(case)))
    packed = 0
    for which, (prog, operands) in made.items():
        args = [rng.standard_normal(s).astype(NP[dtype]) for s in operands]
        packed += any(isinstance(u.source, Layouts) for u in plan_units(prog))
        prepared = prog.prepare(be)
        slots = [be.malloc(a.nbytes, a) for a in args]
        want = expected(which, args, shapes, stride, pad, dilation)
        for _ in range(2):
            out, = prog.execute(be, slots, prepared)
            got = np.frombuffer(bytes(be.readSync(out)), NP[dtype]).reshape(want.shape).astype(np.float64)
            be.decRef(out)
            # float32 sums of n products of unit variance: each of up to n roundings is half a unit in the last place of a partial sum of
            # at most a few sqrt(n); float16 results round once more, to 2^-11 of themselves
            n = dict(forward=shapes[1][1] * case[5] ** 2, image=shapes[1][0] * case[5] ** 2, filter=shapes[2][0] * shapes[2][2] ** 2)[which]
            bound = n * 2.0 ** -24 * 4 * np.sqrt(n) + (2.0 ** -11 * np.abs(want) + 2.0 ** -24 if dtype == "f16" else 0.0)
            assert np.all(np.abs(got - want) <= bound), (which, float(np.max(np.abs(got - want) / bound)))
        for s in slots:
            be.decRef(s)
    assert packed


@pytest.mark.gpu
def test_an_operand_that_the_epilogue_reads_too():
    """The image joins the result behind the convolution: it is laid out beside its own buffer, which the epilogue reads."""
    p = ConvParams(0, [1, 1], [(1, 1), (1, 1)], [1, 1], [1, 1])
    x, w = ShapedArray((3, 41, 19, 19), DType.Float32), ShapedArray((41, 41, 3, 3), DType.Float32)
    prog = J.jit(lambda x, w: J.conv(x, w, p).add(x), [x, w])
    assert any(isinstance(u.source, Layouts) for u in plan_units(prog))
    warm([prog])
    be = backend()
    rng = np.random.default_rng(5)
    args = [rng.standard_normal(a.shape).astype(np.float32) for a in (x, w)]
    slots = [be.malloc(a.nbytes, a) for a in args]
    out, = prog.execute(be, slots, prog.prepare(be))
    got = np.frombuffer(bytes(be.readSync(out)), np.float32).reshape(args[0].shape)
    want = expected("forward", args, (x.shape, w.shape, None), 1, 1, 1) + args[0]
    n = 41 * 9
    assert np.max(np.abs(got - want)) <= (n + 1) * 2.0 ** -24 * 4 * np.sqrt(n)
    for s in slots + [out]:
        be.decRef(s)


def evaluate(e, env):
    """An index or mask expression with C's division, which a masked element may come to with a negative operand."""
    from jaxjs_hip.alu import AluOp

    if e.op == AluOp.Const:
        return np.int64(int(e.arg))
    if e.op == AluOp.Special:
        return env[e.arg[0]]
    a = [np.asarray(evaluate(x, env)).astype(np.int64) for x in e.src]
    if e.op in (AluOp.Idiv, AluOp.Mod):
        q = np.abs(a[0]) // a[1] * np.sign(a[0])
        return q if e.op == AluOp.Idiv else a[0] - q * a[1]
    r = {AluOp.Add: lambda: a[0] + a[1], AluOp.Sub: lambda: a[0] - a[1], AluOp.Mul: lambda: a[0] * a[1], AluOp.Cmplt: lambda: a[0] < a[1],
         AluOp.Cmpne: lambda: a[0] != a[1], AluOp.Cast: lambda: a[0], AluOp.Where: lambda: np.where(a[0] != 0, a[1], a[2])}[e.op]()
    return r != 0 if e.dtype == DType.Bool else r


@pytest.mark.parametrize("case", CASES, ids=str)
def test_layouts_hold_the_elements_of_their_views(case):
    """Every element of a layout by its (row, k) expression against the Kernel's own index expression, and zeros behind the axis."""
    from jaxjs_hip.alu import AluExp
    from jaxjs_hip.patches import pack

    for prog, _operands in programs(*case)[0].values():
        for u in prog.steps:
            if u.kind != "execute" or u.kernel is None or (found := pack(u.kernel)) is None:
                continue
            for x, _gid, _to in found.layouts:
                rows = int(np.prod(x.rows))
                r, k = np.arange(0, rows, max(1, rows // 61), dtype=np.int64)[:, None], np.arange(x.st.shape[-1], dtype=np.int64)[None, :]
                cond, load = x.place()
                names = dict(row=r, k=k)
                index = np.broadcast_to(evaluate(load.src[0], names), (r.shape[0], k.shape[1]))
                inside = np.ones(index.shape, bool) if cond is None else np.broadcast_to(evaluate(cond, names), index.shape)
                at, rest = [], r
                for n in reversed(x.rows):
                    at.insert(0, rest % n)
                    rest = rest // n
                axes = [AluExp.special(DType.Int32, f"x{i}", n) for i, n in enumerate(x.st.shape)]
                ref, valid = x.st.toAluExp(axes)
                env = {f"x{i}": v for i, v in enumerate(at + [k])}
                ok = np.broadcast_to(evaluate(valid, env), index.shape)
                assert np.array_equal(inside, ok)
                assert np.array_equal(index[ok], np.broadcast_to(evaluate(ref, env), index.shape)[ok])
                assert not ok.any() or (index[ok].min() >= 0 and index[ok].max() < load.arg[1])


@pytest.mark.parametrize("stride,taken", [(1 << 10, True), ((1 << 31) // 32, True), (1 << 27, False)], ids=str)
def test_operands_past_32_bit_indices_are_not_laid_out(stride, taken):
    """A plain operand whose rows lie far apart, beside a gathered one: element 2^31 of its buffer has no 32-bit index."""
    from jaxjs_hip.alu import AluExp, AluOp
    from jaxjs_hip.lowering import reduceKernel
    from jaxjs_hip.patches import pack
    from jaxjs_hip.shape import ShapeTracker, View

    M, N, K = 256, 32, 70
    a = ShapeTracker.fromShape([M, K - 2]).pad([(0, 0), (1, 1)]).reshape([M, 1, K]).expand([M, N, K])
    b = ShapeTracker([View.create([N, K], [stride, 1], 0, None)]).reshape([1, N, K]).expand([M, N, K])
    found = pack(reduceKernel([M, N, K], [(DType.Float16, a), (DType.Float16, b)], AluExp.mul, AluOp.Add))
    assert (found is not None) == taken


@pytest.mark.parametrize("B,ci,co,size,window,stride,laid_out", [(6, 20, 461, 28, 4, 4, False), (1, 171, 299, 60, 4, 1, False), (2, 388, 65, 40, 4, 2, False), (2, 3, 713, 32, 8, 8, False),
                                                                 (8, 11, 652, 24, 3, 2, True)], ids=str)
def test_windows_with_vector_loads_are_not_laid_out(B, ci, co, size, window, stride, laid_out):
    p = ConvParams(0, [stride] * 2, [(0, 0)] * 2, [1, 1], [1, 1])
    prog = J.jit(lambda x, w: J.conv(x, w, p), [ShapedArray((B, ci, size, size), DType.Float16), ShapedArray((co, ci, window, window), DType.Float16)])
    assert any(isinstance(u.source, Layouts) for u in plan_units(prog)) == laid_out


@pytest.mark.gpu
@pytest.mark.parametrize("case", [CASES[0], CASES[6]], ids=str)
def test_laid_out_operands_under_capture_and_one_dispatch_at_a_time(case):
    """Replays of a graph with other values in between, and the dispatches of a traced run, against the launch list."""
    from jaxjs_hip.graph import GraphedProgram

    warm(prog for prog, _operands in programs(*case)[0].values())
    be = backend()
    for prog, operands in programs(*case)[0].values():
        prepared = prog.prepare(be)
        if not any(isinstance(u.source, Layouts) for u in prepared.schedule.units):
            continue
        rng = np.random.default_rng(3)
        slots = [be.malloc(a.nbytes, a) for a in (rng.standard_normal(s).astype(NP[case[0]]) for s in operands)]
        graph = GraphedProgram(be, prog, slots)
        for _ in range(3):
            for s, shape in zip(slots, operands):
                be.dev.h2d(be.slotPointer(s), rng.standard_normal(shape).astype(NP[case[0]]).tobytes())
            out, = prog.execute(be, slots, prepared)
            apart, = prepared.schedule._run_by_unit(slots)
            graph.launch()
            want = bytes(be.readSync(out))
            assert bytes(be.readSync(apart)) == want and bytes(be.readSync(graph.outputs[0])) == want
            be.decRef(out)
            be.decRef(apart)
        graph.close()
        for s in slots:
            be.decRef(s)


@pytest.mark.gpu
@pytest.mark.parametrize("case", [CASES[0], CASES[6]], ids=str)
def test_programs_without_room_for_layouts(case, monkeypatch):
    """Executed, under capture and one dispatch at a time: the bits of the schedule that lays out nothing."""
    from jaxjs_hip.errors import DeviceMemoryError
    from jaxjs_hip.graph import GraphedProgram
    from jaxjs_hip.schedule import Schedule

    made, shapes = programs(*case)
    prog, operands = made["forward"]
    warm([prog])
    be = backend()
    rng = np.random.default_rng(11)
    slots = [be.malloc(a.nbytes, a) for a in (rng.standard_normal(s).astype(NP[case[0]]) for s in operands)]
    want, = Schedule(be, prog, layouts=False).run(slots)
    size, plain = int(np.prod(shapes[2])) * np.dtype(NP[case[0]]).itemsize, be._alloc

    def small(n):
        if n > size:
            raise DeviceMemoryError(f"no room for {n} bytes")
        return plain(n)
    before = be.live_slots()
    monkeypatch.setattr(be, "_alloc", small)
    schedule = Schedule(be, prog)
    monkeypatch.setattr(be, "scheduleProgram", lambda p: Schedule(be, p))
    assert schedule.laid_out
    outs = schedule.run(slots) + schedule.run(slots) + Schedule(be, prog)._run_by_unit(slots)
    graph = GraphedProgram(be, prog, slots)
    for _ in range(2):
        graph.launch()
        for o in outs + graph.outputs:
            assert bytes(be.readSync(o)) == bytes(be.readSync(want))
    graph.close()
    for o in outs:
        be.decRef(o)
    assert be.live_slots() == before
    for s in slots + [want]:
        be.decRef(s)


@pytest.mark.parametrize("case,options", [(("f16", 16, 24, 64, 38, 3, 1, 1, 1), dict(thin_rows=True)), (("f16", 2, 61, 21, 21, 3, 1, 1, 1), {}),
                                          (("f32", 9, 28, 25, 18, 5, 2, 2, 1), dict(allow_gemm=False, row_lanes=64)), (("f32", 10, 67, 21, 55, 3, 1, 1, 1), None)], ids=str)
def test_few_rows_behind_a_layout(case, options):
    """Products of few rows: tiles, and a float32 sum by lanes that stays one, or stays where it was (`options` None), for the cotangent
    towards the image (of the first), the forward direction (of the second and third) and the filter's (of the last)."""
    made, _ = programs(*case)
    prog = made["image" if case[1] == 16 else "filter" if options is None else "forward"][0]
    units = plan_units(prog)
    assert any(isinstance(u.source, Layouts) for u in units) == (options is not None)
    if options is not None:
        assert {k: v for k, v in units[-1].options.items()} == options
