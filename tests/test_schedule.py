"""Host logic of a jit program's schedule: index forms against direct evaluation, placement of intermediates."""
import numpy as np
import pytest

from jaxjs_hip.alu import AluExp, AluVar, DType
from jaxjs_hip.rowchain import index_form
from jaxjs_hip.schedule import Unit, place_intermediates
from jaxjs_hip.shape import ShapeTracker


@pytest.mark.parametrize("seed", range(40))
def test_index_form_has_the_value_of_its_expression(seed):
    rng = np.random.default_rng(seed)
    R, C = int(rng.integers(1, 30)), int(rng.integers(1, 40))
    row, col = AluExp.special(DType.Int32, "gidx", R), AluExp.special(DType.Int32, "ridx", C)
    flat = AluExp.add(AluExp.mul(row, AluExp.i32(C)), col)
    e = flat
    for _ in range(int(rng.integers(1, 5))):
        n = int(rng.choice([1, 2, 3, 5, C, 2 * C, C * R, max(1, C // 2)]))
        e = [lambda: AluExp.mod(e, AluExp.i32(n)), lambda: AluExp.idiv(e, AluExp.i32(n)),
             lambda: AluExp.add(AluExp.mul(AluExp.idiv(flat, AluExp.i32(n)), AluExp.i32(n)), AluExp.mod(flat, AluExp.i32(n))),
             lambda: AluExp.add(AluExp.mul(e, AluExp.i32(n)), row)][int(rng.integers(0, 4))]()
    f = index_form(e, {"gidx": R, "ridx": C})
    if f is None:
        return
    for r in range(R):
        for c in range(C):
            got = sum(v * (1 if k is None else (r if k[0] == "gidx" else c) // k[1]) for k, v in f.items())
            assert got == e.evaluate({"gidx": r, "ridx": c}), (str(e), f, r, c)


def test_unravelled_and_ravelled_positions_have_the_form_of_the_position():
    R, C = 98304, 1024
    row, col = AluExp.special(DType.Int32, "gidx", R), AluExp.special(DType.Int32, "ridx", C)
    i = lambda e, n: AluExp.idiv(e, AluExp.i32(n))  # noqa: E731
    m = lambda e, n: AluExp.mul(e, AluExp.i32(n))  # noqa: E731
    flat = AluExp.add(m(row, C), col)
    e = AluExp.add(m(i(flat, 12 * C * C), 12 * C * C), AluExp.add(m(AluExp.mod(i(flat, C * C), AluExp.i32(12)), C * C),
                                                                 AluExp.add(m(AluExp.mod(row, AluExp.i32(C)), C), col)))
    assert index_form(e, {"gidx": R, "ridx": C}) == {("gidx", 1): C, ("ridx", 1): 1}


def test_intermediates_that_are_alive_together_do_not_overlap():
    rng = np.random.default_rng(5)
    for _ in range(30):
        n = int(rng.integers(2, 14))
        sizes = {k: int(rng.integers(0, 4000)) for k in range(n)}
        units = [Unit(None, [int(x) for x in rng.choice(k, min(k, 2), replace=False)] if k else [], [k]) for k in range(n)]
        placed = place_intermediates(units, sizes, {n - 1})
        last = {k: max([k] + [j for j, u in enumerate(units) if k in u.inputs]) for k in range(n)}
        for a in range(n - 1):
            assert placed[a] % 256 == 0 and placed[a] + sizes[a] <= placed[-1]
            for b in range(a):
                if last[b] >= a:  # b is still read when a is written
                    assert placed[a] + sizes[a] <= placed[b] or placed[b] + sizes[b] <= placed[a], (a, b)


def test_an_elementwise_kernel_joins_the_contraction_that_only_it_reads():
    from jaxjs_hip import jit as J
    from jaxjs_hip import library as L
    from jaxjs_hip.jit import ShapedArray
    from jaxjs_hip.schedule import plan_units
    avals = [ShapedArray(s, DType.Float16) for s in ((64, 128), (128, 256), (256,))]

    def count(f):
        return len(plan_units(J.jit(f, avals)))

    hidden = lambda x, w, b: L.matmul(x, w).add(b)  # noqa: E731
    assert count(lambda x, w, b: L.gelu(hidden(x, w, b))) == 1
    assert count(lambda x, w, b: (lambda h: [L.gelu(h), h])(hidden(x, w, b))) == 2            # the product is kept
    assert count(lambda x, w, b: (lambda h: h.mul(h).mul(L.swapaxes(h, 0, 1)))(L.matmul(x, L.swapaxes(x, 0, 1)))) == 2  # read at another position too


def _stand_in(limit=4096):
    """A backend without a device: kernels are generated, not compiled, and launch lists are kept instead of launched."""
    from collections import OrderedDict

    from jaxjs_hip import backend as B
    from test_backend_cache import make_backend
    be = make_backend(limit)
    be.numerics, be._programs, be.programLimit, be.trace, be._slots, be._next_slot = "fast", OrderedDict(), 512, None, {}, 1
    be._pool, be._pool_bytes, be._pool_limit = {}, 0, 1 << 30
    made = []

    def build(source, ks, blobs=None):
        made.append(B.Executable(source, B._Prepared(ks, [100 + len(made)] * len(ks.steps), [7] * len(ks.scratch_bytes), [1])))
        return made[-1]
    be._build = build
    return be


_MASKS = {"tril": 0, "one above": 1, "one below": -1, "argument": None}


def _masked_attention(k, shape=(1, 48, 48, 2, 32)):
    from jaxjs_hip import jit as J
    from jaxjs_hip import library as L
    from jaxjs_hip.jit import ShapedArray
    B, l, s, n, h = shape

    def attend(mask, q, key, v):
        scores = L.einsum("BLNH,BSNH->BNLS", q, key).mul(h ** -0.5)
        return L.einsum("BNLS,BSNH->BLNH", L.softmax(J.where(mask, scores, -np.inf), -1), v)
    operands = [ShapedArray((B, t, n, h), DType.Float16) for t in (l, s, s)]
    if k is None:
        return J.jit(attend, [ShapedArray((l, s), DType.Bool)] + operands)
    return J.jit(lambda q, key, v: attend(L.tri_const(l, s, k), q, key, v), operands)


@pytest.mark.parametrize("order", [list(_MASKS), list(_MASKS)[::-1]], ids=["tril first", "tril last"])
def test_a_schedule_is_found_again_only_for_the_constants_it_was_made_for(order):
    """Four programs with the same dispatches: only the one whose mask is the lower triangle has a causal attention."""
    be = _stand_in()
    for _ in range(2):
        for name in order:
            units = be.scheduleProgram(_masked_attention(_MASKS[name])).units
            assert any(getattr(u.source, "params", None) for u in units) == (name == "tril"), name
    assert len(be._programs) == 4


def test_a_schedule_keeps_the_program_that_its_key_was_made_from():
    """The key names expressions by identity: they have to live as long as it does, rewritten program or not."""
    import gc
    import weakref
    be = _stand_in()
    prog = _masked_attention(0)
    nodes = [weakref.ref(k.exp) for k in prog.kernels]
    be.scheduleProgram(prog)
    del prog
    gc.collect()
    assert all(n() is not None for n in nodes)


@pytest.mark.parametrize("total,top", [("row", "row"), ("column", "row"), ("row", "column"), ("column", "column")])
@pytest.mark.parametrize("masked", [False, True], ids=["full", "causal"])
def test_a_softmax_that_uses_a_row_s_sum_or_maximum_along_the_columns_stays_as_it_is(masked, total, top):
    """With as many queries as keys the sums of the rows fit the columns as well: that is another function."""
    from jaxjs_hip import jit as J
    from jaxjs_hip import library as L
    from jaxjs_hip.jit import ShapedArray
    from jaxjs_hip.rewrite import fuse_attention
    B, T, N, H = 2, 24, 3, 64
    spread = {"row": [B, N, T, 1], "column": [B, N, 1, T]}

    def f(q, k, v):
        scores = L.einsum("BLNH,BSNH->BNLS", q, k).mul(0.125)
        if masked:
            scores = J.where(L.tri_const(T, T, 0), scores, -np.inf)
        e = J.exp(scores.sub(J.stopGradient(scores.max(-1).reshape(spread[top]))))
        return L.einsum("BNLS,BSNH->BLNH", e.div(e.sum(-1).reshape(spread[total])), v)
    prog = J.jit(f, [ShapedArray((B, T, N, H), DType.Float16)] * 3)
    assert (fuse_attention(prog.jaxpr, prog.consts) is not None) == (total == top == "row")


@pytest.mark.parametrize("limit", [1, 2, 3])
def test_a_schedule_of_more_executables_than_the_cache_holds_launches_all_of_them(limit):
    """Nothing that a schedule is made of is evicted while the rest of it is prepared; afterwards it is, as anything else."""
    from jaxjs_hip import jit as J
    from jaxjs_hip import library as L
    from jaxjs_hip.jit import ShapedArray
    be = _stand_in(limit)
    avals = [ShapedArray(s, DType.Float32) for s in ((64, 128), (128, 256), (256, 512), (512, 64))]
    prog = J.jit(lambda x, a, b, c: L.matmul(L.matmul(L.matmul(x, a), b), c), avals)
    s = be.scheduleProgram(prog)
    assert len(s.units) == 3 and s.live() and s._n_steps == sum(len(u.exe.data.ks.steps) for u in s.units) >= 3
    assert not any(u.exe.data.pins or u.exe.data.released for u in s.units)
    assert be.scheduleProgram(prog) is s
    be.prepareKernelSync(J.jit(lambda x: L.matmul(x, x), [ShapedArray((96, 96), DType.Float32)]).kernels[0])
    assert len(be._exes) <= limit and not s.live()
    again = be.scheduleProgram(prog)
    assert again is not s and again.live() and again._n_steps == s._n_steps
    with pytest.raises(ValueError, match="released"):
        s.run([0, 1, 2, 3])


def test_a_schedule_that_cannot_be_prepared_leaves_nothing_pinned():
    from jaxjs_hip import jit as J
    from jaxjs_hip import library as L
    from jaxjs_hip.jit import ShapedArray
    be = _stand_in()
    prog = J.jit(lambda x, a, b: L.matmul(L.matmul(x, a), b), [ShapedArray(s, DType.Float32) for s in ((64, 128), (128, 256), (256, 64))])
    build, calls = be._build, []

    def second_fails(*a):
        calls.append(a)
        if len(calls) == 2:
            raise RuntimeError("no memory")
        return build(*a)
    be._build = second_fails
    with pytest.raises(RuntimeError, match="no memory"):
        be.scheduleProgram(prog)
    assert not be._programs and [e.data.pins for e in be._exes.values()] == [0]


@pytest.mark.parametrize("scale", [float("inf"), -float("inf"), float("nan"), 70000.0, 0.125, -2.0, 0.0])
def test_attention_under_a_scale_that_is_not_a_finite_float16_stays_as_it_is(scale):
    """The routine's source holds the scale as a number; the composition multiplies by whatever it is given."""
    from jaxjs_hip import jit as J
    from jaxjs_hip import library as L
    from jaxjs_hip.jit import ShapedArray
    from jaxjs_hip.rewrite import fuse_attention
    from jaxjs_hip.routinegen import generateRoutine
    from jaxjs_hip.runtime import compile_source
    prog = J.jit(lambda q, k, v: L.dotProductAttention(q, k, v, scale=scale), [ShapedArray((1, 40, 2, 32), DType.Float16)] * 3)
    fused = fuse_attention(prog.jaxpr, prog.consts)
    assert (fused is not None) == (abs(scale) < 65520)
    if fused is not None:
        for source in generateRoutine(J.jitCompile(fused, prog.consts).routines[0], "fast").sources:
            compile_source(source)


@pytest.mark.parametrize("heads,queries,keys,size,causal,routine", [
    # decode: microseconds of the routine and of the composition at these shapes
    (96, 1, 1025, 64, False, True),     # 6 and 14
    (12, 4, 4096, 64, False, True),     # 12 and 17
    (12, 1, 16384, 64, False, False),   # 52 and 20
    (1, 4, 65536, 64, False, False),    # 162 and 36
    (12, 1, 16384, 128, False, False),  # 99 and 27
    (384, 1, 8192, 64, False, False),   # 156 and 144
    (384, 2, 2048, 64, False, True),    # 43 and 51: in tiles
    (192, 2, 8192, 64, False, False),   # 119 and 107
    (192, 4, 8192, 64, False, True),    # 118 and 152
    # prefill
    (12, 5, 512, 64, False, True),      # 8 and 12
    (12, 5, 4096, 64, False, False),    # 52 and 17
    (12, 128, 16384, 64, False, False),  # 204 and 55
    (96, 128, 4096, 64, False, True),   # 54 and 106
    (96, 16, 4096, 128, False, True),   # 79 and 179
    (96, 1024, 1024, 64, True, True),   # 27 and 203
    (1, 128, 16384, 64, True, True),    # 6 and 22: the mask hides all but 128 keys
    (1, 1024, 1024, 64, True, False),   # 18 and 11
], ids=str)
def test_attention_runs_as_the_routine_where_that_is_the_faster_one(heads, queries, keys, size, causal, routine):
    from jaxjs_hip import jit as J
    from jaxjs_hip import library as L
    from jaxjs_hip.jit import ShapedArray
    from jaxjs_hip.rewrite import fuse_attention
    shapes = [(1, t, heads, size) for t in (queries, keys, keys)]
    prog = J.jit(lambda q, k, v: L.dotProductAttention(q, k, v, isCausal=causal), [ShapedArray(s, DType.Float16) for s in shapes])
    assert (fuse_attention(prog.jaxpr, prog.consts) is not None) == routine


@pytest.mark.parametrize("seed", range(4))
def test_what_is_recognised_as_attention_computes_what_the_composition_does(seed, monkeypatch):
    """Variations of the composition (along which axis sums and maxima go, masks, scales, operands in another order, values
    used twice), with extents that coincide: whatever is rewritten gives the composition's results on the checker."""
    import random

    from jaxjs_hip import jit as J
    from jaxjs_hip import library as L
    from jaxjs_hip import rewrite
    from jaxjs_hip.jit import ShapedArray, jitCompile
    from jit_util import run_program
    from oracle.backend import OracleBackend
    monkeypatch.setattr(rewrite, "routine_is_faster", lambda *a: True)
    rng, values = random.Random(seed), np.random.default_rng(seed)
    mostly = lambda usual, *others: usual if rng.random() < 0.8 else rng.choice(others)  # noqa: E731
    fused = 0
    for _ in range(150):
        B, N, H, T = rng.choice([1, 2]), rng.choice([1, 2, 3]), rng.choice([32, 64]), rng.choice([2, 5, 8])
        S = mostly(T, 3, 9)
        top, total = (mostly("row", "column", "all") for _ in range(2))
        mask, scale, again = mostly(0, 1, None, "none"), mostly(0.125, -0.5, 1.0, "twice"), mostly("no", "probabilities", "scores")
        order, shift = mostly("exp first", "sum first"), mostly("minus", "from")

        def along(x, how):
            return x.max() if how == "all" else x.reshape([B, N, 1, T] if how == "column" and T == S else [B, N, T, 1])

        def f(*args):
            q, k, v = args[-3:]
            s = L.einsum("BLNH,BSNH->BNLS", q, k)
            s = s.mul(0.5).mul(0.25) if scale == "twice" else s if scale == 1.0 else s.mul(scale)
            if mask != "none":
                s = J.where(args[0] if mask is None else L.tri_const(T, S, mask), s, -np.inf)
            m = J.stopGradient(along(s.max(-1), top))
            e = J.exp(s.sub(m) if shift == "minus" else m.sub(s))
            r = J.reciprocal(along(e.sum(-1), total))
            p = e.mul(r) if order == "exp first" else r.mul(e)
            out = L.einsum("BNLS,BSNH->BLNH", p, v)
            return [out, p] if again == "probabilities" else [out, s] if again == "scores" else [out]
        avals = [ShapedArray((B, t, N, H), DType.Float16) for t in (T, S, S)]
        arrays = [values.standard_normal(a.shape).astype(np.float16) for a in avals]
        if mask is None:
            avals = [ShapedArray((T, S), DType.Bool)] + avals
            arrays = [((values.random((T, S)) < 0.6) | (np.arange(S) == 0)).astype(np.int32)] + arrays
        prog = J.jit(f, avals)
        other = rewrite.fuse_attention(prog.jaxpr, prog.consts)
        if other is None:
            continue
        fused += 1
        want, got = (run_program(OracleBackend(), p, arrays)[0].astype(np.float64) for p in (prog, jitCompile(other, prog.consts)))
        what = (B, N, T, S, H, top, total, mask, scale, again, order, shift)
        np.testing.assert_allclose(got, want, rtol=1e-2, atol=3e-3 * max(1.0, np.nanmax(np.abs(want))), equal_nan=True, err_msg=str(what))
    assert fused >= 15


@pytest.mark.parametrize("shape,dtype,f,launches", [
    # microseconds joined and in two launches
    ((512, 512, 512), DType.Float16, "erfc", 2),     # 13.5 and 8.7
    ((512, 512, 512), DType.Float16, "sin", 2),      # 12.8 and 8.6
    ((512, 512, 512), DType.Float16, "atan", 2),     # 10.5 and 8.4
    ((8192, 3072, 768), DType.Float16, "erfc", 2),   # 78 and 73
    ((512, 512, 512), DType.Float16, "tanh", 1),     # 8.4 and 8.5 (gelu)
    ((8192, 3072, 768), DType.Float16, "tanh", 1),
    ((8, 3072, 768), DType.Float16, "erfc", 1),      # 5.7 and 8.7: the kernel for few rows
    ((2048, 2048, 64), DType.Float16, "erfc", 1),    # 12.7 and 15.5
    ((512, 512, 512), DType.Float32, "erfc", 1),     # 12.5 and 12.9
    ((8000, 1000, 100), DType.Float32, "sin", 1),
], ids=str)
def test_a_long_epilogue_stays_a_launch_of_its_own_behind_float16_tiles(shape, dtype, f, launches):
    from jaxjs_hip import jit as J
    from jaxjs_hip import library as L
    from jaxjs_hip.jit import ShapedArray
    from jaxjs_hip.schedule import plan_units
    m, n, k = shape
    act = dict(erfc=J.erfc, sin=J.sin, atan=J.atan, tanh=L.tanh)[f]
    prog = J.jit(lambda x, w: (lambda h: h.mul(act(h)))(L.matmul(x, w)), [ShapedArray(s, dtype) for s in ((m, k), (k, n))])
    assert len(plan_units(prog)) == launches


@pytest.mark.parametrize("room", [0, 1, 2])
def test_a_call_that_runs_out_of_memory_gives_back_what_it_took(room):
    """Outputs and the workspace are taken one after the other; whichever fails, the call leaves no slot behind."""
    from jaxjs_hip import jit as J
    from jaxjs_hip import library as L
    from jaxjs_hip.jit import ShapedArray
    be = _stand_in()
    shapes = ((64, 128), (128, 256), (256, 64))
    prog = J.jit(lambda x, a, b: (lambda h: [L.matmul(h, b), J.exp(x)])(L.matmul(x, a)), [ShapedArray(s, DType.Float32) for s in shapes])
    taken = []

    def malloc(n):
        if len(taken) == room:
            raise MemoryError(n)
        taken.append(n)
        return 4096 * len(taken)
    be.dev.malloc = malloc
    be._alloc = lambda n: malloc(n) if n else 0
    schedule = be.scheduleProgram(prog)
    assert schedule._work[-1] > 0 and len(schedule._made) == 2
    be._slots = {i + 1: dict(ptr=1 << 20, size=1 << 20, ref=1) for i in range(3)}
    be._next_slot = 4
    with pytest.raises(MemoryError):
        schedule.run([1, 2, 3])
    assert list(be._slots) == [1, 2, 3] and sum(len(free) for free in be._pool.values()) == room


def test_elementwise_kernels_share_a_launch_until_one_reads_another():
    from jaxjs_hip import jit as J
    from jaxjs_hip import library as L
    from jaxjs_hip.composite import Maps
    from jaxjs_hip.jit import ShapedArray
    from jaxjs_hip.schedule import plan_units

    def f(a, b, c):
        p, q = a.mul(2.0), b.add(1.0)        # two results that the program returns
        m = L.matmul(p, q)
        r, t = m.sub(c), c.mul(3.0)
        return [p, q, m, r, t, J.exp(r.mul(t))]
    prog = J.jit(f, [ShapedArray((48, 48), DType.Float32)] * 3)
    units = plan_units(prog)
    groups = [len(u.outputs) for u in units if isinstance(u.source, Maps)]
    assert groups and groups[0] == 2
    for u in units:
        if isinstance(u.source, Maps):
            assert not set(u.inputs) & set(u.outputs) and len(u.inputs) == sum(k.nargs for k in u.source.kernels)
    made = [o for u in units for o in u.outputs]
    assert len(made) == len(set(made)) and set(prog.outputs) <= set(made)


def wide_programs():
    """Programs whose Kernels, joined, would read more buffers than a step of a launch list takes, by name; and the
    arguments of the launches each keeps."""
    from jaxjs_hip import jit as J
    from jaxjs_hip import library as L
    from jaxjs_hip.jit import ShapedArray

    def total(xs):
        return xs[0] if len(xs) == 1 else total(xs[1:]).add(xs[0])

    def maps(kernels):
        return lambda *xs: [total(xs).mul(float(k + 1)) for k in range(kernels)]

    def product_behind_rows(first, along, behind):
        def f(w, x, *v):
            h = x.add(total(v[:first]))
            return L.matmul(h.sub(h.max(-1, keepdims=True)).add(total(v[first:first + along])), w).add(total(v[first + along:]))
        return J.jit(f, [f32(256, 128), f32(8, 256)] + [f32(256)] * (first + along) + [f32(128)] * behind)

    def rows_behind_product(before, top, along):
        def f(a, w, *v):
            h = L.matmul(a, w).add(total(v[:before]))
            return h.sub(h.add(total(v[before:before + top])).max(-1, keepdims=True)).add(total(v[before + top:]))
        return J.jit(f, [f32(64, 64), f32(64, 16)] + [f32(16)] * (before + top + along))
    f32 = lambda *shape: ShapedArray(shape, DType.Float32)  # noqa: E731
    return {"8 maps of 15": (J.jit(maps(8), [f32(1000)] * 15), [128]), "8 maps of 16": (J.jit(maps(8), [f32(1000)] * 16), [119, 17]),
            "8 maps of 20": (J.jit(maps(8), [f32(1000)] * 20), [126, 42]), "3 maps of 60": (J.jit(maps(3), [f32(1000)] * 60), [122, 61]),
            "product behind rows, 128": (product_behind_rows(5, 60, 60), [128]), "product behind rows, 143": (product_behind_rows(20, 60, 60), [82, 63]),
            "rows behind a product, 128": (rows_behind_product(60, 4, 61), [128]), "rows behind a product, 129": (rows_behind_product(60, 5, 61), [63, 68])}


WIDE = ["8 maps of 15", "8 maps of 16", "8 maps of 20", "3 maps of 60", "product behind rows, 128", "product behind rows, 143", "rows behind a product, 128",
        "rows behind a product, 129"]


@pytest.mark.parametrize("name", WIDE)
def test_no_launch_takes_more_arguments_than_a_launch_list(name):
    import os
    import re
    from jaxjs_hip.runtime import LAUNCH_ARGS
    from jaxjs_hip.schedule import Schedule
    header = open(os.path.join(os.path.dirname(os.path.dirname(__file__)), "include", "jaxhip.h")).read()
    assert int(re.search(r"#define JH_LAUNCH_ARGS (\d+)", header).group(1)) == LAUNCH_ARGS
    prog, args = wide_programs()[name]
    s = Schedule(_stand_in(), prog)
    assert [c.num_args for c in s._steps[:s._n_steps]] == args, [type(u.source).__name__ for u in s.units]


@pytest.mark.parametrize("rows,columns_first,joined", [(4194240, False, True), (4194241, False, False), (5000000, False, False), (5000000, True, True)])
def test_rows_behind_a_product_stay_within_the_grid(rows, columns_first, joined):
    """65535 tiles of 64 rows where the rows are the short operand's (the third dimension of the grid); along the first there is room."""
    from jaxjs_hip import jit as J
    from jaxjs_hip import library as L
    from jaxjs_hip.jit import ShapedArray
    from jaxjs_hip.rowproduct import ProductRows
    from jaxjs_hip.schedule import Schedule
    prog = J.jit(lambda x, w: L.softmax(L.matmul(x, L.swapaxes(w, 0, 1) if columns_first else w), -1),
                 [ShapedArray((rows, 32), DType.Float32), ShapedArray((10, 32) if columns_first else (32, 10), DType.Float32)])
    s = Schedule(_stand_in(), prog)
    assert any(isinstance(u.source, ProductRows) for u in s.units) == joined, [type(u.source).__name__ for u in s.units]
    assert all(c.grid[1] <= 65535 and c.grid[2] <= 65535 for c in s._steps[:s._n_steps])


@pytest.mark.parametrize("dtype,order,rows,cols,k,joined", [
    (DType.Float32, "kn", 100000, 32, 512, True), (DType.Float32, "kn", 100000, 33, 512, False), (DType.Float32, "nk", 200000, 48, 1024, False),
    (DType.Float32, "first along rows", 60000, 32, 864, True), (DType.Float32, "first along rows", 60000, 33, 864, False),
    (DType.Float16, "nk", 90000, 33, 2048, False), (DType.Float16, "nk", 90000, 16, 512, False), (DType.Float16, "kn", 90000, 64, 256, False),
    (DType.Float16, "kn", 60000, 33, 1260, True), (DType.Float16, "kn", 60000, 33, 1261, False), (DType.Float16, "kn", 60000, 40, 1260, False),
    (DType.Float16, "first along rows", 94000, 24, 1024, True), (DType.Float16, "first along rows", 94000, 25, 1024, False),
    (DType.Float16, "first along rows", 94001, 40, 512, True), (DType.Float16, "nk", 1024, 64, 256, True), (DType.Float32, "kn", 1000000, 10, 64, True)], ids=str)
def test_which_rows_behind_a_product_of_many_join(dtype, order, rows, cols, k, joined):
    """Both sides of the rule for products that come in rounds of workgroups, and below its estimate."""
    from jaxjs_hip import jit as J
    from jaxjs_hip import library as L
    from jaxjs_hip.jit import ShapedArray
    from jaxjs_hip.rowproduct import ProductRows
    from jaxjs_hip.schedule import plan_units
    t = lambda x, yes: L.swapaxes(x, 0, 1) if yes else x  # noqa: E731
    prog = J.jit(lambda a, b: L.softmax(L.matmul(t(a, order == "first along rows"), t(b, order != "kn")), -1),
                 [ShapedArray((k, rows) if order == "first along rows" else (rows, k), dtype), ShapedArray((k, cols) if order == "kn" else (cols, k), dtype)])
    units = plan_units(prog)
    assert any(isinstance(u.source, ProductRows) for u in units) == joined, [type(u.source).__name__ for u in units]


@pytest.mark.parametrize("dtype,rows,k,cols,order,joined", [
    (DType.Float32, 2, 1216, 4096, "kn", True), (DType.Float32, 2, 1856, 4096, "nk", True), (DType.Float32, 2, 1856, 4097, "nk", False),
    (DType.Float32, 8, 1423, 8192, "kn", True), (DType.Float32, 8, 1423, 9152, "kn", False), (DType.Float16, 8, 1728, 9088, "kn", False),
    (DType.Float16, 3, 1664, 11328, "nk", True), (DType.Float16, 8, 768, 3072, "kn", True)], ids=str)
def test_rows_are_made_in_workgroups_that_all_have_a_place(dtype, rows, k, cols, order, joined):
    from jaxjs_hip import jit as J
    from jaxjs_hip import library as L
    from jaxjs_hip.jit import ShapedArray
    from jaxjs_hip.rowproduct import RowProduct
    from jaxjs_hip.schedule import plan_units
    prog = J.jit(lambda x, g, w: L.matmul(L.standardize(x).mul(g), L.swapaxes(w, 0, 1) if order == "nk" else w),
                 [ShapedArray((rows, k), dtype), ShapedArray((k,), dtype), ShapedArray((cols, k) if order == "nk" else (k, cols), dtype)])
    units = plan_units(prog)
    assert any(isinstance(u.source, RowProduct) for u in units) == joined, [type(u.source).__name__ for u in units]


def test_schedules_ask_for_direct_loads_of_float32_products():
    from jaxjs_hip import DType, jit as J, library as L
    from jaxjs_hip.jit import ShapedArray
    from jaxjs_hip.kernelgen import generate
    from jaxjs_hip.schedule import plan_units

    def units(dtype, m, n, k):
        return plan_units(J.jit(lambda a, b: L.matmul(a, b), [ShapedArray((m, k), dtype), ShapedArray((k, n), dtype)]))
    for shape, takes in (((512, 512, 512), True), ((1032, 1028, 100), True), ((1032, 1028, 101), False), ((1032, 1027, 100), False), ((132, 196, 60), False)):
        unit, = units(DType.Float32, *shape)
        assert unit.options == (dict(direct_f32=True) if takes else {})
        assert ("global_load_lds_dwordx4" in generate(unit.source, **unit.options).sources[0]) == takes
    assert units(DType.Float16, 512, 512, 512)[0].options == {}


def test_an_attention_is_joined_with_the_copies_that_extend_its_caches():
    from jaxjs_hip import DType, jit as J, library as L
    from jaxjs_hip.jit import ShapedArray, jitCompile
    from jaxjs_hip.rewrite import fuse_attention
    from jaxjs_hip.schedule import plan_units

    def kinds(queries, times=1, third=False):
        def f(q, keys, values, k, v, x):
            keys, values = L.concatenate([keys] + [k] * times, 1), L.concatenate([values] + [v] * times, 1)
            out = [L.dotProductAttention(q, keys, values), keys, values]
            return out + [x.mul(2)] if third else out
        prog = J.jit(f, [ShapedArray((2, n, 4, 64), DType.Float16) for n in (queries, 300, 300, 1, 1, 1)])
        prog = jitCompile(fuse_attention(prog.jaxpr, prog.consts), prog.consts, 30)
        return [(type(u.source).__name__, len(u.outputs)) for u in plan_units(prog)]
    assert kinds(1) == [("CachedAttention", 3)]
    assert ("CachedAttention", 3) in kinds(1, third=True)  # beside another elementwise Kernel
    assert kinds(2) == [("Maps", 2), ("Routine", 1)]       # two workgroups read a head's keys
    assert kinds(1, times=2)[-1] == ("Routine", 1)         # three parts


def test_products_in_front_of_rotations_keep_their_order_of_sums():
    """The Gram matrix of an SVD, also by way of other Kernels: an eigenvector's sign hangs on its last bits.  The product behind
    the rotations is as any other."""
    from jaxjs_hip import DType, jit as J, library as L
    from jaxjs_hip.gemm import is_direct_product
    from jaxjs_hip.jit import ShapedArray
    from jaxjs_hip.routine import Routines
    from jaxjs_hip.schedule import plan_units

    x = ShapedArray((1024, 128), DType.Float32)
    for f in (lambda a: list(L.svd(a)), lambda a: list(L.eigh(J.sin(L.matmul(L.swapaxes(a, 0, 1), a))))):
        units = plan_units(J.jit(f, [x]))
        at = next(i for i, u in enumerate(units) if getattr(u.source, "name", None) == Routines.JacobiEigh)
        assert is_direct_product(units[0].source) and not any(u.options for u in units[:at])
    assert plan_units(J.jit(lambda a: L.matmul(L.swapaxes(a, 0, 1), a), [x]))[0].options == dict(direct_f32=True)


def _filter_cotangent_program(behind):
    """A convolution's filter cotangent whose operands are laid out, the copy that exchanges its channels joined, and what is behind."""
    from jaxjs_hip import DType, jit as J
    from jaxjs_hip.convolution import ConvParams
    from jaxjs_hip.jit import ShapedArray

    p = ConvParams(0, [1, 1], [(2, 2), (2, 2)], [1, 1], [1, 1])
    return J.jit(lambda x, ct: behind(J.convTransposeRhs(x, ct, [54, 43, 5, 5], p)), [ShapedArray((9, 43, 37, 37), DType.Float32), ShapedArray((9, 54, 37, 37), DType.Float32)])


def test_a_copy_is_not_joined_for_layouts_that_are_held_back(monkeypatch):
    """In front of rotations no operands are laid out, and nothing is joined because they would be."""
    from jaxjs_hip import jit as J, library as L, schedule
    from jaxjs_hip.patches import Layouts

    assert [type(u.source) for u in schedule.plan_units(_filter_cotangent_program(lambda w: w))][0] is Layouts

    def gram(w):
        m = w.reshape([54, 43 * 25])
        return [w] + list(L.eigh(L.matmul(m, L.swapaxes(m, 0, 1))))
    prog = _filter_cotangent_program(gram)
    units = [(u.source.key() if hasattr(u.source, "reduction") else type(u.source), u.options) for u in schedule.plan_units(prog)]
    monkeypatch.setattr(schedule, "packs", lambda *a: None)
    assert units == [(u.source.key() if hasattr(u.source, "reduction") else type(u.source), u.options) for u in schedule.plan_units(prog)]


def test_an_epilogue_that_ends_the_layouts_stays_a_launch_of_its_own(monkeypatch):
    from types import SimpleNamespace

    from jaxjs_hip import schedule
    from jaxjs_hip.alu import Kernel
    from jaxjs_hip.patches import Layouts, packs

    made = _filter_cotangent_program(lambda w: w)
    last = [s for s in made.steps if s.kind == "execute"][-1]
    n = last.kernel.size
    twice = Kernel(1, n, AluExp.mul(AluExp.globalView(DType.Float32, 0, ShapeTracker.fromShape([n]), [AluVar.gidx]), AluExp.const(DType.Float32, 2.0)))
    step = SimpleNamespace(kind="execute", kernel=twice, routine=None, inputs=[last.output], output=last.output + 1, outputs=[], size=0)
    prog = SimpleNamespace(steps=made.steps + [step], outputs=[step.output], nargs=made.nargs)
    assert [type(u.source) is Layouts for u in schedule.plan_units(prog)] == [True, False]  # the product with the copy and the factor
    calls = []

    def once(*a):
        calls.append(a)
        return packs(*a) if len(calls) != 2 else None
    monkeypatch.setattr(schedule, "packs", once)
    units = schedule.plan_units(prog)
    assert [type(u.source) is Layouts for u in units] == [True, False, False]


def test_a_program_without_room_for_layouts_runs_without_them():
    from types import SimpleNamespace

    from jaxjs_hip.errors import DeviceMemoryError
    from jaxjs_hip.graph import GraphedProgram
    from jaxjs_hip.schedule import Schedule

    prog = _filter_cotangent_program(lambda w: w)
    size = 9 * 54 * 37 * 37 * 4  # of the larger input

    def device(most):
        be, launched = _stand_in(), []

        def alloc(n):
            if n > most:
                raise DeviceMemoryError(f"no room for {n} bytes")
            return 64
        be._alloc, be._release = alloc, lambda ptr, n: None
        be.dev.lib = SimpleNamespace(jh_launch_list=lambda steps, n, refs, buf: launched.append(n) or 0)
        return be, launched, [be.malloc(size) for _ in range(2)]
    be, launched, inputs = device(1 << 40)
    schedule = Schedule(be, prog)
    assert schedule.laid_out and len(schedule.run(inputs)) == 1
    be, launched, inputs = device(size)
    schedule = Schedule(be, prog)
    for n in (1, 2):
        assert len(schedule.run(inputs)) == 1 and len(launched) == n
        assert be.live_slots() == 2 + n  # what the attempt with layouts made was given back
    lean = schedule.without_layouts()
    assert not lean.laid_out and launched == [lean._n_steps] * 2
    graph = GraphedProgram.__new__(GraphedProgram)
    graph.backend, graph._slots, graph._owned = be, {}, []
    with pytest.raises(DeviceMemoryError):
        graph._make_room(schedule)
    assert be.live_slots() == 4 and not graph._owned
    graph._make_room(lean)
    assert be.live_slots() == 4 + len(graph._owned)
    before, be.dispatch = be.live_slots(), lambda exe, ins, outs: None
    assert len(Schedule(be, prog)._run_by_unit(inputs)) == 1 and be.live_slots() == before + 1 and len(launched) == 3


@pytest.mark.parametrize("m,n", [(1024, 128), (2048, 256), (4096, 136), (3264, 400)], ids=str)
def test_float16_products_in_front_of_rotations_keep_their_order_of_sums(m, n):
    from jaxjs_hip import DType, jit as J, library as L
    from jaxjs_hip.gemm import is_sliced_product
    from jaxjs_hip.jit import ShapedArray
    from jaxjs_hip.routine import Routines
    from jaxjs_hip.schedule import plan_units

    x = ShapedArray((m, n), DType.Float16)
    for f in (lambda a: list(L.svd(a)), lambda a: list(L.eigh(L.matmul(L.swapaxes(a, 0, 1), a)))):
        units = plan_units(J.jit(f, [x]))
        at = next(i for i, u in enumerate(units) if getattr(u.source, "name", None) == Routines.JacobiEigh)
        assert is_sliced_product(units[0].source) and not any(u.options for u in units[:at])


@pytest.mark.parametrize("m,n,k,alone,block", [(192, 224, 896, False, False), (1344, 224, 896, False, False), (768, 192, 768, False, False), (1536, 256, 1024, False, False),
                                               (462, 256, 1024, True, True), (1680, 288, 1152, False, True), (512, 821, 1280, False, False), (384, 1664, 1344, False, True),
                                               (768, 640, 2560, True, True), (615, 768, 3072, True, True), (2240, 576, 2304, True, True)], ids=str)
def test_whole_operands_are_cut_only_where_the_slices_are_worth_the_fold(m, n, k, alone, block):
    """As a product of its own, and behind the bias and the residual of a transformer block's second MLP product."""
    from jaxjs_hip import jit as J, library as L
    from jaxjs_hip.jit import ShapedArray
    from jaxjs_hip.schedule import plan_units

    a, b, bt, bias, rest = (ShapedArray(s, DType.Float16) for s in ((m, k), (k, n), (n, k), (n,), (m, n)))
    plain, = plan_units(J.jit(L.matmul, [a, b]) if n % 4 == 0 else J.jit(lambda a, b: L.matmul(a, L.swapaxes(b, 0, 1)), [a, bt]))
    assert bool(plain.options) == alone
    if n % 4 == 0:
        behind, = plan_units(J.jit(lambda a, b, bias, rest: rest.add(L.matmul(a, b).add(bias)), [a, b, bias, rest]))
        assert bool(behind.options) == block


def test_schedules_ask_for_uneven_slices_of_float16_products():
    from jaxjs_hip import DType, jit as J, library as L
    from jaxjs_hip.jit import ShapedArray
    from jaxjs_hip.schedule import plan_units

    for (m, n, k, t), takes in (((448, 395, 3264, True), True), ((2176, 265, 3843, True), True), ((1984, 1543, 1281, True), True), ((3520, 355, 666, True), False),
                                ((704, 320, 3600, False), False), ((2048, 2048, 2048, False), False), ((8192, 8192, 8192, False), False)):
        shapes = [ShapedArray((m, k), DType.Float16), ShapedArray((n, k) if t else (k, n), DType.Float16)]
        unit, = plan_units(J.jit(lambda a, b: L.matmul(a, L.swapaxes(b, 0, 1) if t else b), shapes))
        assert unit.options == (dict(sliced_f16=True) if takes else {}), (m, n, k)
