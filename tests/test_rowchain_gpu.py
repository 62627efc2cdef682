"""Runs of Kernels over the same rows in one launch, against the same program on the CPU checker, at row lengths around the
vector width, the lane counts and the register limit."""
import numpy as np
import pytest

from gpu_util import WARM_ONLY, backend, compile_units
from jaxjs_hip import DType
from jaxjs_hip import jit as J
from jaxjs_hip import library as L
from jaxjs_hip import workloads as W
from jaxjs_hip.jit import ShapedArray
from jaxjs_hip.rowchain import RowChain
from jaxjs_hip.rowproduct import ProductRows, RowProduct
from jaxjs_hip.schedule import plan_units
from jit_util import run_program
from oracle.backend import OracleBackend
from test_schedule import WIDE, wide_programs

pytestmark = pytest.mark.gpu
OPS = {"softmax": lambda x: L.softmax(x, -1), "logsoftmax": lambda x: L.logSoftmax(x, -1), "standardize": lambda x: L.standardize(x, -1),
       "argmax": lambda x: L.argmax(x, -1), "softmax_of_masked": lambda x: L.softmax(J.where(L.tri_const(x.shape[-2], x.shape[-1], 0), x, -1e30), -1)}
SHAPES = [(1, 2), (3, 7), (64, 10), (5, 64), (300, 66), (2, 33, 257), (1100, 1024), (7, 4097), (3, 50257)]


def check(prog, arrays, f16, chained=True, terms=0):
    """`terms` of a product behind the chain: each of as many additions rounds a partial sum of up to 4 by 2^-23 at most, on either
    side and in an order of its own, so the two differ by a random walk of 2 sqrt(terms) such steps and a few times that.  In float16 the product and the two sums
    behind it are rounded, values of up to 4 (2^-9 apart below) that may cancel in the result: an ulp for each."""
    chains = [u.source for u in plan_units(prog) if isinstance(u.source, RowChain)]
    assert len(chains) == 1 or not chained, [type(u.source).__name__ for u in plan_units(prog)]
    if WARM_ONLY:
        compile_units(prog)
        pytest.skip("warm-up run: compiled only")
    be = backend()
    before = be.live_slots()
    got, want = run_program(be, prog, arrays), run_program(OracleBackend(), prog, arrays)
    assert be.live_slots() == before
    for g, w in zip(got, want):
        if g.dtype.kind in "iu":
            np.testing.assert_array_equal(g, w)
        else:
            np.testing.assert_allclose(g.astype(np.float64), w.astype(np.float64), rtol=1e-2 if f16 else 2e-5, atol=2e-3 + (3 * 2.0 ** -9 if terms else 0) if f16 else 2e-6 + 8 * terms ** 0.5 * 2.0 ** -23)


class OneByOne:
    """A program whose Kernels are dispatched one after the other, each in a launch of its own."""

    def __init__(self, prog):
        self.consts, self.steps, self.outputs, self.prog = prog.consts, prog.steps, prog.outputs, prog

    def execute(self, be, slots):
        return self.prog.execute(be, slots, {k: be.prepareKernelSync(s.kernel) for k, s in enumerate(self.steps) if s.kind == "execute"})


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("dtype", [DType.Float32, DType.Float16], ids=lambda d: d.value)
@pytest.mark.parametrize("op", list(OPS))
def test_row_chains(op, dtype, shape):
    if op == "softmax_of_masked" and shape[-1] > 5000:
        pytest.skip("the mask constant alone is large")
    f16 = dtype == DType.Float16
    x = np.random.default_rng(shape[-1]).standard_normal(shape).astype(np.float16 if f16 else np.float32)
    check(J.jit(OPS[op], [ShapedArray(tuple(shape), dtype)]), [x], f16)


def test_a_chain_keeps_what_is_read_behind_it():
    """Results of the middle of a chain that the program returns or a later Kernel reads are stored as well."""
    def f(x, w):
        m = x.max(-1, keepdims=True)
        e = J.exp(x.sub(m))
        s = e.sum(-1, keepdims=True)
        y = e.div(s)
        return [y, m.reshape([40]), e, L.matmul(y, w)]
    rng = np.random.default_rng(3)
    x, w = rng.standard_normal((40, 96)).astype(np.float32), rng.standard_normal((96, 48)).astype(np.float32)
    check(J.jit(f, [ShapedArray(x.shape, DType.Float32), ShapedArray(w.shape, DType.Float32)]), [x, w], False, chained=False)


def test_row_statistics_of_the_benchmark_program():
    x = np.random.default_rng(1).standard_normal((333, 4096)).astype(np.float32)
    check(W.rowSoftmaxArgmaxProgram(333, 4096), [x], False)


@pytest.mark.parametrize("mnk", [(8, 512, 256), (130, 257, 100), (512, 512, 256), (128, 128, 2048), (1, 96, 64)], ids=str)
@pytest.mark.parametrize("dtype", [DType.Float32, DType.Float16], ids=lambda d: d.value)
def test_an_elementwise_kernel_in_a_contractions_epilogue(dtype, mnk):
    m, n, k = mnk
    rng, t = np.random.default_rng(m), np.float16 if dtype == DType.Float16 else np.float32
    arrays = [rng.standard_normal((m, k)).astype(t), (rng.standard_normal((k, n)) * k ** -0.5).astype(t), rng.standard_normal(n).astype(t)]
    prog = J.jit(lambda x, w, b: L.gelu(L.matmul(x, w).add(b)), [ShapedArray(a.shape, dtype) for a in arrays])
    check(prog, arrays, dtype == DType.Float16, chained=False)


@pytest.mark.parametrize("cols", [2, 37, 257, 1024, 4097])
@pytest.mark.parametrize("op", ["max", "min"])
def test_largest_and_smallest_of_rows_with_values_that_are_no_ordinary_numbers(op, cols):
    """A NaN at any place is the result, infinities are values, and -0 is below +0: bit for bit, on every lane of the row."""
    rng = np.random.default_rng(cols)
    x = rng.standard_normal((9, cols)).astype(np.float32)
    x[0, 0] = x[1, -1] = x[2, cols // 2] = np.nan
    x[3, cols // 3], x[4, cols // 3] = np.inf, -np.inf
    x[5], x[6] = np.copysign(0.0, -1), 0.0
    x[7], x[7, -1], x[8], x[8, 0] = np.copysign(0.0, -1), 0.0, -np.inf, np.nan

    def f(v):
        m = getattr(v, op)(-1, keepdims=True)
        return [m.reshape([9]), v.sub(m)]
    prog = J.jit(f, [ShapedArray(x.shape, DType.Float32)])
    assert [type(u.source) for u in plan_units(prog)] == [RowChain]
    if WARM_ONLY:
        check(prog, [x], False)
    m, y = run_program(backend(), prog, [x])
    m = np.asarray(m).reshape(9)
    # the order of the operation: -0 below +0, anything below a NaN
    key = lambda v: (1, 0.0, 0) if np.isnan(v) else (0, float(v), 0 if np.signbit(v) else 1)  # noqa: E731
    low = lambda v: (0, 0.0, 0) if np.isnan(v) else (1, float(v), 0 if np.signbit(v) else 1)  # noqa: E731
    want = np.array([max(r, key=key) if op == "max" else min(r, key=low) for r in x], np.float32)
    np.testing.assert_array_equal(m, want)
    np.testing.assert_array_equal(np.signbit(m[5:8]), np.signbit(want[5:8]))
    with np.errstate(invalid="ignore"):
        np.testing.assert_array_equal(np.asarray(y).reshape(x.shape), x - want[:, None])


@pytest.mark.parametrize("count", [2, 8, 11])
@pytest.mark.parametrize("size", [1, 7, 1000, 262145])
def test_elementwise_kernels_side_by_side(count, size):
    """Sizes off the vector width, several types, more Kernels than one launch takes; a masked read; one operand for all.  The
    same bits as from the Kernels dispatched one by one."""
    rng = np.random.default_rng(size)
    arrays = [rng.standard_normal(size).astype(np.float16 if i % 3 == 2 else np.float32) for i in range(count)]
    arrays.append(rng.integers(-9, 9, size).astype(np.int32))

    def f(*a):
        return [x.mul(float(i + 1)).add(x) if i % 2 else L.concatenate([x, x], 0) for i, x in enumerate(a[:-1])] + [a[-1].add(3)]
    prog = J.jit(f, [ShapedArray(x.shape, {"f": DType.Float32, "e": DType.Float16, "i": DType.Int32}[x.dtype.char]) for x in arrays])
    assert [len(u.outputs) for u in plan_units(prog)] == {2: [3], 8: [8, 1], 11: [8, 4]}[count]
    check(prog, arrays, True, chained=False)
    for i, (together, apart) in enumerate(zip(run_program(backend(), prog, arrays), run_program(backend(), OneByOne(prog), arrays))):
        assert together.dtype == apart.dtype and together.tobytes() == apart.tobytes(), i


@pytest.mark.parametrize("name", WIDE)
def test_launches_of_as_many_arguments_as_a_launch_list_takes(name):
    """Small whole numbers: every sum is exact."""
    prog, _ = wide_programs()[name]
    if WARM_ONLY:
        pytest.skip("warm-up run")
    rng = np.random.default_rng(len(name))
    arrays = [rng.integers(-2, 3, v.aval.shape).astype(np.float32) for v in prog.jaxpr.inBinders]
    for got, want in zip(run_program(backend(), prog, arrays), run_program(OracleBackend(), prog, arrays)):
        np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("rows,k,n", [(2, 256, 130), (16, 100, 200), (5, 100, 333), (8, 768, 2304), (13, 333, 777), (33, 256, 260), (64, 512, 1000), (8, 2048, 512)], ids=str)
@pytest.mark.parametrize("dtype", [DType.Float32, DType.Float16], ids=lambda d: d.value)
@pytest.mark.parametrize("transposed", [False, True])
def test_rows_made_in_the_launch_of_their_product(transposed, dtype, rows, k, n):
    """Rows and columns off the tile and the vector width, more rows than a workgroup makes at once, a k axis in slices."""
    rng, t = np.random.default_rng(k), np.float16 if dtype == DType.Float16 else np.float32
    arrays = [rng.standard_normal((rows, k)).astype(t), (1 + 0.1 * rng.standard_normal(k)).astype(t), (0.1 * rng.standard_normal(k)).astype(t),
              (rng.standard_normal((n, k) if transposed else (k, n)) * k ** -0.5).astype(t), rng.standard_normal(n).astype(t), rng.standard_normal((rows, n)).astype(t)]

    def f(x, g, b, w, c, r):
        return r.add(L.matmul(L.standardize(x).mul(g).add(b), L.swapaxes(w, 0, 1) if transposed else w).add(c))
    prog = J.jit(f, [ShapedArray(a.shape, dtype) for a in arrays])
    few = any(isinstance(u.source, RowProduct) for u in plan_units(prog))
    assert few or transposed and k < 512, [type(u.source).__name__ for u in plan_units(prog)]  # (short rows of such weights are dot products)
    check(prog, arrays, dtype == DType.Float16, chained=False, terms=k)


def test_rows_that_something_else_reads_stay_a_launch_of_their_own():
    def f(x, w, v):
        h = L.standardize(x)
        return [L.matmul(h, w), L.matmul(h, v)]
    def g(x, w):
        h = L.standardize(x)
        return [h, L.matmul(h, w)]
    rng = np.random.default_rng(0)
    x, w, v = (rng.standard_normal(s).astype(np.float32) for s in ((8, 256), (256, 96), (256, 64)))
    for fn, arrays in ((f, [x, w, v]), (g, [x, w])):
        prog = J.jit(fn, [ShapedArray(a.shape, DType.Float32) for a in arrays])
        assert not any(isinstance(u.source, RowProduct) for u in plan_units(prog))
        check(prog, arrays, False, chained=False, terms=256)


@pytest.mark.parametrize("rows,k,n", [(3, 40, 2), (64, 256, 10), (33, 64, 10), (17, 100, 33), (200, 96, 64), (1024, 512, 16), (8200, 64, 46)], ids=str)
@pytest.mark.parametrize("order", ["kn", "nk", "first along rows"])
@pytest.mark.parametrize("dtype", [DType.Float32, DType.Float16], ids=lambda d: d.value)
@pytest.mark.parametrize("op", ["softmax", "argmax"])
def test_rows_of_a_narrow_product_in_its_launch(op, dtype, order, rows, k, n):
    """Rows off the tile, columns off the vector width and up to the widest tile, operands in all orders the kernel reads;
    the result alone, and an argmax (whose ties and order are exact)."""
    rng, t = np.random.default_rng(k), np.float16 if dtype == DType.Float16 else np.float32
    x, w = rng.standard_normal((rows, k)).astype(t), (rng.standard_normal((k, n)) * k ** -0.5).astype(t)
    if op == "argmax":  # small integers: the same sums in any order
        x, w = rng.integers(-2, 3, (rows, k)).astype(t), rng.integers(-1, 2, (k, n)).astype(t)
    arrays = [np.ascontiguousarray(x.T) if order == "first along rows" else x, np.ascontiguousarray(w.T) if order != "kn" else w, np.zeros(n, t)]

    def f(a, b, c):
        a = L.swapaxes(a, 0, 1) if order == "first along rows" else a
        return OPS[op](L.matmul(a, L.swapaxes(b, 0, 1) if order != "kn" else b).add(c))
    prog = J.jit(f, [ShapedArray(a.shape, dtype) for a in arrays])
    assert any(isinstance(u.source, ProductRows) for u in plan_units(prog)), [type(u.source).__name__ for u in plan_units(prog)]
    check(prog, arrays, dtype == DType.Float16, chained=False, terms=k)
