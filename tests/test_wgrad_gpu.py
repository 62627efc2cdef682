"""The filter cotangent of a convolution with its bands in LDS (`wgrad_f16.hip.inc`): which Kernels it is chosen for, and its
sums against the definition, tap by tap."""
import numpy as np
import pytest

from gpu_util import WARM_ONLY, backend, device_run
from jaxjs_hip import DType, jit as J
from jaxjs_hip.convolution import ConvParams
from jaxjs_hip.jit import ShapedArray
from jaxjs_hip.kernelgen import generate
from jaxjs_hip.schedule import plan_units

RNG = np.random.default_rng(11)


def cotangent_program(batch, cin, cout, h, w, kh, kw, pad, stride=1, dtype=DType.Float16, dilation=1):
    """(program of the filter's cotangent, shape of the cotangent); pad: ((top, bottom), (left, right))."""
    p = ConvParams(0, [stride] * 2, list(pad), [1, 1], [dilation] * 2)
    oh = (h + sum(pad[0]) - (kh - 1) * dilation - 1) // stride + 1
    ow = (w + sum(pad[1]) - (kw - 1) * dilation - 1) // stride + 1
    avals = [ShapedArray((batch, cin, h, w), dtype), ShapedArray((batch, cout, oh, ow), dtype)]
    prog = J.jit(lambda x, ct: J.convTransposeRhs(x, ct, [cout, cin, kh, kw], p), avals)
    return prog, (batch, cout, oh, ow)


def cotangent_kernel(*args, **kw):
    prog, shape = cotangent_program(*args, **kw)
    return [s.kernel for s in prog.steps if s.kind == "execute"][0], shape


SAME = lambda k: ((k // 2, k // 2),) * 2  # noqa: E731

CASES = [
    # batch, cin, cout, h, w, kh, kw, padding        what it reaches
    (2, 64, 64, 16, 16, 3, 3, SAME(3)),              # whole groups of eight, one launch
    (2, 40, 72, 20, 24, 3, 3, SAME(3)),              # channels past the last tile of either operand
    (4, 33, 31, 37, 41, 3, 3, SAME(3)),              # rows that are no whole groups, bands with fewer rows at the end
    (3, 32, 64, 28, 28, 5, 5, SAME(5)),              # a workgroup per window row, two dwords' worth of padding
    (2, 64, 48, 20, 20, 5, 5, ((0, 0), (0, 0))),     # no padding: the image is wider than the cotangent
    (6, 48, 48, 33, 9, 3, 3, ((0, 0), (1, 0))),      # padding on one side, nine columns
    (9, 32, 32, 9, 57, 3, 2, ((1, 1), (0, 1))),      # an even window, odd numbers of groups
    (2, 64, 64, 24, 24, 4, 4, ((3, 3), (3, 3))),     # full padding: the cotangent is wider than the image
    (9, 64, 96, 56, 56, 3, 3, SAME(3)),              # slices over the bands, more of them than a multiple of eight
]


@pytest.mark.parametrize("case", CASES, ids=str)
def test_plan_covers_the_case(case):
    kernel, _ = cotangent_kernel(*case)
    info = generate(kernel, filter_bands=True).info
    assert "wgrad" in info, info
    assert "wgrad" not in generate(kernel).info  # by itself it keeps the general templates
    units = plan_units(cotangent_program(*case)[0])
    assert [u.options for u in units] == [dict(filter_bands=True)]  # and the exchange of its channels goes with it
    joined = generate(units[0].source, filter_bands=True).info
    assert joined["wgrad"] == info["wgrad"]


# What is done with a cotangent: (from the cotangent, the same in numpy, the Kernels of the schedule: buffers they read and write).
# Buffer 2 is the product in its own order, where that is a result of its own.
READERS = {
    "returned": (lambda c: [c()], lambda c: [c], [([0, 1], 3)]),
    "squared": (lambda c: [(lambda v: v.mul(v))(c())], lambda c: [c * c], [([0, 1], 3)]),
    "exchanged again": (lambda c: (lambda v: [v, J.transpose(v, [1, 0, 2, 3]).mul(2.0)])(c()), lambda c: [c, 2 * c.transpose(1, 0, 2, 3)], [([0, 1], 3), ([3], 4)]),
    "flipped": (lambda c: [J.flip(c(), [2])], lambda c: [c[:, :, ::-1]], [([0, 1], 2), ([2], 3)]),
    "read at two places": (lambda c: (lambda v: [v.add(J.flip(v, [3]))])(c()), lambda c: [c + c[..., ::-1]], [([0, 1], 2), ([2], 3)]),
    "two of them": (lambda c: [c().mul(c())], lambda c: [c * c], [([0, 1], 2), ([0, 1], 3), ([2, 3], 4)]),
}


def reader_program(name, case):
    p = ConvParams(0, [1, 1], list(case[7]), [1, 1], [1, 1])
    _, cts = cotangent_program(*case)
    ws = [case[2], case[1], case[5], case[6]]
    avals = [ShapedArray((case[0], case[1], case[3], case[4]), DType.Float16), ShapedArray(cts, DType.Float16)]
    return J.jit(lambda x, ct: READERS[name][0](lambda: J.convTransposeRhs(x, ct, ws, p)), avals)


@pytest.mark.parametrize("name", list(READERS))
def test_an_exchange_that_is_more_than_one_stays_a_launch(name):
    """What reads the cotangent besides its own transpose, or reads it at other positions, is not joined."""
    units = plan_units(reader_program(name, CASES[0]))
    assert [(u.inputs, u.outputs[0]) for u in units] == READERS[name][2]
    assert [u.options == dict(filter_bands=True) for u in units] == [u.inputs == [0, 1] for u in units]


@pytest.mark.parametrize("kw", [dict(stride=2), dict(dilation=2), dict(dtype=DType.Float32), dict(w=7), dict(kh=1), dict(batch=1, cin=16, cout=16)], ids=str)
def test_what_the_kernel_does_not_cover_stays_where_it_was(kw):
    args = dict(dict(batch=4, cin=64, cout=64, h=24, w=24, kh=3, kw=3, pad=SAME(3)), **kw)
    kernel, _ = cotangent_kernel(**args)
    assert "wgrad" not in generate(kernel, filter_bands=True).info
    assert plan_units(cotangent_program(**args)[0])[0].options == {}


def reference(x, ct, kh, kw, pad):
    """sums[c, o, ky, kx] in 64 bits and the sums of the terms' magnitudes."""
    xp = np.pad(x.astype(np.float64), ((0, 0), (0, 0)) + tuple(pad))
    c64 = ct.astype(np.float64).transpose(1, 0, 2, 3).reshape(ct.shape[1], -1)
    oh, ow = ct.shape[2:]
    want, scale = (np.empty((x.shape[1], ct.shape[1], kh, kw)) for _ in range(2))
    for ky in range(kh):
        for kx in range(kw):
            win = xp[:, :, ky:ky + oh, kx:kx + ow].transpose(1, 0, 2, 3).reshape(x.shape[1], -1)
            with np.errstate(invalid="ignore"):
                want[:, :, ky, kx], scale[:, :, ky, kx] = win @ c64.T, np.abs(win) @ np.abs(c64).T
    return want, scale


def sparse_integers(shape, rng):
    """Mostly zeros, the rest 1 or -1: sums of products that float16 holds, to which every term left out or taken twice shows."""
    return ((rng.random(shape) < 0.25) * rng.choice([-1, 1], shape)).astype(np.float16)


def run(prog, arrays):
    """The program's results, in their own types."""
    be = backend()
    slots = [be.malloc(v.nbytes, np.ascontiguousarray(v).tobytes()) for v in arrays]
    outs = prog.execute(be, slots, prog.prepare(be))
    got = [np.frombuffer(be.readSync(o), np.float16) for o in outs]
    for s in slots + outs:
        be.decRef(s)
    return got


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=str)
def test_sums_of_whole_numbers_are_exact(case):
    """By the Kernel itself, and in the filter's own order by its program."""
    batch, cin, cout, h, w, kh, kw, pad = case
    kernel, cts = cotangent_kernel(*case)
    rng = np.random.default_rng(batch * h + kw)
    x, ct = sparse_integers((batch, cin, h, w), rng), sparse_integers(cts, rng)
    want, scale = reference(x, ct, kh, kw, pad)
    assert scale.max() <= 2048
    got = device_run(kernel, [x.reshape(-1), ct.reshape(-1)], filter_bands=True)[0].reshape(cin, cout, kh, kw)
    np.testing.assert_array_equal(got.astype(np.float64), want)
    own, = run(cotangent_program(*case)[0], [x, ct])
    np.testing.assert_array_equal(own.reshape(cout, cin, kh, kw).astype(np.float64), want.transpose(1, 0, 2, 3))


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(READERS))
def test_what_reads_the_cotangent_gets_it(name):
    batch, cin, cout, h, w, kh, kw, pad = case = CASES[0]
    rng = np.random.default_rng(len(name))
    cts = cotangent_program(*case)[1]
    x, ct = sparse_integers((batch, cin, h, w), rng), sparse_integers(cts, rng)
    want = READERS[name][1](reference(x, ct, kh, kw, pad)[0].transpose(1, 0, 2, 3))
    assert max(np.abs(v).max() for v in want) <= 2048
    if WARM_ONLY:
        pytest.skip("warm-up run")
    for got, w in zip(run(reader_program(name, case), [x, ct]), want):
        np.testing.assert_array_equal(got.reshape(w.shape).astype(np.float64), w)


def rounding_bound(want, n):
    """Float32 sums of n exact products of standard normals: partial sums of up to 5 sqrt(n), each addition off by at most
    2^-24 of that and by 3^-1/2 of it in the mean square, n of them at random: four deviations are 12 n 2^-24.  (A row or a column of an
    image left out changes a sum by its square root and more.)  Then one rounding to float16."""
    return np.abs(want) * 2.0 ** -11 + 12 * n * 2.0 ** -24 + 2.0 ** -25


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=str)
def test_sums_against_the_definition(case):
    batch, cin, cout, h, w, kh, kw, pad = case
    kernel, cts = cotangent_kernel(*case)
    x = RNG.standard_normal((batch, cin, h, w)).astype(np.float16)
    ct = RNG.standard_normal(cts).astype(np.float16)
    got = device_run(kernel, [x.reshape(-1), ct.reshape(-1)], filter_bands=True)[0].reshape(cin, cout, kh, kw).astype(np.float64)
    want, _ = reference(x, ct, kh, kw, pad)
    assert np.all(np.abs(got - want) <= rounding_bound(want, batch * cts[2] * cts[3]))


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES[:5] + CASES[-1:], ids=str)
def test_a_program_gets_the_filters_own_order(case):
    batch, cin, cout, h, w, kh, kw, pad = case
    prog, cts = cotangent_program(*case)
    x = RNG.standard_normal((batch, cin, h, w)).astype(np.float16)
    ct = RNG.standard_normal(cts).astype(np.float16)
    if WARM_ONLY:
        pytest.skip("warm-up run")
    got = run(prog, [x, ct])[0].reshape(cout, cin, kh, kw).astype(np.float64)
    want = reference(x, ct, kh, kw, pad)[0].transpose(1, 0, 2, 3)
    assert np.all(np.abs(got - want) <= rounding_bound(want, batch * cts[2] * cts[3]))


@pytest.mark.gpu
@pytest.mark.parametrize("size", [24, 29])
def test_infinities_and_nans_reach_the_taps_that_see_them(size):
    """A pixel or a cotangent that is no finite number spoils exactly the sums it is a term of: what lies beside a row in LDS, or
    past the end of a group of eight, is a term of none.  (Padding is a zero that is multiplied.)"""
    case = (2, 40, 40, size, size, 3, 3, SAME(3))
    kernel, cts = cotangent_kernel(*case)
    x = RNG.integers(-3, 4, (2, 40, size, size)).astype(np.float16)
    ct = RNG.integers(1, 4, cts).astype(np.float16)
    for c, (y, xx) in enumerate([(0, 0), (0, size - 1), (size - 1, 0), (size - 1, size - 1), (7, 8), (8, 7), (5, size - 1), (11, 0), (0, 12)]):
        x[c % 2, c, y, xx] = [np.inf, -np.inf, np.nan][c % 3]
    ct[0, 37, 0, 0], ct[1, 38, size - 1, size - 1] = np.inf, np.nan
    got = device_run(kernel, [x.reshape(-1), ct.reshape(-1)], filter_bands=True)[0].reshape(40, 40, 3, 3).astype(np.float64)
    want, _ = reference(x, ct, 3, 3, SAME(3))
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(got[~np.isnan(want)], want[~np.isnan(want)].astype(np.float16).astype(np.float64))


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(2, 64, 64, 12, 3), (3, 128, 64, 10, 3)], ids=str)
def test_weights_of_several_convolutions_are_laid_out_by_one_launch(shape):
    """Two convolutions of the same Kernel over different filters, one behind them, a cotangent that reads its filter flipped, and
    one whose filter the program computes (it keeps its own pre-pass); small integers, twice over with the filters exchanged."""
    from jaxjs_hip.composite import Weights
    from jaxjs_hip.schedule import Schedule
    from jit_util import run_program
    B, C, O, S, K = shape
    p, q = ConvParams(0, [1, 1], [(K // 2, K // 2)] * 2, [1, 1], [1, 1]), ConvParams(0, [1, 1], [(0, 0)] * 2, [1, 1], [1, 1])
    rng = np.random.default_rng(C)
    x = rng.integers(-1, 2, (B, C, S, S)).astype(np.float16)
    w1, w2 = (((rng.random((O, C, K, K)) < 0.2) * rng.integers(-1, 2, (O, C, K, K))).astype(np.float16) for _ in range(2))
    w3 = ((rng.random((64, O, 1, 1)) < 0.1) * rng.integers(-1, 2, (64, O, 1, 1))).astype(np.float16)

    def f(x, w1, w2, w3):
        a, b = J.conv(x, w1, p), J.conv(x, w2, p)
        return [a, b, J.conv(a, w3, q), J.convTransposeLhs(b, w2, [B, C, S, S], p), J.conv(x, w1.mul(2.0).add(w2), p)]

    def same(x, w):  # whole numbers: every sum is exact
        windows = np.lib.stride_tricks.sliding_window_view(np.pad(x, [(0, 0)] * 2 + [(w.shape[2] // 2,) * 2] * 2), w.shape[2:], (2, 3))
        return np.tensordot(windows, w, ([1, 4, 5], [1, 2, 3])).transpose(0, 3, 1, 2)
    prog = J.jit(f, [ShapedArray(v.shape, DType.Float16) for v in (x, w1, w2, w3)])
    if WARM_ONLY:
        pytest.skip("warm-up run")
    sch = Schedule(backend(), prog)
    assert isinstance(sch.units[0].source, Weights) and len(sch.units[0].outputs) == 3 and sum(isinstance(u.source, Weights) for u in sch.units) == 1
    assert len({u.early for u in sch.units if u.early is not None}) == len(sch.units[0].outputs)
    before = backend().live_slots()
    for arrays in ([x, w1, w2, w3], [x, w2, w1, w3]):
        got = run_program(backend(), prog, arrays)
        vx, v1, v2, v3 = (v.astype(np.float32) for v in arrays)
        a, b = same(vx, v1), same(vx, v2)
        want = [a, b, same(a, v3), same(b, v2.transpose(1, 0, 2, 3)[:, :, ::-1, ::-1]), same(vx, 2 * v1 + v2)]
        for u, v in zip(got, want):
            assert np.abs(v).max() <= 2048
            np.testing.assert_array_equal(u.astype(np.float32), v.reshape(u.shape))
    assert backend().live_slots() == before


def image_cotangent(B, C, O, S, K):
    p = ConvParams(0, [1, 1], [(K // 2, K // 2)] * 2, [1, 1], [1, 1])
    rng = np.random.default_rng(B * C + S)
    ct, w = (rng.integers(-3, 4, s).astype(np.float16) for s in ((B, O, S, S), (O, C, K, K)))
    prog = J.jit(lambda ct, w: [J.convTransposeLhs(ct, w, [B, C, S, S], p)], [ShapedArray(v.shape, DType.Float16) for v in (ct, w)])
    return next(s.kernel for s in prog.steps if s.kind == "execute"), ct, w


@pytest.mark.parametrize("shape,patch", [((2, 128, 128, 14, 3), True), ((3, 64, 64, 13, 5), True), ((2, 64, 256, 10, 3), True), ((4, 64, 192, 14, 5), False), ((24, 64, 192, 14, 5), False),
                                         ((48, 64, 192, 14, 5), True)], ids=str)
def test_the_cotangent_towards_the_image_is_left_whole(shape, patch):
    """Both sides of the rule: up to k = 4096, and behind it by the number of tiles."""
    kernel, *_ = image_cotangent(*shape)
    assert (generate(kernel, "fast").info.get("conv") is not None) == patch


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(2, 128, 128, 14, 3), (3, 64, 64, 13, 5), (2, 64, 256, 10, 3), (2, 64, 128, 7, 3)], ids=str)
def test_the_cotangent_towards_the_image_by_patches(shape):
    """Small integers: every sum is exact up to its rounding to float16."""
    B, C, O, S, K = shape
    kernel, ct, w = image_cotangent(*shape)
    got = device_run(kernel, [v.reshape(-1) for v in (ct, w)])[0].reshape(B, C, S, S)
    windows = np.lib.stride_tricks.sliding_window_view(np.pad(ct.astype(np.float32), [(0, 0)] * 2 + [(K // 2,) * 2] * 2), (K, K), (2, 3))
    want = np.tensordot(windows, w.astype(np.float32).transpose(1, 0, 2, 3)[:, :, ::-1, ::-1], ([1, 4, 5], [1, 2, 3])).transpose(0, 3, 1, 2)
    np.testing.assert_array_equal(got, want.astype(np.float16))
