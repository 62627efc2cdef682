"""Scatter, TriangularSolve, Cholesky, LU, JacobiEigh and Fft as GPU kernels against the CPU checker.

The linear-algebra kernels keep the reference's arithmetic (double scalars, stores rounded to the element type --
float32, float64 or float16 --, the same order per stored element), so their results must be bit-identical to the checker's.  Scatter is bit-identical except float
accumulation onto repeated destinations (atomic adds in any order: compared within a sum-scaled bound).  Fft takes
its sines and cosines from the device math library, whose last-place differences from the host's can decide a
float32 rounding tie in a butterfly (seen for radix-3 stages behind an even stride; power-of-two and prime sizes come
out bit-identical): compared within 1e-5 of the row's largest magnitude."""
import itertools
import math

import numpy as np
import pytest

import routine_util as R
from jaxjs_hip import DType
from jaxjs_hip.errors import UnsupportedRoutineError

pytestmark = pytest.mark.gpu
RNG = np.random.default_rng(77)
F32 = np.float32


def both(routine, arrays):
    got, ks = R.run_gpu(routine, arrays)
    return got, R.run_oracle(routine, arrays), ks


def assert_bits(got, want, what=""):
    for i, (g, w) in enumerate(zip(got, want)):
        if not R.bits_equal(g, w):
            bad = np.flatnonzero((g.reshape(-1) != w.reshape(-1)) & ~(np.isnan(g.reshape(-1)) & np.isnan(w.reshape(-1)))) if g.dtype.kind == "f" else np.flatnonzero(g.reshape(-1) != w.reshape(-1))
            raise AssertionError(f"{what} output {i}: {len(bad)} of {g.size} elements differ; first at {bad[:5]}: "
                                 f"{g.reshape(-1)[bad[:5]]} vs {w.reshape(-1)[bad[:5]]}")


def spd(batch, n):
    a = RNG.standard_normal(batch + (n, n))
    return (a @ np.swapaxes(a, -1, -2) + n * np.eye(n)).astype(F32)


@pytest.mark.parametrize("shape", [(1, 1), (2, 2), (3, 3), (5, 17, 17), (2, 3, 64, 64), (191, 191), (192, 192), (200, 200), (2, 333, 333),
                                   (1100, 1100), (2048, 2048)], ids=str)
def test_cholesky(shape):
    x = spd(tuple(shape[:-2]), shape[-1])
    x = x + np.triu(RNG.standard_normal(x.shape), 1).astype(F32)  # the upper triangle must not matter
    got, want, ks = both(R.cholesky(x), [x])
    assert ("panels" in ks.info) == (shape[-1] >= 192)  # large matrices run panel by panel over the whole chip
    assert_bits(got, want, f"cholesky {shape} {ks.info}")


@pytest.mark.parametrize("shape", [(200, 200), (2, 333, 333), (1100, 1100)], ids=str)
def test_cholesky_left_looking_panels_when_the_double_copy_is_too_large(shape, monkeypatch):
    """The right-looking variant keeps a double-precision copy of every matrix; beyond its size limit the left-looking
    panels run instead.  Same sums in the same order: identical bits."""
    from jaxjs_hip import routinegen
    x = spd(tuple(shape[:-2]), shape[-1])
    right, k1 = R.run_gpu(R.cholesky(x), [x])
    monkeypatch.setattr(routinegen, "CHOLESKY_RIGHT_LOOKING_MAX_BYTES", 0)
    from gpu_util import backend
    backend().clearCache()  # prepared routines are cached by structure: the limit is read when a plan is generated
    left, k2 = R.run_gpu(R.cholesky(x), [x])
    backend().clearCache()
    assert k1.info.get("variant") == "right-looking" and "variant" not in k2.info and "panels" in k2.info
    assert_bits(left, right, f"cholesky variants {shape}")


@pytest.mark.parametrize("dt", [F32, np.float16, np.float64], ids=lambda d: np.dtype(d).name)
@pytest.mark.parametrize("n", [9, 32, 33, 70])
def test_cholesky_pivots_that_are_no_ordinary_numbers(n, dt):
    """Roots and quotients without the compiler's scaling and special cases: zero, negative, infinite and undefined pivots, and
    elements at either end of the range, in the first columns, inside a panel, at its end and behind it."""
    x = RNG.standard_normal((8, n, n))
    base = (x @ np.swapaxes(x, -1, -2) / n + np.eye(n)).astype(dt)
    tiny, big = np.finfo(dt).tiny, np.finfo(dt).max
    mats = []
    for at in sorted({0, 1, 2, 3, n // 2, min(31, n - 1), n - 1}):
        for value in (0.0, -0.0, -1.0, np.inf, -np.inf, np.nan, tiny, tiny / 4, big):
            m = base[at % 8].copy()
            m[at, at] = value
            if value in (0.0, -1.0):
                m[at, :at] = m[:at, at] = 0
            mats.append(m)
    scales = [tiny / 8, tiny * 4, big / 64]
    with np.errstate(over="ignore", under="ignore"):
        mats += [(base[i].astype(np.float64) * s).astype(dt) for i, s in enumerate(scales)]
    a = np.stack(mats)
    got, want, _ = both(R.cholesky(a), [a])
    assert_bits(got, want, f"cholesky {n} {np.dtype(dt).name}")


def _squares(total, bits):
    """Whole numbers of at most `bits` bits whose squares add up to `total`, the larger ones first."""
    parts = []
    while total > 4000:
        m = math.isqrt(total)
        low = max(0, m.bit_length() - bits)
        parts.append(m >> low << low)
        total -= parts[-1] ** 2
    for a, b, c in itertools.product(range(math.isqrt(total) + 1), repeat=3):
        d = total - a * a - b * b - c * c
        if d >= 0 and math.isqrt(d) ** 2 == d:
            return parts + [a, b, c, math.isqrt(d)]


@pytest.mark.parametrize("dt,bits", [(F32, 24), (np.float16, 11)], ids=["float32", "float16"])
@pytest.mark.parametrize("before", [0, 5, 26, 40])
def test_cholesky_pivots_whose_root_is_subnormal(before, dt, bits):
    """A pivot that products cancel down to a few units of the product of two smallest numbers: its rounded root is far from the
    root itself (1 for 1.41), and the quotients below are by the rounded one.  Inside a panel, across two and in the second."""
    unit = 2.0 ** -149 if dt == F32 else 2.0 ** -24  # smallest number of the type
    mats, pivots = [], []
    for left in (1, 2, 3, 5, 6, 7, 30, 200, 2000):  # what is left of the pivot, in units squared
        parts = _squares(int(1 / unit) - left, bits)
        p = before + len(parts)
        a = np.eye(before + 48)
        a[p, before:p] = np.array(parts, dtype=np.float64) * unit
        a[p, p] = unit
        a[p + 1:, before] = -unit * np.arange(1, len(a) - p)
        mats.append(a.astype(dt))
        pivots.append((p, dt(math.sqrt(left) * unit)))
    a = np.stack(mats)
    got, want, _ = both(R.cholesky(a), [a])
    assert np.isfinite(want[0]).all() and [w[p, p] for w, (p, _) in zip(want[0], pivots)] == [v for _, v in pivots]
    assert_bits(got, want, f"cholesky {a.shape} {np.dtype(dt).name}")


def test_cholesky_not_positive_definite_and_empty():
    x = np.array([[[1, 2], [2, 1]], [[4, 2], [2, 3]]], F32)
    got, want, _ = both(R.cholesky(x), [x])
    assert np.isnan(got[0][0, 1, 1]) and got[0][1, 1, 1] == np.float32(np.sqrt(2.0))
    assert_bits(got, want)
    big = spd((), 256)
    big[100, 100] = -5.0  # pivot 100 goes negative: NaNs from there on, in the same places, also panel by panel
    got, want, ks = both(R.cholesky(big), [big])
    assert "panels" in ks.info and np.isnan(got[0][100, 100]) and np.isfinite(got[0][:100, :100]).all()
    assert_bits(got, want, "non-PD through panels")
    e = np.zeros((0, 4, 4), F32)
    got, _ = R.run_gpu(R.cholesky(e), [e])
    assert got[0].shape == (0, 4, 4)
    with pytest.raises(ValueError):
        R.run_gpu(R.cholesky(np.zeros((2, 3), F32)), [np.zeros((2, 3), F32)])


@pytest.mark.parametrize("case", [((2, 2), 1), ((9, 9), 4), ((3, 30, 30), 7), ((2, 2, 16, 16), 100), ((300, 300), 300), ((64, 64), 1000),
                                  ((2, 131, 131), 70), ((128, 128), 3), ((1024, 1024), 64)], ids=str)
@pytest.mark.parametrize("unit", [False, True])
def test_triangular_solve(case, unit):
    ashape, m = case
    n = ashape[-1]
    a = (np.triu(RNG.standard_normal(ashape)) * (0.3 if unit else 1.0) + (0 if unit else 1) * np.sqrt(n) * np.eye(n)
         + np.tril(RNG.standard_normal(ashape), -1)).astype(F32)  # the strictly lower part must not matter
    b = RNG.standard_normal(ashape[:-2] + (m, n)).astype(F32)
    got, want, ks = both(R.triangular_solve(a, b, unit), [a, b])
    assert ks.info["variant"] == "few"
    assert_bits(got, want, f"triangular_solve {case} {ks.info}")


@pytest.mark.parametrize("shape", [(2, 2), (1, 5), (5, 1), (2, 7, 5), (3, 12, 20), (2, 2, 30, 30), (150, 97), (260, 300), (255, 400),
                                   (2, 300, 256), (513, 300), (1024, 1024)], ids=str)
def test_lu(shape):
    a = RNG.uniform(-1, 1, shape).astype(F32)
    got, want, ks = both(R.lu(a), [a])
    assert ks.info["variant"] == ("by matrix" if shape == (1, 5) else "by panels")
    assert_bits(got, want, f"lu {shape} {ks.info}")


@pytest.mark.parametrize("shape,dt", [((2, 260, 260), F32), ((1, 4100, 200), F32), ((2, 4099, 193), F32), ((1, 4100, 200), np.float64), ((1, 4100, 200), np.float16)],
                         ids=lambda v: np.dtype(v).name if isinstance(v, type) else str(v))
def test_lu_zero_pivot_and_nan_columns_of_larger_matrices(shape, dt):
    """The special cases of the test below, in panels and, of more than 4096 rows, column by column: a zero pivot column
    (that step eliminates nothing), equal magnitudes (the first row wins), a NaN that must not win."""
    a = RNG.uniform(-1, 1, shape).astype(dt)
    a[0, :, 3] = 0.0   # stays zero through every update: step 3 meets a zero pivot
    a[-1, 10, 5] = np.nan
    a[-1, 20:23, 7] = [0.75, -0.75, 0.75]
    a[-1, :, 11] = np.sign(a[-1, :, 11])
    got, want, ks = both(R.lu(a), [a])
    assert ks.info["variant"] == ("by panels" if shape[1] <= 4096 else "by columns")
    assert_bits(got, want, "lu, special columns")


def test_lu_ties_zero_pivots_and_nans():
    a = np.array([[[1, 2, 3], [-1, 5, 6], [1, 8, 9]],      # equal magnitudes: the first row wins
                  [[0, 1, 2], [0, 2, 3], [0, 5, 1]],       # zero pivot column: nothing eliminated in that step
                  [[np.nan, 1, 2], [3, 2, 3], [4, 5, 1]],  # NaN in the starting row keeps it
                  [[1, 1, 2], [np.nan, 2, 3], [4, 5, 1]]], F32)  # NaN elsewhere never wins
    got, want, _ = both(R.lu(a), [a])
    assert_bits(got, want, "lu special rows")
    got, want, _ = both(R.lu(np.zeros((2, 3, 0), F32)), [np.zeros((2, 3, 0), F32)])
    assert got[2].tolist() == [[0, 1, 2]] * 2
    assert_bits(got, want)


@pytest.mark.parametrize("shape", [(1, 1), (2, 2), (3, 3), (4, 20, 20), (2, 64, 64), (100, 100), (2, 128, 128), (150, 150)], ids=str)
def test_jacobi_eigh(shape):
    a = RNG.standard_normal(shape)
    sym = (a + np.swapaxes(a, -1, -2)).astype(F32) + np.triu(RNG.standard_normal(shape), 1).astype(F32)
    got, want, ks = both(R.jacobi_eigh(sym), [sym])
    assert ks.info["in_lds"] == (shape[-1] <= 138)
    assert_bits(got, want, f"jacobi_eigh {shape} {ks.info}")


@pytest.mark.parametrize("n", [12, 13, 15, 17, 65, 129, 139, 160])
def test_jacobi_eigh_by_blocks_at_ragged_orders(n):
    """Partial last blocks, one to three waves of chains, both block sizes; and pairs that are left alone (zeros, negative
    zeros among them) beside pairs that turn."""
    a = RNG.standard_normal((2, n, n))
    sym = (a + np.swapaxes(a, -1, -2)).astype(F32)
    sym[1, : n // 2, n // 2:] = sym[1, n // 2:, : n // 2] = -0.0
    sym[1, 1, :1] = sym[1, :1, 1] = 0.0
    got, want, ks = both(R.jacobi_eigh(sym, 3, 0.0), [sym])
    assert ("block" in ks.info) == (n >= 13)
    assert_bits(got, want, f"jacobi_eigh {n} {ks.info}")


@pytest.mark.parametrize("dt", [np.float16, F32, np.float64], ids=lambda d: np.dtype(d).name)
@pytest.mark.parametrize("n", [16, 31, 35, 61, 64, 65])
def test_jacobi_eigh_by_blocks_around_half_a_wave_per_block(n, dt):
    """Fewer rows above a block than half a wave has lanes, as many, more; a partial last block; the order behind."""
    a = RNG.standard_normal((2, n, n))
    sym = (a + np.swapaxes(a, -1, -2)).astype(dt)
    got, want, ks = both(R.jacobi_eigh(sym, 2, 0.0), [sym])
    assert ks.info["block"] == 4
    assert_bits(got, want, f"jacobi_eigh {n} {np.dtype(dt).name}")


@pytest.mark.parametrize("scale", [1e-44, 1e-30, 1e30, 1e38])
@pytest.mark.parametrize("n", [14, 65])
def test_jacobi_eigh_at_the_ends_of_the_element_range(n, scale):
    """Rotations without scaled quotients: elements that are denormal, and elements that overflow on the way (the result then
    holds infinities and NaNs, the same ones); a widely graded diagonal makes the smallest and largest angles."""
    a = RNG.uniform(-1, 1, (3, n, n)) * 10.0 ** RNG.integers(-6, 1, (3, 1, n))
    a[2] += np.diag(3.0 * 10.0 ** RNG.integers(-12, 1, n))
    with np.errstate(over="ignore"):
        sym = ((a + np.swapaxes(a, -1, -2)) * scale).astype(F32)
    got, want, _ = both(R.jacobi_eigh(sym, 4, 0.0), [sym])
    assert_bits(got, want, f"jacobi_eigh {n} scale {scale}")


def test_jacobi_eigh_sweep_limits_and_special_values():
    a = RNG.standard_normal((3, 12, 12))
    sym = (a + np.swapaxes(a, -1, -2)).astype(F32)
    for sweeps, tol in ((0, 1e-7), (1, 1e-7), (2, 0.0), (30, 1e-3)):
        got, want, _ = both(R.jacobi_eigh(sym, sweeps, tol), [sym])
        assert_bits(got, want, f"maxSweeps={sweeps} tolerance={tol}")
    d = np.diag(np.array([3, 1, 2], F32))
    got, want, _ = both(R.jacobi_eigh(d), [d])
    assert np.diagonal(got[0]).tolist() == [3, 1, 2]
    assert_bits(got, want)
    bad = sym.copy()
    bad[1, 5, 2] = np.nan  # a NaN makes the threshold NaN: no sweep runs (Math.max propagates it)
    got, want, _ = both(R.jacobi_eigh(bad), [bad])
    assert_bits(got, want, "NaN input")


@pytest.mark.parametrize("n", [1, 2, 3, 4, 8, 12, 30, 49, 64, 11, 97, 210, 1024, 4096, 1009])
@pytest.mark.parametrize("inverse", [False, True])
def test_fft(n, inverse):
    rows = (2, 3) if n < 1000 else (3,)
    re, im = RNG.standard_normal(rows + (n,)).astype(F32), RNG.standard_normal(rows + (n,)).astype(F32)
    got, want, ks = both(R.fft(re, im, inverse), [re, im])
    scale = max(np.abs(want[0]).max(), np.abs(want[1]).max())
    for g, w in zip(got, want):
        np.testing.assert_allclose(g, w, rtol=0, atol=1e-5 * scale, err_msg=str(ks.info))


@pytest.mark.parametrize("shape", [(3, 8), (2, 60), (1, 1000), (5, 1024), (70, 4096), (2, 8192)], ids=str)
def test_fft_single_launch_and_staged_paths_give_the_same_bits(shape):
    """Short rows run in one launch with the stages in LDS, long or few rows one launch per stage through HBM: the
    same operations per element in the same order, so not a bit may differ (forward and inverse)."""
    from jaxjs_hip.routine import Routine
    re, im = RNG.standard_normal(shape).astype(F32), RNG.standard_normal(shape).astype(F32)
    for inverse in (False, True):
        base = R.fft(re, im, inverse)
        one = Routine(base.name, base.type, dict(base.params, singleLaunch=True))
        many = Routine(base.name, base.type, dict(base.params, singleLaunch=False))
        a, ka = R.run_gpu(one, [re, im])
        b, kb = R.run_gpu(many, [re, im])
        assert ka.info["launches"] == 1 and kb.info["launches"] == 1 + len(base.params["factors"])
        assert_bits(a, b, f"{shape} inverse={inverse}")


@pytest.mark.parametrize("shape", [(2,), (3, 16), (5, 143), (9, 2310), (1, 8192), (300, 4096), (2, 12288), (3, 70875), (1, 4 * 11 * 13 * 49), (1, 1 << 23)], ids=str)
@pytest.mark.parametrize("dt", [F32, np.float64, np.float16], ids=lambda d: np.dtype(d).name)
def test_fft_in_passes(shape, dt):
    """One, two and three passes over memory, lone and many rows, every butterfly size, against numpy in double."""
    if dt != F32 and shape[-1] > 100000:
        pytest.skip("the pass structure does not depend on the element type")
    re, im = RNG.standard_normal(shape).astype(dt), RNG.standard_normal(shape).astype(dt)
    for inverse in (False, True):
        got, ks = R.run_gpu(R.fft(re, im, inverse), [re, im])
        z = re.astype(np.complex128) + 1j * im.astype(np.complex128)
        want = np.fft.ifft(z) if inverse else np.fft.fft(z)
        err = np.abs(got[0].astype(np.complex128) + 1j * got[1] - want).max() / np.abs(want).max()
        assert "passes" in ks.info and err < {"float32": 5e-7, "float64": 1e-14, "float16": 2e-3}[np.dtype(dt).name], (ks.info, err)


@pytest.mark.parametrize("shape", [(1, 6), (3, 9), (2, 10), (5, 12), (1, 14), (7, 15), (2, 90), (3, 140 * 15), (2, 120), (3, 12 * 12 * 9), (2, 8000), (1, 10 * 12 * 14 * 15), (2, 9 ** 5)], ids=str)
def test_fft_butterflies_made_of_two_smaller_ones(monkeypatch, shape):
    """Every such size first, last and alone, and more butterflies than threads, also where a length of so few rows keeps to
    the smaller ones by itself."""
    from jaxjs_hip import routinegen
    monkeypatch.setattr(routinegen, "_fft_stages", lambda L, *rest: routinegen._fft_fewest(L) if L > 1 else [1])
    re, im = RNG.standard_normal(shape).astype(F32), RNG.standard_normal(shape).astype(F32)
    for inverse in (False, True):
        got, ks = R.run_gpu(R.fft(re, im, inverse), [re, im])
        z = re.astype(np.complex128) + 1j * im.astype(np.complex128)
        want = np.fft.ifft(z) if inverse else np.fft.fft(z)
        # a rounding to float32 a stage, of values as large as the result's, over a handful of stages
        assert np.abs(got[0].astype(np.complex128) + 1j * got[1] - want).max() <= 5e-7 * np.abs(want).max(), ks.info


def test_fft_factor_orders_and_validation():
    re, im = RNG.standard_normal((2, 60)).astype(F32), RNG.standard_normal((2, 60)).astype(F32)
    for factors in ([4, 3, 5], [5, 3, 4], [2, 2, 15], [60]):
        got, want, _ = both(R.fft(re, im, False, factors), [re, im])
        for g, w in zip(got, want):
            np.testing.assert_allclose(g, w, rtol=0, atol=1e-5 * np.abs(w).max())
    with pytest.raises(ValueError):
        R.run_gpu(R.fft(re, im, False, [4, 4]), [re, im])


# ---- float64 and float16 elements: the same kernels with another stored type (every kernel variant once per type)
ELEMS = [np.float64, np.float16]


@pytest.mark.parametrize("dt", ELEMS, ids=lambda d: np.dtype(d).name)
@pytest.mark.parametrize("shape", [(3, 3), (2, 3, 64, 64), (200, 200), (2, 333, 333)], ids=str)
def test_cholesky_other_element_types(shape, dt, monkeypatch):
    n = shape[-1]
    x = (spd(tuple(shape[:-2]), n).astype(np.float64) / (1.0 if dt == np.float64 else n)).astype(dt)
    got, want, ks = both(R.cholesky(x), [x])
    assert got[0].dtype == dt and ("panels" in ks.info) == (n >= 192)
    assert_bits(got, want, f"cholesky {shape} {np.dtype(dt).name} {ks.info}")
    if n >= 192:  # and the left-looking panels
        from jaxjs_hip import routinegen
        from gpu_util import backend
        monkeypatch.setattr(routinegen, "CHOLESKY_RIGHT_LOOKING_MAX_BYTES", 0)
        backend().clearCache()
        left, k2 = R.run_gpu(R.cholesky(x), [x])
        backend().clearCache()
        assert "variant" not in k2.info and "panels" in k2.info
        assert_bits(left, want, f"cholesky left-looking {shape} {np.dtype(dt).name}")


@pytest.mark.parametrize("dt", ELEMS, ids=lambda d: np.dtype(d).name)
@pytest.mark.parametrize("case", [((9, 9), 4), ((2, 2, 16, 16), 100), ((2, 131, 131), 70), ((300, 300), 300)], ids=str)
@pytest.mark.parametrize("unit", [False, True])
def test_triangular_solve_other_element_types(case, unit, dt):
    ashape, m = case
    n = ashape[-1]
    a = (np.triu(RNG.standard_normal(ashape)) * (0.3 if unit else 1.0) + (0 if unit else 1) * np.sqrt(n) * np.eye(n)
         + np.tril(RNG.standard_normal(ashape), -1)).astype(dt)
    b = RNG.standard_normal(ashape[:-2] + (m, n)).astype(dt)
    got, want, ks = both(R.triangular_solve(a, b, unit), [a, b])
    assert got[0].dtype == dt and ks.info["variant"] == "few"
    assert_bits(got, want, f"triangular_solve {case} {np.dtype(dt).name} {ks.info}")


@pytest.mark.parametrize("dt", ELEMS, ids=lambda d: np.dtype(d).name)
@pytest.mark.parametrize("shape", [(2, 7, 5), (3, 12, 20), (150, 97), (260, 300), (2, 300, 256)], ids=str)
def test_lu_other_element_types(shape, dt):
    a = RNG.uniform(-1, 1, shape).astype(dt)
    if shape == (260, 300):
        a[:, 3] = 0       # a zero pivot column
        a[10, 5] = np.nan  # a NaN that must not win the pivot search
        a[20:23, 7] = [0.75, -0.75, 0.75]
    got, want, ks = both(R.lu(a), [a])
    assert got[0].dtype == dt and ks.info["variant"] == "by panels"
    assert_bits(got, want, f"lu {shape} {np.dtype(dt).name} {ks.info}")


@pytest.mark.parametrize("dt", ELEMS, ids=lambda d: np.dtype(d).name)
@pytest.mark.parametrize("shape", [(2, 2), (4, 20, 20), (2, 64, 64), (100, 100), (150, 150)], ids=str)
def test_jacobi_eigh_other_element_types(shape, dt):
    a = RNG.standard_normal(shape)
    sym = (a + np.swapaxes(a, -1, -2)).astype(dt) + np.triu(RNG.standard_normal(shape), 1).astype(dt)
    tol = 1e-14 if dt == np.float64 else 1e-3
    got, want, ks = both(R.jacobi_eigh(sym, 30 if dt == np.float64 else 6, tol), [sym])
    eb = np.dtype(dt).itemsize
    assert got[0].dtype == dt and ks.info["in_lds"] == (2 * shape[-1] ** 2 * eb <= 150 * 1024)
    assert_bits(got, want, f"jacobi_eigh {shape} {np.dtype(dt).name} {ks.info}")


@pytest.mark.parametrize("dt", ELEMS, ids=lambda d: np.dtype(d).name)
@pytest.mark.parametrize("n", [1, 4, 12, 49, 97, 210, 1024, 4096])
def test_fft_other_element_types(n, dt):
    """float64 results carry the device sine/cosine's last-place differences from the host's unrounded: compared within
    1e-13 of the row's magnitude per stage; float16 within one unit of its last place of that magnitude."""
    from jaxjs_hip.routine import Routine
    rows = (2, 3) if n < 1000 else (70,)
    re, im = RNG.standard_normal(rows + (n,)).astype(dt), RNG.standard_normal(rows + (n,)).astype(dt)
    for inverse in (False, True):
        base = R.fft(re, im, inverse)
        got, want, ks = both(base, [re, im])
        scale = float(max(np.abs(want[0].astype(np.float64)).max(), np.abs(want[1].astype(np.float64)).max()))
        atol = (1e-13 * max(1, len(base.params["factors"])) if dt == np.float64 else 1e-3) * scale
        for g, w in zip(got, want):
            assert g.dtype == dt
            np.testing.assert_allclose(g.astype(np.float64), w.astype(np.float64), rtol=0, atol=atol, err_msg=str(ks.info))
        if n <= (4096 if dt == np.float64 else 8192) and n > 1:  # single launch and one launch per stage: the same bits
            one = Routine(base.name, base.type, dict(base.params, singleLaunch=True))
            many = Routine(base.name, base.type, dict(base.params, singleLaunch=False))
            a, ka = R.run_gpu(one, [re, im])
            b, kb = R.run_gpu(many, [re, im])
            assert ka.info["launches"] == 1 and kb.info["launches"] == 1 + len(base.params["factors"])
            assert_bits(a, b, f"fft paths n={n} {np.dtype(dt).name} inverse={inverse}")


def _sc(updates, indices, op, shape, axis, out_dim, unique=False, dtype=None):
    return R.scatter(updates, indices, op, shape, axis, out_dim, unique, dtype), [updates] + list(indices)


def test_scatter_reference_tables():
    i32 = lambda x: np.array(x, np.int32)  # noqa: E731
    cases = [
        _sc(np.array([[10, 20], [30, 40], [50, 60]], F32), [i32([1, 3]), i32([0, 1])], "update", [2, 3, 4], [2, 0], 1, True),
        _sc(np.array([1, 2, 3], F32), [i32([1, 1, 3])], "add", [4], [0], 0),
        _sc(np.array([1, 2, 3, 4], np.float16), [i32([0, 1, 0, 1])], "add", [2], [0], 0),
        _sc(np.array([1, 2, 3], np.int32), [i32([1, 1, 3])], "add", [4], [0], 0),
        _sc(np.array([1, 2, 3], np.uint32), [i32([1, 1, 3])], "add", [4], [0], 0),
        _sc(np.array([0, 1, 1], np.int32), [i32([1, 1, 3])], "add", [4], [0], 0, dtype=DType.Bool),
        _sc(np.array([10, 20, 30], F32), [i32([3, 0, 2])], "add", [4], [0], 0, True),
        _sc(np.array([[1, 2, 3], [4, 5, 6]], F32), [i32([[0], [2]]), i32([[0, 1, 1]])], "add", [3, 4], [0, 1], 0),
    ]
    expected = [[[[0, 10, 0, 0], [0, 30, 0, 0], [0, 50, 0, 0]], [[0, 0, 0, 20], [0, 0, 0, 40], [0, 0, 0, 60]]],
                [0, 3, 0, 3], [4, 6], [0, 3, 0, 3], [0, 3, 0, 3], [0, 1, 0, 1], [20, 0, 30, 10],
                [[1, 5, 0, 0], [0, 0, 0, 0], [4, 11, 0, 0]]]
    for (routine, arrays), exp in zip(cases, expected):
        got, want, _ = both(routine, arrays)
        np.testing.assert_array_equal(got[0], np.array(exp))
        assert_bits(got, want)


SCATTER_CASES = [
    ((7,), [(7,)], (5,), [0], 0),
    ((6, 3), [(6,)], (4, 3), [0], 0),
    ((3, 6), [(6,)], (3, 4), [1], 1),
    ((2, 5, 3), [(5,), (5,)], (2, 4, 6, 3), [1, 2], 1),
    ((4, 3, 2), [(4, 1), (1, 3)], (5, 2, 5), [2, 0], 0),
    ((2, 2, 3, 2), [(2, 3)], (2, 6, 2), [1], 1),
    ((5000, 8), [(5000,)], (300, 8), [0], 0),       # many repeated destinations
    ((100000,), [(100000,)], (1000003,), [0], 0),   # sparse
]


@pytest.mark.parametrize("case", SCATTER_CASES, ids=lambda c: "x".join(map(str, c[0])))
@pytest.mark.parametrize("op", ["add", "update"])
@pytest.mark.parametrize("dtype", [DType.Float32, DType.Int32, DType.Uint32, DType.Float16, DType.Bool, DType.Float64], ids=lambda d: d.value)
def test_scatter_random(case, op, dtype):
    ushape, ishapes, oshape, axis, out_dim = case
    npdt = {DType.Float32: F32, DType.Int32: np.int32, DType.Uint32: np.uint32, DType.Float16: np.float16, DType.Bool: np.int32,
            DType.Float64: np.float64}[dtype]
    if dtype == DType.Bool:
        upd = RNG.integers(0, 2, ushape).astype(npdt)
    elif dtype in (DType.Int32, DType.Uint32):
        upd = RNG.integers(0, 1 << 32, ushape, dtype=np.uint64).astype(np.uint32).view(npdt).reshape(ushape)  # sums wrap
    else:
        upd = RNG.integers(-9, 10, ushape).astype(npdt)  # small integers: float sums are exact in any order
    idx = [RNG.integers(-1, oshape[a] + 1, s).astype(np.int32) for s, a in zip(ishapes, axis)]  # some out of range
    got, want, ks = both(*_sc(upd, idx, op, list(oshape), axis, out_dim, dtype=dtype))
    assert_bits(got, want, f"scatter {case} {op} {dtype} {ks.info}")


def test_scatter_float_accumulation_within_bound_and_unique_promise():
    upd = RNG.standard_normal((20000,)).astype(F32)
    idx = RNG.integers(0, 50, (20000,)).astype(np.int32)
    got, want, _ = both(*_sc(upd, [idx], "add", [50], [0], 0))
    bound = np.zeros(50)
    np.add.at(bound, idx, np.abs(upd))
    assert np.all(np.abs(got[0].astype(np.float64) - want[0]) <= 400 * 2.0 ** -24 * bound + 1e-30)  # ~K/50 adds per slot
    perm = RNG.permutation(1000).astype(np.int32)
    vals = RNG.standard_normal((1000, 4)).astype(F32)
    for op in ("add", "update"):
        got, want, ks = both(*_sc(vals, [perm], op, [1000, 4], [0], 0, True))
        assert ks.info["mode"] == 0
        assert_bits(got, want)
    with pytest.raises(UnsupportedRoutineError):
        R.run_gpu(*_sc(np.zeros(3, F32), [np.zeros(3, F32)], "add", [4], [0], 0))  # index arrays must be integers


def test_outputs_are_fully_initialised_without_updates():
    got, want, _ = both(*_sc(np.zeros((0, 3), F32), [np.zeros((0,), np.int32)], "add", [4, 3], [0], 0))
    assert np.all(got[0] == 0)
    assert_bits(got, want)


@pytest.mark.parametrize("shape,dt", [((70, 1, 1), F32), ((5, 9, 9), F32), ((2, 3, 27, 27), F32), ((64, 64), F32), ((3, 8, 8), np.float64),
                                      ((2, 27, 27), np.float64), ((2, 43, 43), np.float16), ((4, 63, 63), np.float16)], ids=str)
def test_cholesky_with_a_wave_per_matrix(shape, dt, monkeypatch):
    """The plan of many small matrices, at every order that a wave can hold a row per lane of: the checker's bits."""
    from gpu_util import WARM_ONLY, backend
    from jaxjs_hip import routinegen
    n = shape[-1]
    x = (spd(tuple(shape[:-2]), n).astype(np.float64) / n + np.triu(RNG.standard_normal(shape), 1)).astype(dt)
    monkeypatch.setattr(routinegen, "_cholesky_plan", lambda *a: "wave per matrix")
    if not WARM_ONLY:
        backend().clearCache()  # prepared routines are cached by structure
    got, want, ks = both(R.cholesky(x), [x])
    backend().clearCache()
    assert [s.name for s in ks.steps] == ["jh_cholesky"]
    assert_bits(got, want, f"cholesky {shape} {np.dtype(dt).name}")


@pytest.mark.parametrize("shape,dt", [((192, 192), F32), ((2, 333, 333), F32), ((3, 200, 200), np.float64), ((2, 333, 333), np.float16)], ids=str)
def test_cholesky_with_two_launches_per_panel(shape, dt, monkeypatch):
    from gpu_util import WARM_ONLY, backend
    from jaxjs_hip import routinegen
    n = shape[-1]
    x = (spd(tuple(shape[:-2]), n).astype(np.float64) / n).astype(dt)
    monkeypatch.setattr(routinegen, "_cholesky_plan", lambda *a: "two launches")
    if not WARM_ONLY:
        backend().clearCache()  # prepared routines are cached by structure
    got, want, ks = both(R.cholesky(x), [x])
    backend().clearCache()
    assert ks.info["variant"] == "two launches" and ks.info["panels"] == -(-n // 32)
    assert_bits(got, want, f"cholesky {shape} {np.dtype(dt).name}")


@pytest.mark.parametrize("n,batch", [(9, 513), (16, 1025), (27, 1537)])
def test_cholesky_of_many_small_matrices(n, batch):
    """The least number of matrices at which each order takes a wave per matrix."""
    x = spd((batch,), n)
    got, want, ks = both(R.cholesky(x), [x])
    assert [s.name for s in ks.steps] == ["jh_cholesky"]
    assert_bits(got, want, f"cholesky {batch} x {n}")


@pytest.mark.parametrize("n,batch", [(13, 256), (13, 257), (20, 300)])
def test_jacobi_eigh_of_many_small_matrices(n, batch):
    """Either side of the line between a matrix per CU, by blocks, and several that rotate one pair after the other."""
    a = RNG.standard_normal((batch, n, n))
    sym = (a + np.swapaxes(a, -1, -2)).astype(F32)
    got, want, ks = both(R.jacobi_eigh(sym), [sym])
    assert ("block" in ks.info) == (batch <= 256)
    assert_bits(got, want, f"jacobi_eigh {batch} x {n}")


@pytest.mark.parametrize("shape,dt", [((33, 31), F32), ((64, 40), F32), ((3, 32, 65), F32), ((40, 7), np.float64), ((9, 2500), F32), ((1024, 33), F32), ((1025, 40), F32),
                                      ((2049, 20), F32), ((3073, 17), np.float16), ((4096, 9), F32), ((1030, 34), np.float64), ((2200, 12), np.float64), ((3, 1), F32),
                                      ((0, 5, 5), F32), ((300, 8, 8), F32)], ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else np.dtype(v).name)
def test_lu_panels_at_their_edges(shape, dt):
    """Panels that are not whole, one to four rows a thread and the widths that go with them, columns behind the last panel.  Elements of few values: equal
    magnitudes in many waves, of which the first row has to win, and zero columns."""
    a = RNG.integers(-2, 3, shape).astype(dt)
    if a.ndim == 2 and min(shape) > 4:
        a[shape[0] // 2:, :] *= 0.5
        a[:, 2] = a[:, 1]  # cancels: a zero pivot column
    got, want, ks = both(R.lu(a), [a])
    assert_bits(got, want, f"lu {shape} {np.dtype(dt).name} {ks.info}")


@pytest.mark.parametrize("dt", ELEMS, ids=lambda d: np.dtype(d).name)
@pytest.mark.parametrize("shape", [(1, 2), (40, 2, 300), (90, 5, 257), (70, 9, 3000), (300, 17, 130), (900, 33, 65), (64, 48, 1100), (8192, 3, 4), (7, 1, 65)], ids=str)
def test_lu_of_many_wide_matrices(shape, dt):
    """A workgroup per matrix, of one wave to sixteen: rows and columns that are not whole waves, few values of which the first row has to win, a zero column, a NaN."""
    a = RNG.integers(-2, 3, shape).astype(dt)
    if a.ndim == 3:
        a[0, :, 0], a[-1, -1, 1] = 0.0, np.nan
        a[len(a) // 2] = RNG.uniform(-1, 1, shape[1:]).astype(dt)
    got, want, ks = both(R.lu(a), [a])
    assert ks.info["variant"] == "by matrix"
    assert_bits(got, want, f"lu {shape} {np.dtype(dt).name} {ks.info}")


@pytest.mark.parametrize("shape", [(5, 40, 70), (23, 9, 11)], ids=str)
def test_lu_strips_in_several_launches(shape, monkeypatch):
    """More strips than a launch holds, with the bound lowered to seven of them: launches that begin and end inside a matrix."""
    from jaxjs_hip import routinegen
    monkeypatch.setattr(routinegen, "LAUNCH_THREADS", 7 * 512 + 511)
    a = RNG.uniform(-1, 1, shape).astype(F32)
    got, want, ks = both(R.lu(a), [a])
    assert max(s.grid[0] for s in ks.steps if s.name == "jh_lu_strip") == 7
    assert_bits(got, want, f"lu {shape} {ks.info}")


@pytest.mark.parametrize("dt", [F32, np.float64, np.float16], ids=lambda d: np.dtype(d).name)
@pytest.mark.parametrize("n,m,mats,variant", [(9, 16400, 1, "plain"), (21, 19, 900, "plain"), (130, 16400, 1, "staged"), (2050, 3, 1, "staged")], ids=str)
def test_triangular_solve_of_many_right_hand_sides(n, m, mats, variant, dt):
    """More than LDS takes, of a workgroup or of all CUs; the diagonal and right-hand sides of the test of few."""
    a = (np.triu(RNG.standard_normal((mats, n, n))) + np.sqrt(n) * np.eye(n)).astype(dt)
    b = RNG.standard_normal((mats, m, n)).astype(dt)
    a[0, 1, 1], a[0, 2, 2], a[0, 3, 3] = 0.0, np.inf, np.finfo(dt).smallest_subnormal
    b[0, 0, 0], b[0, m - 1, n // 2] = np.inf, np.nan
    a += np.tril(np.full((n, n), np.nan), -1).astype(dt)  # the strictly lower part must not matter
    got, want, ks = both(R.triangular_solve(a, b), [a, b])
    assert ks.info["variant"] == variant
    assert_bits(got, want, f"triangular_solve {mats} x {n} x {m} {np.dtype(dt).name} {ks.info}")


@pytest.mark.parametrize("shape,dt", [((5, 41, 70), F32), ((7, 9, 3), np.float16)], ids=str)
def test_lu_of_matrices_a_few_at_a_time(shape, dt, monkeypatch):
    """The workspace lowered to the multipliers of two matrices: the last launches have one."""
    from jaxjs_hip import routinegen
    monkeypatch.setattr(routinegen, "LU_SCRATCH", 2 * (32 if shape[1] > 16 else 8) * shape[1] * 8)
    a = RNG.uniform(-1, 1, shape).astype(dt)
    got, want, ks = both(R.lu(a), [a])
    assert {s.grid[0] for s in ks.steps if s.name == "jh_lu_panel"} == {1, 2}
    assert_bits(got, want, f"lu {shape} {ks.info}")


@pytest.mark.parametrize("n,m,mats,dt", [(1, 1, 1, F32), (7, 8, 1, F32), (8, 9, 3, F32), (9, 1, 2, F32), (17, 2049, 1, F32), (25, 4100, 1, F32), (40, 8200, 1, F32), (127, 17, 1, F32),
                                         (640, 9, 1, F32), (900, 20, 1, F32), (1300, 3, 1, F32), (1900, 5, 1, F32), (500, 10, 1, np.float64), (333, 12, 1, np.float16),
                                         (70, 1, 600, F32), (45, 11, 300, F32), (261, 2, 270, F32), (90, 40, 280, np.float64)],
                         ids=lambda v: np.dtype(v).name if isinstance(v, type) else str(v))
def test_triangular_solve_of_few_right_hand_sides(n, m, mats, dt):
    """Groups of eight entries and rows of a staged block that are not whole, 8 to 64 right-hand sides a workgroup, lanes without one; a zero, an infinite and
    a subnormal pivot, right-hand sides of infinities and NaN, which have no part in rows that they do not belong to."""
    a = (np.triu(RNG.standard_normal((mats, n, n))) + np.sqrt(n) * np.eye(n)).astype(dt) if n > 1 else np.full((mats, 1, 1), 3, dt)
    b = RNG.standard_normal((mats, m, n)).astype(dt)
    if n > 4:
        a[0, 1, 1], a[0, 2, 2], a[0, 3, 3] = 0.0, np.inf, np.finfo(dt).smallest_subnormal
        b[0, 0, 0], b[0, m - 1, n // 2] = np.inf, np.nan
        a += np.tril(np.full((n, n), np.nan), -1).astype(dt)  # the strictly lower part must not matter
    got, want, ks = both(R.triangular_solve(a, b), [a, b])
    assert_bits(got, want, f"triangular_solve {mats} x {n} x {m} {np.dtype(dt).name} {ks.info}")
