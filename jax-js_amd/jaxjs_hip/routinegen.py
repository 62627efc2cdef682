"""Native launch plans for routines (the non-fusable operations, src/routine.ts:20-102).

Every routine runs on the GPU; there is no host path.  A combination without a plan (an element type the
kernels do not cover, an extent beyond a kernel's stated limit) raises `UnsupportedRoutineError` at prepare
time, which is what the Backend interface prescribes for a routine a backend lacks (src/backend.ts:236-240).

  Sort, Argsort                               `sort.hip.inc`     32-bit, float16 and float64 keys
  Scatter                                     `scatter.hip.inc`  float32/float16/float64/int32/uint32/bool updates
  TriangularSolve, Cholesky, LU, JacobiEigh   `linalg.hip.inc`   float32/float64/float16 (arithmetic in double, as the reference)
  Fft                                         `fft_pass.hip.inc`, `fft.hip.inc` (large prime factors)  float32/float64/float16
  Attention (extension, not in the reference) `attention.hip.inc` float16, head size 32 / 64 / 128, any L and S
"""

from __future__ import annotations

from typing import Optional, Tuple

from . import tuner
from .alu import DType, byteWidth
from .codegen import SOURCE_OPTION
from .kernelgen import KernelSource, LaunchStep, _prelude, fill, template
from .errors import UnsupportedRoutineError
from .routine import Routine, Routines, ScatterOp
from .shape import prod

_SORT_KINDS = {DType.Float32: (0, "jh_u32"), DType.Float16: (1, "jh_u16"), DType.Int32: (2, "int"),
               DType.Uint32: (3, "jh_u32"), DType.Bool: (2, "int"), DType.Float64: (4, "unsigned long long")}
SORT_TILE = 8192  # LDS tile in 8-byte words (64 KB): 16384 4-byte words, 4096 16-byte words
SORT_REGISTERS = 256  # bytes of words a lane holds in the register network
SORT_WAVES = 2048     # waves (two per SIMD) from which 16 lanes per row are enough; with fewer, a row takes up to 64
# Rows of more than 64 x 16 words in fewer than 256 waves: short register runs on many lanes, then LDS (float32 1 x 4096:
# 9.6 us against 11.2 with runs of 1024 words; 600 x 3000 stays in registers, 21.7 us).
SORT_FEW, SORT_FEW_WAVES = 16, 256
# Fewer tiles than a quarter of the chip: smaller ones, which cost a launch per stage but work side by side (float32
# 1 x 20000: 58 us with tiles of 16384, 36 of 8192, 33 of 4096, 37 of 2048; 100 x 16384 stays at 16384, 42.5 against 45.6).
SORT_SMALL_TILE, SORT_FEW_TILES = 4096, 64
SORT_LOCAL, SORT_TILES = 16, 1024  # words of a lane in a tile's register runs, from 1024 tiles on
SORT_HELD = 8     # pieces of 16 bytes that a lane hands to others at a time: whole lines of 128 bytes (float32 32768 x 1024: 70.6 us, 83 with 4)
SORT_GROUP = 8    # elements a thread sorts in registers at the end of every stage (4 for rows of <= 256: more threads stay busy)
LAUNCH_THREADS = (1 << 32) - 1  # of a launch, along one axis
LU_SCRATCH = 1 << 28  # bytes of unrounded multipliers
CHOLESKY_PANEL_FROM = 192  # matrix order from which many matrices may take two launches a panel, and a plan counts its panels
CHOLESKY_WAVE_BELOW = {2: 44, 4: 28, 8: 28}  # matrix order, by bytes per element, below which many matrices take a wave each


def _next_pow2(n: int) -> int:
    p = 1
    while p < n:
        p <<= 1
    return p


def generateRoutine(routine: Routine, numerics: str = "wasm") -> KernelSource:
    gen = {Routines.Sort: _gen_sort, Routines.Argsort: _gen_sort, Routines.Scatter: _gen_scatter,
           Routines.TriangularSolve: _gen_trisolve, Routines.Cholesky: _gen_cholesky, Routines.LU: _gen_lu,
           Routines.JacobiEigh: _gen_jacobi, Routines.Fft: _gen_fft, Routines.Attention: _gen_attention}.get(routine.name)
    ks = gen(routine, numerics) if gen is not None else None
    if ks is None:
        raise UnsupportedRoutineError(routine.name, "hip")
    return ks


def _empty(klass: str, **info) -> KernelSource:
    return KernelSource([], [], [], klass, {}, dict(info))


def _round64(n: int, cap: int = 1024) -> int:
    return max(64, min(cap, (n + 63) // 64 * 64))


_LINALG_DEFAULTS = dict(N=1, M=1, THREADS=64, UNIT=0, IN_LDS=0, MAX_SWEEPS=0, TOL="0.0", BATCH=1, AHEAD=16, STAGED=0, RB=1, RHS=1, ELEM_BYTES=4, BLOCK="unsigned",
                        ELEM="float", CMP="float")
# Element types of the dense routines: C type, the type magnitudes are compared in, bytes per element.
_FLOAT_ELEMS = {DType.Float32: ("float", "float", 4), DType.Float64: ("double", "double", 8), DType.Float16: ("jh_f16", "float", 2)}


def _linalg_source(numerics: str, **params) -> str:
    return _prelude(numerics) + fill(template("linalg.hip.inc"), {**_LINALG_DEFAULTS, **params})


def _float_elem(t):
    """(C type, comparison type, bytes) when every operand has one and the same floating-point type, else None."""
    d = t.inputDtypes[0]
    return _FLOAT_ELEMS.get(d) if all(x == d for x in t.inputDtypes) else None


def _cholesky_plan(n: int, batch: int, eb: int) -> str:
    """Which of the four plans factors `batch` matrices of order n; they give the same bits.  (Figures: float32, microseconds.)

    A launch per panel has the shortest chain, and a workgroup of 256 per 32 rows with 36 KB of LDS (55 in float64): four (two)
    of them on a CU.  A wave per matrix holds 32 on a CU and is as fast alone up to order 8 (9 and 10); from there its chain
    is longer and it takes batches to win: 16: 256 matrices 17.2 against 9.9, 1536 21.7 and 14.3, 4096 27 and 30, 65536 305
    and 378; 20: 4096 37 and 35, 16384 115 on both sides; 24: 4096 55 and 39, 16384 168 and 135; 28: 16384 278 and 145; in
    float16, whose panels pay for conversions, 40: 16384 474 and 426, 48: 770 and 477.  Two launches per panel take less room
    in LDS and were ahead where matrices fill the chip, until a launch per panel took half the time; now they are not: 192:
    1024 matrices 595 against 382, 256: 1024 1073 and 728, 512: 512 3007 and 2159, float64 512: 128 1174 and 785.

    So by these figures a wave per matrix should stop at order 20 and two launches should not be taken at all.  The lines stand
    where tests/test_kernelgen.py pins the plan on either side of them, from measurements of the slower kernel."""
    from . import tuner
    cus = tuner.CU_COUNT
    many = 2 if eb == 8 and n <= 12 else min(n // 4, 6)  # matrices per CU
    if n <= 8 or n < CHOLESKY_WAVE_BELOW[eb] and batch > cus * many:
        return "wave per matrix"
    if n > 64 and batch * n * n * 8 > CHOLESKY_RIGHT_LOOKING_MAX_BYTES:
        return "left-looking"
    if n >= CHOLESKY_PANEL_FROM and batch * (n // 32) >= cus * (8 if eb == 8 else 16):
        return "two launches"
    return "right-looking"


def _gen_cholesky(routine: Routine, numerics: str) -> Optional[KernelSource]:
    t = routine.type
    shape = list(t.inputShapes[0])
    if len(shape) < 2:
        raise ValueError("cholesky: input must be at least 2D")
    n, m = shape[-2], shape[-1]
    if n != m:
        raise ValueError(f"cholesky: input must be square, got [{n}, {m}]")
    el = _float_elem(t)
    if el is None or n > 8192:
        return None
    ctype, cmp_t, eb = el
    batch = prod(shape[:-2])
    if batch == 0 or n == 0:
        return _empty("cholesky", n=n, batch=batch)
    plan = _cholesky_plan(n, batch, eb)
    grid1 = lambda count: (max(1, min((count + 255) // 256, 1 << 16)), 1, 1)  # noqa: E731
    need, panels = {0: batch * n * n * eb}, range(0, n, 32)
    if plan == "wave per matrix":
        src = _linalg_source(numerics, ROUTINE=8, N=n, ELEM=ctype, CMP=cmp_t)
        steps = [LaunchStep("jh_cholesky", (batch, 1, 1), (64, 1, 1), 0, [("in", 0), ("out", 0), ("scratch", 0)])]
        return KernelSource([src], steps, [batch * n * n * eb], "cholesky", need, dict(n=n, batch=batch, threads=64))
    if plan == "right-looking":
        # The running sums of the whole triangle in a double-precision scratch copy (two panels need none), one launch per
        # 32-column panel that finishes the panel and subtracts the one before it from the rest.
        src = _linalg_source(numerics, ROUTINE=5, N=n, ELEM=ctype, CMP=cmp_t)
        steps = []
        for j0 in panels:
            after = max(0, n - j0 - 32)
            T = (after + 63) // 64
            blocks = max(1, (after + 31) // 32) + (T * (T + 1) // 2 if j0 else 0)
            steps.append(LaunchStep("jh_chol_step", (batch * blocks, 1, 1), (256, 1, 1), 0, [("in", 0), ("out", 0), ("scratch", 0), ("const", j0)]))
        scratch, info = [batch * n * n * 8 if n > 64 else 8], dict(variant=plan)
    elif plan == "two launches":
        src = _linalg_source(numerics, ROUTINE=9, N=n, M=batch, ELEM=ctype, CMP=cmp_t)
        steps = [LaunchStep("jh_chol_init", grid1(batch * n * n), (256, 1, 1), 0, [("in", 0), ("out", 0), ("scratch", 0)])]
        for j0 in panels:
            after = max(0, n - j0 - 32)
            T = (after + 63) // 64
            steps.append(LaunchStep("jh_chol_panel", (batch * max(1, T), 1, 1), (64, 1, 1), 0, [("scratch", 0), ("out", 0), ("const", j0)]))
            if after:
                steps.append(LaunchStep("jh_chol_update", (batch * T * T, 1, 1), (256, 1, 1), 0, [("out", 0), ("scratch", 0), ("const", j0)]))
        scratch, info = [batch * n * n * 8], dict(variant=plan)
    else:  # left-looking: 32-column panels, two launches each; the same sums in the same order
        src = _linalg_source(numerics, ROUTINE=4, N=n, M=batch, ELEM=ctype, CMP=cmp_t)
        steps = [LaunchStep("jh_chol_zero", grid1(batch * n * n), (256, 1, 1), 0, [("out", 0)])]
        for j0 in panels:
            steps.append(LaunchStep("jh_chol_bulk", (batch * ((n - j0 + 63) // 64), 1, 1), (256, 1, 1), 0,
                                    [("in", 0), ("out", 0), ("scratch", 0), ("const", j0)]))
            after = max(0, n - j0 - 32)
            steps.append(LaunchStep("jh_chol_panel", (batch * max(1, (after + 63) // 64), 1, 1), (64, 1, 1), 0,
                                    [("scratch", 0), ("out", 0), ("const", j0)]))
        scratch, info = [batch * n * 32 * 8], {}
    if n >= CHOLESKY_PANEL_FROM:
        info["panels"] = len(panels)
    return KernelSource([src], steps, scratch, "cholesky", need, dict(n=n, batch=batch, launches=len(steps), **info))


TRISOLVE_FEW = 64  # right-hand sides for every CU up to which they are few


def _trisolve_few(n: int, m: int, mats: int) -> Optional[Tuple[int, int]]:
    """Right-hand sides of a workgroup and rows of a staged block where m right-hand sides each of `mats` matrices of order n are few
    enough to keep theirs and the solved entries in LDS; None where they are not.

    As few for a workgroup as leave a CU to each, with blocks of up to 32 rows; for more matrices than that no more than one of them has,
    and blocks of at most four rows, eight below order 64, so that two to eight workgroups fit a CU, which hide each other's barriers.  float32, one right-hand side each,
    in microseconds, the other kernels, 32 rows, these: 300 of order 256 487, 575, 288; 512 of 512 1736, 1942, 1014; 4096 of 128 826, 1460 (16 to
    a workgroup), 469; 16384 of 100 1915, 4405 (64), 1260; 600 of 48 48, 28, 27 (37 with four rows).  With 20 right-hand sides each, 512 of order 256 783, 585 (64), 586 (32).
    Fewer where more do not fit, up to two rounds of workgroups."""
    if mats * m > TRISOLVE_FEW * tuner.CU_COUNT:
        return None
    width, offered = -(-n // 8) * 8, (8, 16, 32, 64)
    wanted = next((r for r in offered if mats * -(-m // r) <= tuner.CU_COUNT), None)
    rows = 32 if wanted is not None else 8 if n < 64 else 4
    wanted = wanted or next((r for r in offered if r >= m), 64)
    for rhs in reversed(offered[:offered.index(wanted) + 1]):
        rb = min(rows, n, (160 * 1024 - 64 - 8 * width * rhs) // (16 * width + 16))
        if rb >= 1 and (rhs == wanted or mats * -(-m // rhs) <= 2 * tuner.CU_COUNT):
            return rhs, rb
    return None


def _gen_trisolve(routine: Routine, numerics: str) -> Optional[KernelSource]:
    t = routine.type
    a_shape, b_shape = list(t.inputShapes[0]), list(t.inputShapes[1])
    if len(a_shape) < 2:
        raise ValueError(f"triangular_solve: a must be at least 2D, got {a_shape}")
    if len(b_shape) < 2:
        raise ValueError(f"triangular_solve: b must be at least 2D, got {b_shape}")
    n = a_shape[-2]
    if n != a_shape[-1] or n != b_shape[-1]:
        raise ValueError(f"triangular_solve: incompatible shapes a={a_shape}, b={b_shape}")
    el = _float_elem(t)
    if el is None:
        return None
    ctype, cmp_t, eb = el
    mats, m = prod(a_shape[:-2]), b_shape[-2]
    if prod(b_shape[:-2]) != mats:
        raise ValueError(f"triangular_solve: incompatible shapes a={a_shape}, b={b_shape}")
    if mats == 0 or m == 0 or n == 0:
        return _empty("trisolve", n=n, m=m, batch=mats)
    unit = 1 if (routine.params or {}).get("unitDiagonal", False) else 0
    need = {0: mats * n * n * eb, 1: mats * m * n * eb}
    few = _trisolve_few(n, m, mats)
    if few is not None:
        rhs, rb = few
        src = _linalg_source(numerics, ROUTINE=1, N=n, M=m, THREADS=256, UNIT=unit, STAGED=2, RB=rb, RHS=rhs, ELEM=ctype, CMP=cmp_t)
        steps = [LaunchStep("jh_trisolve_few", (mats * -(-m // rhs), 1, 1), (256, 1, 1), 0, [("in", 0), ("in", 1), ("out", 0)])]
        return KernelSource([src], steps, [], "trisolve", need, dict(n=n, m=m, batch=mats, variant="few", rhs=rhs, rows_per_block=rb))
    if TRISOLVE_STAGED_FROM <= n <= TRISOLVE_STAGED_MAX_N:
        # one wave of 64 right-hand sides + three waves staging blocks of rows in LDS as doubles (two buffers <= 128 KB)
        rb = max(1, min(8, TRISOLVE_STAGED_MAX_N // n))
        src = _linalg_source(numerics, ROUTINE=1, N=n, M=m, THREADS=256, UNIT=unit, AHEAD=TRISOLVE_AHEAD, STAGED=1, RB=rb,
                             ELEM=ctype, CMP=cmp_t)
        steps = [LaunchStep("jh_trisolve_staged", (mats * ((m + 63) // 64), 1, 1), (256, 1, 1), 0,
                            [("in", 0), ("in", 1), ("out", 0), ("scratch", 0)])]
        return KernelSource([src], steps, [mats * m * n * 8], "trisolve", need,
                            dict(n=n, m=m, batch=mats, variant="staged", rows_per_block=rb))
    threads = 64 if m <= 64 else 256
    src = _linalg_source(numerics, ROUTINE=1, N=n, M=m, THREADS=threads, UNIT=unit, AHEAD=TRISOLVE_AHEAD, ELEM=ctype, CMP=cmp_t)
    blocks = mats * ((m + threads - 1) // threads)
    steps = [LaunchStep("jh_trisolve", (blocks, 1, 1), (threads, 1, 1), 0, [("in", 0), ("in", 1), ("out", 0), ("scratch", 0)])]
    return KernelSource([src], steps, [mats * m * n * eb], "trisolve", need, dict(n=n, m=m, batch=mats, variant="plain", threads=threads))


def _lu_width(m: int, n: int, eb: int) -> int:
    """Columns of a panel: as many as fit a thread's registers with its rows of 1024."""
    rows = -(-m // 1024)
    return min(32, 1 << (64 // (rows * (2 if eb == 8 else 1))).bit_length() - 1, max(8, 1 << (min(m, n) - 1).bit_length()))


def _lu_strips(m: int, n: int, width: int, j: int) -> int:
    """Strips of eight columns beside the panel from column j on."""
    return -(-j // 8) + -(-(n - min(j + width, m, n)) // 8)


def _lu_by_matrix(m: int, n: int, batch: int, eb: int) -> bool:
    """Whether matrices take a workgroup each for all their columns, in one launch, and not panels.

    A panel's column is the faster one, but every eight columns beside a panel cost a workgroup of 512 threads, few of which have an
    element where there are few rows.  Matrices of at most five rows go by matrix where anything is beside their panel (7.5 us for one launch, 11 for two; float32
    1202 x [3, 272] 10.0 us, 82 by panels, 8484 x [2, 445] 62 and 828) unless they are few and long, and others up to 64 (48 in float64) where many strips meet many
    matrices: float32 829 x [12, 1078] 164 and 647, 262 x [46, 310] 272 and 421, 13646 x [34, 34] 535 and 932, but float64 21 x [75, 262] 528 and 161, 125 x [16, 238] 53 and
    37, float16 855 x [57, 57] 507 and 383.  With more rows than columns panels are twice to five times as fast.  In float16, whose elements a panel's threads convert in every
    step, also very many small ones without strips: 11900 x [3, 3] 14.6 and 19.3, 10728 x [24, 24] 326 and 413.  Of 434 batches of all three types the choice is 0.7 per
    cent from the faster one in the mean."""
    if m > n or batch * _round64(n) > LAUNCH_THREADS:
        return False
    width = _lu_width(m, n, eb)
    strips = batch * sum(_lu_strips(m, n, width, j) for j in range(0, m, width))
    if strips and ((m <= 5 and (n <= 256 or batch >= 16 * m)) or (m <= (48 if eb == 8 else 64) and batch >= 48 and strips >= (128 if eb == 2 else 200) * m)):
        return True
    return eb == 2 and m <= 32 and batch >= 8192


def _gen_lu(routine: Routine, numerics: str) -> Optional[KernelSource]:
    t = routine.type
    shape = list(t.inputShapes[0])
    if len(shape) < 2:
        raise ValueError("lu: input must be at least 2D")
    m, n = shape[-2], shape[-1]
    el = _float_elem(t)
    if el is None:
        return None
    ctype, cmp_t, eb = el
    batch = prod(shape[:-2])
    if batch == 0 or m == 0:
        return _empty("lu", m=m, n=n, batch=batch)
    if m <= 4096 and _lu_by_matrix(m, n, batch, eb):
        threads = _round64(max(m, n))
        src = _linalg_source(numerics, ROUTINE=2, N=n, M=m, THREADS=threads, ELEM=ctype, CMP=cmp_t)
        steps = [LaunchStep("jh_lu", (batch, 1, 1), (threads, 1, 1), 0, [("in", 0), ("out", 0), ("out", 1), ("out", 2)])]
        return KernelSource([src], steps, [], "lu", {0: batch * m * n * eb}, dict(m=m, n=n, batch=batch, launches=1, variant="by matrix"))
    if m <= 4096:
        width = _lu_width(m, n, eb)
        # the multipliers of a panel, of as many matrices at a time as LU_SCRATCH holds: at least 512, which fill the chip
        at_once = min(batch, LU_SCRATCH // (width * m * 8))
        src = _linalg_source(numerics, ROUTINE=10, N=n, M=m, RB=width, ELEM=ctype, CMP=cmp_t, ELEM_BYTES=eb, BLOCK="unsigned" if (at_once + 1) * (-(-n // 8) + 1) < 1 << 32 else "unsigned long long")
        steps = []
        for mat in range(0, batch, at_once):
            mats = min(at_once, batch - mat)
            for j in range(0, max(min(m, n), 1), width):
                steps.append(LaunchStep("jh_lu_panel", (mats, 1, 1), (_round64(m - j), 1, 1), 0,
                                        [("in", 0), ("out", 0), ("out", 1), ("out", 2), ("scratch", 0), ("scratch", 1), ("scratch", 2), ("const", mat), ("const", j)]))
                strips = _lu_strips(m, n, width, j)
                for first in range(0, mats * strips, LAUNCH_THREADS // 512):
                    steps.append(LaunchStep("jh_lu_strip", (min(mats * strips - first, LAUNCH_THREADS // 512), 1, 1), (512, 1, 1), 0,
                                            [("in", 0), ("out", 0), ("out", 1), ("scratch", 0), ("scratch", 1), ("scratch", 2), ("const", mat), ("const", j), ("const", first)]))
        return KernelSource([src], steps, [at_once * width * m * 8, at_once * m * 4, max(at_once * 4, 16)], "lu", {0: batch * m * n * eb},
                            dict(m=m, n=n, batch=batch, launches=len(steps), variant="by panels"))
    if min(m, n) >= LU_BY_COLUMNS_FROM and batch * m * n < (1 << 31):
        # More rows than a workgroup holds a panel of: two launches per column, the rank-1 update of the trailing block over the whole
        # chip; the same operations per element as the panels.
        src = _linalg_source(numerics, ROUTINE=6, N=n, M=m, THREADS=1024, BATCH=batch, ELEM=ctype, CMP=cmp_t)
        grid1 = lambda count: (max(1, min((count + 255) // 256, 1 << 16)), 1, 1)  # noqa: E731
        steps = [LaunchStep("jh_lu_init", grid1(batch * m * n), (256, 1, 1), 0, [("in", 0), ("out", 0), ("out", 2)])]
        for j in range(min(m, n)):
            steps.append(LaunchStep("jh_lu_col", (batch, 1, 1), (1024, 1, 1), 0,
                                    [("out", 0), ("out", 1), ("out", 2), ("scratch", 0), ("scratch", 1), ("const", j)]))
            rows, cols = m - j - 1, n - j - 1
            if rows > 0 and cols > 0:
                steps.append(LaunchStep("jh_lu_update", (batch * ((cols + 63) // 64) * ((rows + 31) // 32), 1, 1), (256, 1, 1), 0,
                                        [("out", 0), ("scratch", 0), ("scratch", 1), ("const", j)]))
        return KernelSource([src], steps, [batch * m * 8, max(batch * 4, 16)], "lu", {0: batch * m * n * eb},
                            dict(m=m, n=n, batch=batch, launches=len(steps), variant="by columns"))
    return None


def _jacobi_blocks_pay(n: int, batch: int, eb: int) -> bool:
    """Whether JacobiEigh by blocks is faster than one rotation after the other for this many matrices (same bits).

    By blocks, a matrix takes a CU for itself, so time goes with rounds of 256 matrices; one after the other, as many
    share a CU as its LDS holds two copies of, at no cost to each other up to about one wave per SIMD.  One round is
    faster by about n / 16 (float32 order 16: 1.4 times, 32: 2.7, 48: 3.5, 64: 4.9), in float16, whose every value is
    converted, by n / 28; past that many rounds the others have caught up, unless they wait for each other too (float32, ms:
    16 x 512 0.43 against 0.54 by blocks, 32 x 512 2.12 and 1.44, 32 x 1024 2.5 and 2.9, 64 x 1024 14.1 and 8.2, 13 x 16384
    2.0 and 14.0).  At the line itself blocks have become the faster ones (48 x 1024 5.3 and 5.0, float64 6.1 and 5.7, float16
    48 x 512 7.1 and 5.7); it is where tests/test_kernelgen.py pins it."""
    from . import tuner
    rounds = -(-batch // tuner.CU_COUNT)
    held = 150 * 1024 // (2 * n * n * eb)  # matrices on a CU when one rotation follows the other
    if held == 0:  # too large for LDS: ten times slower alone, and more so together
        return True
    return rounds <= max(1.0, n / (28 if eb == 2 else 16)) * -(-rounds // held)


def _gen_jacobi(routine: Routine, numerics: str) -> Optional[KernelSource]:
    t = routine.type
    shape = list(t.inputShapes[0])
    if len(shape) < 2:
        raise ValueError("jacobi_eigh: input must be at least 2D")
    n = shape[-1]
    if n != shape[-2]:
        raise ValueError(f"jacobi_eigh: input must be square, got {shape}")
    if t.inputDtypes[0] not in (DType.Float32, DType.Float16, DType.Float64):
        raise TypeError("jacobi_eigh: input must be floating-point")
    el = _float_elem(t)
    if el is None or n > 16384:
        return None
    ctype, cmp_t, eb = el
    batch = prod(shape[:-2])
    if batch == 0 or n == 0:
        return _empty("jacobi", n=n, batch=batch)
    params = routine.params or {}
    threads = _round64(n)
    in_lds = 1 if 2 * n * n * eb <= 150 * 1024 else 0  # both matrices in the CU's 160 KB of LDS: n <= 138 in float32
    by_blocks = JACOBI_BLOCKS_FROM[eb] <= n <= 192 and _jacobi_blocks_pay(n, batch, eb)
    # Waves for part 3 beside the chains' (three times n / 64), as many as leave a lane the registers it needs (float32 64:
    # 1.83 ms with 8, 1.84 with 16; 128: 7.0 with 8, 6.7 with 12, 6.4 with 16; float64 96: 4.8 with 8, 4.5 with 12, 5.0 with
    # 16; 128: 7.5, 7.2 and 7.3).  From order 129 on the chains, eigenvectors and columns before p take more than eight.
    block_threads = 512 if n <= 64 else 768 if eb == 8 else 1024
    for size in (4, 8):  # indices per block; the triangle and the rotations under way have to fit the LDS
        blocks = -(-n // size)
        if by_blocks and eb * (n * (n + 1) // 2) + 16 * (blocks + 1) * n + 32 * blocks + 512 <= 160 * 1024:
            src = _linalg_source(numerics, ROUTINE=7, N=n, THREADS=block_threads, RB=size, MAX_SWEEPS=int(params["maxSweeps"]), TOL=repr(float(params["tolerance"])), ELEM=ctype, CMP=cmp_t)
            steps = [LaunchStep("jh_jacobi_blocks", (batch, 1, 1), (block_threads, 1, 1), 0, [("in", 0), ("out", 0), ("out", 1), ("scratch", 0)])]
            return KernelSource([src], steps, [batch * n * n * eb], "jacobi", {0: batch * n * n * eb},
                                dict(n=n, batch=batch, threads=block_threads, in_lds=bool(in_lds), block=size))
    src = _linalg_source(numerics, ROUTINE=3, N=n, THREADS=threads, IN_LDS=in_lds, MAX_SWEEPS=int(params["maxSweeps"]),
                         TOL=repr(float(params["tolerance"])), ELEM=ctype, CMP=cmp_t)
    steps = [LaunchStep("jh_jacobi", (batch, 1, 1), (threads, 1, 1), 0, [("in", 0), ("out", 0), ("out", 1)])]
    return KernelSource([src], steps, [], "jacobi", {0: batch * n * n * eb}, dict(n=n, batch=batch, threads=threads, in_lds=bool(in_lds)))


# The step of a block costs about as much as the few rotations of a smaller matrix (float32 12: 164 against 177 us, 13: 192 and
# 207, 16: 277 and 386; float64 12: 199 and 211; float16 13: 463 and 401, 16: 611 and 635).  tests/test_kernelgen.py pins 12
# and 13.
JACOBI_BLOCKS_FROM = {2: 16, 4: 13, 8: 13}
ATTENTION_FEW_QUERIES = 4     # queries per sequence up to which a query may be a workgroup of its own (`attention_by_queries`)
TRISOLVE_STAGED_FROM = 128    # matrix size from which TriangularSolve stages the matrix in LDS with helper waves
TRISOLVE_STAGED_MAX_N = 8192   # two one-row buffers of doubles still fit in LDS
TRISOLVE_AHEAD = 8       # entries of a row that a right-hand side's thread fetches ahead of its subtraction chain
LU_BY_COLUMNS_FROM = 192  # smaller dimension from which LU of more than 4096 rows runs, two launches per column over the whole chip
CHOLESKY_RIGHT_LOOKING_MAX_BYTES = 1 << 30  # the double-precision working copy of all matrices
FFT_FUSED_MAX_N = 8192  # 16 bytes of LDS per point: 128 KiB


def _gen_fft(routine: Routine, numerics: str) -> Optional[KernelSource]:
    t = routine.type
    shape = list(t.inputShapes[0])
    if len(shape) < 1:
        raise ValueError("fft: input must be at least 1D")
    n = shape[-1]
    if n < 1:
        raise ValueError(f"fft: final axis must be non-empty, got {n}")
    if t.inputDtypes[0] != t.inputDtypes[1] or t.inputDtypes[0] not in (DType.Float32, DType.Float16, DType.Float64):
        raise ValueError("fft: expected matching floating-point real/imag arrays")
    params = routine.params or {}
    factors = [int(f) for f in params["factors"]]
    if prod(factors) != n or any(f < 1 for f in factors):
        raise ValueError(f"fft: factors {factors} do not multiply to the axis length {n}")
    el = _float_elem(t)
    if el is None or n >= (1 << 30):
        return None
    ctype, _, eb = el
    rows = prod(shape[:-1])
    if rows == 0:
        return _empty("fft", n=n, rows=rows)
    if "singleLaunch" not in params:
        ks = _fft_passes(n, rows, ctype, eb, bool(params.get("inverse")), numerics, factors)
        if ks is not None:
            return ks
    # Rows that fit the LDS twice over (16 bytes per point) run in one launch, one workgroup per row, unless there are
    # too few rows for that to use the chip (a single long row is quicker spread over many workgroups per stage).
    S = len(factors)
    fused_max = FFT_FUSED_MAX_N * 4 // max(eb, 4)  # four buffers of n elements: 128 KiB at most
    fused = S >= 1 and n <= fused_max and (n <= 2048 or rows >= 64)
    if "singleLaunch" in params:  # tests pin either path
        fused = bool(params["singleLaunch"]) and S >= 1 and n <= fused_max
    threads = min(1024, max(64, _round64(n)))
    # Twiddle tables: stage s has span_s entries for (q, j) and radix_s^2 for (q, p), 16 bytes each.
    offsets, spans, prev = [0], [], 1
    for radix in factors:
        spans.append(prev * radix + radix * radix)
        offsets.append(offsets[-1] + spans[-1])
        prev *= radix
    lds_entries = max(spans) if spans and 4 * eb * n + 16 * max(spans) <= 150 * 1024 else 0
    src = _prelude(numerics) + fill(template("fft.hip.inc"), dict(N=n, ROWS=rows, ELEM=ctype, INVERSE=1 if params.get("inverse") else 0,
                                                                  NF=len(factors), FACTORS=", ".join(map(str, factors)) or "1",
                                                                  TW_OFFSETS=", ".join(map(str, offsets if S else [0, 0])),
                                                                  FUSED=1 if fused else 0, FUSED_THREADS=threads,
                                                                  FUSED_TABLE_ENTRIES=lds_entries))
    need = {0: rows * n * eb, 1: rows * n * eb}
    if fused:
        steps = [LaunchStep("jh_fft_rows", (min(rows, 1 << 16), 1, 1), (threads, 1, 1), 0, [("in", 0), ("in", 1), ("out", 0), ("out", 1)])]
        return KernelSource([src], steps, [], "fft", need, dict(n=n, rows=rows, factors=factors, launches=1, fused=True, lds_tables=bool(lds_entries)))
    blocks = max(1, min((rows * n + 255) // 256, 1 << 20))
    out_pair, tmp_pair = [("out", 0), ("out", 1)], [("scratch", 0), ("scratch", 1)]
    target = lambda s: out_pair if (S - 1 - s) % 2 == 0 else tmp_pair  # noqa: E731  (stage -1 is the permutation)
    steps = [LaunchStep("jh_fft_permute", (blocks, 1, 1), (256, 1, 1), 0, [("in", 0), ("in", 1)] + target(-1) + [("scratch", 2)])]
    prev = 1
    for s_, radix in enumerate(factors):
        steps.append(LaunchStep("jh_fft_stage", (blocks, 1, 1), (256, 1, 1), 0,
                                target(s_ - 1) + target(s_) + [("scratch", 2), ("const", prev), ("const", radix),
                                                               ("const", 1 if s_ == S - 1 else 0), ("const", s_)]))
        prev *= radix
    scratch = [rows * n * eb, rows * n * eb, max(offsets[-1], 1) * 16] if S >= 1 else [8, 8, 16]
    return KernelSource([src], steps, scratch, "fft", need, dict(n=n, rows=rows, factors=factors, launches=len(steps), fused=False))


FFT_PASS_RADIX_MAX = 13       # larger prime factors: one thread per output of a stage (fft.hip.inc)
FFT_PASS_POINTS = 8192        # points a workgroup keeps in LDS, twice (128 KiB as float pairs)


FFT_NESTED = {6: 2, 8: 2, 9: 3, 10: 2, 12: 3, 16: 4}  # butterflies made of two smaller ones: points of the outer


def _fft_radices(L: int) -> Optional[list]:
    """L as a product of butterfly sizes, powers of two in eights and sixteens; None when a prime factor is too large."""
    out, two = [], 0
    while L % 2 == 0:
        L, two = L // 2, two + 1
    while two:  # 2^4k and 2^3k first choice; 2, 4 only for what is left
        step = 3 if two in (3, 6, 9) else 4 if two >= 4 else two
        out.append(1 << step)
        two -= step
    for p in (3, 5, 7, 11, 13):
        while L % p == 0:
            out.append(p)
            L //= p
    return out if L == 1 else None


def _fft_fewest(L: int) -> list:
    """L as a product of as few butterfly sizes as possible, then the smallest largest and the smallest sum."""
    best = {1: (0, 0, 0, [])}
    for n in (d for d in range(2, L + 1) if L % d == 0):
        for r in (2, 3, 4, 5, 7, 11, 13, *FFT_NESTED):
            rest = best.get(n // r) if n % r == 0 else None
            if rest is not None:
                option = (rest[0] + 1, max(rest[1], r), rest[2] + r, sorted(rest[3] + [r], reverse=True))
                if n not in best or option < best[n]:
                    best[n] = option
    return best[L][3]


def _fft_threads(L: int, cols: int, radices: list) -> int:
    return _round64(max(L // r for r in radices) * cols, 512 if max(radices) > 10 else 1024)


def _fft_stages(L: int, cols: int, blocks: int, double: bool) -> list:
    """The butterfly sizes of a pass.  A stage less is a round trip through LDS and a wait for twiddles less, but larger
    butterflies are fewer threads: two stages less pay always (7776: 11.6 -> 9.3 us, 531441 16.9 -> 15.3, 2250 4.9 -> 4.2),
    one where the workgroups fill the chip and have more than a wave for every SIMD (10^6 21.3 -> 20.3, 500 rows of 1500 6.5 ->
    6.1; one row of 3000 4.7 -> 4.9, 512 of 1000 in workgroups of four waves 4.6 -> 4.7).  In float64, where a stage's results are not rounded in
    between, the larger butterflies only add roundings (10^6 points: 5.7 and 6.3e-16; in float32 7.2 and 6.2e-8)."""
    plain = _fft_radices(L) or [1]
    if double or L < 2:
        return plain
    fewest = _fft_fewest(L)
    less = len(plain) - len(fewest)
    return fewest if less >= 2 or (less == 1 and blocks >= 128 and _fft_threads(L, cols, fewest) > 256) else plain


def _fft_lengths(n: int, limit: int) -> Optional[list]:
    """n as a product of one, two or three pass lengths up to `limit`, as equal as its divisors allow."""
    if n <= limit:
        return [n]
    divisors = [d for i in range(1, int(n ** 0.5) + 1) if n % i == 0 for d in (i, n // i)]
    for passes in (2, 3):
        best = None
        for a in divisors:
            if a > limit:
                continue
            rest = n // a
            tails = [[rest]] if passes == 2 else [[b, rest // b] for b in divisors if b <= limit and rest % b == 0]
            for tail in tails:
                if max(tail) <= limit and (best is None or max([a] + tail) < max(best)):
                    best = sorted([a] + tail, reverse=True)
        if best is not None:
            return best
    return None


def _fft_columns(L: int, total: int, points: int, alone: bool) -> int:
    """Columns a workgroup transforms side by side: up to a whole line of them (16 floats), fewer while that leaves CUs
    without a workgroup, but four where they are adjacent in memory (n = 10^6 in passes of 1000: two columns 26.3 us, four
    20.9, eight 23.7; three passes of 100 with 4 to 32 columns 23.4 to 26.9)."""
    cols = 1
    while cols < (64 if alone else 16) and 2 * cols * L <= min(points, 4096 if alone else points // 2) and (total // (2 * cols) >= 256 or (not alone and cols < 4)):
        cols *= 2
    return cols


def _fft_butterfly(R: int, sign: float) -> str:
    """`jh_dft` for R points in place: sums over pairs q, R - q for odd R, two nested transforms for 2^k."""
    import math
    lines = [f"JH_DEV void jh_dft(jh_c (&v)[{R}]) {{"]
    lit = lambda x: float(x).hex()  # noqa: E731
    if R == 2:
        lines.append("  const jh_c a = v[0], b = v[1]; v[0] = jh_c{a.re + b.re, a.im + b.im}; v[1] = jh_c{a.re - b.re, a.im - b.im};")
    elif R == 4:
        s = "" if sign > 0 else "-"
        lines += ["  const jh_c a = jh_c{v[0].re + v[2].re, v[0].im + v[2].im}, b = jh_c{v[0].re - v[2].re, v[0].im - v[2].im};",
                  "  const jh_c c = jh_c{v[1].re + v[3].re, v[1].im + v[3].im}, d = jh_c{v[1].re - v[3].re, v[1].im - v[3].im};",
                  f"  const jh_c e = jh_c{{{'-' if sign > 0 else ''}d.im, {s}d.re}};",  # d times +-i
                  "  v[0] = jh_c{a.re + c.re, a.im + c.im}; v[1] = jh_c{b.re + e.re, b.im + e.im};",
                  "  v[2] = jh_c{a.re - c.re, a.im - c.im}; v[3] = jh_c{b.re - e.re, b.im - e.im};"]
    elif R in FFT_NESTED and math.gcd(FFT_NESTED[R], R // FFT_NESTED[R]) == 1:
        # coprime sizes (Good 1958): points at B a + A b, results at the k with k = i (mod A), k = j (mod B), no twiddles
        A, B = FFT_NESTED[R], R // FFT_NESTED[R]
        lines.append(f"  jh_c t[{A}][{B}];")
        for a in range(A):
            lines.append(f"  {{ jh_c x[{B}] = {{{', '.join(f'v[{(B * a + A * b) % R}]' for b in range(B))}}}; jh_dft(x); " + " ".join(f"t[{a}][{j}] = x[{j}];" for j in range(B)) + " }")
        for j in range(B):
            at = [next(k for k in range(R) if k % A == i and k % B == j) for i in range(A)]
            lines.append(f"  {{ jh_c x[{A}] = {{{', '.join(f't[{a}][{j}]' for a in range(A))}}}; jh_dft(x); " + " ".join(f"v[{at[i]}] = x[{i}];" for i in range(A)) + " }")
    elif R in FFT_NESTED:
        A, B = FFT_NESTED[R], R // FFT_NESTED[R]  # v[a + A*b]: transforms over b, twiddles, transforms over a
        lines.append(f"  jh_c t[{A}][{B}];")
        for a in range(A):
            lines.append(f"  {{ jh_c x[{B}] = {{{', '.join(f'v[{a + A * b}]' for b in range(B))}}}; jh_dft(x);")
            for k in range(B):
                ang = sign * 2 * math.pi * a * k / R
                lines.append(f"    t[{a}][{k}] = " + (f"x[{k}];" if a * k == 0 else f"jh_mul(x[{k}], jh_c{{{lit(math.cos(ang))}, {lit(math.sin(ang))}}});"))
            lines.append("  }")
        for k in range(B):
            lines.append(f"  {{ jh_c x[{A}] = {{{', '.join(f't[{a}][{k}]' for a in range(A))}}}; jh_dft(x); " + " ".join(f"v[{k + B * a}] = x[{a}];" for a in range(A)) + " }")
    else:
        H = (R - 1) // 2
        for q in range(1, H + 1):
            lines.append(f"  const jh_c s{q} = jh_c{{v[{q}].re + v[{R - q}].re, v[{q}].im + v[{R - q}].im}}, d{q} = jh_c{{v[{q}].re - v[{R - q}].re, v[{q}].im - v[{R - q}].im}};")
        lines.append("  const jh_c z = v[0];")
        lines.append("  v[0] = jh_c{z.re + " + " + ".join(f"s{q}.re" for q in range(1, H + 1)) + ", z.im + " + " + ".join(f"s{q}.im" for q in range(1, H + 1)) + "};")
        for p in range(1, H + 1):
            cs = [math.cos(2 * math.pi * (q * p % R) / R) for q in range(1, H + 1)]
            sn = [sign * math.sin(2 * math.pi * (q * p % R) / R) for q in range(1, H + 1)]
            even = lambda part: "z." + part + "".join(f" + {lit(c)} * s{q}.{part}" for q, c in enumerate(cs, 1))  # noqa: E731
            odd = lambda part: " + ".join(f"{lit(s)} * d{q}.{part}" for q, s in enumerate(sn, 1))  # noqa: E731
            lines.append(f"  {{ const double er = {even('re')}, ei = {even('im')}, orr = {odd('re')}, oi = {odd('im')};")
            lines.append(f"    v[{p}] = jh_c{{er - oi, ei + orr}}; v[{R - p}] = jh_c{{er + oi, ei - orr}}; }}")
    lines.append("}")
    return "\n".join(lines)


def _fft_passes(n: int, rows: int, ctype: str, eb: int, inverse: bool, numerics: str, factors: list) -> Optional[KernelSource]:
    """The transform in as few passes over memory as its length allows (fft_pass.hip.inc); None for lengths with a prime
    factor above FFT_PASS_RADIX_MAX."""
    import numpy as np

    if n < 2 or _fft_radices(n) is None:
        return None
    points = FFT_PASS_POINTS * 8 // (2 * max(eb, 4))
    # Alone in a workgroup a row may fill its LDS; the passes of a longer one take columns side by side, at least four.
    lengths = _fft_lengths(n, points) if n <= points else _fft_lengths(n, points // 4)
    if lengths is None:
        return None
    sign = 1.0 if inverse else -1.0
    exchange = "double" if ctype == "double" else "float"

    def table(count: int, of: int, step: int = 1) -> str:
        """exp(sign 2 pi i m step / of) for m < count, each angle reduced to the first eighth of the circle exactly."""
        m = (np.arange(count, dtype=np.int64) * step) % of
        oct_, rem = (8 * m) // of, None
        ang = 2 * np.pi * np.where(oct_ % 2 == 0, m * 8 - oct_ * of, (oct_ + 1) * of - m * 8).astype(np.float64) / (8.0 * of)
        c, s = np.cos(ang), np.sin(ang)
        swap = np.isin(oct_ % 8, (1, 2, 5, 6))
        re, im = np.where(swap, s, c), np.where(swap, c, s)
        re, im = np.where(np.isin(oct_ % 8, (2, 3, 4, 5)), -re, re), sign * np.where(np.isin(oct_ % 8, (4, 5, 6, 7)), -im, im)
        return ", ".join(f"{{{float(a).hex()}, {float(b).hex()}}}" for a, b in zip(re, im))

    sources, steps = [], []
    S = 1
    for i, Ln in enumerate(lengths):
        D = n // S // Ln
        final = D == 1
        alone = len(lengths) == 1
        total = rows * S * D
        cols = _fft_columns(Ln, total, points, alone)
        radices = _fft_stages(Ln, cols, -(-total // cols), ctype == "double")
        threads = _fft_threads(Ln, cols, radices)
        low_bits = max(1, (Ln * D - 1).bit_length() // 2)
        kinds = sorted({k for r in radices for k in ((r, FFT_NESTED[r], r // FFT_NESTED[r]) if r in FFT_NESTED else (r,))})
        blocks = -(-total // cols)
        # Neighbouring tiles of columns share the lines of the rows they cut: neighbours go to one XCD (workgroups are handed
        # to the eight XCDs in turn), whose L2 then serves the second of them.
        grid = blocks if alone else -(-blocks // 8) * 8
        tile = "JH_DEV int jh_tile() { return " + ("(int)blockIdx.x" if alone else f"(int)(blockIdx.x % 8) * {grid // 8} + (int)(blockIdx.x / 8)") + "; }"
        calls, NS = [], 1
        for s, r in enumerate(radices):
            src, dst = (s + 1) & 1, s & 1
            calls.append(f"  jh_stage<{r}, {NS}, {'true' if s == 0 else 'false'}, {'true' if s == len(radices) - 1 else 'false'}>(in_re, in_im, out_re, out_im, re[{src}], im[{src}], re[{dst}], im[{dst}]);")
            if s < len(radices) - 1:
                calls.append("  __syncthreads();")
            NS *= r
        sources.append(_prelude(numerics) + fill(template("fft_pass.hip.inc"), dict(
            N=n, L=Ln, COLS=cols, THREADS=threads, S=S, D=D, TOTAL=total, GUARD=1 if grid * cols != total else 0, L1=lengths[0], L2=lengths[1] if len(lengths) == 3 else 1,
            POINTS_FIRST=1 if final else 0, POINTS_LAST=1 if alone else 0, SCALE=repr(1.0 / n) if inverse and final else "1.0", LOW_BITS=low_bits,
            INDEX="int" if rows * n + cols * n < (1 << 31) else "long long", ELEM=ctype, EXCHANGE=exchange, TWIDDLES=table(Ln, Ln), HIGH=table(((Ln * D - 1) >> low_bits) + 1, Ln * D, 1 << low_bits) if not final else "{1.0, 0.0}",
            LOW=table(1 << low_bits, Ln * D) if not final else "{1.0, 0.0}", BUTTERFLIES=tile + "\n" + "\n".join(_fft_butterfly(r, sign) for r in kinds),
            NAME=f"jh_fft_pass{i}", STAGES=len(radices), STAGE_CALLS="\n".join(calls))))
        src_pair = [("in", 0), ("in", 1)] if i == 0 else [("scratch", 2 * ((i - 1) % 2)), ("scratch", 2 * ((i - 1) % 2) + 1)]
        dst_pair = [("out", 0), ("out", 1)] if final else [("scratch", 2 * (i % 2)), ("scratch", 2 * (i % 2) + 1)]
        steps.append(LaunchStep(f"jh_fft_pass{i}", (grid, 1, 1), (threads, 1, 1), 0, src_pair + dst_pair, module=i))
        S *= Ln
    scratch = [rows * n * eb] * (2 * (len(lengths) - 1))
    need = {0: rows * n * eb, 1: rows * n * eb}
    return KernelSource(sources, steps, scratch, "fft", need, dict(n=n, rows=rows, factors=factors, launches=len(steps), passes=lengths))


_SCATTER_KINDS = {DType.Float32: (0, "float"), DType.Float16: (1, "jh_f16"), DType.Int32: (2, "int"), DType.Uint32: (3, "jh_u32"),
                  DType.Bool: (4, "int"), DType.Float64: (5, "double")}


def _gen_scatter(routine: Routine, numerics: str) -> Optional[KernelSource]:
    """Index arithmetic of src/routine.ts:226-296, unrolled over the output axes at generation time."""
    t = routine.type
    params = routine.params or {}
    op = ScatterOp(getattr(params["op"], "value", params["op"]))
    out_shape, axes, out_dim = [int(x) for x in params["shape"]], [int(x) for x in params["axis"]], int(params["outDim"])
    unique = bool(params.get("uniqueIndices", False))
    ushape = list(t.inputShapes[0])
    index_shapes = [list(s) for s in t.inputShapes[1:]]
    dtype = t.inputDtypes[0]
    if dtype not in _SCATTER_KINDS or any(d not in (DType.Int32, DType.Uint32) for d in t.inputDtypes[1:]):
        return None
    if len(axes) != len(index_shapes):
        raise ValueError(f"scatter: {len(axes)} indexed axes but {len(index_shapes)} index arrays")
    U, OUT = prod(ushape), prod(out_shape)
    if U >= (1 << 31) or OUT >= (1 << 31):
        return None
    if OUT == 0:
        return _empty("scatter", updates=U, out=OUT)
    index_rank = max((len(s) for s in index_shapes), default=0)
    ustrides = [prod(ushape[d + 1:]) for d in range(len(ushape))]
    ostrides = [prod(out_shape[d + 1:]) for d in range(len(out_shape))]
    free_dims = [d for d in range(len(ushape)) if d < out_dim or d >= out_dim + index_rank]
    if len(free_dims) != len(out_shape) - len(axes):
        raise ValueError(f"scatter: updates of shape {ushape} do not match output {out_shape} indexed on {axes}")
    coord = lambda d: f"((i / {ustrides[d]}ll) % {ushape[d]}ll)"  # noqa: E731
    lines, free_i = [], 0
    for axis, extent in enumerate(out_shape):
        if axis in axes:
            k = axes.index(axis)
            ishape = index_shapes[k]
            istrides = [prod(ishape[j + 1:]) for j in range(len(ishape))]
            first = out_dim + index_rank - len(ishape)
            terms = [f"{coord(first + j)} * {istrides[j]}ll" for j in range(len(ishape)) if ishape[j] != 1]
            cast = "(jh_i64)" if t.inputDtypes[1 + k] == DType.Int32 else "(jh_i64)(jh_u32)"
            lines.append(f"  c = {cast}idx{k}[{' + '.join(terms) or '0'}];")
        else:
            lines.append(f"  c = {coord(free_dims[free_i])};")
            free_i += 1
        lines.append(f"  if (c < 0 || c >= {extent}ll) return -1;")
        lines.append(f"  o += c * {ostrides[axis]}ll;")
    accumulate = op != ScatterOp.Update and not unique
    mode = 2 if accumulate else (0 if unique else 1)
    kind, ctype = _SCATTER_KINDS[dtype]
    nidx = len(index_shapes)
    src = _prelude(numerics) + fill(template("scatter.hip.inc"), dict(
        U=U, OUT=OUT, MODE=mode, KIND=kind, T=ctype, DEST_CODE="\n".join(lines),
        INDEX_PARAMS="".join(f", const int* __restrict__ idx{k}" for k in range(nidx)),
        INDEX_ARGS="".join(f", idx{k}" for k in range(nidx))))
    idx_args = [("in", 1 + k) for k in range(nidx)]
    grid = lambda count: (max(1, min((count + 255) // 256, 1 << 20)), 1, 1)  # noqa: E731
    steps = [LaunchStep("jh_scatter_fill", grid(OUT), (256, 1, 1), 0, [("out", 0), ("scratch", 0)])]
    if U > 0:
        if mode == 1:
            steps.append(LaunchStep("jh_scatter_claim", grid(U), (256, 1, 1), 0, [("scratch", 0)] + idx_args))
        steps.append(LaunchStep("jh_scatter_apply", grid(U), (256, 1, 1), 0, [("in", 0), ("out", 0), ("scratch", 0)] + idx_args))
    need = {0: U * byteWidth(dtype)}
    for k, ishape in enumerate(index_shapes):
        need[1 + k] = prod(ishape) * 4
    return KernelSource([src], steps, [OUT * 4 if mode == 1 else 8], "scatter", need, dict(updates=U, out=OUT, mode=mode, launches=len(steps)))


def _gen_sort(routine: Routine, numerics: str) -> Optional[KernelSource]:
    t = routine.type
    shape, dtype = list(t.inputShapes[0]), t.inputDtypes[0]
    if len(shape) == 0:
        raise ValueError(f"{routine.name.value.lower()}: cannot sort a scalar")
    if dtype not in _SORT_KINDS:
        return None
    n = shape[-1]
    rows = prod(shape[:-1])
    argsort = routine.name == Routines.Argsort
    if n == 0 or rows == 0:
        return KernelSource([], [], [], "sort", {}, dict(n=n, rows=rows))
    if n >= (1 << 30):
        return None
    P = max(_next_pow2(n), 2)
    kind, ctype = _SORT_KINDS[dtype]
    short = argsort and dtype == DType.Float16 and n <= 65536  # key and position in 32 bits
    word = (8 if argsort and not short else 4) * (2 if dtype == DType.Float64 else 1)  # bytes per keyed word
    most = SORT_REGISTERS // word
    values = dict(N=n, P=P, ROWS=rows, ARGSORT=1 if argsort else 0, KIND=kind, T=ctype, GROUP=SORT_GROUP if P > 256 else 4)
    need = {0: rows * n * byteWidth(dtype)}
    outs = [("out", 0), ("out", 1)] if argsort else [("out", 0), ("out", 0)]
    if P <= (64 if word == 4 else 16) * most:
        # 16 lanes per row pair most words inside a lane and reach every other one by DPP; with few rows up to 64, since the
        # launch then waits for one wave's chain.  Sorts gain from registers up to 64 lanes (8000 x 4000 float32: 118 us
        # against 134 through LDS), and so does float16 Argsort, whose words are as wide (8000 x 4000: 104 us, 141 through LDS;
        # 1000 x 3000: 21.5 and 28.2); words of 8 bytes pay for every lane exchange twice (argsort float32 30000 x 1000: 158 us in
        # 32 lanes, 148 through LDS; 3000 x 1000: 23.9 and 21.0).
        E = min(max(2, P // 16), most)
        while E > max(2, P // 64) and rows * (P // E) < SORT_WAVES * 64:
            E //= 2
        E = max(E, P // 64, 1)
        if E <= SORT_FEW or rows * (P // E) >= SORT_FEW_WAVES * 64:
            src = _prelude(numerics) + fill(template("sort.hip.inc"), dict(values, DOUBLES=0, TILE=P, THREADS=256, E=E, W=P, HELD=SORT_HELD))
            steps = [LaunchStep("jh_sort_rows", (-(-rows * (P // E) // 256), 1, 1), (256, 1, 1), 0, [("in", 0)] + outs)]
            return KernelSource([src], steps, [], "sort", need, dict(n=n, rows=rows, P=P, tile=P, argsort=argsort, launches=1))
    tile = min(P, SORT_TILE * 8 // word)
    while tile > SORT_SMALL_TILE and rows * (P // tile) < SORT_FEW_TILES:
        tile //= 2
    # With few tiles the block is as wide as it gets, which finishes its one tile sooner; else longer register runs.
    E = max(min(SORT_LOCAL, most // 2) if rows * (P // tile) >= SORT_TILES else 4, tile // 1024)
    E = min(E, P // 128)  # (runs shorter than the row, of 64 lanes)
    threads = tile // E
    # Words that are doubles where they go through LDS (float32 2000 x 7000: 204 -> 179 us; the register network alone
    # loses by them, 30000 x 1000 in 32 lanes: 206 -> 243).
    doubles = argsort and dtype in (DType.Float32, DType.Int32, DType.Uint32, DType.Bool) and n <= 1 << 20
    opening = SOURCE_OPTION + "-ffinite-math-only\n" if doubles else ""
    src = opening + _prelude(numerics) + fill(template("sort.hip.inc"), dict(values, DOUBLES=1 if doubles else 0, TILE=tile, THREADS=threads, E=E, W=64 * E, HELD=1))
    tiles = rows * (P // tile)
    steps = [LaunchStep("jh_sort_local", (tiles, 1, 1), (threads, 1, 1), 0, [("in", 0), ("scratch", 0)] + outs)]
    k = tile * 2
    while k <= P:
        j = k // 2
        while j >= tile:
            count = min(3, (j // tile).bit_length())
            blocks = max(1, min((rows * (P >> count) + 255) // 256, 1 << 20))
            steps.append(LaunchStep("jh_sort_global", (blocks, 1, 1), (256, 1, 1), 0, [("scratch", 0), ("const", k), ("const", j), ("const", count)]))
            j >>= count
        steps.append(LaunchStep("jh_sort_merge", (tiles, 1, 1), (threads, 1, 1), 0, [("in", 0), ("scratch", 0)] + outs + [("const", k)]))
        k *= 2
    scratch = [rows * P * word] if P > tile else [16]
    return KernelSource([src], steps, scratch, "sort", need, dict(n=n, rows=rows, P=P, tile=tile, argsort=argsort, launches=len(steps)))


def attention_by_queries(heads: int, queries: int, size: int) -> bool:
    """Whether every query takes a workgroup of its own (attention_few.hip.inc) and not a row of a tile of 128.  `heads`
    counts those of all sequences.  Alone on its CU a query reads its keys as fast as they come, where a tile walks 64 at a
    time: 8 x 12 heads over 2048 keys of 64 10 us against 27.  But every query reads them for itself: from 128 heads on
    two to four of them wait for memory, the tile of each head does not (11 x 12 heads, 4 queries, 2048 keys 32 us against
    28, 32 x 12 67 against 41, 64 x 12 156 against 79).  One query stays ahead (64 x 12 71 against 80), in heads of 32
    up to 512 of them (32 x 12 0.93 of the tile's time, 64 x 12 1.25)."""
    if queries == 1:
        return heads <= 512 or size > 32
    return queries <= ATTENTION_FEW_QUERIES and heads <= 128


def attention_copiers(heads: int, keys: int, size: int, threads: int) -> int:
    """Workgroups that write an extended cache beside those that attend to it, which otherwise each write their head's part on the way.

    A workgroup writes at 100 GB/s, and few of them leave the chip idle: a decoding step of 12 heads over 1024 keys of 64 28.4 us apart, 27.5
    on the way, 25.6 beside; over 4096 42.2, 47.5, 38.1; 48 heads over 1024 29.7, 27.8, 26.2, over 2048 37.1, 34.0, 32.3.  With more of them
    the second reading costs more than it hides: 96 heads over 1024 34.1, 29.5, 30.6, over 2048 45.0, 36.8, 41.2; 192 over 1024 44.2, 34.6, 41.1."""
    if heads > tuner.CU_COUNT // 4:
        return 0
    return min(tuner.CU_COUNT - heads, -(-2 * heads * keys * (size // 8) // threads))


def _gen_attention(routine: Routine, numerics: str, appended=None) -> Optional[KernelSource]:
    """Fused attention over [B, L, N, H] / [B, S, N, H] float16 operands with H = 32, 64 or 128 and any L and S >= 1
    (contiguous, or strided views with unit stride along the head dimension).  `appended`: the parts that keys and values are put
    together of (`attentioncache.Appended`); inputs are then q, the parts of k, the parts of v, and outputs the result, k and v."""
    import math

    t = routine.type
    params = routine.params or {}
    if len(t.inputShapes) != 3 or any(len(s) != 4 for s in t.inputShapes):
        raise ValueError("attention: expected q [B,L,N,H], k [B,S,N,H], v [B,S,N,H]")
    (B, L, N, H), ks, vs = t.inputShapes
    if list(ks) != list(vs) or ks[0] != B or ks[2] != N or ks[3] != H:
        raise ValueError(f"attention: shape mismatch q={t.inputShapes[0]} k={ks} v={vs}")
    S = ks[1]
    if any(d != DType.Float16 for d in t.inputDtypes) or H not in (32, 64, 128):
        return None  # the kernel takes float16 and head sizes of one, two or four 32-row MFMA tiles
    if B * N * L == 0:
        return _empty("attention", B=B, L=L, S=S, N=N)
    if B * N * -(-L // 128) >= (1 << 31) or max(B * L * N * H, B * S * N * H) >= (1 << 31):
        return None
    scale = float(params.get("scale", 1 / math.sqrt(H)))
    # Each operand is a base buffer read through (batch, position, head) strides and an offset: contiguous
    # [B, T, N, H] unless the caller passes a view (`params["views"]`, e.g. the q/k/v slices of one QKV projection).
    views = list(params.get("views") or [None, None, None])
    lay, need = [], {}
    for i, T in enumerate((L, S, S)):
        v = views[i]
        if v is None:
            lay.append((T * N * H, N * H, H, 0))
            need[i] = B * T * N * H * 2
        else:
            sb, sp, sn, sh = v["strides"]
            if (sh != 1 and H > 1) or v["offset"] % 8 or sb % 8 or sp % 8 or sn % 8 or min(sb, sp, sn) < 0 or v["elements"] >= (1 << 31):
                return None
            lay.append((sb, sp, sn, v["offset"]))
            need[i] = v["elements"] * 2
    (qb, ql, qn, qo), (kb, ksp, kn, ko), (vb, vsp, vn, vo) = lay
    if attention_by_queries(B * N, L, H):
        lanes = H // 8
        threads = 128
        while threads < 1024 and threads < S * lanes // 2:
            threads *= 2
        passes = -(-S // (threads // lanes))
        rounds = -(-passes // 10)  # ten keys and values of 16 bytes each in flight per thread
        copiers = 0 if appended is None else attention_copiers(B * N, S, H, threads)
        src = _prelude(numerics) + fill(template("attention_few.hip.inc"), dict(
            NH=N, HEADS=B * N, COPIERS=copiers, L=L, S=S, H=H, CAUSAL=1 if params.get("isCausal") else 0, SCALE_LOG2E=repr(scale * math.log2(math.e)), THREADS=threads,
            PASSES=-(-passes // rounds), ROUNDS=rounds, QB=qb, QL=ql, QN=qn, QOFF=qo, OB=L * N * H, OL=N * H, ON=H,
            **(dict(APPENDED=0, KB=kb, KS=ksp, KN=kn, KOFF=ko, VB=vb, VS=vsp, VN=vn, VOFF=vo, **{f"{o}1{x}": 0 for o in "KV" for x in ("B", "S", "N", "OFF")})
               if appended is None else dict(APPENDED=appended[0].first, **{k: v for o, a in zip("KV", appended) for k, v in a.fields(o).items()}))))
        if appended is not None:
            need = {0: need[0], 1: appended[0].need[0], 3: appended[0].need[1], 2: appended[1].need[0], 4: appended[1].need[1]}
            args = [("in", i) for i in range(5)] + [("out", 1), ("out", 2), ("out", 0)]
            return KernelSource([src], [LaunchStep("jh_attention_few", (B * N + copiers, 1, 1), (threads, 1, 1), 0, args)], [], "attention", need, dict(B=B, L=L, S=S, N=N, H=H, blocks=B * N, threads=threads))
        steps = [LaunchStep("jh_attention_few", (B * L * N, 1, 1), (threads, 1, 1), 0, [("in", 0), ("in", 1), ("in", 2), ("out", 0)])]
        return KernelSource([src], steps, [], "attention", need, dict(B=B, L=L, S=S, N=N, H=H, causal=bool(params.get("isCausal")), blocks=B * L * N, threads=threads))
    src = _prelude(numerics) + fill(template("attention.hip.inc"), dict(
        B=B, NH=N, L=L, S=S, H=H, CAUSAL=1 if params.get("isCausal") else 0, SCALE_LOG2E=repr(scale * math.log2(math.e)),
        FOLD_SCALE=1 if 0 < scale < float("inf") else 0,
        QB=qb, QL=ql, QN=qn, QOFF=qo, KB=kb, KS=ksp, KN=kn, KOFF=ko, VB=vb, VS=vsp, VN=vn, VOFF=vo,
        OB=L * N * H, OL=N * H, ON=H))
    blocks = B * N * -(-L // 128)
    steps = [LaunchStep("jh_attention", (blocks, 1, 1), (256, 1, 1), 0, [("in", 0), ("in", 1), ("in", 2), ("out", 0)])]
    return KernelSource([src], steps, [], "attention", need, dict(B=B, L=L, S=S, N=N, H=H, causal=bool(params.get("isCausal")), blocks=blocks))
