"""Plan generation on the host (no GPU): properties every kernel plan must have."""
import pytest

from jaxjs_hip import DType
from jaxjs_hip.kernelgen import generate


def test_every_contraction_shape_gets_a_plan():
    """Plan generation must not raise whatever the extents: rows and columns from 2 to 14336 across the tile sizes, k
    from 32 to 8192 (multiples of the slab depths and not), both layouts of B, float16 and float32.  (A k split folded
    inside the launch used to be chosen for tiles that only the general template can run, which has no such fold.)"""
    import random
    from jaxjs_hip.lowering import matmulKernel
    rng = random.Random(1)
    shapes = [(100, 14336, 4096), (65, 4096, 4096), (127, 14336, 4096), (96, 1000, 4096), (8192, 100, 4096), (300, 300, 8192)]
    rows = [2, 33, 64, 65, 100, 128, 129, 200, 256, 300, 1000, 4096]
    for _ in range(60):
        shapes.append((rng.choice(rows), rng.choice(rows + [14336]), rng.choice([32, 64, 100, 256, 768, 1000, 2048, 4096, 4100, 8192])))
    for dt in (DType.Float16, DType.Float32):
        for shape in shapes:
            for bt in (False, True):
                ks = generate(matmulKernel(*shape, dt, b_transposed=bt), "fast")
                assert ks.steps and ks.sources, (dt, shape, bt)


PINNED_PLANS = [
    # dtype, M, N, K, B stored [N,K] -> what the plan must say
    # whole tiles
    (DType.Float16, 8192, 8192, 8192, False, dict(BM=256, BN=256, direct_lds=True, splitk=1)),
    (DType.Float16, 2048, 2048, 2048, False, dict(BM=128, BN=128, BK=64, stages=4, direct_lds=True, splitk=1)),
    # edge tiles on the direct-to-LDS template: clamped loads
    (DType.Float16, 8000, 8000, 8000, False, dict(BM=256, BN=256, direct_lds=True, splitk=1)),
    (DType.Float16, 1000, 1001, 512, True, dict(BM=128, BN=128, direct_lds=True)),
    (DType.Float16, 100, 14336, 4096, False, dict(BM=128, BN=128, BK=32, direct_lds=True, splitk=2, fused_fold=True)),
    # rows of B off the 16-byte grid: repack pre-pass when the other side has >= 512 rows, the general template below
    (DType.Float16, 8192, 50257, 768, False, dict(BM=256, BN=256, direct_lds=True, repack="b")),
    (DType.Float16, 300, 1001, 512, False, dict(direct_lds=False)),
    # a k axis that is not whole slabs: both operands copied with k padded to 32 (zeros), unless the copies are huge or the
    # shape is small
    (DType.Float16, 4100, 4100, 4100, False, dict(BM=128, BN=256, direct_lds=True, repack="ab")),
    (DType.Float16, 1000, 1000, 1000, True, dict(BM=128, BN=128, direct_lds=True, repack="ab")),
    (DType.Float16, 8192, 768, 50257, False, dict(direct_lds=True, repack="ab")),
    (DType.Float16, 16384, 16384, 16400, False, dict(direct_lds=False, repack=None)),
    (DType.Float16, 300, 300, 1000, False, dict(direct_lds=False, repack=None)),
    # a few rows against a large matrix: clamped rows on 128x128 tiles, k in slices, fold launch
    (DType.Float16, 4, 14336, 4096, False, dict(BM=128, BN=128, BK=32, stages=4, direct_lds=True, splitk=2)),
    (DType.Float16, 31, 4096, 4096, True, dict(BM=128, BN=128, direct_lds=True, splitk=4)),
    (DType.Float16, 16, 14336, 4000, False, dict(BM=64, BN=128, direct_lds=False)),
    # short k under many tiles: shallow stages, several workgroups per CU
    (DType.Float16, 8192, 3072, 768, False, dict(BM=128, BN=256, BK=32, stages=2, direct_lds=True)),
    (DType.Float16, 8192, 768, 3072, False, dict(BM=128, BN=256, stages=4, direct_lds=True)),
    # f32: small shapes in 64x64 tiles with in-launch k slices, the rest unchanged
    (DType.Float32, 256, 256, 256, False, dict(BM=64, BN=64, splitk=4, fused_fold=True)),
    (DType.Float32, 512, 512, 512, True, dict(BM=64, BN=64, splitk=4, fused_fold=True)),
    (DType.Float32, 1024, 1024, 1024, False, dict(BM=128, BN=64, splitk=4, fused_fold=True)),
    (DType.Float32, 4096, 4096, 4096, False, dict(BM=128, BN=128, splitk=1)),
]


def test_gemm_plans_are_pinned():
    """The launch plan the tile chooser picks for the shapes its rules were measured on."""
    from jaxjs_hip.lowering import matmulKernel
    for dt, M, N, K, bt, want in PINNED_PLANS:
        ks = generate(matmulKernel(M, N, K, dt, b_transposed=bt), "fast")
        assert ks.klass.startswith("gemm"), (M, N, K, ks.klass)
        got = {key: ks.info.get(key) for key in want}
        assert got == want, ((dt.value, M, N, K, bt), got, want)
        if want.get("repack"):
            assert [s.name.rsplit("_", 2)[-2] for s in ks.steps][:len(want["repack"])] == ["repack"] * len(want["repack"])
            assert len(ks.scratch_bytes) == len(want["repack"])
        if want.get("repack") == "b" and not bt:
            assert ks.scratch_bytes[0] == K * (-(-N // 8) * 8) * 2


def _direct_lds_load_offsets(rows, bk, nwaves, k_contiguous, row_stride, k_stride, last):
    """Element offsets (from the tile's first row and the slab's first k) of every 16-byte load of one operand slab, as the
    direct-to-LDS template computes them: (tile row or first row of the group, k or first k of the chunk, offset)."""
    out = []
    for q in range(rows * bk * 2 // 1024 // nwaves):
        for wave in range(nwaves):
            inst = q * nwaves + wave
            for lane in range(64):
                if k_contiguous:
                    lpr = bk // 8
                    row = inst * (64 // lpr) + lane // lpr
                    swz = (row >> 2) & 3 if bk == 32 else (row >> 1) & 7
                    lc = (lane % lpr) ^ swz
                    out.append((row, lc * 8, min(row, last) * row_stride + lc * 8))
                else:
                    row_bytes = rows * 2
                    off = lane * 16
                    k = inst * (1024 // row_bytes) + off // row_bytes
                    pc = (off % row_bytes) >> 4
                    lchunk = (((pc >> 2) ^ (k & 3)) << 2) | (pc & 3)
                    lastc = (last + 1) // 8 - 1
                    out.append((lchunk * 8, k, k * k_stride + min(lchunk, lastc) * 8))
    return out


def test_clamped_edge_loads_stay_inside_the_operand():
    """A model of the direct-to-LDS loaders' source addresses (the arithmetic of `jh_lane_offset` with its clamp to the
    last row, or last whole group of eight rows, that exists): for operands whose extent is not whole tiles every
    16-byte load lies inside the operand, and the rows that exist read their own elements."""
    cases = [(8000, 64, 256, 32, 4, True), (8000, 128, 256, 64, 4, True), (8000, 64, 256, 32, 4, False), (136, 64, 128, 32, 4, False),
             (100, 64, 128, 32, 4, True), (50257, 64, 256, 32, 4, True), (50264, 64, 128, 64, 4, False), (8, 64, 128, 32, 4, False),
             (1, 64, 128, 32, 4, True), (4104, 96, 256, 32, 8, False)]
    for extent, K, tile, bk, nwaves, k_contiguous in cases:
        row_stride, k_stride = (K, 1) if k_contiguous else (1, extent)
        for t in range(-(-extent // tile)):
            r0 = t * tile
            last = min(extent - 1 - r0, tile - 1)
            for slab in range(K // bk):
                base = r0 * row_stride + slab * bk * k_stride
                for r, kk, src in _direct_lds_load_offsets(tile, bk, nwaves, k_contiguous, row_stride, k_stride, last):
                    a = base + src
                    assert 0 <= a and a + 8 <= extent * K, (extent, K, tile, t, slab, r, kk)
                    if k_contiguous and r <= last:
                        assert a == (r0 + r) * K + slab * bk + kk
                    if not k_contiguous and r + 7 <= last:
                        assert a == (slab * bk + kk) * extent + r0 + r


def test_interval_form_of_a_mask_matches_the_mask_element_by_element():
    """`gemm.interval_mask_form`: a conjunction of comparisons affine in `e` (coefficient +-1) and terms without `e` is
    rewritten as invariant terms and bounds lo <= e < hi.  Checked against the condition itself on random values of the
    other variables, for every e of a group; conditions outside the form (a coefficient of 2, a comparison of something
    not affine in e) are refused."""
    import random
    from jaxjs_hip.alu import AluExp
    from jaxjs_hip.gemm import interval_mask_form
    I, S = AluExp.i32, AluExp.special
    row, k, e = S(DType.Int32, "row", 4096), S(DType.Int32, "k", 100352), S(DType.Int32, "e", 8)
    NOT = lambda c: AluExp.cmpne(c, AluExp.bool(True))
    x = AluExp.add(AluExp.mod(k, I(56)), AluExp.mod(row, I(3)))          # column of a padded window, before e
    y = AluExp.add(AluExp.mod(AluExp.idiv(k, I(56)), I(56)), AluExp.idiv(row, I(3)))
    conds = {
        "window": AluExp.mul(AluExp.mul(AluExp.cmplt(y, I(57)), NOT(AluExp.cmplt(y, I(1)))),
                             AluExp.mul(AluExp.cmplt(AluExp.add(x, e), I(57)), NOT(AluExp.cmplt(AluExp.add(x, e), I(1))))),
        "flipped": AluExp.mul(AluExp.cmplt(I(3), AluExp.sub(x, e)), NOT(AluExp.cmplt(I(40), AluExp.sub(x, e)))),   # 3 < x - e <= 40
        "both sides": AluExp.cmplt(AluExp.add(e, I(2)), AluExp.sub(x, I(20))),
        "double negation": NOT(NOT(AluExp.cmplt(AluExp.add(e, x), I(30)))),
        "no e at all": AluExp.cmplt(y, I(20)),
    }
    rng = random.Random(5)
    for name, cond in conds.items():
        form = interval_mask_form(cond)
        assert form is not None, name
        inv, lows, highs = form
        for _ in range(300):
            ctx = {"row": rng.randrange(4096), "k": rng.randrange(100352)}
            signed = lambda v: v - (1 << 32) if v >= (1 << 31) else v  # bounds are signed 32-bit values
            lo = max([0] + [signed(b.evaluate(ctx)) for b in lows])
            hi = min([8] + [signed(b.evaluate(ctx)) for b in highs])
            ok = all(bool(t.evaluate(ctx)) for t in inv)
            for ev in range(8):
                want = bool(cond.evaluate(dict(ctx, e=ev)))
                assert want == (ok and lo <= ev < hi), (name, ctx, ev)
    assert interval_mask_form(AluExp.cmplt(AluExp.add(x, AluExp.mul(e, I(2))), I(57))) is None
    assert interval_mask_form(AluExp.cmplt(AluExp.mod(AluExp.add(x, e), I(7)), I(3))) is None


def test_float16_sources_carry_their_compiler_option_and_unknown_options_are_refused():
    """Float16 map and reduce kernels, and matrix kernels with a float16 epilogue beyond bias / ReLU, open with the line
    that switches the SLP vectorizer off for that source; float32 kernels and plain epilogues do not.  The line is
    honoured only for options on the fixed list."""
    import pytest
    from jaxjs_hip import jit as J, library as Lb
    from jaxjs_hip.codegen import SOURCE_OPTION
    from jaxjs_hip.errors import HipRuntimeError
    from jaxjs_hip.jit import ShapedArray
    from jaxjs_hip.runtime import compile_source
    line = SOURCE_OPTION + "-fno-slp-vectorize\n"

    def sources(fn, shapes, dtype):
        prog = J.jit(fn, [ShapedArray(s, dtype) for s in shapes])
        return [generate(k, "fast") for k in prog.kernels]

    for dtype, expect in ((DType.Float16, True), (DType.Float32, False)):
        gens = sources(lambda x: Lb.logSoftmax(x, -1), [(16, 1001)], dtype)
        assert {g.klass for g in gens} == {"reduce_row", "map"}
        assert all(g.sources[0].startswith(line) == expect for g in gens)
    mm = [(256, 256), (256, 256)]
    (neg,) = sources(lambda a, b: J.neg(Lb.matmul(a, b)), mm, DType.Float16)
    (relu,) = sources(lambda a, b: Lb.relu(Lb.matmul(a, b)), mm, DType.Float16)
    (neg32,) = sources(lambda a, b: J.neg(Lb.matmul(a, b)), mm, DType.Float32)
    assert neg.klass == relu.klass == neg32.klass == "gemm"
    assert neg.sources[0].startswith(line) and not relu.sources[0].startswith(line) and not neg32.sources[0].startswith(line)
    with pytest.raises(HipRuntimeError, match="not on the list"):
        compile_source(SOURCE_OPTION + "-O0\nextern \"C\" __global__ void k() {}\n", use_cache=False)


def test_wide_load_of_a_looked_up_row_reads_what_the_guarded_element_loads_read():
    """The claim behind the `vector_gm` load class, by brute force over int32 ids (extremes, multiples of the table
    length of either sign, values whose product with the row width wraps): with x = wrap(wrap(id * W) + r0 + lane),
    element loads read `x % C` (C remainder, sign of x) when it lies in [0, C) and element 0 otherwise; the wide load
    reads `x0 % C + lane` when x0 >= 0 and the remainder is in range, element 0 in every lane otherwise."""
    import numpy as np
    from jaxjs_hip import jit as J, library as Lb
    from jaxjs_hip.jit import ShapedArray

    def wrap(v):
        return (v + 2**31) % 2**32 - 2**31

    def crem(a, b):
        return a - b * int(a / b)  # truncating division, exact for |a| < 2^53

    rng = np.random.default_rng(5)
    for rows, W, V in ((50257, 768, 8), (77, 64, 8), (1000, 8, 4), (3, 16, 8)):
        C = rows * W
        ids = [0, 1, -1, rows - 1, rows, -rows, 2 * rows, -2 * rows, 2**31 - 1, -2**31, 2**31 // W, -(2**31 // W), 2**32 // W + 1]
        ids += [int(v) for v in rng.integers(-2**31, 2**31, 200)] + [int(v) for v in rng.integers(-3 * rows, 3 * rows, 200)]
        for i in ids:
            for r0 in range(0, W, V):
                x0 = wrap(wrap(i * W) + r0)
                each = [crem(wrap(x0 + lane), C) for lane in range(V)]
                each = [f if 0 <= f < C else 0 for f in each]
                f0 = crem(x0, C)
                inside = x0 >= 0 and 0 <= f0 < C
                assert each == ([f0 + lane for lane in range(V)] if inside else [0] * V), (rows, W, i, r0)
    prog = J.jit(lambda t, i: Lb.take(t, i, 0), [ShapedArray((1000, 768), DType.Float16), ShapedArray((64,), DType.Int32)])
    from jaxjs_hip.tuner import tuneHip
    assert "vector_gm" in tuneHip(prog.kernels[0]).vector_loads.values()


@pytest.mark.parametrize("order,batch,dtype,plan", [
    # microseconds of a wave per matrix against a launch per panel, when the lines were drawn -> as the kernels are now
    (8, 1, DType.Float32, "wave per matrix"), (8, 65536, DType.Float64, "wave per matrix"),              # 7 and 7; -> 132 and 466
    (12, 768, DType.Float32, "right-looking"), (12, 1024, DType.Float32, "wave per matrix"),             # 12 and 9; 12 and 15 -> 14 and 10; 15 and 11
    (12, 512, DType.Float64, "right-looking"), (12, 768, DType.Float64, "wave per matrix"),              # 9 and 9; 9 and 16 -> 11 and 9; 11 and 12
    (24, 1024, DType.Float32, "right-looking"), (24, 4096, DType.Float32, "wave per matrix"),            # 27 and 19; 47 and 56 -> 30 and 14; 55 and 39
    (28, 16384, DType.Float32, "right-looking"), (28, 4096, DType.Float16, "wave per matrix"),           # 266 and 249; 65 and 99 -> 278 and 145; 71 and 56
    (40, 4096, DType.Float16, "wave per matrix"), (48, 16384, DType.Float16, "right-looking"),           # 128 and 168; 768 and 725 -> 136 and 122; 770 and 477
    (191, 1024, DType.Float32, "right-looking"),
    # of two launches per panel against one, likewise
    (192, 512, DType.Float32, "right-looking"), (192, 1024, DType.Float32, "two launches"),              # 379 and 327; 576 and 604 -> 401 and 221; 595 and 382
    (512, 128, DType.Float32, "right-looking"), (512, 512, DType.Float32, "two launches"),               # 1174 and 1000; 3000 and 3501 -> 1189 and 651; 3007 and 2159
    (512, 128, DType.Float64, "two launches"), (1024, 32, DType.Float64, "right-looking"),               # 1188 and 1235; 2135 and 1896 -> 1174 and 785; 2125 and 1211
    (1024, 1, DType.Float32, "right-looking"), (1024, 256, DType.Float32, "left-looking"),               # (2 GiB of running sums)
], ids=str)
def test_cholesky_s_plan_follows_the_number_of_matrices(order, batch, dtype, plan):
    from jaxjs_hip.alu import byteWidth
    from jaxjs_hip.routine import Routine, Routines, RoutineType
    from jaxjs_hip.routinegen import _cholesky_plan, generateRoutine
    assert _cholesky_plan(order, batch, byteWidth(dtype)) == plan
    shape = [batch, order, order]
    first = generateRoutine(Routine(Routines.Cholesky, RoutineType([shape], [dtype], [shape], [dtype]))).steps[0].name
    assert first == {"wave per matrix": "jh_cholesky", "right-looking": "jh_chol_step", "two launches": "jh_chol_init", "left-looking": "jh_chol_zero"}[plan]


@pytest.mark.parametrize("order,batch,dtype,blocks", [
    # milliseconds by blocks against one rotation after the other
    (16, 256, DType.Float32, True), (16, 257, DType.Float32, False),      # 0.32 and 0.46; 0.55 and 0.43 (300)
    (32, 512, DType.Float32, True), (32, 513, DType.Float32, False),      # 1.44 and 2.12; 2.16 and 2.18 (768)
    (48, 768, DType.Float32, True), (48, 1024, DType.Float32, False),     # 4.3 and 5.4; 5.0 and 5.3
    (64, 2048, DType.Float32, True), (128, 4096, DType.Float32, True),    # 16.5 and 28.3: those wait for each other too; 103 and 776
    (64, 2048, DType.Float64, True), (48, 1024, DType.Float64, False),    # 16.5 and 46.0; 5.7 and 6.1
    (48, 512, DType.Float16, False), (64, 512, DType.Float16, True),      # 5.7 and 7.1; 9.2 and 14.2
    (64, 1024, DType.Float16, False), (160, 4096, DType.Float32, True),   # 18.3 and 16.7; (too large for LDS)
    (13, 2, DType.Float32, True), (13, 2, DType.Float16, False), (12, 1, DType.Float32, False),
], ids=str)
def test_jacobi_eigh_s_plan_follows_the_number_of_matrices(order, batch, dtype, blocks):
    from jaxjs_hip.routine import Routine, Routines, RoutineType
    from jaxjs_hip.routinegen import generateRoutine
    shape = [batch, order, order]
    ks = generateRoutine(Routine(Routines.JacobiEigh, RoutineType([shape], [dtype], [shape] * 2, [dtype] * 2), dict(maxSweeps=30, tolerance=1e-7)))
    assert ks.steps[0].name == ("jh_jacobi_blocks" if blocks else "jh_jacobi") and ("block" in ks.info) == blocks


FEW = "few"  # gemm_few.hip.inc
PRODUCT_PLANS = [
    # dtype, M, N, K, B stored [N, K] -> the kernel that takes it, and microseconds of it and of what it is chosen over
    (DType.Float32, 64, 256, 784, False, FEW),                # 4.0 and 22.3 in tiles
    (DType.Float32, 300, 300, 300, False, FEW),               # 3.4 and 10.1
    (DType.Float32, 45, 2133, 3712, True, "gemm"),            # 27 and 35
    (DType.Float32, 61, 10492, 1444, True, "gemm"),           # 38 and 58
    (DType.Float32, 56, 5248, 1856, False, "gemm"),           # 28 and 41
    (DType.Float16, 64, 256, 784, False, FEW),                # 2.9 and 12.0
    (DType.Float16, 64, 1024, 1024, False, FEW),              # 3.3 and 8.0
    (DType.Float16, 64, 2048, 4096, False, "gemm+fold"),      # 10.2 and 11.9
    (DType.Float16, 16, 14336, 4096, False, "gemm+fold"),     # 25.8 and 32
    (DType.Float16, 3, 9287, 5632, False, FEW),               # 33 and 46.5: rows off the 16-byte grid
    (DType.Float16, 64, 10112, 4416, True, "gemm"),           # 30 and 53
    (DType.Float16, 40, 8896, 704, True, "gemm"),             # 7.2 and 9.6
    (DType.Float16, 42, 10240, 512, False, FEW),              # 5.8 and 9.0
    (DType.Float16, 64, 2304, 5248, True, "gemm+fold"),       # 20 and 29
    # a handful of rows: of the reductions
    (DType.Float16, 1, 768, 768, False, FEW),                 # 3.1 and 6.3
    (DType.Float16, 1, 768, 3072, True, "reduce_row"),        # 3.0 and 4.9
    (DType.Float16, 12, 54, 576, False, FEW),                 # 2.7 and 5.6
    (DType.Float16, 1, 11008, 4096, False, "reduce_col+fold"),
    (DType.Float32, 22, 452, 1280, False, FEW),               # 5.3 and 6.7
    (DType.Float32, 30, 94, 1504, False, "reduce_col+fold"),  # 5.3 and 6.6
    (DType.Float32, 26, 128, 3072, False, "reduce_col+fold"),  # 6.0 and 11.4
]


@pytest.mark.parametrize("dtype,m,n,k,transposed,taken", PRODUCT_PLANS, ids=str)
def test_products_of_few_rows_or_tiles_take_the_kernel_that_was_measured_faster(dtype, m, n, k, transposed, taken):
    from jaxjs_hip.lowering import matmulKernel
    ks = generate(matmulKernel(m, n, k, dtype, b_transposed=transposed), "fast")
    assert (FEW if ks.info.get("few") else ks.klass) == taken


@pytest.mark.parametrize("heads,queries,size,by_queries", [
    # microseconds of a workgroup per query and of tiles, 2048 keys
    ((8, 12), 1, 64, True), ((64, 12), 1, 64, True), ((64, 12), 1, 128, True),     # 10 and 27; 71 and 80
    ((32, 12), 1, 32, True), ((64, 12), 1, 32, False),                             # 0.93 and 1.25 of the tiles' time
    ((8, 12), 4, 64, True), ((4, 32), 4, 64, True), ((11, 12), 4, 64, False),      # 21 and 27; 21 and 29; 32 and 28
    ((32, 12), 2, 64, False), ((64, 12), 4, 128, False), ((1, 1), 5, 64, False),   # 57 and 43; 1.8 of the tiles' time
], ids=str)
def test_attention_takes_a_workgroup_per_query_only_for_few_queries_of_few_heads(heads, queries, size, by_queries):
    from jaxjs_hip.routine import Routine, Routines, RoutineType
    from jaxjs_hip.routinegen import generateRoutine
    B, N = heads
    shapes = [[B, t, N, size] for t in (queries, 2048, 2048)]
    ks = generateRoutine(Routine(Routines.Attention, RoutineType(shapes, [DType.Float16] * 3, [shapes[0]], [DType.Float16]), dict(scale=0.125)))
    assert [s.name for s in ks.steps] == ["jh_attention_few" if by_queries else "jh_attention"]


@pytest.mark.parametrize("shape", [(140000, 8, 512), (3, 8, 100_000_000), (9_000_000, 8, 16), (2_000_000, 70, 33), (1 << 25, 1, 1200), (70000, 65, 800)], ids=str)
def test_lu_s_launches_hold_fewer_than_2_to_the_32_threads(shape):
    """Every strip of every matrix once, in launches of the size that the device takes."""
    from jaxjs_hip.routine import Routine, Routines, RoutineType
    from jaxjs_hip.routinegen import generateRoutine

    batch, m, n = shape
    ks = generateRoutine(Routine(Routines.LU, RoutineType([shape], [DType.Float32], [shape, (batch, min(m, n)), (batch, m)], [DType.Float32, DType.Int32, DType.Int32])))
    assert all(s.grid[0] * s.block[0] < 1 << 32 for s in ks.steps)
    if ks.info["variant"] == "by matrix":
        assert [s.grid for s in ks.steps] == [(batch, 1, 1)]
        return
    done = {}
    for s in ks.steps:
        if s.name == "jh_lu_strip":
            mat, j, first = (c for kind, c in s.args if kind == "const")
            assert first == done.get((mat, j), 0)
            done[mat, j] = first + s.grid[0]
    width = max(8, min(32, 1 << (min(m, n) - 1).bit_length()))
    panels = [(s.args[-2][1], s.args[-1][1], s.grid[0]) for s in ks.steps if s.name == "jh_lu_panel"]
    assert sum(mats for _mat, j, mats in panels if j == 0) == batch
    for mat, j, mats in panels:
        assert done.get((mat, j), 0) == mats * (-(-j // 8) + -(-(n - min(j + width, m, n)) // 8))
    assert max(done.values(), default=0) < 1 << 32 or "(unsigned long long)first + blockIdx.x" in ks.sources[0]


@pytest.mark.parametrize("batch,m,n,eb,by_matrix", [(1202, 3, 272, 4, True), (1, 5, 256, 4, True), (24, 3, 2000, 4, False), (829, 12, 1078, 4, True), (40, 12, 1078, 4, False), (13646, 34, 34, 4, True),
                                                    (855, 57, 57, 2, False), (21, 75, 262, 8, False), (500, 49, 900, 8, False), (500, 49, 900, 4, True), (5000, 100, 64, 4, False),
                                                    (11900, 3, 3, 2, True), (11900, 3, 3, 4, False), (5681, 14, 3, 2, False), (1 << 25, 1, 1200, 4, False), (9000, 27, 6, 2, False)], ids=str)
def test_which_lu_goes_by_matrix(batch, m, n, eb, by_matrix):
    from jaxjs_hip import routinegen

    assert routinegen._lu_by_matrix(m, n, batch, eb) == by_matrix


@pytest.mark.parametrize("shape", [(1 << 20, 4096, 1), (2_000_000, 64, 64), (500_000, 130, 200), (1 << 22, 9, 7), (3, 4096, 4096)], ids=str)
@pytest.mark.parametrize("dtype", [DType.Float16, DType.Float32, DType.Float64], ids=str)
def test_lu_s_workspace_does_not_grow_with_the_batch(shape, dtype):
    """Multipliers of a panel in double are up to sixteen times as large as a batch of thin matrices."""
    from jaxjs_hip.routine import Routine, Routines, RoutineType
    from jaxjs_hip.routinegen import LU_SCRATCH, generateRoutine

    batch, m, n = shape
    ks = generateRoutine(Routine(Routines.LU, RoutineType([shape], [dtype], [shape, (batch, min(m, n)), (batch, m)], [dtype, DType.Int32, DType.Int32])))
    if ks.info["variant"] == "by matrix":
        assert not ks.scratch_bytes
        return
    assert ks.scratch_bytes[0] <= LU_SCRATCH and sum(ks.scratch_bytes) <= 1.2 * LU_SCRATCH
    sizes = [s.grid[0] for s in ks.steps if s.name == "jh_lu_panel"]
    assert min(sizes[:1]) >= min(batch, 512)


@pytest.mark.parametrize("m,n,k", [(652, 896, 704), (512, 1408, 768), (192, 3904, 832), (448, 1536, 576), (2072, 256, 640), (608, 832, 576), (1080, 512, 640), (1024, 1024, 1024),
                                   (960, 384, 3696), (256, 256, 256)], ids=str)
def test_direct_loads_make_no_chain_of_roundings_longer(m, n, k):
    """A wave adds half of its part of a slice in a row; staged in registers it is a whole slice."""
    from jaxjs_hip import gemm, tuner
    from jaxjs_hip.lowering import matmulKernel

    kernel = matmulKernel(m, n, k, DType.Float32)
    assert gemm.is_direct_product(kernel)
    g = tuner.tuneHip(kernel).gemm
    staged, direct = gemm.choose_tile(dict(g, direct=False)), gemm.choose_tile(dict(g, direct=True))
    assert not staged.get("DLDS") and direct["DLDS"]
    assert 2 * direct["WK"] * direct.get("SPLITK", 1) >= staged.get("SPLITK", 1)


@pytest.mark.parametrize("batch,m,n,k,direct", [
    (2, 224, 128, 1792, False), (3, 192, 256, 512, False), (6, 96, 224, 2048, False), (1, 256, 48, 30720, False), (1, 32, 576, 26624, False), (1, 60, 192, 18432, False), (2, 64, 64, 128, False),
    (2, 256, 512, 256, True), (2, 256, 512, 512, False), (2, 512, 512, 512, True), (2, 512, 512, 1024, False), (24, 128, 128, 512, False), (24, 256, 256, 512, True), (12, 512, 512, 32, False), (12, 512, 512, 64, True), (1, 48, 320, 17408, False), (1, 32, 576, 17408, True)],
    ids=str)
def test_products_cut_finer_than_direct_loads_cut_them_keep_their_plan(batch, m, n, k, direct):
    """Batches, which direct loads cut into no slices, and few rows behind a long axis, staged in up to 64 of them."""
    from jaxjs_hip import gemm, jit as J, library as L, tuner
    from jaxjs_hip.jit import ShapedArray
    from jaxjs_hip.kernelgen import generate
    from jaxjs_hip.schedule import plan_units

    lead = (batch,) if batch > 1 else ()
    unit, = plan_units(J.jit(lambda a, b: L.matmul(a, b), [ShapedArray(lead + (m, k), DType.Float32), ShapedArray(lead + (k, n), DType.Float32)]))
    generate(unit.source, **unit.options)
    g = tuner.tuneHip(unit.source).gemm
    staged, taken = gemm.choose_tile(dict(g, direct=False)), gemm.choose_tile(dict(g, direct=bool(unit.options)))
    assert unit.options == (dict(direct_f32=True) if direct else {}) and bool(taken.get("DLDS")) == direct
    assert taken == staged or 2 * taken["WK"] * taken.get("SPLITK", 1) >= staged.get("SPLITK", 1)


@pytest.mark.parametrize("m,n,k,reads,direct", [(784, 3664, 64, True, False), (784, 3664, 64, False, True), (3852, 684, 184, True, False), (1900, 484, 88, True, True),
                                                (3300, 2144, 352, True, True), (2264, 3808, 60, True, False), (4096, 4096, 64, True, False), (4096, 4096, 64, False, True)], ids=str)
def test_epilogues_that_read_behind_short_axes_keep_products_staged(m, n, k, reads, direct):
    from jaxjs_hip import jit as J, library as L
    from jaxjs_hip.jit import ShapedArray
    from jaxjs_hip.kernelgen import generate
    from jaxjs_hip.schedule import plan_units

    a, b, c = (ShapedArray(s, DType.Float32) for s in ((m, k), (k, n), (m, n)))
    unit, = plan_units(J.jit(lambda a, b, *c: L.matmul(a, b).add(c[0]) if c else L.matmul(a, b), [a, b, c] if reads else [a, b]))
    assert ("global_load_lds_dwordx4" in generate(unit.source, **unit.options).sources[0]) == direct


@pytest.mark.parametrize("n,m,mats,plan", [(256, 1, 300, (8, 4)), (128, 1, 4096, (8, 4)), (100, 1, 16384, (8, 4)), (48, 1, 600, (8, 8)), (256, 20, 512, (32, 4)), (128, 1, 256, (8, 32)),
                                           (609, 14, 1, (8, 12)), (1284, 28, 68, (8, 3)), (64, 65, 250, (64, 4)), (100, 1, 16385, None), (2048, 8, 1, None)], ids=str)
def test_few_right_hand_sides_are_counted_by_workgroup(n, m, mats, plan):
    """No workgroup holds right-hand sides of two matrices: what makes them few is how many workgroups that is."""
    from jaxjs_hip import routinegen

    assert routinegen._trisolve_few(n, m, mats) == plan
