"""The fused attention kernel (an extension routine, `Routines.Attention`) on the GPU against the float64 checker, and
the GPT-2 block traced with it against the block traced the reference's way.  Float16 in, float16 out, f32 softmax
statistics: bound = 1e-2 relative + a few f16 ulps of values of order 1 (the stated f16 tolerance)."""
import math

import numpy as np
import pytest

import routine_util as R
from gpu_util import WARM_ONLY, backend
from jaxjs_hip import DType
from jaxjs_hip import workloads as W
from jaxjs_hip.errors import UnsupportedRoutineError
from jaxjs_hip.routine import Routine, Routines, RoutineType
from jit_util import run_program
from test_jit import block_inputs, block_reference

pytestmark = pytest.mark.gpu
F16 = DType.Float16


def attention_routine(B, L, S, N, causal, scale=None, H=64):
    t = RoutineType([[B, L, N, H], [B, S, N, H], [B, S, N, H]], [F16] * 3, [[B, L, N, H]], [F16])
    return Routine(Routines.Attention, t, dict(scale=1 / math.sqrt(H) if scale is None else scale, isCausal=causal))


CASES = [(1, 128, 64, 1, 64), (1, 128, 128, 1, 64), (2, 256, 256, 3, 64), (1, 384, 192, 2, 64), (1, 128, 320, 2, 64), (2, 1024, 1024, 4, 64),
         # other head sizes, and lengths that are not whole tiles (a last query block and a last key tile that are partly
         # empty, fewer queries than a wave holds, one key)
         (2, 256, 256, 2, 32), (1, 256, 192, 3, 128), (1, 100, 128, 1, 64), (1, 128, 100, 1, 64), (2, 77, 333, 3, 32), (1, 130, 65, 2, 128),
         (1, 1, 1, 1, 64), (3, 5, 700, 2, 64), (1, 1000, 1000, 2, 128), (2, 513, 511, 1, 32)]


@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "B%d_L%d_S%d_N%d_H%d" % c)
def test_attention_matches_float64(case, causal):
    B, L, S, N, H = case
    rng = np.random.default_rng(B * 1000 + L + S + N + H)
    q, k, v = [rng.standard_normal((B, T, N, H)).astype(np.float16) for T in (L, S, S)]
    routine = attention_routine(B, L, S, N, causal, H=H)
    got, ks = R.run_gpu(routine, [q, k, v])
    want = R.run_oracle(routine, [q, k, v])
    np.testing.assert_allclose(got[0].astype(np.float64), want[0].astype(np.float64), rtol=1e-2, atol=3e-3, err_msg=str(ks.info))


@pytest.mark.parametrize("case", [(2, 1, 1, 3, 64), (1, 2, 2, 1, 32), (3, 1, 63, 2, 128), (2, 4, 129, 2, 64), (8, 1, 1025, 12, 64), (1, 3, 1281, 2, 64), (1, 1, 5000, 2, 32)],
                         ids=lambda c: "B%d_L%d_S%d_N%d_H%d" % c)
@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
def test_attention_of_few_queries(case, causal):
    """One workgroup per query: one pass and several, several rounds, key counts around the passes, every head size."""
    B, L, S, N, H = case
    rng = np.random.default_rng(S + H)
    q, k, v = [rng.standard_normal((B, T, N, H)).astype(np.float16) for T in (L, S, S)]
    routine = attention_routine(B, L, S, N, causal, H=H)
    got, ks = R.run_gpu(routine, [q, k, v])
    want = R.run_oracle(routine, [q, k, v])
    assert ks.info["blocks"] == B * L * N
    np.testing.assert_allclose(got[0].astype(np.float64), want[0].astype(np.float64), rtol=2e-3, atol=1e-3, err_msg=str(ks.info))


def test_attention_is_stable_for_large_scores_and_peaked_rows():
    rng = np.random.default_rng(4)
    q, k, v = [rng.standard_normal((1, 256, 2, 64)).astype(np.float16) for _ in range(3)]
    q *= np.float16(6.0)   # scores of order +-50: exp would overflow f16/f32 without the running maximum
    k[:, 17] *= np.float16(4.0)  # one dominant key
    for causal in (False, True):
        routine = attention_routine(1, 256, 256, 2, causal, scale=1.0)
        got, _ = R.run_gpu(routine, [q, k, v])
        want = R.run_oracle(routine, [q, k, v])
        assert np.isfinite(got[0]).all()
        np.testing.assert_allclose(got[0].astype(np.float64), want[0].astype(np.float64), rtol=1e-2, atol=4e-3)


@pytest.mark.parametrize("scale", [-0.125, 0.0, 1e-3, 3.0], ids=lambda s: "scale%g" % s)
def test_attention_takes_any_scale(scale):
    """A scale that is zero or negative does not commute with the row maximum (the kernel then scales the scores before
    taking it); ragged lengths so the masked key tile and the diagonal are covered under both forms."""
    rng = np.random.default_rng(11)
    q, k, v = [rng.standard_normal((2, T, 2, 64)).astype(np.float16) for T in (200, 200, 200)]
    for causal in (False, True):
        routine = attention_routine(2, 200, 200, 2, causal, scale=scale)
        got, _ = R.run_gpu(routine, [q, k, v])
        want = R.run_oracle(routine, [q, k, v])
        assert np.isfinite(got[0]).all()
        np.testing.assert_allclose(got[0].astype(np.float64), want[0].astype(np.float64), rtol=1e-2, atol=4e-3)


def _view(strides, offset, shape):
    return dict(strides=list(strides), offset=offset, elements=offset + sum((d - 1) * s for d, s in zip(shape, strides)) + 1)


@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
def test_attention_reads_operands_through_strides(causal):
    """q, k and v as three windows of one [B, L, 3*N*64] buffer (the output of a fused QKV projection), and k/v stored
    head-major ([B, N, S, 64]): the routine takes the base buffers with strides and offsets, no copies."""
    B, L, N, H = 2, 256, 3, 64
    rng = np.random.default_rng(11)
    qkv = rng.standard_normal((B, L, 3 * N * H)).astype(np.float16)
    t = RoutineType([[B, L, N, H]] * 3, [F16] * 3, [[B, L, N, H]], [F16])
    st = (L * 3 * N * H, 3 * N * H, H, 1)
    views = [_view(st, i * N * H, (B, L, N, H)) for i in range(3)]
    routine = Routine(Routines.Attention, t, dict(scale=0.125, isCausal=causal, views=views))
    got, ks = R.run_gpu(routine, [qkv, qkv, qkv])
    q, k, v = [qkv[..., i * N * H:(i + 1) * N * H].reshape(B, L, N, H) for i in range(3)]
    want = R.run_oracle(attention_routine(B, L, L, N, causal), [q, k, v])
    np.testing.assert_allclose(got[0].astype(np.float64), want[0].astype(np.float64), rtol=1e-2, atol=3e-3)
    np.testing.assert_array_equal(R.run_oracle(routine, [qkv, qkv, qkv])[0], want[0])  # the checker reads views too
    # head-major keys and values, contiguous queries
    kh, vh = [np.ascontiguousarray(np.transpose(a, (0, 2, 1, 3))) for a in (k, v)]
    hm = _view((N * L * H, H, L * H, 1), 0, (B, L, N, H))
    routine = Routine(Routines.Attention, t, dict(scale=0.125, isCausal=causal, views=[None, hm, hm]))
    got2, _ = R.run_gpu(routine, [np.ascontiguousarray(q), kh, vh])
    np.testing.assert_array_equal(got2[0], got[0])


def test_strided_operands_the_kernel_cannot_load_are_refused():
    if WARM_ONLY:
        pytest.skip("nothing to compile")
    B, L, N, H = 1, 128, 1, 64
    t = RoutineType([[B, L, N, H]] * 3, [F16] * 3, [[B, L, N, H]], [F16])
    for bad in (_view((L * N * H, N * H, H, 1), 4, (B, L, N, H)), _view((L * N * H * 2, N * H * 2, H * 2, 2), 0, (B, L, N, H)),
                _view((L * 68, 68, 68, 1), 0, (B, L, N, H))):
        with pytest.raises(UnsupportedRoutineError):
            backend().prepareRoutineSync(Routine(Routines.Attention, t, dict(scale=0.125, isCausal=False, views=[bad, None, None])))


def test_shapes_outside_the_kernel_are_refused_not_faked():
    if WARM_ONLY:
        pytest.skip("nothing to compile")
    be = backend()
    t32 = RoutineType([[1, 128, 1, 64]] * 3, [DType.Float32] * 3, [[1, 128, 1, 64]], [DType.Float32])
    for routine in (attention_routine(1, 128, 128, 1, False, H=16), attention_routine(1, 128, 128, 1, False, H=96),
                    Routine(Routines.Attention, t32, dict(scale=0.125, isCausal=False))):
        with pytest.raises(UnsupportedRoutineError):
            be.prepareRoutineSync(routine)


def test_reference_attention_tables_on_the_fused_kernel():
    """test/nn.test.ts:275-390 on the fused kernel.  The tables use head sizes of 2 and 4; the operands are padded with
    zeros to 32 (dot products and the meaningful output columns are unchanged) and the scale is the table's own
    1/sqrt(H).  Two or three queries and keys: every tile is ragged."""
    def run(q, k, v, scale, causal):
        H0 = np.asarray(q).shape[-1]
        pad = lambda a: np.pad(np.asarray(a, np.float16), [(0, 0)] * 3 + [(0, 32 - H0)])  # noqa: E731
        q, k, v = pad(q), pad(k), pad(v)
        routine = attention_routine(q.shape[0], q.shape[1], k.shape[1], q.shape[2], causal, scale=scale, H=32)
        got, _ = R.run_gpu(routine, [q, k, v])
        out = got[0].astype(np.float64).reshape(q.shape)
        assert not out[..., H0:].any()
        return out[..., :H0]
    q = [[[[1, 0, 0, 0]], [[0, 1, 0, 0]]]]
    out = run(q, q, [[[[1, 2, 3, 4]], [[5, 6, 7, 8]]]], 0.5, False)
    np.testing.assert_allclose(out[0, 0, 0], [0.62245935 * a + 0.37754068 * b for a, b in zip((1, 2, 3, 4), (5, 6, 7, 8))], rtol=2e-3)
    e = [[[[1, 0]], [[0, 1]]]]
    out = run(e, e, e, 1.0, False)
    np.testing.assert_allclose(out[0, 0, 0], [0.7310586, 0.26894143], rtol=2e-3)
    out = run([[[[1, 0]], [[0.2, 0.2]], [[1, 1]]]], [[[[1, 0]], [[0, 1]], [[1, 1]]]], [[[[1, 0]], [[0, 1]], [[0, 0]]]], 1 / math.sqrt(2), True)
    np.testing.assert_allclose(out[0, 0, 0], [1, 0], atol=1e-3)
    np.testing.assert_allclose(out[0, 1, 0], [0.5, 0.5], rtol=2e-3)
    np.testing.assert_allclose(out[0, 2, 0], [1 / (2 + math.exp(math.sqrt(0.5)))] * 2, rtol=2e-3)


def test_gpt2_block_with_fused_attention():
    """Small block (d=128, 2 heads of 64): fused against the float64 block restatement and against the unfused program
    on the same GPU.  The front-end switch falls back to the reference's composition when the shapes do not fit."""
    batch, seq, d, heads, d_ff = 2, 128, 128, 2, 512
    fused = W.gpt2BlockProgram(batch, seq, d, heads, d_ff, fusedAttention=True)
    plain = W.gpt2BlockProgram(batch, seq, d, heads, d_ff)
    assert [r.name for r in fused.routines] == [Routines.Attention] and not plain.routines
    assert len(fused.kernels) == len(plain.kernels) - 7  # seven attention kernels out; q, k, v are views of the QKV output
    assert all(v is not None for v in fused.routines[0].params["views"])
    assert not W.gpt2BlockProgram(batch, seq, d, 8, d_ff, fusedAttention=True).routines  # heads of 16: composition kept
    assert W.gpt2BlockProgram(batch, 100, d, 4, d_ff, fusedAttention=True).routines     # heads of 32, a ragged length: fused
    if WARM_ONLY:
        from test_programs_gpu import warm
        warm(fused)
    arrs = block_inputs(batch, seq, d, d_ff, np.float16)
    order = ["x"] + list(W.GPT2_BLOCK_PARAMS)
    arrays = [arrs[n] for n in order]
    (y,) = run_program(backend(), fused, arrays)
    (y0,) = run_program(backend(), plain, arrays)
    want = block_reference(arrs["x"].astype(np.float64), {n: arrs[n].astype(np.float64) for n in order[1:]}, heads)
    np.testing.assert_allclose(y.astype(np.float64).reshape(batch, seq, d), want, rtol=3e-2, atol=3e-2)
    np.testing.assert_allclose(y.astype(np.float64), y0.astype(np.float64), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("shape", [(2, 40, 40, 3, 32), (1, 1, 77, 4, 64), (2, 130, 65, 1, 128)], ids=str)
def test_composed_attention_runs_as_the_routine(shape, causal):
    """The front-end's composition is recognised when a program is scheduled: same result within float16."""
    from jaxjs_hip import jit as J
    from jaxjs_hip import library as L_
    from jaxjs_hip.jit import ShapedArray
    from jaxjs_hip.schedule import Schedule
    from oracle.backend import OracleBackend
    B, L, S, N, H = shape
    rng = np.random.default_rng(S)
    arrays = [rng.standard_normal((B, T, N, H)).astype(np.float16) for T in (L, S, S)]
    prog = J.jit(lambda q, k, v: L_.dotProductAttention(q, k, v, isCausal=causal), [ShapedArray(a.shape, F16) for a in arrays])
    assert not prog.routines
    if WARM_ONLY:
        pytest.skip("warm-up run")
    be = backend()
    names = [str(getattr(u.source, "name", "")) for u in Schedule(be, prog).units]
    assert names == ["Attention"], names
    got, want = run_program(be, prog, arrays), run_program(OracleBackend(), prog, arrays)
    np.testing.assert_allclose(got[0].astype(np.float64), want[0].astype(np.float64), rtol=1e-2, atol=3e-3)


def test_a_chain_whose_scores_are_used_elsewhere_stays_as_it_is():
    from jaxjs_hip import jit as J
    from jaxjs_hip import library as L_
    from jaxjs_hip.jit import ShapedArray
    from jaxjs_hip.rewrite import fuse_attention

    def f(q, k, v):
        scores = L_.einsum("BLNH,BSNH->BNLS", q, k)
        p = L_.softmax(scores, -1)
        return [L_.einsum("BNLS,BSNH->BLNH", p, v), p]
    prog = J.jit(f, [ShapedArray((1, 8, 2, 32), F16)] * 3)
    assert fuse_attention(prog.jaxpr, prog.consts) is None


@pytest.mark.parametrize("shape", [(1, 1, 77, 2, 64), (2, 3, 1025, 1, 32), (1, 40, 77, 2, 128), (1, 130, 65, 1, 64)], ids=str)
def test_an_infinite_value_of_the_last_key_stays_one(shape):
    """Keys past the last one are read from its row: their weight is zero, and zero times infinity is not."""
    B, L, S, N, H = shape
    rng = np.random.default_rng(L)
    q, k, v = (rng.standard_normal((B, T, N, H)).astype(np.float16) for T in (L, S, S))
    v[:, -1, :, 5], v[:, -1, :, 6] = np.inf, -np.inf
    y = R.run_gpu(attention_routine(B, L, S, N, False, H=H), [q, k, v])[0][0]
    assert (y[..., 5] == np.inf).all() and (y[..., 6] == -np.inf).all()
    rest = [i for i in range(H) if i not in (5, 6)]
    assert np.isfinite(y[..., rest]).all()


def _composed(mask, T, N, H, sums="row"):
    """Attention under a mask that the program closes over (`mask` a diagonal) or takes (None), its softmax written out."""
    from jaxjs_hip import jit as J
    from jaxjs_hip import library as L_
    from jaxjs_hip.jit import ShapedArray

    def attend(m, q, k, v):
        s = J.where(m, L_.einsum("BLNH,BSNH->BNLS", q, k).mul(H ** -0.5), -np.inf)
        e = J.exp(s.sub(J.stopGradient(s.max(-1, keepdims=True))))
        total = e.sum(-1).reshape([2, N, T, 1] if sums == "row" else [2, N, 1, T])
        return L_.einsum("BNLS,BSNH->BLNH", e.div(total), v)
    operands = [ShapedArray((2, T, N, H), F16)] * 3
    if mask is None:
        return J.jit(attend, [ShapedArray((T, T), DType.Bool)] + operands)
    return J.jit(lambda q, k, v: attend(L_.tri_const(T, T, mask), q, k, v), operands)


@pytest.mark.parametrize("order", [(0, 1, -1, None), (None, -1, 1, 0)], ids=["causal first", "causal last"])
def test_masks_of_one_shape_do_not_run_as_each_other(order):
    """Programs with the same dispatches on one backend: each under its own mask, whichever was prepared first."""
    if WARM_ONLY:
        pytest.skip("warm-up run")
    from oracle.backend import OracleBackend
    be, (T, N, H) = backend(), (72, 2, 32)
    be._programs.clear()
    rng = np.random.default_rng(6)
    qkv = [rng.standard_normal((2, T, N, H)).astype(np.float16) for _ in range(3)]
    free = (rng.random((T, T)) < 0.5) | np.eye(T, dtype=bool)
    for mask in order:
        prog, arrays = _composed(mask, T, N, H), qkv if mask is not None else [free.astype(np.int32)] + qkv
        got, want = run_program(be, prog, arrays)[0], run_program(OracleBackend(), prog, arrays)[0]
        if mask == -1:  # the first row sees no key: NaN in both
            assert np.isnan(want.reshape(2, T, -1)[:, 0]).all() and np.isnan(got.reshape(2, T, -1)[:, 0]).all()
        np.testing.assert_allclose(got.astype(np.float64), want.astype(np.float64), rtol=1e-2, atol=3e-3, equal_nan=True, err_msg=str(mask))


def test_sums_along_the_columns_are_not_taken_for_a_softmax():
    if WARM_ONLY:
        pytest.skip("warm-up run")
    from oracle.backend import OracleBackend
    T, N, H = 64, 2, 64
    rng = np.random.default_rng(8)
    arrays = [rng.standard_normal((2, T, N, H)).astype(np.float16) for _ in range(3)]
    row, column = _composed(0, T, N, H), _composed(0, T, N, H, "column")
    got = [run_program(backend(), p, arrays)[0].astype(np.float64) for p in (row, column)]
    want = run_program(OracleBackend(), column, arrays)[0].astype(np.float64)
    np.testing.assert_allclose(got[1], want, rtol=1e-2, atol=3e-3 * np.abs(want).max())
    assert np.abs(got[0] - got[1]).max() > 0.1


# Caches extended in the launch that attends to them: heads that write their own part (more than a quarter of the CUs) and copiers beside them, a cache
# of one row, several new rows, new rows in front, key counts around the passes and several rounds, every head size; B, S, new, N, H, in front.
@pytest.mark.parametrize("case", [(1, 1, 1, 1, 64, False), (2, 127, 1, 3, 64, False), (1, 128, 3, 5, 32, True), (3, 700, 1, 2, 128, False), (8, 1024, 1, 12, 64, False), (13, 129, 2, 5, 128, True),
                                  (1, 2600, 1, 2, 64, False), (10, 1400, 1, 7, 32, False)], ids=str)
def test_attention_over_caches_that_the_program_extends(case):
    if WARM_ONLY:
        pytest.skip("warm-up run")
    from jaxjs_hip import jit as J, library as L
    from jaxjs_hip.attentioncache import CachedAttention
    from jaxjs_hip.jit import ShapedArray
    B, S, T, N, H, front = case

    def f(q, keys, values, qkv):
        k, v = (J.shrink(qkv, [(0, B), (0, T), (i * N * H, (i + 1) * N * H)]).reshape([B, T, N, H]) for i in (0, 1))
        keys, values = (L.concatenate([n, o] if front else [o, n], 1) for o, n in ((keys, k), (values, v)))
        return [L.dotProductAttention(q, keys, values), keys, values]
    shapes = [(B, 1, N, H), (B, S, N, H), (B, S, N, H), (B, T, 2 * N * H)]
    prog = J.jit(f, [ShapedArray(s, F16) for s in shapes])
    rng = np.random.default_rng(S)
    q, keys, values, qkv = [rng.standard_normal(s).astype(np.float16) for s in shapes]
    keys[0, 0, 0, :8] = -0.0  # the sum of both padded parts makes these positive
    be = backend()
    assert any(isinstance(u.source, CachedAttention) for u in be.scheduleProgram(prog).units)
    k, v = (qkv[:, :, i * N * H:(i + 1) * N * H].reshape(B, T, N, H) for i in (0, 1))
    k, v = (np.concatenate([n, o] if front else [o, n], 1) + np.float16(0) for o, n in ((keys, k), (values, v)))
    for _ in range(2):
        got = run_program(be, prog, [q, keys, values, qkv])
        np.testing.assert_array_equal(got[1].view(np.uint16), k.reshape(-1).view(np.uint16))
        np.testing.assert_array_equal(got[2].view(np.uint16), v.reshape(-1).view(np.uint16))
        want = R.run_oracle(attention_routine(B, 1, S + T, N, False, H=H), [q, k, v])[0]
        np.testing.assert_allclose(got[0].astype(np.float64).reshape(want.shape), want.astype(np.float64), rtol=2e-3, atol=1e-3)
