"""What the speed of this framework is measured on: whole calls through its public entry points.

Every case is a traced program (`jit.jit` over `library` / `workloads`), prepared once for the backend and then executed
on resident operands (`JitProgram.prepare`, `JitProgram.execute`), which is how a front-end drives the device.  A pass
returns every output of the program as a tensor over the output slot's own memory.  Sizes are those of the
repository's configurations and benches, and ranges around them."""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("jax-js_amd"))

from jaxjs_hip import DType, getBackend, init  # noqa: E402
from jaxjs_hip import jit as J  # noqa: E402
from jaxjs_hip import library as L  # noqa: E402
from jaxjs_hip import workloads as W  # noqa: E402
from jaxjs_hip.convolution import ConvParams  # noqa: E402
from jaxjs_hip.jit import ShapedArray  # noqa: E402

_TYPES = {"f32": (DType.Float32, torch.float32, "<f4", 4), "f16": (DType.Float16, torch.float16, "<f2", 2), "i32": (DType.Int32, torch.int32, "<i4", 4)}
_BY_DTYPE = {d: (t, s, b) for d, t, s, b in _TYPES.values()}


# ---- the cases -------------------------------------------------------------------------------------------------------

def listed():
    return [
        # A small dense classifier on a batch of flattened images: a handful of tiny launches, bound by latency and host work.
        dict(name="mlp_f32_b64", kind="mlp", dtype="f32", batch=64, d_in=784, hidden=256, classes=10),
        # The reference's matmul bench, and this backend's parity configuration: ordinary float32 products.
        dict(name="matmul_f32_1024", kind="matmul", dtype="f32", m=1024, n=1024, k=1024, transposed=False),
        # The headline configuration: the largest dense product, float16 operands with float32 sums.
        dict(name="matmul_f16_8192", kind="matmul", dtype="f16", m=8192, n=8192, k=8192, transposed=False),
        # One token through a linear layer of a language model (weights stored [out, in]): bound by reading the weights.
        dict(name="linear_f16_1x11008x4096", kind="linear", dtype="f16", m=1, n=11008, k=4096, transposed=True),
        # Fused softmax-style row statistics and argmax over wide float32 rows.
        dict(name="rows_f32_8192x4096", kind="rows", op="stats", dtype="f32", rows=8192, cols=4096),
        # Prefill: one pre-LayerNorm transformer block forward over full sequences, as the front-end composes it.
        dict(name="block_f16_b8_l1024", kind="block", batch=8, seq=1024, heads=12, head=64, fused=False),
        # Decode: the same block on one new position per sequence, keys and values appended to a cache.
        dict(name="decode_f16_b8_s1024", kind="decode", batch=8, seq=1024, heads=12, head=64),
        # A training step's share of one convolution layer: forward, and the cotangents of activations and filter.
        dict(name="conv_train_f16_56", kind="conv", dtype="f16", batch=32, cin=64, cout=64, size=56, window=3, stride=1),
        # The reference's sort bench.
        dict(name="sort_f32_32768x1024", kind="sort", op="sort", dtype="f32", rows=32768, cols=1024),
        # The reference's largest FFT bench.
        dict(name="fft_f32_1000000", kind="fft", rows=1, n=1000000, inverse=False),
        # The reference's Cholesky bench at its middle size.
        dict(name="cholesky_f32_1024", kind="linalg", op="cholesky", batch=1, n=1024, rhs=0),
        # The reference's SVD bench: a tall matrix, thin factors.
        dict(name="svd_f32_1024x128", kind="svd", op="svd", m=1024, n=128),
    ]


def _log(rng, low, high):
    """A whole number between the two, spread over the logarithm; odd and ragged values as they come."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _size(rng, low, high):
    """As `_log`; half of the time rounded to a multiple of 64, as layers and batches mostly are."""
    v = _log(rng, low, high)
    return max(low, (v + 32) // 64 * 64) if v >= 64 and rng.random() < 0.5 else v


def draw(rng):
    kind = rng.choice(["mlp", "matmul", "matmul", "linear", "rows", "block", "decode", "conv", "sort", "fft", "linalg", "svd"])
    if kind == "mlp":
        return dict(kind=kind, dtype=rng.choice(["f32", "f16"]), batch=_log(rng, 1, 512), d_in=_size(rng, 16, 1024), hidden=_size(rng, 32, 1024),
                    classes=_log(rng, 2, 1000))
    if kind == "matmul":
        dtype = rng.choice(["f32", "f16"])
        m, n, k = (_size(rng, *((64, 4096) if dtype == "f32" else (256, 8192))) for _ in range(3))
        return dict(kind=kind, dtype=dtype, m=m, n=n, k=k, transposed=rng.random() < 0.5)
    if kind == "linear":
        return dict(kind=kind, dtype="f16", m=_log(rng, 1, 64), n=_size(rng, 512, 16384), k=_size(rng, 512, 8192), transposed=rng.random() < 0.5)
    if kind == "rows":
        dtype = rng.choice(["f32", "f16"])
        cols = _log(rng, 64, 50257)
        return dict(kind=kind, op=rng.choice(["stats", "softmax", "logsoftmax", "standardize"]) if dtype == "f32" else
                    rng.choice(["softmax", "logsoftmax", "standardize"]), dtype=dtype, rows=_log(rng, 16, min(65536, (32 << 20) // cols)), cols=cols)
    if kind == "block":
        return dict(kind=kind, batch=rng.randint(1, 8), seq=_size(rng, 64, 1024), heads=rng.randint(4, 12), head=rng.choice([32, 64]), fused=rng.random() < 0.3)
    if kind == "decode":
        return dict(kind=kind, batch=_log(rng, 1, 16), seq=_log(rng, 64, 1024), heads=rng.randint(4, 12), head=rng.choice([32, 64]))
    if kind == "conv":
        size = _log(rng, 7, 56)
        cin, cout = (_size(rng, 16, 256) for _ in range(2))
        window = rng.choice([1, 3, 3, 5])
        batch = max(1, min(32, _log(rng, 1, 32), (32 * 64 * 56 * 56 * 64 * 9) // (cin * cout * size * size * window * window)))
        return dict(kind=kind, dtype=rng.choice(["f32", "f16"]), batch=batch, cin=cin, cout=cout, size=size, window=window, stride=rng.choice([1, 1, 2]))
    if kind == "sort":
        cols = _log(rng, 16, 65536)
        return dict(kind=kind, op=rng.choice(["sort", "argsort"]), dtype=rng.choice(["f32", "f32", "f16", "i32"]), rows=_log(rng, 1, min(32768, (32 << 20) // cols)), cols=cols)
    if kind == "fft":
        n = 1
        while n < 64:
            n = 1
            target = _log(rng, 64, 1000000)
            while n * 2 <= target:
                step = rng.choice([2, 2, 2, 3, 5, 5, 7])
                if n * step > target:
                    break
                n *= step
        return dict(kind=kind, rows=_log(rng, 1, max(1, min(4096, 1000000 // n))), n=n, inverse=rng.random() < 0.5)
    if kind == "linalg":
        op, n = rng.choice(["cholesky", "solve"]), _log(rng, 16, 1024)
        return dict(kind=kind, op=op, batch=_log(rng, 1, max(1, min(64, (1024 // n) ** 2))), n=n, rhs=_log(rng, 1, 64) if op == "solve" else 0)
    n = _log(rng, 16, 128)
    return dict(kind="svd", op=rng.choice(["svd", "svdvals"]), m=_log(rng, 2 * n, 4096), n=n)


# ---- programs, operands, work ----------------------------------------------------------------------------------------

def _aval(dtype, *shape):
    return ShapedArray(tuple(shape), _TYPES[dtype][0])


def _mlp(x, w1, b1, w2, b2):
    return L.softmax(L.matmul(L.relu(L.matmul(x, w1).add(b1)), w2).add(b2))


def _decode_step(B, N, H):
    """One new position per sequence: keys and values appended to the cache along the position axis, attention over it."""
    D = N * H

    def f(x, keys, values, ln1_g, ln1_b, w_qkv, b_qkv, w_o, b_o, ln2_g, ln2_b, w_fc1, b_fc1, w_fc2, b_fc2):
        h = L.standardize(x).mul(ln1_g).add(ln1_b)
        qkv = L.matmul(h, w_qkv).add(b_qkv)
        q, k, v = (J.shrink(qkv, [(0, B), (0, 1), (i * D, (i + 1) * D)]).reshape([B, 1, N, H]) for i in range(3))
        keys, values = L.concatenate([keys, k], 1), L.concatenate([values, v], 1)
        a = L.dotProductAttention(q, keys, values).reshape([B, 1, D])
        x = x.add(L.matmul(a, w_o).add(b_o))
        h = L.standardize(x).mul(ln2_g).add(ln2_b)
        m = L.gelu(L.matmul(h, w_fc1).add(b_fc1))
        return [x.add(L.matmul(m, w_fc2).add(b_fc2)), keys, values]
    return f


def _conv_step(c):
    pad = c["window"] // 2
    p = ConvParams(0, [c["stride"]] * 2, [(pad, pad)] * 2, [1, 1], [1, 1])
    xs, ws = [c["batch"], c["cin"], c["size"], c["size"]], [c["cout"], c["cin"], c["window"], c["window"]]

    def f(x, w, ct):
        return [J.conv(x, w, p), J.convTransposeLhs(ct, w, xs, p), J.convTransposeRhs(x, ct, ws, p)]
    return f


def _block_operands(c, decode):
    """(name, shape, spread or None for ones / zeros) in the program's order."""
    B, S, D = c["batch"], c["seq"], c["heads"] * c["head"]
    shapes = W.gpt2BlockShapes(B, 1 if decode else S, D, 4 * D)
    ops = [("f16", shapes["x"], 1.0)]
    if decode:
        ops += [("f16", (B, S, c["heads"], c["head"]), 1.0)] * 2
    for name in W.GPT2_BLOCK_PARAMS:
        ops.append(("f16", shapes[name], 0.02 if name.startswith("w") else 0.1))
    return ops


def _operands(c):
    """(type, shape, standard deviation) of every operand."""
    k = c["kind"]
    if k == "mlp":
        d, h, o, t = c["d_in"], c["hidden"], c["classes"], c["dtype"]
        return [(t, (c["batch"], d), 1.0), (t, (d, h), d ** -0.5), (t, (h,), 0.1), (t, (h, o), h ** -0.5), (t, (o,), 0.1)]
    if k in ("matmul", "linear"):
        b = (c["n"], c["k"]) if c["transposed"] else (c["k"], c["n"])
        return [(c["dtype"], (c["m"], c["k"]), 1.0), (c["dtype"], b, c["k"] ** -0.5)]
    if k == "rows":
        return [(c["dtype"], (c["rows"], c["cols"]), 1.0)]
    if k in ("block", "decode"):
        return _block_operands(c, k == "decode")
    if k == "conv":
        out = _conv_out(c)
        return [(c["dtype"], (c["batch"], c["cin"], c["size"], c["size"]), 1.0), (c["dtype"], (c["cout"], c["cin"], c["window"], c["window"]), 0.05),
                (c["dtype"], (c["batch"], c["cout"], out, out), 1.0)]
    if k == "sort":
        return [(c["dtype"], (c["rows"], c["cols"]), 1.0)]
    if k == "fft":
        return [("f32", (c["rows"], c["n"]), 1.0)] * 2
    if k == "linalg":
        lead = (c["batch"],) if c["batch"] > 1 else ()
        return [("f32", lead + (c["n"], c["n"]), 1.0)] + ([("f32", lead + (c["n"], c["rhs"]), 1.0)] if c["op"] == "solve" else [])
    return [("f32", (c["m"], c["n"]), 1.0)]


def _conv_out(c):
    return (c["size"] + 2 * (c["window"] // 2) - c["window"]) // c["stride"] + 1


def _program(c):
    k, avals = c["kind"], [_aval(t, *s) for t, s, _ in _operands(c)]
    if k == "mlp":
        return J.jit(_mlp, avals)
    if k in ("matmul", "linear"):
        t = c["transposed"]
        return J.jit(lambda a, b: L.matmul(a, L.swapaxes(b, 0, 1) if t else b), avals)
    if k == "rows":
        if c["op"] == "stats":
            return W.rowSoftmaxArgmaxProgram(c["rows"], c["cols"])
        op = {"softmax": L.softmax, "logsoftmax": L.logSoftmax, "standardize": L.standardize}[c["op"]]
        return J.jit(lambda x: op(x, -1), avals)
    if k == "block":
        D = c["heads"] * c["head"]
        return W.gpt2BlockProgram(c["batch"], c["seq"], D, c["heads"], 4 * D, fusedAttention=c["fused"])
    if k == "decode":
        return J.jit(_decode_step(c["batch"], c["heads"], c["head"]), avals)
    if k == "conv":
        return J.jit(_conv_step(c), avals)
    if k == "sort":
        return J.jit(lambda x: L.sort(x) if c["op"] == "sort" else L.argsort(x), avals)
    if k == "fft":
        return J.jit(lambda re, im: list(L.fft(re, im, -1, c["inverse"])), avals)
    if k == "linalg":
        return J.jit(L.solve if c["op"] == "solve" else L.cholesky, avals)
    return J.jit(lambda a: list(L.svd(a)) if c["op"] == "svd" else L.svdvals(a), avals)


def _values(c, i, gen):
    """Operand `i` as a host array, from the generator alone."""
    t, shape, spread = _operands(c)[i]
    dtype = _TYPES[t][1]
    if dtype is torch.int32:
        return torch.randint(-(1 << 30), 1 << 30, shape, generator=gen, device="cuda", dtype=dtype).cpu().numpy()
    x = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * spread
    if c["kind"] == "linalg" and i == 0:  # well-conditioned systems: a positive definite matrix, a dominant diagonal
        eye = torch.eye(c["n"], device="cuda")
        if c["op"] == "cholesky":
            x = torch.matmul(x, x.transpose(-1, -2).contiguous()) / c["n"] + eye
        else:
            x = x + 2.0 * c["n"] ** 0.5 * eye
    if c["kind"] in ("block", "decode") and (i - (2 if c["kind"] == "decode" else 0)) in (1, 7):  # LayerNorm gains
        x = x + 1.0
    return x.to(dtype).cpu().numpy()


def _result_types(c):
    """(type, shape) of every output, in the program's order."""
    k = c["kind"]
    if k == "mlp":
        return [(c["dtype"], (c["batch"], c["classes"]))]
    if k in ("matmul", "linear"):
        return [(c["dtype"], (c["m"], c["n"]))]
    if k == "rows":
        return [("f32", (c["rows"],)), ("i32", (c["rows"],))] if c["op"] == "stats" else [(c["dtype"], (c["rows"], c["cols"]))]
    if k == "block":
        return [("f16", (c["batch"], c["seq"], c["heads"] * c["head"]))]
    if k == "decode":
        return [("f16", (c["batch"], 1, c["heads"] * c["head"]))] + [("f16", (c["batch"], c["seq"] + 1, c["heads"], c["head"]))] * 2
    if k == "conv":
        out = _conv_out(c)
        return [(c["dtype"], (c["batch"], c["cout"], out, out)), (c["dtype"], (c["batch"], c["cin"], c["size"], c["size"])),
                (c["dtype"], (c["cout"], c["cin"], c["window"], c["window"]))]
    if k == "sort":
        return [("i32" if c["op"] == "argsort" else c["dtype"], (c["rows"], c["cols"]))]
    if k == "fft":
        return [("f32", (c["rows"], c["n"]))] * 2
    if k == "linalg":
        lead = (c["batch"],) if c["batch"] > 1 else ()
        return [("f32", lead + ((c["n"], c["rhs"]) if c["op"] == "solve" else (c["n"], c["n"])))]
    s = [("f32", (c["n"],))]
    return s if c["op"] == "svdvals" else [("f32", (c["m"], c["n"]))] + s + [("f32", (c["n"], c["n"]))]


class _Owner:
    """Holds a program's slots and gives them back when the last tensor over them is gone."""

    def __init__(self, be, slots):
        self.be, self.slots = be, list(slots)

    def swap(self, slots):
        old, self.slots = self.slots, slots
        for s in old:
            self.be.decRef(s)

    def __del__(self):
        self.swap([])


class _Memory:
    """A slot's device memory, as torch takes it in."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr=typestr, data=(ptr, False), version=2)


class _State:
    pass


def prepare(case, seed):
    init("hip")
    be = getBackend("hip")
    s = _State()
    s.be, s.prog = be, _program(case)
    s.prepared = s.prog.prepare(be)
    slots = []
    for const in s.prog.consts:  # closed-over constants come first
        kernel = const.kernel()
        slots.append(be.malloc(kernel.bytes))
        be.dispatch(be.prepareKernelSync(kernel), [], [slots[-1]])
    gen = torch.Generator(device="cuda")
    for i in range(len(_operands(case))):
        gen.manual_seed(seed * 64 + i)
        x = _values(case, i, gen)
        slots.append(be.malloc(x.nbytes, x))
    s.inputs, s.outputs, s.views = _Owner(be, slots), _Owner(be, []), {}
    s.results = [(shape, _TYPES[t][2]) for t, shape in _result_types(case)]
    return s


def run(state):
    be = state.be
    outs = state.prog.execute(be, state.inputs.slots, state.prepared)
    state.outputs.swap(outs)
    got = []
    for i, slot in enumerate(outs):
        key = (i, be.slotPointer(slot))
        view = state.views.get(key)
        if view is None:  # the pool hands the same few buffers out again: their tensors are kept
            view = state.views[key] = torch.as_tensor(_Memory(state.outputs, key[1], *state.results[i]), device="cuda")
        got.append(view)
    return got


def _count(t, shape):
    return math.prod(shape) * _TYPES[t][3]


def work(case):
    c, k = case, case["kind"]
    moved = sum(_count(t, s) for t, s, _ in _operands(c)) + sum(_count(t, s) for t, s in _result_types(c))
    if k == "mlp":
        flops = 2 * c["batch"] * c["hidden"] * (c["d_in"] + c["classes"])
    elif k in ("matmul", "linear"):
        flops = 2 * c["m"] * c["n"] * c["k"]
    elif k == "rows":
        flops = 8 * c["rows"] * c["cols"]
    elif k in ("block", "decode"):
        B, S, D = c["batch"], c["seq"], c["heads"] * c["head"]
        rows = B * (1 if k == "decode" else S)
        # four projections and the MLP (12 D^2 weights); scores and values, the visible half of a causal matrix
        flops = 2 * rows * 12 * D * D + (4 * B * (S + 1) * D if k == "decode" else 2 * B * S * (S + 1) * D)
    elif k == "conv":
        flops = 3 * 2 * c["batch"] * c["cin"] * c["cout"] * (c["window"] * _conv_out(c)) ** 2
    elif k == "sort":
        flops = c["rows"] * c["cols"] * max(1, c["cols"].bit_length())
    elif k == "fft":
        flops = 5 * c["rows"] * c["n"] * math.log2(c["n"])
    elif k == "linalg":
        flops = c["batch"] * (c["n"] ** 3 / 3 if c["op"] == "cholesky" else 2 * c["n"] ** 3 / 3 + 2 * c["n"] ** 2 * c["rhs"])
    else:  # the Gram product, its eigendecomposition (about 9 n^3), and the other factor
        flops = 2 * c["m"] * c["n"] ** 2 * (2 if c["op"] == "svd" else 1) + 9 * c["n"] ** 3
    return {"bytes": float(moved), "flops": float(flops)}


def tolerance(case):
    k = case["kind"]
    if k == "sort":
        return "exact"
    if k in ("block", "decode"):  # a chain of float16 roundings
        return {"rel": 5e-3}
    if case.get("dtype") == "f16":
        return {"rel": 2e-3}
    if k == "linalg" and case["op"] == "solve":  # an elimination in float32 before the two substitutions
        return {"rel": 1e-4}
    if k == "svd":  # vectors of a float32 Gram matrix, whose closest eigenvalues are a small part of the largest apart
        return {"rel": 2e-3 if case["op"] == "svd" else 2e-5}
    return {"rel": 1e-5}
