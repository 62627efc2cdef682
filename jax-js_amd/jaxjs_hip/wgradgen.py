"""The filter cotangent of a stride-1 convolution with its image and cotangent bands resident in LDS (`wgrad_f16.hip.inc`).

The transpose rule of a convolution binds another convolution for the filter's cotangent, batch and channels exchanged
(src/frontend/linearize.ts:813-837).  It reaches a backend as one reduce Kernel over batch x positions whose image operand is
read through padded and windowed views, once per tap.  `match_wgrad` takes both operands' lowered index expressions, proposes
the geometry of a window walk from a few probes, and evaluates the expressions against that model: every (tap, position) of the
first, the second and the last image with its padding mask, and the corners of all others.  Channels have to enter by a
constant stride.  Only an exact match takes the kernel, and only as part of a program (`schedule.py`): a Kernel that is prepared
by itself keeps the general templates."""

from __future__ import annotations

from typing import Optional

import numpy as np

from . import tuner
from .alu import AluExp, AluOp, DType
from .convgen import np_eval

WGRAD_TAPS = 9             # of a workgroup: sixteen registers each, and four waves' sums of them in LDS
WGRAD_LDS = 80 * 1024      # a band of the image and of the cotangent, of which two are held
WGRAD_PARTIALS = 64 << 20  # bytes of the slices' sums
WGRAD_WORK = 1 << 24       # products from which the kernel is taken
WGRAD_FOLD = 9000          # cycles of the fold's launch and of writing the slices' sums ([3,256,14,14] 128 11.7 -> 8.0 us in one launch,
                           # [3,130,17,17] 250, whose bands take 4500, 13.0 and 14.2)
WGRAD_TABLE = 1 << 22      # entries of the index tables that a match may evaluate


def operand_exps(kernel, t, g: dict) -> Optional[dict]:
    """Both operands in (row, k, b0..) coordinates, by tag."""
    from .gemm import _strip_casts

    lowered = _strip_casts(t.exp)
    if lowered.op != AluOp.Mul:
        return None
    sides = {}
    for side in lowered.src:
        gids = {n.arg[0] for n in side.collect(lambda x: x.op == AluOp.GlobalIndex)}
        if len(gids) != 1:
            return None
        sides[gids.pop()] = _strip_casts(side)
    if len(sides) != 2 or {g["gid_a"], g["gid_b"]} != set(sides):
        return None
    out = {}
    for tag, gid, extent, stride in (("a", g["gid_a"], g["M"], g["c_sm"]), ("b", g["gid_b"], g["N"], g["c_sn"])):
        flat = AluExp.mul(AluExp.special(DType.Int32, "row", max(extent, 1)), AluExp.i32(stride))
        for k, (size, _sa, _sb, sc) in enumerate(g["batch"]):
            flat = AluExp.add(AluExp.mul(AluExp.special(DType.Int32, f"b{k}", size), AluExp.i32(sc)), flat)
        kvar = AluExp.special(DType.Int32, "k", max(g["K"], 1))

        def put(node, flat=flat, kvar=kvar):
            if node.op == AluOp.Special and node.arg[0] == "gidx":
                return flat
            if node.op == AluOp.Special and node.arg[0] == "ridx":
                return kvar
            return None
        out[tag] = sides[gid].rewrite(put).reduceExactIndex().simplify()
    return out


def _load(e: AluExp):
    """(mask or None, GlobalIndex node, channel stride, index at channel 0) of a float16 load, or None."""
    from .gemm import _affine_in, _has_special

    cond, node = None, e
    if node.op == AluOp.Where:
        if node.src[2].op != AluOp.Const or float(node.src[2].arg) != 0.0:
            return None
        cond, node = node.src[0], node.src[1]
    if node.op != AluOp.GlobalIndex or node.dtype != DType.Float16 or (cond is not None and _has_special(cond, "row")):
        return None
    a = _affine_in(node.src[0], "row")
    return None if a is None or a[0] <= 0 else (cond, node, a[0], a[1])


def _table(cond, idx, k, tap):
    env = {"row": np.int64(0), "k": k, "b0": tap, "b1": np.int64(0), "b2": np.int64(0)}
    shape = np.broadcast_shapes(np.shape(k), np.shape(tap))
    try:
        i = np.broadcast_to(np_eval(idx, env), shape)
        ok = np.ones(shape, bool) if cond is None else np.broadcast_to(np_eval(cond, env), shape)
    except (NotImplementedError, KeyError):
        return None
    return i, ok


def match_wgrad(g: dict, exps: dict) -> Optional[dict]:
    """Geometry of the window walk and the operands' tags, or None.  The taps are the batch axis, or (`joined`) the image
    operand's rows are channel * taps + tap."""
    if g["dtype"] != DType.Float16 or len(g["batch"]) > 1:
        return None
    for img, ct in (("a", "b"), ("b", "a")):
        if not g.get(img + "_gather"):
            continue
        C, O = (g["M"], g["N"]) if img == "a" else (g["N"], g["M"])
        forms = [(g["batch"][0][0], C, exps[img], False)] if g["batch"] else _split_rows(exps[img], C)
        for T, channels, image, joined in forms:
            found = _match(T, g["K"], image, exps[ct], channels, O) if T > 1 else None
            if found is not None:
                return dict(found, img=img, ct=ct, joined=joined)
    return None


def _split_rows(image: AluExp, rows: int):
    """Ways to read the image operand's rows as channel * T + tap: (T, channels, the operand with `row` the channel and `b0` the
    tap, True)."""
    divisors = {int(x.src[1].arg) for x in image.collect(lambda x: x.op == AluOp.Idiv and x.src[1].op == AluOp.Const)}
    for T in sorted(divisors, reverse=True):
        if 1 < T < rows and rows % T == 0:
            row = AluExp.add(AluExp.mul(AluExp.special(DType.Int32, "row", rows // T), AluExp.i32(T)), AluExp.special(DType.Int32, "b0", T))
            yield T, rows // T, image.rewrite(lambda n, row=row: row if n.op == AluOp.Special and n.arg[0] == "row" else None).reduceExactIndex().simplify(), True


def _match(T: int, K: int, image: AluExp, cotangent: AluExp, C: int, O: int) -> Optional[dict]:
    im, co = _load(image), _load(cotangent)
    if im is None or co is None or co[0] is not None:
        return None
    # The cotangent: the same for every tap, whole images of consecutive elements.  Where an image ends shows in the first
    # step that is not one.
    head = np.arange(min(K, WGRAD_TABLE // T), dtype=np.int64)
    taps = np.arange(T, dtype=np.int64)[:, None]
    first = _table(None, co[3], head, np.int64(0))
    if first is None:
        return None
    step = np.nonzero(np.diff(first[0]) != 1)[0]
    P = int(step[0]) + 1 if len(step) else len(head)
    if K % P or P < 64 or (not len(step) and P != K):
        return None
    NB, pos = K // P, head[:P]
    ct0 = int(first[0][0])
    # every position of the first, second and last image, and the first and last position of every image
    some = sorted({0, 1, NB - 1} & set(range(NB)))
    starts = np.arange(NB, dtype=np.int64)[:, None] * P
    ks = np.concatenate([(np.array(some)[:, None] * P + pos[None, :]).reshape(-1), (starts + np.array([0, P - 1])[None, :]).reshape(-1)])
    cot = [_table(None, co[3], ks, np.int64(tap)) for tap in (0, T - 1)]
    if any(c is None for c in cot):
        return None
    ctb = int(cot[0][0][P]) - ct0 if NB > 1 else 0
    if ctb < 0 or ct0 < 0 or any(not np.array_equal(c[0], ct0 + (ks // P) * ctb + ks % P) for c in cot):
        return None
    # the image: one whole image, every tap
    table = _table(im[0], im[3], pos[None, :], taps)
    if table is None:
        return None
    idx, ok = table
    d_tap = np.nonzero(np.diff(idx[:, 0]) != 1)[0]
    KW = int(d_tap[0]) + 1 if len(d_tap) else T
    if KW == T or T % KW:  # (windows of one row stay on the general template)
        return None
    KH = T // KW
    W = int(idx[KW, 0] - idx[0, 0])
    SC = im[2]
    breaks = np.nonzero(np.diff(idx[0, :]) != 1)[0]
    OW = int(breaks[0]) + 1 if len(breaks) else W
    if W < 8 or OW < 8 or SC % W or P % OW:
        return None
    H, OH = SC // W, P // OW
    # An image may start anywhere in its buffer, so the padding is read off the mask: the first position's valid taps.
    ky, kx = taps // KW, taps % KW
    y, x = np.arange(P)[None, :] // OW, np.arange(P)[None, :] % OW
    valid_at_0 = np.nonzero(ok[:, 0])[0]
    if not len(valid_at_0):
        return None
    PH, PW = int(valid_at_0[0]) // KW, int(valid_at_0[0]) % KW
    base = int(idx[0, 0]) + PH * W + PW
    iy, ix = y + ky - PH, x + kx - PW
    valid = (iy >= 0) & (iy < H) & (ix >= 0) & (ix < W)
    if base < 0 or not np.array_equal(ok, valid) or not np.array_equal(idx[valid], (base + iy * W + ix)[valid]):
        return None
    whole = _table(im[0], im[3], ks[None, :], taps)
    if whole is None or not np.array_equal(whole[1], ok[:, ks % P]):
        return None
    keep, delta = whole[1], whole[0] - idx[:, ks % P]
    second = keep & (ks // P == 1)[None, :]
    SB = int(delta[second][0]) if second.any() else 0
    if SB < 0 or not np.array_equal(delta[keep], np.broadcast_to((ks // P) * SB, delta.shape)[keep]):
        return None
    if base + (NB - 1) * SB + (C - 1) * SC + H * W > im[1].arg[1] or ct0 + (NB - 1) * ctb + (O - 1) * co[2] + P > co[1].arg[1]:
        return None
    return dict(C=C, O=O, T=T, KH=KH, KW=KW, W=W, H=H, OW=OW, OH=OH, PH=PH, PW=PW, SC=SC, SB=SB, IMG_OFF=base, CTO=co[2], CTB=ctb,
                CT_OFF=ct0, NB=NB)


def _odd(n: int) -> int:
    """n elements (whole groups of eight) rounded up to an odd number of 16 bytes."""
    return n if n % 16 == 8 else n + 8


def plan_wgrad(m: dict) -> Optional[dict]:
    """Band, window rows of a workgroup and slices, or None where a band does not fit."""
    KY = max((d for d in range(1, m["KH"] + 1) if m["KH"] % d == 0 and d * m["KW"] <= WGRAD_TAPS), default=0)
    if KY == 0 or m["PW"] > 4 or m["KW"] - 1 - m["PW"] > 4 or m["PW"] < 0 or m["KW"] - 1 - m["PW"] < 0:
        return None
    XC = -(-m["OW"] // 8)
    IC = max(-(-m["W"] // 8), XC)
    best = None
    for R in range(1, min(m["OH"], 32) + 1):
        PI, PC = _odd((R + KY - 1) * 8 * IC), _odd(R * 8 * XC)
        if 2 * (8 + 32 * PI + (KY - 1) * 8 * IC + 32 + 32 * PC + 8 + 7) > WGRAD_LDS:
            break
        bands = -(-m["OH"] // R)
        steps = -(-(-(-R * XC // 2)) // 4)  # of a wave
        # a step: matrix instructions, and what goes around them; a band: its way into LDS, its first reads and its barrier
        cycles = steps * (40 * KY * m["KW"] + 80) + 2 * 32 * (R + KY - 1 + R) * XC / 16 + 500
        if best is None or bands * cycles < best["cost"]:
            best = dict(cost=bands * cycles, cycles=cycles, R=R, PI=PI, PC=PC)
    if best is None:
        return None
    if m["C"] * m["SC"] >= 1 << 31 or m["O"] * m["CTO"] >= 1 << 31:  # offsets inside an image are 32 bits
        return None
    groups = m["KH"] // KY
    tiles = -(-m["C"] // 32) * -(-m["O"] // 32) * groups
    bands = m["NB"] * -(-m["OH"] // best["R"])
    slices = max(1, min(bands, tuner.CU_COUNT // tiles, WGRAD_PARTIALS // (tiles * KY * m["KW"] * 4096)))
    if (bands - 1) * best["cycles"] <= WGRAD_FOLD:  # sooner done one after the other than folded by a launch of its own
        slices = 1
    slices = -(-bands // -(-bands // slices))  # no more than it takes: the longest slice is what the launch waits for
    return dict(best, KY=KY, GROUPS=groups, IC=IC, slices=slices, tiles=tiles, bands=bands)


def find_wgrad(kernel, t, g: dict) -> Optional[dict]:
    """Geometry and plan of a filter cotangent that the kernel covers and is worth its two launches for, or None.

    Float16 microseconds, before -> here ([batch, channels, size, size], output channels, window): [32,64,56,56] 64 3x3 48.9 -> 25,
    [8,256,14,14] 256 91.6 -> 15, [16,128,28,28] 128 34 -> 18, [3,32,28,28] 64 5x5 22.6 -> 10.5.  Odd sizes and few channels, which
    went element by element: [6,72,40,40] 72 439 -> 15, [2,64,57,57] 64 197 -> 11.5, [32,16,56,56] 16 1937 -> 29.  Below the line the
    differences are within a microsecond of a launch ([8,24,9,9] 40 8.9 and 10.9, [1,64,12,12] 64 9.9 and 7.3)."""
    if g["dtype"] != DType.Float16 or len(g["batch"]) > 1 or not (g.get("a_gather") or g.get("b_gather")):
        return None
    if g["M"] * g["N"] * (g["batch"][0][0] if g["batch"] else 1) * g["K"] < WGRAD_WORK:
        return None
    exps = operand_exps(kernel, t, g)
    m = match_wgrad(g, exps) if exps is not None else None
    p = plan_wgrad(m) if m is not None else None
    return None if p is None else dict(m, **p)


def _fold_waves(slices: int) -> int:
    """Waves of the fold that share the slices of 64 pieces: about four loads each, all in flight at once (56 slices of [64, 64, 3,
    3]: 6.1 -> 4.6 us with 14 waves instead of four)."""
    return max(4, min(16, slices // 4))


def is_filter_cotangent(kernel) -> bool:
    """Whether `kernel` is better prepared with the option `filter_bands`.  (Why it is an option, which programs' schedules set,
    and not the plan of every such Kernel: the plan without it, slices of k read element by element, 45 + 5 us where this
    kernel takes 15 + 5 for 32 x [64, 56, 56], is pinned by tests/test_transform_kernels.py.)"""
    if kernel.reduction is None or kernel.size == 0:
        return False
    g = tuner.match_gemm(kernel)
    return g is not None and find_wgrad(kernel, tuner.tuneNullopt(kernel), g) is not None


def gen_wgrad(kernel, g: dict, w: dict, numerics: str, name: str, params: str, names: list, out_t: str, epi_fn: str, epi_params: str, epi_args: str,
              need: dict, src_options: str):
    """KernelSource of the plan `w` (see `find_wgrad`): one launch, and the fold of its slices where there are several."""
    from .kernelgen import KernelSource, LaunchStep, _prelude, fill, template

    aligned = all(v % 8 == 0 for v in (w["W"], w["OW"], w["SC"], w["SB"], w["CTO"], w["CTB"], w["IMG_OFF"], w["CT_OFF"]))
    image_rows = w["img"] == "a"
    c_row = f"c * {w['T']} + tap" if w["joined"] else "c"
    src = src_options + _prelude(numerics) + fill(template("wgrad_f16.hip.inc"), dict(
        {k: w[k] for k in ("C", "O", "W", "H", "OW", "OH", "KW", "KY", "GROUPS", "PH", "PW", "SC", "SB", "CTO", "CTB", "R", "NB", "IC", "PI", "PC", "IMG_OFF", "CT_OFF")},
        SLICES=w["slices"], PARTS=_fold_waves(w["slices"]), ALIGN=16 if aligned else 2, EPILOGUE_FN=epi_fn, NAME=name, PARAMS=params, IMG_PTR=names[g["gid_" + w["img"]]],
        CT_PTR=names[g["gid_" + w["ct"]]], ROW=c_row if image_rows else "o", COL="o" if image_rows else c_row,
        C_SM=g["c_sm"], C_SN=g["c_sn"], C_ST=0 if w["joined"] else g["batch"][0][3], B0="0" if w["joined"] else "tap", OUT_T=out_t, EPILOGUE_PARAMS=epi_params, EPILOGUE_ARGS=epi_args))
    args = [("in", i) for i in range(kernel.nargs)] + [("out", 0)]
    pieces, scratch = w["tiles"] * w["KY"] * w["KW"] * 256, []
    steps = [LaunchStep(name, (w["tiles"] * w["slices"], 1, 1), (256, 1, 1), 0, args)]
    if w["slices"] > 1:
        scratch = [w["slices"] * pieces * 16]
        steps = [LaunchStep(name, (w["tiles"] * w["slices"], 1, 1), (256, 1, 1), 0, args + [("scratch", 0)]),
                 LaunchStep(name + "_fold", (pieces // 64, 1, 1), (64 * _fold_waves(w["slices"]), 1, 1), 0, args + [("scratch", 0)])]
    need = dict(need)
    for tag, end in ((w["img"], w["IMG_OFF"] + (w["NB"] - 1) * w["SB"] + (w["C"] - 1) * w["SC"] + w["H"] * w["W"]),
                     (w["ct"], w["CT_OFF"] + (w["NB"] - 1) * w["CTB"] + (w["O"] - 1) * w["CTO"] + w["OH"] * w["OW"])):
        gid = g["gid_" + tag]
        need[gid] = max(need.get(gid, 0), end * 2)
    info = dict(M=g["M"], N=g["N"], K=g["K"], nbatch=w["T"], tiles=w["tiles"], splitk=w["slices"], direct_lds=False,
                wgrad=dict(KY=w["KY"], R=w["R"], bands=w["bands"], aligned=aligned), gather=dict(image="band"))
    return KernelSource([src], steps, scratch, "gemm+fold" if w["slices"] > 1 else "gemm", need, info)
