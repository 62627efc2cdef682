"""Plan and source of a GEMM too small for LDS tiles to fill the chip (`gemm_few.hip.inc`)."""

from __future__ import annotations

from typing import Optional

from . import tuner
from .alu import DType
from .kernelgen import fill, template

FEW_LDS = 128 * 1024  # float32 sums of all waves
FEW_ROWS = 64         # short operands up to this many rows are what the kernel is made for
FEW_DEEP = 4096       # longest k axis for more rows, or across 16-byte lines: each wave of a tile would walk too many steps
FEW_WORKGROUPS = 64   # tile plans with as many workgroups stand against more rows (see `_tiles_stand`)


def _loads(g: dict, tag: str, along_k: bool) -> float:
    """Cost of a load of 16 bytes a lane against one from even addresses: float16 rows at odd elements straddle."""
    srow, other = (g["a_sm"], g["a_sk"]) if tag == "a" else (g["b_sn"], g["b_sk"])
    if g["dtype"] == DType.Float32 or (srow if along_k else other) % 2 == 0:
        return 1.0
    return 3.0 if along_k else 1.5


def _operands(g: dict) -> Optional[dict]:
    """The short operand, which has to run along k, the wide one, along k or along its rows, and their extents; None where
    the kernel does not apply."""
    if g["dtype"] not in (DType.Float16, DType.Float32) or g.get("a_gather") or g.get("b_gather") or g["a_k0"] != g["K"] or g["b_k0"] != g["K"] or g["K"] < 32:
        return None
    nb = 1
    for b in g["batch"]:
        nb *= b[0]
    if nb > 65535:
        return None
    row, rows = {"a": "a_sm", "b": "b_sn"}, {"a": g["M"], "b": g["N"]}
    short = "a" if g["M"] <= g["N"] else "b"
    if g[short + "_sk"] != 1:
        short = "b" if short == "a" else "a"
    wide = "b" if short == "a" else "a"
    if g[short + "_sk"] != 1:
        return None
    along_k = g[wide + "_sk"] == 1
    if not along_k and not (g[row[wide]] == 1 and g[wide + "_sk"] > 0):
        return None
    loose = bool(g.get("a_loose") or g.get("b_loose"))
    R, C, K = rows[short], rows[wide], g["K"]
    if K > FEW_DEEP and (R > FEW_ROWS or along_k and loose):
        return None
    eb = 4 if g["dtype"] == DType.Float32 else 2
    return dict(R=R, C=C, K=K, short=short, wide=wide, along_k=along_k, loose=loose, nbatch=nb, row=row, eb=eb, w_bytes=C * K * eb * nb)


def _shape(g: dict, o: dict) -> Optional[dict]:
    """The workgroup's tile (MT 16-row and VN 16-column pieces), its waves, and the launch's estimated microseconds: 2.6
    to start; per step of a workgroup 28 cycles for each 16-row piece of an operand and the matrix instructions of four
    SIMDs; 16 cycles per wave and 16 x 16 tile for the sums; and the wide operand again from beyond the L2 for every row
    tile when it is more than 4 MB."""
    f32, along_k, R, C = o["eb"] == 4, o["along_k"], o["R"], o["C"]
    step = 64 // o["eb"]
    steps = -(-o["K"] // step)
    wx, ww = _loads(g, o["short"], True), _loads(g, o["wide"], along_k)
    best = None
    for MT in (1, 2, 4):
        if MT > 1 and 8 * MT >= R:
            break
        for VN in ((1, 2, 4) if f32 or along_k else (2, 4, 8)):
            if MT * VN > 16 or (not along_k and C < VN) or (VN > 1 and 8 * VN >= C and VN != 2):
                continue
            waves = max(1, min(16, o["K"] // step or 1, FEW_LDS // (MT * 16 * (16 * VN + 1) * 4)))
            row_tiles = -(-R // (16 * MT))
            count = row_tiles * -(-C // (16 * VN)) * o["nbatch"]
            cycles = steps * (28 * (MT * wx + VN * ww) + MT * VN * (32 if f32 else 4)) + waves * MT * VN * 16
            work = max(1.0, count / tuner.CU_COUNT) * cycles / 2400
            again = row_tiles * o["w_bytes"] / 10e6 if o["w_bytes"] > 4 << 20 else 0.0
            if row_tiles <= 65535 and (best is None or 2.6 + work + again < best["us"]):
                best = dict(us=2.6 + work + again, work=work, count=count, MT=MT, VN=VN, waves=waves)
    return best


def _slices(steps: int, count: int) -> int:
    """Workgroups that share the k steps of each of `count` tiles (folded inside the launch by the last of them).

    A long k axis in a few workgroups is bound by what one CU can have in flight and by its matrix instructions, and the fold
    costs about 1.3 us, so the axis is cut where a slice keeps 24 steps of 64 bytes (64 in two slices, 32 in eight) and every
    slice's workgroup still has a CU to itself.  microseconds with the weights in the L2 / from beyond it: float16 8 x 768 x
    3072 4.8 / 7.5 whole, 4.4 / 5.1 in four slices, 24 x 512 x 4096 7.1 / 10.7 and 5.1 / 6.2; float32 8 x 512 x 2048 7.1 / 8.3
    and 4.6 / 5.1, 64 x 128 x 4096 14.8 / 15.1 and in eight 5.9 / 5.8, 64 x 512 x 4096 (128 tiles) 15.4 / 15.9 and in two
    10.3 / 10.8.  Shorter axes lose from the L2 what they win from memory (float16 2 x 1024 x 2048 3.3 / 6.0 and 4.1 / 5.1)."""
    for slices, least in ((8, 256), (4, 96), (2, 128)):
        if steps >= least and count * slices <= tuner.CU_COUNT:
            return slices
    return 1


def _tile_launch(g: dict, o: dict, tile: dict) -> dict:
    """The tile plan's workgroups, whether it is on the direct-to-LDS path, and its estimated microseconds: 2.5 to start
    (2.8 where whole 16-byte groups are staged through registers), 2 for folding a k split, and a time
    per element of k that depends on the loader."""
    BM, BN, split = tile["BM"], tile["BN"], tile.get("SPLITK", 1)
    count = -(-g["M"] // BM) * -(-g["N"] // BN) * o["nbatch"] * split
    direct = o["eb"] == 2 and BM >= 128 and BN >= 128 and o["K"] % 32 == 0 and not o["loose"]
    start = 2.5 if direct or o["loose"] else 2.8
    if o["eb"] == 4:
        per_k = (0.026 if o["loose"] else 0.024) * BM * BN / 4096
    elif direct:
        per_k = 0.0045 * BM * BN / 16384
    elif o["along_k"]:
        per_k = 0.008 if o["loose"] else 0.0066
    else:
        per_k = 0.025 if g.get(o["wide"] + "_loose") else 0.012
    us = start + (2.0 if split > 1 else 0.0) + max(1.0, count / tuner.CU_COUNT) * o["K"] / split * per_k
    return dict(count=count, direct=direct, us=us)


def _tiles_stand(o: dict, t: dict) -> bool:
    """Tile plans that no estimate is asked about: with enough workgroups to hide their loads behind each other, against
    more rows than a few (64; twice as many for float32 with a k axis of under 256, one per CU for float16 off the
    16-byte grid, any on the direct-to-LDS path), or against weights that stream from memory anyway."""
    if o["eb"] == 4:
        many = 2 * FEW_WORKGROUPS if o["loose"] or o["K"] < 256 else FEW_WORKGROUPS
    else:
        many = 0 if t["direct"] else tuner.CU_COUNT if o["loose"] else FEW_WORKGROUPS
    return t["count"] >= many and o["R"] > FEW_ROWS or t["count"] >= FEW_WORKGROUPS and o["w_bytes"] > 96 << 20 and not o["loose"]


def _in_steps(best: dict, o: dict, slices: int) -> dict:
    """The plan of a shape: steps in equal shares for the waves, in equal batches of what the registers of a full workgroup hold
    in flight."""
    MT, VN, steps = best["MT"], best["VN"], max(1, o["K"] // (64 // o["eb"]))
    waves = min(best["waves"], -(-steps // slices))
    share = -(-steps // (waves * slices))
    most = max(1, (104 - 4 * MT * VN) // (4 * (MT + VN)))
    return dict(R=o["R"], MT=MT, C=o["C"], short=o["short"], wide=o["wide"], along_k=o["along_k"], VN=VN, waves=-(-steps // (share * slices)), slices=slices,
                batch=-(-share // -(-share // most)), nbatch=o["nbatch"], row=o["row"])


def plan_whole_rows(g: dict) -> Optional[dict]:
    """The plan of `g` in tiles that hold whole rows of the result, or None; with the launch's estimated microseconds."""
    o = _operands(g)
    if o is None or g["batch"]:
        return None
    f32, step = o["eb"] == 4, 64 // o["eb"]
    best = None
    for MT in (1, 2, 4):
        for VN in ((1, 2, 4) if f32 or o["along_k"] else (2, 4, 8)):
            across, down = (16 * VN, 16 * MT) if o["short"] == "a" else (16 * MT, 16 * VN)
            if MT * VN > 16 or across < g["N"] or (not o["along_k"] and o["C"] < VN) or -(-o["R"] // (16 * MT)) > 65535:  # (gridDim.z)
                continue
            waves = max(1, min(16, o["K"] // step or 1, FEW_LDS // (MT * 16 * (16 * VN + 1) * 4)))
            cycles = -(-o["K"] // step) * (28 * (MT * _loads(g, o["short"], True) + VN * _loads(g, o["wide"], o["along_k"])) + MT * VN * (32 if f32 else 4)) + waves * MT * VN * 16
            us = 2.6 + max(1.0, -(-g["M"] // down) / tuner.CU_COUNT) * cycles / 2400
            if best is None or us < best["us"]:
                best = dict(us=us, MT=MT, VN=VN, waves=waves)
    return dict(_in_steps(best, o, 1), us=best["us"]) if best is not None else None


def plan_few(g: dict, tiles_of=None) -> Optional[dict]:
    """Workgroup shape for `g` (see tuner.match_gemm) if one operand runs along k, the other along either axis, and this
    kernel is expected to beat the LDS tiles, else None.  `tiles_of()` gives the tile plan to compare with.

    The choice is between two estimates that are fits to both sides measured at 1072 shapes (rows and columns up to 16384,
    k up to 8192).  Of the 809 that take this kernel it is the slower side by more than a fifth at eleven, mostly wide
    outputs of a short or ragged k axis (float16 3392 x 256 x 63: 10.1 us against 5.7, 106 x 8500 x 56: 8.6 and 5.9); the
    estimate is raised by a third for more than 16 rows of whole 16-byte groups, where it was low and the tiles' was not.
    microseconds, tiles -> here: float32 64 x 256 x 784 22.3 -> 4.0, 128 x 1000 x 1000 28.1 -> 7.0, 300 x 300 x 300
    10.1 -> 3.4; float16 64 x 256 x 784 12.0 -> 2.9, 200 x 300 x 300 12.5 -> 2.6, 64 x 1024 x 1024 8.0 -> 3.3, 12 x 805 x
    1906 47 -> 6.0, 3 x 9287 x 5632 46.5 -> 33.  With the tiles stay float16 64 x 2048 x 4096 (10.2 against 11.9),
    16 x 14336 x 4096 (25.8 against 32), 64 x 10112 x 4416 of weights along k (30 against 53), 64 x 2304 x 5248 (20 against
    29) and float32 45 x 2133 x 3712 (27 against 35), 61 x 10492 x 1444 (38 against 58)."""
    o = _operands(g)
    best = _shape(g, o) if o is not None else None
    if best is None:
        return None
    if tiles_of is not None:
        t = _tile_launch(g, o, tiles_of())
        us = best["us"] + (0.35 * best["work"] if best["MT"] > 1 and not o["loose"] else 0.0)
        stream = o["w_bytes"] / 4.5e6  # the weights from memory, which either waits for
        if _tiles_stand(o, t) or max(us, stream) >= 0.95 * max(t["us"], stream):
            return None
    return _in_steps(best, o, _slices(max(1, o["K"] // (64 // o["eb"])), best["count"]))


def chain_pitch(K: int, dtype: DType) -> int:
    """Elements from row to row of a short operand in LDS: whole 16-byte groups, and rows start four banks apart."""
    group = 8 if dtype == DType.Float16 else 4
    return -(-K // group) * group + group


def gen_few(g: dict, p: dict, name: str, params: str, names, epi_fn: str, epi_args: str, decode: str, rows=None, behind=None, made_t: str = "float"):
    """(source text behind the prelude, grid, block).  `rows`: the short operand's rows as a `RowText` with outputs of its own
    name, made in LDS.  `behind`: what happens to the rows of the result (of type `made_t`), as a `RowText` that reads them from
    LDS; a workgroup's tile has to hold them whole."""
    s, w = p["short"], p["wide"]
    text = ((rows or behind).machinery if rows or behind else "") + fill(template("gemm_few.hip.inc"), dict(
        F32=1 if g["dtype"] == DType.Float32 else 0, R=p["R"], MT=p["MT"], C=p["C"], K=g["K"], WK=1 if p["along_k"] else 0, VN=p["VN"],
        WAVES=p["waves"], BATCH=p["batch"], SLICES=p["slices"], CHAIN=1 if rows else 0, PITCH=chain_pitch(g["K"], g["dtype"]),
        X_NONE=f"  const jh_val* const {names[g['gid_' + s]]} = nullptr;  // (the epilogue's parameters name every operand)" if rows else "",
        CHAIN_LOADS=(rows or behind).loads if rows or behind else "", CHAIN_STAGES=(rows or behind).stages if rows or behind else "",
        BEHIND=1 if behind else 0, HEIGHT=g["M"], MADE_ROWS=16 * (p["MT"] if s == "a" else p["VN"]), FIRST_ROW="r0" if s == "a" else "c0", MADE_T=made_t, EPILOGUE_FN=epi_fn, NAME=name, PARAMS=params, A_OFF=g["a_off"], B_OFF=g["b_off"], BATCH_DECODE=decode, X_PTR=names[g["gid_" + s]], W_PTR=names[g["gid_" + w]], X_BASE=s + "_base", W_BASE=w + "_base",
        X_ROW=g[p["row"][s]], W_ROW=g[p["row"][w]], W_K=g[w + "_sk"], ROW="rr" if s == "a" else "c", COL="c" if s == "a" else "rr", C_SM=g["c_sm"], C_SN=g["c_sn"],
        EPILOGUE_ARGS=epi_args))
    return text, (-(-p["C"] // (16 * p["VN"])) * p["slices"], p["nbatch"], -(-p["R"] // (16 * p["MT"]))), (64 * p["waves"], 1, 1)
