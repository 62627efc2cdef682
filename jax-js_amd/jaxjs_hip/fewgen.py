"""Plan and source of a GEMM too small for LDS tiles to fill the chip (`gemm_few.hip.inc`)."""

from __future__ import annotations

from typing import Optional

from .alu import DType
from .kernelgen import fill, template
from .tuner import CU_COUNT

FEW_LDS = 128 * 1024  # float32 sums of all waves
# Tile plans with at least this many workgroups stand, unless the operand along k has at most FEW_ROWS rows; with a float32
# k axis of under 256 twice as many, with float16 off the 16-byte grid one for every CU, and any the direct-to-LDS path takes.
FEW_WORKGROUPS = 64
FEW_ROWS = 64
FEW_DEEP = 4096       # longest k axis: each wave of a tile would walk too many steps


def _loads(g: dict, tag: str, along_k: bool) -> float:
    """Cost of a load of 16 bytes a lane against one from even addresses: float16 rows at odd elements straddle."""
    srow, other = (g["a_sm"], g["a_sk"]) if tag == "a" else (g["b_sn"], g["b_sk"])
    if g["dtype"] == DType.Float32 or (srow if along_k else other) % 2 == 0:
        return 1.0
    return 3.0 if along_k else 1.5


def plan_few(g: dict, tiles_of=None) -> Optional[dict]:
    """Workgroup shape for `g` (see tuner.match_gemm) if one operand runs along k, the other along either axis, and this
    kernel is expected to beat the LDS tiles, else None.  `tiles_of()` gives the tile plan to compare with.

    The estimates are fits to measurements (us, at 2.4 GHz).  Here: 2.6 for the launch; per step of a workgroup 28 cycles
    for each 16-row piece of an operand and the matrix instructions of four SIMDs; 16 cycles per wave and 16 x 16 tile for the
    sums; and W again from beyond the L2 for every row tile when it is more than 4 MB.  Tiles: 2.5 for the launch, 2 for
    folding a k split, and a time per element of k: float32 0.026 for a 64 x 64 tile; float16 0.0045 on the direct-to-LDS
    path, else 0.008 along k, 0.012 across and 0.025 across rows off the 16-byte grid.  They leave (before -> here):
    float32 64 x 256 x 784 22.3 -> 4.0, 128 x 1000 x 1000 28.1 -> 7.0, 300 x 300 x 300 10.1 -> 3.4; float16 64 x 256 x 784
    12.0 -> 2.9, 200 x 300 x 300 12.5 -> 2.6, 64 x 1024 x 1024 8.0 -> 3.3, 12 x 805 x 1906 47 -> 6.0, 3 x 9287 x 5632
    46.5 -> 33; but 64 x 2048 x 4096 (10.2 against 11.9) and 16 x 14336 x 4096 (25.8 against 32) stay with the tiles."""
    if g["dtype"] not in (DType.Float16, DType.Float32) or g.get("a_gather") or g.get("b_gather") or g["a_k0"] != g["K"] or g["b_k0"] != g["K"] or g["K"] < 32:
        return None
    nb = 1
    for b in g["batch"]:
        nb *= b[0]
    if nb > 65535:
        return None
    f32 = g["dtype"] == DType.Float32
    eb = 4 if f32 else 2
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
    R, C, K = rows[short], rows[wide], g["K"]
    if R > FEW_ROWS and K > FEW_DEEP or along_k and K > FEW_DEEP and (g.get("a_loose") or g.get("b_loose")):
        return None
    step = 64 // eb
    steps = -(-K // step)
    wx, ww = _loads(g, short, True), _loads(g, wide, along_k)
    w_bytes = C * K * eb * nb
    best = None
    for MT in (1, 2, 4):
        if MT > 1 and 8 * MT >= R:
            break
        for VN in ((1, 2, 4) if f32 or along_k else (2, 4, 8)):
            if MT * VN > 16 or (not along_k and C < VN) or (VN > 1 and 8 * VN >= C and VN != 2):
                continue
            waves = max(1, min(16, K // step or 1, FEW_LDS // (MT * 16 * (16 * VN + 1) * 4)))
            row_tiles = -(-R // (16 * MT))
            count = row_tiles * -(-C // (16 * VN)) * nb
            cycles = steps * (28 * (MT * wx + VN * ww) + MT * VN * (32 if f32 else 4)) + waves * MT * VN * 16
            us = 2.6 + max(1.0, count / CU_COUNT) * cycles / 2400 + (row_tiles * w_bytes / 10e6 if w_bytes > 4 << 20 else 0.0)
            if row_tiles <= 65535 and (best is None or us < best[0]):
                best = (us, MT, VN, waves)
    if best is None:
        return None
    us, MT, VN, waves = best
    if tiles_of is not None:
        tile = tiles_of()
        BM, BN, split = tile["BM"], tile["BN"], tile.get("SPLITK", 1)
        count = -(-g["M"] // BM) * -(-g["N"] // BN) * nb * split
        loose = g.get("a_loose") or g.get("b_loose")
        direct = not f32 and BM >= 128 and BN >= 128 and K % 32 == 0 and not loose
        many = 0 if direct else FEW_WORKGROUPS if not loose and not (f32 and K < 256) else FEW_WORKGROUPS * 2 if f32 else CU_COUNT
        if count >= many and R > FEW_ROWS or count >= FEW_WORKGROUPS and w_bytes > 96 << 20 and not loose:
            return None
        if f32:
            per_k = 0.026 * BM * BN / 4096
        elif direct:
            per_k = 0.0045 * BM * BN / 16384
        else:
            per_k = 0.008 if along_k else 0.012 if not g.get(wide + "_loose") else 0.025
        tiles_us = 2.5 + (2.0 if split > 1 else 0.0) + max(1.0, count / CU_COUNT) * K / split * per_k
        stream = w_bytes / 4.5e6
        if max(us, stream) >= 0.95 * max(tiles_us, stream):
            return None
    # Steps in equal shares for the waves, in equal batches of what the registers of a full workgroup hold in flight.
    share = -(-max(1, K // step) // waves)
    waves = -(-max(1, K // step) // share)
    most = max(1, (104 - 4 * MT * VN) // (4 * (MT + VN)))
    batch = -(-share // -(-share // most))
    return dict(R=R, MT=MT, C=C, short=short, wide=wide, along_k=along_k, VN=VN, waves=waves, batch=batch, nbatch=nb, row=row)


def gen_few(g: dict, p: dict, name: str, params: str, names, epi_fn: str, epi_args: str, decode: str):
    """(source text behind the prelude, grid, block)."""
    s, w = p["short"], p["wide"]
    text = fill(template("gemm_few.hip.inc"), dict(
        F32=1 if g["dtype"] == DType.Float32 else 0, R=p["R"], MT=p["MT"], C=p["C"], K=g["K"], WK=1 if p["along_k"] else 0, VN=p["VN"],
        WAVES=p["waves"], BATCH=p["batch"], EPILOGUE_FN=epi_fn, NAME=name, PARAMS=params, A_OFF=g["a_off"], B_OFF=g["b_off"], BATCH_DECODE=decode, X_PTR=names[g["gid_" + s]], W_PTR=names[g["gid_" + w]], X_BASE=s + "_base", W_BASE=w + "_base",
        X_ROW=g[p["row"][s]], W_ROW=g[p["row"][w]], W_K=g[w + "_sk"], ROW="rr" if s == "a" else "c", COL="c" if s == "a" else "rr", C_SM=g["c_sm"], C_SN=g["c_sn"],
        EPILOGUE_ARGS=epi_args))
    return text, (-(-p["C"] // (16 * p["VN"])), p["nbatch"], -(-p["R"] // (16 * p["MT"]))), (64 * p["waves"], 1, 1)
