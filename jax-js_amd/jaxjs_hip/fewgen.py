"""Plan and source of a float16 GEMM with few rows on one side (`gemm_f16_few.hip.inc`)."""

from __future__ import annotations

from typing import Optional

from .alu import DType
from .kernelgen import fill, template

FEW_ROWS = 64          # rows of the short operand at most: four 16-row matrix tiles
FEW_LDS = 128 * 1024   # float32 sums of all waves


def plan_few(g: dict) -> Optional[dict]:
    """Workgroup shape when `g` (see tuner.match_gemm) has at most 64 rows on one side and a plain, unit-stride operand pair,
    else None.  The short operand has to run along k, the wide one along either axis."""
    if g["dtype"] != DType.Float16 or g.get("a_gather") or g.get("b_gather") or g["a_k0"] != g["K"] or g["b_k0"] != g["K"] or g["K"] < 32:
        return None
    nb = 1
    for b in g["batch"]:
        nb *= b[0]
    if nb > 65535:
        return None
    short = "a" if g["M"] <= g["N"] else "b"
    wide = "b" if short == "a" else "a"
    R, C = min(g["M"], g["N"]), max(g["M"], g["N"])
    row = {"a": "a_sm", "b": "b_sn"}
    if R > FEW_ROWS or g[short + "_sk"] != 1:
        return None
    if g[wide + "_sk"] == 1:
        along_k = True
    elif g[row[wide]] == 1 and g[wide + "_sk"] > 0:
        along_k = False
    else:
        return None
    MT = -(-R // 16)
    # Against the direct-to-LDS tile.  This kernel reads the short operand again for every step of every narrow tile, so it
    # gains while W is small or the short operand is one matrix tile, and loses on a deep k axis under few tiles (us before
    # -> here, [out, in] / [in, out] weights): 4 x 2048 x 2048 9.2 -> 4.9 / 9.6 -> 5.7, 8 x 768 x 3072 11.6 -> 6.0 /
    # 12.2 -> 5.5, 32 x 4096 x 2048 10.2 -> 9.4 / 10.1 -> 9.2, 64 x 1024 x 1024 7.5 -> 7.5 / 8.0 -> 6.3; but 16 x 4096 x 4096
    # 11.3 -> 9.4 / 11.8 -> 14.3, 32 x 4096 x 4096 11.5 -> 16.6 / 12.5 -> 17.0, 16 x 14336 x 4096 31.2 -> 36.2 / 25.8 -> 32.1.
    # Off the 16-byte grid, or on a k axis that is not whole slabs, the other choice is the general tile, several times
    # slower: 4 x 3000 x 1500 17.1 -> 5.0 / 21.9 -> 6.3, 64 x 5000 x 3333 - / 48.3 -> 38.1, 3 x 9287 x 5632 - / 49.6 -> 35.5;
    # odd rows of [out, in] weights make every load straddle, 64 x 5000 x 3333 42.1 -> 51.6.
    bytes_w = 2 * C * g["K"] * nb
    if g["K"] % 32 == 0 and not g.get("a_loose") and not g.get("b_loose"):
        if not (bytes_w <= 48 << 20 if along_k and MT == 1 else bytes_w <= 16 << 20 and g["K"] * MT <= 4096 and g["K"] < 4096):
            return None
    elif along_k and (g["K"] > 4096 or (g["K"] % 2 and MT > 2)):
        return None
    # Columns per workgroup: whole lines of W where there are workgroups enough, narrower while half the chip would have
    # none; wider tiles read the short operand less often.
    if along_k:
        VN = 1 if MT == 1 else 2
        while VN < 4 and C * nb >= 16 * 2 * VN * 512:
            VN *= 2
    else:
        VN = 8 if MT <= 2 else 4
        while VN > 2 and -(-C // (16 * VN)) * nb < 96:
            VN //= 2
        if C < VN:
            return None
    # Steps in equal shares for the waves, in equal batches of what the registers of a full workgroup hold in flight.
    steps = g["K"] // 32 or 1
    share = -(-steps // max(1, min(16, FEW_LDS // (MT * 16 * (16 * VN + 1) * 4))))
    waves = -(-steps // share)
    most = max(1, (104 - 4 * MT * VN) // (4 * (MT + VN)))
    batch = -(-share // -(-share // most))
    return dict(R=R, C=C, short=short, wide=wide, along_k=along_k, VN=VN, waves=waves, batch=batch, nbatch=nb, row=row)


def gen_few(g: dict, p: dict, name: str, params: str, names, epi_fn: str, epi_args: str, decode: str):
    """(source text behind the prelude, grid, block)."""
    s, w = p["short"], p["wide"]
    text = fill(template("gemm_f16_few.hip.inc"), dict(
        R=p["R"], C=p["C"], K=g["K"], WK=1 if p["along_k"] else 0, VN=p["VN"], WAVES=p["waves"], BATCH=p["batch"], EPILOGUE_FN=epi_fn, NAME=name, PARAMS=params,
        A_OFF=g["a_off"], B_OFF=g["b_off"], BATCH_DECODE=decode, X_PTR=names[g["gid_" + s]], W_PTR=names[g["gid_" + w]], X_BASE=s + "_base", W_BASE=w + "_base",
        X_ROW=g[p["row"][s]], W_ROW=g[p["row"][w]], W_K=g[w + "_sk"], ROW="r" if s == "a" else "c", COL="c" if s == "a" else "r", C_SM=g["c_sm"], C_SN=g["c_sn"],
        EPILOGUE_ARGS=epi_args))
    return text, (-(-p["C"] // (16 * p["VN"])), p["nbatch"], 1), (64 * p["waves"], 1, 1)
