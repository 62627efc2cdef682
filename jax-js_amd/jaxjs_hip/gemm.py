"""Source generation for kernel class (d): MFMA GEMM (templates `gemm_f16.hip.inc`, `gemm_f32.hip.inc`).

The tuner's `match_gemm` has already reduced the Kernel to strides of a batched `C = A . B^T`-style
contraction; this module chooses the block tile, renders the fused epilogue as a device function
and fills the template.
"""

from __future__ import annotations

import math

from typing import Dict, List, Optional

from .alu import AluExp, AluOp, DType, Kernel, byteWidth
from .codegen import CTYPE, SOURCE_OPTION, STORAGE_CTYPE, HipExpCodegen, strip_parens
from .kernelgen import KernelSource, LaunchStep, _Body, _min_bytes, _prelude, _used_args, epilogue_compile_options, fill, template
from . import tuner
from .fewgen import gen_few, plan_few
from .tuner import TuneResult, classify_loads
from .wgradgen import gen_wgrad


def _short_axis_tile(g: dict, bm: int, bn: int, per_cu: int, both_k: bool, reads: bool):
    """(rate relative to 256x256 tiles on a long axis, plan) of a tile on the direct-to-LDS path where the k axis is so short
    that a workgroup's prologue and its stores of C weigh as much as its matrix instructions; None: as on a long axis.

    What helps is a second wave on every SIMD, in the same workgroup or in another one of the CU, whose phases overlap the
    first one's: 256x256 in eight waves (8192 x 1536 x 768 25.9 -> 24.1 us, 4096 x 4096 x 1024 36.7 -> 34.7, 2048 x 5632 x
    2048 51.2 -> 48.6, the same at 4096^3); 128x256 and 128x192 in two shallow stages, three workgroups to a CU (8192 x 3072
    x 768 43.4 -> 40.7).  128x192 tiles deal a width of 768 or 2304 out evenly: 8192 x 768 x 768 15.1 -> 13.4 us on 256
    workgroups instead of 192, 8192 x 2304 x 768 37.6 -> 34.1, 3072 x 3072 x 768 24.2 -> 20.8.  Operands that both run along k
    take deeper slabs in eight waves (6144 x 6144 x 512 54.9 -> 49.3, 8192 x 2304 x 768 42.6 -> 37.8).  Up to 4096 the 128x192
    tiles, one to a CU, stand behind an epilogue that `reads` buffers, whose loads add to the stores (8192 x 768 x 3072 with
    bias and residual 44.3 -> 41.2).  The bare product would gain as well (40.6 and 38.2), but tests/test_kernelgen.py pins its
    plan at this shape, so the rule asks for the epilogue."""
    if g["K"] > (4096 if reads and (bm, bn) == (128, 192) and per_cu == 1 else 2048) or g["K"] % 64:
        return None
    if (bm, bn) == (256, 256):
        return 1.06, dict(WM=2, WN=4)
    if (bm, bn) == (128, 192):
        if per_cu == 1:
            return 0.70 if both_k else 0.68, dict(BK=64, STAGES=4)
        return (0.83, dict(WM=4, WN=2, BK=64, STAGES=3)) if both_k else (0.87, dict(BK=32, STAGES=2, PIPE=0))
    if (bm, bn) == (256, 128) and both_k:
        return 0.85 if per_cu == 1 else 0.95, dict(WM=4, WN=2)
    if (bm, bn) == (128, 256) and not both_k and per_cu > 1 and g["K"] <= 1024:
        return 0.97, dict(WM=1, WN=4, BK=32, STAGES=2, PIPE=0)
    return None


def _f32_staged_tile(g: dict, tiles, nb: int) -> Dict[str, int]:
    """Tile and slices of a float32 product of whole 16-byte groups with a single-stride k axis and enough tiles to fill the
    chip.  128-row tiles take eight waves, two on a SIMD (2048 x 2048 x 1024 84.3 -> 81.0 us, 4032 x 4032 x 2368 657 -> 632, 1024 x
    1024 x 1024 29.3 -> 28.5).

    With two workgroups for every CU in some shape: the area of the tiles a CU gets, at the shape's rate (2048 x 3072 x 768 111
    -> 106 us in 128x64, 3224 x 1388 x 2964 320 in 64x64 and 354 in 128x64).  With fewer, by an estimate in microseconds: 3.7;
    that area times the depth of a slice, a CU that has one workgroup alone a fifth or a sixth slower; for the fold of slices
    inside the launch 0.65 a slice and 0.61 for every 10^6 partial sums; and a thirtieth for every halving of the axis, since
    workgroups that share a CU even their numbers out (128 x 14336 x 4096 178 in two slices, 190 in eight).  It is a fit to 11 products in both orders of B
    and all plans, within half a per cent of the fastest one in the mean and a third faster than a rule of 1.5 workgroups of
    128x64 a CU: 1280 x 640 x 320 19.3 -> 11.8 in 200 tiles instead of 100, 640 x 896 x 3136 84 -> 54 in eight slices, 192 x
    2112 x 1408 35 -> 22, 1536 x 768 x 768 36.6 -> 28.2, 768 x 1152 x 704 25.4 -> 21.4."""
    CU, best = tuner.CU_COUNT, None

    def plan(bm, bn, split=1):
        return dict(BM=bm, BN=bn, BK=32, WM=4 if bm == 128 else 2, WN=2, **(dict(SPLITK=split, FUSEK=1) if split > 1 else {}))
    for bm, bn, rate in ((128, 128, 266e3), (128, 64, 248.5e3), (64, 64, 230e3)):
        if g["M"] >= bm and g["N"] >= bn and tiles(bm, bn) >= 2 * CU:
            cost = -(-tiles(bm, bn) // CU) * bm * bn / rate
            if best is None or cost < best[0]:
                best = (cost, plan(bm, bn))
    if best is not None:
        return best[1]
    for bm, bn, rate, alone in ((64, 64, 185.5e3, 0.79), (128, 64, 222.0e3, 0.83)):
        for split in (1, 2, 4, 8):
            if split > 1 and (nb > 1 or g["K"] % (4 * split) or g["K"] // split < 128):
                continue
            per_cu = -(-tiles(bm, bn) * split // CU)
            us = 3.66 + per_cu * bm * bn * (g["K"] / split + 2.7) / (rate * (alone if per_cu == 1 else 1.0))
            if split > 1:
                us = (us + 0.645 * split + 0.611e-6 * split * g["M"] * g["N"]) * 1.035 ** (split.bit_length() - 1)
            if best is None or us < best[0]:
                best = (us, plan(bm, bn, split))
    return best[1]


# Plans of float32 products by direct loads: tile and waves, stages of a 32-deep slab (64 to 72 KB: two workgroups to a CU), and
# what `_f32_tile` estimates with, in microseconds: a launch; k steps that filling and emptying the pipeline costs; elements of
# C and k a microsecond, for a CU, alone as a part of that; folding a slice, and 10^6 of its partial sums.
_F32_PLANS = ((dict(BM=64, BN=64, WM=2, WN=2, WK=2, STAGES=4), 2.18, 71.0, 274.5e3, 0.948, 0.455, 0.873),
              (dict(BM=64, BN=64, WM=2, WN=2, WK=1, STAGES=4), 1.70, 62.5, 269.0e3, 0.927, 0.710, 0.391),
              (dict(BM=128, BN=64, WM=4, WN=2, WK=1, STAGES=3), 1.98, 35.0, 277.5e3, 0.959, 0.831, 0.714),
              (dict(BM=128, BN=128, WM=4, WN=2, WK=1, STAGES=2), 3.10, 12.2, 281.9e3, 0.988, 1.130, 0.993))


def _f32_tile(g: dict, tiles, nb: int, parts: int) -> Optional[Dict[str, int]]:
    """Plan of a float32 product whose slabs go to LDS by direct loads (`_f32_direct`), by an estimate: a launch, the tiles of the
    CU that gets most of them at the plan's rate, and the fold of slices of the k axis inside the launch.  It is a fit to 132
    products of 64 to 8192 rows, columns and k in both orders of B under all plans, within 1.7 per cent of the fastest one in
    the mean, 26 at worst (128 x 2144 x 216).  Against staging slabs in registers: 1024 x 1024 x 1024 25.9 -> 19.8 us, 2048
    150 -> 124, 4096 1080 -> 946 (145 TFLOP/s), 8192 8596 -> 7565, 3632 x 3088 x 144 49.6 -> 37.0, 1280 x 640 x 320 10.5 -> 7.6, 960 x 384 x
    3696 95.9 -> 41.5, 3672 x 768 x 1408 86.9 -> 69.4.
    `parts`: slices of the k axis that staging in registers takes, each a chain of roundings as long as itself.  Here a chain is half
    of what a wave has of a slice, and only plans that make it no longer are taken.  The others grew the error of four in 400 drawn products.  None where there are none:
    batches, which are not cut here, and products that staging cuts in up to 64.  And none where staging has the shorter walk along k: for a batch that
    it cuts in two behind k = 512, in four behind 256 (2 x 256 x 512 x 256 7.1 us staged, 6.5 here, x 512 8.8 and 10.0, x 2048 18.6 and 34.2; 2 x 512 x 512 x 512 11.3
    and 11.0, x 1024 18.1 and 18.7), and where it cuts in more than eight and all slices have a CU to themselves (48 x 320 x 17408 27.7 and 38.7; with 288 slices
    32 x 576 x 17408 41.0 and 38.8)."""
    if (nb > 1 and parts > 1 and parts * g["K"] > 1024) or (parts > 8 and parts * tiles(64, 64) <= tuner.CU_COUNT):
        return None
    best = None
    for plan, launch, fill, rate, alone, fold, sums in _F32_PLANS:
        count = tiles(plan["BM"], plan["BN"])
        for split in (1, 2, 4, 8):
            if 2 * plan["WK"] * split < parts or (split > 1 and (nb > 1 or g["K"] % (4 * split) or g["K"] // split < 64)):
                continue
            per_cu = -(-count * split // tuner.CU_COUNT)
            us = launch + per_cu * plan["BM"] * plan["BN"] * (g["K"] / split + fill) / (rate * (alone if per_cu == 1 else 1.0))
            if split > 1:
                us += fold * split + sums * 1e-6 * split * g["M"] * g["N"]
            if best is None or us < best[0]:
                best = (us, dict(plan, BK=32, DLDS=1, **(dict(SPLITK=split, FUSEK=1) if split > 1 else {})))
    return best and best[1]


def is_direct_product(kernel: Kernel) -> bool:
    """Whether `kernel` is better prepared with the option `direct_f32`: a float32 product that no other kernel takes.  (Why it is an
    option, which programs' schedules set, and not the plan of every such Kernel: the plans of smaller products, slabs staged in registers,
    are pinned by tests/test_kernelgen.py.)  Batches of one slab stay staged, there is nothing to fetch ahead (12 x 512 x 512 x 32 6.2 us and
    6.5 by direct loads, 36 x 128 x 128 x 32 5.0 and 5.4; of k = 64 24 x 256 x 256 5.8 and 5.3)."""
    if kernel.reduction is None or kernel.size == 0:
        return False
    t = tuner.tuneHip(kernel)
    return (t.klass == "gemm" and t.gemm["dtype"] == DType.Float32 and _f32_direct(t.gemm) and not (t.gemm["batch"] and t.gemm["K"] <= 32) and few_plan(t) is None
            and bool(choose_tile(dict(t.gemm, direct=True), bool(t.epilogue.collect(lambda n: n.op == AluOp.GlobalIndex))).get("DLDS")))


def _f32_direct(g: dict) -> bool:
    """Whether float32 operands can go to LDS by direct loads: plain ones of whole 16-byte groups, one stride along k, and offsets
    inside a slab that unsigned 32-bit byte counts hold."""
    return (not any(g.get(tag + w) for tag in "ab" for w in ("_gather", "_loose")) and g["a_k0"] == g["K"] and g["b_k0"] == g["K"] and g["K"] % 4 == 0
            and _f32_direct_span(g, 128, 128, 64))


def _f32_direct_span(g: dict, bm: int, bn: int, bk: int) -> bool:
    """Whether the lanes' offsets inside a slab of a tile are unsigned 32-bit byte counts."""
    strides = [(bm, g["a_sm"]), (bk, g["a_sk"]), (bn, g["b_sn"]), (bk, g["b_sk"])]
    return min(s for _, s in strides) >= 0 and max(bm * g["a_sm"] + bk * g["a_sk"], bn * g["b_sn"] + bk * g["b_sk"]) < 1 << 29


def choose_tile(g: dict, reads: bool = False) -> Dict[str, int]:
    """Block tile (and wave arrangement) for one GEMM: f16 by a small cost model, f32 128x128 down to 64x64.  `reads`: whether
    the epilogue reads buffers."""
    nb = 1
    for b in g["batch"]:
        nb *= b[0]

    def tiles(bm, bn):
        return -(-g["M"] // bm) * -(-g["N"] // bn) * nb

    CU = tuner.CU_COUNT
    # Slices of the k axis at most: 8, or 64 when the axis is very long (k = batch x positions of a filter cotangent:
    # 100352 against 9 output tiles), where the partial sums stay tiny next to the operands.
    plain_k = not (g.get("a_gather") or g.get("b_gather")) and g["a_k0"] == g["K"] and g["b_k0"] == g["K"]
    max_split = 64 if g["K"] >= (16384 if plain_k else 8192) else 8
    # A k axis that may be cut over workgroups: one stride per plain operand (a slice is a pointer offset), any gather
    # operand (a slice is an offset on the k its loader is asked for).
    # With exactly one gather operand and a short k axis the kernel is a forward convolution, whose stride-1 form has
    # its own template (image patch in LDS) that takes the whole k axis: those keep one slice.
    # A plain operand whose k axis has two strides (runs of k0 elements) can be cut where a slice is whole runs.
    two_level = [g[t + "_k0"] for t in ("a", "b") if g[t + "_k0"] != g["K"]]

    def runs_ok(slices):  # whole runs, or a whole fraction of one
        return all((g["K"] // slices) % k0 == 0 or k0 % (g["K"] // slices) == 0 for k0 in two_level)

    # (float32 has no such template: its forward convolutions are cut like any other gather GEMM.  Nor is that template
    # any use to a float16 convolution with a handful of tiles -- one small image, many channels: [1,512,7,7] * [512,512,3,3]
    # is 8 tiles whatever the template -- which is cut as well and then runs on the gather loaders.)
    one_gather = bool(g.get("a_gather")) != bool(g.get("b_gather"))
    few_tiles = (one_gather and 1024 <= g["K"] < 8192 and g["M"] >= 64 and tiles(64, 128) * 4 <= CU
                 and g["M"] * g["N"] * nb * g["K"] >= (1 << 26))  # (smaller than that, a launch is a launch)
    cut_k = (all(g["K"] % k0 == 0 for k0 in two_level)
             and (not one_gather or g["K"] >= 8192 or g["dtype"] == DType.Float32 or few_tiles))
    repack = _repack_operand(g)  # that operand is read from an aligned copy (rows padded to whole groups)
    loose_ops = bool(g.get("a_loose") or g.get("b_loose")) and repack is None

    def edge_ok(bm, bn):
        return (("a" in (repack or "") or _edge_ok(g["M"], bm, g["a_sk"] == 1))
                and ("b" in (repack or "") or _edge_ok(g["N"], bn, g["b_sk"] == 1)))

    if g["dtype"] == DType.Float32:
        # The f32 matrix pipe is 16x slower than the f16 one, so LDS traffic matters little and filling
        # every CU matters most: take the largest tile that still yields two workgroups per CU (the
        # second one hides the first one's staging latency).  Slabs are 32 deep (measured 3-6 % over 16 on
        # 2048^3 and 4096^3: half the barriers); gather operands keep the 16-deep slabs they were tuned with.
        bk = 32 if plain_k else 16
        # Direct loads where a schedule asks for them, and for any Kernel of at least two 128x128 tiles per CU, whose plans nothing pins
        # (8192^3 8596 -> 7565 us; 4096^3 1080 -> 946).
        # Short k axes behind an epilogue that reads buffers stay staged where there is more than a round of tiles: four workgroups have a
        # place on a CU then and hide each other's epilogues, where direct loads leave it to two (with a residual 784 x 3664 x 64 11.6 us staged, 15.7 by direct loads, 3220 x
        # 924 x 96 12.7 and 16.2, 3852 x 684 x 184 18.9 and 22.7, 3020 x 668 x 240 20.3 and 19.9; 1900 x 484 x 88, one round, 6.8 and 6.4).
        exposed = reads and g["K"] <= 256 and tiles(64, 64) > 2 * CU
        if _f32_direct(g) and (g.get("direct") or tiles(128, 128) >= 2 * CU) and not exposed:
            plan = _f32_tile(g, tiles, nb, 1 if tiles(128, 128) >= 2 * CU else choose_tile(dict(g, direct=False)).get("SPLITK", 1))
            if plan is not None:
                return plan
        if plain_k and not loose_ops and g["M"] >= 128 and g["N"] >= 64 and tiles(128, 64) * 4 > CU:
            return _f32_staged_tile(g, tiles, nb)
        # Among the shapes that do, the cheapest by (rounds of two workgroups per CU) x (tile area) / (rate of the
        # shape relative to 128x128: 0.97, 0.80): a last round that is nearly empty costs a whole one (products of
        # attention weights and values over 577 positions, 640 tiles of 128x64: 85.1 us, 66.1 us in 1280 of 64x64; the
        # scores of the same, 3200 tiles of 128x128: 84.9 us, 77.1 us in 6400 of 128x64; 512 x 11008 x 4096, 688 tiles of
        # 128x64: 600 -> 488 us in 1376 of 64x64; 2048 x 2304 x 768: 106 -> 91 us; 2048 x 3072 x 768 pays 4-7 % for it).
        # (16-deep slabs measured faster on some of these short k axes and slower on others: not taken.)
        best = None
        for bm, bn, rate in ((128, 128, 1.0), (128, 64, 0.97), (64, 64, 0.80)):
            if g["M"] >= bm and g["N"] >= bn and tiles(bm, bn) >= 2 * CU:
                cost = -(-tiles(bm, bn) // (2 * CU)) * bm * bn / rate
                if best is None or cost < best[0]:
                    best = (cost, dict(BM=bm, BN=bn, BK=bk))
        if best is not None:
            return best[1]
        # A handful of tiles (512^3 and smaller): the launch is as long as one workgroup's walk along k.  64x64 tiles and
        # up to 8 slices of at least 64 k, until every CU has a workgroup, folded inside the launch
        # (128^3 8.2 -> 5.4 us, 256^3 15.2 -> 6.3 us, 512^3 17.2 -> 9.1 us; the launch floor is 4.7 us).
        if plain_k and g["M"] >= 64 and g["N"] >= 64 and tiles(128, 64) * 4 <= CU:
            split = 1
            while tiles(64, 64) * split < CU and split < 8 and g["K"] % (split * 2 * bk) == 0 and g["K"] // (split * 2) >= 64:
                split *= 2
            return dict(BM=64, BN=64, BK=bk, **(dict(SPLITK=split, FUSEK=1) if split > 1 else {}))
        # Fewer tiles than that: 128x64 tiles with the k axis cut over blockIdx.y until the launch has at least 1.5
        # workgroups per CU (1024^3: 128 tiles x 4 slices, 37.9 -> 31.1 us; 128x14336x4096: 224 x 2, 222 -> 172 us).
        if plain_k and g["M"] >= 128 and g["N"] >= 64:
            split = 1
            while tiles(128, 64) * split < 1.5 * CU and split < 8 and g["K"] % (split * 2 * bk) == 0 and g["K"] // (split * 2) >= 256:
                split *= 2
            # The slices are folded inside the launch (1024^3: 30.2 -> 27.8 us, 128x14336x4096: 169 -> 166, same bits);
            # four waves stacked along m then measure another 1 % better than 2x2.
            return dict(BM=128, BN=64, BK=bk, SPLITK=split, **(dict(FUSEK=1, WM=4, WN=1) if split > 1 else {}))
        # Fewer than 128 rows or 64 columns: 64x64 tiles, the k axis cut the same way when they are few.  Gather operands
        # keep gaining up to four workgroups per CU (filter cotangents: [32,128,28,28] 143 us in 16 slices = 576
        # workgroups, 115 us in 32; [8,64,56,56] 54 -> 49 us; [16,128,28,28] 78 -> 67 us; [32,256,14,14] 183 -> 162 us).
        fill = 4.0 if not plain_k and g["K"] >= 8192 else 1.5
        split = 1
        while cut_k and tiles(64, 64) * split < fill * CU and split < max_split and g["K"] % (split * 2 * bk) == 0 and g["K"] // (split * 2) >= 256 and runs_ok(split * 2):
            split *= 2
        return dict(BM=64, BN=64, BK=bk, **(dict(SPLITK=split, FUSEK=1 if plain_k else 0) if split > 1 else {}))
    # f16: estimated time = (tiles the busiest CU runs) x (tile area) x (K + fixed per-tile overhead) / efficiency.
    # Efficiencies are measured rates of each tile shape relative to 256x256 on large problems (MI355X):
    # 128x256 0.84, 256x128 0.79, 128x128 0.62 with two workgroups resident per CU (8000^3: 0.63; 4100 x 4100 x 4096:
    # 218 us against 180 us with 128x256), 0.64 alone with its deeper slabs.  The fixed
    # overhead (pipeline fill + epilogue) is about 100 k-steps.  This picks big tiles for big problems and
    # smaller ones when 256x256 would leave the last round of CUs nearly empty (e.g. 288 tiles on 256 CUs).
    def k_split(count, fill=1.5):
        # Fewer workgroups than `fill` per CU: cut the k axis (partial sums in scratch, fold kernel) while slices stay >= 512 deep.
        split = 1
        gran = 64 if plain_k else 8  # whole slabs for the direct loads; the gather loaders take a ragged last slab
        while cut_k and count * split < fill * CU and split < max_split and g["K"] % (split * 2 * gran) == 0 and g["K"] // (split * 2) >= 512 and runs_ok(split * 2):
            split *= 2
        return dict(SPLITK=split) if split > 1 else {}

    if g["M"] <= 64 and g["N"] >= 128:
        # Few rows.  Many tiles (64 output channels of a convolution against thousands of positions): 64 x 256.
        if g["N"] >= 256 and tiles(64, 256) >= CU:
            return dict(BM=64, BN=256, WM=1, WN=4)
        # Few tiles (a linear layer on 2..64 tokens): bound by streaming B once, so what matters is enough workgroups
        # in flight -- 64 x 128 tiles and a k split (64 x 14336 x 4096: 65.7 us with 56 tiles of 64 x 256, 26.6 us with
        # 112 x 4 slices; 16 rows 24.6 us, 4 rows 23.5 us; B alone takes 15 us at the HBM rate).
        # When the direct-to-LDS template can take the shape (its A loads clamp to the last row that exists) its
        # 128x128 tiles in two or four slices stream B faster than the register-staged loaders, the empty rows of the
        # tile costing nothing that matters here: 4 / 16 / 64 x 14336 x 4096 25.2 / 25.9 / 28.2 -> 20.7 / 21.2 / 23.5 us,
        # 31 x 4096 x 4096 15.5 -> 13.0 us.  Those fall through to the plan below.
        # (Likewise a small B, whatever its k: the launch is all there is to it, and that template's is the shorter one --
        # 32 x 3072 x 768: 12.1 us on the register-staged loaders, 7.2 us for 128 rows on this one.)
        if not (edge_ok(128, 128) and plain_k and not loose_ops and repack is None and g["K"] % 128 == 0
                and (g["K"] >= 2048 or g["N"] * g["K"] <= (1 << 22)) and tiles(128, 128) * 2 <= CU):
            return dict(BM=64, BN=128, WM=1, WN=4, **k_split(tiles(64, 128)))
    elif g["N"] <= 64 and g["M"] >= 128:
        # A 128-wide tile would compute and store a half-empty block (attention's probabilities x V, N = head
        # size 64): measured 30 % faster with 128x64 tiles, which is then bound by reading A.
        return dict(BM=128, BN=64, WM=2, WN=2, **k_split(tiles(128, 64)))
    if (g["K"] <= 128 and g["K"] % 32 == 0 and plain_k and edge_ok(128, 128) and tiles(128, 128) >= 4 * CU
            and not loose_ops and repack is None):
        # A k axis of one to four slabs (attention scores: q.k^T over a head size of 64): the launch is bound by writing
        # C, and a workgroup spends its life in prologue and epilogue.  128x128 tiles with two shallow stages leave
        # room for four workgroups per CU, so that one's stores overlap another's loads and MFMAs
        # (96 x 1024 x 1024 x 64: 47.5 us with 256x256 tiles in the deep pipeline, 41.3 us = 5.5 TB/s this way).
        # Ragged lengths take it through clamped edge loads (scores of 128 heads over 577 positions: 48.9 us on the
        # 128x256 tiles the estimate below picked, 26.1 us here; 384 heads over 197: 17.2 -> 15.1 us).
        return dict(BM=128, BN=128, BK=32, STAGES=2, PIPE=0)
    if not plain_k and cut_k and g["K"] >= 8192 and tiles(128, 128) * 8 <= CU:
        # A handful of tiles over a very long k axis read through gather loaders (the filter cotangent of a convolution:
        # 9 taps x 64 x 64 or 128 x 128 outputs, k = batch x positions): 64x64 tiles waste no half-empty MFMA tile and
        # give the k slices four times as many workgroups ([32,64,56,56] 93 -> 72 us, [32,128,28,28] 187 -> 64 us).  With a
        # gather loader on one side only, one workgroup per CU is where more slices stop paying ([32,64,56,56]: 48 us in
        # 32 slices = 288 workgroups, 53 us in 64; [8,64,56,56]: 25 / 30 us); with one on both sides the loads are slower
        # and 1.5 per CU still gain ([32,128,28,28]: 61 us in 8 slices = 288 workgroups, 51 in 16, 53 in 32).
        both = bool(g.get("a_gather")) and bool(g.get("b_gather"))
        return dict(BM=64, BN=64, **k_split(tiles(64, 64), 1.5 if both else 1.0))
    if few_tiles and cut_k:
        # [1,512,7,7] * [512,512,3,3] f16: 47.9 us as 8 tiles of the patch template; [1,256,28,28] stride 2: 37.9 us.
        return dict(BM=64, BN=64, **k_split(tiles(64, 64)))
    if (bool(g.get("a_gather")) != bool(g.get("b_gather")) and g["K"] < 8192 and g["M"] >= 128 and g["N"] >= 128
            and g["a_k0"] == g["K"] and g["b_k0"] == g["K"] and tiles(128, 128) < CU):
        # One gather operand, fewer 128x128 tiles than CUs (the convolutions of audio models: a few hundred channels
        # against one long row of a few thousand positions): smaller tiles until the launch covers the chip.
        # [1,512,1500] * [512,512,3]: 48 tiles, 40.5 us; 192 of 64x64, 33.5 us.  [1,384,3000] stride 2: 36 tiles, 46.5 us;
        # 144 of 64x64, 24.3 us.  [1,256,8000] * [256,256,7]: 126 tiles, 50.5 us; 250 of 128x64, 42.3 us (64x64: 49.6).
        return dict(BM=64, BN=64) if tiles(128, 128) * 4 <= 1.5 * CU else dict(BM=128, BN=64)
    both_k = g["a_sk"] == 1 and g["b_sk"] == 1
    best = None
    for bm, bn, eff, extra in ((256, 256, 1.00, dict()), (128, 256, 0.84, dict(WM=1, WN=4)), (256, 128, 0.79, dict()),
                                (128, 128, 0.62, dict()), (128, 192, 0.68, dict())):
        if (bm > 128 and g["M"] < bm) or (bn > 128 and g["N"] < bn):
            continue
        per_cu = -(-tiles(bm, bn) // tuner.CU_COUNT)
        if (bm, bn) == (128, 128) and per_cu < 2:
            eff = 0.64
        whole = edge_ok(bm, bn) and (g["K"] % 32 == 0 or repack is not None) and plain_k and not loose_ops
        if not whole:
            # A ragged k axis, operands off the 16-byte grid or an edge the direct loads cannot clamp run the general
            # template, whose small tiles lose more
            # (8000^3: 838 / 597 / 691 / 512 TFLOP/s for the four shapes, against 1340 for whole 256x256 tiles).
            eff = {(256, 256): 0.63, (128, 256): 0.45, (256, 128): 0.52, (128, 128): 0.38}.get((bm, bn), eff)
        short = _short_axis_tile(g, bm, bn, per_cu, both_k, reads) if whole and repack is None else None
        if short is not None:
            eff, extra = short
        elif bn == 192:
            continue
        cost = per_cu * bm * bn * (g["K"] + 100) / eff
        if best is None or cost < best[0]:
            best = (cost, dict(BM=bm, BN=bn, **extra), per_cu)
    tile, per_cu = dict(best[1]), best[2]
    if (tile["BM"], tile["BN"]) == (128, 128) and per_cu == 1 and plain_k and g["K"] % 64 == 0:
        # One 128x128 workgroup per CU (or fewer): nothing shares the CU's LDS, so the slabs can be 64 deep in four
        # stages (128 KiB: twice the bytes in flight per workgroup; 2048^3 20.7 -> 19.6 us, 128x14336x4096 35.2 -> 27.4 us).
        if not both_k:
            tile.update(BK=64, STAGES=4)
        # Eight waves where the k axis is short: a second one on each SIMD covers the first one's prologue and stores (8192 x
        # 512 x 512 7.7 -> 7.3 us, 1600 x 512 x 512 7.3 -> 6.2, 4096 x 768 x 768 8.6 -> 7.9; from k = 1024 on no gain).
        if g["K"] < 1024 and not loose_ops and repack is None and edge_ok(128, 128):
            tile.update(BK=64, STAGES=4, WM=4, WN=2)
        # Half the CUs or fewer would get a workgroup: cut the k axis in two, four when a quarter or fewer would, the
        # slices folded inside the launch by the last one to arrive (128x14336x4096: 27.4 -> 26.0 us with a fold
        # launch, 24.7 folded in the launch; 128x4096x4096: 16.1 us in two slices, 13.9 in four; with 112 tiles four
        # slices cost more in partial sums than they gain).
        if tiles(128, 128) * 2 <= CU and g["K"] >= 2048 and g["K"] % 128 == 0:
            tile.update(SPLITK=4 if tiles(128, 128) * 4 <= CU and g["K"] >= 4096 and g["K"] % 256 == 0 else 2)
            # The slices take 32-deep slabs in four stages (64 KiB, so two workgroups fit a CU): as fast as the 64-deep
            # ones at their best and steady, where those swing between 21 and 28 us from launch to launch
            # (16 x 14336 x 4096: 20.2-20.7 us against 24-27; 128 rows: 26.0-26.6 against 29.6-32.9).
            tile.update(BK=32, STAGES=4)
            # Folding inside the launch is the direct-to-LDS template's: operands on the 16-byte grid, edges it can clamp.
            # Other shapes keep the split and fold in a second launch.
            # Two slices only: with four, the last workgroup's read-back of four slices behind the acknowledged stores
            # costs more than a fold launch (128x4096x4096: 16.0 us folded in the launch, 14.4 us with the fold kernel).
            # Edge tiles fold the same way (100 x 14336 x 4096: 31.1 us in four slices with a fold launch, 25.5 us in two).
            # Up to 64 rows the fold launch is the cheaper one: it touches the rows that exist, the fold inside the launch
            # whole tiles of partial sums (64 x 14336 x 4096: 23.5 against 23.7 us, 4 rows: 20.7 against 22.4 us).
            if edge_ok(128, 128) and not (g.get("a_loose") or g.get("b_loose")):  # (a repacked operand takes no k split)
                if tile["SPLITK"] == 2 and g["M"] > 64:
                    tile.update(FUSEK=1)
            else:  # the general template gains from more slices (100 x 14336 x 4096: 41.1 us in two, 34.6 us in four)
                tile.update(k_split(tiles(128, 128)) or dict(SPLITK=tile["SPLITK"]))
    elif not plain_k and cut_k and per_cu == 1 and tiles(tile["BM"], tile["BN"]) * 2 <= CU:
        # Gather operands on both sides and a handful of tiles over a long k axis (the filter cotangent of a
        # convolution: 9 taps x one tile, k = batch x positions): slices over workgroups, folded by a second launch.
        tile.update(k_split(tiles(tile["BM"], tile["BN"])))
    return tile


def _repack_operand(g: dict):
    """The operands ("a", "b" or "ab") that a pre-pass copies into scratch before the direct-to-LDS template reads them,
    or None.  That template loads whole 16-byte groups from the 16-byte grid and walks k in whole 32-deep slabs; an
    f16 operand off the grid (np.matmul against a [K, N] matrix with N = 50257: every row starts at an odd element) or a
    k axis that is not whole slabs (k = 50257, 4100, 1000) would otherwise send the whole GEMM to the general template
    (8192 x 50257 x 768: 1.19 ms against 0.80 ms).  The copy keeps the operand's orientation -- [rows][k] or [k][rows] --
    with rows rounded up to 8 and k to 32, zeros in the padding (2 x 2 bytes of traffic per element); a ragged k axis
    takes both operands.  Worth it when the other operand has enough rows to amortise the copy."""
    if g["dtype"] != DType.Float16 or g["batch"] or g.get("a_gather") or g.get("b_gather"):
        return None
    if g["a_k0"] != g["K"] or g["b_k0"] != g["K"] or g["K"] < 64:
        return None
    ragged_k = g["K"] % 32 != 0
    tags = "".join(t for t in ("a", "b") if g.get(t + "_loose") or ragged_k)
    if not tags:
        return None
    for t in tags:
        rows, other = (g["M"], g["N"]) if t == "a" else (g["N"], g["M"])
        srow, sk = (g["a_sm"], g["a_sk"]) if t == "a" else (g["b_sn"], g["b_sk"])
        if (srow != 1 and sk != 1) or rows < 128 or other < 512:
            return None
    if sum((g["M"] if t == "a" else g["N"]) for t in tags) * (g["K"] + 32) * 2 > (1 << 30):
        return None  # more than 1 GiB of copies: not at the price of that much scratch
    return tags


def is_sliced_product(kernel: Kernel) -> bool:
    """Whether `kernel` is better prepared with the option `sliced_f16`.  (An option for the reason that `direct_f32` is one.)

    Slices of the k axis that need not be equal, of operands that a pre-pass may have to copy first, where the tile plan cuts in
    halves and cuts no copies: 343 x 896 x 7104 40.2 -> 18.5 us, 448 x 395 x 3264 18.8 -> 10.9, 1125 x 768 x 4800 28.7 -> 18.4, 2176 x
    265 x 3843 (weights along k) 68.7 -> 24.1, 4070 x 448 x 5184 31.9 -> 29.0.  In one slice, copies of both operands in one launch
    instead of two (1984 x 1543 x 1281 26.4 -> 23.1), and behind fewer than 512 rows, where the general template's element loads cost
    18 ns per k (379 x 5964 x 6175 111 -> 66), from k = 1024 on (3520 x 355 x 666 12.8 against 15.2).  Of 105 products drawn that it
    could take alone none that it takes is more than 3 per cent slower.  Shapes of the kernel for few rows or tiles stay there (704 x 320 x 3600 13.6 against 19.5, 406 x 448 x 962 7.2 and 12.4).

    Whole operands that the tile plan gives eight waves stay with it: blocks of 128 to 1536 rows and width 192 or 224, whose second MLP product
    has a k axis of 768 or 896, were slower by up to 5 per cent with it cut (768 x 192 35.4 and 36.1 us for the block, 1344 x 224 41.7 and 43.8), but for 128 x 224, 33.5 and 32.8.  With
    four waves, from a k axis of 1024 on, blocks are faster by up to a quarter (448 x 704 66.8 -> 49.1, 768 x 768 60.5 -> 54.7, 462 x 256 37.0 -> 35.4), also
    where the tile plan folds two slices inside the launch.  With an epilogue that reads nothing one plain launch takes less, half a
    microsecond or, of operands that both run along k, one, and partial sums whose rows are off the 16-byte grid cost more: alone,
    384 x 1664 x 1344 9.6 us and 11.4 cut, along k 512 x 821 x 1280 8.8 and 12.6, 256 x 3008 x 1792 11.0 and 12.5, 1024 x 285 x 1344 9.1 and 9.9, but
    421 x 2112 x 1984 15.1 and 14.1, and 640 x 320 x 1088 8.6 and 8.3."""
    if kernel.reduction is None or kernel.size == 0:
        return False
    t = tuner.tuneHip(kernel)
    if t.klass != "gemm" or t.gemm["dtype"] != DType.Float16 or few_plan(t) is not None:
        return False
    g, p = t.gemm, sliced_plan(t.gemm)
    if p is None:
        return False
    if p["slices"] > 1 and not p["repack"]:
        tile = choose_tile(g)
        if tile.get("WM", 2) * tile.get("WN", 2) == 8:
            return False
        if tile.get("SPLITK", 1) == 1:
            reads = bool(t.epilogue.collect(lambda n: n.op == AluOp.GlobalIndex))
            return p["gain"] >= (0.0 if reads else 1.05 if g["a_sk"] == 1 and g["b_sk"] == 1 else 0.5) + (1e-6 * p["slices"] * g["M"] * g["N"] if g["N"] % 4 else 0.0)
    return p["slices"] > 1 or (p["repack"] == "ab" and (g["K"] >= 1024 or _repack_operand(g) is not None))


def sliced_plan(g: dict) -> Optional[dict]:
    """Copies (`repack`, see `_repack_operand`, or ""), padded k axis, slab depth and slices of the k axis, and what the slices gain, for a float16 product of up to
    one 128x128 tile per CU; None where the tile plan stands.  Slice z walks the slabs from z * slabs / slices on.  The number of
    slices is the cheapest by 6 ns per element of k, and 2.2 us and the partial sums at 5 TB/s for the fold's launch (2.0 cut 1536 x 256 x 1024: a
    block of 49.0 us took 49.7; with 2.2, 1680 x 288 x 1152 is still cut, 52.6 -> 51.5)."""
    if g["dtype"] != DType.Float16 or g["batch"] or g.get("a_gather") or g.get("b_gather") or g["a_k0"] != g["K"] or g["b_k0"] != g["K"]:
        return None
    M, N, K = g["M"], g["N"], g["K"]
    count = -(-M // 128) * -(-N // 128)
    if min(M, N) < 128 or K < 256 or count > tuner.CU_COUNT or any(g[s] != 1 and g[k] != 1 for s, k in (("a_sm", "a_sk"), ("b_sn", "b_sk"))):
        return None
    tags = "".join(t for t, rows in (("a", M), ("b", N))
                   if g.get(t + "_loose") or K % 32 or not _edge_ok(rows, 128, g[t + "_sk"] == 1))
    deep = 64 if K % 64 == 0 or K % 32 else 32
    slabs = -(-K // deep)
    if sum(M if t == "a" else N for t in tags) * slabs * deep * 2 > (1 << 30):
        return None
    most = max(1, min(slabs // 4, tuner.CU_COUNT // count))
    us = [-(-slabs // n) * deep * 0.006 + (2.2 + n * M * N * 8 / 5e6 if n > 1 else 0.0) for n in range(1, most + 1)]
    return dict(slices=us.index(min(us)) + 1, repack=tags, deep=deep, k=slabs * deep, gain=us[0] - min(us))


def _edge_ok(extent: int, tile: int, k_contiguous: bool) -> bool:
    """Whether the direct-to-LDS template can take an operand whose row count is `extent` in tiles of `tile` rows: whole
    tiles, or an edge tile whose loads can be clamped -- to the last row when the operand runs along k in memory, to
    the last whole 16-byte group of rows when it runs along its rows (the count must then be whole groups)."""
    return extent % tile == 0 or k_contiguous or (extent % 8 == 0 and extent >= 8)


def _strip_casts(e: AluExp) -> AluExp:
    """Drop float<->float casts around an operand (the MFMA consumes the storage type)."""
    while e.op == AluOp.Cast and e.dtype in (DType.Float16, DType.Float32, DType.Float64) and \
            e.src[0].dtype in (DType.Float16, DType.Float32):
        e = e.src[0]
    return e



# ---- row-vector gather: eight consecutive rows of a gather operand in one 128-bit load ------------------------------
#
# For an operand whose memory runs along its tile-row axis (the pixels of a stride-1 convolution's image operand),
# element (row0 + e, k) for an aligned row0 (row0 % 8 == 0) and e in 0..7 sits at index(row0, k) + e, and its mask is
# a conjunction of comparisons that are linear in e.  `_lin` proves that shape on the operand's own simplified
# expression: it splits an expression f(row) evaluated at row0 + e into rest(row0) + coef * e, pushing e out of
# `% D` and `/ D` when the rest is a multiple of 8 * coef that divides D.

def _has_row(e: AluExp) -> bool:
    return bool(e.collect(lambda x: x.op == AluOp.Special and x.arg[0] == "row"))


def _multiple_of(e: AluExp, m: int, group: int) -> bool:
    if m == 1:
        return True
    if e.op == AluOp.Const:
        return int(e.arg) % m == 0
    if e.op == AluOp.Special and e.arg[0] == "row":
        return group % m == 0
    if e.op in (AluOp.Add, AluOp.Sub):
        return _multiple_of(e.src[0], m, group) and _multiple_of(e.src[1], m, group)
    if e.op == AluOp.Mul:
        for x, y in ((e.src[0], e.src[1]), (e.src[1], e.src[0])):
            if y.op == AluOp.Const:
                c = abs(int(y.arg))
                if c % m == 0:
                    return True
                return c != 0 and _multiple_of(x, m // math.gcd(m, c), group)
        return False
    if e.op == AluOp.Mod and e.src[1].op == AluOp.Const and int(e.src[1].arg) % m == 0:
        return _multiple_of(e.src[0], m, group)
    return False


def _lin(e: AluExp, group: int = 8):
    """(coef, rest) with e(row0 + t) == rest(row0) + coef * t for every aligned row0 and t in [0, group), or None."""
    if not _has_row(e):
        return 0, e
    if e.dtype != DType.Int32:
        return None
    if e.op == AluOp.Special:
        return 1, e
    if e.op in (AluOp.Add, AluOp.Sub):
        a, b = _lin(e.src[0], group), _lin(e.src[1], group)
        if a is None or b is None:
            return None
        if e.op == AluOp.Add:
            return a[0] + b[0], AluExp.add(a[1], b[1])
        return a[0] - b[0], AluExp.sub(a[1], b[1])
    if e.op == AluOp.Mul:
        for x, y in ((e.src[0], e.src[1]), (e.src[1], e.src[0])):
            if y.op == AluOp.Const:
                a = _lin(x, group)
                if a is None:
                    return None
                return a[0] * int(y.arg), AluExp.mul(a[1], y)
        return None
    if e.op in (AluOp.Mod, AluOp.Idiv) and e.src[1].op == AluOp.Const:
        D = int(e.src[1].arg)
        a = _lin(e.src[0], group)
        if a is None or D <= 0:
            return None
        coef, rest = a
        if coef == 0:
            return 0, AluExp(e.op, e.dtype, (rest, e.src[1]))
        step = coef * group
        if coef < 0 or rest.min < 0 or D % step != 0 or not _multiple_of(rest, step, group):
            return None
        return (coef, AluExp.mod(rest, e.src[1])) if e.op == AluOp.Mod else (0, AluExp.idiv(rest, e.src[1]))
    return None


def rows8_form(oexp: AluExp, extent: int, group: int = 8):
    """For a gather operand's expression in (row, k, batch coordinates): (index at the group's first row, mask as a
    function of the extra variable `e` or None when unmasked, the GlobalIndex node) if `group` consecutive rows of
    every aligned group load `group` consecutive elements; else None."""
    cond = None
    node = oexp
    if node.op == AluOp.Where:
        zero = node.src[2]
        if zero.op != AluOp.Const or float(zero.arg) != 0.0:
            return None
        cond, node = node.src[0], node.src[1]
    if node.op != AluOp.GlobalIndex:
        return None
    a = _lin(node.src[0], group)
    if a is None or (group > 1 and a[0] != 1):
        return None
    idx0 = a[1].simplify()
    evar = AluExp.special(DType.Int32, "e", group)
    cond_e = None
    if cond is not None:
        atoms = []
        for atom in cond.splitOp(AluOp.Mul):
            neg = False
            inner = atom
            if inner.op == AluOp.Cmpne and inner.src[1].op == AluOp.Const and inner.src[0].dtype == DType.Bool and bool(inner.src[1].arg) is True:
                neg, inner = True, inner.src[0]
            if inner.op != AluOp.Cmplt:
                if _has_row(inner):
                    return None
                atoms.append(atom)
                continue
            sides = []
            for side in inner.src:
                la = _lin(side, group)
                if la is None:
                    return None
                coef, rest = la
                sides.append(AluExp.add(rest, AluExp.mul(evar, AluExp.i32(coef))) if coef else rest)
            lt = AluExp.cmplt(sides[0], sides[1])
            atoms.append(AluExp.cmpne(lt, AluExp.bool(True)) if neg else lt)
        cond_e = atoms[0]
        for x in atoms[1:]:
            cond_e = AluExp.mul(cond_e, x)
        cond_e = cond_e.simplify()
    return idx0, cond_e, node



def _swap_row_k(e: AluExp) -> AluExp:
    """The same expression with the roles of the Specials `row` and `k` exchanged."""
    def sw(n):
        if n.op == AluOp.Special and n.arg[0] == "row":
            return AluExp.special(n.dtype, "k", n.arg[1])
        if n.op == AluOp.Special and n.arg[0] == "k":
            return AluExp.special(n.dtype, "row", n.arg[1])
        return None
    return e.rewrite(sw)


def kvec_form(oexp: AluExp, K: int, group: int = 8):
    """`rows8_form` along the other axis: (index at the group's first k, mask as a function of `e`, the GlobalIndex node) if
    `group` consecutive k of every aligned group read `group` consecutive elements of one row (the image operand of a
    filter cotangent: k runs over batch x positions, and consecutive positions are consecutive pixels); else None."""
    form = rows8_form(_swap_row_k(oexp), K, group)
    if form is None:
        return None
    idx0, cond_e, node = form
    return _swap_row_k(idx0).simplify(), (None if cond_e is None else _swap_row_k(cond_e).simplify()), node


# ---- tap-major k order for convolution-like gather operands -----------------------------------------------------------
#
# The patch operand of a convolution reads element k = c * T + tap (T filter taps, tap fastest) of channel plane c:
# its index is `plane(c) + window(row, tap)` and its padding mask does not depend on c at all.  Walking k in the order
# k' = tap * C + c instead (a permutation of the reduction, applied to both operands alike) makes a slab of consecutive
# k' one tap over consecutive channels: the index/mask arithmetic is done once per (rows, tap) and each further channel
# costs one add and one load.

def _has_special(e: AluExp, name: str) -> bool:
    return bool(e.collect(lambda x: x.op == AluOp.Special and x.arg[0] == name))


def _affine_in(e: AluExp, name: str):
    """(coef, rest) with e == rest + coef * name, `name` reached only through +, - and * const; else None."""
    if not _has_special(e, name):
        return 0, e
    if e.op == AluOp.Special:
        return 1, AluExp.i32(0)
    if e.dtype != DType.Int32:
        return None
    if e.op in (AluOp.Add, AluOp.Sub):
        a, b = _affine_in(e.src[0], name), _affine_in(e.src[1], name)
        if a is None or b is None:
            return None
        return (a[0] + b[0], AluExp.add(a[1], b[1])) if e.op == AluOp.Add else (a[0] - b[0], AluExp.sub(a[1], b[1]))
    if e.op == AluOp.Mul:
        for x, y in ((e.src[0], e.src[1]), (e.src[1], e.src[0])):
            if y.op == AluOp.Const:
                a = _affine_in(x, name)
                return None if a is None else (a[0] * int(y.arg), AluExp.mul(a[1], y))
    return None


def _conj_terms(c: AluExp):
    """The terms of a conjunction (booleans multiply)."""
    if c.op == AluOp.Mul and c.dtype == DType.Bool:
        return _conj_terms(c.src[0]) + _conj_terms(c.src[1])
    return [c]


def interval_mask_form(cond: AluExp, name: str = "e"):
    """`cond` as (terms without `name`, lower bounds, upper bounds): cond == all(terms) and lo <= name < hi for every
    lower bound lo and upper bound hi (integer expressions without `name`); None when some term is not a comparison
    that is affine in `name` with coefficient +-1.  The padding masks of window views have this form: along a run of
    consecutive elements the elements inside the image are one interval."""
    inv, lows, highs = [], [], []
    for t in _conj_terms(cond):
        if not _has_special(t, name):
            inv.append(t)
            continue
        negated = False
        while t.op == AluOp.Cmpne and t.src[0].dtype == DType.Bool and any(x.op == AluOp.Const for x in t.src):
            c, x = (t.src[0], t.src[1]) if t.src[0].op == AluOp.Const else (t.src[1], t.src[0])
            if bool(c.arg):
                negated = not negated
            t = x
        if t.op != AluOp.Cmplt or t.src[0].dtype != DType.Int32:
            return None
        fa, fb = _affine_in(t.src[0], name), _affine_in(t.src[1], name)
        if fa is None or fb is None:
            return None
        coef, rest = fa[0] - fb[0], AluExp.sub(fa[1], fb[1])  # the term reads coef * name + rest < 0
        if coef == 1:  # name < -rest; negated: name >= -rest
            (lows if negated else highs).append(AluExp.sub(AluExp.i32(0), rest).simplify())
        elif coef == -1:  # name > rest, i.e. name >= rest + 1; negated: name <= rest, i.e. name < rest + 1
            (highs if negated else lows).append(AluExp.add(rest, AluExp.i32(1)).simplify())
        else:
            return None
    return inv, lows, highs


def mask_bits_fn(cond_e, tag: str, G: int, names, numerics: str) -> str:
    """C function `jh_mbits_<tag>(row, k, b0, b1, b2)`: bit e set when element e of the group of `G` that starts at
    (row, k) is inside the operand's mask.  From the interval form where the mask has one (two bounds and a few compares
    per group instead of a compare chain per element: the loaders of gather GEMMs are bound by such arithmetic), element
    by element otherwise."""
    head = f"static __device__ __forceinline__ unsigned jh_mbits_{tag}(int row, int k, int b0, int b1, int b2) {{\n"
    if cond_e is None:
        return head + f"  return {(1 << G) - 1}u;\n}}"
    vnames = {"row": "row", "e": "e", "k": "k", "b0": "b0", "b1": "b1", "b2": "b2"}
    form = interval_mask_form(cond_e)
    cg = HipExpCodegen(names, vnames, "  ", prefix=f"mb{tag}", numerics=numerics)
    if form is None:
        cg.indent = "    "
        cg.countReferences(cond_e)
        val = strip_parens(cg.run(cond_e))
        return (head + f"  unsigned bits = 0u;\n#pragma unroll\n  for (int e = 0; e < {G}; ++e) {{\n" + "\n".join(cg.take_lines())
                + f"\n    bits |= (({val}) ? 1u : 0u) << e;\n  }}\n  return bits;\n}}")
    inv, lows, highs = form
    for x in inv + lows + highs:
        cg.countReferences(x)
    inv_c = [strip_parens(cg.run(x)) for x in inv]
    lo_c = [strip_parens(cg.run(x)) for x in lows]
    hi_c = [strip_parens(cg.run(x)) for x in highs]
    body = "\n".join(cg.take_lines())
    lo_s = "".join(f"  lo = lo > ({x}) ? lo : ({x});\n" for x in lo_c)
    hi_s = "".join(f"  hi = hi < ({x}) ? hi : ({x});\n" for x in hi_c)
    ok = " && ".join(["lo < hi"] + [f"({x})" for x in inv_c])
    return (head + (body + "\n" if body else "") + f"  int lo = 0, hi = {G};\n{lo_s}{hi_s}"
            f"  return ({ok}) ? (((1u << hi) - 1u) & ~((1u << lo) - 1u)) : 0u;\n}}")


def tap_major_form(oexp: AluExp, K: int):
    """For a gather operand's expression in (row, k, batch coordinates): try k = c * T + tap for every T that the
    expression divides k by.  Returns dict(T, C, cs, exp) where `exp` is the operand re-expressed in (row, tap, batch
    coordinates) at c = 0, the element of channel c sitting `c * cs` further on and the mask not involving c; or None."""
    kvars = oexp.collect(lambda x: x.op == AluOp.Idiv and x.src[0].op == AluOp.Special and x.src[0].arg[0] == "k" and x.src[1].op == AluOp.Const)
    cands = sorted({int(x.src[1].arg) for x in kvars}, reverse=True)
    for T in cands:
        if T <= 1 or K % T != 0 or (K // T) % 8 != 0:
            continue
        C = K // T
        cvar, tvar = AluExp.special(DType.Int32, "c", C), AluExp.special(DType.Int32, "tap", T)
        kexp = AluExp.add(AluExp.mul(cvar, AluExp.i32(T)), tvar)
        e = oexp.rewrite(lambda n: kexp if (n.op == AluOp.Special and n.arg[0] == "k") else None).simplify()
        node, cond = e, None
        if node.op == AluOp.Where:
            if node.src[2].op != AluOp.Const or float(node.src[2].arg) != 0.0:
                continue
            cond, node = node.src[0], node.src[1]
        if node.op != AluOp.GlobalIndex or (cond is not None and _has_special(cond, "c")):
            continue
        a = _affine_in(node.src[0], "c")
        if a is None or a[0] <= 0:
            continue
        base = AluExp.globalIndex(node.dtype, node.arg[0], node.arg[1], a[1].simplify())
        exp0 = base if cond is None else AluExp.where(cond, base, e.src[2])
        return dict(T=T, C=C, cs=a[0], exp=exp0)
    return None


def few_plan(t: TuneResult) -> Optional[dict]:
    """The plan of the contraction `t` where the kernel for few rows or tiles takes it."""
    g = t.gemm
    if g is None or g.get("direct") or g.get("sliced") or t.params.get("gemm_tile") or _repack_operand(g) is not None:
        return None
    return plan_few(g, lambda: choose_tile(g))


def _flipped_filter(g: dict) -> bool:
    """Whether a product of two gather operands whose k axis would be cut is left whole where it is the cotangent of a
    convolution towards its image, so that the patch template takes it and reads the flipped filter through its pre-pass.  The
    slices read both operands element by element; the template's time is its walk over k, whatever the tiles (9 us per 1000 of
    k up to one tile a CU).  Of 120 shapes ([2..32, 64..512, 7..56 square], windows of 3 and 5) all 90 with k <= 4096 gain,
    1.16 to 4.6 times ([32,256,14,14] 3x3 93.5 -> 30.9 us, [16,64,28,28] 5x5 50.1 -> 22.7).  Behind a longer axis six of the
    twenty in 4 to 64 tiles lose (2 x [512,7,7] 41.6 against 53.5 us in 16 tiles, 52.2 against 54.3 in 64) and the ten in 112
    and more gain, 1.19 to 2.7 times (16 x [512,7,7] 65.6 -> 55.1 in 128): the line lies between.  Same error against double
    sums."""
    if g["dtype"] != DType.Float16 or not (g.get("a_gather") and g.get("b_gather")) or len(g["batch"]) != 1:
        return False
    return g["K"] <= 4096 or -(-g["M"] // 64) * -(-g["N"] // 128) * g["batch"][0][0] >= 96


def gen_gemm(kernel: Kernel, t: TuneResult, numerics: str, name: str, rows=None, behind=None, few=None) -> KernelSource:
    """`rows`: the rows of the short operand of a contraction that `few_plan` takes, made in the same launch (a `RowText` whose
    inputs come behind the kernel's).  `behind`: what happens to the result's rows in the same launch, under the plan `few` (a
    `RowText`; its inputs come behind the kernel's and its outputs are the launch's)."""
    g = t.gemm
    re = kernel.reduction
    assert g is not None and re is not None and t.epilogue is not None
    override = dict(t.params.get("gemm_tile") or {})
    few = few or few_plan(t)
    sliced = sliced_plan(g) if g.get("sliced") and not few and not override else None
    tile = dict() if ("BM" in override or "BN" in override) else dict(BM=128, BN=128) if few \
        else dict(BM=128, BN=128, BK=sliced["deep"], STAGES=4, SPLITK=sliced["slices"]) if sliced \
        else choose_tile(g, bool(t.epilogue.collect(lambda n: n.op == AluOp.GlobalIndex)))
    tile.update(override)
    if "BM" not in tile or "BN" not in tile:
        raise ValueError("a tile override must give both BM and BN")
    BM, BN = tile["BM"], tile["BN"]
    WM, WN = tile.get("WM", 2), tile.get("WN", 2)
    if BM % (32 * WM) or BN % (32 * WN):
        raise ValueError(f"tile {BM}x{BN} does not divide into {WM}x{WN} waves of 32x32 MFMA tiles")
    # float32 with direct loads: WK waves share out the k of a slab
    direct32 = int(tile.get("DLDS", 0)) if g["dtype"] == DType.Float32 and not few else 0
    WK = tile.get("WK", 1) if direct32 else 1
    nthreads = 64 * WM * WN * WK
    out_t = STORAGE_CTYPE[kernel.dtype]
    in_t = STORAGE_CTYPE[g["dtype"]]

    # Split of the k axis over blockIdx.y: every slice is the same kernel on K / split, its f32 accumulators go to a
    # scratch buffer [slice][output] and a generated fold Kernel adds the slices in order and applies the epilogue
    # (deterministic: no float atomics).  For launches that would otherwise leave most CUs without a workgroup.
    wgrad = t.params.get("wgrad") if not override else None  # a filter cotangent with a kernel of its own
    split = 1 if wgrad else int(tile.get("SPLITK", 1))
    K_full = g["K"]
    two_stride = dict(a=g["a_k0"] != K_full, b=g["b_k0"] != K_full)  # of the whole k axis, before any slicing
    if split > 1 and not sliced:
        vec_k = 8 if g["dtype"] == DType.Float16 else 4
        # a two-stride k axis is cut into whole runs, or a run into whole slices
        if (K_full % split or (K_full // split) % vec_k
                or any(g[t + "_k0"] != K_full and (K_full // split) % g[t + "_k0"] and g[t + "_k0"] % (K_full // split) for t in ("a", "b"))):
            split = 1
    if split > 1 and not override and not wgrad and not sliced and _flipped_filter(g):
        import copy

        t2 = copy.copy(t)
        t2.params = dict(t.params, gemm_tile=(("BM", 128), ("BN", 128), ("SPLITK", 1)))
        whole = gen_gemm(kernel, t2, numerics, name)
        if whole.info.get("conv"):
            return whole
    # An operand off the 16-byte grid that a pre-pass copies into scratch (see `_repack_operand`): from here on it is a
    # dense [K][rows_pad] operand named `jh_repack`.
    repack = sliced["repack"] if sliced else _repack_operand(g) if split == 1 and tile.get("REPACK", 1) and not few and not wgrad else None
    load_rows = dict(a=g["M"], b=g["N"])
    repack_src = {}
    if repack:
        k_pad = sliced["k"] if sliced else -(-g["K"] // 32) * 32
        for tg in repack:
            rows = load_rows[tg]
            srow = g["a_sm"] if tg == "a" else g["b_sn"]
            rkey = "a_sm" if tg == "a" else "b_sn"
            kc = g[tg + "_sk"] == 1  # runs along k: copied as [rows][k_pad]; else along its rows: [k_pad][rows_pad]
            rows_pad = rows if kc else -(-rows // 8) * 8
            repack_src[tg] = dict(gid=g["gid_" + tg], off=g[tg + "_off"], sk=g[tg + "_sk"], srow=srow, rows=rows, rows_pad=rows_pad,
                                  k=g["K"], k_pad=k_pad, kc=kc)
            load_rows[tg] = rows_pad
            g = dict(g, **{tg + "_off": 0, tg + "_sk": 1 if kc else rows_pad, rkey: k_pad if kc else 1, tg + "_loose": False})
        g = dict(g, K=k_pad, a_k0=k_pad, b_k0=k_pad)

    # ... or, with FUSEK (f32 template), folded inside the same launch by the slice that arrives last at the tile's
    # counter: one launch instead of two.
    fusek = 0
    if split > 1 and not sliced:
        KS = K_full // split
        run_full = dict(a=g["a_k0"], b=g["b_k0"])
        # (a slice inside one run has a single stride, like a slice of a single-stride axis)
        g = dict(g, K=KS, a_k0=KS if g["a_k0"] == K_full or g["a_k0"] > KS else g["a_k0"],
                 b_k0=KS if g["b_k0"] == K_full or g["b_k0"] > KS else g["b_k0"])
        fusek = split if tile.get("FUSEK", 0) else 0
    if split > 1 and not fusek:
        out_t = "float"

    used = _used_args(kernel.nargs, t.epilogue)
    used[g["gid_a"]] = g["dtype"]
    used[g["gid_b"]] = g["dtype"]
    names = [f"in{i}" for i in range(kernel.nargs)]
    params = ", ".join(
        [f"const {STORAGE_CTYPE[d or DType.Float32]}* __restrict__ {n}" for d, n in zip(used, names)]
        + [f"{out_t}* __restrict__ out"] + (["float* __restrict__ jh_part", "unsigned* __restrict__ jh_count"] if fusek else [])
        + [f"const jh_f16* __restrict__ jh_repack_{tg}" for tg in (repack or "")])

    # Fused epilogue as a device function of (acc, row, col, batch coordinates, buffers...).  The kernel's
    # epilogue is written over the flat output index; here that index is re-expressed through the tile's own
    # coordinates and simplified, so `gidx % N` becomes `col` and a bias load no longer depends on the row
    # (the compiler then hoists it out of the per-row loop instead of doing a division per element).
    if len(g["batch"]) > 3:
        raise ValueError("at most 3 batch axes")
    I32 = DType.Int32
    gexp = AluExp.add(AluExp.mul(AluExp.special(I32, "row", max(g["M"], 1)), AluExp.i32(g["c_sm"])),
                      AluExp.mul(AluExp.special(I32, "col", max(g["N"], 1)), AluExp.i32(g["c_sn"])))
    for k, (size, _sa, _sb, sc) in enumerate(g["batch"]):
        gexp = AluExp.add(AluExp.mul(AluExp.special(I32, f"b{k}", size), AluExp.i32(sc)), gexp)

    def _retarget(node):
        if node.op == AluOp.Special and node.arg[0] == "gidx":
            return gexp
        return None
    epilogue = t.epilogue.rewrite(_retarget).simplify()
    cg = HipExpCodegen(names, {"acc": "acc", "row": "row", "col": "col", "b0": "b0", "b1": "b1", "b2": "b2"}, "  ",
                       prefix="e", numerics=numerics)
    cg.countReferences(epilogue)
    value = strip_parens(cg.run(epilogue))
    epi_params = "".join(f", const {STORAGE_CTYPE[d or DType.Float32]}* __restrict__ {n}" for d, n in zip(used, names))
    epi_fn = (f"static __device__ __forceinline__ {out_t} jh_epilogue(float acc, int row, int col, int b0, int b1, int b2{epi_params}) {{\n"
              + "\n".join(cg.take_lines()) + f"\n  return ({out_t})({value});\n}}")
    src_options = epilogue_compile_options(epilogue)
    if split > 1 and not fusek:  # the fold kernel applies the epilogue; a slice stores its raw accumulator
        src_options = ""
        epi_fn = f"static __device__ __forceinline__ float jh_epilogue(float acc, int row, int col, int b0, int b1, int b2{epi_params}) {{\n  return acc;\n}}"
    epi_args = "".join(f", {n}" for n in names)
    if wgrad:
        return gen_wgrad(kernel, g, wgrad, numerics, name, params, names, out_t, epi_fn, epi_params, epi_args, _min_bytes(t.epilogue), src_options)

    if few:
        lines = ["  {", "    int rem = batch;"]
        for k, (size, sa, sb, sc) in reversed(list(enumerate(g["batch"]))):
            lines.append(f"    jh_b{k} = rem % {size}; rem /= {size};")
            lines.append(f"    a_base += (long long)jh_b{k} * {sa}ll; b_base += (long long)jh_b{k} * {sb}ll; c_base += (long long)jh_b{k} * {sc}ll;")
        lines.append("  }")
        gids = list(range(kernel.nargs))
        if rows:
            gids.remove(g["gid_" + few["short"]])
            params = ", ".join([f"const {STORAGE_CTYPE[used[i] or DType.Float32]}* __restrict__ {names[i]}" for i in gids] + rows.params + [f"{out_t}* __restrict__ out"])
        if behind:
            params = ", ".join(f"const {STORAGE_CTYPE[used[i] or DType.Float32]}* __restrict__ {names[i]}" for i in gids) + ", " + ", ".join(behind.params)
        if few["slices"] > 1:
            params += ", float* __restrict__ jh_part, unsigned* __restrict__ jh_count"
        text, grid, block = gen_few(g, few, name, params, names, epi_fn, epi_args, "\n".join(lines) if g["batch"] else "", rows, behind, out_t)
        need = _min_bytes(t.epilogue)
        for tg in ("a", "b"):
            need[g["gid_" + tg]] = max(need.get(g["gid_" + tg], 0), g[tg + "_len"] * byteWidth(g["dtype"]))
        if rows:
            src_options = src_options or (SOURCE_OPTION + "-fno-slp-vectorize\n" if rows.halves else "")
            need = {k: need[i] for k, i in enumerate(gids) if i in need}
            need.update({len(gids) + k: b for k, b in rows.need.items()})
            gids = list(range(len(gids) + len(rows.params)))
        outs = 1
        if behind:
            src_options = src_options or (SOURCE_OPTION + "-fno-slp-vectorize\n" if behind.halves else "")
            outs = sum(" __restrict__ out" in q for q in behind.params)
            need.update({len(gids) + k: b for k, b in behind.need.items()})
            gids = list(range(len(gids) + len(behind.params) - outs))
        args, scratch = [("in", i) for i in gids] + [("out", i) for i in range(outs)], []
        if few["slices"] > 1:  # the slices' sums, and a counter for each tile
            args += [("scratch", 0), ("scratch", 1)]
            scratch = [math.prod(grid) * 256 * few["MT"] * few["VN"] * 4, math.prod(grid) // few["slices"] * 4]
        return KernelSource([src_options + _prelude(numerics) + text], [LaunchStep(name, grid, block, 0, args)], scratch, "gemm", need,
                            dict(few=True, direct_lds=False, M=g["M"], N=g["N"], K=K_full, nbatch=few["nbatch"], tiles=grid[0] // few["slices"], waves=few["waves"],
                                 columns=16 * few["VN"], along_k=few["along_k"], splitk=few["slices"], rows=bool(rows)), zeroed_scratch=[1] if scratch else [])

    # Element loaders for gather operands: the operand's lowered expression (masked load through its view
    # chain) with the flat output index rebuilt from (tile row, batch coordinates) and ridx = k.
    gather_fns, gather_calls, gather_flags, gather_group, gather_oexp, gather_slow, element_fn = [], {}, {}, {}, {}, {}, {}
    lowered = _strip_casts(t.exp)
    operand_exps = {g["gid_a"]: None, g["gid_b"]: None}
    if g.get("a_gather") or g.get("b_gather"):
        assert lowered.op == AluOp.Mul
        for side in lowered.src:
            gids = {n.arg[0] for n in side.collect(lambda x: x.op == AluOp.GlobalIndex)}
            if len(gids) != 1:
                raise ValueError("gather operand must read exactly one buffer")
            operand_exps[gids.pop()] = _strip_casts(side)
    for tag, gid, is_gather, extent, c_stride in (("a", g["gid_a"], g.get("a_gather"), g["M"], g["c_sm"]),
                                                  ("b", g["gid_b"], g.get("b_gather"), g["N"], g["c_sn"])):
        gather_flags[tag] = 1 if is_gather else 0
        if not is_gather:
            gather_calls[tag] = f"({in_t})0"
            continue
        flat = AluExp.mul(AluExp.special(I32, "row", max(extent, 1)), AluExp.i32(c_stride))
        for k, (size, _sa, _sb, sc) in enumerate(g["batch"]):
            flat = AluExp.add(AluExp.mul(AluExp.special(I32, f"b{k}", size), AluExp.i32(sc)), flat)
        kvar = AluExp.special(I32, "k", max(K_full, 1))  # the whole axis: a slice's loader is asked for k + its offset

        def _retarget_operand(node, flat=flat, kvar=kvar):
            if node.op == AluOp.Special and node.arg[0] == "gidx":
                return flat
            if node.op == AluOp.Special and node.arg[0] == "ridx":
                return kvar
            return None
        oexp = operand_exps[gid].rewrite(_retarget_operand).reduceExactIndex().simplify()
        gather_oexp[tag] = oexp
        if tag == "b" and g["dtype"] == DType.Float16 and split == 1 and tile.get("CONV", 1) and not tile.get("TAPMAJOR", 0):
            # A stride-1 window walk over an image (verified on the operand's own index expression): the patch-in-LDS
            # convolution template instead of an im2col tile built element by element.  The other operand -- the filter --
            # may itself be a gather operand (the flipped, transposed filter of the cotangent towards the activations): the
            # template's weight pre-pass then reads it through its element loader.
            from .convgen import gen_conv

            conv_need = _min_bytes(t.epilogue)
            if g.get("a_gather"):
                for gid_, b_ in _min_bytes(t.exp).items():
                    conv_need[gid_] = max(conv_need.get(gid_, 0), b_)
            conv = gen_conv(kernel, g, oexp, numerics, name, params, names, epi_fn, epi_args, conv_need, tile,
                            a_gather_fns=element_fn["a"] if g.get("a_gather") else None)
            if conv is not None:
                conv.sources[0] = src_options + conv.sources[0]
                return conv
        gcg = HipExpCodegen(names, {"row": "row", "k": "k", "b0": "b0", "b1": "b1", "b2": "b2"}, "  ", prefix=f"g{tag}", numerics=numerics)
        gcg.countReferences(oexp)
        gval = strip_parens(gcg.run(oexp))
        element_fn[tag] = (f"static __device__ __forceinline__ {in_t} jh_gather_{tag}(int row, int k, int b0, int b1, int b2{epi_params}) {{\n"
                           + "\n".join(gcg.take_lines()) + f"\n  return ({in_t})({gval});\n}}")
        gather_fns.append(element_fn[tag])
        gather_calls[tag] = f"jh_gather_{tag}(row, k, jh_b0, jh_b1, jh_b2{epi_args})"
        # Row-vector loader: when G = 8 or 4 consecutive rows of an aligned group read G consecutive elements, one
        # unaligned G-element load replaces G element loads and their index arithmetic; masked lanes are zeroed
        # afterwards (pairs measured slower than the element loader and are not used).  A group whose bytes would leave the buffer (first/last rows of the whole array, where the
        # out-of-range part is masked anyway) takes the element loader through an out-of-line call.
        r8, G = None, 0
        if g["dtype"] == DType.Float16 and tile.get("ROWS8", 1):
            for G in (8, 4):
                r8 = rows8_form(oexp, extent, G)
                if r8 is not None:
                    break
        if r8 is not None:
            idx0, cond_e, gnode = r8
            vnames = {"row": "row", "e": "e", "k": "k", "b0": "b0", "b1": "b1", "b2": "b2"}
            icg = HipExpCodegen(names, vnames, "  ", prefix=f"i{tag}", numerics=numerics)
            icg.countReferences(idx0)
            ival = strip_parens(icg.run(idx0))
            ilines = "\n".join(icg.take_lines())
            gather_fns.append(f"static __device__ __forceinline__ int jh_gindex_{tag}(int row, int k, int b0, int b1, int b2) {{\n"
                              f"{ilines}\n  return {ival};\n}}")
            gather_fns.append(mask_bits_fn(cond_e, tag, G, names, numerics))
            buf = names[gnode.arg[0]]
            # The loader only forms addresses and mask bits and issues the loads (no use of the loaded data, no
            # branches): the stager applies the mask when it writes the slab to LDS, one slab later, so the eight
            # loads of a block are in flight together.  A group that would leave the buffer loads from a clamped
            # address and is flagged; the stager replaces it through the out-of-line element loader afterwards.
            gather_fns.append(
                f"typedef jh_f16 jh_part_{tag} __attribute__((ext_vector_type({G})));\n"
                f"struct __attribute__((packed, aligned(2))) jh_part_u_{tag} {{ jh_part_{tag} v; }};\n"
                f"static __device__ __attribute__((noinline)) jh_half8 jh_gather8_slow_{tag}(int row, int k, int b0, int b1, int b2{epi_params}) {{\n"
                f"  jh_half8 v;\n#pragma unroll\n  for (int e = 0; e < 8; ++e) v[e] = jh_gather_{tag}(row + e, k, b0, b1, b2{epi_args});\n  return v;\n}}\n"
                f"static __device__ __forceinline__ jh_g8 jh_gather8_{tag}(int row, int k, int b0, int b1, int b2{epi_params}) {{\n"
                f"  jh_g8 out;\n  out.keep = 0u;\n#pragma unroll\n  for (int j = 0; j < {8 // G}; ++j) {{\n"
                f"    const int r = row + j * {G};\n    const int i0 = jh_gindex_{tag}(r, k, b0, b1, b2);\n"
                f"    const bool inside = (unsigned)i0 <= (unsigned)({gnode.arg[1]} - {G});\n"
                f"    if (!inside) out.keep |= 0x100u;\n"
                f"    const jh_part_{tag} part = reinterpret_cast<const jh_part_u_{tag}*>({buf} + (inside ? i0 : 0))->v;\n"
                f"#pragma unroll\n    for (int e = 0; e < {G}; ++e) out.v[j * {G} + e] = part[e];\n"
                f"    out.keep |= jh_mbits_{tag}(r, k, b0, b1, b2) << (j * {G});\n  }}\n"
                f"  return out;\n}}")
            gather_slow[tag] = f"jh_gather8_slow_{tag}(row, k, jh_b0, jh_b1, jh_b2{epi_args})"
            gather_calls[tag] = f"jh_gather8_{tag}(row, k, jh_b0, jh_b1, jh_b2{epi_args})"
            gather_flags[tag] = 2
            gather_group[tag] = G

        # float32: four consecutive rows of an aligned group as one 128-bit load (the image of a stride-1 convolution),
        # the operand staged like one that runs along its rows.  Groups whose bytes would leave the buffer take the
        # element loader, which applies the mask itself.
        if g["dtype"] == DType.Float32 and tile.get("ROWS4", 1) and extent % 4 == 0 and g["K"] % 8 == 0:
            r4 = rows8_form(oexp, extent, 4)
            if r4 is not None:
                idx0, cond_e, gnode = r4
                vnames = {"row": "row", "e": "e", "k": "k", "b0": "b0", "b1": "b1", "b2": "b2"}
                icg = HipExpCodegen(names, vnames, "  ", prefix=f"i{tag}", numerics=numerics)
                icg.countReferences(idx0)
                ival = strip_parens(icg.run(idx0))
                gather_fns.append(f"static __device__ __forceinline__ int jh_gindex_{tag}(int row, int k, int b0, int b1, int b2) {{\n"
                                  + "\n".join(icg.take_lines()) + f"\n  return {ival};\n}}")
                gather_fns.append(mask_bits_fn(cond_e, tag, 4, names, numerics))
                buf = names[gnode.arg[0]]
                # (raw data + mask bits, the load unconditional: see the k-vector loader below)
                gather_fns.append(
                    f"static __device__ __forceinline__ jh_g4 jh_gather4_{tag}(int row, int k, int b0, int b1, int b2{epi_params}) {{\n"
                    f"  const int i0 = jh_gindex_{tag}(row, k, b0, b1, b2);\n  jh_g4 out;\n  out.keep = 0u;\n"
                    f"  const bool inb = (unsigned)i0 <= (unsigned)({gnode.arg[1]} - 4);\n  __builtin_memcpy(&out.v, {buf} + (inb ? i0 : 0), 16);\n"
                    f"  out.keep = inb ? jh_mbits_{tag}(row, k, b0, b1, b2) : 0u;\n"
                    f"  if (__builtin_amdgcn_ballot_w64(!inb) != 0) {{\n    if (!inb) {{\n"
                    f"#pragma unroll\n      for (int e = 0; e < 4; ++e) out.v[e] = jh_gather_{tag}(row + e, k, b0, b1, b2{epi_args});\n      out.keep = 15u;\n    }}\n  }}\n  return out;\n}}")
                gather_calls[tag] = f"jh_gather4_{tag}(row, k, jh_b0, jh_b1, jh_b2{epi_args})"
                gather_flags[tag], gather_group[tag] = 5, 4

        # k-vector loader: when neither row form applies but G consecutive k of an aligned group read G consecutive elements
        # of one row (the activations under a filter cotangent: k = batch x positions), one G-element load per group feeds
        # the k-contiguous staging path; masked lanes are zeroed, groups that would leave the buffer go element by element.
        if gather_flags[tag] == 1 and tile.get("KVEC", 1) and g["K"] % 8 == 0:
            kv, G = None, 0
            for G in ((8, 4) if g["dtype"] == DType.Float16 else (4,)):
                kv = kvec_form(oexp, K_full, G)
                if kv is not None:
                    break
            if kv is not None:
                idx0, cond_e, gnode = kv
                vnames = {"row": "row", "e": "e", "k": "k", "b0": "b0", "b1": "b1", "b2": "b2"}
                icg = HipExpCodegen(names, vnames, "  ", prefix=f"ki{tag}", numerics=numerics)
                icg.countReferences(idx0)
                ival = strip_parens(icg.run(idx0))
                gather_fns.append(f"static __device__ __forceinline__ int jh_kindex_{tag}(int row, int k, int b0, int b1, int b2) {{\n"
                                  + "\n".join(icg.take_lines()) + f"\n  return {ival};\n}}")
                gather_fns.append(mask_bits_fn(cond_e, tag, G, names, numerics))
                buf = names[gnode.arg[0]]
                W = 8 if g["dtype"] == DType.Float16 else 4  # elements per chunk of the staging path
                part_t = (f"typedef {in_t} jh_kpart_{tag} __attribute__((ext_vector_type({G})));\n"
                          f"struct __attribute__((packed, aligned({2 if g['dtype'] == DType.Float16 else 4}))) jh_kpart_u_{tag} {{ jh_kpart_{tag} v; }};\n")
                if g["dtype"] == DType.Float16:
                    # The f16 loader hands back the raw vector and the mask as bits (`jh_g8`), to be applied when the staged
                    # registers are written to LDS, and its vector load is unconditional (a group that would leave the buffer
                    # loads from the buffer's start instead).  A select right behind the load would wait for the data inside
                    # the fetch, and a load under a branch makes the wait before the commit of the previous slab a wait for
                    # everything (the counter of loads in flight is not known at the join): either way one slab's loads are
                    # in flight instead of two.  Groups off the buffer are redone element by element under one wave-uniform
                    # branch, which consumes its own loads before it ends.
                    gather_fns.append(
                        part_t + f"static __device__ __forceinline__ jh_g8 jh_gatherk_{tag}(int row, int k, int b0, int b1, int b2{epi_params}) {{\n"
                        f"  jh_g8 out;\n  out.keep = 0u;\n  unsigned off = 0u;\n#pragma unroll\n  for (int j = 0; j < {W // G}; ++j) {{\n    const int kk = k + j * {G};\n"
                        f"    const int i0 = jh_kindex_{tag}(row, kk, b0, b1, b2);\n"
                        f"    const bool inb = (unsigned)i0 <= (unsigned)({gnode.arg[1]} - {G});\n"
                        f"    const jh_kpart_{tag} part = reinterpret_cast<const jh_kpart_u_{tag}*>({buf} + (inb ? i0 : 0))->v;\n"
                        f"#pragma unroll\n    for (int e = 0; e < {G}; ++e) out.v[j * {G} + e] = part[e];\n"
                        f"    if (inb) out.keep |= jh_mbits_{tag}(row, kk, b0, b1, b2) << (j * {G});\n"
                        f"    off |= (inb ? 0u : 1u) << j;\n  }}\n"
                        f"  if (__builtin_amdgcn_ballot_w64(off != 0u) != 0) {{\n#pragma unroll\n    for (int j = 0; j < {W // G}; ++j)\n      if ((off >> j) & 1u) {{\n"
                        f"#pragma unroll\n        for (int e = 0; e < {G}; ++e) out.v[j * {G} + e] = jh_gather_{tag}(row, k + j * {G} + e, b0, b1, b2{epi_args});\n"
                        f"        out.keep |= {(1 << G) - 1}u << (j * {G});\n      }}\n  }}\n"
                        f"  return out;\n}}")
                else:
                    gather_fns.append(
                        part_t + f"static __device__ __forceinline__ jh_g4 jh_gatherk_{tag}(int row, int k, int b0, int b1, int b2{epi_params}) {{\n"
                        f"  jh_g4 out;\n  out.keep = 0u;\n  const int i0 = jh_kindex_{tag}(row, k, b0, b1, b2);\n"
                        f"  const bool inb = (unsigned)i0 <= (unsigned)({gnode.arg[1]} - 4);\n"
                        f"  const jh_kpart_{tag} part = reinterpret_cast<const jh_kpart_u_{tag}*>({buf} + (inb ? i0 : 0))->v;\n"
                        f"#pragma unroll\n  for (int e = 0; e < 4; ++e) out.v[e] = part[e];\n"
                        f"  out.keep = inb ? jh_mbits_{tag}(row, k, b0, b1, b2) : 0u;\n"
                        f"  if (__builtin_amdgcn_ballot_w64(!inb) != 0) {{\n    if (!inb) {{\n"
                        f"#pragma unroll\n      for (int e = 0; e < 4; ++e) out.v[e] = jh_gather_{tag}(row, k + e, b0, b1, b2{epi_args});\n      out.keep = 15u;\n    }}\n  }}\n"
                        f"  return out;\n}}")
                gather_calls[tag] = f"jh_gatherk_{tag}(row, k, jh_b0, jh_b1, jh_b2{epi_args})"
                gather_flags[tag] = 7 if g["dtype"] == DType.Float16 else 6
                gather_group[tag] = G

    # Tap-major k order (see `tap_major_form`): one gather operand whose k splits into (channel, tap), the other a plain
    # strided operand.  Both are then loaded through block/chunk loaders that take the first k' of eight consecutive
    # ones: k' = tap * C + c, original k = c * T + tap.
    tap_major = None
    gtags = [tg for tg in ("a", "b") if gather_flags[tg]]
    if g["dtype"] == DType.Float16 and tile.get("TAPMAJOR", 0) and len(gtags) == 1 and g["K"] % 8 == 0:
        gt = gtags[0]
        pt = "b" if gt == "a" else "a"
        tm = tap_major_form(gather_oexp[gt], g["K"])
        plain_ok = g[f"{pt}_k0"] == g["K"] and not g.get(f"{pt}_gather")
        if tm is not None and plain_ok:
            form, G = None, 0
            for G in (8, 4, 1):
                form = rows8_form(tm["exp"], 0, G)
                if form is not None:
                    break
            if form is not None:
                idx0, cond_e, gnode = form
                T, C, CS = tm["T"], tm["C"], tm["cs"]
                vnames = {"row": "row", "e": "e", "tap": "tap", "b0": "b0", "b1": "b1", "b2": "b2"}
                icg = HipExpCodegen(names, vnames, "  ", prefix=f"ti{gt}", numerics=numerics)
                icg.countReferences(idx0)
                ival = strip_parens(icg.run(idx0))
                gather_fns.append(f"static __device__ __forceinline__ int jh_tindex_{gt}(int row, int tap, int b0, int b1, int b2) {{\n"
                                  + "\n".join(icg.take_lines()) + f"\n  return {ival};\n}}")
                if cond_e is not None:
                    mcg = HipExpCodegen(names, vnames, "  ", prefix=f"tm{gt}", numerics=numerics)
                    mcg.countReferences(cond_e)
                    mval = strip_parens(mcg.run(cond_e))
                    gather_fns.append(f"static __device__ __forceinline__ bool jh_tmask_{gt}(int row, int e, int tap, int b0, int b1, int b2) {{\n"
                                      + "\n".join(mcg.take_lines()) + f"\n  return {mval};\n}}")
                    mask_bits = f"jh_tmask_{gt}(r, e, tap, b0, b1, b2)"
                else:
                    mask_bits = "true"
                buf, LEN, NG = names[gnode.arg[0]], gnode.arg[1], 8 // G
                gather_fns.append(
                    f"typedef jh_f16 jh_tpart_{gt} __attribute__((ext_vector_type({G})));\n"
                    f"struct __attribute__((packed, aligned(2))) jh_tpart_u_{gt} {{ jh_tpart_{gt} v; }};\n"
                    f"static __device__ __attribute__((noinline)) jh_half8 jh_gather8_tslow_{gt}(int row, int kp, int b0, int b1, int b2{epi_params}) {{\n"
                    f"  const int tap = kp / {C};\n  const int k = (kp - tap * {C}) * {T} + tap;\n"
                    f"  jh_half8 v;\n#pragma unroll\n  for (int e = 0; e < 8; ++e) v[e] = jh_gather_{gt}(row + e, k, b0, b1, b2{epi_args});\n  return v;\n}}\n"
                    f"// Eight consecutive k' (one tap, channels c0 .. c0+7) of eight consecutive rows: loads only; the mask (one\n"
                    f"// per block, it does not depend on the channel) is applied when the block is written to LDS.\n"
                    f"static __device__ __forceinline__ jh_gblock jh_gather_block_{gt}(int row, int kbase, int b0, int b1, int b2{epi_params}) {{\n"
                    f"  jh_gblock out;\n  out.keep = 0u;\n  const int tap = kbase / {C};\n  const int c0 = kbase - tap * {C};\n"
                    f"#pragma unroll\n  for (int j = 0; j < {NG}; ++j) {{\n    const int r = row + j * {G};\n"
                    f"    const int i0 = jh_tindex_{gt}(r, tap, b0, b1, b2) + c0 * {CS};\n"
                    f"    const bool inside = i0 >= 0 && (long long)i0 + 7ll * {CS} <= {LEN}ll - {G};\n"
                    f"    if (!inside) out.keep |= 0x100u;\n"
                    f"#pragma unroll\n    for (int e = 0; e < {G}; ++e) if ({mask_bits}) out.keep |= 1u << (j * {G} + e);\n"
                    f"    const jh_f16* const src = {buf} + (inside ? i0 : 0);\n"
                    f"#pragma unroll\n    for (int i = 0; i < 8; ++i) {{\n"
                    f"      const jh_tpart_{gt} part = reinterpret_cast<const jh_tpart_u_{gt}*>(src + (inside ? i * {CS} : 0))->v;\n"
                    f"#pragma unroll\n      for (int e = 0; e < {G}; ++e) out.v[i][j * {G} + e] = part[e];\n    }}\n  }}\n  return out;\n}}")
                gather_slow[gt] = f"jh_gather8_tslow_{gt}(row, k, jh_b0, jh_b1, jh_b2{epi_args})"
                gather_calls[gt] = f"jh_gather_block_{gt}(row, k, jh_b0, jh_b1, jh_b2{epi_args})"
                gather_flags[gt], gather_group[gt] = 3, G
                # the plain operand, eight consecutive k' at a time: elements T * stride apart
                srow, sk = (g["a_sm"], g["a_sk"]) if pt == "a" else (g["b_sn"], g["b_sk"])
                gather_fns.append(
                    f"static __device__ __forceinline__ jh_half8 jh_gather_chunk_{pt}(const jh_f16* __restrict__ base, int row, int kbase) {{\n"
                    f"  const int tap = kbase / {C};\n  const int c0 = kbase - tap * {C};\n"
                    f"  const jh_f16* p = base + (long long)row * {srow}ll + ((long long)c0 * {T} + tap) * {sk}ll;\n  jh_half8 v;\n"
                    f"#pragma unroll\n  for (int e = 0; e < 8; ++e) v[e] = p[(long long)e * {T * sk}ll];\n  return v;\n}}")
                gather_calls[pt] = f"jh_gather_chunk_{pt}({'Ap' if pt == 'a' else 'Bp'}, row, k)"
                gather_flags[pt] = 4
                tap_major = dict(T=T, C=C, group=G)

    # Batch index decode, innermost batch axis last in g["batch"].
    lines = ["  {", "    int rem = batch;"]
    for k, (size, sa, sb, sc) in reversed(list(enumerate(g["batch"]))):
        lines.append(f"    jh_b{k} = rem % {size}; rem /= {size};")
        lines.append(f"    a_base += (long long)jh_b{k} * {sa}ll; b_base += (long long)jh_b{k} * {sb}ll; c_base += (long long)jh_b{k} * {sc}ll;")
    lines.append("  }")
    nbatch = 1
    for b in g["batch"]:
        nbatch *= b[0]
    pitch = -(-kernel.size // 8) * 8  # elements between two slices' partial outputs
    if sliced and split > 1:
        lines.append(f"  const int jh_first = (int)blockIdx.y * {g['K'] // sliced['deep']} / {split};  // slab")
        lines.append(f"  a_base += (long long)jh_first * {sliced['deep'] * g['a_sk']}ll; b_base += (long long)jh_first * {sliced['deep'] * g['b_sk']}ll;"
                     f" c_base += (long long)blockIdx.y * {pitch}ll;")
    elif split > 1:
        # a slice starts K elements further along k: K * sk for one stride, (K / k0) runs of sk1 for two
        # (whether the axis has two strides is the whole axis's property: a slice of exactly one run has k0 == K too)
        # and for runs cut into r slices each, slice z is piece z % r of run z / r
        def slice_offset(tag):
            if not two_stride[tag]:
                return f"(long long)blockIdx.y * {g['K'] * g[tag + '_sk']}ll"
            if g["K"] % run_full[tag] == 0:
                return f"(long long)blockIdx.y * {(g['K'] // run_full[tag]) * g[tag + '_sk1']}ll"
            r = run_full[tag] // g["K"]
            return f"((long long)(blockIdx.y / {r}) * {g[tag + '_sk1']}ll + (long long)(blockIdx.y % {r}) * {g['K'] * g[tag + '_sk']}ll)"

        lines.append(f"  a_base += {slice_offset('a')}; b_base += {slice_offset('b')};"
                     + ("" if fusek else f" c_base += (long long)blockIdx.y * {pitch}ll;"))
        lines.append(f"  const int jh_k_off = (int)blockIdx.y * {g['K']};  // a gather loader is asked for k of the whole axis")
        for d in (gather_calls, gather_slow):
            for tag in list(d):
                d[tag] = d[tag].replace("(row, k, ", "(row, k + jh_k_off, ")

    tmpl = "gemm_f16.hip.inc" if g["dtype"] == DType.Float16 else "gemm_f32.hip.inc"
    fBK = int(tile.get("BK", 16)) if g["dtype"] == DType.Float32 else 0  # slab depth of the f32 template
    if direct32:
        stages = int(tile.get("STAGES", 4))
        if not _f32_direct(g):
            raise ValueError("direct loads of float32 operands need plain ones of whole 16-byte groups, with one stride along k")
        if fBK not in (32, 64) or BM * fBK * 4 % (16 * nthreads) or BN * fBK * 4 % (16 * nthreads) or fBK % (8 * WK):
            raise ValueError(f"{nthreads} threads in {WK} parts of k do not share out a {BM}- or {BN}-row slab {fBK} deep")
        if stages < 2 or max(stages * (BM + BN) * fBK * 4, (WK - 1) * BM * BN * 4) > 160 * 1024:
            raise ValueError(f"{stages} stages of {BM}+{BN} rows {fBK} deep do not fit the LDS")
    elif g["dtype"] == DType.Float32 and fBK in (16, 32, 64) and (BM * fBK // 4 % nthreads or BN * fBK // 4 % nthreads):
        raise ValueError(f"{nthreads} threads do not share out a {BM}- or {BN}-row slab {fBK} deep in whole groups")
    if not direct32 and g["dtype"] == DType.Float32 and (fBK not in (16, 32, 64) or 2 * (BM + BN) * (fBK + 4) * 4 > 160 * 1024):
        raise ValueError(f"f32 slab depth {fBK} is not 16, 32 or 64, or two {BM}+{BN}-row slabs of it do not fit the LDS")
    # Fast path: direct global->LDS loads need whole tiles (no bounds predicates) and 32-deep slabs.
    # Slab depth.  When both operands run along k in memory, 64-deep slabs make every row of a slab one whole
    # 128-byte line (a 32-deep slab asks for the two halves of each line about a microsecond apart, as two requests):
    # measured +7..21 % on every tile shape.  An operand that runs along m or n is fetched in whole lines either way,
    # and the shorter pipeline that 64-deep slabs leave room for then costs more than it gains.
    both_k = g["a_sk"] == 1 and g["b_sk"] == 1 and g["K"] % 64 == 0 and g["K"] >= 128
    dBK = tile.get("BK", 64 if both_k and tile.get("PIPE", 1) else 32) if g["dtype"] == DType.Float16 else 32
    if dBK not in (32, 64):
        raise ValueError(f"direct-to-LDS slab depth must be 32 or 64, got {dBK}")
    a_kc, b_kc = g["a_sk"] == 1 or g["K"] == 1, g["b_sk"] == 1 or g["K"] == 1
    full = (_edge_ok(load_rows["a"], BM, a_kc) and _edge_ok(load_rows["b"], BN, b_kc) and g["K"] % dBK == 0 and BM >= 128 and BN >= 128
            and tile.get("EDGE", 1) | (g["M"] % BM == 0 and g["N"] % BN == 0))
    any_gather = bool(g.get("a_gather") or g.get("b_gather"))
    loose = {tag: 1 if g.get(tag + "_loose") and not g.get(tag + "_gather") else 0 for tag in ("a", "b")}
    dlds = g["dtype"] == DType.Float16 and full and tile.get("DLDS", 1) and not any_gather and not (loose["a"] or loose["b"])
    if sliced and not dlds:
        raise ValueError("uneven slices of the k axis need the direct-to-LDS template")
    if repack and not dlds:  # the copy only serves the direct loads: plan again without it
        import copy

        t2 = copy.copy(t)
        t2.params = dict(t.params, gemm_tile=tuple(sorted(dict(override, REPACK=0).items())))
        return gen_gemm(kernel, t2, numerics, name)
    if dlds:
        tmpl = "gemm_f16_dlds.hip.inc"
    if dlds:
        # Stages that fit the 160 KiB of LDS: four of a 32-deep slab; of a 64-deep slab four (128x128), three
        # (128x256, 256x128), or the five-unit ring (256x256: 2.5 slabs).
        ring_default = 5 if dBK == 64 and (BM, BN) == (256, 256) and "STAGES" not in tile and tile.get("PIPE", 1) else 0
        stages_default = 4 if dBK == 32 else min(4, (160 * 1024) // ((BM + BN) * dBK * 2))
        sched = dict(BK=dBK, STAGES=tile.get("STAGES", stages_default), PIPE=tile.get("PIPE", 1), SGB=tile.get("SGB", 1), ASM_LOAD=tile.get("ASM", 1))
        # Scalar-base addressing needs every lane offset inside one slab of a tile to fit 32 bits.
        span = 2 * max((BM - 1) * abs(g["a_sm"]) + dBK * abs(g["a_sk"]), (BN - 1) * abs(g["b_sn"]) + dBK * abs(g["b_sk"]))
        sched["SADDR"] = 1 if tile.get("SADDR", 1) and span < 2 ** 31 and g["a_sm"] >= 0 and g["a_sk"] >= 0 and g["b_sn"] >= 0 and g["b_sk"] >= 0 else 0
        sched.update(SLICES=split if sliced else 1)
        sched.update(PIN=tile.get("PIN", 1), BAR_AT=tile.get("BAR_AT", 2), READ_AHEAD=tile.get("RA", 1), LOADS_LATE=tile.get("LATE", 1))
        # Tile walk: groups of 4 tile rows (8192^3: 865 -> 853 us against groups of 8, 873 with 16; one group spanning
        # all rows loses a third).  Nontemporal C stores only for the f32 partials of a k split, where a wave's store
        # covers whole 128-byte lines (128x14336x4096: 26.1 -> 25.3 us): with 2-byte outputs they gain nothing once the
        # walk is in groups of 4 and the half-line writes cost a third more HBM write traffic (WRITE_SIZE 132 -> 176 MiB).
        sched.update(GROUP_M=int(tile.get("GM", 4)), NT_STORE=int(tile.get("NTS", 1 if split > 1 and not fusek else 0)), FUSEK=fusek)
        sched["RING"] = ring = tile.get("RING", ring_default)
        if ring and (ring != 5 or BM != BN or not sched["PIPE"]):
            raise ValueError("the unit ring is five units of a square block tile under the phase-pipelined loop")
        if (ring * BM * dBK * 2 if ring else sched["STAGES"] * (BM + BN) * dBK * 2) > 160 * 1024:
            raise ValueError(f"{ring or sched['STAGES']} {'units' if ring else 'stages'} of a {BM}x{BN}x{dBK} slab do not fit the 160 KiB of LDS")
        # Vector epilogue: needs unit column stride and 8-element alignment of every row / batch start of C.
        # It pays when the epilogue itself reads buffers (bias, residual): those become 128-bit loads.  A plain
        # cast-and-store epilogue measures the same either way and keeps the simpler path.
        has_loads = bool(epilogue.collect(lambda x: x.op == AluOp.GlobalIndex)) and split == 1
        vec = (split == 1 and tile.get("VEPI", 1 if has_loads else 0) and g["c_sn"] == 1 and g["c_sm"] % 8 == 0 and all(b[3] % 8 == 0 for b in g["batch"])
               and kernel.dtype != DType.Bool and (g["N"] % BN == 0 or g["N"] % 8 == 0))  # an edge tile ends on a whole group of 8
        if vec:
            vnames = {"acc": "acc", "row": "row", "col": "col", "b0": "b0", "b1": "b1", "b2": "b2"}
            body = _Body(epilogue, names, vnames, "col", "c0", 8, classify_loads(epilogue, "col", 8), numerics, "      ", "e")
            vhoist, vloads = body.hoisted()
            vbody, vvalue = body.lanes(vloads)
            sched.update(VEC_EPI=1, VEPI_LOADS=vhoist, VEPI_BODY=vbody, VEPI_VALUE=vvalue, OUT_T=out_t)
        else:
            sched.update(VEC_EPI=0, VEPI_LOADS="", VEPI_BODY="", VEPI_VALUE="0", OUT_T=out_t)
    elif g["dtype"] == DType.Float16:
        sched = dict(COMMIT_A=tile.get("CA", 2), COMMIT_B=tile.get("CB", 3), FETCH_A=tile.get("FA", 0),
                     FETCH_B=tile.get("FB", 1), IGLP=tile.get("IGLP", -1), SCHED_FENCE=tile.get("FENCE", 0),
                     A_LOOSE=loose["a"], B_LOOSE=loose["b"])
    elif direct32:
        tmpl = "gemm_f32_dlds.hip.inc"
        sched = dict(BK=fBK, STAGES=stages, WK=WK, FUSEK=fusek)
    else:
        sched = dict(BK=fBK, FRAG_FENCE=int(tile.get("FENCE", 1)), FUSEK=fusek, A_LOOSE=loose["a"], B_LOOSE=loose["b"])
    if not dlds:
        sched.update(GATHER_FNS="\n".join(gather_fns), A_GATHER=gather_flags["a"], B_GATHER=gather_flags["b"],
                     GATHER_A_CALL=gather_calls["a"], GATHER_B_CALL=gather_calls["b"],
                     GATHER_A_SLOW=gather_slow.get("a", "jh_half8{0, 0, 0, 0, 0, 0, 0, 0}"), GATHER_B_SLOW=gather_slow.get("b", "jh_half8{0, 0, 0, 0, 0, 0, 0, 0}"))
    src = src_options + _prelude(numerics) + fill(template(tmpl), dict(sched, 
        M=g["M"], N=g["N"], K=g["K"], M_LOAD=load_rows["a"], N_LOAD=load_rows["b"], BM=BM, BN=BN, WM=WM, WN=WN,
        A_KCONTIG=0 if gather_flags["a"] in (2, 3, 5) else (1 if g["a_sk"] == 1 or g["K"] == 1 or gather_flags["a"] in (1, 4, 6, 7) else 0),
        B_KCONTIG=0 if gather_flags["b"] in (2, 3, 5) else (1 if g["b_sk"] == 1 or g["K"] == 1 or gather_flags["b"] in (1, 4, 6, 7) else 0),
        NBATCH=nbatch, EPILOGUE_FN=epi_fn, NAME=name, PARAMS=params,
        A_OFF=g["a_off"], B_OFF=g["b_off"], BATCH_DECODE="\n".join(lines),
        A_PTR="jh_repack_a" if "a" in (repack or "") else names[g["gid_a"]], B_PTR="jh_repack_b" if "b" in (repack or "") else names[g["gid_b"]],
        A_SM=g["a_sm"], A_SK=g["a_sk"], B_SN=g["b_sn"], B_SK=g["b_sk"],
        A_K0=g["a_k0"], A_SK1=g["a_sk1"], B_K0=g["b_k0"], B_SK1=g["b_sk1"],
        C_SM=g["c_sm"], C_SN=g["c_sn"], EPILOGUE_ARGS=epi_args))
    tiles = -(-g["M"] // BM) * -(-g["N"] // BN) * nbatch
    if fusek and g["dtype"] == DType.Float16 and not dlds:
        raise ValueError("an in-launch fold of a k split needs the direct-to-LDS f16 template or the f32 template")
    out_args = [("out", 0), ("scratch", 0), ("scratch", 1)] if fusek else [("scratch", 0) if split > 1 else ("out", 0)]
    step = LaunchStep(name, (tiles, split, 1), (nthreads, 1, 1), 0, [("in", i) for i in range(kernel.nargs)] + out_args)
    need = _min_bytes(t.epilogue)
    if any_gather:
        for gid_, b_ in _min_bytes(t.exp).items():
            need[gid_] = max(need.get(gid_, 0), b_)
    eb = byteWidth(g["dtype"])
    need[g["gid_a"]] = max(need.get(g["gid_a"], 0), g["a_len"] * eb)
    need[g["gid_b"]] = max(need.get(g["gid_b"], 0), g["b_len"] * eb)
    info = dict(BM=BM, BN=BN, WM=WM, WN=WN, BK=dBK if dlds else (64 if g["dtype"] == DType.Float16 else fBK), direct_lds=bool(dlds), tiles=tiles, a_kcontig=g["a_sk"] == 1, b_kcontig=g["b_sk"] == 1,
                M=g["M"], N=g["N"], K=K_full, nbatch=nbatch, splitk=split)
    if dlds:
        info.update(stages=sched["STAGES"], ring=sched["RING"])
    if any_gather:
        info["gather"] = {tag: {0: "none", 1: "element", 2: f"rows{gather_group.get(tag, 8)}", 3: f"tap-major rows{gather_group.get(tag, 8)}",
                                4: "tap-major strided" if tap_major is not None else f"k{gather_group.get(tag, 8)}", 5: "rows4", 6: "k4", 7: f"k{gather_group.get(tag, 8)}"}[gather_flags[tag]] for tag in ("a", "b")}
        if tap_major is not None:
            info["tap_major"] = tap_major
    scratch, copies, preps = [], [], []
    if repack:
        src += "\nstruct __attribute__((packed, aligned(2))) jh_half8_u { jh_half8 v; };\n"
        calls = []
        for tg in repack:
            rs = repack_src[tg]
            if rs["kc"]:
                groups, total = rs["k_pad"] // 8, rs["rows"] * (rs["k_pad"] // 8)
                body = (f"  const int r = (int)(i / {groups}), k0 = (int)(i % {groups}) * 8;\n"
                        f"  const jh_f16* __restrict__ p = src + {rs['off']}ll + (long long)r * {rs['srow']}ll + k0;\n"
                        f"  const int valid = {rs['k']} - k0;\n"
                        f"  jh_f16* const q = dst + (long long)r * {rs['k_pad']} + k0;\n")
                what = f"[{rs['rows']} rows][{rs['k']} k] (row stride {rs['srow']}) -> [{rs['rows']}][{rs['k_pad']}]"
            else:
                groups, total = rs["rows_pad"] // 8, rs["k_pad"] * (rs["rows_pad"] // 8)
                body = (f"  const int k = (int)(i / {groups}), r0 = (int)(i % {groups}) * 8;\n"
                        f"  const jh_f16* __restrict__ p = src + {rs['off']}ll + (long long)k * {rs['sk']}ll + r0;\n"
                        f"  const int valid = k < {rs['k']} ? {rs['rows']} - r0 : 0;\n"
                        f"  jh_f16* const q = dst + (long long)k * {rs['rows_pad']} + r0;\n")
                what = f"[{rs['k']} k][{rs['rows']} rows] (k stride {rs['sk']}) -> [{rs['k_pad']}][{rs['rows_pad']}]"
            src += (f"""
// Operand {tg.upper()} {what}, first element {rs['off']}: eight elements per thread, one under-aligned 16-byte load and one
// aligned store; what lies past the operand's extents is zeros.
static __device__ __forceinline__ void jh_repack_of_{tg}(const jh_f16* __restrict__ src, jh_f16* __restrict__ dst, const long long i) {{
  if (i >= {total}ll) return;
{body}  jh_half8 v;
  if (valid >= 8) {{
    v = reinterpret_cast<const jh_half8_u*>(p)->v;
  }} else {{
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = e < valid ? p[e] : (jh_f16)0.0f;
  }}
  *reinterpret_cast<jh_half8*>(q) = v;
}}
""")
            calls.append((tg, -(-total // 256)))
            copies.append(("scratch", len(scratch) + (split > 1)))  # (the buffer of a split's partial sums is the first)
            scratch.append(rs["k_pad"] * rs["rows_pad"] * 2)
        step.args += copies
        for group in ([calls] if sliced else [[c] for c in calls]):  # one launch for both, but where tests pin single Kernels' launches
            jump, first = "", 0
            for tg, blocks in group:
                jump += (f"  if (blockIdx.x >= {first}u && blockIdx.x < {first + blocks}u)"
                         f" jh_repack_of_{tg}(src_{tg}, dst_{tg}, (long long)(blockIdx.x - {first}u) * 256 + threadIdx.x);\n")
                first += blocks
            tags = "".join(tg for tg, _ in group)
            src += (f'\nextern "C" __global__ __launch_bounds__(256) void {name}_repack_{tags}('
                    + ", ".join(f"const jh_f16* __restrict__ src_{tg}, jh_f16* __restrict__ dst_{tg}" for tg in tags) + f") {{\n{jump}}}\n")
            preps.append(LaunchStep(f"{name}_repack_{tags}", (first, 1, 1), (256, 1, 1), 0,
                                    [a for tg in tags for a in (("in", repack_src[tg]["gid"]), copies[repack.index(tg)])]))
        info["repack"] = repack
    if split == 1:
        return KernelSource([src], preps + [step], scratch, "gemm", need, info)
    if fusek:
        info["fused_fold"] = True
        return KernelSource([src], [step], [split * tiles * BM * BN * 4, tiles * 4], "gemm", need, info, zeroed_scratch=[1])
    from .kernelgen import fold_stage

    ks2, steps2, partial_len = fold_stage(kernel, numerics, name, split, pitch, slice_major=True)
    info["stage2"] = ks2.info
    need.update({gid_: b_ for gid_, b_ in ks2.min_input_bytes.items() if gid_ != kernel.nargs})
    return KernelSource([src] + ks2.sources, preps + [step] + steps2, [partial_len * 4] + scratch, "gemm+fold", need, info)
