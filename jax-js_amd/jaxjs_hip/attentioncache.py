"""Attention of one new position over a cache that the same program extends by it.

A decoding step appends the position's keys and values to their caches (`concatenate`, src/library/numpy.ts: two padded views added up)
and attends to the result.  As dispatches that is a copy of both caches, which reads and writes them once, and an attention
that reads them again; in one launch every cached row is read once, scored, and written on the way."""

from __future__ import annotations

from typing import Dict, List, Optional, Sequence, Tuple

from .alu import AluOp, AluVar, DType, Kernel
from .composite import Composite, Maps
from .kernelgen import KernelSource, _min_bytes
from .routine import Routine, Routines
from .shape import unravelAlu
from .tuner import tuneHip


class Appended:
    """Keys (or values) [B, S, N, H] as a sum of two padded views: positions below `first` of one array, the others of another."""

    def __init__(self, first: int, parts: Sequence[Tuple[int, int, Tuple[int, ...]]], need: Dict[int, int]):
        self.first = first
        self.gids = [gid for gid, _, _ in parts]
        self.parts = [(offset, strides) for _, offset, strides in parts]
        self.need = [need[gid] for gid in self.gids]

    def fields(self, name: str) -> Dict[str, int]:
        """What the template calls them."""
        out = {}
        for tag, (offset, (sb, sp, sn, _)) in zip((name, name + "1"), self.parts):
            out.update({tag + "B": sb, tag + "S": sp, tag + "N": sn, tag + "OFF": offset})
        return out


def match_appended(kernel: Kernel, shape: Sequence[int]) -> Optional[Appended]:
    """`kernel` as an array of `shape` put together along its axis 1, if rows along the last axis are whole and aligned ones."""
    e = kernel.exp
    if kernel.reduction is not None or kernel.dtype != DType.Float16 or e.op != AluOp.Add or any(s.op != AluOp.GlobalView or s.dtype != DType.Float16 for s in e.src):
        return None
    walk = [u.simplify() for u in unravelAlu(list(shape), AluVar.gidx)]
    parts = []
    for s in e.src:
        st = s.arg[1]
        v = st.views[0]
        if len(st.views) != 1 or list(v.shape) != list(shape) or v.mask is None or [u.simplify() for u in s.src] != walk:
            return None
        if any(m != (0, n) for k, (m, n) in enumerate(zip(v.mask, shape)) if k != 1):
            return None
        sb, sp, sn, sh = v.strides
        lo, hi = v.mask[1]
        if sh != 1 or min(sb, sp, sn) < 0 or sb % 8 or sp % 8 or sn % 8 or v.offset % 8 or v.offset + lo * sp < 0:
            return None
        parts.append((lo, hi, (s.arg[0], v.offset, v.strides)))
    parts.sort(key=lambda p: p[0])
    (lo0, hi0, first), (lo1, hi1, second) = parts
    if lo0 != 0 or hi0 != lo1 or hi1 != shape[1] or not 0 < hi0 < hi1:
        return None
    return Appended(hi0, [first, second], _min_bytes(tuneHip(kernel).exp))


class CachedAttention(Composite):
    """`attention` over keys and values that `kernels` put together, which it writes as well: outputs are its result, keys, values."""

    def __init__(self, attention: Routine, kernels: Sequence[Kernel], appended: Sequence[Appended], inputs: Sequence[int]):
        self.attention, self.kernels, self.appended, self.inputs = attention, list(kernels), list(appended), list(inputs)

    def key(self) -> tuple:
        from .backend import routineKey
        return ("cached attention", routineKey(self.attention), tuple(k.key() for k in self.kernels))

    def output_bytes(self) -> List[int]:
        B, L, N, H = self.attention.type.outputShapes[0]
        return [B * L * N * H * 2] + [k.bytes for k in self.kernels]

    def generate(self, numerics: str) -> KernelSource:
        from .routinegen import _gen_attention
        return _gen_attention(self.attention, numerics, self.appended)

    def extents(self) -> List[int]:
        return [k.size for k in self.kernels]

    def label(self):
        return "CachedAttention", [("kernels", "3"), ("size", str(self.extents()[0]))]


def join_cache(maps: Maps, outputs: Sequence[int], routine: Routine, inputs: Sequence[int]) -> Optional[Tuple[CachedAttention, List[int]]]:
    """The Attention `routine` (reading `inputs`) with the two Kernels of `maps` (which write `outputs`) that make its keys and values, and
    where they stand in `maps`; or None."""
    from .routinegen import attention_by_queries
    if routine.name != Routines.Attention or inputs[1] == inputs[2] or inputs[1] not in outputs or inputs[2] not in outputs or inputs[0] in (inputs[1], inputs[2]):
        return None
    (B, L, N, H), shape, _ = routine.type.inputShapes
    if L != 1 or not attention_by_queries(B * N, L, H):
        return None
    S = shape[1]
    whole = [S * N * H, N * H, H, 1]
    views = list((routine.params or {}).get("views") or [None, None, None])
    if any(v is not None and (v["offset"] or any(n > 1 and a != b for n, a, b in zip(shape, v["strides"], whole))) for v in views[1:]):
        return None
    at = [outputs.index(i) for i in inputs[1:3]]
    kernels = [maps.kernels[k] for k in at]
    appended = [match_appended(k, shape) for k in kernels]
    if any(a is None for a in appended) or appended[0].first != appended[1].first:
        return None
    ids = [inputs[0]]
    for k, a in zip(at, appended):
        first = sum(m.nargs for m in maps.kernels[:k])
        ids += [maps.inputs[first + g] for g in a.gids]
    ids[2], ids[3] = ids[3], ids[2]  # q, both caches, both new parts
    return CachedAttention(routine, kernels, appended, ids), at
