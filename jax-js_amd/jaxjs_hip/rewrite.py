"""Rewrites of a traced program before it is scheduled on the `hip` backend.

`fuse_attention` recognises scaled-dot-product attention as the front-end composes it (src/library/nn.ts:478-583: two Dots
around scale, mask and softmax, seven Kernels over a [B, N, L, S] score tensor) and puts the backend's Attention routine in
its place, which keeps scores in registers and in float32 where the composition rounds them to float16 and moves them
through memory seven times.  Only what the routine computes: float16, head size 32, 64 or 128, no mask or the lower
triangle, and no part of the chain used by anything else; and only where the routine is the faster one
(`routine_is_faster`): it never splits the keys, which the composition spreads over the whole chip.
"""

from __future__ import annotations

from typing import Dict, List, Optional

import numpy as np

from .alu import AluOp, DType
from .jit import Atom, ConstArray, Jaxpr, JaxprEqn, Lit, ShapedArray, Var


class _Graph:
    def __init__(self, jaxpr: Jaxpr):
        self.made: Dict[Var, JaxprEqn] = {v: e for e in jaxpr.eqns for v in e.outBinders}
        self.uses: Dict[Var, int] = {}
        for e in jaxpr.eqns:
            for x in e.inputs:
                if isinstance(x, Var):
                    self.uses[x] = self.uses.get(x, 0) + 1
        for x in jaxpr.outs:
            if isinstance(x, Var):
                self.uses[x] = self.uses.get(x, 0) + 100  # kept whatever else happens to it

    def by(self, x: Atom, primitive: str, uses: int = 1) -> Optional[JaxprEqn]:
        """The equation that makes `x` when it is this primitive and `x` is read `uses` times in all."""
        e = self.made.get(x) if isinstance(x, Var) else None
        return e if e is not None and e.primitive == primitive and self.uses.get(x, 0) == uses else None

    def through(self, x: Atom, *primitives: str) -> Atom:
        """`x` behind any of these one-operand primitives, each read once."""
        while isinstance(x, Var) and x in self.made and self.made[x].primitive in primitives and self.uses.get(x, 0) == 1:
            x = self.made[x].inputs[0]
        return x


def _lower_triangle(x: Atom, jaxpr: Jaxpr, consts: List[ConstArray], L: int, S: int) -> bool:
    from .library import tri_const
    if not isinstance(x, Var) or x not in jaxpr.inBinders[:len(consts)]:
        return False
    c = consts[jaxpr.inBinders.index(x)]
    t = tri_const(L, S, 0)
    return tuple(c.shape) == tuple(t.shape) and c.dtype == t.dtype and c.exp.simplify() is t.exp.simplify()


def _match(g: _Graph, values: JaxprEqn, jaxpr: Jaxpr, consts: List[ConstArray]) -> Optional[dict]:
    """`values` is the Dot of the probabilities with the values: operands, scale and mask of the chain behind it."""
    p, z = values.inputs
    out = values.outBinders[0].aval
    if not isinstance(z, Var) or not isinstance(p, Var) or out.dtype != DType.Float16 or len(out.shape) != 4:
        return None
    B, N, L, H = out.shape
    if len(z.aval.shape) != 5 or len(p.aval.shape) != 5 or H not in (32, 64, 128):
        return None
    S = z.aval.shape[4]
    if tuple(p.aval.shape) != (B, N, L, 1, S) or tuple(z.aval.shape) != (B, N, 1, H, S) or S < 2 or B * N * L * S * H == 0:
        return None
    share = g.by(g.through(p, "Reshape"), "Mul")
    # Operands broadcast, and reshapes are looked through: a value per row has to be read as one, next to whole rows.
    rows, row = (B, N, L, S), (B, N, L, 1)
    if share is None or tuple(share.outBinders[0].aval.shape) != rows:
        return None
    for e, r in (share.inputs, share.inputs[::-1]):  # exp(...) times 1 / its sum
        inverse = g.by(r, "Reciprocal")
        exp = g.by(e, "Exp", uses=2)
        if inverse is not None and exp is not None and tuple(r.aval.shape) == row and tuple(e.aval.shape) == rows:
            break
    else:
        return None
    total = g.by(g.through(inverse.inputs[0], "Reshape"), "Reduce")
    if total is None or total.params["op"] != AluOp.Add or list(total.params["axis"]) != [3] or total.inputs[0] is not e:
        return None
    shifted = g.by(exp.inputs[0], "Add")
    if shifted is None:
        return None
    for scores, m in (shifted.inputs, shifted.inputs[::-1]):  # scores minus their maximum
        minus = g.by(m, "Neg")
        if minus is not None and tuple(m.aval.shape) == row and tuple(scores.aval.shape) == rows:
            break
    else:
        return None
    top = g.by(g.through(minus.inputs[0], "StopGradient", "Reshape"), "Reduce")
    if top is None or top.params["op"] != AluOp.Max or list(top.params["axis"]) != [3] or top.inputs[0] is not scores:
        return None
    causal, x = False, scores
    where = g.by(x, "Where", uses=2)
    if where is not None:
        mask, x, floor = where.inputs
        if tuple(x.aval.shape) != rows or not (isinstance(floor, Lit) and floor.value == -np.inf and _lower_triangle(mask, jaxpr, consts, L, S)):
            return None
        causal = True
    scale, reads = 1.0, 1 if causal else 2
    scaled = g.by(x, "Mul", uses=reads)
    if scaled is not None and any(isinstance(i, Lit) for i in scaled.inputs):
        lit = next(i for i in scaled.inputs if isinstance(i, Lit))
        x = next((i for i in scaled.inputs if not isinstance(i, Lit)), None)
        with np.errstate(over="ignore"):
            scale, reads = float(np.float16(lit.value)), 1
        if not np.isfinite(scale):  # the routine's source holds it as a number
            return None
    dot = g.by(x, "Dot", uses=reads)
    if dot is None or tuple(x.aval.shape) != rows:
        return None
    q, k = dot.inputs
    if not isinstance(q, Var) or not isinstance(k, Var) or tuple(q.aval.shape) != (B, N, L, 1, H) or tuple(k.aval.shape) != (B, N, 1, S, H):
        return None
    if any(v.aval.dtype != DType.Float16 for v in (q, k, z)):
        return None
    if not routine_is_faster(B, N, L, S, H, causal):
        return None
    return dict(q=q, k=k, z=z, B=B, N=N, L=L, S=S, H=H, scale=scale, causal=causal)


# Microseconds per key that a workgroup of the tile kernel walks, by head size (16384 keys: 162, 206 and 304 us).
_TILE_US_PER_KEY = {32: 0.0100, 64: 0.0126, 128: 0.0188}


def routine_is_faster(B: int, N: int, L: int, S: int, H: int, causal: bool) -> bool:
    """Whether the Attention routine beats the composition.  From both sides measured at B N = 1 .. 768, L = 1 .. 4096 and
    S = 128 .. 65536 in all head sizes: of 640 shapes the rule takes the slower side by more than a fifth at five (by 1.54
    at most, at S = 5001), where the routine everywhere would lose that much at 153, and up to 21 times.

    A workgroup per query reads keys and values at 100 GB/s, so 4096 keys of 64 take it 12 us and 65536 take 162, when the
    composition's launches and all CUs' reading take 14 and 33.  With many workgroups both are bound by reading the cache:
    from 50 million multiplications (in heads of 64) on the composition is level (384 heads x 3072 55.5 against 54.6 us).

    Workgroups of 128 rows, one to a CU at first, walk all keys they see (half of them on average under the mask).  The
    composition costs 10 us of launches and moves the scores several times: 1.8 us per million of them, and 3.2 where its
    products' tiles of 64 rows are partly empty (12 x 64 x 2048 x 64: 27.6 against 16.3 us; 12 x 512 x 2048: 28.4 against 36;
    96 x 128 x 4096: 54 against 106; 1 x 4096 x 4096, causal: 62 against 48).  Up to four queries it has no such tiles and
    reads the cache at 4.3 TB/s for two of them (192 x 2 x 2048 x 64: 28 against 30 us, 8192: 119 and 107; 4 x 8192: 118 and
    152; 384 x 4 x 1024: 23 and 36)."""
    from .routinegen import ATTENTION_FEW_QUERIES, attention_by_queries
    if attention_by_queries(B * N, L, H):
        return S * H <= 4096 * 64 and B * N * L * S * max(H, 64) <= 3 << 24
    tiles = B * N * -(-L // 128)
    walked = min(S, L) if causal else S
    routine = 2 + _TILE_US_PER_KEY[H] * walked * max(1.0, tiles * (0.6 if causal else 1.0) / 256)
    if L <= ATTENTION_FEW_QUERIES:
        return 1.1 * routine <= 12 + (0.6 + 0.2 * L) * 4 * B * N * S * H / 4.3e6
    return routine <= 10 + (3.2 if L <= 64 else 1.8) * B * N * max(L, 64) * S / 1e6


def fuse_attention(jaxpr: Jaxpr, consts: List[ConstArray]) -> Optional[Jaxpr]:
    """The program with every recognised attention as one routine, or None where there is none."""
    g = _Graph(jaxpr)
    found = {id(e): m for e in jaxpr.eqns if e.primitive == "Dot" for m in [_match(g, e, jaxpr, consts)] if m is not None}
    if not found:
        return None
    eqns: List[JaxprEqn] = []
    alias: Dict[Var, Var] = {}

    def view(x: Var, primitive: str, params: dict, shape) -> Var:
        v = Var(ShapedArray(tuple(shape), x.aval.dtype, x.aval.weak))
        eqns.append(JaxprEqn(primitive, [x], params, [v]))
        return v

    def heads_behind(x: Var, flat, perm) -> Var:
        """A Dot's operand without its broadcast axis, as [batch, position, head, size]."""
        x = view(alias.get(x, x), "Reshape", dict(shape=flat), flat)
        return view(x, "Transpose", dict(perm=perm), [flat[i] for i in perm])

    for source in jaxpr.eqns:
        m = found.get(id(source))
        e = JaxprEqn(source.primitive, [alias.get(x, x) if isinstance(x, Var) else x for x in source.inputs], source.params, source.outBinders)
        if m is not None:
            B, N, L, S, H = (m[i] for i in "BNLSH")
            q = heads_behind(m["q"], (B, N, L, H), [0, 2, 1, 3])
            k = heads_behind(m["k"], (B, N, S, H), [0, 2, 1, 3])
            v = heads_behind(m["z"], (B, N, H, S), [0, 3, 1, 2])
            out = Var(ShapedArray((B, L, N, H), DType.Float16, False))
            eqns.append(JaxprEqn("Attention", [q, k, v], dict(scale=m["scale"], isCausal=m["causal"]), [out]))
            # the front-end moves the heads behind the positions next: that is how the routine writes them
            readers = [r for r in jaxpr.eqns if e.outBinders[0] in r.inputs]
            if len(readers) == 1 and readers[0].primitive == "Transpose" and list(readers[0].params["perm"]) == [0, 2, 1, 3] and e.outBinders[0] not in jaxpr.outs:
                alias[readers[0].outBinders[0]] = out
            eqns.append(JaxprEqn("Transpose", [out], dict(perm=[0, 2, 1, 3]), e.outBinders))
            continue
        eqns.append(e)
    outs = [alias.get(x, x) if isinstance(x, Var) else x for x in jaxpr.outs]
    return Jaxpr(list(jaxpr.inBinders), eqns, outs).simplify()
