"""A chain of Kernels over rows and a product of those rows, or whose result they are, in one launch (`gemm_few.hip.inc`).

A layer normalisation in front of a linear layer on a few tokens is a launch of a few microseconds whose result the
product's workgroups read at once.  Here each of them makes the rows it needs in LDS, while its first share of the matrix
is on its way: the same work many times over, but beside a wait that is there anyway, and a launch less.  layer normalisation
and a linear layer, microseconds in two launches -> in one: float16 8 x 768 x 2304 5.4 -> 4.0, 8 x 768 x 3072 6.7 -> 4.1, 64 x
512 x 1536 5.2 -> 3.6, 16 x 2048 x 2048 7.5 -> 5.6; float32 8 x 768 x 3072 6.6 -> 4.2, 64 x 1024 x 1000 8.2 -> 6.1, 8 x 2048 x
2048 9.3 -> 8.5; a decode step of a transformer block 38.0 -> 35.1.

`ProductRows` is the other way round: a softmax behind a narrow output layer works on the rows of a result of which a
workgroup holds whole rows, before they are stored.
"""

from __future__ import annotations

from typing import List, Optional, Sequence

from . import tuner
from .alu import AluOp, Kernel, byteWidth
from .composite import Composite
from .gemm import few_plan, gen_gemm
from .kernelgen import KernelSource
from .rowchain import RowChain, plan_rows, row_text
from .runtime import LAUNCH_ARGS
from .fewgen import chain_pitch, plan_whole_rows

ROWS_MOST = 64             # rows of the product: every 16 of them are made by all of its column tiles
ROWS_BYTES = 96 * 1024     # of a workgroup's rows: 12 x 2048 float32 9.5 -> 9.1 us, 16 x 2048 9.9 -> 10.0
LANE_ELEMENTS = 32         # of a row in a lane's registers
LDS_BYTES = 160 * 1024 - 256


class RowProduct(Composite):
    """`kernel`, whose operand `gid` is the one output of `chain`."""

    def __init__(self, chain: RowChain, kernel: Kernel, gid: int, inputs: Sequence[int]):
        self.chain, self.kernel, self.gid = chain, kernel, gid
        self.inputs = [b for i, b in enumerate(inputs[:kernel.nargs]) if i != gid] + list(chain.inputs)

    def key(self) -> tuple:
        return ("row product", self.chain.key(), self.kernel.key(), self.gid)

    def output_bytes(self) -> List[int]:
        return [self.kernel.bytes]

    def extents(self) -> List[int]:
        return [self.kernel.size, self.kernel.reduction.size]

    def label(self):
        return "RowProduct", [("kernels", str(len(self.chain.stages) + 1)), ("size", str(self.kernel.size))]

    def generate(self, numerics: str) -> KernelSource:
        t = tuner.tuneHip(self.kernel)
        p = few_plan(t)
        plan = lane_plan(self.chain, p["waves"], min(self.chain.R, 16 * p["MT"]))
        text = row_text(self.chain, plan, numerics, "row")
        j = self.chain.outputs[0]
        text.params = [q for q in text.params if not q.endswith(f" out{j}")]
        text.stages = text.stages.replace(f"(out{j} + put + c0,", "(&jh_short[0][0] + put + c0,")
        return gen_gemm(self.kernel, t, numerics, "jh_row_product", rows=text)


class ProductRows(Composite):
    """`kernel` and `chain`, whose input `local` is the kernel's result and nothing else's."""

    def __init__(self, kernel: Kernel, inputs: Sequence[int], chain: RowChain, local: int, few: dict):
        self.kernel, self.chain, self.local, self.few = kernel, chain, local, few
        self.inputs = list(inputs[:kernel.nargs]) + [b for k, b in enumerate(chain.inputs) if k != local]

    def key(self) -> tuple:
        return ("product rows", self.kernel.key(), self.chain.key(), self.local)

    def output_bytes(self) -> List[int]:
        return self.chain.output_bytes()

    def extents(self) -> List[int]:
        return [self.kernel.size, self.kernel.reduction.size]

    def label(self):
        return "ProductRows", [("kernels", str(len(self.chain.stages) + 1)), ("size", str(self.kernel.size))]

    def generate(self, numerics: str) -> KernelSource:
        t = tuner.tuneNullopt(self.kernel)
        t.klass, t.gemm = "gemm", tuner.match_gemm(self.kernel)
        p = self.few
        plan = lane_plan(self.chain, p["waves"], 16 * (p["MT"] if p["short"] == "a" else p["VN"]), 2)
        text = row_text(self.chain, plan, numerics, "row", self.local)
        # inputs of the chain are numbered through without the local one
        text.need = {k - (k > self.local): b for k, b in text.need.items()}
        return gen_gemm(self.kernel, t, numerics, "jh_product_rows", behind=text, few=p)


# Whole rows in a workgroup are few, wide tiles: taken up to this estimate, and where they come in rounds anyway by what they
# replace (`_rounds_pay`).  softmax behind a linear layer, rows x columns x k, microseconds in two launches -> in one: float32 16 x
# 2 x 64 5.8 -> 3.4, 64 x 10 x 256 5.5 -> 3.8, 64 x 10 x 1024 5.9 -> 4.3, 1024 x 46 x 256 5.4 -> 4.0; float16 1024 x 64 x 256 5.6 ->
# 4.0, 8192 x 10 x 1024 7.1 -> 5.4.  Past the line 64 x 46 x 1024 6.4 -> 8.6, float16 64 x 64 x 1024 5.6 -> 7.3.
BEHIND_US = 5.0


def _rounds_pay(kernel: Kernel, g: dict, p: dict, rows: int) -> bool:
    """Whether whole rows in two rounds of workgroups and more beat the product's own launch and the rows' behind it: always where
    the product alone is a dot product per element, and else by the tiles it would take, which read the operands once for all
    columns and are the better the fuller they are.

    Of 440 products of up to 360000 rows, 4 to 64 columns and k from 32 to 4096, time in one launch over time in two: dot products 0.03
    to 0.63; float32 up to 32 columns 0.06 to 1.0 (one 1.12; 70000 x 10 x 512 64 -> 27 us, 116672 x 32 x 416 77 -> 62), more columns 1.0
    to 1.64 (100000 x 64 x 1024 164 -> 207); float16 with a wide operand off the 16-byte grid, which tiles load element by element,
    0.4 to 1.04 (50000 x 33 x 2048 108 -> 65) unless the other one is off the 4-byte grid too (0.6 to 1.5), with the rows along memory
    and up to 24 columns 0.75 to 1.05, and otherwise 0.56 to 2.2 and 1.17 in the mean (95323 x 33 x 1727 95 -> 208)."""
    if kernel.size // g["N"] < 2 * tuner.CU_COUNT * rows:
        return False
    if not tuner.tuneHip(kernel).klass.startswith("gemm"):
        return True
    if byteWidth(g["dtype"]) == 4:
        return g["N"] <= 32
    s, w = p["short"], p["wide"]
    return not p["along_k"] and (g[w + "_sk"] % 8 != 0 and g[p["row"][s]] % 2 == 0 or s == "b" and g["N"] <= 24)


def join_behind(kernel: Kernel, inputs: Sequence[int], buffer: int, chain: RowChain) -> Optional[ProductRows]:
    """`kernel`, which writes `buffer`, in one launch with `chain`, the only reader of that result; or None."""
    if kernel.reduction is None or buffer not in chain.inputs or kernel.size != chain.R * chain.C:
        return None
    local = chain.inputs.index(buffer)
    for st in chain.stages:
        for n in st.exp.collect(lambda n: n.op == AluOp.GlobalIndex) + (st.epilogue.collect(lambda n: n.op == AluOp.GlobalIndex) if st.epilogue is not None else []):
            if st.refs[n.arg[0]] == ("in", local) and (id(n) not in st.full or n.dtype != kernel.dtype):
                return None
    g = tuner.match_gemm(kernel)
    if g is None or g["M"] != chain.R or g["N"] != chain.C or g["c_sn"] != 1 or g["c_sm"] != chain.C or g["gid_a"] == g["gid_b"]:
        return None
    p = plan_whole_rows(g)
    if p is None:
        return None
    rows = 16 * (p["MT"] if p["short"] == "a" else p["VN"])
    if p["us"] > BEHIND_US and not _rounds_pay(kernel, g, p, rows):
        return None
    lanes = lane_plan(chain, p["waves"], rows, 2)
    sums = p["waves"] * 16 * p["MT"] * (16 * p["VN"] + 1) * 4
    if lanes["iters"] * lanes["V"] > LANE_ELEMENTS or sums + rows * (chain.C + 16) * byteWidth(kernel.dtype) > LDS_BYTES:
        return None
    joined = ProductRows(kernel, inputs, chain, local, p)
    return joined if len(joined.inputs) + len(chain.outputs) <= LAUNCH_ARGS else None


def lane_plan(chain: RowChain, waves: int, rows: int, least: int = 16) -> dict:
    """Lanes of a row inside one wave, as many as let the workgroup make all its rows at once."""
    p = dict(plan_rows(chain))
    V, groups = p["V"], chain.C // p["V"]
    T = 64
    while T > least and (waves * 64 // T < rows or T >= 2 * groups):
        T //= 2
    iters = -(-groups // T)
    p.update(T=T, iters=iters, full=sum(1 for i in range(iters) if (i + 1) * T * V <= chain.C))
    return p


def join_rows(chain: RowChain, buffer: int, kernel: Kernel, inputs: Sequence[int]) -> Optional[RowProduct]:
    """`chain`, whose only stored result is `buffer`, in one launch with `kernel`, the only reader of that result; or None."""
    if kernel.reduction is None or len(chain.outputs) != 1 or chain.R > ROWS_MOST or chain.stages[chain.outputs[0]].kind != "map" or chain.outputs[0] != len(chain.stages) - 1:
        return None
    t = tuner.tuneHip(kernel)
    g = t.gemm
    p = few_plan(t) if t.klass.startswith("gemm") and not t.params.get("wgrad") else None
    if p is None:
        return None
    rows, eb = min(chain.R, 16 * p["MT"]), byteWidth(g["dtype"])
    lanes = lane_plan(chain, p["waves"], rows)
    lds = p["waves"] * 16 * p["MT"] * (16 * p["VN"] + 1) * 4 + 16 * p["MT"] * chain_pitch(g["K"], g["dtype"]) * eb
    if rows * chain.C * eb > ROWS_BYTES or lanes["iters"] * lanes["V"] > LANE_ELEMENTS or lds > LDS_BYTES:
        return None
    # Workgroups that wait for a place make their rows beside no other's wait: float32 2 x 1856 x 5739 16.7 -> 20.0 us, 8 x 1423 x 9152
    # 25.6 -> 29.3, float16 8 x 1728 x 9088 17.5 -> 18.8, all with one to a CU; where a CU holds two, 3 x 1664 x 11328 12.5 -> 11.8.
    count = -(-p["C"] // (16 * p["VN"])) * p["slices"] * -(-chain.R // (16 * p["MT"]))
    if count > tuner.CU_COUNT * min(LDS_BYTES // lds, 32 // p["waves"]):
        return None
    s = p["short"]
    gid = g["gid_" + s]
    dtype = chain.stages[chain.outputs[0]].kernel.dtype
    if inputs[gid] != buffer or any(b == buffer for i, b in enumerate(inputs[:kernel.nargs]) if i != gid) or g["gid_a"] == g["gid_b"] \
            or t.epilogue.collect(lambda n: n.op == AluOp.GlobalIndex and n.arg[0] == gid):
        return None
    if dtype != g["dtype"] or (p["R"], g["K"]) != (chain.R, chain.C) or g["batch"] or g[s + "_off"] or g[p["row"][s]] != chain.C:
        return None
    joined = RowProduct(chain, kernel, gid, inputs)
    return joined if len(joined.inputs) + (3 if p["slices"] > 1 else 1) <= LAUNCH_ARGS else None  # (slices have sums and counters)
