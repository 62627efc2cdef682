"""Several dispatches of a program in one launch."""

from __future__ import annotations

from typing import List, Sequence, Tuple

from . import tuner
from .alu import Kernel
from .kernelgen import KernelSource, LaunchStep, _prelude, gen_maps


class Composite:
    """What the sources of such launches have in common: `inputs` (the caller's buffer ids, in parameter order) and the methods
    below.  A `Kernel` and a `Routine` are the other two kinds of source."""

    inputs: List[int]

    def key(self) -> tuple:
        raise NotImplementedError

    def output_bytes(self) -> List[int]:
        raise NotImplementedError

    def generate(self, numerics: str) -> KernelSource:
        raise NotImplementedError

    def extents(self) -> List[int]:
        """What a trace names the launch's size by."""
        raise NotImplementedError

    def label(self) -> Tuple[str, List[Tuple[str, str]]]:
        """Name and properties in a trace."""
        raise NotImplementedError


MAPS_MOST = 8  # Kernels in one launch


class Maps(Composite):
    """Elementwise Kernels that do not read each other's results, their workgroups one after the other in one launch.

    A launch costs about 2.2 us beside its work and ends with a chip that runs empty; programs leave such Kernels behind one
    another where they do the same to several arrays (the keys and values of an attention cache, the parameters of a
    model).  microseconds, apart -> in one: float32 x 0.9 + y 0.1 over 2 x 1000 10.9 -> 8.0, 8 x 10^5 33.5 -> 16.0, 4 x 2^20 20.5
    -> 11.8, 2 x 2^22 19.5 -> 17.6, 2 x 2^24 69.5 -> 67.8, 2 x 2^26 239 -> 239; 5 x 3000001 halves 28.3 -> 16.3; both halves of a
    1024-position cache extended by one 11.8 -> 9.9.  None of forty sizes was slower."""

    def __init__(self, kernels: Sequence[Kernel], inputs: Sequence[int]):
        self.kernels, self.inputs = list(kernels), list(inputs)

    def key(self) -> tuple:
        return ("maps", tuple(k.key() for k in self.kernels))

    def output_bytes(self) -> List[int]:
        return [k.bytes for k in self.kernels]

    def generate(self, numerics: str) -> KernelSource:
        return gen_maps(self.kernels, numerics)

    def extents(self) -> List[int]:
        return [sum(k.size for k in self.kernels)]

    def label(self):
        return "Maps", [("kernels", str(len(self.kernels))), ("size", str(sum(k.size for k in self.kernels)))]


def joins_maps(kernel) -> bool:
    """Whether `kernel` is a Kernel whose launch is a plain elementwise one."""
    return isinstance(kernel, Kernel) and kernel.reduction is None and kernel.size > 0 and tuner.tuneHip(kernel).klass == "map"


WEIGHTS_MOST = 16  # layouts in one launch


class Weights(Composite):
    """The weights of several Kernels, laid out by one launch at the front of a program instead of a launch before each of them
    (forward and both cotangents of 32 x 64 x 56 x 56 float16 by 64 x 64 x 3 x 3: 54.9 -> 53.1 us; each launch took 4.7 us of
    which the layout itself is a fraction)."""

    def __init__(self, kernels: Sequence[Kernel], sources: Sequence[KernelSource], inputs: Sequence[int]):
        self.kernels, self.early, self.inputs = list(kernels), [ks.early for ks in sources], list(inputs)
        self.need = [ks.min_input_bytes[ks.early.gid] for ks in sources]

    def key(self) -> tuple:
        return ("weights", tuple((k.key(), e.text) for k, e in zip(self.kernels, self.early)))

    def output_bytes(self) -> List[int]:
        return [e.bytes for e in self.early]

    def generate(self, numerics: str) -> KernelSource:
        params, lines, args, first = [], [], [], 0
        for k, e in enumerate(self.early):
            params += [f"const jh_f16* __restrict__ w{k}", f"jh_f16* __restrict__ wt{k}"]
            call = f"jh_{k}::jh_weights(w{k}, wt{k}, block{f' - {first}' if first else ''});"
            lines.append(f"  {'else ' if k else ''}{f'if (block < {first + e.blocks}) ' if k + 1 < len(self.early) else ''}{call}")
            args += [("in", k), ("out", k)]
            first += e.blocks
        src = _prelude(numerics) + "".join(e.text.replace("namespace jh_0 {", f"namespace jh_{k} {{", 1) for k, e in enumerate(self.early)) + (
            f"extern \"C\" __global__ __launch_bounds__(256) void jh_weights_of({', '.join(params)}) {{\n  const int block = (int)blockIdx.x;\n" + "\n".join(lines) + "\n}\n")
        return KernelSource([src], [LaunchStep("jh_weights_of", (first, 1, 1), (256, 1, 1), 0, args)], [], "weights", dict(enumerate(self.need)), dict(parts=len(self.early)))

    def extents(self) -> List[int]:
        return [sum(e.bytes for e in self.early) // 2]

    def label(self):
        return "Weights", [("kernels", str(len(self.early))), ("size", str(self.extents()[0]))]
