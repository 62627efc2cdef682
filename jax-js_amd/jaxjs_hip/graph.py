"""A compiled jit program captured into a HIP graph.

`JitProgram.execute` (src/frontend/jit.ts:111-162) is a fixed list of kernel dispatches over buffers whose
sizes are known at compile time.  `GraphedProgram` allocates every intermediate and output once, records the
dispatches into one graph (`jh_graph_begin/end`) and replays them with a single `jh_graph_launch`: no host
work per kernel, no allocator traffic per call.  Inputs are bound at capture time: write new data into the
same input slots (or capture again) to run on other values.
"""

from __future__ import annotations

from typing import Dict, List, Sequence

from .errors import DeviceMemoryError
from .jit import JitProgram


class GraphedProgram:
    def __init__(self, backend, prog: JitProgram, inputs: Sequence[int]):
        if len(inputs) != prog.nargs:
            raise ValueError(f"jit program takes {prog.nargs} inputs, got {len(inputs)}")
        self.backend, self.prog = backend, prog
        self._slots: Dict[int, int] = {i: s for i, s in enumerate(inputs)}
        self._owned: List[int] = []
        # The units of the program's schedule, compiled and loaded before any capture; a routine is several launches and
        # outputs, recorded the same way.
        schedule = backend.scheduleProgram(prog)
        try:
            self._make_room(schedule)
        except DeviceMemoryError:
            if not schedule.laid_out:
                raise
            schedule = schedule.without_layouts()
            self._make_room(schedule)
        for s in inputs:
            backend.incRef(s)
            self._owned.append(s)
        prog, units = schedule.prog, schedule.units
        # The graph launches these executables' code objects and writes their scratch buffers without going through
        # dispatch: pin them so that neither cache eviction nor clearCache() can release them under a replay.
        self._exes = []
        for u in units:
            backend.pin(u.exe)
            self._exes.append(u.exe)

        def issue():
            for u in units:
                backend.dispatch(u.exe, [self._slots[i] for i in u.inputs], [self._slots[o] for o in u.outputs])

        issue()  # one eager pass: every code object is resident before the capture starts
        backend.dev.sync()
        self._graph = None
        trace, backend.trace = backend.trace, None  # event records are not part of the graph
        backend.capturing = True                    # nor is the profiler hook's event pair (it synchronises)
        try:
            backend.dev.graph_begin()
            try:
                issue()
            finally:
                self._graph = backend.dev.graph_end()
        finally:
            backend.trace, backend.capturing = trace, False
        self.outputs = [self._slots[o] for o in prog.outputs]
        self.kernels = len(units)

    def _make_room(self, schedule) -> None:
        """A slot for every buffer that the schedule's units write."""
        made: Dict[int, int] = {}
        try:
            for u in schedule.units:
                for o in u.outputs:
                    made[o] = self.backend.malloc(schedule.size_of(o))
        except BaseException:
            for s in made.values():
                self.backend.decRef(s)
            raise
        self._slots.update(made)
        self._owned.extend(made.values())

    def launch(self) -> None:
        """Queue one replay of the whole program (asynchronous, in order with everything else)."""
        if self._graph is None:
            raise ValueError("the graphed program was closed")
        if any(exe.data.released for exe in self._exes):
            raise ValueError("an executable of this graph was released: capture the program again")
        self.backend.dev.graph_launch(self._graph)

    def close(self) -> None:
        if self._graph is not None:
            self.backend.dev.sync()
            self.backend.dev.graph_destroy(self._graph)
            self._graph = None
            for exe in self._exes:
                self.backend.unpin(exe)
            self._exes = []
            for s in self._owned:
                self.backend.decRef(s)
            self._owned = []
