"""What the sorts' sources ask the compiler for.  Sources whose words are doubles are compiled for finite values only; the
elements, among which NaN and infinity are ordinary, must not be floating-point values to the compiler there."""
import re
import subprocess

import pytest

from jaxjs_hip import DType
from jaxjs_hip.kernelgen import _prelude
from jaxjs_hip.routine import Routine, Routines, RoutineType
from jaxjs_hip.routinegen import generateRoutine


def _source(op, dtype, shape):
    outs = [dtype] if op == Routines.Sort else [dtype, DType.Int32]
    return generateRoutine(Routine(op, RoutineType([shape], [dtype], [shape] * len(outs), outs)), "fast").sources[0]


@pytest.mark.parametrize("dtype", [DType.Float32, DType.Float16, DType.Int32, DType.Uint32, DType.Bool, DType.Float64], ids=lambda d: d.value)
@pytest.mark.parametrize("op", [Routines.Sort, Routines.Argsort], ids=lambda o: o.value)
@pytest.mark.parametrize("shape", [[4, 100], [3000, 300], [4, 5000], [2, 70000], [1, (1 << 20) + 1]], ids=str)
def test_a_sort_compiled_for_finite_values_has_no_element_in_a_floating_type(op, dtype, shape):
    source = _source(op, dtype, shape)
    if "-ffinite-math-only" not in source:
        return
    own = source[source.index(_prelude("fast")) + len(_prelude("fast")):]
    text = subprocess.run(["gcc", "-E", "-P", "-x", "c++", "-"], input=own, capture_output=True, text=True, check=True).stdout
    left = text.replace("__builtin_bit_cast(double, a)", "").replace("__builtin_bit_cast(double, b)", "")  # the words
    assert len(left) < len(text) and not re.findall(r"\b(?:float|double|jh_f16|_Float16)\b.*", left)


def test_the_option_is_asked_for_where_the_words_are_doubles():
    asked = lambda *a: "-ffinite-math-only" in _source(*a)  # noqa: E731
    assert asked(Routines.Argsort, DType.Float32, [4, 5000]) and asked(Routines.Argsort, DType.Int32, [2, 70000])
    assert not asked(Routines.Sort, DType.Float32, [4, 5000]) and not asked(Routines.Argsort, DType.Float16, [2, 70000])
    assert not asked(Routines.Argsort, DType.Float64, [4, 5000]) and not asked(Routines.Argsort, DType.Float32, [1, (1 << 20) + 1])
