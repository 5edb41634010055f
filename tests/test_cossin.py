"""cossin_turn (the phase factors of the steering and direct imagers) on the CPU, against
float64: no larger an error than the runtime's sincospif, which it stands for, has on the GPU
(5.212e-8 for the cosine and 5.209e-8 for the sine over 2^27 evenly spaced arguments)."""
import subprocess

import pytest

from test_host_memory import compile_host


@pytest.fixture(scope="module")
def errors(tmp_path_factory):
    exe = compile_host(str(tmp_path_factory.mktemp("cossin") / "cossin"), "cossin_harness.cpp")
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120, check=True).stdout
    print(out)
    return [float(x) for x in out.split()]


def test_error_bound(errors):
    assert errors[0] <= 5.212e-8


def test_small_arguments(errors):
    """The sine keeps its relative accuracy towards zero: half a unit in the last place of the
    last operation (6.0e-8) and the smaller terms before it, below one unit."""
    assert errors[1] <= 1.2e-7
