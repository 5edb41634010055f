"""The tables of the spreading kernel's Fourier transform on the CPU: no larger an error against
long double than the sum with a cosine per node and entry has."""
import subprocess

from test_host_memory import compile_host


def test_table_errors(tmp_path):
    exe = compile_host(str(tmp_path / "es_ft"), "es_ft_harness.cpp")
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120, check=True).stdout
    print(out)
    table, plain = ([float(x) for x in line.split()] for line in out.splitlines())
    assert all(t <= p for t, p in zip(table, plain))
