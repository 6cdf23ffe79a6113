"""The chunked line solve of the fused sweeps, from the tables the kernels read,
on the CPU over every line length, chunk length and end condition they take
(tests/cpp/test_chunk_solve.cpp)."""
import os
import subprocess

import pytest

EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "_bin", "test_chunk_solve")


def test_chunked_solve_matches_whole_line_recurrences():
    if not os.path.exists(EXE):
        pytest.fail(f"{EXE} is not built (run __graft_entry__.build())")
    r = subprocess.run([EXE], capture_output=True, text=True, timeout=300)
    print(r.stdout, r.stderr)
    assert r.returncode == 0
