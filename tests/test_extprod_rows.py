"""CPU check of the key rows the one-launch external product requests
(extprod_rows.hpp): in every round of every shape it takes, each row is
requested at its own place, and a request past the last row stays inside the
key."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "concrete-fft_amd", "csrc")


def test_key_rows_stay_inside_the_key(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "extprod_rows")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC,
                    os.path.join(HERE, "native", "extprod_rows.cpp"), "-o", exe], check=True)
    seen, past = {}, 0
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout
    for line in out.splitlines():
        log2n, k1, glwes, levels, r0, rr, i, rows, row = map(int, line.split())
        assert 0 <= row < rows, line
        if r0 + rr + i < rows:
            assert row == r0 + rr + i, line
            seen.setdefault((log2n, k1, glwes, levels), set()).add(row)
        else:
            past += 1
    assert past > 0
    for (log2n, k1, glwes, levels), rows in seen.items():
        assert rows == set(range(k1 * levels)), (log2n, k1, glwes, levels)
