"""CPU checks of the one-launch external product's host arithmetic
(extprod_rows.hpp): the key rows it requests, and which calls run on it."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "concrete-fft_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("rows") / "extprod_rows")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC,
                    os.path.join(HERE, "native", "extprod_rows.cpp"), "-o", exe], check=True)
    return exe


def test_key_rows_stay_inside_the_key(program):
    """In every round of every shape, each row is requested at its own place,
    and a request past the last row stays inside the key."""
    seen, past = {}, 0
    out = subprocess.run([program], check=True, capture_output=True, text=True).stdout
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


# (N, k1, levels, base_log): batches on which each form measured faster, 256 CUs
FASTER = [
    ((2048, 2, 3, 8), [1, 100, 257, 1100], []),
    ((4096, 2, 2, 15), [1, 257, 512, 2200], []),
    ((4096, 2, 6, 6), [2, 16, 600], []),
    ((2048, 2, 2, 32), [1, 256, 257, 1100], []),
    ((4096, 4, 3, 8), [40, 600], [2, 4, 16]),
    ((4096, 4, 3, 11), [100, 257], [2, 8, 16]),
    ((4096, 4, 4, 10), [100, 260], [40]),
    ((4096, 4, 5, 6), [100, 260], [16, 50]),
    ((4096, 4, 6, 5), [200], [72]),
    ((4096, 3, 4, 10), [16, 40, 200, 357, 513], [1, 4, 8, 257, 297]),
    ((4096, 3, 4, 7), [1, 16, 257, 300], []),
    ((4096, 3, 2, 16), [1, 200, 256, 357, 513, 600], [257, 300, 337]),
    ((4096, 3, 1, 32), [1, 257, 300, 600], []),
    ((2048, 3, 1, 32), [1, 257, 512, 693, 1060], [533, 613, 673]),
    ((2048, 3, 1, 23), [1, 257, 600], []),
    ((2048, 3, 2, 16), [257, 600, 1100], []),
    ((1024, 3, 1, 32), [1, 600, 1385, 2049], [1070, 1160, 1250]),
    ((2048, 4, 5, 7), [40, 260], [2, 4, 8]),
    ((2048, 4, 5, 6), [1, 2, 40], []),
    ((2048, 4, 8, 3), [40], [24]),
]


def test_calls_run_on_the_faster_form(program):
    calls = [(shape, b, want) for shape, one, split in FASTER
             for bs, want in ((one, 1), (split, 0)) for b in bs]
    text = "".join("%d %d %d %d %d 256\n" % (s + (b,)) for s, b, _ in calls)
    out = subprocess.run([program, "rule"], input=text, check=True, capture_output=True,
                         text=True).stdout.split()
    wrong = [(s, b, want) for (s, b, want), got in zip(calls, out) if int(got) != want]
    assert len(out) == len(calls) and not wrong, wrong


def test_other_shapes_keep_the_split_form(program):
    shapes = [(512, 2, 3, 8), (8192, 2, 3, 8), (2048, 1, 3, 8), (2048, 5, 3, 8), (2048, 64, 1, 8)]
    text = "".join("%d %d %d %d 100 256\n" % s for s in shapes)
    out = subprocess.run([program, "rule"], input=text, check=True, capture_output=True,
                         text=True).stdout.split()
    assert out == ["0"] * len(shapes)
