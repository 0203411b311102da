"""CPU check of the server's test for requests of one device batch that write
over each other's inputs (serve_overlap.hpp), against the definition."""
import os
import random
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "concrete-fft_amd", "csrc")


def test_outputs_over_other_inputs(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "serve_overlap")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC,
                    os.path.join(HERE, "native", "serve_overlap.cpp"), "-o", exe], check=True)
    L = 64
    cases = [
        [(0, 64), (128, 192)],           # buffers of their own
        [(0, 0), (64, 64), (128, 128)],  # each in place
        [(0, 64), (64, 128)],            # a chain
        [(64, 128), (0, 64)],
        [(0, 32), (256, 512)],           # over its own input, shifted
        [(0, 512), (0, 1024)],           # one input, two readers
        [(0, 0), (0, 1024)],             # ... and written by one of them
        [(0, 127), (64, 256)], [(0, 128), (64, 256)], [(0, 1), (64, 256)], [(0, 0), (64, 256)],
    ]
    rng = random.Random(5)
    for _ in range(2000):
        m, room = rng.randint(1, 12), rng.choice([8, 40, 400])
        cases.append([(8 * rng.randrange(room), 8 * rng.randrange(room)) for _ in range(m)])
    text = "".join("%d %d %s\n" % (L, len(c), " ".join("%d %d" % p for p in c)) for c in cases)
    got = subprocess.run([exe], input=text, check=True, capture_output=True, text=True).stdout.split()
    want = [any(abs(c[i][1] - c[j][0]) < L for i in range(len(c)) for j in range(len(c)) if i != j)
            for c in cases]
    assert [g == "1" for g in got] == want and 0 < sum(want) < len(want)
