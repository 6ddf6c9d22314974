"""The split of a gated batch into runs, compiled for the host: every instance in exactly one run, no
empty run, runs of at most eight and the first of at most four, for any number of them."""

import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def split(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("runs") / "gated_runs")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-o", exe,
                    os.path.join(HERE, "cpp", "gated_runs.cpp")], check=True)

    def run(n, width):
        out = subprocess.run([exe, str(n), str(width)], capture_output=True, text=True, timeout=60)
        assert out.returncode == 0, out.stderr
        return [int(v) for v in out.stdout.split(":")[1].split()]
    return run


# Runs of one (neighbours that cannot share a launch) and of eight, either side of 62 runs, and the
# largest batches (64 beams of 32 coarse channels).
@pytest.mark.parametrize("width", [1, 3, 8])
@pytest.mark.parametrize("n", [1, 4, 5, 12, 13, 62, 63, 64, 65, 492, 493, 2048, 4096])
def test_every_instance_in_one_run(split, n, width):
    runs = split(n, width)
    want, left = [], n
    while left:
        want.append(min(width, left, 8 if want else 4))
        left -= want[-1]
    assert runs == want
