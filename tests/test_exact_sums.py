"""The rule by which the sampler takes double sums of floats for exact
(bitmamba.c_amd/csrc/bm_exact.h), compiled for the CPU: never a set whose sums
differ with their order, and not too careful to be of use."""
import os
import subprocess
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_exact_sums():
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "exact_sums")
        subprocess.run(["g++", "-O2", "-ffp-contract=off", "-std=c++17",
                        "-I" + os.path.join(ROOT, "bitmamba.c_amd", "csrc"),
                        os.path.join(ROOT, "tests", "csrc", "exact_sums.cpp"), "-o", exe], check=True)
        out = subprocess.run([exe], check=True, stdout=subprocess.PIPE, text=True, timeout=300).stdout
    lines = [[int(v) for v in line.split()] for line in out.splitlines()]
    kinds, limits = lines[:-1], lines[-1]
    assert len(kinds) == 6
    for sets, exact, bad in kinds:
        assert sets == 4000 and bad == 0, kinds
    # terms within a factor of 20 (a min_p cut), and of e^8: always exact
    assert kinds[0][1] == 4000 and kinds[5][1] == 4000, kinds
    # mixed spreads fall on both sides of the rule
    for k in (1, 2, 4):
        assert 0 < kinds[k][1] < 4000, kinds
    assert limits == [1, 0, 1, 1, 0]
