"""The rules that cut sweeps into work-groups (awflcloud_amd/csrc/awfl_cut.hpp),
built for the host with g++: what they may not exceed, over many sizes, and the
sizes at which the other choice was measured slower."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "native", "cut_test.cpp")


@pytest.fixture(scope="module")
def cuts(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("cut") / "cut_test")
    subprocess.run(["g++", "-O1", "-std=c++17", SRC, "-o", exe], check=True)

    def ask(lines):
        r = subprocess.run([exe], input="\n".join(lines) + "\n", capture_output=True, text=True, timeout=120, check=True)
        return [ln.split() for ln in r.stdout.splitlines()]
    return ask


def test_adjoint_groups_fit(cuts):
    asked = [(n, lines) for n in range(1, 769) for lines in (1, 100, 256, 257, 600, 5000, 100000)]
    for (n, lines), (m,) in zip(asked, cuts(["adj %d %d" % a for a in asked])):
        assert 1 <= int(m) <= 768 // n, (n, lines, m)        # lanes of a work-group; 20 doubles of LDS each


def test_adjoint_lines_of_five_waves_share_a_group(cuts):
    # one line of 257 to 384 cells to a group leaves a CU with five or six waves
    for n in (257, 289, 300, 320, 384):
        for lines in (257, 312, 1008, 6400):
            assert cuts(["adj %d %d" % (n, lines)]) == [["2"]]
        assert cuts(["adj %d 224" % n]) == [["1"]]
