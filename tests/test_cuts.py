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


def test_small_grids_without_colliding_pairs(cuts):
    # two groups of two waves on a CU share a SIMD: slower at each of these, by the
    # adjoint (cells of a line, lines) and by three tracers along x
    for n, lines in ((36, 636), (45, 650), (43, 585), (34, 864)):
        assert cuts(["adj %d %d" % (n, lines)]) == [["1"]]
    for grid in ((63, 5, 154), (34, 12, 72), (40, 30, 30)):
        assert cuts(["tracers 0 3 %d %d %d 3" % grid])[0][1] == "1"


def _check_tile(n, per, cut, lanes):
    cols, rows, nseg, seglen, threads, lds = (int(v) for v in cut)
    assert cols >= 1 and cols * rows <= threads <= lanes and threads % 64 == 0 and lds <= 160 * 1024
    assert nseg * seglen >= n and (nseg - 1) * seglen < n            # every segment has a cell
    # a segment holds its neighbours' end cells too, where the line has them
    assert rows >= (n if nseg == 1 else seglen + (1 if not per and nseg == 2 else 2))
    return cols, nseg


def test_tiles_fit(cuts):
    asked = [(d, n, nline, other, per, 0) for d in (0, 1, 2) for n in list(range(1, 600)) + [683, 700, 768, 1000, 1024, 1027, 1364]
             for nline, other in ((1, 1), (37, 5), (160, 64)) for per in (0, 1)]
    for a, cut in zip(asked, cuts(["tile %d %d %d %d %d %d" % a for a in asked])):
        _check_tile(a[1], a[4], cut, 512)


def test_lines_updated_in_place_are_whole(cuts):
    asked = [(0, n, nline, 5, per, 1) for n in range(1, 1025) for nline in (1, 160) for per in (0, 1)]
    for a, cut in zip(asked, cuts(["tile %d %d %d %d %d %d" % a for a in asked])):
        assert _check_tile(a[1], a[4], cut, 1024)[1] == 1


def test_long_x_lines_run_in_segments(cuts):
    # a group of nine waves or more was slower than the segments at each of these
    for n in (513, 560, 600, 640, 700, 800, 1000, 1024):
        for nline, other in ((48, 32), (160, 64)):
            (cut,) = cuts(["tile 0 %d %d %d 1 0" % (n, nline, other)])
            assert int(cut[2]) >= 2 and int(cut[4]) <= 256


def test_short_x_lines_fill_a_wave(cuts):
    for n, nline, other in ((8, 91, 9), (2, 100, 50), (6, 50, 6), (16, 40, 30), (20, 60, 60), (33, 40, 30)):
        (cut,) = cuts(["tile 0 %d %d %d 1 0" % (n, nline, other)])
        assert int(cut[0]) >= 64 // n


# bits, direction, ord, grid, the form that was measured faster
MEASURED = [
    (64, 2, 3, (1000, 160, 64), "walker"),
    (64, 2, 3, (600, 160, 64), "walker"),
    (64, 2, 3, (1101, 616, 6), "walker"),
    (64, 2, 3, (512, 256, 128), "walker"),
    (64, 2, 3, (512, 100, 60), "tile"),
    (64, 2, 3, (128, 128, 64), "tile"),
    (64, 2, 3, (64, 64, 32), "tile"),
    (64, 1, 3, (1000, 160, 64), "walker"),
    (64, 1, 3, (130, 96, 64), "tile"),
    (64, 1, 3, (541, 2, 340), "walker"),
    (64, 2, 5, (256, 256, 128), "walker"),
    (64, 2, 5, (96, 300, 200), "tile"),
    (32, 2, 3, (600, 160, 64), "walker"),
    (32, 2, 3, (192, 192, 96), "walker"),
    (64, 2, 3, (332, 317, 5), "walker"),
    (64, 2, 3, (1214, 40, 75), "walker"),
    (32, 2, 3, (518, 102, 66), "walker"),
    (32, 2, 3, (795, 186, 30), "walker"),
    (32, 1, 3, (760, 22, 216), "walker"),
    (32, 2, 3, (100, 90, 75), "tile"),
    (32, 2, 3, (128, 128, 64), "tile"),
    (32, 1, 3, (512, 100, 60), "walker"),
    (32, 2, 5, (512, 512, 256), "walker"),
    (32, 2, 5, (128, 128, 64), "tile"),
]


@pytest.mark.parametrize("bits,d,ord,grid,form", MEASURED)
def test_form_is_the_one_measured_faster(cuts, bits, d, ord, grid, form):
    assert cuts(["form %d %d %d %d %d %d %d" % ((bits, d, ord) + grid + (int(d < 2),))]) == [[form]]


def test_tracer_tiles_fit(cuts):
    asked = [(d, o, nx, ny, nz, ntr) for d in (0, 1, 2) for o in (3, 5) for ntr in (0, 1, 3, 8)
             for nx, ny, nz in ((1, 1, 1), (7, 5, 6), (63, 65, 64), (1024, 2, 3), (2, 1025, 9), (3, 4, 700), (300, 200, 100))]
    for a, (form, cols, lds) in zip(asked, cuts(["tracers %d %d %d %d %d %d" % a for a in asked])):
        n = a[2 + a[0]]
        assert form == "tile" or a[0] == 0 or n >= 8          # shorter lines have no walker
        assert int(cols) * n <= 1024 and (form == "walker" or int(lds) <= 160 * 1024)


# direction, ord, grid, tracers, the form that was measured faster
@pytest.mark.parametrize("d,ord,grid,ntr,form", [
    (1, 3, (39, 456, 215), 1, "walker"),
    (1, 3, (92, 449, 80), 3, "walker"),
    (1, 3, (59, 189, 181), 3, "walker"),
    (1, 3, (156, 228, 160), 2, "walker"),
    (1, 3, (288, 237, 52), 2, "walker"),
    (1, 3, (66, 210, 76), 3, "tile"),
    (1, 3, (224, 134, 62), 2, "tile"),
    (1, 3, (237, 147, 116), 5, "tile"),
    (1, 3, (170, 249, 7), 2, "tile"),
    (1, 3, (17, 520, 10), 5, "tile"),
    (2, 3, (57, 6, 388), 8, "tile"),
    (2, 3, (51, 11, 367), 1, "tile"),
    (1, 5, (256, 256, 128), 3, "tile"),
    (2, 5, (256, 256, 128), 3, "tile"),
    (1, 5, (155, 287, 109), 3, "walker"),
    (2, 5, (778, 23, 267), 3, "walker"),
])
def test_tracer_form_is_the_one_measured_faster(cuts, d, ord, grid, ntr, form):
    assert cuts(["tracers %d %d %d %d %d %d" % ((d, ord) + grid + (ntr,))])[0][0] == form
