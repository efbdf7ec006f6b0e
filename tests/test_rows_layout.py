"""Assembled row storage on the host: built from the sources, no GPU."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "opentelemac_amd", "csrc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("rows") / "check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC,
                    os.path.join(HERE, "rows_layout_check.cpp"),
                    os.path.join(CSRC, "layout.cpp"), os.path.join(CSRC, "rows_layout.cpp"),
                    "-rdynamic", "-lpthread", "-ldl", "-o", exe], check=True)
    return exe


# (max workgroups, block nodes, systems): ragged members before one whose rows
# have only entries of another workgroup's columns; 1, 2, 4 and 8 slabs
@pytest.mark.parametrize("args", [
    (256, 64, "100", "far2048"), (256, 1024, "100", "far2048"), (256, 64, "700", "far4096", "3"),
    (4, 64, "1300", "far4096"), (2, 1024, "100", "far4096"), (2, 64, "9000", "far8192"),
    (256, 1024, "1024"), (256, 1024, "1025"),
    # more workgroups than fit: narrow systems, wide ones, both
    (16, 64, *["9000"] * 20), (16, 64, *["30000"] * 9), (16, 64, "100", "80000", *["9000"] * 20),
    (16, 64, *["9000"] * 17, "131072", "100"),
])
def test_ids_stay_within_their_workgroup(check, args):
    out = subprocess.run([check, *map(str, args)], capture_output=True, text=True)
    assert out.stdout == "ok\n", (out.stdout, out.returncode)


def _run(check, fail, *args):
    out = subprocess.run([check, *args], capture_output=True, text=True,
                         env=dict(os.environ, CHECK_FAIL=fail))
    assert out.returncode == 0, (out.returncode, out.stdout, out.stderr)
    return out.stdout


MANY = ("256", "64", "60000", "far40960")  # enough workgroups for several threads


def test_rows_are_built_without_threads(check):
    assert _run(check, "threads", *MANY) == "ok\n"


def test_a_failed_allocation_reaches_the_caller(check):
    """In the caller's thread or in another, first and last ones among them."""
    got = [_run(check, f"memory={n}", *MANY) for n in (0, 1, 5, 20, 60, 200, 1000, 5000, 20000)]
    assert set(got) <= {"bad_alloc\n", "built\n"} and got[0] == "bad_alloc\n"
    assert got.count("bad_alloc\n") >= 6


@pytest.mark.parametrize("systems,group", [
    (["1024"] * 128, 1), (["131072"], 1), (["131073"], 2), (["262145"], 2), (["530000"], 4),
    # many small ones: no empty slabs for fewer workgroups, or hardly fewer
    (["100"] * 300, 1), (["1500"] * 300, 2), (["3000"] * 300, 4), (["9000"] * 60, 4),
    (["100"] * 300 + ["20000"] * 2, 1),
    # a system that needs them sets the group of all
    (["100"] * 300 + ["1050000"], 8),
])
def test_slabs_per_workgroup(check, systems, group):
    out = subprocess.run([check, "256", "1024", *systems], capture_output=True, text=True,
                         env=dict(os.environ, CHECK_PRINT="1"))
    assert out.stdout == f"{group}\n"


def test_halos_beyond_the_lds_are_refused(check):
    """Joined halves of 2 slabs need a halo of 2 slabs each; of 4, too much."""
    for n, want in (("far4096", "ok\n"), ("far8192", "no rows (0)\n")):
        assert subprocess.run([check, "2", "64", n], capture_output=True, text=True).stdout == want
