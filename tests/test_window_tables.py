"""The tables of places of the several-steps launch (CPU only): every window's
table has entries of its own, also past 2^32 of them (a FP16 ensemble of some
7,300 400x100 cylinders, 16 windows of 64x64 cells each)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
pytestmark = pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include"),
                                reason="g++ or the HIP headers not available")


@pytest.fixture(scope="module")
def tool(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("place") / "place_check")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-isystem", "/opt/rocm/include",
                    "-I", os.path.join(ROOT, "imexlb-1.0_amd", "csrc"),
                    os.path.join(ROOT, "tests", "sanitize", "place_check.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("cells", [256, 512, 1024, 2048, 4096])
def test_tables_do_not_overlap(tool, cells):
    wrap = 2 ** 32 // (9 * cells)  # the first table that ends past 2^32
    tables = [0, 1, wrap - 1, wrap, wrap + 1, 2 * wrap + 1, 2 ** 31 - 1]
    out = subprocess.run([tool, str(cells), *map(str, tables)], capture_output=True, text=True, check=True).stdout
    for t, line in zip(tables, out.splitlines(), strict=True):
        assert [int(v) for v in line.split()] == [t * 9 * cells, (t + 1) * 9 * cells - 1], t


def test_runs_of_several_steps_per_launch(tmp_path):
    """Launches of odd numbers of steps, the last of enough, a single step left;
    no steps at all where the run is too short."""
    exe = str(tmp_path / "multi_run_check")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-isystem", "/opt/rocm/include",
                    "-I", os.path.join(ROOT, "imexlb-1.0_amd", "csrc"),
                    os.path.join(ROOT, "tests", "sanitize", "multi_run_check.cpp"), "-o", exe,
                    "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib"], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, check=True).stdout.splitlines()
    assert len(out) == 4 * 2 * 2 * 400
    for line in out:
        halo, least, first, n, full, last, done = map(int, line.split())
        assert done == full * halo + last
        if done == 0:
            assert last == full == 0 and (n < first or n - 1 < max(least, 3) or (n - 1) < halo), line
            continue
        assert n >= first and done <= n - 1 and last % 2 == 1 and (last >= least or last == halo), line
        assert n - 1 - done < max(least, 3) + 1, line  # nothing left that a launch would have taken


def test_kernels_index_through_the_table_base():
    """Both kernels and both allocations take the table's place from there."""
    src = os.path.join(ROOT, "imexlb-1.0_amd", "csrc")
    text = {f: open(os.path.join(src, f)).read() for f in ("lbm_kernels.hip", "capi.cpp", "batch.cpp")}
    assert [text[f].count("place_base(") for f in text] == [2, 1, 1]
