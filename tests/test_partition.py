"""The partition of the resident solve on the CPU: every table that the kernel
reads, checked against the tets and colours it was made from."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CSRC = ROOT / "avbd_amd" / "csrc"
LDS = 160 * 1024 - 1024   # what a workgroup of an MI355X may use
CUS = 256


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    exe = tmp_path_factory.mktemp("partition") / "partition_check"
    subprocess.run([shutil.which("g++"), "-std=c++20", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{CSRC}", f"-I{ROOT / 'include'}", str(ROOT / "tests" / "native" / "partition_check.cpp"),
                    str(CSRC / "resident_host.cpp"), str(CSRC / "host_graph.cpp"), "-o", str(exe)], check=True)

    def run(*args):
        r = subprocess.run([str(exe), *map(str, args)], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
        return r.stdout.split()
    return run


def scenes(checker, cells, target=1000, real=4, damp=0, fixed=0, cus=CUS, lds=LDS):
    cells = cells if isinstance(cells, (list, tuple)) else [cells]
    return checker("scenes", ",".join(map(str, cells)), target, real, damp, fixed, cus, lds)


def even(n):   # the target of one cube of n cells
    return max(1000, -(-24 * n ** 3 // CUS))


# one tet patch, one patch, the first cut, ragged patches, patches that fill the LDS;
# a cut that does not fit and is refined (a small LDS); fixed particles
@pytest.mark.parametrize("cells,target,real,damp,fixed,lds", [
    (1, 1000, 4, 0, 0, LDS), (2, 1000, 8, 0, 1, LDS), (5, 1000, 4, 0, 0, LDS), (8, 200, 4, 0, 1, LDS),
    (6, 30, 8, 0, 1, LDS), (15, 1000, 8, 1, 0, LDS), (24, even(24), 4, 1, 0, LDS), (32, even(32), 8, 0, 0, LDS),
    (32, even(32), 4, 0, 0, LDS), (10, 10 ** 6, 8, 0, 0, 30000), ([3, 7, 1, 9, 4], 2000, 4, 0, 0, 40000)])
def test_every_table_of_the_partition(checker, cells, target, real, damp, fixed, lds):
    assert scenes(checker, cells, target, real, damp, fixed, lds=lds)[0] == "fits"


@pytest.mark.parametrize("cells", [14, 16])
def test_a_first_cut_beyond_16_bits_is_refined(checker, cells):
    """A batch of a thousand scenes aims at more incidences per patch than its
    16-bit offsets hold: such a cut is refined like one that overfills the LDS."""
    assert 24 * cells ** 3 > 0xFFFF
    out = scenes(checker, [cells, 5], target=10 ** 6)
    assert out[0] == "fits" and int(out[1]) > 2


def test_a_failed_allocation_comes_out_as_an_error(checker):
    assert checker("memory")[:2] == ["every", "failure"]
