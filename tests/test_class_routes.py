"""The rules that choose a class's kernel, built for the host: no GPU needed."""
import ctypes
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("routes") / "libroutes.so")
    subprocess.run(["/opt/rocm/bin/hipcc", "-O1", "-std=c++17", "-fPIC", "-shared", "--offload-arch=gfx950",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-o", out,
                    os.path.join(ROOT, "tests", "class_routes_host.hip")], check=True, stderr=subprocess.DEVNULL)
    lib = ctypes.CDLL(out)
    lib.jk_runs_rys.argtypes = [ctypes.c_int] * 6 + [ctypes.c_longlong] + [ctypes.c_double] * 2
    return lib


def _rys(lib, cls, mixed, quartets, longest, heaviest):
    return bool(lib.jk_runs_rys(*(int(x) for x in cls), int(mixed), 0, quartets, longest, heaviest))


# shell quartets, primitive quartets of the longest work item and of the heaviest shell quartet
@pytest.mark.parametrize("cls,quartets,longest,heaviest,rys", [
    ("1111", 1, 81, 81, True),        # water, STO-3G
    ("1111", 55, 810, 81, False),     # C4H10, STO-3G: rows of ten kets of 81 primitive quartets each
    ("1111", 104, 1215, 81, False),   # (H2O)5, STO-3G
    ("1111", 55, 256, 256, True),     # water, cc-pVDZ
    ("1111", 20000, 81, 81, False),   # beyond latency, the shell quartets decide
    ("2110", 3600, 1072, 144, False),
    ("2011", 70, 144, 144, True),
    ("2111", 474, 176, 64, True),
    ("2210", 333, 232, 36, False),
])
def test_jk_low_l_by_its_longest_item(lib, cls, quartets, longest, heaviest, rys):
    assert _rys(lib, cls, False, quartets, longest, heaviest) == rys
    assert not _rys(lib, cls, True, quartets, longest, heaviest)  # mixed builds: from L = 7 only


@pytest.mark.parametrize("cls", ["2211", "2121", "2022", "2220", "2221", "2122", "2222"])
def test_jk_high_l_always(lib, cls):
    for work in ((1, 1, 1), (10 ** 7, 1e5, 1)):
        assert _rys(lib, cls, False, *work)
        assert _rys(lib, cls, True, *work) == (sum(map(int, cls)) >= 7)


@pytest.mark.parametrize("np", [0, 1, 2, 9, 81])
def test_gradient_slices_load_stored_primitives(lib, np):
    # a slice without primitives of its own loads one of the pair's, which stores one at least
    for k in range(100):
        assert lib.grad_first_prim(k, np) == (k if k < np else max(np - 1, 0))
