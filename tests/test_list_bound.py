"""The source lists of the sweeps take room for a bound of their entries: per
element of level l at most l + 1 sources up to its own level among nested cells,
2 l + 1 among touching ones, and as many pairs as the finer of the two, less
itself.  Here the pairs are counted from the tables themselves on a full fiber,
and all of them lie in the relation that the sweep-by-sweep form walks."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "adaptive-multiresolution-dg_amd", "csrc")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("lists") / "list_pairs.so")
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-shared", "-fPIC", "-ffp-contract=off", "-pthread", "-o", so,
                           os.path.join(HERE, "helpers", "list_pairs.cpp"), os.path.join(CSRC, "setup.cpp")])
    return ctypes.CDLL(so)


@pytest.mark.parametrize("k", [1, 2, 3])
@pytest.mark.parametrize("table,family,m", [(0, 0, 1), (0, 0, 2), (0, 0, 3), (0, 0, 4), (0, 1, 3), (1, 0, 1), (1, 0, 2),
                                            (1, 0, 3), (1, 0, 4), (1, 1, 3), (2, 0, 3)])
@pytest.mark.parametrize("n", [1, 4, 6])
def test_entries_stay_in_their_room(lib, table, family, k, m, n):
    out = (ctypes.c_long * (n + 3))()
    cells = lib.list_pairs(table, family, k, m, n, out)
    assert out[0] == 0, "pairs outside the relation"
    for level in range(n + 1):
        assert 1 <= out[1 + level] <= (level + 1 if table == 0 else 2 * level + 1), level
    assert out[n + 2] <= cells * (2 * n + 1 if table == 0 else 4 * n + 1)
