"""The MFMA product's slots of small V-stack units (acoustic_reliefs_amd/csrc/lr_units.h), compiled for the host, at every
number of wavefronts per workgroup that the product can be built with: no two units share a slot, none lies past the
slots that the list is made with, those are whole workgroups, and a workgroup has up to four units."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "acoustic_reliefs_amd", "csrc")

SRC = r'''
#include "lr_units.h"
extern "C" int slot(int n, int waves) { return (int)arh::lr_slot(n, waves); }
extern "C" int slots(int n, int waves) { return (int)arh::lr_slots(n, waves); }
'''


@pytest.fixture(scope="module")
def units(tmp_path_factory):
    d = tmp_path_factory.mktemp("units")
    (d / "u.cpp").write_text(SRC)
    subprocess.run(["g++", "-shared", "-fPIC", "-std=c++17", "-I" + CSRC, str(d / "u.cpp"), "-o", str(d / "u.so")],
                   check=True)
    return ctypes.CDLL(str(d / "u.so"))


@pytest.mark.parametrize("waves", [1, 2, 4, 8, 16])
def test_slots(units, waves):
    per = min(4, waves)
    for n in range(0, 40):
        total = units.slots(n, waves)
        got = [units.slot(u, waves) for u in range(n)]
        assert len(set(got)) == n and total % waves == 0
        assert not got or (min(got) >= 0 and max(got) < total)
        groups = [s // waves for s in got]
        assert all(groups.count(q) <= per for q in set(groups)) and total // waves == (n + per - 1) // per
        assert all(s % waves < per for s in got)
