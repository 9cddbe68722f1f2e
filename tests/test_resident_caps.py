"""The plan of the LDS-resident factorization at the capacities the kernels have
in each precision (taken from the header), executed on the CPU by
tests/cpp/resident_check.cpp: the FP64 top part holds 2527 slots."""
import os
import subprocess

import pytest

from mapol_amd import synth
from tests.test_resident import ROOT, check  # noqa: F401


@pytest.fixture(scope="module")
def caps(tmp_path_factory):
    d = tmp_path_factory.mktemp("caps")
    (d / "caps.cpp").write_text(
        '#include <cstdio>\n#include "resident.hpp"\nusing namespace bpf;\nint main() {\n'
        '  for (int s : {4, 8}) printf("%d %d ", resident_cap(RES_TOP_LDS, s), '
        'resident_cap(RES_SMALL_LDS, s));\n}\n')
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "mapol_amd", "csrc"),
                    str(d / "caps.cpp"), "-o", str(d / "caps")], check=True)
    v = [int(x) for x in subprocess.run([str(d / "caps")], capture_output=True,
                                        text=True).stdout.split()]
    return {"fp32": tuple(v[:2]), "fp64": tuple(v[2:])}


def test_capacities(caps):
    assert caps == {"fp32": (5055, 1021), "fp64": (2527, 510)}


@pytest.mark.parametrize("name,ordering,tail", [("pf118x200", 1, 8), ("pf1354x200", 0, 0),
                                                ("pf2869x100", 0, 40), ("pf9241x200", 0, 0)])
def test_fp64_plan_at_its_capacity(check, caps, name, ordering, tail):  # noqa: F811
    case, _ = synth.workload(name, T=2)
    check(case.bus_type, case.br_from, case.br_to, ordering, tail, caps["fp64"])

