"""The plan of the LDS-resident factorization, executed on the CPU
(tests/cpp/resident_check.cpp): the factors, the forward substitution and the
tail's Schur complement it gives equal a plain block elimination's, every
operand is final when it is read, and every part fits its capacity.  Grids
from 14 to 9241 buses, the capacities of both precisions and small ones (many
parts, three and more stages), both orderings, no and small dense tails, an
islanded grid with an isolated bus."""
import os
import subprocess

import numpy as np
import pytest

from mapol_amd import synth

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
FP32, FP64 = (5055, 1021), (2526, 510)     # slots of the last part, of the others


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("resident") / "resident_check")
    src = [os.path.join(ROOT, "tests", "cpp", "resident_check.cpp")] + [
        os.path.join(ROOT, "mapol_amd", "csrc", f) for f in ("symbolic.cpp", "resident.cpp")]
    subprocess.run(["g++", "-std=c++17", "-O2", *src, "-o", exe], check=True, capture_output=True)

    def run(types, f, t, ordering, tail, caps):
        text = (f"{len(types)} {len(f)} {ordering} {tail} {caps[0]} {caps[1]}\n"
                + " ".join(map(str, types)) + "\n"
                + "\n".join(f"{a} {b}" for a, b in zip(f, t)) + "\n")
        r = subprocess.run([exe], input=text, capture_output=True, text=True)
        assert r.returncode == 0, (r.stdout, r.stderr)
        stages, parts = r.stdout.split()[1], r.stdout.split()[3]
        return int(stages), int(parts)

    return run


@pytest.mark.parametrize("name,ordering,tail,caps,stages", [
    ("pf14", 0, 0, FP32, 1), ("pf14", 0, 1, (13, 13), None),
    ("pf118x200", 0, 0, FP32, 1), ("pf118x200", 1, 8, FP64, 1),
    ("pf118x200", 0, 8, (60, 40), None), ("pf118x200", 0, 1, (64, 24), None),
    ("pf1354x200", 0, 0, FP32, 2), ("pf1354x200", 1, 0, FP64, 2),
    ("pf1354x200", 0, 16, (400, 100), None),
    ("pf2869x100", 0, 0, FP32, 2), ("pf2869x100", 0, 40, FP64, None),
    ("pf9241x200", 0, 0, FP32, 2), ("pf9241x200", 1, 0, FP64, None)])
def test_plan_factors_like_a_plain_elimination(check, name, ordering, tail, caps, stages):
    case, _ = synth.workload(name, T=2)
    got, parts = check(case.bus_type, case.br_from, case.br_to, ordering, tail, caps)
    assert stages is None or got == stages
    assert parts >= got


def test_islands_and_an_isolated_bus(check):
    a, b = (synth.workload(n, T=2)[0] for n in ("pf118x200", "pf14"))
    types = np.r_[a.bus_type, b.bus_type, 1]
    f = np.r_[a.br_from, b.br_from + a.nbus]
    t = np.r_[a.br_to, b.br_to + a.nbus]
    for caps in (FP32, (60, 40)):
        check(types, f, t, 0, 0, caps)
