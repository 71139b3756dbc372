"""The row dealing of the on-chip solvers (fortranfvcell_amd/csrc/
fvc_resplan.h), which the device code shares, built for the CPU with
sanitizers and checked against what it promises."""
import os

from test_sanitize import HERE, _build_and_run


def test_resident_plans_sanitized(tmp_path):
    out = _build_and_run(tmp_path, "g++", ["-std=c++17", os.path.join(HERE, "sanitize", "resplan_checks.cpp")],
                         "resplan_checks")
    assert " 0 failures" in out
