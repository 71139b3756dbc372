"""The on-chip solvers' launch shapes, shared memory and plans for each of the
four methods (fortranfvcell_amd/csrc/fvc_resplan.h), built for the CPU with
sanitizers."""
import os

from test_sanitize import HERE, _build_and_run


def test_resident_plans_of_every_method(tmp_path):
    out = _build_and_run(tmp_path, "g++", ["-std=c++17", os.path.join(HERE, "sanitize", "resplan_kinds.cpp")],
                         "resplan_kinds")
    assert " 0 failures" in out
