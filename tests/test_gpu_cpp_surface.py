"""The host backend's tensor surface from C++: a solver template written against that surface
only (tests/cpp/template_surface.cpp, built by __graft_entry__.build()) runs on HipVector /
HipCrsMatrix and agrees with the backend's fused ConjugateGradient. Solvers whose operator changes
between update and apply (tests/cpp/changed_operator.cpp)."""
import subprocess
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu

BIN = Path(__file__).resolve().parent / "cpp" / "template_surface"
CHANGED = BIN.with_name("changed_operator")


def test_templated_solver_on_hip_tensors():
    assert BIN.exists(), f"{BIN} not built (run __graft_entry__.build())"
    r = subprocess.run([str(BIN)], capture_output=True, text=True, timeout=120)
    print(r.stdout, r.stderr)
    assert r.returncode == 0 and r.stdout.strip().endswith("OK")


@pytest.mark.parametrize("check", ["mprgp_replanned", "sweep_values", "sweep_values_row_blocks", "multigrid_values",
                                   "bounds_mprgp", "bounds_pgs", "loop_in_loop"])
def test_solvers_whose_operator_or_surroundings_change(check):
    assert CHANGED.exists(), f"{CHANGED} not built (run __graft_entry__.build())"
    r = subprocess.run([str(CHANGED), check], capture_output=True, text=True, timeout=120)
    print(r.stdout, r.stderr)
    assert r.returncode == 0 and r.stdout.strip().endswith("OK")
