"""The kernels' reciprocal (v_rcp_f32 and one Newton step) is the correctly
rounded 1/x wherever its residual is accepted: every significand, whole
numbers, and denormals (tests/cpp/recip_test.hip)."""
import subprocess
from pathlib import Path

import pytest

EXE = Path(__file__).resolve().parents[1] / "cu-reconstruction_amd" / "lib" / "recip_test"


@pytest.mark.gpu
def test_reciprocal_equals_division(cuda):
    r = subprocess.run([str(EXE)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "significands 0 whole 0 denormal 0" in r.stdout
