"""The reciprocals that the projection and the raster set-up rest on
(rcp_newton, rcp_any, rcp_normal in q-pso_amd/csrc/qpso_math.h) against the
correctly rounded division, for all 2^32 inputs on this device."""
import os
import subprocess

import pytest

import qpso

pytestmark = pytest.mark.gpu


def test_reciprocals_over_all_inputs():
    exe = os.path.join(qpso.HERE, "lib", "qpso_rcp_check")
    p = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert p.returncode == 0, p.stdout + p.stderr
    counts = dict((k, int(v)) for k, v in (line.split() for line in p.stdout.splitlines()))
    assert counts == {"newton_wrong": 0, "any_wrong": 0, "normal_wrong": 0, "division_wrong": 0, "normal_rejected": 0,
                      "other_accepted": 0}
