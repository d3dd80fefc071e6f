"""near_sqrt and near_rcp (fluids3_amd/csrc/fx_near.hpp) against sqrtf and the division, at every float of their range."""
import json
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu

CHECK = os.path.join(os.path.dirname(os.path.abspath(__file__)), "near", "near")


def test_every_float_of_the_range():
    if not os.path.exists(CHECK):
        raise RuntimeError("tests/near/near is not built (run __graft_entry__.build())")
    r = subprocess.run([CHECK], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    got = json.loads(r.stdout.strip().splitlines()[-1])
    assert got == {"inside": 2 ** 30, "bad_sqrt": 0, "bad_rcp": 0}
