"""Builds with an item length the list build cannot hold are refused: lengths 0 to
APO_ITEM_STEPS have a lane and a 64-entry histogram row each, and are compared
bit by bit, so the limit is a power of two below 64."""
import os
import subprocess

import pytest

from apocharmm_amd import build

pytestmark = pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="needs hipcc")


@pytest.mark.parametrize("steps,ok", [(16, True), (32, True), (64, False), (48, False)])
def test_item_steps(steps, ok):
    cmd = [build.HIPCC] + build.FLAGS + ["-DAPO_ITEM_STEPS=%d" % steps, "--cuda-device-only",
                                         "-fsyntax-only", "-x", "hip",
                                         os.path.join(build.CSRC, "nblist.hip")]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert (r.returncode == 0) == ok, r.stderr[-2000:]
    assert ok or "one lane per item length" in r.stderr
