"""The reference build without the reference: an absent or empty checkout
builds nothing and is no error, so that the library's own build goes on."""
import os
import subprocess
import sys

import pytest

SCRIPT = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle", "build_ref.py")


@pytest.mark.parametrize("exists", [False, True])
def test_no_reference_is_no_error(tmp_path, exists):
    ref = tmp_path / "reference"
    if exists:
        ref.mkdir()
    r = subprocess.run([sys.executable, SCRIPT, "--ref", str(ref)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    assert "nothing to build" in r.stdout
