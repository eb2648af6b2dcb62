"""The Font fix's correctly rounded pow: its short method against the full-length one
on the host, bit for bit (the device evaluates the same IEEE operations)."""
import os
import subprocess
import tempfile

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_short_pow_gives_the_full_methods_bits():
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "pow_check")
        subprocess.run([HIPCC, "--offload-arch=gfx950", "-O2", "-ffp-contract=off", "-o", exe,
                        os.path.join(HERE, "pow_check.hip")], check=True, capture_output=True, cwd=d)
        out = subprocess.run([exe, "3000000"], check=False, capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout + out.stderr
    assert "checked 3000000 mismatches 0" in out.stdout
