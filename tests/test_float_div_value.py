"""div_const2 (csrc/common.h) tests only its result for the cases that take a
true division; this runs the exhaustive proof (tests/float_div_value.c) that a
result that is neither NaN nor subnormal is the IEEE quotient."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("d", [60, 12])
def test_result_equals_ieee_division_unless_nan_or_subnormal(tmp_path, d):
    cc = shutil.which("gcc")
    if cc is None:
        pytest.skip("gcc not found")
    exe = str(tmp_path / "float_div_value")
    subprocess.run([cc, "-O2", "-mfma", "-ffp-contract=off", "-o", exe, os.path.join(HERE, "float_div_value.c"),
                    "-lpthread", "-lm"], check=True)
    r = subprocess.run([exe, str(d)], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stdout
    assert int(r.stdout.split("fast-path inputs")[1].split()[0]) > 4_000_000_000
