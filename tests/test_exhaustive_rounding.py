"""The quantizers inside the decode GEMMs (gemm_common.h, gemm_token_quant.h) replace a division by one Markstein step on a shared reciprocal
and roundf by an addition and a truncation.  exhaustive_rounding.c runs both against the operators they replace, over every input."""
import os
import shutil
import subprocess

import pytest


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs a C compiler")
def test_every_quotient_and_every_rounding(tmp_path):
    source = os.path.join(os.path.dirname(os.path.abspath(__file__)), "exhaustive_rounding.c")
    program = str(tmp_path / "exhaustive_rounding")
    subprocess.run(["gcc", "-O3", "-march=native", "-std=c11", "-ffp-contract=off", "-fno-math-errno", "-fopenmp", "-o", program, source, "-lm"], check=True)
    out = subprocess.run([program], check=True, capture_output=True, text=True, timeout=600).stdout
    assert out.split() == ["0", "0", "0"], out
