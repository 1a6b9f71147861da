"""TG_GEMM=vector, the products without the matrix cores, on the projection and contraction
tests of test_gpu_parity.py in a child process (the variable is read once).  It covers the
contraction as well: TG_GROUPED_VARIANT=99 names no tile, which only the matrix-core
contraction refuses."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
KEY = "test_projection_matches_reference or test_fields or test_gradient_matches_reference"


@pytest.mark.parametrize("variant,passes", [("", True), ("vector", True), ("mfma", False)])
def test_parity_with_vector_products(variant, passes):
    env = {k: v for k, v in os.environ.items() if k not in ("TG_GEMM", "TG_GROUPED_VARIANT")}
    if variant:
        env.update(TG_GEMM=variant, TG_GROUPED_VARIANT="99")
    print("TG_GEMM", variant, flush=True)
    cmd = [sys.executable, "-m", "pytest", os.path.join(HERE, "test_gpu_parity.py"), "-x", "-q",
           "-p", "no:cacheprovider", "-k", KEY]
    r = subprocess.run(cmd, env=env, cwd=os.path.dirname(HERE), capture_output=True, text=True,
                       timeout=200)
    tail = "\n".join((r.stdout + r.stderr).splitlines()[-15:])
    assert (r.returncode == 0) == passes, tail
    assert passes or "bad tile variant" in r.stdout, tail
