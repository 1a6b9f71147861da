"""The bits of a projection do not depend on which tile shapes the autotuner picks: it picks
by timing, so two runs of one input may differ in them.  A child process per tile (the
forced shapes are read once per process) prints a digest of every output; all must agree,
and with the child that tunes for itself.  Orders 24, 40 and 140 (remainders of 16 and 32),
14 and 36 angles."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHILD = """
import hashlib, sys
import numpy as np
sys.path.insert(0, %r)
from taurus_vap_amd import gpu, hamiltonian as H, host, inputs as I
for name, M in (("sd", 7), ("pf", 6), ("emax4", 6)):
    w = I.WORKLOADS[name]
    h = H.workload_hamiltonian(w, 1234)
    b = h["basis"]
    U, V = host.seed_state(w, b, 5)
    cb = host.construct_canonical_basis(U, V)
    ctx = gpu.Context(b.dim, b.sp_2mj, b.sp_2mt, b.sp_l, b.sp_tr, h["H0"], h["H1"], h["abcd"], h["H2"],
                      h["trperm"])
    r = ctx.project_wavefunction(U, V, cb["D"], cb["nocc"], cb["nemp"], cb["ovac"], cb["voveru"], M,
                                 M if name != "sd" else 2, 2.0 * np.pi, float(w.Z), float(w.N))
    ctx.close()
    for k in sorted(r):
        print(name, k, hashlib.sha256(np.asarray(r[k]).tobytes()).hexdigest())
"""


def _digests(**env):
    e = {k: v for k, v in os.environ.items() if not k.startswith("TG_G")}
    r = subprocess.run([sys.executable, "-c", CHILD % ROOT], env=dict(e, **env), capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    return r.stdout.splitlines()


def test_bits_do_not_depend_on_the_tile_shapes():
    ref = _digests()
    assert len(ref) == 3 * 12, ref
    for v in range(11):
        print("tile", v, flush=True)
        out = _digests(TG_GEMM_VARIANT=str(v), TG_GROUPED_VARIANT=str(v % 5))
        assert out == ref, [(a, b) for a, b in zip(out, ref) if a != b]
