"""Device memory of a projection: per (state, angle) item thirteen work matrices, A_phi and G,
four matrices of contraction layouts and, without a fully occupied level, two of the
Pfaffian: 21 n^2 complex numbers, with 4 % for rows filled up to whole lines, R6 and the like.
A work matrix that nothing reads would be another 5 %, and make every chunk of a
projection that is short of memory smaller."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _free():
    """Free device memory, from the HIP runtime that the library has loaded."""
    paths = {l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l}
    path = sorted(p for p in paths if "/torch/" not in p)[0]
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL(path).hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_projection_holds_no_more_than_its_work():
    from taurus_vap_amd import gpu, hamiltonian as H, host, inputs as I
    w = I.WORKLOADS["emax4"]
    h = H.workload_hamiltonian(w, 1234)
    b = h["basis"]
    n, M = b.dim, 15
    U, V = host.seed_state(w, b, 5)
    cb = host.construct_canonical_basis(U, V)
    assert cb["nocc"] == 0
    ctx = gpu.Context(n, b.sp_2mj, b.sp_2mt, b.sp_l, b.sp_tr, h["H0"], h["H1"], h["abcd"], h["H2"],
                      h["trperm"])
    try:
        free = _free()
        ctx.project_wavefunction(U, V, cb["D"], cb["nocc"], cb["nemp"], cb["ovac"], cb["voveru"], M, M,
                                 2.0 * np.pi, float(w.Z), float(w.N))
        used = free - _free()
    finally:
        ctx.close()
    print("bytes per item over n^2 complex:", used / (16.0 * n * n * M * M), flush=True)
    assert used <= 1.04 * 21 * 16.0 * n * n * M * M
