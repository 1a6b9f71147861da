"""Device memory of a projection: per (state, angle) item thirteen work matrices, A_phi and G,
four matrices of contraction layouts and, without a fully occupied level, two of the
Pfaffian: 21 n^2 complex numbers, with 4 % for rows filled up to whole lines, R6 and the like.
A work matrix that nothing reads would be another 5 %, and make every chunk of a
projection that is short of memory smaller."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_projection_holds_no_more_than_its_work():
    torch = pytest.importorskip("torch")
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
        free = torch.cuda.mem_get_info()[0]
        ctx.project_wavefunction(U, V, cb["D"], cb["nocc"], cb["nemp"], cb["ovac"], cb["voveru"], M, M,
                                 2.0 * np.pi, float(w.Z), float(w.N))
        used = free - torch.cuda.mem_get_info()[0]
    finally:
        ctx.close()
    print("bytes per item over n^2 complex:", used / (16.0 * n * n * M * M), flush=True)
    assert used <= 1.04 * 21 * 16.0 * n * n * M * M
