"""One gradient step without constraints: U1 = (U0 + V0 Z) L^-T, V1 = (V0 + U0 Z) L^-T with
L L^T = 1 + Z^T Z and Z = -eta H20, against the oracle's evolve_wavefunction with the
projected H20 of the same state.  The orders are one block of 32 columns and less (24), a
remainder of 8 (40), whole blocks (64), of 16 (80) and of 12 (140).

Tolerance 1e-11: H20 of two runs differs by rounding (below 1e-12 of its largest entry, a
few tens of MeV, times eta), and n steps of rounding at 1.1e-16 grow by the condition
number of 1 + Z^T Z, below 100 here.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SPACES = {"sd": (4, 4, 0.1), "pf": (4, 4, 0.1), "sdpf": (6, 6, 0.1), "emax3": (6, 6, 0.03),
          "emax4": (8, 8, 0.02)}


@pytest.mark.parametrize("eta", [0.01, 0.1])
@pytest.mark.parametrize("space", list(SPACES))
def test_evolution_matches_oracle(space, eta):
    from oracle import pnvap
    from taurus_vap_amd import gpu, hamiltonian as H, host, inputs as I
    Z, N, sigma = SPACES[space]
    if space in I.WORKLOADS:
        b = I.WORKLOADS[space]
        w = I.Workload(space, b.space, Z, N, b.M, b.sigma, b.pairing, b.spe, decay=b.decay, hw=b.hw,
                       seed_sigma=sigma)
    else:
        w = I.Workload(space, space, Z, N, 9, 2.0, 0.0, "hw", decay=4.0, seed_sigma=sigma)
    h = H.workload_hamiltonian(w, 1234)
    b = h["basis"]
    U, V = host.seed_state(w, b, 5)
    cb = host.construct_canonical_basis(U, V)
    ctx = gpu.Context(b.dim, b.sp_2mj, b.sp_2mt, b.sp_l, b.sp_tr, h["H0"], h["H1"], h["abcd"], h["H2"],
                      h["trperm"])
    args = (U, V, cb["D"], cb["nocc"], cb["nemp"], cb["ovac"], cb["voveru"], 3, 3, 2.0 * np.pi, float(Z),
            float(N))
    n = b.dim
    H20 = np.asarray(ctx.project_wavefunction(*args)["H20v"]).reshape(n, n, order="F")
    ctx.set_gradient(eta, 0.0)
    ctx.set_state(*args)
    ctx.iterate(0.0)
    U1, V1 = ctx.get_state()
    Uo, Vo = pnvap.evolve_wavefunction(U, V, -eta * H20)[:2]
    assert np.abs(np.asarray(U1) - Uo).max() <= 1e-11
    assert np.abs(np.asarray(V1) - Vo).max() <= 1e-11
