"""One gradient step at the orders above the named model spaces: the one-launch Cholesky and
inverse up to order 512 (340: last block of 20 columns; 388: of 4; 512: the LDS full) and the
blocked form above it (516, 576), against the oracle's evolve_wavefunction with the
projected H20 of the same state, mean field only.

One shell of n / 2 states per species and no two-body elements, so that the blocks of the
contraction stay small; the one-body part is a dense symmetric matrix.  Tolerance 1e-11 as for
the smaller orders: H20 is the library's own, and n steps of rounding at 1.1e-16 grow by the
condition number of 1 + Z^T Z, below 100 here."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [340, 388, 512, 516, 576])
def test_evolution_at_large_orders(n):
    from oracle import pnvap
    from taurus_vap_amd import gpu, host
    h = n // 2
    rng = np.random.default_rng(n)
    m = np.tile(np.arange(-(h - 1), h, 2), 2).astype(np.int32)
    t = np.repeat([-1, 1], h).astype(np.int32)
    partner = np.concatenate([np.arange(h)[::-1], h + np.arange(h)[::-1]])
    H1 = rng.normal(size=(n, n)) / np.sqrt(n)
    H1 = H1 + H1.T + np.diag(np.linspace(0.0, 10.0, n))
    # paired states, rotated
    th = rng.uniform(0.1, 1.2, size=n)
    th = np.where(m > 0, th, th[partner])
    U, V = np.diag(np.cos(th)), np.zeros((n, n))
    V[np.arange(n), partner] = np.sin(th) * np.sign(m)
    X = rng.normal(size=(n, n)) * 0.01
    U, V = host.evolve(U, V, X - X.T)
    cb = host.construct_canonical_basis(U, V)
    ctx = gpu.Context(n, m, t, np.full(n, h - 1), partner + 1, 0.0, H1.astype(complex), np.zeros(0),
                      np.zeros(0), np.zeros(0))
    try:
        args = (U, V, cb["D"], cb["nocc"], cb["nemp"], cb["ovac"], cb["voveru"], 1, 1, 2.0 * np.pi,
                float(h // 2), float(h // 2))
        print("projection of order", n, flush=True)
        H20 = np.asarray(ctx.project_wavefunction(*args)["H20v"]).reshape(n, n, order="F")
        ref = U.T @ H1 @ V
        ref = ref - ref.T
        assert np.abs(H20 - ref).max() <= 1e-10
        for eta in (0.01, 0.1):
            ctx.set_gradient(eta, 0.0)
            ctx.set_state(*args)
            print("step", eta, flush=True)
            ctx.iterate(0.0)
            U1, V1 = ctx.get_state()
            Uo, Vo = pnvap.evolve_wavefunction(U, V, -eta * H20)[:2]
            assert np.abs(np.asarray(U1) - Uo).max() <= 1e-11
            assert np.abs(np.asarray(V1) - Vo).max() <= 1e-11
    finally:
        ctx.close()
