"""Iterations of so many states that the real products of the constraint steps take their
other form (32 x 32 tiles; 750 to 2000 tiles of 16 x 16 by operand order and length): orders
24, 40, 64 and 80 with remainders of 8, 8, 0 and 16 in a tile, a little above and below each
line.  Every state against a context that holds it alone: 1e-11 of the scalars, 1e-10 on
the evolved state, as for the batches of few states."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SPACES = {"sd": (4, 4, 0.1, [180, 188, 251]), "pf": (4, 4, 0.1, [83, 84, 112]),
          "sdpf": (6, 6, 0.1, [46, 47, 63]), "emax3": (6, 6, 0.03, [30, 31, 41])}


@pytest.mark.parametrize("space", list(SPACES))
def test_iteration_of_many_states_matches_single_ones(space):
    from taurus_vap_amd import gpu, hamiltonian as H, host, inputs as I
    Z, N, sigma, counts = SPACES[space]
    if space in I.WORKLOADS:
        b = I.WORKLOADS[space]
        w = I.Workload(space, b.space, Z, N, b.M, b.sigma, b.pairing, b.spe, decay=b.decay, hw=b.hw,
                       seed_sigma=sigma)
    else:
        w = I.Workload(space, space, Z, N, 9, 2.0, 0.0, "hw", decay=4.0, seed_sigma=sigma)
    h = H.workload_hamiltonian(w, 1234)
    b = h["basis"]
    ops = np.stack(host.number_operators(b))
    vals = np.array([float(Z), float(N)])
    states = []
    for seed in (5, 6, 7):
        U, V = host.seed_state(w, b, seed)
        states.append((U, V, host.construct_canonical_basis(U, V)))

    def run(sts):
        ctx = gpu.Context(b.dim, b.sp_2mj, b.sp_2mt, b.sp_l, b.sp_tr, h["H0"], h["H1"], h["abcd"],
                          h["H2"], h["trperm"])
        try:
            ctx.set_constraints(ops, vals)
            ctx.set_gradient(0.01, 0.0)
            ctx.set_states(sts, 1, 1, 2.0 * np.pi, float(Z), float(N))
            r = ctx.iterate(0.0)
            U, V = ctx.get_state()
        finally:
            ctx.close()
        return ([r], [U], [V]) if len(sts) == 1 else (r, U, V)

    single = [run([st]) for st in states]
    for S in counts:
        print(space, S, flush=True)
        r, U, V = run([states[k % 3] for k in range(S)])
        for k in sorted({0, 1, 2, S // 2, S - 2, S - 1}):
            rs, Us, Vs = (x[0] for x in single[k % 3])
            assert r[k]["adjust_iterations"] == rs["adjust_iterations"]
            for key in ("ener", "prot", "neut", "gradient_norm"):
                assert abs(r[k][key] - rs[key]) <= 1e-11 * max(1.0, abs(rs[key])), (S, k, key)
            assert np.max(np.abs(U[k] - Us)) <= 1e-10 and np.max(np.abs(V[k] - Vs)) <= 1e-10, (S, k)
