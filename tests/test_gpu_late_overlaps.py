"""Overlaps that start after the densities: orders of 66 to 150 with more than 128 angles at
once.  80 states with 12 x 12 angles against the same with a batch limit of 128 and of 37
items, where they start first; eager and as a captured graph, with the parity overlaps, and
with the canonical basis deferred to the second stream.  The runs add the same numbers in
the same order but for the chunks, so the tolerances are those of the chunk tests: 1e-11 of
the scalars, 1e-10 on H20 and the gradient."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

M = 12
KEYS = ("over", "ener", "prot", "neut", "prot2", "neut2", "pari")


@pytest.fixture(scope="module")
def case():
    from taurus_vap_amd import hamiltonian as H, host, inputs as I
    w = I.Workload("emax3", "emax3", 6, 6, 9, 2.0, 0.0, "hw", decay=4.0, seed_sigma=0.03)
    h = H.workload_hamiltonian(w, 1234)
    U, V = host.seed_state(w, h["basis"], 5)
    return h, U, V, host.construct_canonical_basis(U, V)


def _ctx(h, **kw):
    from taurus_vap_amd import gpu
    b = h["basis"]
    return gpu.Context(b.dim, b.sp_2mj, b.sp_2mt, b.sp_l, b.sp_tr, h["H0"], h["H1"], h["abcd"], h["H2"],
                       h["trperm"], **kw)


def _set(ctx, case, iprint):
    _, U, V, cb = case
    ctx.set_state(U, V, cb["D"], cb["nocc"], cb["nemp"], cb["ovac"], cb["voveru"], M, M, 2.0 * np.pi,
                  6.0, 6.0, iprint=iprint)


@pytest.mark.parametrize("iprint", [0, 1])
@pytest.mark.parametrize("graph", [False, True])
def test_late_overlaps_match_early_ones(case, graph, iprint):
    out = {}
    for limit in (128, 37, 0):
        ctx = _ctx(case[0], graph=graph and limit == 0)
        try:
            ctx.set_batch_limit(limit)
            ctx.set_gradient(0.01, 0.3)
            _set(ctx, case, iprint)
            for rep in range(4):       # eager, captured, replayed when graph
                print("graph" if graph else "eager", "limit", limit, "pass", rep, flush=True)
                ctx.project_resident()
                out[limit, rep] = (ctx.get_results(), ctx.get_gradient()[0])
        finally:
            ctx.close()
    for limit in (37, 0):
        for rep in range(4):
            (r, Z), (ref, Zref) = out[limit, rep], out[128, rep]
            for k in KEYS:
                assert abs(r[k] - ref[k]) <= 1e-11 * max(1.0, abs(ref[k])), (limit, rep, k)
            assert np.max(np.abs(r["H20v"] - ref["H20v"])) <= 1e-10, (limit, rep)
            assert np.max(np.abs(Z - Zref)) <= 1e-10, (limit, rep)


def test_deferred_basis_beside_many_angles(case):
    """iterate_canonical against canonical_basis and iterate, three iterations."""
    runs = []
    for deferred in (True, False):
        ctx = _ctx(case[0])
        try:
            ctx.set_gradient(0.01, 0.2)
            _set(ctx, case, 0)
            res = [ctx.iterate(0.0)]
            for it in range(3):
                print("deferred" if deferred else "in turn", it, flush=True)
                if deferred:
                    res.append(ctx.iterate_canonical()[0])
                else:
                    ctx.canonical_basis()
                    res.append(ctx.iterate(0.0))
            runs.append((res, ctx.get_state()))
        finally:
            ctx.close()
    for a, b in zip(runs[0][0], runs[1][0]):
        for k in KEYS[:6] + ("gradient_norm",):
            assert abs(a[k] - b[k]) <= 1e-11 * max(1.0, abs(b[k])), k
    for x, y in zip(runs[0][1], runs[1][1]):
        assert np.max(np.abs(x - y)) <= 1e-10
