"""Launch shapes that the named workloads do not reach: chunks of two to five angles (the
matrix-vector contraction for two to four rows, the packed layout of its pair rows, the first
matrix-core one), and runs of neighbouring states of one occupation shape that share an
overlap launch.  Against the same work in other launches, to the chunk and batch tests'
1e-11 of the scalars and 1e-10 on H20 and the gradient."""
import numpy as np
import pytest

from conftest import golden_canon, load_golden

pytestmark = pytest.mark.gpu

KEYS = ("over", "ener", "prot", "neut", "prot2", "neut2", "pari")


def _ctx(g, **kw):
    from taurus_vap_amd import gpu
    return gpu.Context(int(g["ndim"]), g["sp_2mj"], g["sp_2mt"], g["sp_l"], g["sp_tr"],
                       complex(g["H0"]), g["H1"], g["abcd"], g["H2"], g["trperm"], **kw)


def _setup(g):
    return (int(g["Mphip"]), int(g["Mphin"]), float(g["facpi"]), float(g["valence_Z"]),
            float(g["valence_N"]), float(g["factor_delta"]))


def _same(r, Z, ref, Zref):
    for k in KEYS:
        assert abs(r[k] - ref[k]) <= 1e-11 * max(1.0, abs(ref[k])), k
    assert np.max(np.abs(r["H20v"] - ref["H20v"])) <= 1e-10
    assert np.max(np.abs(Z - Zref)) <= 1e-10


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("case", ["sd64", "pf64"])
def test_chunks_of_few_angles(case, fp32):
    g = load_golden(case)
    cb = golden_canon(g)
    H2 = g["H2"].astype(np.float32) if fp32 else g["H2"]
    out = {}
    for limit in (0, 2, 3, 4, 5):
        ctx = _ctx(dict(g, H2=H2), tbme_fp32=fp32)
        try:
            ctx.set_batch_limit(limit)
            ctx.set_gradient(0.01, 0.3)
            ctx.set_state(g["U0"], g["V0"], cb["D"].real, cb["nocc"], cb["nemp"], cb["ovac"],
                          cb["voveru"], *_setup(g), iprint=1)
            print(case, "fp32" if fp32 else "fp64", "limit", limit, flush=True)
            ctx.project_resident()
            out[limit] = (ctx.get_results(), ctx.get_gradient()[0])
        finally:
            ctx.close()
    for limit in (2, 3, 4, 5):
        _same(*out[limit], *out[0])


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("pattern", ["PPSPP", "SSPPP", "PSPSS", "PPPSS"])
def test_runs_of_one_occupation_shape(pattern, graph):
    """Paired states (P) and Slater determinants (S) side by side in one context."""
    from taurus_vap_amd import host
    g = load_golden("batch_sd")
    n = int(g["ndim"])
    rng = np.random.default_rng(2)

    def slater(shift):
        occ = np.zeros(n, dtype=bool)
        occ[shift:shift + 4] = True
        occ[n // 2 + shift:n // 2 + shift + 4] = True
        return np.diag((~occ).astype(float)), np.diag(occ.astype(float))

    states = []
    for k, c in enumerate(pattern):
        if c == "S":
            U, V = slater(k % 3)
        else:
            X = rng.normal(size=(n, n)) * 0.03
            U, V = host.evolve(np.asarray(g["U0"][0]), np.asarray(g["V0"][0]), X - X.T)
        states.append((U, V, host.construct_canonical_basis(U, V)))
    ctx = _ctx(g, graph=graph)
    try:
        ctx.set_gradient(0.01, 0.0)
        ctx.set_states(states, *_setup(g))
        for rep in range(4 if graph else 1):
            print(pattern, "graph" if graph else "eager", rep, flush=True)
            ctx.project_resident()
            got = [(ctx.get_results(k), ctx.get_gradient(k)[0]) for k in range(len(states))]
    finally:
        ctx.close()
    for k, st in enumerate(states):
        single = _ctx(g)
        try:
            single.set_gradient(0.01, 0.0)
            single.set_states([st], *_setup(g))
            single.project_resident()
            _same(*got[k], single.get_results(), single.get_gradient()[0])
        finally:
            single.close()
