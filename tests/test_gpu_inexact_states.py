"""Projections of states that are orthonormal only to 1e-9 or 1e-6 (U and V read with few
digits, or left by another program's step).  Their Thouless matrix and pairing tensors are
not skew beyond that, so nothing may take half of one for the whole.

Expected values: the oracle's formulas on the same U, V, the pair channel of its fields fed
with the pairing tensor as the contraction takes it (the elements (x, y) that follow each
other in the order of 2mt, 2mj, parity, and minus them at (y, x); equal for an exact state).
Tolerances are those of exact states: 1e-10 on the matrices, 1e-11 of the sums on
the scalars; half products in place of whole ones miss them by a factor of 500 at 1e-9.
"""
import numpy as np
import pytest

from conftest import golden_canon, golden_ham, load_golden

pytestmark = pytest.mark.gpu

SCALARS = ("over", "ener", "prot", "neut", "prot2", "neut2")


def _ctx(g, **kw):
    from taurus_vap_amd import gpu
    return gpu.Context(int(g["ndim"]), g["sp_2mj"], g["sp_2mt"], g["sp_l"], g["sp_tr"],
                       complex(g["H0"]), g["H1"], g["abcd"], g["H2"], g["trperm"], **kw)


def _noisy(g, eps, seed=3):
    rng = np.random.default_rng(seed)
    U, V = np.asarray(g["U0"]), np.asarray(g["V0"])
    return U + eps * rng.normal(size=U.shape), V + eps * rng.normal(size=V.shape)


def _setup(g):
    return (int(g["Mphip"]), int(g["Mphin"]), float(g["facpi"]), float(g["valence_Z"]),
            float(g["valence_N"]), float(g["factor_delta"]))


def _project(ctx, g, U, V, cb):
    return ctx.project_wavefunction(U, V, cb["D"].real, cb["nocc"], cb["nemp"], cb["ovac"],
                                    cb["voveru"], *_setup(g))


def _same(r, ref, tol=1e-10, rel=1e-11, mats=("A", "H20", "AH20", "H20v")):
    for k in SCALARS:
        assert abs(r[k] - ref[k]) <= rel * max(1.0, abs(ref[k])), (k, r[k], ref[k])
    for k in mats:
        assert np.max(np.abs(r[k] - ref[k])) <= tol, k


@pytest.mark.parametrize("case", ["sd64", "pf64"])
@pytest.mark.parametrize("eps", [1e-9, 1e-6])
def test_projection_of_inexact_state_matches_oracle(case, eps, monkeypatch):
    from oracle import pnvap
    g = load_golden(case)
    n = int(g["ndim"])
    order = sorted(range(n), key=lambda i: (g["sp_2mt"][i], g["sp_2mj"][i], g["sp_l"][i] % 2))
    rank = np.empty(n, int)
    rank[order] = np.arange(n)
    keep = rank[:, None] > rank[None, :]
    fields = pnvap.calculate_fields

    def with_skew_kappa(rho, kLR, kRL, *a):
        return fields(rho, *(np.where(keep, k, 0) - np.where(keep, k, 0).T for k in (kLR, kRL)), *a)

    monkeypatch.setattr(pnvap, "calculate_fields", with_skew_kappa)
    cb = golden_canon(g)
    U, V = _noisy(g, eps)
    basis = dict(sp_2mj=g["sp_2mj"], sp_tr=g["sp_tr"].astype(int) - 1)
    ref = pnvap.project_wavefunction(U, V, golden_ham(g), basis, *_setup(g)[:5], canon=cb,
                                     factor_delta=float(g["factor_delta"]))
    ref["H20v"] = np.asarray(ref["H20v"]).reshape(-1, order="F")
    for limit in (0, 5):
        ctx = _ctx(g)
        try:
            ctx.set_batch_limit(limit)
            print(case, eps, "batch limit", limit, flush=True)
            _same(_project(ctx, g, U, V, cb), ref)
        finally:
            ctx.close()


def test_exact_and_inexact_states_in_one_context():
    """States of a batch, and states that follow each other through one context, are
    judged each for itself."""
    g = load_golden("sd64")
    cb = golden_canon(g)
    cb = dict(cb, D=cb["D"].real)
    exact = (np.asarray(g["U0"]), np.asarray(g["V0"]), cb)
    noisy = (*_noisy(g, 1e-6), cb)
    single = {}
    for name, st in (("exact", exact), ("noisy", noisy)):
        ctx = _ctx(g)
        try:
            single[name] = _project(ctx, g, *st)
        finally:
            ctx.close()
    assert np.max(np.abs(single["exact"]["H20v"] - single["noisy"]["H20v"])) > 1e-7
    names = ["exact", "noisy", "exact", "noisy"]
    ctx = _ctx(g)
    try:
        ctx.set_states([exact if k == "exact" else noisy for k in names], *_setup(g))
        for rep in range(2):
            ctx.project_resident()
            for k, name in enumerate(names):
                _same(ctx.get_results(k), single[name], mats=("H20v",))
    finally:
        ctx.close()
    for graph in (False, True):
        ctx = _ctx(g, graph=graph)
        try:
            # (graph: the second projection is captured, the later ones are replays)
            for name in ("exact", "exact", "noisy", "exact", "noisy", "noisy", "exact"):
                print("graph" if graph else "eager", name, flush=True)
                _same(_project(ctx, g, *(exact if name == "exact" else noisy)), single[name])
        finally:
            ctx.close()
