"""Fields of interactions that have only some of the symmetries the contraction's blocks may
be reduced by, against the oracle's loop over the stored list: charge independent, charge
dependent, and every element changed by itself, stored in 32 and 64 bits, for one and for
several sets of densities (a projection of a few angles).  Tolerance 1e-10 as for the
reference's own interactions (elements below 20, densities below 1)."""
import numpy as np
import pytest

from conftest import golden_canon, golden_ham, load_golden

pytestmark = pytest.mark.gpu


def _list(g, kind):
    H2 = g["H2"].astype(np.float64).copy()
    rng = np.random.default_rng(4)
    h = int(g["ndim"]) // 2
    abcd = g["abcd"].reshape(-1, 4)
    if kind == "charge":                       # proton pairs 3 % stronger
        H2[(abcd <= h).all(axis=1)] *= 1.03
    elif kind == "each":
        H2 *= 1.0 + 0.1 * rng.normal(size=H2.size)
    return H2


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("kind", ["stored", "charge", "each"])
@pytest.mark.parametrize("case", ["sd32", "pf64"])
def test_fields_and_projection_match_oracle(case, kind, fp32):
    from oracle import pnvap
    from taurus_vap_amd import gpu
    g = load_golden(case)
    n = int(g["ndim"])
    H2 = _list(g, kind)
    if fp32:
        H2 = H2.astype(np.float32)
    ham = dict(golden_ham(g), H2=H2.astype(np.float64))
    sp_tr = g["sp_tr"].astype(int) - 1
    ctx = gpu.Context(n, g["sp_2mj"], g["sp_2mt"], g["sp_l"], g["sp_tr"], complex(g["H0"]), g["H1"],
                      g["abcd"], H2, g["trperm"], tbme_fp32=fp32)
    try:
        ph, pp = ctx.contraction_size()
        print(case, kind, "fp32" if fp32 else "fp64", "blocks", ph, pp, flush=True)
        rng = np.random.default_rng(1)
        rho = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
        k1, k2 = (rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n)) for _ in range(2))
        k1, k2 = k1 - k1.T, k2 - k2.T
        sc = 1.0 / max(1.0, np.abs(rho).max(), np.abs(k1).max(), np.abs(k2).max())
        args = [sc * x for x in (rho, k1, k2)]
        for x, y in zip(ctx.calculate_fields(*args), pnvap.calculate_fields(*args, ham, g["sp_2mj"], sp_tr)):
            assert np.max(np.abs(x - y)) <= 1e-10
        cb = golden_canon(g)
        setup = (3, 2, 2.0 * np.pi, float(g["valence_Z"]), float(g["valence_N"]))
        r = ctx.project_wavefunction(g["U0"], g["V0"], cb["D"].real, cb["nocc"], cb["nemp"],
                                     cb["ovac"], cb["voveru"], *setup)
        ref = pnvap.project_wavefunction(g["U0"], g["V0"], ham, dict(sp_2mj=g["sp_2mj"], sp_tr=sp_tr),
                                         *setup, canon=cb)
        assert abs(r["ener"] - ref["ener"]) <= 1e-10 * max(1.0, abs(ref["ener"]))
        H20v = np.asarray(ref["H20v"]).reshape(-1, order="F")
        assert np.max(np.abs(r["H20v"] - H20v)) <= 1e-10
    finally:
        ctx.close()


def test_reduction_follows_the_symmetries():
    """Fewer multiply-adds with more symmetry.  Proton pairs of their own strength leave the
    pair blocks as they are: the reflection maps proton pairs to neutron pairs, another
    class, and splits the proton-neutron ones alone."""
    from taurus_vap_amd import gpu
    g = load_golden("sd32")
    n = int(g["ndim"])
    m, t, l = (g[k].astype(int) for k in ("sp_2mj", "sp_2mt", "sp_l"))
    whole = [0, 0]
    for q in range(2):
        count = {}
        for y in range(n):
            for x in range(y + 1 if q else 0, n):
                s = 1 if q else -1
                key = (m[x] + s * m[y], t[x] + s * t[y], (l[x] + l[y]) & 1)
                count[key] = count.get(key, 0) + 1
        whole[q] = sum(v * v for v in count.values())
    size = {}
    for kind in ("stored", "charge", "each"):
        ctx = gpu.Context(n, g["sp_2mj"], g["sp_2mt"], g["sp_l"], g["sp_tr"], complex(g["H0"]), g["H1"],
                          g["abcd"], _list(g, kind).astype(np.float32), g["trperm"], tbme_fp32=True)
        size[kind] = ctx.contraction_size()
        ctx.close()
    assert size["stored"][0] < size["charge"][0] < size["each"][0] <= whole[0], (size, whole)
    assert size["stored"][1] == size["charge"][1] < size["each"][1] <= whole[1], (size, whole)
