"""Engine against the oracle on molecules whose sizes cut the kernels' tiles: electron
counts around 16 and 64, centre counts that 4 does not divide, few quadrature pairs,
unequal spins, and e-e-n orders 2, 3 and 5."""
import numpy as np
import pytest

from champ_amd import system as S
from champ_amd.engine import PREC_FP64, PREC_MIXED, Engine
from oracle import ffi
from tests.gpu_helpers import ENGINE_LIB, relnorm

pytestmark = pytest.mark.gpu

# heavy atoms, hydrogens, electrons, e-e-n order, pseudopotential
SHAPES = [(2, 0, 2, 4, True), (2, 1, 9, 2, True), (3, 2, 17, 3, True), (5, 0, 33, 5, True), (4, 3, 16, 4, True),
          (9, 4, 65, 4, True), (3, 3, 15, 5, False)]


def molecule(nheavy, nh, nelec, order, ecp):
    return S.make_system("shape", nheavy, nh, nelec, "ssppd", "sp", nloc=4 if ecp else 0, nordc=order)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "-".join(map(str, s)))
@pytest.mark.parametrize("prec", [PREC_FP64, PREC_MIXED])
def test_hpsi_of_odd_shapes(require_gpu, shape, prec):
    sy = molecule(*shape)
    nw = 3
    x = sy.initial_walkers(nw, seed=4)
    eng = Engine(sy, nw, precision=prec, lib_path=ENGINE_LIB)
    eng.set_walkers(x)
    g = eng.hpsi()
    # FP64: the rounding of sums of a few thousand terms, and of a Slater inverse
    # of condition up to 1e6 in the energies; mixed: FP32 terms summed in FP64
    tol_j, tol_e = (1e-12, 1e-9) if prec == PREC_FP64 else (2e-6, 2e-5)
    ref = []
    for w in range(nw):
        o = ffi.walker(sy)
        o.set_x(x[w])
        if sy.nloc:
            o.set_quad(sy.xq0, sy.yq0, sy.zq0)
        ref.append(o.hpsi())
        assert relnorm(eng.array("vj")[w], o.vj()) < max(tol_j, 1e-12) * 10
    for key, tol in (("psij", tol_j), ("ekin", tol_e), ("energy", tol_e)):
        r = np.array([d[key] for d in ref])
        # the terms of E_L cancel: relative to their own size
        scale = np.maximum(1.0, np.abs(r)) if key != "energy" else np.maximum(np.abs(r), np.abs([d["ekin"] for d in ref]))
        assert np.all(np.abs(g[key] - r) <= tol * np.maximum(1.0, scale)), (key, g[key], r)


def drop_ao(sy, it, i):
    """The system without AO i of type it: its shell is no whole set any more."""
    first = np.concatenate([[0], np.cumsum([sy.nbastyp[t] for t in sy.iwctype])])
    gone = [first[c] + i for c, t in enumerate(sy.iwctype) if t == it]
    sy.coef = np.ascontiguousarray(np.delete(sy.coef, gone, axis=1))
    for name in ("iwrwf", "iwlbas"):
        a = getattr(sy, name).copy()
        a[it, i:-1] = a[it, i + 1:]
        setattr(sy, name, a)
    sy.nbastyp = sy.nbastyp.copy()
    sy.nbastyp[it] -= 1
    return sy


@pytest.mark.parametrize("heavy,hyd,drop", [("spf", "s", None), ("sspd", "sp", (0, 3)), ("fd", "p", (0, 12)), ("s", "f", (1, 0))])
def test_quadrature_of_shell_sets(require_gpu, heavy, hyd, drop):
    """s, p, d and f sets, and shells that miss one of their monomials, in the
    quadrature's psi ratio (all of E_L against the oracle)."""
    sy = S.make_system("shells", 3, 2, 11, heavy, hyd, nloc=4, nordc=4)
    if drop is not None:
        sy = drop_ao(sy, *drop)
    nw = 2
    x = sy.initial_walkers(nw, seed=9)
    eng = Engine(sy, nw, lib_path=ENGINE_LIB)
    eng.set_walkers(x)
    g = eng.hpsi()
    for w in range(nw):
        o = ffi.walker(sy)
        o.set_x(x[w])
        o.set_quad(sy.xq0, sy.yq0, sy.zq0)
        d = o.hpsi()
        assert abs(g["energy"][w] - d["energy"]) <= 1e-9 * max(1.0, abs(d["energy"]), abs(d["ekin"]))


# (2, 1, 9): one pass of 16 lanes; 33 and 65 electrons: a full pass and a remainder of 1;
# 97: 64 + 33 (two passes of 64 lanes); 40: one pass; spins above 32, 80 (five and ten
# columns of the update) through 65 and 170 electrons
@pytest.mark.parametrize("shape", [(2, 1, 9, 2, True), (5, 0, 33, 5, True), (9, 4, 65, 4, True), (13, 7, 97, 3, False),
                                   (6, 2, 40, 4, True), (22, 0, 170, 4, True)], ids=lambda s: "-".join(map(str, s)))
@pytest.mark.parametrize("nwalk", [3, 1030])
@pytest.mark.parametrize("mover", [1, 6])
def test_sweep_of_odd_shapes(require_gpu, shape, nwalk, mover):
    """One sweep against the oracle's, with few walkers (several wavefronts per
    walker) and with many (one per walker); the first and last walkers are compared."""
    if "emu" in ENGINE_LIB and nwalk > 100:
        pytest.skip("population too large for the host emulation")
    if mover == 6 and shape[2] > 128:
        pytest.skip("ill-conditioned start: its small determinant ratios amplify roundings to 1e-7, in any kernel")
    sy = molecule(*shape)
    x = sy.initial_walkers(nwalk, seed=6)
    eng = Engine(sy, nwalk, lib_path=ENGINE_LIB)
    eng.set_walkers(x)
    st = np.random.default_rng(5).integers(1, 2 ** 63 - 1, size=(nwalk, 4), dtype=np.uint64)
    eng.set_rng(st)
    eng.hpsi()
    r = eng.metrop1(1, 0.3) if mover == 1 else eng.metrop6(1)
    assert 0 < r["accepted"] <= r["proposed"]
    # a proposal outside every AO's cut radius has the ratio 0, which flags the walker (2)
    assert not np.any(eng.status() & ~2)
    got, sc, rng = eng.get_walkers(), eng.scalars(), eng.get_rng()
    for w in (0, 1, nwalk - 1):
        o = ffi.walker(sy)
        o.set_x(x[w])
        o.set_rng(st[w])
        if sy.nloc:
            o.set_quad(sy.xq0, sy.yq0, sy.zq0)
        o.hpsi()
        o.sweep(0.3) if mover == 1 else o.sweep6()
        d = o.scalars()
        # the same decisions, positions to the rounding of the drifts, ln psi and E_L
        # to that of an inverse updated once per electron
        assert np.array_equal(rng[w], o.get_rng())
        assert np.max(np.abs(got[w] - o.get_x())) < 1e-8
        assert abs(sc["psijo"][w] - d["psijo"]) < 1e-8 * max(1.0, abs(d["psijo"]))
        assert abs(sc["eold"][w] - d["eold"]) < 1e-6 * max(1.0, abs(d["eold"]))


@pytest.mark.parametrize("prec", [PREC_FP64, PREC_MIXED])
@pytest.mark.parametrize("order", [4, 5])
def test_quadrature_forms_agree(require_gpu, order, prec):
    """The matrix-core form against the vector-pipe form at several partner tiles, centre
    steps and resident blocks: 97 electrons, 20 centres, 40 walkers."""
    if "emu" in ENGINE_LIB:
        pytest.skip("population too large for the host emulation")
    sy = molecule(13, 7, 97, order, True)
    x = sy.initial_walkers(40, seed=12)
    e = []
    for form, p in ((0, prec), (1, PREC_FP64)):
        eng = Engine(sy, len(x), precision=p, lib_path=ENGINE_LIB)
        eng.set_tuning(quadrature=form)
        eng.set_walkers(x)
        h = eng.hpsi()
        e.append(h["energy"])
    # FP64: the rounding of sums of a few thousand terms; mixed: FP32 terms summed in FP64
    tol = 1e-9 if prec == PREC_FP64 else 2e-5
    assert np.all(np.abs(e[0] - e[1]) <= tol * np.maximum(1.0, np.maximum(np.abs(e[1]), np.abs(h["ekin"]))))


# 9 and 64 electrons: one wavefront per walker, alone in its block or four to a block
# (above 512 walkers; two where four walkers' tables of 120 centres would not fit);
# 65: a wavefront per 64 partners
@pytest.mark.parametrize("shape", [(2, 1, 9, 4, False), (6, 3, 64, 5, False), (100, 20, 64, 5, False), (6, 3, 65, 4, False)],
                         ids=lambda s: "-".join(map(str, s)))
@pytest.mark.parametrize("prec", [PREC_FP64, PREC_MIXED])
def test_psie_does_not_depend_on_the_population(require_gpu, shape, prec):
    """ln J and its gradient at a proposal, the same bits for a walker among 3 and among 517."""
    if "emu" in ENGINE_LIB:
        pytest.skip("population too large for the host emulation")
    sy = molecule(*shape)
    x = sy.initial_walkers(517, seed=14)
    xn = x[:, 1] + 0.2
    got = []
    for part in (slice(0, 3), slice(0, 517)):
        eng = Engine(sy, len(x[part]), precision=prec, lib_path=ENGINE_LIB)
        eng.set_walkers(x[part])
        eng.hpsi()
        got.append((eng.psie(1, np.ascontiguousarray(xn[part]))[1], eng.array("vjn")))
    for small, large in zip(*got):
        assert np.array_equal(small, large[:3])


def sweep_against_oracle(sy, nwalk, walkers, lu_every=None, tau=0.3):
    x = sy.initial_walkers(nwalk, seed=6)
    eng = Engine(sy, nwalk, lib_path=ENGINE_LIB)
    if lu_every is not None:
        eng.set_lu_every(lu_every)
    eng.set_walkers(x)
    st = np.random.default_rng(5).integers(1, 2 ** 63 - 1, size=(nwalk, 4), dtype=np.uint64)
    eng.set_rng(st)
    eng.hpsi()
    eng.metrop1(1, tau)
    got, sc, rng = eng.get_walkers(), eng.scalars(), eng.get_rng()
    for w in walkers:
        o = ffi.walker(sy)
        o.set_x(x[w])
        o.set_rng(st[w])
        if sy.nloc:
            o.set_quad(sy.xq0, sy.yq0, sy.zq0)
        o.hpsi()
        o.sweep(tau)
        d = o.scalars()
        # as in test_sweep_of_odd_shapes
        assert np.array_equal(rng[w], o.get_rng())
        assert np.max(np.abs(got[w] - o.get_x())) < 1e-8
        assert abs(sc["psijo"][w] - d["psijo"]) < 1e-8 * max(1.0, abs(d["psijo"]))
        assert abs(sc["eold"][w] - d["eold"]) < 1e-6 * max(1.0, abs(d["eold"]))


# spins of 132 and 131: a second pass over the orbitals beside ten columns of the update
@pytest.mark.parametrize("nwalk", [2, 600])
def test_sweep_of_large_spins(require_gpu, nwalk):
    if "emu" in ENGINE_LIB:
        pytest.skip("system too large for the host emulation")
    sweep_against_oracle(molecule(40, 4, 263, 4, False), nwalk, (nwalk - 1,))


# spins of 166 and 165: the update row by row.  Steps of 0.03 bohr: the determinant ratios
# stay near 1, so that roundings add up and are not multiplied by small ratios' inverses
@pytest.mark.parametrize("nwalk", [2, 600])
def test_row_by_row_update(require_gpu, nwalk):
    if "emu" in ENGINE_LIB:
        pytest.skip("system too large for the host emulation")
    sweep_against_oracle(molecule(40, 4, 331, 4, False), nwalk, (nwalk - 1,), tau=1e-3)


@pytest.mark.parametrize("every", [1, 7, 32])
def test_sweep_split_by_the_refresh(require_gpu, every):
    """The inverse recomputed inside the sweep, every step but the last a whole one."""
    sweep_against_oracle(molecule(5, 3, 33, 4, True), 3, (0, 2), lu_every=every)


# 20 electrons: a walker per block, four to a block; 33 and 97: a block per walker,
# then four walkers to a block (with a last block that is not full)
@pytest.mark.parametrize("prec", [PREC_FP64, PREC_MIXED])
@pytest.mark.parametrize("shape", [(4, 2, 20, 4, True), (5, 3, 33, 5, True), (13, 7, 97, 4, False)],
                         ids=lambda s: "-".join(map(str, s)))
def test_sweep_does_not_depend_on_the_population(require_gpu, shape, prec):
    """The same bits for a walker among 3 and among 517."""
    if "emu" in ENGINE_LIB:
        pytest.skip("population too large for the host emulation")
    sy = molecule(*shape)
    x = sy.initial_walkers(517, seed=15)
    st = np.random.default_rng(16).integers(1, 2 ** 63 - 1, size=(517, 4), dtype=np.uint64)
    got = []
    for n in (3, 517):
        eng = Engine(sy, n, precision=prec, lib_path=ENGINE_LIB)
        eng.set_tuning(orbital_gemm=0, ecp_rows_gemm=0 if sy.nloc else -1)  # hpsi's products too
        eng.set_walkers(x[:n])
        eng.set_rng(st[:n])
        eng.hpsi()
        eng.metrop1(2, 0.3)
        sc = eng.scalars()
        got.append((eng.get_walkers(), eng.get_rng(), sc["psijo"], sc["psido"]))
    for small, large in zip(*got):
        assert np.array_equal(small, large[:3])
