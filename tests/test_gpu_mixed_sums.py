"""Sums of the mixed path that two kernels form, one of them to subtract the other's:
the pair sums of hpsi against those of the moves and of the quadrature."""
import numpy as np
import pytest

from champ_amd import system as S
from champ_amd.engine import PREC_FP64, PREC_MIXED, Engine
from tests.gpu_helpers import ENGINE_LIB

pytestmark = pytest.mark.gpu

NWALK = 16 if "emu" in ENGINE_LIB else 64


def molecule(nheavy, nh, nelec, order, ecp):
    return S.make_system("sums", nheavy, nh, nelec, "ssppd", "sp", nloc=4 if ecp else 0, nordc=order)


def change_of_ln_psi(sy, prec, x, moves):
    eng = Engine(sy, len(x), precision=prec, lib_path=ENGINE_LIB)
    eng.set_walkers(x)
    psij = eng.hpsi()["psij"]
    return np.array([eng.psie(i, xi)[1] - psij for i, xi in moves])


@pytest.mark.parametrize("shape", [(9, 4, 60, 4, True), (5, 3, 33, 5, True), (5, 3, 33, 3, False)],
                         ids=lambda s: "-".join(map(str, s)))
def test_errors_of_a_moves_jastrow_scatter_about_zero(require_gpu, shape):
    """ln J of a proposal minus that of hpsi: on the mixed path the roundings of the two
    are independent from pair to pair, so their mean over n moves is within five standard
    errors of 0; a constant rounded in one of them only shifts every pair the same way."""
    sy = molecule(*shape)
    x = sy.initial_walkers(NWALK, seed=21)
    rng = np.random.default_rng(22)
    moves = [(i, np.ascontiguousarray(x[:, i] + 0.3 * rng.standard_normal((NWALK, 3))))
             for i in range(0, sy.nelec, sy.nelec // 8)]
    d = change_of_ln_psi(sy, PREC_MIXED, x, moves) - change_of_ln_psi(sy, PREC_FP64, x, moves)
    assert abs(d.mean()) < 5 * d.std() / np.sqrt(d.size), (d.mean(), d.std(), d.size)


@pytest.mark.parametrize("order,form", [(1, -1), (4, 1)])
def test_vector_pipe_quadrature_of_the_mixed_path(require_gpu, order, form):
    """The vector-pipe quadrature subtracts hpsi's FP64 pair sums and forms its own the
    same way: a mixed hpsi with it has no FP32 operation left, so the energies are those
    of the FP64 path to the rounding of sums of a few thousand terms."""
    sy = molecule(4, 3, 25, order, True)
    x = sy.initial_walkers(8, seed=23)
    e = {}
    for prec in (PREC_FP64, PREC_MIXED):
        eng = Engine(sy, len(x), precision=prec, lib_path=ENGINE_LIB)
        eng.set_tuning(quadrature=form)
        eng.set_walkers(x)
        e[prec] = eng.hpsi()["energy"]
    assert np.all(np.abs(e[PREC_MIXED] - e[PREC_FP64]) <= 1e-12 * np.maximum(1.0, np.abs(e[PREC_FP64])))


@pytest.mark.parametrize("shape", [(5, 3, 33, 5, False), (4, 4, 20, 4, False), (3, 1, 65, 1, False)],
                         ids=lambda s: "-".join(map(str, s)))
def test_pair_sums_without_a_quadrature_are_fp32(require_gpu, shape):
    """An all-electron system has no quadrature that subtracts hpsi's pair sums: the
    mixed path forms them in FP32 (their values differ from the FP64 ones), to the
    rounding of FP32 terms."""
    sy = molecule(*shape)
    x = sy.initial_walkers(8, seed=24)
    h = {}
    for prec in (PREC_FP64, PREC_MIXED):
        eng = Engine(sy, len(x), precision=prec, lib_path=ENGINE_LIB)
        eng.set_walkers(x)
        h[prec] = eng.hpsi()
    for key, tol in (("psij", 2e-6), ("ekin", 2e-5)):
        d = np.abs(h[PREC_MIXED][key] - h[PREC_FP64][key])
        assert np.all(d <= tol * np.maximum(1.0, np.abs(h[PREC_FP64][key]))), key
    assert np.any(h[PREC_MIXED]["ekin"] != h[PREC_FP64]["ekin"])


@pytest.mark.parametrize("shape", [(5, 3, 33, 5, True), (4, 4, 20, 4, True)], ids=lambda s: "-".join(map(str, s)))
def test_pair_sums_under_a_quadrature_are_fp64(require_gpu, shape):
    """With a pseudopotential hpsi's pair sums, orbitals and inverse are FP64 on both
    paths: ln J and the kinetic energy agree to the rounding of sums of a few thousand terms."""
    sy = molecule(*shape)
    x = sy.initial_walkers(8, seed=25)
    h = {}
    for prec in (PREC_FP64, PREC_MIXED):
        eng = Engine(sy, len(x), precision=prec, lib_path=ENGINE_LIB)
        eng.set_walkers(x)
        h[prec] = eng.hpsi()
    for key in ("psij", "ekin"):
        d = np.abs(h[PREC_MIXED][key] - h[PREC_FP64][key])
        assert np.all(d <= 1e-12 * np.maximum(1.0, np.abs(h[PREC_FP64][key]))), key
