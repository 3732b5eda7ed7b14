"""bench.py's work counts: the polynomial's operations against the Horner evaluation they
count, the sweep kernel's work per launch, and what its headline roofline says it is."""
import numpy as np
import pytest

import bench
from champ_amd import system as S


class Counted:
    """A number that counts the multiplications and additions made with it."""
    ops = 0

    def __mul__(self, other):
        Counted.ops += 1
        return Counted()

    __add__ = __mul__


@pytest.mark.parametrize("order", [2, 3, 4, 5])
def test_polynomial_operations(order):
    # sum_k u^k sum_n A_kn y^n with d/du, d/dy and the rows of dA/dx, by Horner's rule
    # with the first step of each derivative a copy
    Counted.ops = 0
    nz = {(k, n) for k, l, m in S.een_terms(order) for n in (m, l + m)}
    kmax = max(k for k, _ in nz)
    y = u = Counted()
    P = Pu = Py = Px = None
    for k in range(kmax, -1, -1):
        rows = [n for kk, n in nz if kk == k]
        q, q1, r = Counted(), Counted(), Counted()
        for step, n in enumerate(range(max(rows) - 1, -1, -1) if rows else ()):
            q1 = q if step == 0 else q1 * y + q
            q = q * y + Counted() if (k, n) in nz else q * y
            r = r * y + Counted() if (k, n) in nz else r * y
        if P is None:
            P, Py, Px = q, q1, r
        else:
            Pu = P if Pu is None else Pu * u + P
            P, Py, Px = P * u + q, Py * u + q1, Px * u + r
    assert bench.een_eval_flops(order) == Counted.ops


@pytest.mark.parametrize("path,launches", [("fp64", 6), ("mixed", 12)])
def test_work_of_the_sweep_kernel(path, launches):
    """Six sweeps in one launch each, or in two (split by the refresh): the same work."""
    sy = S.config("c60")
    kt = {"moves": (600.0, launches), "hpsi_jastrow": (120.0, 6), "hpsi_nonloc": (50.0, 6)}
    nxq = np.full(512, 240)
    d = bench.per_kernel(sy, 512, kt, nxq, path, 0.4)["moves"]
    sweep = 512 * sy.nelec * bench.flops_move_pairs(sy.nelec, sy.ncent, sy.nordc, path)
    assert d["work_per_launch"] * launches == pytest.approx(6 * sweep, rel=1e-12)
    assert d["achieved"] == pytest.approx(6 * sweep / 0.6 / 1e12, abs=1e-3)
    r = bench.roofline(sy, 512, kt, nxq, path, 0.4)
    assert r["kernel"] == "moves" and r["bound"] == "valu" and r["utilisation"] is True
