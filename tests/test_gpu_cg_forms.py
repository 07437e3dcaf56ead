"""The FP64 and QED CG in the forms their kernels are instantiated for: complex
and real s-matrices on both sides of the 8 / 12 / 16 / 24 / 32 row instances,
and lattices where the block sums go through a reduction kernel (more than 4096
of them), against the oracles' loops at iteration limits."""

import numpy as np
import pytest

import qlattice_amd as q
from oracle import oracle as O
from oracle import qed as Q
from tests.helpers import rand_field, rand_gauge, rel

pytestmark = pytest.mark.gpu


def omega(ls):
    """Complex zMoebius coefficients that keep M_ee well conditioned."""
    w = [complex(1.1 - 0.7 * s / ls) for s in range(ls)]
    w[-1], w[-2] = complex(0.45, 0.05), complex(0.45, -0.05)
    return w


def make(site, ls, z):
    kw = dict(mass=0.1, ls=ls, m5=1.8, mobius_scale=1.0 if z else 2.0, omega=omega(ls) if z else None)
    U = rand_gauge(site, 0.4, 50 + ls)
    geo = q.Geometry(site)
    gf = q.GaugeField(geo)
    gf.data = U
    return geo, q.InverterDomainWall(gf=gf, fa=q.FermionAction(**kw)), O.OracleInverter(site, U, **kw)


def compare(geo, inv, orc, ls, limits):
    """Each application of Mpc^+ Mpc is within 1e-12 of the oracle's (the bar
    of the operator tests); a relative change of the source comes back in the
    iterates of the first eight iterations with a factor of 1.0 (measured with
    the oracle on these systems), so 1e-11 bounds eight applications."""
    b = rand_field((geo.total_volume() // 2, ls, 12), 80)
    src = q.FermionField5d(geo, ls, 1)
    src.data = b
    for limit in limits:
        sol = q.FermionField5d(geo, ls, 1)
        it = q.cg_with_herm_sym_2(sol, src, inv, stop_rsd=1e-8, max_num_iter=limit)
        want, it_want = orc.cg_with_herm_sym_2(b, stop_rsd=1e-8, max_num_iter=limit)
        assert it == it_want == limit + 1
        assert rel(sol.data, want) < 1e-11, limit


@pytest.mark.parametrize("ls,z", [(5, True), (7, True), (12, True), (16, True), (21, True), (28, True), (24, False),
                                  (28, False)])
def test_cg_instances(ls, z):
    print(f"\n[gpu] FP64 CG Ls{ls} complex {z}", flush=True)
    geo, inv, orc = make((4, 4, 2, 6), ls, z)
    compare(geo, inv, orc, ls, (1, 2, 3, 8))
    b = rand_field((geo.total_volume() // 2, ls, 12), 81)
    src = q.FermionField5d(geo, ls, 1)
    src.data = b
    sol = q.FermionField5d(geo, ls, 1)
    it = q.cg_with_herm_sym_2(sol, src, inv, stop_rsd=1e-8, max_num_iter=500)
    # (the iterated residual leaves the true one by rounding, far below 1e-8)
    assert it <= 500
    assert rel(orc.apply_half("hermop_sym2", sol.data, 1), b) < 1.01e-8


# Ls 9 has blocks of 16 sites: 4096 and 4352 block sums of Re <p, Ap>
@pytest.mark.parametrize("site,z", [((16, 16, 16, 32), False), ((16, 16, 16, 34), False), ((16, 16, 16, 34), True)])
def test_cg_on_both_sides_of_the_reduction(site, z):
    print(f"\n[gpu] FP64 CG {site} Ls9 complex {z}", flush=True)
    geo, inv, orc = make(site, 9, z)
    compare(geo, inv, orc, 9, (2,))


# elements of 4096 and 4097 blocks: the same for the QED CG (its bar per
# application is 1e-13)
@pytest.mark.parametrize("site,ls", [((8, 8, 16, 32), 8), ((1, 1, 241, 17), 64)])
def test_qed_cg_on_both_sides_of_the_reduction(site, ls):
    print(f"\n[gpu] QED CG {site} Ls{ls}", flush=True)
    rng = np.random.default_rng(7)
    V = int(np.prod(site))
    g = np.exp(1j * rng.uniform(0, 2 * np.pi, (V, 4)))
    x = rng.standard_normal((V, ls, 4)) + 1j * rng.standard_normal((V, ls, 4))
    sol, it = q.cg_with_m_dwf_qed(x, g, 0.1, 1.0, ls, site, None, False, 1e-10, 2)
    ref, it_ref = Q.cg_with_m_dwf_qed(x, g, 0.1, 1.0, ls, site, None, False, 1e-10, 2)
    assert it == it_ref == 3
    assert rel(sol, ref) < 1e-11
