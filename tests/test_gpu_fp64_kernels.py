"""The FP64 kernels at the edges of their tiles: Ls below, at and between the
4-row steps and the 8 / 12 / 16 / 24 / 32 instances of the s-matrix products,
lattices whose half volume is no multiple of a block, and the block sizes the
dispatch switches to on larger lattices, against the CPU oracle."""

import numpy as np
import pytest

import qlattice_amd as q
from oracle import oracle as O
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


OPS = [("m_e_e", q.multiply_m_e_e), ("mdag_e_e_inv", q.multiply_mdag_e_e_inv), ("m_e_o", q.multiply_m_e_o),
       ("mdag_e_o", q.multiply_mdag_e_o), ("mpc_sym2", q.multiply_mpc_sym2), ("mpcdag_sym2", q.multiply_mpcdag_sym2),
       ("hermop_sym2", q.multiply_hermop_sym2)]


# the bar of the operator tests (FP64 sums of at most 32 terms and 8
# directions, four deep: a few 1e-15)
@pytest.mark.parametrize("z", [False, True])
@pytest.mark.parametrize("ls", [2, 3, 4, 5, 7, 8, 9, 13, 16, 17, 21, 25, 32])
def test_operators_at_the_edges_of_ls(ls, z):
    geo, inv, orc = make((2, 6, 2, 10), ls, z)
    for eo in (1, 2):
        x = rand_field((geo.total_volume() // 2, ls, 12), 60 + eo)
        f = q.FermionField5d(geo, ls, eo)
        f.data = x
        for name, fn in OPS:
            assert rel(fn(None, f, inv).data, orc.apply_half(name, x, eo)) < 1e-12, name


# half volumes of 8192 (32-site blocks of the fused hop for Ls <= 8), 12800
# (64-site blocks of the plain hop) and one site block more, ragged
@pytest.mark.parametrize("site,ls", [((8, 8, 8, 32), 3), ((10, 8, 16, 20), 2), ((10, 14, 10, 20), 6), ((6, 14, 14, 22), 9)])
def test_operators_on_larger_blocks(site, ls):
    geo, inv, orc = make(site, ls, False)
    x = rand_field((geo.total_volume() // 2, ls, 12), 70)
    f = q.FermionField5d(geo, ls, 1)
    f.data = x
    assert rel(q.multiply_hermop_sym2(None, f, inv).data, orc.apply_half("hermop_sym2", x, 1)) < 1e-12


@pytest.mark.parametrize("ls,z", [(3, False), (6, False), (10, False), (18, False)])
def test_cg_iterations_and_limits(ls, z):
    """The queued iterations of the CG stop where the oracle's loop stops:
    at convergence, at odd and even limits, and at a limit reached exactly."""
    geo, inv, orc = make((4, 4, 2, 6), ls, z)
    b = rand_field((geo.total_volume() // 2, ls, 12), 80)
    src = q.FermionField5d(geo, ls, 1)
    src.data = b
    ref, it_ref = orc.cg_with_herm_sym_2(b, stop_rsd=1e-8, max_num_iter=500)
    for limit in (1, 2, 3, 8, it_ref - 1, it_ref, it_ref + 1, 500):
        sol = q.FermionField5d(geo, ls, 1)
        it = q.cg_with_herm_sym_2(sol, src, inv, stop_rsd=1e-8, max_num_iter=limit)
        want, it_want = orc.cg_with_herm_sym_2(b, stop_rsd=1e-8, max_num_iter=limit)
        assert it == it_want, limit
        assert rel(sol.data, want) < 1e-9, limit
