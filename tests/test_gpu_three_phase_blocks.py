"""The three-phase hop kernels at the ends of a lattice that fills no whole
block, for every block of sites that has a kernel at an Ls: FP32 storage, FP16
storage with FP16 products and with FP32 arithmetic, real and complex
s-matrices."""

import numpy as np
import pytest

import qlattice_amd as q
from tests.helpers import rand_field, rand_gauge, rel

pytestmark = pytest.mark.gpu

# (Ls, sites per block) with a kernel: whole waves, 6 <= Ls <= 24
BLOCKS = [(6, 32), (8, 16), (8, 32), (10, 32), (12, 16), (12, 32), (14, 32), (16, 8), (16, 16), (16, 32), (20, 16),
          (24, 8), (24, 16)]


# half volumes of 24 (less than a block of 32), 120 and 360 sites
@pytest.mark.parametrize("site,z", [((6, 2, 2, 2), False), ((2, 2, 6, 10), True), ((2, 6, 10, 6), False)])
@pytest.mark.parametrize("ls,sb", BLOCKS)
def test_ragged_lattices(monkeypatch, site, ls, sb, z):
    """FP32: the bar of the FP32 operator tests.  FP16 storage rounds the input
    and three intermediate fields to 11 bits of the site's largest component
    and the links likewise: four passes of sqrt(24) * 2^-12 or less against the
    site's norm and as much from the links, times the operator's growth of the
    first errors (below 2 on these fields), is below 3e-3."""
    print(f"\n[gpu] three-phase {site} Ls{ls} blocks of {sb}", flush=True)
    monkeypatch.setenv("QLAT_DWF_TP_SB", str(sb))
    monkeypatch.setenv("QLAT_DWF_RHS_TILE", "1")
    geo = q.Geometry(site)
    gf = q.GaugeField(geo)
    gf.data = rand_gauge(site, 0.4, 7)
    omega = [complex(0.6 + 0.1 * s, 0.02 * s) for s in range(ls)] if z else None
    fa = q.FermionAction(mass=0.05, ls=ls, m5=1.8, mobius_scale=0.0 if z else 2.0, omega=omega)
    x = rand_field((geo.total_volume() // 2, ls, 12), 11)
    for solver, h2, bar in (("mixed", "1", 2e-6), ("mixed16", "1", 3e-3), ("mixed16", "0", 3e-3)):
        monkeypatch.setenv("QLAT_DWF_H2", h2)
        inv = q.InverterDomainWall(gf=gf, fa=fa, solver=solver)
        for eo in (1, 2):
            f = q.FermionField5d(geo, ls, eo)
            f.data = x
            exact = q.multiply_hermop_sym2(None, f, inv).data
            assert rel(q.multiply_hermop_sym2_fp32(None, f, inv).data, exact) < bar, (solver, h2, eo)
        if not z:  # the block really is the one asked for
            inv.set_max_num_iter(2)
            inv.set_max_mixed_precision_cycle(1)
            full = q.FermionField5d(geo, ls, 0)
            full.data = rand_field((geo.total_volume(), ls, 12), 12)
            q.invert_batch([inv], [full])
            assert inv.stats()["sites_per_block"] == sb


@pytest.mark.parametrize("site,ls", [((6, 6, 6, 10), 4), ((10, 8, 16, 20), 3)])
@pytest.mark.parametrize("by,bz", [(1, 1), (2, 2), (2, 0), (0, 2), (0, 0)])
def test_site_orders_of_the_fp64_hop(monkeypatch, site, ls, by, bz):
    """Every tile of the site order gives the reference's operators on both
    blocks of the plain FP64 hop (16 sites, and 64 from a half volume of 12800
    on); 0: no tiles.  The bar of the operator tests."""
    from oracle import oracle as O

    print(f"\n[gpu] site order {site} tiles {by} x {bz}", flush=True)
    monkeypatch.setenv("QLAT_DWF_TILE_Y", str(by or site[1]))
    monkeypatch.setenv("QLAT_DWF_TILE_Z", str(bz or site[2]))
    kw = dict(mass=0.1, ls=ls, m5=1.8, mobius_scale=2.0)
    U = rand_gauge(site, 0.4, 31)
    geo = q.Geometry(site)
    gf = q.GaugeField(geo)
    gf.data = U
    inv, orc = q.InverterDomainWall(gf=gf, fa=q.FermionAction(**kw)), O.OracleInverter(site, U, **kw)
    x = rand_field((geo.total_volume() // 2, ls, 12), 40)
    for eo in (1, 2):
        f = q.FermionField5d(geo, ls, eo)
        f.data = x
        for name, fn in (("m_e_o", q.multiply_m_e_o), ("mdag_e_o", q.multiply_mdag_e_o),
                         ("hermop_sym2", q.multiply_hermop_sym2)):
            assert rel(fn(None, f, inv).data, orc.apply_half(name, x, eo)) < 1e-12, name
    y = q.FermionField5d(geo, ls, 0)
    y.data = rand_field((geo.total_volume(), ls, 12), 41)
    assert rel(q.multiply_d_minus(None, y, inv).data, orc.apply_full("d_minus", y.data)) < 1e-12
