"""The FP16-storage hop kernels where their site blocks, neighbour table and
power-of-two scales can go wrong: volumes that end inside a block, every
block shape, lattices of extent 2, and inputs far from 1."""

import numpy as np
import pytest

import qlattice_amd as q
from tests.helpers import rand_field, rand_gauge, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sb", [8, 16, 32])
@pytest.mark.parametrize("site,ls,scale", [((2, 2, 6, 10), 8, 2.0), ((2, 6, 10, 6), 12, 0.0), ((4, 6, 2, 14), 24, 2.0),
                                           ((6, 2, 2, 2), 5, 2.0)])
def test_fp16_hermop_on_ragged_blocks(monkeypatch, site, ls, scale, sb):
    """Mpc^+ Mpc rounds its input and three intermediate fields to 11 bits of
    the site's largest component and the FP16 links likewise: four passes of
    sqrt(24) * 2^-12 or less against the site's norm and as much from the
    links, times the operator's growth of the first errors (below 2 on these
    fields), is below 3e-3.  A power of two in the input passes through
    exactly."""
    print(f"\n[gpu] FP16 hermop {site} Ls{ls} blocks of {sb}", flush=True)
    monkeypatch.setenv("QLAT_DWF_TP_SB", str(sb))
    geo = q.Geometry(site)
    gf = q.GaugeField(geo)
    gf.data = rand_gauge(site, 0.4, 7)
    omega = None if scale else [complex(0.6 + 0.1 * s, 0.02 * s) for s in range(ls)]
    fa = q.FermionAction(mass=0.05, ls=ls, m5=1.8, mobius_scale=scale, omega=omega)
    inv = q.InverterDomainWall(gf=gf, fa=fa, solver="mixed16")
    f = q.FermionField5d(geo, ls, 1)
    x = rand_field((geo.total_volume() // 2, ls, 12), 11)
    f.data = x
    exact = q.multiply_hermop_sym2(None, f, inv).data
    got = q.multiply_hermop_sym2_fp32(None, f, inv).data
    assert rel(got, exact) < 3e-3
    for e in (-60, 30):
        f.data = x * 2.0**e
        assert np.array_equal(q.multiply_hermop_sym2_fp32(None, f, inv).data, got * 2.0**e)
