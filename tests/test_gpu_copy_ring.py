"""Host arrays of sizes at the edges of the staging ring's pieces, with the
ring made: it is there from the third transfer on, as long as an inverter
lives."""

import numpy as np
import pytest
import torch

import qlattice_amd as q
from qlattice_amd import _lib
from tests.helpers import rand_gauge

pytestmark = pytest.mark.gpu


def make(site, ls):
    geo = q.Geometry(site)
    gf = q.GaugeField(geo)
    gf.data = rand_gauge(site, 0.3, 5)
    return geo, q.InverterDomainWall(gf=gf, fa=q.FermionAction(mass=0.05, ls=ls, m5=1.8, mobius_scale=2.0))


def apply_both(geo, inv, ls, seed):
    """Mpc^+ Mpc of a host field and of the same field in device memory."""
    f = q.FermionField5d(geo, ls, 1)
    g = np.random.Generator(np.random.PCG64(seed))
    f.data = g.standard_normal(f.data.shape) + 1j * g.standard_normal(f.data.shape)
    x = torch.from_numpy(f.data).cuda()
    out = torch.empty_like(x)
    _lib.load().multiply_hermop_sym2_device(inv.cdata, _lib.dev_ptr(out), _lib.dev_ptr(x), 1)
    torch.cuda.synchronize()
    return q.multiply_hermop_sym2(None, f, inv).data, out.cpu().numpy()


@pytest.fixture(scope="module")
def ring():
    """An inverter kept alive past the first transfers; every one, before and
    after the ring is made, arrives whole."""
    print("\n[gpu] host copies until the ring is made", flush=True)
    geo, inv = make((8, 8, 16, 16), 8)
    for i in range(4):
        a, b = apply_both(geo, inv, 8, i)
        assert np.array_equal(a, b)
    return inv


# pieces of 2 MiB: 4.1 MiB (three pieces, the last short), 6 (exactly three),
# 7.5 (four), 11.8 (six), 16.5 (nine, one more than the ring), 34 and 46
@pytest.mark.parametrize("site,ls", [((6, 6, 8, 12), 13), ((8, 8, 8, 16), 8), ((8, 8, 16, 16), 5), ((8, 8, 8, 12), 21),
                                     ((8, 8, 16, 16), 11), ((12, 12, 8, 16), 20), ((12, 12, 12, 24), 12)])
def test_arrays_through_the_ring(ring, site, ls):
    print(f"\n[gpu] host copies {site} Ls{ls}", flush=True)
    geo, inv = make(site, ls)
    for seed in (1, 2):
        a, b = apply_both(geo, inv, ls, seed)
        assert np.array_equal(a, b)
