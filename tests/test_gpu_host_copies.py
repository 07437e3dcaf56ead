"""Host arrays through the staging ring against the device entry points: the
bytes have to arrive whatever the size, from pinned memory, and while another
thread's transfer holds the ring."""

import threading

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


def field(geo, ls, seed):
    f = q.FermionField5d(geo, ls, 1)
    g = np.random.Generator(np.random.PCG64(seed))
    f.data = g.standard_normal(f.data.shape) + 1j * g.standard_normal(f.data.shape)
    return f


def on_device(f, inv):
    x = torch.from_numpy(f.data).cuda()
    out = torch.empty_like(x)
    _lib.load().multiply_hermop_sym2_device(inv.cdata, _lib.dev_ptr(out), _lib.dev_ptr(x), 1)
    torch.cuda.synchronize()
    return out.cpu().numpy()


# half fields of 0.4, 4.1 (the smallest in the ring: three pieces, the last
# short), 11.8 (six), 7.5 (four), 16.5 (nine, one more than the ring) and 34 MB
@pytest.mark.parametrize("site,ls", [((4, 4, 4, 8), 8), ((6, 6, 8, 12), 13), ((8, 8, 8, 12), 21), ((8, 8, 16, 16), 5),
                                     ((8, 8, 16, 16), 11), ((12, 12, 8, 16), 20)])
def test_host_arrays_arrive_whole(site, ls):
    print(f"\n[gpu] host copies {site} Ls{ls}", flush=True)
    geo, inv = make(site, ls)
    for seed in (1, 2):
        f = field(geo, ls, seed)
        assert np.array_equal(q.multiply_hermop_sym2(None, f, inv).data, on_device(f, inv))
    pinned = torch.from_numpy(f.data).pin_memory()
    g = q.FermionField5d(geo, ls, 1)
    g.data = pinned.numpy()
    assert np.array_equal(q.multiply_hermop_sym2(None, g, inv).data, on_device(f, inv))


def test_threads_share_the_ring():
    print("\n[gpu] host copies from three threads", flush=True)
    site, ls = (8, 8, 16, 16), 8
    work = [(*make(site, ls), field(q.Geometry(site), ls, 10 + i)) for i in range(3)]
    want = [on_device(f, inv) for _, inv, f in work]
    got = [[] for _ in work]

    def run(i):
        for _ in range(6):
            got[i].append(q.multiply_hermop_sym2(None, work[i][2], work[i][1]).data)

    th = [threading.Thread(target=run, args=(i,)) for i in range(3)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for w, g in zip(want, got):
        assert len(g) == 6 and all(np.array_equal(w, x) for x in g)
