"""The QED operator, one thread per (site, s, spin), at its edges: extents of
1 and odd ones, Ls 1 (both walls on one slice) and 2, element counts that are
no multiple of a block, with and without Wick phases, against the numpy
restatement; and the queued iterations of its CG at their limits."""

import numpy as np
import pytest

import qlattice_amd as q
from oracle import qed as Q
from tests.helpers import rel

pytestmark = pytest.mark.gpu


def fields(site, ls, seed):
    rng = np.random.default_rng(seed)
    V = int(np.prod(site))
    g = np.exp(1j * rng.uniform(0, 2 * np.pi, (V, 4))) * (1 + 0.2 * rng.standard_normal((V, 4)))
    wick = 1.1 * np.exp(1j * rng.uniform(-0.3, 0.3, site[3]))
    return g, wick, rng.standard_normal((V, ls, 4)) + 1j * rng.standard_normal((V, ls, 4))


# the bar of tests/test_gpu_qed.py for one application
@pytest.mark.parametrize("site,ls", [((1, 3, 2, 5), 1), ((3, 1, 5, 2), 2), ((2, 2, 1, 1), 3), ((5, 3, 7, 3), 5),
                                     ((4, 4, 4, 8), 8)])
@pytest.mark.parametrize("dag", [False, True])
@pytest.mark.parametrize("phases", [False, True])
def test_operator_edges(site, ls, dag, phases):
    g, wick, x = fields(site, ls, 5 + ls)
    w = wick if phases else None
    got = q.multiply_m_dwf_qed(x, g, 0.1, 1.8, ls, site, w, dag)
    assert rel(got, Q.multiply_m_dwf_qed(x, g, 0.1, 1.8, ls, site, w, dag)) < 1e-13


@pytest.mark.parametrize("limit", [1, 2, 3, 4, 7])
def test_cg_limits(limit):
    """After a few iterations the iterates of both sides still agree to
    rounding (1e-13 an application, a few applications each)."""
    site, ls = (3, 4, 2, 5), 4
    g, wick, x = fields(site, ls, 9)
    sol, it = q.cg_with_m_dwf_qed(x, g, 0.1, 1.0, ls, site, wick, False, 1e-10, limit)
    ref, it_ref = Q.cg_with_m_dwf_qed(x, g, 0.1, 1.0, ls, site, wick, False, 1e-10, limit)
    assert it == it_ref == limit + 1
    assert rel(sol, ref) < 1e-11


@pytest.mark.parametrize("bad", [0.0, np.nan, 1e200])
def test_cg_ends_where_the_residual_is_not_finite(bad):
    """A zero source (alpha = 0/0), a NaN and a norm that overflows: no later
    iteration can converge, so the solve returns at once, with the count that
    says so, whatever its limit (at 1e9 iterations it would take hours)."""
    site, ls, limit = (3, 4, 2, 5), 4, 10**9
    g, wick, x = fields(site, ls, 9)
    x[7, 1, 2] = bad
    if bad == 0.0:
        x[:] = 0.0
    print(f"\n[gpu] QED CG, source with {bad}", flush=True)
    sol, it = q.cg_with_m_dwf_qed(x, g, 0.1, 1.0, ls, site, wick, False, 1e-10, limit)
    assert it == limit + 1
    if bad == 0.0:
        out, it = q.invert_dwf_qed(x[:, 0], g, 0.1, 1.0, ls, site, wick, False, 1e-10, limit)
        assert it == limit + 1
