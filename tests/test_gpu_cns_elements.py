"""cns element residual on the matrix cores: 16-element groups (2, 18 and 130 elements), every
order, the low-Mach, sonic and inviscid branches of tau, and inadmissible states."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu
INFLOW = 0b1110


def _pair(oracle_mod, n, log2p, mach, mu, seed=3):
    from hpmp import mesh as M, workloads as W
    from hpmp.tri_hp import TriHpCns
    m = M.unit_square(n, 0.2, 2, essential_mask=INFLOW)
    st, bc = W.cns_gaussian_state(m, 1 << log2p, seed=seed, mach=mach, amp=0.05, width=0.3, noise=2e-2)
    g = TriHpCns(m, log2p=log2p, mu=mu, bc=bc)
    o = oracle_mod.TriHpCns(m, log2p=log2p, mu=mu, bc=bc)
    return m, st, g, o


@pytest.mark.parametrize("log2p", [0, 1, 2])
@pytest.mark.parametrize("n", [1, 3, 65])
@pytest.mark.parametrize("mach,mu", [(0.3, 1e-3), (0.0, 1e-2), (1.0, 1e-3), (1.7, 0.0), (0.5, 0.0)])
def test_residual_over_regimes(oracle_mod, n, log2p, mach, mu):
    print(f"cns residual n={n} log2p={log2p} mach={mach} mu={mu}", flush=True)
    m, st, g, o = _pair(oracle_mod, n, log2p, mach, mu)
    for x in (g, o):
        x.set_state(*st)
    for stage in (0, 1, 2, g.nstage):
        g.rsdl(stage)
        o.rsdl(stage)
        # fluxes of size gamma / (gamma - 1) p summed over at most 25 points and 6 elements,
        # relative to the largest residual (0.05 p / p^2 of them at least)
        assert rel_err(g.get_residual(), o.get_res()) < 2e-12


def test_negative_temperature_gives_nan_where_the_oracle_does(oracle_mod):
    print("cns residual with RT < 0 at one vertex", flush=True)
    m, st, g, o = _pair(oracle_mod, 3, 2, 0.5, 1e-3)
    st[0][5, 3] = -3.0
    for x in (g, o):
        x.set_state(*st)
        x.rsdl()
    for a, b in zip(g.get_residual(), o.get_res()):
        assert np.array_equal(np.isnan(a), np.isnan(b))
        assert np.isnan(b).any() and not np.isnan(b).all()
