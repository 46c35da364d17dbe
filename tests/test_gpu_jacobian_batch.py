"""Batched ins element Jacobians at the edges of their launch: (element, column) entries in
16-entry groups, slices of 2^25 / N^2 elements, and a first stage without viscous part."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solver(n, log2p, cls=None, **kw):
    from hpmp import mesh as M, workloads as W
    from hpmp.tri_hp import TriHpIns
    m = M.unit_square(n, 0.2, 4)
    st = W.noisy_freestream(m, 1 << log2p, seed=9, scale=0.3)
    g = (cls or TriHpIns)(m, log2p=log2p, mu=1e-2, **kw)
    g.set_state(*st)
    return m, g


@pytest.mark.parametrize("log2p,nel", [(0, 1), (0, 7), (1, 3), (1, 33), (2, 1), (2, 17)])
def test_batch_edges_match_the_oracle_with_inviscid_first_stage(oracle_mod, log2p, nel):
    print(f"element jacobian log2p={log2p} nel={nel} beta0=0", flush=True)
    beta = (0.0, 1.0, 5.0 / 9.0, 0.0, 4.0 / 9.0)
    m, g = _solver(5, log2p, beta=beta)
    _, o = _solver(5, log2p, oracle_mod.TriHpIns, beta=beta)
    t = np.random.default_rng(nel).choice(m.ntri, nel, replace=False)
    K = g.element_jacobian(t, 1e-4, 1e-4)
    for j, e in enumerate(t):
        Ko = o.element_jacobian(int(e), 1e-4, 1e-4)
        # residual rounding 1e-14 over a step of 1e-4
        assert np.abs(K[j] - Ko).max() <= 1e-9 * np.abs(Ko).max()


def test_slices_of_a_large_batch():
    print("element jacobian over two slices", flush=True)
    m, g = _solver(92, 2)
    cut = (1 << 25) // 45 ** 2   # elements of the first slice
    assert cut < m.ntri
    t = np.random.default_rng(1).permutation(m.ntri)[:cut + 5]
    K = g.element_jacobian(t)
    for j in (0, cut - 1, cut, cut + 4):
        assert np.array_equal(K[j], g.element_jacobian([t[j]])[0])
