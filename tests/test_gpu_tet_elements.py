"""Element residual of the p = 2 tets (16 elements per wave): element counts around the
wave's 16 and with a ragged last group, every record form (full and inviscid stages), and
the listed elements of the Jacobian, against the CPU oracle."""
import numpy as np
import pytest

from conftest import rel_err
from test_gpu_tet import RSDL_TOL, _pair

pytestmark = pytest.mark.gpu


# 6 n^3 elements: 6 (one partial group), 48 (three whole groups), 162 and 1296 (remainders 2 and 0)
@pytest.mark.parametrize("n", [1, 2, 3, 6])
@pytest.mark.parametrize("mu", [0.0, 1e-2])
def test_element_residual_sizes(oracle_mod, n, mu):
    print(f"\n[gpu-case] tet elements n={n} mu={mu}", flush=True)
    m, st, G, O = _pair(n, 1, mu=mu, seed=n)
    G.setup_preconditioner()
    O.setup_preconditioner()
    for s in (5, 0, 1, 2, 3):  # full, full, inviscid (compact records), full, inviscid
        G.rsdl(s)
        O.rsdl(s)
        err = rel_err(G.get_residual(), O.get_res())
        print("stage", s, "rel err", err, flush=True)
        assert err < RSDL_TOL


@pytest.mark.parametrize("n", [1, 2, 3, 6])
@pytest.mark.parametrize("mu", [0.0, 1e-2])
def test_cns_element_residual_sizes(oracle_mod, n, mu):
    import test_gpu_tet_cns as C
    print(f"\n[gpu-case] tet cns elements n={n} mu={mu}", flush=True)
    m, st, G, O = C._pair(n, 1, mu=mu, seed=n)
    G.setup_preconditioner()
    O.setup_preconditioner()
    for s in (5, 0, 1, 2, 3):
        G.rsdl(s)
        O.rsdl(s)
        err = rel_err(G.get_residual(), O.get_res())
        print("stage", s, "rel err", err, flush=True)
        assert err < C.RSDL_TOL
