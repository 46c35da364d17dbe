"""Element residual at p = 4 (16 elements per wave, a group's data loaded a group ahead):
one partial group, a ragged last group, whole groups, and the full and inviscid stages with
their record lengths, against the CPU oracle."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


# 2 n^2 elements: 2, 18 (16 + 2), 32, 392 (24 groups + 8)
@pytest.mark.parametrize("n", [1, 3, 4, 14])
@pytest.mark.parametrize("mu", [0.0, 1e-2])
def test_element_residual_sizes(oracle_mod, n, mu):
    print(f"\n[gpu-case] ins p=4 elements n={n} mu={mu}", flush=True)
    from hpmp import mesh as M, workloads as W
    from hpmp.tri_hp import TriHpIns
    m = M.unit_square(n, 0.2, 3, essential_mask=0)
    st = W.noisy_freestream(m, 4, seed=n, scale=0.3)
    g, o = TriHpIns(m, log2p=2, mu=mu), oracle_mod.TriHpIns(m, log2p=2, mu=mu)
    for x in (g, o):
        x.set_state(*st)
        assert x.setup_preconditioner() == 0
    for stage in (5, 0, 1, 2, 3):  # full, full, inviscid, full, inviscid
        g.rsdl(stage)
        o.rsdl(stage)
        err = rel_err(g.get_residual(), o.get_res())
        print("stage", stage, "rel err", err, flush=True)
        assert err < 1e-12
