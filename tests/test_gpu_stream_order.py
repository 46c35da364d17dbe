"""Contexts of a multigrid stack have a stream each: what a call leaves queued on one of them
has to be done before a neighbour's stream uses the same arrays."""
import numpy as np
import pytest

from test_gpu_hmg import _case, _stacks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("physics", ["ins", "cns"])
def test_upload_to_the_fine_mesh_between_restriction_and_prolongation(oracle_mod, physics):
    """mg_prolongate runs on the coarse stream and adds to the fine state: to the uploaded one."""
    _case(f"set_state, set_residual, mg_prolongate {physics} 8x8 -> 4x4 p=2")
    _, (G, Gc), _ = _stacks(oracle_mod, physics, 8, 1, 2)
    base, res = G.get_state(), [1e-3 * np.random.default_rng(3).standard_normal(s) for s in G.shapes()]
    st = [1.0 + 0.1 * np.random.default_rng(7).standard_normal(s) for s in G.shapes()]
    out = []
    for wait in (False, True):
        G.set_state(*base)
        G.set_residual(*res)
        Gc.mg_restrict()
        assert Gc.setup_preconditioner() == 0
        Gc.update()
        for _ in range(3):
            G.set_state(*st)
            G.set_residual(*st)
        if wait:
            G.synchronize()
            Gc.synchronize()
        Gc.mg_prolongate()
        out.append([*G.get_state(), *G.get_residual()])
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    assert not np.array_equal(out[0][0], st[0])  # the correction is not zero


def test_upload_to_a_coarse_mesh_before_a_replayed_cycle(oracle_mod):
    """A replayed cycle runs on the fine stream and overwrites the coarse states: an upload to
    a coarse context just before it lands before it."""
    _case("coarse set_state, set_residual, update before a replayed cycle, ins 16x16 p=4, 3 grids")
    from hpmp import multigrid as MG
    _, ga, _ = _stacks(oracle_mod, "ins", 16, 2, 3)
    _, gb, _ = _stacks(oracle_mod, "ins", 16, 2, 3)
    rng = np.random.default_rng(11)
    for k in range(6):
        for g in ga[1:]:
            junk = [rng.standard_normal(s) for s in g.shapes()]
            g.set_state(*junk)
            g.set_residual(*junk)
            g.update()
        ea = MG.cycle(ga, 2, 2, 2, 2, fused=True)
        eb = MG.cycle(gb, 2, 2, 2, 2, fused=True)
        assert ea == eb
        for x, y in zip(ga[0].get_state(), gb[0].get_state()):
            assert np.array_equal(x, y)
