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


@pytest.mark.parametrize("physics", ["ins", "cns"])
def test_update_of_the_fine_mesh_between_restriction_and_prolongation(oracle_mod, physics):
    """The correction is added to the fine state that the updates leave."""
    _case(f"fine updates, mg_prolongate {physics} 32x32 -> 16x16 p=2")
    _, (G, Gc), _ = _stacks(oracle_mod, physics, 32, 1, 2)
    if physics == "cns":
        # the explicit compressible relaxation stays admissible at CFL ~ (8 h)^2 / p^3 0.01
        for x in (G, Gc):
            x.set_cfl([0.01 / 16 / 8] * 4)
    base = G.get_state()
    out = []
    for wait in (False, True):
        G.set_state(*base)
        assert G.setup_preconditioner() == 0
        G.rsdl()
        Gc.mg_restrict()
        assert Gc.setup_preconditioner() == 0
        Gc.update()
        Gc.synchronize()
        for _ in range(20):
            G.update()
        if wait:
            G.synchronize()
        Gc.mg_prolongate()
        out.append([*G.get_state(), *G.get_residual()])
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.array_equal(a, b)


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


def test_error_flags_of_failed_and_good_cycles(oracle_mod):
    """A cycle on a state without a valid pseudo-time step reports it, enqueued and replayed,
    as often as it happens and never afterwards."""
    _case("cycles on good and NaN states, ins 16x16 p=4, 3 grids, graph replay")
    from hpmp import multigrid as MG
    _, g, _ = _stacks(oracle_mod, "ins", 16, 2, 3)
    good = g[0].get_state()
    nan = [x.copy() for x in good]
    nan[0][::7] = np.nan
    want = None
    for k, st in enumerate((good, nan, nan, good, nan, good, good)):
        g[0].set_state(*st)
        if st is nan:
            with pytest.raises(FloatingPointError, match="setup_preconditioner"):
                MG.cycle(g, 2, 2, 2, 2, fused=True)
            continue
        e = MG.cycle(g, 2, 2, 2, 2, fused=True)
        assert want is None or e == want
        want = e
    for x in g:
        assert x.setup_preconditioner() == 0


def _failing_call(lib, call):
    """``call`` with an error of an unrelated HIP call pending in this thread: its kernels are
    enqueued, then it reports that error."""
    from hpmp import _lib
    assert lib.hipSetDevice(1 << 20) != 0
    with pytest.raises(_lib.HpgError):
        call()
    lib.hipGetLastError()


def test_flag_of_a_setup_that_was_not_read_is_dropped(oracle_mod):
    _case("setup and cycle that end before their error flag is read")
    import test_gpu_tet_cns as C
    from hpmp import multigrid as MG
    _, g, _ = _stacks(oracle_mod, "ins", 8, 1, 2)
    good = g[0].get_state()
    g[0].set_state(np.full_like(good[0], np.nan), *good[1:])
    _failing_call(g[0].L, lambda: MG.cycle(g, 1, fused=True))
    g[0].set_state(*good)
    assert g[0].setup_preconditioner() == 0
    _, st, G, _ = C._pair(2, 1)
    G.set_state(np.full_like(st[0], np.nan), st[1])
    _failing_call(G.L, G.setup_preconditioner)
    G.set_state(*st)
    assert G.setup_preconditioner() == 0
