"""State exchange through the staging slots: the size classes and their edges, several
contexts and threads at once, and null arrays."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _roundtrip(n, log2p, seed):
    from hpmp import mesh as M
    from hpmp.tri_hp import TriHpIns
    g = TriHpIns(M.unit_square(n, 0.2, 1), log2p=log2p, mu=1e-3)
    rng = np.random.default_rng(seed)
    for _ in range(3):
        st = [rng.standard_normal(s) for s in g.shapes()]
        g.set_state(*st)
        r = [rng.standard_normal(s) for s in g.shapes()]
        g.set_residual(*r)
        for a, b in zip(g.get_state(), st):
            assert np.array_equal(a, b)
        for a, b in zip(g.get_residual(), r):
            assert np.array_equal(a, b)
    return sum(x.nbytes for x in st)


# one small kernel (up to 256 KiB), direct (to 2 MiB), threads (above; 1 MiB chunks)
@pytest.mark.parametrize("n,log2p", [(1, 0), (1, 2), (25, 2), (26, 2), (72, 2), (74, 2), (120, 1), (150, 2)])
def test_roundtrip_over_size_classes(n, log2p):
    print(f"exchange n={n} log2p={log2p}: {_roundtrip(n, log2p, n)} bytes", flush=True)


def test_contexts_in_threads():
    print("exchange from six threads", flush=True)
    bad = []

    def run(k):
        try:
            _roundtrip((3, 40, 110)[k % 3], 2, k)
        except BaseException as e:  # reported below
            bad.append(repr(e))
    th = [threading.Thread(target=run, args=(k,)) for k in range(6)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad


def test_null_array_is_an_error():
    import ctypes as C
    from hpmp import mesh as M
    from hpmp.tri_hp import TriHpIns
    g = TriHpIns(M.unit_square(2, 0.2, 1), log2p=1, mu=1e-3)
    v = np.zeros(g.shapes()[0])
    assert g.L.hpg_set_state(g.h, C.c_void_p(v.ctypes.data), C.c_void_p(0), C.c_void_p(0)) == -1
    assert b"null" in g.L.hpg_last_error(g.h)
