"""Boundary-edge fluxes inside the element launch: one edge block (4 edges), the block edge
(256 and 260 edges) and boundary lists that name a side twice."""
import dataclasses

import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log2p", [0, 1, 2])
@pytest.mark.parametrize("n", [1, 64, 65])
def test_edges_at_block_edges(oracle_mod, n, log2p):
    print(f"edge blocks n={n} log2p={log2p}", flush=True)
    from hpmp import mesh as M, workloads as W
    from hpmp.tri_hp import TriHpIns
    m = M.unit_square(n, 0.2, 3, essential_mask=0)
    st = W.noisy_freestream(m, 1 << log2p, seed=n, scale=0.3)
    g, o = TriHpIns(m, log2p=log2p, mu=1e-2), oracle_mod.TriHpIns(m, log2p=log2p, mu=1e-2)
    for x in (g, o):
        x.set_edge_flux([2] * m.nebd, (1.0, 0.1, 0.2))
        x.set_state(*st)
        x.rsdl()
    ro = o.get_res()
    assert rel_err(g.get_residual(), ro) < 1e-12
    # FP32 element residual: about 200 roundings of terms of the residual's size
    assert rel_err(g.residual_fp32(), ro) < 200 * 2.0 ** -23


def test_side_listed_twice_counts_twice():
    print("boundary side in two lists", flush=True)
    from hpmp import mesh as M, workloads as W
    from hpmp.tri_hp import TriHpIns
    m = M.unit_square(3, 0.2, 3, essential_mask=0)
    st = W.noisy_freestream(m, 4, seed=2, scale=0.3)
    twice = dataclasses.replace(m, ebdry_start=np.append(m.ebdry_start, m.ebdry_start[-1] + 1).astype(np.int32),
                                ebdry_seg=np.append(m.ebdry_seg, m.ebdry_seg[1]).astype(np.int32),
                                ebdry_essential=np.append(m.ebdry_essential, 0).astype(np.int32))
    none = dataclasses.replace(m, ebdry_start=np.zeros(1, np.int32), ebdry_seg=np.zeros(0, np.int32),
                               ebdry_essential=np.zeros(0, np.int32))
    only = dataclasses.replace(m, ebdry_start=np.array([0, 1], np.int32), ebdry_seg=m.ebdry_seg[1:2],
                               ebdry_essential=np.zeros(1, np.int32))
    r = {}
    for k, q in (("m", m), ("twice", twice), ("none", none), ("only", only)):
        g = TriHpIns(q, log2p=2, mu=1e-2)
        g.set_state(*st)
        g.rsdl()
        r[k] = g.get_residual()
    want = [a + (b - c) for a, b, c in zip(r["m"], r["only"], r["none"])]
    assert rel_err(r["twice"], want) < 1e-12


@pytest.mark.parametrize("n", [223, 224])
def test_fp32_edges_on_both_sides_of_their_own_launch(n):
    """p = 4 in FP32: 99 458 elements take the edges in the element launch, 100 352 in one of
    their own, against the FP64 residual."""
    print(f"fp32 edges n={n}", flush=True)
    from hpmp import mesh as M, workloads as W
    from hpmp.tri_hp import TriHpIns
    m = M.unit_square(n, 0.2, 3, essential_mask=0)
    st = W.noisy_freestream(m, 4, seed=n, scale=0.3)
    g = TriHpIns(m, log2p=2, mu=1e-2)
    g.set_edge_flux([2] * m.nebd, (1.0, 0.1, 0.2))
    g.set_state(*st)
    g.rsdl()
    r, f = g.get_residual(), g.residual_fp32()
    b = np.unique(m.ebdry_seg)
    # FP32 element residual: about 200 roundings of terms of the residual's size
    assert rel_err([f[1][b]], [r[1][b]]) < 200 * 2.0 ** -23
    assert rel_err(f, r) < 200 * 2.0 ** -23
