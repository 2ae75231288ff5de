"""Replayed steps against eager ones where state outside the graph changes between
replays while every count stays: each step's dt and state bit for bit, with the host's
own uploads and downloads between the replays."""
import numpy as np
import pytest

from sphgpu import problems

pytestmark = pytest.mark.gpu

FIELDS = ("position", "velocity", "mass density", "specific thermal energy", "H", "pressure", "sound speed")


@pytest.mark.parametrize("n", [8, 37])           # eight lanes to a node, and one
def test_position_unit_changes_between_replays(sphgpu, n):
    """3-D mixed precision without boundaries: H uploaded before every step takes the
    search radius across a power of two and back, and with it the unit of the
    records' positions."""
    print(f"[unit] n={n}", flush=True)
    st, _ = problems.random_state(3, n, seed=40 + n, jitter=0.1)
    N = st["pos"].shape[0]
    base = 2.0 * st["H"] / st["H"][0, 0]         # search radius 2 / 2 = 1
    sims = []
    for graphs in (False, True):
        s = sphgpu.Sim(3)
        s.set_row_order(sphgpu.ROW_ORDER_SEARCH)
        s.set_table_bspline(1000)
        s.set_nodes(N, N)
        # spacing 1 / 3.02: 1.51 nodes to a smoothing length of 1/2
        x = {k: st[k] for k in ("vel", "mass", "rho", "eps")}
        s.upload_state(dict(x, pos=st["pos"] * (n / 3.02), H=base))
        s.eos_gamma_law(1.4)
        s.set_precision(sphgpu.PRECISION_MIXED)
        s.set_graphs(graphs)
        sims.append(s)
    a, b = sims
    hp = sphgpu.hydro_params(precision=sphgpu.PRECISION_MIXED)
    ip = sphgpu.integrator_params(gamma=1.4, dtMax=1.0e-4)
    radii = [0.985] * 6 + [1.015] * 6 + [0.99, 1.01, 0.99, 1.01]
    for k, r in enumerate(radii):
        for s in sims:
            s.upload("H", base / r)
        assert a.rk2_step(hp, ip) == b.rk2_step(hp, ip), k
        for f in FIELDS:
            assert np.array_equal(a.download(f, rows=N), b.download(f, rows=N)), (k, r, f)
    captures, replays = b.graph_counts()
    print(f"[unit] {captures} captures, {replays} replays", flush=True)
    assert captures >= 2 and replays >= 4


def test_slot_lists_grow_between_replays(sphgpu):
    """2-D mixed precision, two NodeLists: a step with more ghosts, and so more slots,
    than any before it with lists comes between replays with fewer.  The records were
    sized by steps without lists before, so only the slots' NodeLists grow."""
    print("[slot lists]", flush=True)
    n = 24
    st, _ = problems.random_state(2, n, seed=71, jitter=0.1, vel_scale=0.05)
    N = st["pos"].shape[0]
    state = {k: st[k] for k in ("pos", "vel", "mass", "rho", "eps", "H")}
    hp = sphgpu.hydro_params(precision=sphgpu.PRECISION_MIXED)
    ip = sphgpu.integrator_params(gamma=1.4, dtMax=1.0e-6)
    sims = []
    for graphs in (False, True):
        s = sphgpu.Sim(2)
        s.set_row_order(sphgpu.ROW_ORDER_SEARCH)
        s.set_table_bspline(1000)
        s.set_boundaries(sphgpu.box_boundaries(2))
        s.set_precision(sphgpu.PRECISION_MIXED)
        s.set_graphs(graphs)
        s.set_nodes(N, N)
        s.upload_state(dict(state, H=state["H"] / 2.0))
        s.eos_gamma_law(1.4)
        s.rk2_step(hp, ip)
        s.set_nodes(N, N)
        s.upload_state(state)
        s.set_node_lists([N // 2, N - N // 2])
        s.eos_gamma_law(1.4)
        sims.append(s)
    a, b = sims
    counts = []
    for k, wide in enumerate([0] * 6 + [1] * 6 + [0, 1] * 3):
        for s in sims:
            s.upload("position", state["pos"])
            s.upload("H", state["H"] / (1.9 if wide else 1.0))
        assert a.rk2_step(hp, ip) == b.rk2_step(hp, ip), k
        counts.append(b.node_counts())
        assert a.node_counts() == counts[-1], k
        for f in FIELDS:
            assert np.array_equal(a.download(f, rows=N), b.download(f, rows=N)), (k, f)
    captures, replays = b.graph_counts()
    print(f"[slot lists] {sorted(set(counts))}, {captures} captures, {replays} replays", flush=True)
    assert captures >= 2 and replays >= 4
