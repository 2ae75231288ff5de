"""The dt vote of mixed 3-D steps on both sides of its size rule, and of ensemble members,
against the vote that gathers every velocity: the same dt to the bit."""
import numpy as np
import pytest

import test_gpu_dispatch as dispatch
from sphgpu import problems

pytestmark = pytest.mark.gpu


def gathered_vote(sg, st):
    s = dispatch.make(sg, 3, st, order=1, precision=1)
    s.eos_gamma_law(1.4)
    s.set_boundaries(sg.box_boundaries(3))
    s.set_ghost_nodes(2.0)
    vote = s.hydro_dt(1.51, 0.25)
    s.close()
    return vote


@pytest.mark.parametrize("n,scale", [(50, 20.0), (50, 0.2), (37, 20.0), (25, 20.0)])
def test_vote_below_the_bounds(sphgpu, n, scale):
    """125000, 50653 and 15625 nodes: the velocities packed by slot are gathered."""
    print(f"[vote] n={n} scale={scale}", flush=True)
    st, _ = problems.random_state(3, n, seed=910 + n, jitter=0.1, vel_scale=scale, h_var=0.1)
    dispatch.test_mixed_vote_bounds(sphgpu, (f"{n}^3", st))


def test_vote_of_members_by_bounds(sphgpu):
    """Two members of 68921 nodes, together beyond the line: each member's dt is its own
    vote.  One member is fast throughout, the other has one fast node."""
    print("[vote] members", flush=True)
    states = []
    for seed, scale in ((920, 5.0), (921, 0.05)):
        st, _ = problems.random_state(3, 41, seed=seed, jitter=0.1, vel_scale=scale, h_var=0.1)
        st = {k: st[k] for k in ("pos", "vel", "mass", "rho", "eps", "H")}
        st["eps"] = st["eps"] * 1.0e-12              # the sound speed limits nothing
        states.append(st)
    states[1]["vel"][33333] = [3.0, -2.0, 1.0]
    votes = [gathered_vote(sphgpu, st) for st in states]
    assert votes[0] != votes[1]
    ip = sphgpu.integrator_params(gamma=1.4, dtGrowth=1.0e30)
    e = sphgpu.Sim(3)
    e.set_row_order(sphgpu.ROW_ORDER_SEARCH)
    e.set_table_bspline(1000)
    e.set_precision(sphgpu.PRECISION_MIXED)
    e.set_boundaries(sphgpu.box_boundaries(3))
    e.ensemble_begin()
    ids = [e.ensemble_add(st, 1.4, 1.0e3, ip) for st in states]
    for i in ids:
        e.ensemble_set_clock(i, 0.0, 1.0e30, 0)
    e.ensemble_step(sphgpu.hydro_params(precision=sphgpu.PRECISION_MIXED), ip)
    assert not e.ensemble_failed()
    got = {m["id"]: m["last_dt"] for m in e.ensemble_members()}
    assert [got[i] for i in ids] == votes
    e.close()
