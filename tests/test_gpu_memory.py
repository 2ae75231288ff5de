"""The device memory an ensemble takes for a row, against what the request loop admits
members by (sphgpu_ensemble_bytes_per_node)."""
import ctypes as C

import pytest

from sphgpu import problems

pytestmark = pytest.mark.gpu

STATES = {1: lambda k: [problems.random_state(1, int(n * k), seed=n, jitter=0.1)[0] for n in (1000000, 1300000)],
          2: lambda k: [problems.random_state(2, int(n * k ** 0.5), seed=n, jitter=0.1)[0] for n in (700, 800)],
          3: lambda k: [problems.random_state(3, int(n * k ** (1 / 3)), seed=n, jitter=0.1)[0] for n in (70, 80)]}


def free_bytes():
    hip = C.CDLL("libamdhip64.so")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def footprint(sg, dim, states, precision):
    """(bytes, rows) of an ensemble that has stepped and lost a member."""
    before = free_bytes()
    e = sg.Sim(dim)
    e.set_row_order(sg.ROW_ORDER_SEARCH)
    e.set_table_bspline(1000)
    e.set_precision(precision)
    e.set_boundaries(sg.box_boundaries(dim))
    e.ensemble_begin()
    ip = sg.integrator_params(gamma=1.4)
    ids = [e.ensemble_add({k: st[k] for k in ("pos", "vel", "mass", "rho", "eps", "H")}, 1.4, 1.0, ip) for st in states]
    hp = sg.hydro_params(precision=precision)
    for _ in range(3):
        e.ensemble_step(hp, ip)
    rows = e.node_counts()[1]
    e.ensemble_remove(ids[:1])
    e.ensemble_step(hp, ip)
    used = before - free_bytes()
    e.close()
    return used, rows


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("dim", [1, 2, 3])
def test_bytes_per_row(sphgpu, dim, precision):
    """Between two sizes, so that what does not grow with the rows drops out; 2.5 % for
    the slots of culled ghosts and the allocations' granules."""
    (b1, n1), (b2, n2) = (footprint(sphgpu, dim, STATES[dim](k), precision) for k in (1.0, 2.5))
    per = (b2 - b1) / (n2 - n1)
    sim = sphgpu.Sim(dim)
    declared = sim.L.sphgpu_ensemble_bytes_per_node(dim)
    sim.close()
    print(f"[memory] {dim}-D precision {precision}: {per:.0f} B a row, declared {declared}", flush=True)
    assert per <= 1.025 * declared
    assert per >= 0.8 * declared
