"""Neighbour grids of a few nodes far apart: tens of millions of empty cells, on both
sides of the cell scan's size rule (33554432 cells), against the oracle's rows."""
import numpy as np
import pytest

from sphgpu import problems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [33554431, 33554432, 33554433, 33554432 + 2048, 60000000])
def test_cells_on_a_line(sphgpu, oracle, cells):
    """1-D, search radius 1 (and the search's margin): the last node's place sets the
    number of cells."""
    print(f"[sparse] 1-D {cells} cells", flush=True)
    R = 1.0 * (1.0 + 1.0e-6) * (1.0 + 1.0e-9)
    rng = np.random.default_rng(5)
    N = 1200
    clumps = np.sort(rng.uniform(0.0, 100.0, (3, N // 3)), axis=1) + np.array([[0.0], [0.37 * cells], [cells - 150.0]])
    pos = np.concatenate([[0.0], clumps.ravel()[1:-1], [(cells - 0.5) * R]])[:, None]
    check(sphgpu, oracle, 1, pos, np.full((N, 1), 2.0))


@pytest.mark.parametrize("dim,n,far", [(2, 20, 900.0), (3, 6, 90.0)])
def test_cells_of_far_clumps(sphgpu, oracle, dim, n, far):
    """Two clumps on the diagonal of a plane and of a box."""
    print(f"[sparse] {dim}-D", flush=True)
    st, _ = problems.random_state(dim, n, seed=6, jitter=0.2)
    pos = st["pos"] + np.where(st["pos"][:, :1] > 0.5, far, 0.0)
    check(sphgpu, oracle, dim, pos, st["H"])


def check(sg, oracle, dim, pos, H):
    N = pos.shape[0]
    st = dict(pos=pos, H=H, vel=np.zeros_like(pos), mass=np.full(N, 1.0 / N), rho=np.ones(N), eps=np.ones(N))
    off, nbr = oracle.connectivity(dim, N, pos, H)
    rho = oracle.sum_density(oracle.Table(dim, 1000), N, pos, st["mass"], H, off, nbr, gather=True)
    s = sg.Sim(dim)
    s.set_row_order(sg.ROW_ORDER_REFERENCE)
    s.set_table_bspline(1000)
    s.set_nodes(N, N)
    s.upload_state(st)
    for _ in range(2):
        s.build_neighbors(2.0)
        o2, n2 = s.neighbors()
        assert np.array_equal(o2, off) and np.array_equal(n2, nbr)
    s.sum_density()
    assert np.array_equal(s.download("mass density", rows=N), rho)
    s.close()
