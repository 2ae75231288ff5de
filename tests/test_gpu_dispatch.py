"""Both sides of every size rule of the device code, against the oracle.

Several lanes to a node, the scans' tiles, the search's workgroups and stage, the
row sort's widths, the dt vote's bounds, the isotropy test and the large downloads
each change their path at a size; the sizes here are the last of one path and the
first of the next.  Bars as elsewhere: neighbour rows identical, reference row order
equal value for value (cube-root fields in 3-D 1e-14), search row order 1e-12, mixed
precision 1e-5, votes and copies exact.
"""
import numpy as np
import pytest

from sphgpu import problems

pytestmark = pytest.mark.gpu

POW_FIELDS = ("weightedNeighborSum", "Hideal")
STATE = ("position", "velocity", "mass density", "specific thermal energy", "H")


def make(sg, dim, st, order=0, precision=0):
    N = st["pos"].shape[0]
    s = sg.Sim(dim)
    s.set_row_order(order)
    s.set_table_bspline(1000)
    s.set_precision(precision)
    s.set_nodes(N, N)
    s.upload_state(st)
    return s


def rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


# nodes: 1-D 32768 | 32769; 2-D 16384 | 16641, 65536 | 66049, 81796 | 82369; 3-D 15625 | 17576,
# 46656 | 50653, 64000 | 68921, 79507 | 85184, 125000 | 132651, 157464 | 166375
SIZES = [(1, 32768), (1, 32769), (2, 128), (2, 129), (2, 256), (2, 257), (2, 286), (2, 287), (3, 25), (3, 26),
         (3, 36), (3, 37), (3, 40), (3, 41), (3, 43), (3, 44), (3, 50), (3, 51), (3, 54), (3, 55)]


@pytest.mark.parametrize("dim,n", SIZES)
def test_pass_across_lanes(sphgpu, oracle, dim, n):
    """Rows of uneven length on both sides of the lanes' lines: neighbours, sum
    density, grad-h correction, every derivative field and the pair count, in
    both row orders and mixed precision."""
    st, _ = problems.random_state(dim, n, seed=300 + n, jitter=0.2, h_var=0.15)
    N = st["pos"].shape[0]
    print(f"[lanes] dim={dim} N={N}", flush=True)
    off, nbr = oracle.connectivity(dim, N, st["pos"], st["H"])
    T = oracle.Table(dim, 1000)
    rho = oracle.sum_density(T, N, st["pos"], st["mass"], st["H"], off, nbr, gather=True)
    full = dict(st, rho=rho)
    ref = oracle.eval_derivs(T, oracle.make_params(), N, full, off, nbr, gather=True)
    om = oracle.omega_gradh(T, N, st["pos"], st["H"], off, nbr)
    pairs = int((np.repeat(np.arange(N), np.diff(off)) < nbr).sum())
    for order, precision, tol in ((0, 0, 0.0), (1, 0, 1e-12), (1, 1, 1e-5)):
        s = make(sphgpu, dim, st, order, precision)
        s.build_neighbors(2.0)
        o2, n2 = s.neighbors()
        assert np.array_equal(o2, off) and np.array_equal(n2, nbr)
        s.sum_density()
        got = s.download("mass density", rows=N)
        assert np.array_equal(got, rho) if order == 0 else rel(got, rho) <= tol
        s.upload("mass density", rho)
        s.evaluate_derivatives(sphgpu.hydro_params(precision=precision))
        assert s.pair_count() == pairs
        if dim == 1 and precision:
            continue                                 # |grad W|^2/r^6 at 3e-5 spacing leaves the FP32 range
        for f in sphgpu.DERIV_ALIASES:
            a = s.derivative(f).reshape(ref[f].shape)
            if order == 0 and not (dim == 3 and f in POW_FIELDS):
                assert np.array_equal(a, ref[f]), f
            else:
                assert rel(a, ref[f]) <= (tol if order else 1e-14), (f, order, precision)
        if order == 0:
            s.omega_gradh()
            assert np.array_equal(s.download("grad h corrections", rows=N), om)
        s.close()


@pytest.mark.parametrize("dim,n", [(2, 128), (2, 221), (2, 222), (3, 25), (3, 43), (3, 44)])
def test_ideal_h_across_lanes(sphgpu, oracle, dim, n):
    """iterateIdealH at 16 lanes to a node, 8 and one (2-D 48841 | 49284, 3-D 79507
    | 85184 nodes), nodes that are done leaving the iteration early."""
    import integrator
    st, _ = problems.random_state(dim, n, seed=400 + n, jitter=0.2, h_var=0.3)
    N = st["pos"].shape[0]
    print(f"[ideal H lanes] dim={dim} N={N}", flush=True)
    Hr, itr, mdr = integrator.iterate_ideal_h(dim, {k: st[k] for k in ("pos", "mass", "rho", "H")},
                                              oracle.box_boundaries(dim), max_iterations=3, tolerance=1.0e-2)
    s = make(sphgpu, dim, st)
    s.set_boundaries(sphgpu.box_boundaries(dim))
    it, md = s.iterate_ideal_h(sphgpu.hydro_params(), 3, 1.0e-2)
    assert it == itr
    Hd = s.download("H", rows=N).reshape(Hr.shape)
    assert np.array_equal(Hd, Hr) if dim < 3 else rel(Hd, Hr) <= 1e-12


@pytest.mark.parametrize("dim,n", [(2, 128), (2, 129), (3, 25), (3, 26)])
def test_compatible_energy_across_lanes(sphgpu, oracle, dim, n):
    """A step with compatible energy at 16 lanes to a node and at 8."""
    import integrator
    st, _ = problems.random_state(dim, n, seed=500 + n, jitter=0.2, h_var=0.1)
    N = st["pos"].shape[0]
    print(f"[compatible lanes] dim={dim} N={N}", flush=True)
    base = {k: st[k] for k in ("pos", "vel", "mass", "rho", "eps", "H")}
    ref = integrator.RK2(dim, base, oracle.box_boundaries(dim), 1.4, compatible=True)
    s = make(sphgpu, dim, base)
    s.eos_gamma_law(1.4)
    s.set_boundaries(sphgpu.box_boundaries(dim))
    dref = ref.step()
    ddev = s.rk2_step(sphgpu.hydro_params(compatibleEnergyEvolution=1), sphgpu.integrator_params(gamma=1.4))
    assert ddev == dref if dim < 3 else ddev == pytest.approx(dref, rel=1e-12)
    for key, f in zip(("pos", "vel", "rho", "eps", "H"), STATE):
        a, b = s.download(f, rows=N).reshape(ref.st[key].shape), ref.st[key]
        assert np.array_equal(a, b) if dim < 3 else rel(a, b) <= 1e-12, key


def test_members_and_plain_runs_take_different_lanes(sphgpu):
    """Members of 12100 and 8281 nodes (16 lanes to a node alone, 8 together) keep
    their plain runs' bits."""
    from test_gpu_ensemble import check_same, ensemble, plain_run, run_ensemble
    members = [dict(state=problems.point_blast(n, seed=700 + n), gamma=5.0 / 3.0, t_end=2.0e-5) for n in (110, 91)]
    hp = sphgpu.hydro_params()
    for order in (sphgpu.ROW_ORDER_REFERENCE, sphgpu.ROW_ORDER_SEARCH):
        print(f"[members lanes] order={order}", flush=True)
        e = ensemble(sphgpu, 2, order)
        got = run_ensemble(sphgpu, e, members, hp, {})
        e.close()
        for q, m in enumerate(members):
            ref, steps = plain_run(sphgpu, 2, m["state"], m["gamma"], m["t_end"], hp, {}, order)
            assert got[q][1] == steps
            check_same(got[q][0], ref, q)


def search_cases():
    out = []
    for dim, n in ((1, 65536), (1, 65537), (2, 90), (2, 200)):     # smoothing scales over a factor 12: level grids
        st, _ = problems.random_state(dim, n, seed=600 + n, jitter=0.1)
        r = np.sqrt(((st["pos"] - 0.5) ** 2).sum(1))
        st["H"] = st["H"] / (1.0 + 11.0 * np.exp(-(r / 0.05) ** 2))[:, None]
        out.append((f"levels{dim}d{n}", dim, st))
    for dim, n in ((2, 60), (2, 181), (2, 257), (3, 12), (3, 40), (3, 41)):
        st, meta = problems.random_state(dim, n, seed=610 + n, jitter=0.2)
        st["H"] = problems.anisotropic_H(dim, st["pos"].shape[0], 1.51 * meta["dx"])
        out.append((f"aniso{dim}d{n}", dim, st))
    # one brick's stage holds all nodes: up to 2239 in LDS, from 2240 on from global
    # memory; rows from 40 to 400 entries, so every width of the row sort
    rng = np.random.default_rng(77)
    for n in (2238, 2239, 2240, 2241):
        pos = rng.uniform(0.0, 1.0, (n, 3))
        h = 0.5 * 0.5 * 2.0 / 5.9
        H = np.zeros((n, 6))
        H[:, [0, 3, 5]] = 1.0 / h
        out.append((f"stage{n}", 3, dict(pos=pos, H=H, vel=np.zeros((n, 3)), mass=np.full(n, 1.0 / n),
                                         rho=np.ones(n), eps=np.ones(n))))
    return out


SEARCH = search_cases()


@pytest.mark.parametrize("case", SEARCH, ids=[c[0] for c in SEARCH])
def test_search_across_lanes_and_stage(sphgpu, oracle, case):
    name, dim, st = case
    N = st["pos"].shape[0]
    print(f"[search] {name} N={N}", flush=True)
    off, nbr = oracle.connectivity(dim, N, st["pos"], st["H"])
    T = oracle.Table(dim, 1000)
    rho = oracle.sum_density(T, N, st["pos"], st["mass"], st["H"], off, nbr, gather=True)
    s = make(sphgpu, dim, st)
    s.build_neighbors(2.0)
    o2, n2 = s.neighbors()
    assert np.array_equal(o2, off) and np.array_equal(n2, nbr)
    assert s.neighbor_count() == off[-1]
    s.sum_density()                                  # the rows' order
    assert np.array_equal(s.download("mass density", rows=N), rho)


@pytest.mark.parametrize("n", [1, 2, 8191, 8192, 8193, 524288, 524289])
def test_ghost_generation_across_scan_tiles(sphgpu, oracle, n):
    """The ghosts of a 1-D box: one scan launch, two with one item a lane, two with
    four."""
    st, _ = problems.random_state(1, n, seed=800 + n % 97, jitter=0.2)
    N = st["pos"].shape[0]
    print(f"[scan] N={N}", flush=True)
    full, off, nbr, info = oracle.ghost_pipeline(1, st, oracle.box_boundaries(1))
    s = make(sphgpu, 1, st)
    s.set_boundaries(sphgpu.box_boundaries(1))
    s.set_ghost_nodes(2.0)
    assert s.node_counts() == (N, full["pos"].shape[0])
    control, sub = s.ghost_controls()
    assert np.array_equal(control, info["control"]) and np.array_equal(sub, info["sub_of"])
    o2, n2 = s.neighbors()
    assert np.array_equal(o2, off) and np.array_equal(n2, nbr)


def vote_cases():
    n = 51                                           # 132651 nodes: the bounds
    out = []
    for name, scale in (("subsonic", 0.2), ("supersonic", 20.0), ("still", 0.0)):
        st, _ = problems.random_state(3, n, seed=900, jitter=0.1, vel_scale=scale, h_var=0.1)
        out.append((name, st))
    st, _ = problems.random_state(3, n, seed=901, jitter=0.1, vel_scale=1.0)
    st["vel"] = 1.0e6 + np.zeros_like(st["vel"])     # one velocity: FP32 differences are zero
    st["vel"][7] += 1.0e-3                           # but one, far below FP32's step
    out.append(("shifted", st))
    st, _ = problems.random_state(3, n, seed=902, jitter=0.1, vel_scale=1.0)
    st["vel"][11] = 3.0e19                           # beyond the bounds' range
    out.append(("huge", st))
    return out


VOTES = vote_cases()


@pytest.mark.parametrize("case", VOTES, ids=[c[0] for c in VOTES])
def test_mixed_vote_bounds(sphgpu, case):
    """A large mixed step's dt equals the vote that gathers every velocity."""
    name, st = case
    print(f"[vote] {name}", flush=True)
    st = {k: st[k] for k in ("pos", "vel", "mass", "rho", "eps", "H")}
    st["eps"] = st["eps"] * 1.0e-12                  # the sound speed limits nothing
    s = make(sphgpu, 3, st, order=1, precision=1)
    s.eos_gamma_law(1.4)
    s.set_boundaries(sphgpu.box_boundaries(3))
    s.set_ghost_nodes(2.0)
    vote = s.hydro_dt(1.51, 0.25)
    s.set_clock(0.0, 1.0e30, 0)
    dt = s.rk2_step(sphgpu.hydro_params(precision=1), sphgpu.integrator_params(gamma=1.4, dtGrowth=1.0e30))
    assert dt == vote


@pytest.mark.parametrize("n", [1023, 1024, 1025])
@pytest.mark.parametrize("dim", [1, 2, 3])
def test_isotropy_of_uploads(sphgpu, dim, n):
    """H = h I is recognised by the host's loop below 1024 rows and the device's from
    there on; mixed precision refuses any other H."""
    rng = np.random.default_rng(n)
    NS = dim * (dim + 1) // 2
    diag = [0] if dim == 1 else ([0, 2] if dim == 2 else [0, 3, 5])
    H = np.zeros((n, NS))
    H[:, diag] = 50.0
    pos = rng.uniform(0, 1, (n, dim))
    s = make(sphgpu, dim, dict(pos=pos, H=H, vel=0 * pos, mass=np.ones(n), rho=np.ones(n), eps=np.ones(n)),
             order=1, precision=1)
    s.eos_gamma_law(1.4)
    s.build_neighbors(2.0)
    s.evaluate_derivatives(sphgpu.hydro_params(precision=1))
    if dim == 1:
        return
    for row, comp, value in ((n - 1, 1, 1.0e-300), (0, diag[-1], np.nextafter(50.0, 60.0))):
        t = make(sphgpu, dim, dict(pos=pos, H=H, vel=0 * pos, mass=np.ones(n), rho=np.ones(n), eps=np.ones(n)),
                 order=1, precision=1)
        t.eos_gamma_law(1.4)
        B = H.copy()
        B[row, comp] = value
        t.upload("H", B)
        t.build_neighbors(2.0)
        with pytest.raises(sphgpu.SphGpuError):
            t.evaluate_derivatives(sphgpu.hydro_params(precision=1))


@pytest.mark.parametrize("n", [1, 524287, 524288, 524289, 917504, 1048579, 2500001])
def test_downloads_across_the_ring(sphgpu, n):
    """Copies below 4 MB, from there on through the slots: whole chunks, a part of
    one, fewer than the slots and several rounds of them."""
    rng = np.random.default_rng(n)
    s = sphgpu.Sim(1)
    s.set_nodes(n, n)
    for _ in range(2):
        a = rng.standard_normal(n)
        s.upload("mass density", a)
        assert np.array_equal(s.download("mass density"), a)
