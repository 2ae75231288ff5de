"""Both sides of the lines between one lane and several lanes to a node, against the
oracle: the lines of each step of 65536 nodes, and the options that the one-lane, 8-lane
and 16-lane kernels take (tensile term, Q multipliers, any H, several NodeLists, stored
pair accelerations).  Bars as elsewhere: reference row order equal value for value
(cube-root fields in 3-D 1e-14), search row order 1e-12, mixed precision 1e-5."""
import numpy as np
import pytest

import test_gpu_dispatch as dispatch
import test_gpu_nodelists as nodelists
from sphgpu import problems

pytestmark = pytest.mark.gpu

# nodes: 2-D 48841 | 49284, 57121 | 57600, 97969 | 98596, 106276 | 106929, 131044 | 131769,
# 262144 | 263169; 3-D 39304 | 42875, 54872 | 59319 | 64000, 91125 | 97336, (132651 |) 140608
SIZES = [(2, 221), (2, 222), (2, 239), (2, 240), (2, 313), (2, 314), (2, 326), (2, 327), (2, 362), (2, 363),
         (2, 512), (2, 513), (3, 34), (3, 35), (3, 38), (3, 39), (3, 45), (3, 46), (3, 52)]


@pytest.mark.parametrize("dim,n", SIZES)
def test_pass_at_the_lines(sphgpu, oracle, dim, n):
    dispatch.test_pass_across_lanes(sphgpu, oracle, dim, n)


def any_H(dim, N, h0, seed):
    """Rotated H of +-20 % anisotropy, all nodes at once."""
    rng = np.random.default_rng(seed)
    Q, _ = np.linalg.qr(rng.standard_normal((N, dim, dim)))
    lam = 1.0 / (h0 * (1.0 + 0.2 * rng.uniform(-1, 1, (N, dim))))
    H = np.einsum("nij,nj,nkj->nik", Q, lam, Q)
    a, b = np.triu_indices(dim)
    return np.ascontiguousarray(H[:, a, b])


def option_state(dim, n, option):
    st, meta = problems.random_state(dim, n, seed=320 + n, jitter=0.15, h_var=0.1)
    N = st["pos"].shape[0]
    kw = {}
    if option == "any H":
        st["H"] = any_H(dim, N, 1.51 * meta["dx"], 330 + n)
    elif option == "multipliers":
        rng = np.random.default_rng(340 + n)
        st.update(fCl=rng.uniform(0.5, 1.5, N), fCq=rng.uniform(0.5, 1.5, N), fshear=rng.uniform(0, 1, N))
        kw["linearInExpansion"] = 1
    else:
        st["P"] = st["P"] * np.where(np.arange(N) % 3 == 0, -1.0, 1.0)      # tension on a third of the nodes
        kw["epsTensile"] = 0.25
    return st, kw


# 16 lanes; 8 lanes; one lane to the pair pass in the first and second step; one lane to the
# density sum and the grad-h correction as well (any H); 3-D: 8 and 16 lanes, one lane to the
# pairs, one lane to all
@pytest.mark.parametrize("option", ["any H", "multipliers", "tensile"])
@pytest.mark.parametrize("dim,n", [(2, 128), (2, 129), (2, 250), (2, 287), (2, 340), (3, 25), (3, 26), (3, 50),
                                   (3, 55)])
def test_options_at_every_lane_count(sphgpu, oracle, dim, n, option):
    st, kw = option_state(dim, n, option)
    N = st["pos"].shape[0]
    print(f"[options] {option} dim={dim} N={N}", flush=True)
    off, nbr = oracle.connectivity(dim, N, st["pos"], st["H"])
    T = oracle.Table(dim, 1000)
    rho = oracle.sum_density(T, N, st["pos"], st["mass"], st["H"], off, nbr, gather=True)
    full = dict(st, rho=rho)
    ref = oracle.eval_derivs(T, oracle.make_params(**kw), N, full, off, nbr, gather=True)
    om = oracle.omega_gradh(T, N, st["pos"], st["H"], off, nbr)
    s = dispatch.make(sphgpu, dim, st)
    s.build_neighbors(2.0)
    s.sum_density()
    assert np.array_equal(s.download("mass density", rows=N), rho)
    s.evaluate_derivatives(sphgpu.hydro_params(**kw))
    for f in sphgpu.DERIV_ALIASES:
        a = s.derivative(f).reshape(ref[f].shape)
        if dim == 3 and f in dispatch.POW_FIELDS:
            assert dispatch.rel(a, ref[f]) <= 1e-14, f
        else:
            assert np.array_equal(a, ref[f]), f
    s.omega_gradh()
    assert np.array_equal(s.download("grad h corrections", rows=N), om)


@pytest.mark.parametrize("dim,n", [(2, 128), (2, 129), (2, 250), (2, 287), (3, 25), (3, 26), (3, 50), (3, 55)])
def test_nodelists_at_every_lane_count(sphgpu, oracle, dim, n):
    nodelists.test_pass_with_nodelists(sphgpu, oracle, (dim, n, "reflecting"), 0, False)


@pytest.mark.parametrize("n", [49, 50, 54])
def test_stored_pair_terms_at_the_lines(sphgpu, oracle, n):
    """Compatible energy in 3-D: 117649 | 125000 nodes and 157464, 8 lanes to the pair
    pass, one, 8."""
    dispatch.test_compatible_energy_across_lanes(sphgpu, oracle, 3, n)


@pytest.mark.parametrize("n", [32768, 32769])
def test_ideal_h_and_compatible_energy_on_a_line(sphgpu, oracle, n):
    """1-D: 8 lanes to a node and one."""
    dispatch.test_ideal_h_across_lanes(sphgpu, oracle, 1, n)
    dispatch.test_compatible_energy_across_lanes(sphgpu, oracle, 1, n)
