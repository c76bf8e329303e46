"""Edges of the one-launch step: the meshes and step modes that it leaves to the patch form also when asked for
(MPS_SPREAD=1), nodes of as many elements as its tables hold, and a time window with energies that ends inside a launch
sequence.  Every comparison of the two forms asserts which form each side ran in."""
import numpy as np
import pytest

import mps_gpu as G
from meshgen import box, clamp_and_pull, perturb
from test_gpu_spread_forms import SERIES, spread
from test_gpu_spread_modes import EXACT, SUMS

pytestmark = pytest.mark.gpu


def fan(k, before):
    """`before` tet4 elements of a bar, then k around a common edge: two nodes of k elements each."""
    m = box(before // 6, 1, 1, tet=True)
    N, ang = m["n_nodes"], 2 * np.pi * np.arange(k) / k
    ring = np.stack([3 + np.cos(ang), 3 + np.sin(ang), np.zeros(k)])
    X = np.concatenate([m["X"].reshape(3, N), [[3.0, 3.0], [3.0, 3.0], [-0.5, 0.5]], ring], axis=1)
    tets = [[N, N + 2 + i, N + 2 + (i + 1) % k, N + 1] for i in range(k)]
    conn = np.concatenate([m["conn"].reshape(-1, 4), tets]).astype(np.int32)
    return dict(n_nodes=X.shape[1], n_elem=len(conn), nen=4, X=np.ascontiguousarray(X.ravel()),
                conn=np.ascontiguousarray(conn.ravel()))


def with_free_node(m):
    N = m["n_nodes"]
    X = np.concatenate([m["X"].reshape(3, N), np.full((3, 1), 2.0)], axis=1)
    return dict(m, n_nodes=N + 1, X=np.ascontiguousarray(X.ravel()))


def both(m, monkeypatch, expected, **kw):
    out = []
    rng = np.random.default_rng(4)
    state = [s * rng.uniform(-1, 1, 3 * m["n_nodes"]) for s in (1e-3, 1e-1, 1e1)]
    for env in "01":
        monkeypatch.setenv("MPS_SPREAD", env)
        with G.Solver(m, n_steps=33, **kw) as s:
            s.set_state(*state)
            assert spread(s) == (expected and env == "1")
            rc, rep = s.run(30)
            assert rc == 0, rep
            f = s.internal_force_dofs(np.arange(3 * m["n_nodes"], dtype=np.int32))
            out.append([*s.get_state(), f, np.array([rep["time"], rep["dt"]])])
    for i, (x, y) in enumerate(zip(*out)):
        assert np.isfinite(x).all() and np.array_equal(x, y), i


@pytest.mark.parametrize("precision", [G.PREC_FP64, G.PREC_FP32_ELEM])
@pytest.mark.parametrize("before", [6, 246])  # in one patch; over the boundary of two
@pytest.mark.parametrize("k", [31, 32, 33])
def test_node_of_many_elements(k, before, precision, monkeypatch):
    both(fan(k, before), monkeypatch, k <= 32, precision=precision)


@pytest.mark.parametrize("tet", [False, True])
def test_node_of_no_element(tet, monkeypatch):
    both(with_free_node(perturb(box(5, 4, 3, tet=tet), 0.1, 3)), monkeypatch, False)


@pytest.mark.parametrize("tet", [False, True])
@pytest.mark.parametrize("precision", [G.PREC_FP64, G.PREC_FP32_ELEM])
@pytest.mark.parametrize("mode", ["plain", "energies", "viscosity", "loads", "pressure", "series", "energies and viscosity"])
def test_form_by_step_mode(mode, precision, tet, monkeypatch):
    """Asked for, the one-launch form runs these steps and no others."""
    monkeypatch.setenv("MPS_SPREAD", "1")
    m = perturb(box(6, 5, 4, tet=tet), 0.1, 3)
    dd, dv = clamp_and_pull(m)
    with G.Solver(m, dir_dof=dd, dir_val=dv, n_steps=10, precision=precision, energy_every=2 * ("energies" in mode)) as s:
        if mode in ("loads", "pressure"):
            blocks = [("gravity", 9.81), ("force", [m["n_nodes"] - 1], [[1.0, 2.0, 3.0]], 0.0, 1.0)]
            if mode == "pressure":
                blocks.append(("pressure_inst", 5.0, 0.0, 1e9, np.array([m["n_elem"] - 1]), np.array([2])))
            s.set_loads(loads=blocks)
        if "viscosity" in mode:
            s.set_viscosity(G.VISC_BULK, c1=0.5, cl=0.06)
        if mode == "series":
            s.set_dof_series(*SERIES)
        runs = mode in ("plain", "energies", "loads") or (mode == "viscosity" and not tet)
        assert spread(s) == (runs and (tet or precision == G.PREC_FP64))


@pytest.mark.parametrize("loads", [False, True])
@pytest.mark.parametrize("every", [1, 2, 7])
@pytest.mark.parametrize("shape,tet", [((6, 5, 4), False), ((11, 9, 7), False), ((5, 4, 3), True)])
def test_time_window_with_energies(shape, tet, every, loads, monkeypatch):
    """The window ends inside a launch sequence, whose last sums the end of the sequence adds up.  Tolerances of the sums:
    3 n additions of n nodes, each within 2^-53 of the largest value, times 8 for cancellation."""
    m = perturb(box(*shape, tet=tet), 0.1, 3)
    dd, dv = clamp_and_pull(m)
    out = []
    for env in "01":
        monkeypatch.setenv("MPS_SPREAD", env)
        with G.Solver(m, dir_dof=dd, dir_val=dv, bc_mode=G.BC_RAMP, tf=0.03, energy_every=every, history_cap=512) as s:
            if loads:
                s.set_loads(loads=[("gravity", 9.81), ("force", [m["n_nodes"] - 1], [[1.0, 2.0, 3.0]], 0.0, 1.0)])
            assert spread(s) == (env == "1")
            rc, rep = s.run(256)
            assert rc == 0 and rep["status"] == G.MPS_DONE and 3 < rep["steps"] < 259
            h = s.history(0, rep["steps"])
            h.update(s.energy_balance(0, rep["steps"]))
            out.append((s.get_state(), h))
    (a, ha), (b, hb) = out
    for x, y in zip(a, b):
        assert np.array_equal(x, y)
    for key in ha:
        if key in EXACT:
            assert np.array_equal(ha[key], hb[key], equal_nan=True), key
        elif key == "e_kin":
            np.testing.assert_allclose(ha[key], hb[key], rtol=1e-13, equal_nan=True)
        else:
            assert key in SUMS
            scale = np.nanmax(np.abs(ha[key]))
            np.testing.assert_allclose(ha[key], hb[key], rtol=0, atol=8 * 3 * m["n_nodes"] * 2.0 ** -53 * scale, equal_nan=True)
