"""Which form of the step a solve takes, and what must hold when the form changes between two runs."""
import ctypes

import numpy as np
import pytest

import mps_gpu as G
from meshgen import box, clamp_and_pull, perturb

pytestmark = pytest.mark.gpu

SERIES = ([G.SERIES_U, G.SERIES_FINT], [5, 50])


def window(m, tf, **kw):
    dd, dv = clamp_and_pull(m)
    return G.Solver(m, dir_dof=dd, dir_val=dv, tf=tf, bc_mode=G.BC_RAMP, **kw)


@pytest.mark.parametrize("tet", [False, True])
@pytest.mark.parametrize("series_first", [False, True])
def test_forces_after_a_run_without_a_step(series_first, tet):
    """A time window that ends with the last step of a run: the next run finds the end and begins no step.  A DOF series set
    or removed in between sends that run through the other form; the forces are still those of the last step."""
    m = perturb(box(8, 7, 5, tet=tet), 0.1, 3)
    dofs = np.arange(3 * m["n_nodes"], dtype=np.int32)
    with window(m, 0.02) as s:
        _, rep = s.run(1 << 20)
        assert rep["status"] == G.MPS_DONE
        n = rep["steps"]
    with window(m, 0.02) as s:
        s.set_dof_series(*(SERIES if series_first else ([], [])))
        s.prepare_run(n)
        rc, rep = s.run(n)
        assert rc == 0 and rep["steps"] == n and rep["status"] == G.MPS_RUNNING
        f = s.internal_force_dofs(dofs)
        s.set_dof_series(*(([], []) if series_first else SERIES))
        s.prepare_run(5)
        rc, rep = s.run(5)
        assert rc == 0 and rep["steps"] == n and rep["status"] == G.MPS_DONE
        assert np.array_equal(s.internal_force_dofs(dofs), f)


@pytest.mark.parametrize("series", [False, True])
def test_forces_after_a_first_step_that_fails(series):
    """The first step ends with its time step too small: the forces are those of the state handed over, in both forms."""
    m = perturb(box(6, 5, 4), 0.1, 3)
    dd, dv = clamp_and_pull(m)
    dofs = np.arange(3 * m["n_nodes"], dtype=np.int32)
    u = 1e-2 * np.random.default_rng(2).uniform(-1, 1, 3 * m["n_nodes"])
    with G.Solver(m, dir_dof=dd, dir_val=dv, n_steps=10, scale=1e-30) as s:
        s.set_state(u)
        if series:
            s.set_dof_series(*SERIES)
        rc, rep = s.run(10)
        assert rc == G.MPS_ERR_DT and rep["steps"] == 0
        f = s.internal_force_dofs(dofs)
    with G.Solver(m, dir_dof=dd, dir_val=dv, n_steps=10) as s:
        s.set_state(u)
        assert np.array_equal(s.internal_force_dofs(dofs), f)


def spread(s):
    """True when the next steps of s run in the spread form: one launch per step and one at the end, where the patch form
    has a node kernel in every step."""
    s.prepare_run(3)
    s.profile(True)
    before = s.kernel_times()["node"][1]
    rc, rep = s.run(3)
    assert rc == 0, rep
    n = s.kernel_times()["node"][1] - before
    s.profile(False)
    assert n in (1, 3), n
    return n == 1


def form(m, **kw):
    dd, dv = clamp_and_pull(m)
    with G.Solver(m, dir_dof=dd, dir_val=dv, n_steps=10, **kw) as s:
        return spread(s)


@pytest.mark.parametrize("shape,tet,precision,every,expected", [
    ((33, 33, 33), False, G.PREC_FP64, 0, True), ((34, 34, 34), False, G.PREC_FP64, 0, False),
    ((34, 34, 34), False, G.PREC_FP64, 1, True), ((34, 34, 34), False, G.PREC_FP64, 2, True),
    ((34, 34, 34), False, G.PREC_FP64, 3, False), ((33, 33, 33), False, G.PREC_FP64, 100, True),
    ((36, 36, 35), False, G.PREC_FP64, 1, False), ((36, 36, 35), False, G.PREC_FP64, 100, False),
    ((22, 22, 22), True, G.PREC_FP64, 0, True), ((22, 23, 22), True, G.PREC_FP64, 0, False),
    ((24, 24, 24), True, G.PREC_FP64, 2, True), ((24, 24, 24), True, G.PREC_FP64, 5, False),
    ((22, 22, 22), True, G.PREC_FP32_ELEM, 100, True), ((24, 24, 24), True, G.PREC_FP32_ELEM, 100, False),
    ((24, 24, 24), True, G.PREC_FP32_ELEM, 1, True), ((25, 25, 26), True, G.PREC_FP64, 1, False),
])
def test_form_by_size_and_energy_interval(shape, tet, precision, every, expected, monkeypatch):
    """The limits of the one-launch form where the energy interval moves them."""
    monkeypatch.delenv("MPS_SPREAD", raising=False)
    assert form(box(*shape, tet=tet), precision=precision, energy_every=every) == expected


@pytest.mark.parametrize("cells,window,precision,every,expected", [
    (14, 1, G.PREC_FP64, 0, True), (14, 512, G.PREC_FP64, 0, False), (14, 256, G.PREC_FP64, 0, True),
    (14, 256, G.PREC_FP32_ELEM, 0, False), (12, 256, G.PREC_FP32_ELEM, 0, True), (8, 1 << 20, G.PREC_FP32_ELEM, 0, False),
    (9, 1 << 20, G.PREC_FP64, 0, True), (17, 1 << 20, G.PREC_FP64, 0, False), (17, 1, G.PREC_FP32_ELEM, 0, True),
    (18, 1, G.PREC_FP32_ELEM, 0, False), (14, 512, G.PREC_FP64, 1, True), (20, 512, G.PREC_FP64, 1, False),
    (14, 512, G.PREC_FP32_ELEM, 50, False), (12, 512, G.PREC_FP32_ELEM, 50, True),
])
def test_form_by_element_order(cells, window, precision, every, expected, monkeypatch):
    """Tet4 elements shuffled in windows: the one-launch form is for meshes whose workgroups share few nodes."""
    monkeypatch.delenv("MPS_SPREAD", raising=False)
    m = box(cells, cells, cells, tet=True)
    rng, ne = np.random.default_rng(1), m["n_elem"]
    order = np.concatenate([i + rng.permutation(min(window, ne - i)) for i in range(0, ne, window)])
    m["conn"] = np.ascontiguousarray(m["conn"].reshape(-1, 4)[order].ravel())
    assert form(m, precision=precision, energy_every=every) == expected


def test_set_up_only_where_it_is_used(monkeypatch):
    """The tables and buffers of the one-launch form (18 MB for this mesh) are those of solves that step in it: not of one
    with a pressure load, nor of one that is only created, and with a series of one from which it is taken away."""
    hip = ctypes.CDLL("libamdhip64.so")
    monkeypatch.delenv("MPS_SPREAD", raising=False)
    m = perturb(box(33, 33, 33), 0.1, 3)
    dd, dv = clamp_and_pull(m)

    def free():
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value / 2 ** 20

    def grown(**kw):
        """MB in use once created, after 3 steps with a pressure load or a series, after 3 more without the series."""
        start = free()
        with G.Solver(m, dir_dof=dd, dir_val=dv, n_steps=10) as s:
            out = [start - free()]
            if kw.get("pressure"):
                s.set_loads(loads=[("pressure_inst", 5.0, 0.0, 1e9, np.array([m["n_elem"] - 1]), np.array([2]))])
            if kw.get("series"):
                s.set_dof_series(*SERIES)
            s.prepare_run(3)
            assert s.run(3)[0] == 0
            out.append(start - free())
            s.set_dof_series([], [])
            s.prepare_run(3)
            assert s.run(3)[0] == 0
            out.append(start - free())
        return np.array(out)

    grown()
    created, run, _ = grown()
    assert run > created + 12
    assert grown(pressure=True).max() < created + 6
    _, with_series, without = grown(series=True)
    assert with_series < created + 6 and without > created + 12


def test_set_up_after_enough_steps(monkeypatch):
    """Without mps_prepare_run the set-up waits for as many steps as pay for it (n^2 / 2^21 of n hex8 elements); the steps
    before it run in the patch form, and the state is the same as in either form alone."""
    m = perturb(box(16, 16, 32), 0.1, 3)  # 8,192 elements: 32 steps
    dd, dv = clamp_and_pull(m)
    out = []
    for env in (None, "0", "1"):
        monkeypatch.setenv("MPS_SPREAD", env) if env else monkeypatch.delenv("MPS_SPREAD", raising=False)
        with G.Solver(m, dir_dof=dd, dir_val=dv, n_steps=100) as s:
            s.profile(True)
            nodes = []
            for n in (15, 15, 1, 1, 36):
                before = s.kernel_times()["node"][1]
                assert s.run(n)[0] == 0
                nodes.append(s.kernel_times()["node"][1] - before)
            assert nodes == {None: [15, 15, 1, 1, 1], "0": [15, 15, 1, 1, 36], "1": [1] * 5}[env]
            out.append([*s.get_state(), s.internal_force_dofs(np.arange(3 * m["n_nodes"], dtype=np.int32))])
    for a, b, c in zip(*out):
        assert np.array_equal(a, b) and np.array_equal(a, c)
    monkeypatch.delenv("MPS_SPREAD", raising=False)
    with G.Solver(m, dir_dof=dd, dir_val=dv, n_steps=31) as s:  # asked for more than the solve has
        s.profile(True)
        assert s.run(1 << 40)[1]["steps"] == 31 and s.kernel_times()["node"][1] == 31
