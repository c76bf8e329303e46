"""Spread form of the step (small meshes; MPS_SPREAD=1 at any size) against the patch form (MPS_SPREAD=0): one launch per
step with an element's work spread over eight lanes, the same arithmetic and the same order of every sum, so the state,
the step history and the internal force are the same bit for bit.  Sizes at the edges of its workgroups (8 hex8, 64 tet4)
and of the patches (256 elements), whose boundary the force sums of a node must respect."""
import numpy as np
import pytest

import mps_gpu as G
from meshgen import box, clamp_and_pull, perturb
from mps_gpu import configs

pytestmark = pytest.mark.gpu


def solve(m, form, monkeypatch, precision, chunks, graphs=True, state=None, **kw):
    monkeypatch.setenv("MPS_SPREAD", form)
    dd, dv = clamp_and_pull(m)
    with G.Solver(m, dir_dof=dd, dir_val=dv, precision=precision, history_cap=256, **kw) as s:
        s.set_graphs(graphs)
        if state is not None:
            s.set_state(*state)
        s.set_loads(loads=[("gravity", 9.81)])
        for c in chunks:
            rc, rep = s.run(c)
            assert rc == 0, rep
        f = s.internal_force_dofs(np.arange(3 * m["n_nodes"], dtype=np.int32))
        h = s.history(0, rep["steps"])
        return [*s.get_state(), f, h["time"], h["dt"], np.array([rep["time"], rep["dt"], rep["steps"], rep["status"]])]


def same(m, monkeypatch, precision=G.PREC_FP64, chunks=(1, 2, 30), **kw):
    a = solve(m, "0", monkeypatch, precision, chunks, **kw)
    b = solve(m, "1", monkeypatch, precision, chunks, **kw)
    for i, (x, y) in enumerate(zip(a, b)):
        assert np.array_equal(x, y, equal_nan=True), (i, np.nanmax(np.abs(x - y)))  # thin cells may go unstable
    return a


@pytest.mark.parametrize("precision", [G.PREC_FP64, G.PREC_FP32_ELEM])
@pytest.mark.parametrize("shape", [(1, 1, 1), (7, 1, 1), (4, 2, 1), (3, 3, 1), (16, 16, 1), (257, 1, 1), (11, 9, 7)])
def test_hex_sizes(shape, precision, monkeypatch):
    same(perturb(box(*shape), 0.1, 7), monkeypatch, precision, n_steps=33)


@pytest.mark.parametrize("precision", [G.PREC_FP64, G.PREC_FP32_ELEM])
@pytest.mark.parametrize("shape", [(1, 1, 1), (5, 2, 1), (11, 1, 1), (43, 1, 1), (7, 6, 5)])
def test_tet_sizes(shape, precision, monkeypatch):
    same(perturb(box(*shape, tet=True), 0.1, 7), monkeypatch, precision, n_steps=33)


@pytest.mark.parametrize("precision", [G.PREC_FP64, G.PREC_FP32_ELEM])
@pytest.mark.parametrize("law", [0, 1, 2, 3])
@pytest.mark.parametrize("tet", [False, True])
def test_laws_and_materials(tet, law, precision, monkeypatch):
    """Per-element materials, a handed-over state with large strains (the library logarithm), every law."""
    m = perturb(box(9, 5, 6, tet=tet), 0.1, 3)
    rng = np.random.default_rng(5)
    E, nu = 10 ** rng.uniform(5, 6, m["n_elem"]), rng.uniform(0.2, 0.4, m["n_elem"])
    x = m["X"]
    state = (0.15 * x * np.sin(3 * x), 0.5 * np.cos(5 * x), 0.1 * x)
    same(m, monkeypatch, precision, n_steps=33, law=law, E=E, nu=nu, state=state)


@pytest.mark.parametrize("mode", [G.BC_RAMP, G.BC_INST])
@pytest.mark.parametrize("graphs", [False, True])
def test_time_window(mode, graphs, monkeypatch):
    """The time-window loop ends inside a launch sequence."""
    m = perturb(box(6, 5, 4), 0.1, 3)
    r = same(m, monkeypatch, chunks=(3, 256, 256), bc_mode=mode, tf=0.05, graphs=graphs)
    assert r[-1][3] == G.MPS_DONE and 3 < r[-1][2] < 515


def test_mirrored_elements(monkeypatch):
    """Cells of alternating orientation: det J < 0 in half of the elements of a wave."""
    same(configs.perturb(configs.box(6, 6, 6, reflected=True), 0.05, 3), monkeypatch, n_steps=33)


def test_forms_hand_over(monkeypatch):
    """A DOF series set between two runs sends the rest of the solve through the patch form, and back when removed."""
    m = perturb(box(8, 7, 5), 0.1, 3)
    dd, dv = clamp_and_pull(m)
    out = []
    for form in ("0", "1"):
        monkeypatch.setenv("MPS_SPREAD", form)
        with G.Solver(m, dir_dof=dd, dir_val=dv, n_steps=60) as s:
            s.run(13)
            s.set_dof_series([G.SERIES_U, G.SERIES_FINT], [5, 50])
            s.run(20)
            ser = s.dof_series(13, 20)
            s.set_dof_series([], [])
            s.run(27)
            out.append([*s.get_state(), ser])
    for x, y in zip(*out):
        assert np.array_equal(x, y)
