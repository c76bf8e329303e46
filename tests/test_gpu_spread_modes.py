"""Spread form of the step (MPS_SPREAD=1) with energies, bulk viscosity and external loads against the patch form
(MPS_SPREAD=0): the state and the element energies are the same bit for bit.  The node sums (works, lumped kinetic and
external energy) are added in another order: at most 3 n additions of n nodes, each within 2^-53 of the sum of the terms'
magnitudes, so their bound is 3 n 2^-53 of the largest value of the column, times 8 for cancellation among the terms.
Sizes at the edges of the workgroups (8 hex8, 64 tet4) and of the patches and sum groups (256)."""
import numpy as np
import pytest

import mps_gpu as G
from meshgen import box, clamp_and_pull, perturb

pytestmark = pytest.mark.gpu

EXACT = ("time", "dt", "e_def", "volume")
SUMS = ("e_ext", "e_kin_lumped", "w_ext", "w_react")


def solve(m, form, monkeypatch, energies=0, visc=False, loads=True, pressure=False, chunks=(1, 2, 30), **kw):
    monkeypatch.setenv("MPS_SPREAD", form)
    dd, dv = clamp_and_pull(m)
    rng = np.random.default_rng(4)
    state = [s * rng.uniform(-1, 1, 3 * m["n_nodes"]) for s in (1e-3, 1e-1, 1e1)]
    top = np.flatnonzero(m["X"][2 * m["n_nodes"]:] >= m["X"][2 * m["n_nodes"]:].max() - 1e-9)
    load = [("gravity", 9.81), ("force", [int(n) for n in top[:9]], [[3.0, -2.0, 1.0]] * len(top[:9]), 0.0, 1.0),
            ("traction_inst", (2.0, 3.0, -4.0), 0.0, 1e9, np.arange(m["n_elem"])[-3:], np.full(min(3, m["n_elem"]), 2))]
    if pressure:
        load.append(("pressure_inst", 5.0, 0.0, 1e9, np.array([m["n_elem"] - 1]), np.array([2])))
    with G.Solver(m, dir_dof=dd, dir_val=dv, n_steps=sum(chunks), history_cap=64, energy_every=energies, **kw) as s:
        s.set_state(*state)
        if loads:
            s.set_loads(loads=load)
        if visc:
            s.set_viscosity(G.VISC_BULK, c1=0.5, cl=0.06)
        for c in chunks:
            rc, rep = s.run(c)
            assert rc == 0, rep
        h = s.history(0, rep["steps"])
        if energies:
            h.update(s.energy_balance(0, rep["steps"]))
        return [*s.get_state(), s.internal_force_dofs(np.arange(3 * m["n_nodes"], dtype=np.int32))], h


def same(m, monkeypatch, **kw):
    (a, ha), (b, hb) = (solve(m, f, monkeypatch, **kw) for f in ("0", "1"))
    for i, (x, y) in enumerate(zip(a, b)):
        assert np.array_equal(x, y, equal_nan=True), (i, np.nanmax(np.abs(x - y)))  # slender bars go unstable in both forms
    for key in ha:
        if key in EXACT:
            assert np.array_equal(ha[key], hb[key], equal_nan=True), key
        elif key == "e_kin":  # a sequence's last step: the pass after it
            np.testing.assert_allclose(ha[key], hb[key], rtol=1e-13, equal_nan=True)
        elif key in SUMS:
            scale = np.nanmax(np.abs(ha[key])) if not np.isnan(ha[key]).all() else 0.0
            np.testing.assert_allclose(ha[key], hb[key], rtol=0, atol=8 * 3 * m["n_nodes"] * 2.0 ** -53 * scale, equal_nan=True)


@pytest.mark.parametrize("law", [0, 1, 2, 3])
@pytest.mark.parametrize("shape,tet,every", [((1, 1, 1), False, 1), ((3, 3, 1), False, 1), ((16, 16, 1), False, 3),
                                             ((257, 1, 1), False, 1), ((21, 11, 9), False, 2), ((1, 1, 1), True, 1),
                                             ((11, 1, 1), True, 1), ((43, 1, 1), True, 3), ((9, 7, 6), True, 2)])
def test_energies(shape, tet, every, law, monkeypatch):
    same(perturb(box(*shape, tet=tet), 0.1, 7), monkeypatch, energies=every, law=law)


@pytest.mark.parametrize("law", [0, 1, 2, 3])
@pytest.mark.parametrize("shape,tet,every", [((1, 1, 1), False, 1), ((16, 16, 1), False, 3), ((21, 11, 9), False, 2),
                                             ((11, 1, 1), True, 1), ((9, 7, 6), True, 2)])
def test_energies_fp32(shape, tet, every, law, monkeypatch):
    """FP32 forces: the energies stay FP64, in the patch form by a pass of its own with other intermediates.  F's diagonal
    is rounded at 2^-53; the strains of the state are 1e-4 and more, so energies of the strain agree to some 1e-12 (1e-11
    here), the volume to 1e-13."""
    m = perturb(box(*shape, tet=tet), 0.1, 7)
    kw = dict(energies=every, law=law, precision=G.PREC_FP32_ELEM)
    (a, ha), (b, hb) = (solve(m, f, monkeypatch, **kw) for f in ("0", "1"))
    for x, y in zip(a, b):
        assert np.array_equal(x, y)
    for key, rtol in (("time", 0), ("dt", 0), ("e_def", 1e-11), ("volume", 1e-13), ("e_kin", 1e-13)):
        np.testing.assert_allclose(ha[key], hb[key], rtol=rtol, equal_nan=True, err_msg=key)
    for key in SUMS:
        scale = np.nanmax(np.abs(ha[key])) if not np.isnan(ha[key]).all() else 0.0
        np.testing.assert_allclose(ha[key], hb[key], rtol=0, atol=8 * 3 * m["n_nodes"] * 2.0 ** -53 * scale, equal_nan=True)


@pytest.mark.parametrize("precision", [G.PREC_FP64, G.PREC_FP32_ELEM])
@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 3, 1), (16, 16, 1), (257, 1, 1), (11, 9, 7)])
def test_viscosity(shape, precision, monkeypatch):
    same(perturb(box(*shape), 0.1, 7), monkeypatch, visc=True, precision=precision, law=1)


@pytest.mark.parametrize("precision", [G.PREC_FP64, G.PREC_FP32_ELEM])
@pytest.mark.parametrize("tet", [False, True])
@pytest.mark.parametrize("pressure", [False, True])
def test_loads(pressure, tet, precision, monkeypatch):
    """Pressure loads need the step's displacement: those solves stay in the patch form."""
    same(perturb(box(9, 8, 7, tet=tet), 0.1, 7), monkeypatch, pressure=pressure, precision=precision)


def test_loads_set_after_the_graphs(monkeypatch):
    """Loads and viscosity set after a chunk was captured are in the steps that follow."""
    m = perturb(box(6, 5, 4), 0.1, 7)
    out = []
    for early in (False, True):
        dd, dv = clamp_and_pull(m)
        with G.Solver(m, dir_dof=dd, dir_val=dv, n_steps=20) as s:
            if early:
                s.prepare_run(20)
            s.set_loads(loads=[("gravity", 9.81), ("force", [m["n_nodes"] - 1], [[1.0, 2.0, 3.0]], 0.0, 10.0)])
            s.set_viscosity(G.VISC_BULK, c1=0.5, cl=0.06)
            assert s.run(20)[0] == 0
            out.append(s.get_state())
    for x, y in zip(*out):
        assert np.array_equal(x, y)
