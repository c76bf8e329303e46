"""Which form of the step a solve takes, and what must hold when the form changes between two runs."""
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
        rc, rep = s.run(n)
        assert rc == 0 and rep["steps"] == n and rep["status"] == G.MPS_RUNNING
        f = s.internal_force_dofs(dofs)
        s.set_dof_series(*(([], []) if series_first else SERIES))
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
